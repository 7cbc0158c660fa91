// What the two GDN2 chunk loops (the forward state, the backward dh) share.
//
// Both walk the chunks of one (batch, head, V tile) with the state in MFMA
// accumulators.  Their operands (w_pseudo, qg, kg [64][K], Aqk [64][64]) go
// from global memory to LDS by loader waves of their own that keep about two
// chunks in flight, so the waves that compute only read LDS and meet two
// barriers a chunk.  Loading MFMA fragments straight from the row-major arrays
// does not pay: sixteen lanes on sixteen rows get 38 GB/s per CU where
// consecutive lanes on consecutive addresses get 150 GB/s (both from L2).
// The LDS rows are not padded (a load writes 1 KB in lane order), so the
// 16-byte pieces of a row are permuted by an XOR with the row number instead:
// that is done in the lanes' global addresses and keeps both the row and the
// transposed fragment reads free of bank conflicts.
#pragma once
#include "gdn2.hpp"

namespace ah {

// Byte offset of element (row, col) of an unpadded [rows][VT] bf16 array: rows
// 8..15 of every 16 half the banks away from rows 0..7, which the transposed
// reads of a half wave pair up.
template <int VT>
__device__ __forceinline__ int seq_off(int row, int col) {
  static_assert(VT == 16 || VT == 32, "32- or 64-byte rows");
  if constexpr (VT == 16) return (row ^ (((row >> 3) & 1) << 2)) * 32 + col * 2;
  else return row * 64 + ((col * 2) ^ (((row >> 3) & 1) << 5));
}
// Fragment with i = column 16 u + (lane & 15), k = row k0 .. k0 + 31 of such an array.
template <int VT>
__device__ __forceinline__ bf16x8 seq_colfrag(const unsigned char* s, int u, int k0) {
  typedef __attribute__((address_space(3))) bf16x4* lds_p;
  const int l = lane_id(), row = 8 * (l >> 4) + ((l & 15) >> 2), col = 16 * u + 4 * (l & 3);
  const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_p)(s + k0 * VT * 2 + seq_off<VT>(row, col)));
  const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_p)(s + k0 * VT * 2 + seq_off<VT>(row + 4, col)));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// The same of a [64][8 NP] block whose 16-byte pieces are permuted: piece p of
// row r at slot p ^ (r & (NP - 1)).
template <int NP>
__device__ __forceinline__ bf16x8 swz_colfrag(const unsigned char* s, int i0, int k0) {
  typedef __attribute__((address_space(3))) bf16x4* lds_p;
  const int l = lane_id(), row = 8 * (l >> 4) + ((l & 15) >> 2), pc = (i0 >> 3) + ((l & 3) >> 1);
  const unsigned char* b = s + k0 * NP * 16 + (l & 1) * 8;
  const bf16x4 lo =
      __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_p)(b + row * NP * 16 + ((pc ^ (row & (NP - 1))) * 16)));
  const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
      (lds_p)(b + (row + 4) * NP * 16 + ((pc ^ ((row + 4) & (NP - 1))) * 16)));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// Fragment with i = row i0 + (lane & 15), k = column 32 ks ... of such a block (i0 a multiple of 16).
template <int NP>
__device__ __forceinline__ bf16x8 swz_rowfrag(const unsigned char* s, int i0, int ks) {
  const int l = lane_id(), r = l & 15;
  return *reinterpret_cast<const bf16x8*>(s + (i0 + r) * NP * 16 + (((4 * ks + (l >> 4)) ^ (r & (NP - 1))) * 16));
}
// A fragment's 16 rows of 32 columns to global rows of ld elements: the 16
// bytes that lane (r, g) holds of row r move to lane 4 r + g, so that four
// consecutive lanes write 64 consecutive bytes.
__device__ __forceinline__ void store_frag_rows(bf16* dst, int ld, bf16x8 a) {
  const int l = lane_id(), from = 4 * ((l >> 2) + 16 * (l & 3));
  const u32x4 p = __builtin_bit_cast(u32x4, a);
  u32x4 q;
#pragma unroll
  for (int i = 0; i < 4; ++i) q[i] = __builtin_amdgcn_ds_bpermute(from, p[i]);
  *reinterpret_cast<u32x4*>(dst + (size_t)(l >> 2) * ld + 8 * (l & 3)) = q;
}

// Kilobyte i of the 16 rows of 32 NK columns that NK fragments hold, rows dense:
// lane l's 16 bytes of it come from fragment (piece / 4), lane (row, piece & 3).
template <int NK>
__device__ __forceinline__ void store_frags_1k(bf16* dst, int i, const bf16x8 (&a)[NK]) {
  constexpr int PP = 4 * NK;  // pieces a row
  const int e = 64 * i + lane_id(), pc = e % PP, from = 4 * (e / PP + 16 * (pc & 3));
  u32x4 q = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int s = 0; s < NK; ++s) {
    const u32x4 p = __builtin_bit_cast(u32x4, a[s]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t x = __builtin_amdgcn_ds_bpermute(from, p[j]);
      q[j] = (pc >> 2) == s ? x : q[j];
    }
  }
  *reinterpret_cast<u32x4*>(dst + e * 8) = q;
}

// dma16, or (AL = false) the same through registers, from any address.  The wave
// that issues these has to see the LDS writes done too before the barrier.
template <bool AL>
__device__ __forceinline__ void copy16(const void* src, void* dst) {
  if constexpr (AL) {
    dma16(src, dst);
  } else {
    u32x4 v;
    __builtin_memcpy(&v, src, 16);
    *reinterpret_cast<u32x4*>(static_cast<unsigned char*>(dst) + lane_id() * 16) = v;
  }
}
template <bool AL>
__device__ __forceinline__ void loader_barrier() {
  if constexpr (AL) bare_barrier();
  else __syncthreads();
}

// Loader wave lw of NL: its share of a [64][K] bf16 block (row pieces permuted
// as above); 64 K 2 / 1024 / NL instructions.
template <int K, int NL, bool AL>
__device__ __forceinline__ void dma_rows(const bf16* src, unsigned char* dst, int lw) {
  constexpr int NP = K / 8, NI = 64 * K * 2 / 1024, RPI = 1024 / (2 * K);
  static_assert(NI % NL == 0, "the instructions split evenly over the loader waves");
  constexpr int UF = AL ? NI / NL : 4;  // through registers: few at a time
#pragma unroll UF
  for (int i = 0; i < NI / NL; ++i) {
    const int ins = lw * (NI / NL) + i;
    const int row = ins * RPI + lane_id() / NP, slot = lane_id() % NP;
    copy16<AL>(src + row * K + ((slot ^ (row & (NP - 1))) * 8), dst + ins * 1024);
  }
}
// One of `parts` equal shares of an array's cache lines into L2.
__device__ __forceinline__ void touch_lines(const void* base, int bytes, int parts, int part, void* scratch) {
  const int lines = bytes / 128 / parts;
  for (int l0 = 0; l0 < lines; l0 += 64)
    if (l0 + lane_id() < lines)
      dma_touch(static_cast<const char*>(base) + (size_t)(part * lines + l0 + lane_id()) * 128, scratch);
}

}  // namespace ah
