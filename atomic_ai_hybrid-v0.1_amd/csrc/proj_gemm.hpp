// bf16 MFMA GEMMs of the Mamba2 projection prologue (gfx950), with the
// kernels around them: weight packing, the element-wise VJP of the
// projection epilogue and the weight-gradient reduction.
//
//   gemm_nt   C[M][N] = A[M][K] . Bt[N][K]^T, both operands K-contiguous with
//             row strides (the in_proj half x_bc is read in place), fp32
//             accumulation, the result handed to an epilogue functor.
//   gemm_tn   P[s][K][N] = sum over the rows m of split s of X[m][K] D[m][N]
//             (the weight gradient X^T D over the tokens), fp32 partials.
//
// Tiles: 256 x 256 per workgroup of eight waves where the sizes allow (the _big
// kernels); else one 128 x BN block of C per workgroup of four waves (2 x 2, each
// 64 x BN/2 as v_mfma_f32_16x16x32_bf16 tiles; BN = 256 where N allows, else
// 128); the reduction dimension in steps of 64 through one LDS stage: the
// next step's 16-byte pieces are loaded into registers while the current
// step's MFMAs run, and stored after a barrier.
#pragma once
#include "common.hpp"

namespace ah {

constexpr int kGT = 128;       // C tile rows (M)
constexpr int kGK = 64;        // reduction step
constexpr int kGP = kGK + 8;   // NT staging row pitch (elements): 16 rows of a fragment read hit distinct banks
constexpr int kTP = kGT + 16;  // TN staging row pitch: four rows of a transposed read hit distinct banks

__device__ __forceinline__ float bf16r(float x) { return (float)(bf16)x; }

// 4 x 4 transpose inside each lane quad: lane (4 a + j) holds v[k] = M[j][k]
// on entry and v[k] = M[k][j] on return (M the quad's 4 x 4 block), by two
// exchange steps (quad partners l ^ 2, then l ^ 1).  Applied to an MFMA
// result tile (lane: rows 4 g + k, column c) it leaves the lane with row
// 4 g + (c & 3) and the four columns (c & ~3) .. + 3, so stores are vectors.
__device__ __forceinline__ void quad_transpose(float (&v)[4]) {
  const int l = lane_id();
  {
    const bool hi = (l & 2) != 0;
    const float s0 = hi ? v[0] : v[2], s1 = hi ? v[1] : v[3];
    const float r0 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s0), 0x4E, 0xF, 0xF, false));
    const float r1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s1), 0x4E, 0xF, 0xF, false));
    v[0] = hi ? r0 : v[0];
    v[1] = hi ? r1 : v[1];
    v[2] = hi ? v[2] : r0;
    v[3] = hi ? v[3] : r1;
  }
  {
    const bool odd = (l & 1) != 0;
    const float s0 = odd ? v[0] : v[1], s1 = odd ? v[2] : v[3];
    const float r0 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s0), 0xB1, 0xF, 0xF, false));
    const float r1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s1), 0xB1, 0xF, 0xF, false));
    v[0] = odd ? r0 : v[0];
    v[2] = odd ? r1 : v[2];
    v[1] = odd ? v[1] : r0;
    v[3] = odd ? v[3] : r1;
  }
}

__device__ __forceinline__ void st4bf(bf16* p, const float (&v)[4]) {
  bf16x4 o;
  o[0] = (bf16)v[0]; o[1] = (bf16)v[1]; o[2] = (bf16)v[2]; o[3] = (bf16)v[3];
  *reinterpret_cast<bf16x4*>(p) = o;
}
__device__ __forceinline__ void ld4bf(const bf16* p, float (&v)[4]) {
  const bf16x4 t = *reinterpret_cast<const bf16x4*>(p);
  v[0] = (float)t[0]; v[1] = (float)t[1]; v[2] = (float)t[2]; v[3] = (float)t[3];
}

// ---------------------------------------------------------------- NT GEMM
struct GemmNT {
  const bf16* A;   // [M][K], row stride lda
  long long lda;
  const bf16* Bt;  // [N][K], row stride ldb
  long long ldb;
  int M, N, K;     // multiples of 128, BN, 64
};

// One 128 x BN tile of C per workgroup: waves in a 2 x 2 grid, each 64 x BN/2
// as 4 x (BN / 32) MFMA tiles.  One LDS stage: the next step's pieces are
// loaded into registers while the current step's MFMAs read the stage, then
// stored after a barrier.  The epilogue gets each wave's block (rows m0..,
// columns n0..) as acc[i][j], the 16 x 16 tile at rows m0 + 16 i, columns n0 + 16 j.
template <int BN, typename Epi>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_nt(GemmNT g, Epi epi) {
  constexpr int NJ = BN / 32, PB = BN / 32;  // tiles per wave along N; Bt pieces per thread
  __shared__ __attribute__((aligned(16))) bf16 sA[kGT * kGP];
  __shared__ __attribute__((aligned(16))) bf16 sB[BN * kGP];
  typedef Mma<bf16>::frag frag;
  const int tid = threadIdx.x, w = wave_id();
  const int ntn = g.N / BN;
  const int tm = blockIdx.x / ntn, tn = blockIdx.x % ntn;  // consecutive workgroups share the A rows
  const bf16* Ag = g.A + (size_t)tm * kGT * g.lda;
  const bf16* Bg = g.Bt + (size_t)tn * BN * g.ldb;
  u32x4 ra[4], rb[PB];
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + 256 * i, r = e >> 3, c = (e & 7) * 8;
      ra[i] = *reinterpret_cast<const u32x4*>(Ag + (size_t)r * g.lda + k0 + c);
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int e = tid + 256 * i, r = e >> 3, c = (e & 7) * 8;
      rb[i] = *reinterpret_cast<const u32x4*>(Bg + (size_t)r * g.ldb + k0 + c);
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + 256 * i, r = e >> 3, c = (e & 7) * 8;
      *reinterpret_cast<u32x4*>(&sA[r * kGP + c]) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int e = tid + 256 * i, r = e >> 3, c = (e & 7) * 8;
      *reinterpret_cast<u32x4*>(&sB[r * kGP + c]) = rb[i];
    }
  };
  f32x4 acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = zero4();
  const int wm = (w >> 1) * 64, wn = (w & 1) * (BN / 2);
  const int nk = g.K / kGK;
  gload(0);
  lstore();
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 1 < nk) gload((kt + 1) * kGK);
#pragma unroll
    for (int ks = 0; ks < kGK; ks += 32) {
      frag af[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = Mma<bf16>::ld_c(sA, kGP, wm + 16 * i, ks);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const frag bfr = Mma<bf16>::ld_c(sB, kGP, wn + 16 * j, ks);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i][j] = Mma<bf16>::mma(af[i], bfr, acc[i][j]);
      }
    }
    if (kt + 1 < nk) {
      __syncthreads();  // every wave is done reading the stage
      lstore();
      __syncthreads();
    }
  }
  epi(tm * kGT + wm, tn * BN + wn, acc);
}

// 256 x 256 tiles, one workgroup of eight waves per CU (each 128 x 64), the
// reduction in steps of 32 through four LDS stages that the waves load without
// registers three steps ahead; one barrier a step.  Per CU a step reads 96 KB
// of fragments for 1024 cycles of MFMA per SIMD.  Stage rows of 64 bytes, their
// four pieces permuted by (row / 4) & 3 (in the loads' global addresses), so
// that a fragment read meets no bank conflict.  Bit-identical to gemm_nt.
// M 32768, bf16 result: 1792 x 1536 0.271 -> 0.239 ms (754 TFLOP/s; 3.5 rounds of
// tiles), 1536 x 1792 0.262 -> 0.215 (839); with their epilogues 0.330 -> 0.282
// and 0.272 -> 0.230.  Two alternating groups of waves
// (one reading LDS, one on MFMA) gave 2 % more here and less in gemm_tn_big.
constexpr int kBigT = 256, kBigK = 32, kBigS = 4;

template <typename Epi>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_nt_big(GemmNT g, Epi epi) {
  constexpr int SB = kBigT * kBigK * 2;   // bytes of one operand's stage
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kBigS * 2 * SB];
  const int w = wave_id(), lane = lane_id();
  int tm, tn;
  xcd_group_map(blockIdx.x, g.M / kBigT, g.N / kBigT, tm, tn);
  const int nk = g.K / kBigK;
  // this wave's four loads of a stage: 16 rows of 64 bytes each (waves 0-3 A, 4-7 B)
  const bool isb = w >= 4;
  const bf16* base = isb ? g.Bt + (size_t)tn * kBigT * g.ldb : g.A + (size_t)tm * kBigT * g.lda;
  const long long ld = isb ? g.ldb : g.lda;
  const char* src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 64 * (w & 3) + 16 * i + (lane >> 2);
    const int piece = (lane & 3) ^ ((row >> 2) & 3);
    src[i] = reinterpret_cast<const char*>(base + (size_t)row * ld + piece * 8);
  }
  const uint32_t l0 = lds_addr(lds) + (isb ? SB : 0) + (w & 3) * 4096;
  auto issue = [&](int t) {
    const uint32_t d = l0 + (t % kBigS) * 2 * SB;
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16_raw(src[i] + (size_t)t * (kBigK * 2), d + i * 1024);
  };
  f32x4 acc[2][4][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][i][j] = zero4();
  const int wm = 128 * (w >> 2), wn = 64 * (w & 3);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int fo = r16 * 64 + ((g4 ^ ((r16 >> 2) & 3)) * 16);   // a fragment row's 16 bytes within its 16 rows
  issue(0); issue(1); issue(2);
  for (int t = 0; t < nk; ++t) {
    if (t + 2 < nk) vm_wait<8>();
    else vm_wait<0>();
    bare_barrier();
    if (t + 3 < nk) issue(t + 3);
    const unsigned char* sA = lds + (t % kBigS) * 2 * SB + wm * 64 + fo;
    const unsigned char* sB = lds + (t % kBigS) * 2 * SB + SB + wn * 64 + fo;
    bf16x8 bf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bf[j] = *reinterpret_cast<const bf16x8*>(sB + j * 1024);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bf16x8 af = *reinterpret_cast<const bf16x8*>(sA + (4 * h + i) * 1024);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[h][i][j] = Mma<bf16>::mma(af, bf[j], acc[h][i][j]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's reads of the stage are done
  }
  // The epilogue takes whole 16-byte row pieces (four consecutive lanes of an MFMA
  // tile hold four rows, and stored from there a wave wrote 32 bytes of each of
  // 16 rows: the forward 0.335 ms): each wave's 64 x 64 halves pass through LDS as bf16.
  __syncthreads();  // the last stage is read
  bf16* st = reinterpret_cast<bf16*>(lds) + w * 64 * 72;
  const int c = tile_col();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v[4] = {acc[h][i][j][0], acc[h][i][j][1], acc[h][i][j][2], acc[h][i][j][3]};
        quad_transpose(v);
        st4bf(st + (16 * i + tile_row(0) + (c & 3)) * 72 + 16 * j + (c & ~3), v);
      }
    wave_lds_sync();
#pragma unroll 2
    for (int p = 0; p < 8; ++p) {
      const int r = 8 * p + (lane >> 3), cc = 8 * (lane & 7);
      float v[8];
      load8(st + r * 72 + cc, v);
      epi.row8(tm * kBigT + wm + 64 * h + r, tn * kBigT + wn + cc, v);
    }
    wave_lds_sync();  // the rows are rewritten next
  }
}

// ---------------------------------------------------------------- TN GEMM
struct GemmTN {
  const bf16* X;  // [M][Kd], row stride ldx
  long long ldx;
  const bf16* D;  // [M][N], row stride ldd
  long long ldd;
  int Kd, N;      // multiples of 128 and BN
  int rows;       // rows per split (a multiple of 64; 32 in gemm_tn_big); split s covers
                  // rows [s rows, (s + 1) rows), in gemm_tn_big no further than M
  float* part;    // [splits][Kd][N]
  int M;
};

// P[s] tile (128 x BN) = X^T D over the split's rows, both operands staged as
// 64-row tiles and read transposed (ds_read_b64_tr_b16) as the MFMA fragments.
template <int BN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_tn(GemmTN g) {
  constexpr int NJ = BN / 32, PD = BN / 32, LD = BN + 16;
  __shared__ __attribute__((aligned(16))) bf16 sX[kGK * kTP];
  __shared__ __attribute__((aligned(16))) bf16 sD[kGK * LD];
  typedef Mma<bf16>::frag frag;
  const int tid = threadIdx.x, w = wave_id();
  const int ntn = g.N / BN, ntk = g.Kd / kGT;
  const int s = blockIdx.x / (ntk * ntn), t = blockIdx.x % (ntk * ntn);
  const int tk = t / ntn, tn = t % ntn;
  const bf16* Xg = g.X + (size_t)s * g.rows * g.ldx + tk * kGT;
  const bf16* Dg = g.D + (size_t)s * g.rows * g.ldd + tn * BN;
  u32x4 ra[4], rb[PD];
  auto gload = [&](int m0) {  // 64 rows x 128 columns of X, 64 x BN of D
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + 256 * i, r = e >> 4, c = (e & 15) * 8;
      ra[i] = *reinterpret_cast<const u32x4*>(Xg + (size_t)(m0 + r) * g.ldx + c);
    }
#pragma unroll
    for (int i = 0; i < PD; ++i) {
      const int e = tid + 256 * i, r = e / (BN / 8), c = (e % (BN / 8)) * 8;
      rb[i] = *reinterpret_cast<const u32x4*>(Dg + (size_t)(m0 + r) * g.ldd + c);
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + 256 * i, r = e >> 4, c = (e & 15) * 8;
      *reinterpret_cast<u32x4*>(&sX[r * kTP + c]) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < PD; ++i) {
      const int e = tid + 256 * i, r = e / (BN / 8), c = (e % (BN / 8)) * 8;
      *reinterpret_cast<u32x4*>(&sD[r * LD + c]) = rb[i];
    }
  };
  f32x4 acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = zero4();
  const int wm = (w >> 1) * 64, wn = (w & 1) * (BN / 2);
  const int nk = g.rows / kGK;
  gload(0);
  lstore();
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 1 < nk) gload((kt + 1) * kGK);
#pragma unroll
    for (int ks = 0; ks < kGK; ks += 32) {
      // A(k, m) = X[m][k] and B(m, n) = D[m][n]: both read transposed from the row tiles
      frag af[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = Mma<bf16>::ld_t(sX, kTP, wm + 16 * i, ks);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const frag bfr = Mma<bf16>::ld_t(sD, LD, wn + 16 * j, ks);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i][j] = Mma<bf16>::mma(af[i], bfr, acc[i][j]);
      }
    }
    if (kt + 1 < nk) {
      __syncthreads();
      lstore();
      __syncthreads();
    }
  }
  // partial tile, stored as 4-column vectors after a quad transpose
  float* P = g.part + (size_t)s * g.Kd * g.N;
  const int c = tile_col();
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      quad_transpose(v);
      const int row = tk * kGT + wm + 16 * i + tile_row(0) + (c & 3);
      const int col = tn * BN + wn + 16 * j + (c & ~3);
      *reinterpret_cast<float4*>(P + (size_t)row * g.N + col) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

// The same in 256 x 256 tiles (see gemm_nt_big): stages of 32 rows of 512 bytes of
// each operand, read transposed; their 16-byte pieces are permuted so that the
// eight rows a half wave reads together lie 32 bytes apart in the banks.
// 1536 x 1792 over 32768 rows: 0.309 -> 0.206 ms (876 TFLOP/s, six splits).
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_tn_big(GemmTN g) {
  constexpr int SB = kBigT * kBigK * 2;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kBigS * 2 * SB];
  const int w = wave_id(), lane = lane_id();
  const int ntn = g.N / kBigT, ntk = g.Kd / kBigT;
  // one split's tiles are consecutive workgroups: they read the same rows at the same
  // time (each XCD fetches them once, since consecutive workgroups go over all XCDs)
  const int tiles = ntk * ntn;
  const int s = blockIdx.x / tiles, tt = blockIdx.x % tiles;
  const int tk = tt / ntn, tn = tt % ntn;
  const int m0 = s * g.rows, m1 = min(m0 + g.rows, g.M);
  const int nk = (m1 - m0) / kBigK;
  const bool isb = w >= 4;
  const bf16* base = isb ? g.D + (size_t)m0 * g.ldd + tn * kBigT : g.X + (size_t)m0 * g.ldx + tk * kBigT;
  const long long ld = isb ? g.ldd : g.ldx;
  auto swz = [](int row) { return 2 * ((row & 3) | (((row >> 3) & 1) << 2)); };
  const char* src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {   // two rows of 512 bytes each
    const int row = 8 * (w & 3) + 2 * i + (lane >> 5);
    src[i] = reinterpret_cast<const char*>(base + (size_t)row * ld + (((lane & 31) ^ swz(row)) * 8));
  }
  const size_t adv = (size_t)kBigK * ld * 2;
  const uint32_t l0 = lds_addr(lds) + (isb ? SB : 0) + (w & 3) * 4096;
  auto issue = [&](int t) {
    const uint32_t d = l0 + (t % kBigS) * 2 * SB;
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16_raw(src[i] + (size_t)t * adv, d + i * 1024);
  };
  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero4();
  const int wm = 128 * (w >> 2), wn = 64 * (w & 3);
  const int r16 = lane & 15, g4 = lane >> 4;
  typedef __attribute__((address_space(3))) bf16x4* lds_p;
  auto frag = [&](const unsigned char* st, int c0) {   // (k = row, i = column c0 + r16)
    const int row = 8 * g4 + (r16 >> 2);
    const int pc = (c0 >> 3) + ((r16 & 3) >> 1), by = (r16 & 1) * 8;
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_p)(st + row * 512 + ((pc ^ swz(row)) * 16) + by));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_p)(st + (row + 4) * 512 + ((pc ^ swz(row + 4)) * 16) + by));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  for (int t = 0; t < 3 && t < nk; ++t) issue(t);
  for (int t = 0; t < nk; ++t) {
    if (t + 2 < nk) vm_wait<8>();
    else vm_wait<0>();
    bare_barrier();
    if (t + 3 < nk) issue(t + 3);
    const unsigned char* sX = lds + (t % kBigS) * 2 * SB;
    const unsigned char* sD = sX + SB;
    bf16x8 bf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bf[j] = frag(sD, wn + 16 * j);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bf16x8 af = frag(sX, wm + 16 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = Mma<bf16>::mma(af, bf[j], acc[i][j]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  float* P = g.part + (size_t)s * g.Kd * g.N;
  const int c = tile_col();
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      quad_transpose(v);
      const int row = tk * kBigT + wm + 16 * i + tile_row(0) + (c & 3);
      const int col = tn * kBigT + wn + 16 * j + (c & ~3);
      *reinterpret_cast<float4*>(P + (size_t)row * g.N + col) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

// ---------------------------------------------------------------- epilogues
__device__ __forceinline__ float m2p_dt_lo() { return bf16r(1e-2f); }
// jax.nn.softplus(x) = logaddexp(x, 0); every use rounds the result to bf16
__device__ __forceinline__ float m2p_softplus(float x) { return fmaxf(x, 0.f) + __logf(1.f + __expf(-fabsf(x))); }
// nan_to_num(clip(x, -c, c))
__device__ __forceinline__ float m2p_sanit(float x, float c) {
  if (__builtin_isnan(x)) return 0.f;
  return fminf(fmaxf(x, -c), c);
}

// Forward epilogue: the columns of [W_dt | W_B | W_C] give
//   dt = sanitize(clip(softplus(bf16(bf16(x W_dt) + bf16(b_dt))), bf16(1e-2), 1), 1e3)
//   B  = sanitize(bf16(x W_B), 1e3)      C = sanitize(bf16(x W_C), 1e3)
// (model.py:425-433); the pre-activations are also stored when asked for.
struct M2ProjEpi {
  int d, n;
  const float* b_dt;               // [d]
  bf16 *dt, *B, *C;                // [M][d], [M][n], [M][n]
  bf16 *dt_pre, *b_pre, *c_pre;    // the same shapes, or NULL
  // eight columns of one row, the products rounded to bf16 (all outputs 16-byte aligned)
  __device__ __forceinline__ void row8(int row, int col, float (&v)[8]) const {
    float o[8];
    if (col < d) {  // uniform over a wave's 64 columns
      float bv[8];
      load8(b_dt + col, bv);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        v[k] = bf16r(v[k] + bf16r(bv[k]));
        o[k] = m2p_sanit(fminf(fmaxf(bf16r(m2p_softplus(v[k])), m2p_dt_lo()), 1.f), 1e3f);
      }
      store8(dt + (size_t)row * d + col, o);
      if (dt_pre) store8(dt_pre + (size_t)row * d + col, v);
    } else {
      const bool isb = col < d + n;
      const int cc = isb ? col - d : col - d - n;
#pragma unroll
      for (int k = 0; k < 8; ++k) o[k] = m2p_sanit(v[k], 1e3f);
      store8((isb ? B : C) + (size_t)row * n + cc, o);
      bf16* pre = isb ? b_pre : c_pre;
      if (pre) store8(pre + (size_t)row * n + cc, v);
    }
  }
  template <int NJ>
  __device__ __forceinline__ void operator()(int m0, int n0, f32x4 (&acc)[4][NJ]) const {
    const int c = tile_col();
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = n0 + 16 * j + (c & ~3);  // this lane's four columns after the transpose
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + 16 * i + tile_row(0) + (c & 3);
        float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        quad_transpose(v);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = bf16r(v[k]);
        if (col < d) {  // uniform over the 16-column tile
          const float4 bb = *reinterpret_cast<const float4*>(b_dt + col);
          const float bv[4] = {bb.x, bb.y, bb.z, bb.w};
          float o[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            v[k] = bf16r(v[k] + bf16r(bv[k]));
            o[k] = m2p_sanit(fminf(fmaxf(bf16r(m2p_softplus(v[k])), m2p_dt_lo()), 1.f), 1e3f);
          }
          st4bf(dt + (size_t)row * d + col, o);
          if (dt_pre) st4bf(dt_pre + (size_t)row * d + col, v);
        } else {
          const bool isb = col < d + n;
          const int cc = isb ? col - d : col - d - n;
          bf16* out = isb ? B : C;
          bf16* pre = isb ? b_pre : c_pre;
          float o[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) o[k] = m2p_sanit(v[k], 1e3f);
          st4bf(out + (size_t)row * n + cc, o);
          if (pre) st4bf(pre + (size_t)row * n + cc, v);
        }
      }
    }
  }
};

// Backward epilogue of dX = dPre [W_dt | W_B | W_C]^T: x_bc's gradient is the
// projections' part (bf16) plus the convolution path's part, written to the
// strided view of the in_proj gradient.
struct M2DxEpi {
  const bf16* dxc;  // [M][d] the convolution path's part
  int d;
  bf16* out;        // [M] rows of stride ldo
  long long ldo;
  __device__ __forceinline__ void row8(int row, int col, float (&v)[8]) const {
    float cv[8];
    load8(dxc + (size_t)row * d + col, cv);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] += cv[k];
    store8(out + (size_t)row * ldo + col, v);
  }
  template <int NJ>
  __device__ __forceinline__ void operator()(int m0, int n0, f32x4 (&acc)[4][NJ]) const {
    const int c = tile_col();
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = n0 + 16 * j + (c & ~3);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + 16 * i + tile_row(0) + (c & 3);
        float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        quad_transpose(v);
        float cv[4];
        ld4bf(dxc + (size_t)row * d + col, cv);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = bf16r(v[k]) + cv[k];
        st4bf(out + (size_t)row * ldo + col, v);
      }
    }
  }
};

// ---------------------------------------------------------------- packing
// W(k, r) for the concatenated [W_dt | W_B | W_C] ([d][d + 2n], fp32 params)
__device__ __forceinline__ float m2p_w(int d, int n, const float* wdt, const float* wb, const float* wc, int k,
                                       int r) {
  return r < d ? wdt[(size_t)k * d + r] : (r < d + n ? wb[(size_t)k * n + r - d] : wc[(size_t)k * n + r - d - n]);
}
// out[k][r] = bf16(W(k, r))  (the layout of the backward's dX GEMM)
__global__ __launch_bounds__(256) void m2p_pack(int d, int n, const float* __restrict__ wdt,
                                                const float* __restrict__ wb, const float* __restrict__ wc,
                                                bf16* __restrict__ out) {
  const int nt = d + 2 * n;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (size_t)d * nt) return;
  out[e] = (bf16)m2p_w(d, n, wdt, wb, wc, (int)(e / nt), (int)(e % nt));
}
// out[r][k] = bf16(W(k, r))  (the forward GEMM's Bt), 64 x 64 tiles through LDS
__global__ __launch_bounds__(256) void m2p_pack_t(int d, int n, const float* __restrict__ wdt,
                                                  const float* __restrict__ wb, const float* __restrict__ wc,
                                                  bf16* __restrict__ out) {
  __shared__ float t[64][65];
  const int nt = d + 2 * n, ntr = nt / 64;
  const int tr = blockIdx.x % ntr, tk = blockIdx.x / ntr;
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int kk = e >> 6, rr = e & 63;
    t[kk][rr] = m2p_w(d, n, wdt, wb, wc, tk * 64 + kk, tr * 64 + rr);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int rr = e >> 6, kk = e & 63;
    out[(size_t)(tr * 64 + rr) * d + tk * 64 + kk] = (bf16)t[kk][rr];
  }
}

// ---------------------------------------------------------------- backward pieces
// cotangent factors of clip(v, -c, c) and of clip(x, lo, hi) (ties split evenly)
__device__ __forceinline__ float m2p_clip_g(float v, float c) {
  const float a = fabsf(v);
  return a < c ? 1.f : (a == c ? 0.5f : 0.f);
}
__device__ __forceinline__ float m2p_range_g(float x, float lo, float hi) {
  const float a = x > lo ? 1.f : (x == lo ? 0.5f : 0.f);
  const float b = x < hi ? 1.f : (x == hi ? 0.5f : 0.f);
  return a * b;
}

// The element-wise VJP of M2ProjEpi into dPre [M][d + 2n] (columns: dt, B, C
// pre-activations), one thread per 4 columns of 32 rows; column sums of the
// dt part (b_dt's gradient) per 32 rows into dbpart [M / 32][d].  Block 0
// also writes dA_log from dA (A = -exp(clip(A_log, +-20)), model.py:420-422).
// Its four transcendentals an element and its 6 bytes take about as long as each
// other: softplus and its derivative share one exponential, the loads of
// eight rows are in flight together, and 4 columns a thread give seven waves per
// SIMD (8 columns, two exponentials: 0.142 ms at 32768 x 1792, now 0.105).
__global__ __launch_bounds__(256) void m2p_vjp(int M, int d, int n, int H, const bf16* __restrict__ dt_pre,
                                               const bf16* __restrict__ b_pre, const bf16* __restrict__ c_pre,
                                               const float* __restrict__ a_log, const bf16* __restrict__ ddt,
                                               const bf16* __restrict__ dB, const bf16* __restrict__ dC,
                                               const float* __restrict__ dA, bf16* __restrict__ dpre,
                                               float* __restrict__ dbpart, float* __restrict__ da_log) {
  const int nt = d + 2 * n, ncg = nt / 4;
  const size_t gi = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (gi < (size_t)(M / 32) * ncg) {
    const int cg = (int)(gi % ncg), rt = (int)(gi / ncg);
    const int col = cg * 4;
    constexpr int U = 8;
    const bool isdt = col < d, isb = col < d + n;
    const int cc = isdt ? col : (isb ? col - d : col - d - n), ld = isdt ? d : n;
    const bf16* pre = (isdt ? dt_pre : (isb ? b_pre : c_pre)) + cc;
    const bf16* gg = (isdt ? ddt : (isb ? dB : dC)) + cc;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int r0 = 0; r0 < 32; r0 += U) {
      bf16x4 rv[U], rg[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const size_t m = (size_t)rt * 32 + r0 + u;
        rv[u] = *reinterpret_cast<const bf16x4*>(pre + m * ld);
        rg[u] = *reinterpret_cast<const bf16x4*>(gg + m * ld);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float o[4];
        if (isdt) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float v = (float)rv[u][j], e = __expf(-fabsf(v));
            const float sp = bf16r(fmaxf(v, 0.f) + __logf(1.f + e));   // m2p_softplus
            // the clip to [lo, 1] keeps its result inside the +-1e3 of the sanitise after it
            const float dsp = bf16r((float)rg[u][j] * m2p_range_g(sp, m2p_dt_lo(), 1.f));
            const float ri = __builtin_amdgcn_rcpf(1.f + e);
            o[j] = bf16r(dsp * (v >= 0.f ? ri : e * ri));  // softplus' = logistic
            acc[j] += o[j];
          }
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = bf16r((float)rg[u][j] * m2p_clip_g((float)rv[u][j], 1e3f));
        }
        st4bf(dpre + ((size_t)rt * 32 + r0 + u) * nt + col, o);
      }
    }
    if (isdt) *reinterpret_cast<float4*>(dbpart + (size_t)rt * d + col) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  }
  if (blockIdx.x == 0)
    for (int h = threadIdx.x; h < H; h += 256) {
      const float al = a_log[h];
      da_log[h] = dA[h] * (-__expf(fminf(fmaxf(al, -20.f), 20.f))) * m2p_clip_g(al, 20.f);
    }
}

// Weight and bias gradients: dW = fp32(bf16(sum of the split partials)) split
// into [W_dt | W_B | W_C]; b_dt's gradient = fp32(bf16(dbsum)) (the bf16
// dot / bias VJPs of the reference, then the cast of the fp32 parameters).
__global__ __launch_bounds__(256) void m2p_dw_finish(int d, int n, int splits, const float* __restrict__ part,
                                                     const float* __restrict__ dbsum, float* __restrict__ dw_dt,
                                                     float* __restrict__ dw_b, float* __restrict__ dw_c,
                                                     float* __restrict__ db_dt) {
  const int nt = d + 2 * n;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t tot = (size_t)d * nt;
  if (e < (size_t)d) db_dt[e] = bf16r(dbsum[e]);
  if (e >= tot) return;
  float s = 0.f;
  for (int sp = 0; sp < splits; ++sp) s += part[(size_t)sp * tot + e];
  const float v = bf16r(s);
  const int k = (int)(e / nt), r = (int)(e % nt);
  if (r < d) dw_dt[(size_t)k * d + r] = v;
  else if (r < d + n) dw_b[(size_t)k * n + r - d] = v;
  else dw_c[(size_t)k * n + r - d - n] = v;
}

}  // namespace ah
