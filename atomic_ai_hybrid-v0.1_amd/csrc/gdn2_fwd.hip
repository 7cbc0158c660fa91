// GDN2 WY chunked forward for gfx950.
//
// gdn2_fwd_intra  (one workgroup per (batch, head, chunk); fully parallel)
//   Follows _build_chunk_wy (atomic_ops/gdn2_wy_reference.py:59-102):
//   gc = cumsum(g); Aqk / Akk intra-chunk scores; A = (I + Akk)^-1;
//   w_pseudo = A (b k e^gc); u = A (w v); kg, qg; gc_last.
//   The pairwise decay exp(gc_i - gc_j) is factorised as
//   (q e^{gc_i}) . (k e^{-gc_j}) so both score matrices are bf16 MFMA GEMMs.
//   The factorisation is exact while every g <= 0 in the chunk (then
//   gc_i - gc_j <= 0 on causal pairs, so the reference's +20 clip never
//   fires) and -gc_last <= kFactorLimit (so k e^{-gc} stays finite).  Pairs
//   whose decay falls below the reference's -20 floor then carry their true
//   (smaller) weight instead of e^-20, a difference below 2e-9 |q||k|.  Any
//   chunk outside those bounds takes an exact pairwise path that applies
//   exp(clip(gc_i - gc_j, -20, 20)) as the reference does.
//
// gdn2_fwd_state  (one workgroup per (batch, head, V tile); sequential over
//   chunks).  Follows the scan step of gdn2_chunked_wy_reference
//   (gdn2_wy_reference.py:125-144) / gdn2_inter_chunk_combine
//   (kernel_d_pipeline.py:94-124): v_new = u - w_pseudo h;
//   o = scale qg h + Aqk v_new; h = sanitize(h e^{gc_last} + kg^T v_new).
//   The fp32 state lives in MFMA accumulators for the whole sequence.
#include "gdn2_seq.hpp"

namespace ah {

constexpr float kFactorLimit = 64.f;

// ------------------------------------------------------------------ cumsum
// Thread map for [C][K] fp32 element-wise passes: column group cg (8
// columns), segment seg (RS consecutive rows).  Whatever the number of
// threads, a wave covers a quarter of the rows: with 256 threads all columns of
// them, with 512 half of the columns in segments of half the length.
template <int C, int K, int NTH = 256>
struct ColMap {
  static constexpr int NCG = K / 8, NSEG = NTH / NCG, RS = C / NSEG;
  static constexpr int U = NTH / 256, WCG = NCG / U;  // column groups of a wave
  static_assert(RS >= 1, "chunk too small for the thread mapping");
  static __device__ __forceinline__ int cg() {
    return U == 1 ? lane_id() % NCG : (wave_id() & 1) * WCG + lane_id() % WCG;
  }
  static __device__ __forceinline__ int seg() {
    return (U == 1 ? wave_id() : wave_id() >> 1) * (64 / WCG) + lane_id() / WCG;
  }
};

// Exclusive scan over the row segments of a ColMap pass: t holds this
// thread's segment total for its 8 columns; out gets the sum over the lower
// segments (REV = false) or the higher ones (REV = true).  Within a wave by
// lane shuffles, across the four waves of a column through sW (4 * K floats).
// With U > 1, U consecutive segments count as one (t is its total in each).
template <int NCG, bool REV, int U = 1>
__device__ __forceinline__ void seg_scan8(const float (&t)[8], float (&out)[8], float* sW) {
  constexpr int UL = NCG;           // lanes of a segment, or of the U that count as one
  constexpr int SPW = 64 / UL;      // segments per wave
  static_assert(SPW * UL == 64, "column groups must tile a wave");
  const int lane = lane_id(), w = U == 1 ? wave_id() : wave_id() >> 1, sl = lane / UL;
  const int cg = U == 1 ? lane % NCG : (wave_id() & 1) * (NCG / U) + lane % (NCG / U);
  float x[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = t[j];
#pragma unroll
  for (int d = 1; d < SPW; d <<= 1) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float y = REV ? __shfl_down(x[j], d * UL) : __shfl_up(x[j], d * UL);
      if (REV ? (sl + d < SPW) : (sl >= d)) x[j] += y;
    }
  }
  if (sl == (REV ? 0 : SPW - 1)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) sW[w * NCG * 8 + cg * 8 + j] = x[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 8; ++j) out[j] = x[j] - t[j];
#pragma unroll
  for (int w2 = 0; w2 < 4; ++w2)
    if (REV ? w2 > w : w2 < w) {
#pragma unroll
      for (int j = 0; j < 8; ++j) out[j] += sW[w2 * NCG * 8 + cg * 8 + j];
    }
}

// x of the lane that the DPP control CTRL selects (within a 16-lane row)
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

// gc = cumsum(g) over one chunk (gdn2_wy_reference.py:63) for this thread's
// RS rows x 8 columns.  Writes gc_last to sGl[K] (sTot: 4 K floats of
// scratch).  Returns, uniformly over the workgroup, whether the factorised
// pairwise decay is unsafe for this chunk: some g > 0, or gc_last below
// -kFactorLimit in some column.  The order of the additions does not depend on
// NTH: with 512 threads two lanes continue one serial sum, so that the
// exponentials, and every bf16 operand rounded from them, are the same bits.
template <int C, int K, int NTH = 256>
__device__ __forceinline__ bool chunk_cumsum(const float* __restrict__ g, size_t rs,
                                             float (&gcr)[ColMap<C, K, NTH>::RS][8], float* sTot,
                                             float* sGl) {
  typedef ColMap<C, K, NTH> M;
  static_assert(M::U == 1 || (M::U == 2 && 16 % (2 * M::WCG) == 0), "one lane a serial sum, or two of a 16-lane row");
  const int cg = M::cg(), seg = M::seg();
  bool positive = false;
#pragma unroll
  for (int rr = 0; rr < M::RS; ++rr) {
    load8(g + (size_t)(seg * M::RS + rr) * rs + cg * 8, gcr[rr]);
#pragma unroll
    for (int j = 0; j < 8; ++j) positive |= gcr[rr][j] > 0.f;
  }
  if constexpr (M::U == 2) {  // an odd segment goes on from the sum of the even one before it
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float s = gcr[0][j];
#pragma unroll
      for (int rr = 1; rr < M::RS; ++rr) s += gcr[rr][j];
      s = dpp_mov<0x110 + M::WCG>(s);  // row_shr
      if (seg & 1) gcr[0][j] += s;
    }
  }
#pragma unroll
  for (int rr = 1; rr < M::RS; ++rr)
#pragma unroll
    for (int j = 0; j < 8; ++j) gcr[rr][j] += gcr[rr - 1][j];
  float tot[8], off[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    tot[j] = gcr[M::RS - 1][j];
    if constexpr (M::U == 2) {
      const float s = dpp_mov<0x100 + M::WCG>(tot[j]);  // row_shl
      if (!(seg & 1)) tot[j] = s;
    }
  }
  seg_scan8<M::NCG, false, M::U>(tot, off, sTot);
#pragma unroll
  for (int rr = 0; rr < M::RS; ++rr)
#pragma unroll
    for (int j = 0; j < 8; ++j) gcr[rr][j] += off[j];
  bool too_deep = false;
  if (seg == M::NSEG - 1) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      sGl[cg * 8 + j] = gcr[M::RS - 1][j];
      too_deep |= gcr[M::RS - 1][j] < -kFactorLimit;
    }
  }
  return __syncthreads_or(positive || too_deep);
}

// ------------------------------------------------------------------ layout
template <typename T, int C, int K, int V>
struct IntraLds {
  static constexpr int NTH = 512, NW = NTH / 64;
  static constexpr int PAD = Pad<T>::v;
  static constexpr int LK = K + PAD, LV = V + PAD;
  static constexpr int LA = C + 4;                 // fp32 score / inverse rows
  static constexpr int LAB = C + PAD;              // operand-type inverse rows
  static constexpr int NCG = K / 8, NSEG = NTH / NCG, RS = C / NSEG;
  static constexpr int NCGV = V / 8, NSEGV = NTH / NCGV, RSV = C / NSEGV;
  static constexpr int OPK = C * LK * (int)sizeof(T);
  static constexpr int OPV = C * LV * (int)sizeof(T);
  static constexpr int AF = C * LA * 4;
  static constexpr int off_q = 0, off_k = OPK, off_b = 2 * OPK, off_w = 3 * OPK;
  static constexpr int end_ops = 3 * OPK + OPV;
  static constexpr bool alias_a = 2 * OPK >= 2 * AF;
  static constexpr int off_af = alias_a ? 0 : end_ops;      // Akk (then operand-type A)
  static constexpr int off_x = off_af + AF;                 // fp32 inverse
  static constexpr int end_a = off_x + AF;
  static constexpr int off_tot = (end_ops > end_a ? end_ops : end_a);
  // cumsum totals of the row quarters; then the solve's products, one a wave
  static constexpr int S16 = 16 * 17 * 4, SOLVE = (C / 16 - 1) * S16;
  static constexpr int TOT = 4 * K * 4 > SOLVE ? 4 * K * 4 : SOLVE;
  static constexpr int off_gl = off_tot + TOT;
  static constexpr int off_flag = off_gl + K * 4;
  static constexpr int total = off_flag + 16;
  // phase 4 (operand-type path): per-wave [16][64] staging of half a row block of
  // w_pseudo / u, placed over the operands that are dead by then (q, k, the
  // fp32 Akk / inverse), after the operand-type inverse
  static constexpr int LS = 64 + PAD;
  static constexpr int off_stage =
      alias_a ? ((off_af + C * (C + PAD) * (int)sizeof(T) + 15) / 16) * 16 : 0;
  static constexpr int stage_end = off_stage + NW * 16 * LS * (int)sizeof(T);
  static constexpr bool stage_fits = stage_end <= off_b && (alias_a || stage_end <= off_af);
  static_assert(RS >= 1 && RSV >= 1, "chunk too small for the thread mapping");
  static_assert(2 * OPK >= C * K * 4, "gc scratch of the exact path must fit in sQ+sK");
};

// Exact pairwise scores for one chunk (reference form, used when the
// factorised form could overflow or a positive gate breaks monotonicity).
template <typename T, int C, int K, int NTH>
__device__ void intra_scores_exact(const float* sgc, const T* q, const T* k, const T* b, size_t sq,
                                   size_t sk, size_t sb, float scale, float* out_qk, float* out_kk) {
  // thread t computes entries e = t, t + NTH, ... of the C x C matrices
  for (int e = threadIdx.x, s = 0; e < C * C; e += NTH, ++s) {
    const int i = e / C, j = e % C;
    float aqk = 0.f, akk = 0.f;
    if (j <= i) {
      const T* qi = q + i * sq;
      const T* ki = k + i * sk;
      const T* bi = b + i * sb;
      const T* kj = k + j * sk;
      for (int d = 0; d < K; ++d) {
        const float dd = sgc[i * K + d] - sgc[j * K + d];
        const float ed = __expf(fminf(fmaxf(dd, -kClipDecay), kClipDecay));
        const float kjd = to_f(kj[d]);
        aqk += to_f(qi[d]) * ed * kjd;
        akk += to_f(bi[d]) * to_f(ki[d]) * ed * kjd;
      }
      aqk *= scale;
      if (j == i) akk = 0.f;
    }
    out_qk[s] = n2n(aqk);
    out_kk[s] = n2n(akk);
  }
}

// What one gdn2_fwd_intra launch builds: the whole per-chunk build (kernels
// A + B + C in one pass), or one of the reference's three kernels over
// caller-owned per-chunk arrays:
//   kIntraScores    A: Aqk and the strict Akk (kernel_a_scores.py:21-66)
//   kIntraSolve     B: A = (I + Akk)^-1 from a given Akk (kernel_b_solve.py)
//   kIntraRecompute C: w_pseudo = A kb, u = A (w v), kg, qg, gc_last from a
//                   given A, all clipped to +-1e4 (kernel_c_recompute.py:46-88)
enum { kIntraAll = 0, kIntraScores = 1, kIntraSolve = 2, kIntraRecompute = 3 };

//
// One chunk is a chain of short phases (loads and cumsum, element-wise operands,
// scores, four 16-row substitutions, the blocks below them column by column, the
// two products), so the kernel is latency, hidden by eight waves per workgroup and
// two workgroups per CU: with four waves one chunk took 17.8 us at B1 T64 H8 K =
// 128 and the kernel 0.367 ms at B4 T8192 H16, so 11.9 us and 0.316 ms, the latter
// 5.0 TB/s of what the kernel has to move and as fast as a large copy.  The
// inverse in two levels of 2 x 2 blocks, and a cumsum whose waves take whole
// rows (0.312 ms), were as fast or faster but add in another order, which
// moved the bf16 gradients by 8e-4 of themselves.
template <typename T, int C, int K, int V, int ST = kIntraAll>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 2 ? 4 : 2, 4))) void gdn2_fwd_intra(Gdn2Dims dm, const T* __restrict__ q,
                                                     const T* __restrict__ k, const T* __restrict__ v,
                                                     const T* __restrict__ w, const T* __restrict__ b,
                                                     const float* __restrict__ g, Gdn2Chunks<T> ck) {
  typedef IntraLds<T, C, K, V> L;
  __shared__ __attribute__((aligned(16))) unsigned char lds[L::total];
  T* sQ = reinterpret_cast<T*>(lds + L::off_q);
  T* sK = reinterpret_cast<T*>(lds + L::off_k);
  T* sB = reinterpret_cast<T*>(lds + L::off_b);
  T* sW = reinterpret_cast<T*>(lds + L::off_w);
  float* sAf = reinterpret_cast<float*>(lds + L::off_af);
  float* sX = reinterpret_cast<float*>(lds + L::off_x);
  float* sTot = reinterpret_cast<float*>(lds + L::off_tot);
  float* sGl = reinterpret_cast<float*>(lds + L::off_gl);
  float* sGcExact = reinterpret_cast<float*>(lds + L::off_q);  // exact path only

  constexpr int NTH = L::NTH, NW = L::NW;
  const int tid = threadIdx.x;
  const int bhn = blockIdx.x;
  const int n = bhn % dm.NT;
  const int bh = bhn / dm.NT;
  const int h = bh % dm.H;
  const int bb = bh / dm.H;
  const size_t t0 = (size_t)bb * dm.T + (size_t)n * C;
  const T* qc = q + t0 * dm.rq + (size_t)h * K;
  const T* kc = k + t0 * dm.rk + (size_t)h * K;
  const T* bc = b + t0 * dm.rb + (size_t)h * K;
  const float* gc_in = g + t0 * dm.rg + (size_t)h * K;
  const T* vc = v + t0 * dm.rv + (size_t)h * V;
  const T* wc = w + t0 * dm.rw + (size_t)h * V;

  // q, k, b, v, w are requested before the cumsum of g, so their latency overlaps it
  typedef ColMap<C, K, L::NTH> M;
  const int cg = M::cg(), seg = M::seg();
  const int cgv = tid % L::NCGV, segv = tid / L::NCGV;
  constexpr bool kRows = ST != kIntraSolve;                          // reads q, k, b, g
  constexpr bool kVals = ST == kIntraAll || ST == kIntraRecompute;   // reads v, w; writes qg, kg
  constexpr bool kScores = ST == kIntraAll || ST == kIntraScores;
  // the stage-level kernel C clips every output to +-1e4 (kernel_c_recompute.py:74-82)
  auto fin = [](float x) { return ST == kIntraRecompute ? sanitize(x) : n2n(x); };
  Raw8<T> rq[L::RS], rk[L::RS], rb[L::RS], rv[L::RSV], rw[L::RSV];
  if constexpr (kRows) {
#pragma unroll
    for (int rr = 0; rr < L::RS; ++rr) {
      const size_t r = (size_t)(seg * L::RS + rr);
      rq[rr].load(qc + r * dm.rq + cg * 8);
      rk[rr].load(kc + r * dm.rk + cg * 8);
      rb[rr].load(bc + r * dm.rb + cg * 8);
    }
  }
  if constexpr (kVals) {
#pragma unroll
    for (int rr = 0; rr < L::RSV; ++rr) {
      const size_t r = (size_t)(segv * L::RSV + rr);
      rv[rr].load(vc + r * dm.rv + cgv * 8);
      rw[rr].load(wc + r * dm.rw + cgv * 8);
    }
  }

  bool exact = false;
  if constexpr (kRows) {
  // ---- phase 0: gc = cumsum(g) over the chunk (gdn2_wy_reference.py:63)
  float gcr[L::RS][8];
  exact = chunk_cumsum<C, K, NTH>(gc_in, (size_t)dm.rg, gcr, sTot, sGl);
  if (kVals && tid < K) ck.gcl[(size_t)bhn * K + tid] = fin(sGl[tid]);

  // ---- phase 1: elementwise operands (gdn2_wy_reference.py:92-100)
  T* g_qg = ck.qg + (size_t)bhn * C * K;
  T* g_kg = ck.kg + (size_t)bhn * C * K;
#pragma unroll
  for (int rr = 0; rr < L::RS; ++rr) {
    const int r = seg * L::RS + rr;
    float qv[8], kv[8], bv[8], o_qg[8], o_kt[8], o_kb[8], o_kg[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) { qv[j] = rq[rr][j]; kv[j] = rk[rr][j]; bv[j] = rb[rr][j]; }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float gcv = gcr[rr][j];
      const float e = __expf(gcv);
      o_qg[j] = qv[j] * e;
      o_kt[j] = kv[j] * __expf(-gcv);
      o_kb[j] = (bv[j] * kv[j]) * e;
      o_kg[j] = kv[j] * __expf(sGl[cg * 8 + j] - gcv);
    }
    store8(sB + r * L::LK + cg * 8, o_kb);
    if constexpr (kScores) {
      if (!exact) {
        store8(sQ + r * L::LK + cg * 8, o_qg);
        store8(sK + r * L::LK + cg * 8, o_kt);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) sGcExact[r * K + cg * 8 + j] = gcr[rr][j];
      }
    }
    if constexpr (kVals) {
      if constexpr (ST == kIntraRecompute) {
#pragma unroll
        for (int j = 0; j < 8; ++j) { o_qg[j] = fin(o_qg[j]); o_kg[j] = fin(o_kg[j]); }
      }
      store8(g_qg + r * K + cg * 8, o_qg);
      store8(g_kg + r * K + cg * 8, o_kg);
    }
  }
  if constexpr (kVals) {
#pragma unroll
    for (int rr = 0; rr < L::RSV; ++rr) {
      const int r = segv * L::RSV + rr;
      float vv[8], wv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) { vv[j] = rv[rr][j]; wv[j] = rw[rr][j]; }
      // w * v is formed in the input dtype before the upcast (gdn2_wy_reference.py:94)
#pragma unroll
      for (int j = 0; j < 8; ++j) wv[j] = to_f(from_f<T>(wv[j] * vv[j]));
      store8(sW + r * L::LV + cgv * 8, wv);
    }
  }
  __syncthreads();
  }  // kRows

  // ---- phase 2: Aqk (causal, scaled) and Akk (strict) (gdn2_wy_reference.py:79-87)
  constexpr int NB = C / 16;
  constexpr int NTRI = NB * (NB + 1) / 2;
  T* g_aqk = ck.aqk + (size_t)bhn * C * C;
  T* g_akk = ck.akk + (size_t)bhn * C * C;  // kernel A alone: Akk leaves in the operand type
  const int wv_id = wave_id();
  if constexpr (kScores) {
  if (!exact) {
    // job: 0 .. NTRI - 1 Aqk's lower tiles, then Akk's; a wave's jobs share each
    // k step, so their MFMA chains overlap (past the last job: that one again)
    constexpr int JPW = (2 * NTRI + NW - 1) / NW;
    f32x4 res[JPW];
    const T* jp[JPW];
    int jm[JPW], jn[JPW];
#pragma unroll
    for (int cnt = 0; cnt < JPW; ++cnt) {
      const int job = min(wv_id + NW * cnt, 2 * NTRI - 1);
      jp[cnt] = job / NTRI ? sB : sQ;
      int t = job % NTRI, mi = 0;
      while (t > mi) { t -= mi + 1; ++mi; }
      jm[cnt] = mi;
      jn[cnt] = t;
      res[cnt] = zero4();
    }
#pragma unroll 4
    for (int k0 = 0; k0 < K; k0 += Mma<T>::KS)
#pragma unroll
      for (int cnt = 0; cnt < JPW; ++cnt)
        res[cnt] = Mma<T>::mma(Mma<T>::ld_c(jp[cnt], L::LK, 16 * jm[cnt], k0),
                               Mma<T>::ld_c(sK, L::LK, 16 * jn[cnt], k0), res[cnt]);
#pragma unroll
    for (int cnt = 0; cnt < JPW; ++cnt) {
      const bool kk = min(wv_id + NW * cnt, 2 * NTRI - 1) >= NTRI;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * jm[cnt] + tile_row(i), c = 16 * jn[cnt] + tile_col();
        const float x = kk ? res[cnt][i] : dm.scale * res[cnt][i];
        const bool keep = kk ? (r > c) : (r >= c);
        res[cnt][i] = keep ? n2n(x) : 0.f;
      }
    }
    __syncthreads();  // sQ / sK are dead from here on; sAf may alias them
#pragma unroll
    for (int cnt = 0; cnt < JPW; ++cnt) {
      const int job = wv_id + NW * cnt;
      if (job >= 2 * NTRI) break;
      if (job < NTRI) store_tile_n(g_aqk, C, 16 * jm[cnt], 16 * jn[cnt], res[cnt]);
      else if constexpr (ST == kIntraScores) store_tile_n(g_akk, C, 16 * jm[cnt], 16 * jn[cnt], res[cnt]);
      else store_tile_n(sAf, L::LA, 16 * jm[cnt], 16 * jn[cnt], res[cnt]);
    }
  } else {
    constexpr int PER = C * C / NTH;
    float eqk[PER], ekk[PER];
    intra_scores_exact<T, C, K, NTH>(sGcExact, qc, kc, bc, dm.rq, dm.rk, dm.rb, dm.scale, eqk, ekk);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < PER; ++s) {
      const int e = tid + NTH * s, i = e / C, j = e % C;
      g_aqk[i * C + j] = from_f<T>(eqk[s]);
      if constexpr (ST == kIntraScores) g_akk[i * C + j] = from_f<T>(ekk[s]);
      else sAf[i * L::LA + j] = ekk[s];
    }
  }
  // upper tiles of Aqk / Akk are zero (in LDS only the lower blocks of Akk are
  // read), and so is the inverse until its blocks are written; 16 bytes an item
  // where the caller's array allows it
  const u32x4 z4 = {0u, 0u, 0u, 0u};
  auto zero_upper = [&](T* p) {
    constexpr int VC = 16 / (int)sizeof(T);
    const bool wide = (reinterpret_cast<uintptr_t>(p) & 15) == 0;
    for (int e = tid; e < C * C / VC; e += NTH) {
      const int i = e / (C / VC), j = (e % (C / VC)) * VC;
      if ((j >> 4) <= (i >> 4)) continue;
      if (wide) {
        *reinterpret_cast<u32x4*>(p + i * C + j) = z4;
      } else {
#pragma unroll
        for (int t = 0; t < VC; ++t) p[i * C + j + t] = from_f<T>(0.f);
      }
    }
  };
  if (!exact) zero_upper(g_aqk);
  if constexpr (ST == kIntraScores) zero_upper(g_akk);
  if constexpr (ST == kIntraAll)
    for (int e = tid; e < C * C / 4; e += NTH)
      *reinterpret_cast<u32x4*>(sX + e / (C / 4) * L::LA + (e % (C / 4)) * 4) = z4;
  if constexpr (ST == kIntraScores) return;
  __syncthreads();
  }  // kScores
  if constexpr (ST == kIntraSolve) {
    // Akk from the caller (only its strictly lower blocks are read below)
    for (int e = tid; e < C * C; e += NTH) {
      const int i = e / C, j = e % C;
      sAf[i * L::LA + j] = to_f(g_akk[i * C + j]);
      sX[i * L::LA + j] = 0.f;
    }
    __syncthreads();
  }

  // ---- phase 3: A = (I + Akk)^-1 (gdn2_wy_reference.py:16-30,89-90)
  T* g_ainv = ck.ainv + (size_t)bhn * C * C;
  const T* opA;
  int ldA;
  if constexpr (ST != kIntraRecompute) {
  static_assert(NB <= NW, "a 16-row block per wave");
  // Diagonal 16x16 blocks by forward substitution (wave w, lane = column).
  {
    const int lane = lane_id();
    if (wv_id < NB && lane < 16) {
      const int o = 16 * wv_id;
      f32x4 row[16][4];  // the block's rows, every lane the same
#pragma unroll
      for (int i = 1; i < 16; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (4 * q < i) row[i][q] = *reinterpret_cast<const f32x4*>(sAf + (o + i) * L::LA + o + 4 * q);
      float x[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = (i == lane) ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < 15; ++j)  // x_j is final: into every later row
#pragma unroll
        for (int i = j + 1; i < 16; ++i) x[i] -= row[i][j / 4][j % 4] * x[j];
#pragma unroll
      for (int i = 0; i < 16; ++i) sX[(o + i) * L::LA + o + lane] = x[i];
    }
  }
  __syncthreads();
  // Off-diagonal blocks, one column block per wave (no wave reads another's column):
  //   A_mn = -A_mm (sum_{k=n}^{m-1} T_mk A_kn)
  if (wv_id < NB - 1) {
    const int nb = wv_id;
    float* scr = sTot + wv_id * (L::S16 / 4);  // private to this wave
    for (int mb = nb + 1; mb < NB; ++mb) {
      const f32x4 p = tile_mma<float, false, true>(zero4(), sAf + 16 * nb, L::LA, sX + 16 * nb * L::LA, L::LA, 16 * mb,
                                                   16 * nb, 16 * (mb - nb));
      store_tile_n(scr, 17, 0, 0, p);
      wave_lds_sync();
      f32x4 a = tile_mma<float, false, true>(zero4(), sX + 16 * mb * L::LA + 16 * mb, L::LA, scr, 17, 0, 0, 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = -a[i];
      store_tile_n(sX, L::LA, 16 * mb, 16 * nb, a);
      wave_lds_sync();  // the next row block reads this one
    }
  }
  __syncthreads();
  // n2n, operand-type copy, global A
  if constexpr (sizeof(T) == 2) {
    T* sAb = reinterpret_cast<T*>(lds + L::off_af);  // Akk is dead
    for (int e = tid; e < C * C / 8; e += NTH) {  // 8 consecutive columns per item
      const int i = e / (C / 8), j = (e % (C / 8)) * 8;
      float x[8];
      load8(sX + i * L::LA + j, x);
#pragma unroll
      for (int t = 0; t < 8; ++t) x[t] = n2n(x[t]);
      store8(sAb + i * (C + Pad<T>::v) + j, x);
      store8(g_ainv + i * C + j, x);
    }
    opA = sAb;
    ldA = C + Pad<T>::v;
  } else {
    for (int e = tid; e < C * C; e += NTH) {
      const int i = e / C, j = e % C;
      const float x = n2n(sX[i * L::LA + j]);
      sX[i * L::LA + j] = x;
      g_ainv[i * C + j] = from_f<T>(x);
    }
    opA = reinterpret_cast<const T*>(sX);
    ldA = L::LA;
  }
  if constexpr (ST == kIntraSolve) return;
  } else {
    // A from the caller, into the operand-type rows phase 4 reads
    if constexpr (sizeof(T) == 2) {
      T* sAb = reinterpret_cast<T*>(lds + L::off_af);
      for (int e = tid; e < C * C / 8; e += NTH) {
        const int i = e / (C / 8), j = (e % (C / 8)) * 8;
        *reinterpret_cast<uint4*>(sAb + i * (C + Pad<T>::v) + j) =
            *reinterpret_cast<const uint4*>(g_ainv + i * C + j);
      }
      opA = sAb;
      ldA = C + Pad<T>::v;
    } else {
      for (int e = tid; e < C * C; e += NTH) {
        const int i = e / C, j = e % C;
        sX[i * L::LA + j] = g_ainv[i * C + j];
      }
      opA = reinterpret_cast<const T*>(sX);
      ldA = L::LA;
    }
  }
  __syncthreads();

  // ---- phase 4: w_pseudo = A kb, u = A wv (gdn2_wy_reference.py:92-96)
  T* g_wt = ck.wt + (size_t)bhn * C * K;
  T* g_u = ck.u + (size_t)bhn * C * V;
  if constexpr (sizeof(T) == 2 && L::stage_fits) {
    // waves 0-3 a row block of w_pseudo each, 4-7 of u: 64 columns at a time, whose
    // tiles share the A reads, go through the wave's LDS staging rows and
    // leave as 16-byte row pieces
    static_assert(NW == 2 * NB && K == V, "a row block of each product per wave");
    T* stg = reinterpret_cast<T*>(lds + L::off_stage) + wv_id * 16 * L::LS;
    const int mi = wv_id % NB;
    const bool isu = wv_id >= NB;
    const T* Bop = isu ? sW : sB;
    T* gout = (isu ? g_u : g_wt) + (size_t)16 * mi * K;
    // A is block lower triangular; a caller's A (kernel C alone) is read whole
    int kr = ST == kIntraRecompute ? C : 16 * (mi + 1);
    kr = ((kr + Mma<T>::KS - 1) / Mma<T>::KS) * Mma<T>::KS;
    if (kr > C) kr = C;
#pragma unroll
    for (int c0 = 0; c0 < K; c0 += 64) {
      f32x4 acc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = zero4();
      tile_mma_row<T, false, true, 4>(acc, opA, ldA, Bop, L::LK, 16 * mi, c0, kr);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[t][i] = fin(acc[t][i]);
        store_tile_n(stg, L::LS, 0, 16 * t, acc[t]);
      }
      wave_lds_sync();
#pragma unroll
      for (int e = lane_id(); e < 16 * 8; e += 64) {
        const int r = e / 8, c = (e % 8) * 8;
        *reinterpret_cast<uint4*>(gout + (size_t)r * K + c0 + c) = *reinterpret_cast<const uint4*>(stg + r * L::LS + c);
      }
      wave_lds_sync();  // the staging rows are rewritten next
    }
  } else {
    // a row block of w_pseudo or u per wave, its column tiles four at a time (their
    // MFMA chains overlap)
    static_assert(NW == 2 * NB && K == V, "a row block of each product per wave");
    const int mi = wv_id % NB;
    const bool isu = wv_id >= NB;
    int kr = ST == kIntraRecompute ? C : 16 * (mi + 1);
    kr = ((kr + Mma<T>::KS - 1) / Mma<T>::KS) * Mma<T>::KS;
    if (kr > C) kr = C;
    for (int c0 = 0; c0 < K; c0 += 64) {
      f32x4 acc[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = zero4();
      tile_mma_row<T, false, true, 4>(acc, opA, ldA, isu ? sW : sB, L::LK, 16 * mi, c0, kr);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[t][i] = fin(acc[t][i]);
        store_tile_n(isu ? g_u : g_wt, K, 16 * mi, c0 + 16 * t, acc[t]);
      }
    }
  }
}

// ------------------------------------------------------------------ state
// gdn2_fwd_state mode bits: keep the per-chunk states and v_new for the
// backward; write o per chunk ([B][H][NT][C][V], the layout of
// gdn2_inter_chunk_combine's result, kernel_d_pipeline.py:94-124) instead of
// [B][T][H][V]; sanitise h0 (nan_to_num(clip(h0, +-1e4)), its _sanitize_h0).
enum { kStateSave = 1, kStateChunkO = 2, kStateSanitizeH0 = 4 };

template <int C, int K, int VT>
struct StateLds {
  static constexpr int RB = K * 2, CB = C * 2, UB = VT * 2;  // row bytes
  // read before a step's first barrier only: two buffers
  static constexpr int s_w = 0, s_q = C * RB, s_u = 2 * C * RB, s_gl = s_u + C * UB;
  static constexpr int WQ = s_gl + K * 4;
  // loaded at the start of a step: three buffers
  static constexpr int s_kg = 0, s_a = C * RB;
  static constexpr int KA = C * RB + C * CB;
  static constexpr int off_wq = 0, off_ka = 2 * WQ, off_h = off_ka + 3 * KA;
  static constexpr int off_vn = off_h + K * UB;
  static constexpr int off_pf = off_vn + C * UB;  // where the prefetch wave's loads land
  static constexpr int total = off_pf + 256;
  static_assert(total <= 160 * 1024, "one workgroup per CU");
};

// bf16 state loop of one (batch, head, VT columns): waves 0-3 compute v_new
// and the state, 4-7 o, the next NL load the chunks (see gdn2_seq.hpp), two more
// store the saves (32 columns), and a last one, when launched, touches the lines
// of the chunk kPrefetch steps on: it hides memory latency that the loaders'
// two chunks in flight do not cover.
// v_new and the state are computed transposed (columns of h as MFMA rows), so
// a lane's four results are four consecutive columns of one row of the LDS
// copies.  Bound by the step's chain of LDS reads, MFMAs and two barriers when
// the operands come from L2 (0.87 us a chunk at 16 columns, 1.3 at 32, K =
// 128; the former kernel, in which every wave loaded, staged and computed,
// 1.40 and 1.7), and by HBM with 256 workgroups and the saves.
// Kernel times, former -> now: B1 T32768 H16 0.822 -> 0.508 ms, with saves 0.902
// -> 0.618; B8 T4096 H6 with saves 0.172 -> 0.150; B4 T8192 H16 0.270 -> 0.231,
// with saves 0.329 -> 0.297; K = 64 with saves, B2 T4096 H16 0.097 -> 0.070, B8
// T4096 H16 0.135 -> 0.137.
// The saves at 32 columns: as 64-byte row pieces by the o waves, inside their MFMA
// chain, they took the same bytes 0.344 ms at B4 T8192 H16 (the pieces by waves of
// their own 0.348), as whole rows 0.321, with the prefetch wave 0.297.  At 16
// columns latency bounds the step and more waves reading LDS lengthen it (B1
// T32768 H16: 0.634 against 0.617), so there the o waves store them.
// The prefetch distance: lines touched too early are gone again when the loader
// waves come.  32 columns, K = 128: two chunks (the one that the loaders request in
// the same step; B4 T8192 H16 with saves 0.297 ms and the bytes of the loaders
// alone; three chunks 1.3 times those and 0.307; B8 T4096 H6 0.150, three 0.152,
// four 1.19 times and 0.155).  Else three (B8 T4096 H12 K = 64 with saves 0.100 ms, two
// 0.105; 16 columns, B1 T32768 H16 with saves 0.618, two 0.623).
// AL = false: per-chunk arrays that are not 16-byte aligned (a caller's own).
template <int C, int K, int V, int VT, int NL, bool AL = true>
__global__ __launch_bounds__(512 + 64 * (NL + 3)) void gdn2_fwd_state(
    Gdn2Dims dm, Gdn2Chunks<bf16> ck, const float* __restrict__ h0, float* __restrict__ o,
    float* __restrict__ h_final, int mode) {
  typedef StateLds<C, K, VT> L;
  typedef Mma<bf16> M;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[L::total];
  constexpr int NVT = V / VT, NTI = VT / 16, RB = K / 64, XK = K / 32, XC = C / 32, PK = K / 8;
  static_assert(C == 64 && K % 64 == 0, "four row blocks");
  constexpr int kPrefetch = VT == 32 && K == 128 ? 2 : 3;
  int bh, vt;
  xcd_group_map(blockIdx.x, dm.B * dm.H, NVT, bh, vt);
  const int h = bh % dm.H, bb = bh / dm.H;
  const int v0 = vt * VT;
  const int wid = wave_id(), w = wid & 3, lane = lane_id(), r16 = lane & 15, g4 = lane >> 4;
  const size_t bh0 = (size_t)bh * dm.NT;
  const int last = dm.NT - 1;
  unsigned char* sH = lds + L::off_h;
  unsigned char* sVn = lds + L::off_vn;

  const bool save = (mode & kStateSave) != 0;
  const int nsave = VT == 32 && save ? 2 : 0;
  if (wid == 8 + NL + nsave) {
    // ---------------- L2 prefetch: the V tiles of a head share an XCD and split its lines
    auto prefetch = [&](int n) {
      if (n > last) return;
      auto part = [&](const void* p, int bytes) { touch_lines(p, bytes, NVT, vt, lds + L::off_pf); };
      part(ck.wt + (bh0 + n) * (C * K), C * K * 2);
      part(ck.qg + (bh0 + n) * (C * K), C * K * 2);
      part(ck.kg + (bh0 + n) * (C * K), C * K * 2);
      part(ck.aqk + (bh0 + n) * (C * C), C * C * 2);
      part(ck.u + (bh0 + n) * (C * V), C * V * 2);
    };
    for (int n = 2; n < kPrefetch; ++n) prefetch(n);
    bare_barrier();
    for (int n = 0; n < dm.NT; ++n) {
      prefetch(n + kPrefetch);
      bare_barrier();
      bare_barrier();
    }
    vm_wait<0>();  // nothing may still be on its way to this workgroup's LDS when it ends
    return;
  }
  if (VT == 32 && wid >= 8 + NL) {
    // ---------------- the saves, state and v_new transposed: a column block a wave
    const int sw = wid - 8 - NL;
    auto put = [&](const unsigned char* src, bf16* dst, auto nk) {
      constexpr int NK = decltype(nk)::value;  // k blocks of 32 columns
      bf16x8 a[NK];
#pragma unroll
      for (int s = 0; s < NK; ++s) a[s] = seq_colfrag<VT>(src, sw, 32 * s);
#pragma unroll
      for (int i = 0; i < NK; ++i) store_frags_1k<NK>(dst + (size_t)(v0 + 16 * sw) * (32 * NK), i, a);
    };
    __syncthreads();
    for (int n = 0; n < dm.NT; ++n) {
      put(sH, ck.hT + (bh0 + n) * (V * K), std::integral_constant<int, XK>());
      __syncthreads();
      put(sVn, ck.vnT + (bh0 + n) * (V * C), std::integral_constant<int, XC>());
      __syncthreads();
    }
    return;
  }
  if (wid >= 8) {
    // ---------------- loader waves
    const int lw = wid - 8;
    auto issue_ka = [&](int n) {
      unsigned char* b = lds + L::off_ka + (n % 3) * L::KA;
      dma_rows<K, NL, AL>(ck.kg + (bh0 + n) * (C * K), b + L::s_kg, lw);
      dma_rows<C, NL, AL>(ck.aqk + (bh0 + n) * (C * C), b + L::s_a, lw);
    };
    auto issue_wq = [&](int n) {
      unsigned char* b = lds + L::off_wq + (n & 1) * L::WQ;
      dma_rows<K, NL, AL>(ck.wt + (bh0 + n) * (C * K), b + L::s_w, lw);
      dma_rows<K, NL, AL>(ck.qg + (bh0 + n) * (C * K), b + L::s_q, lw);
      // u and gc_last: every wave issues the same number of instructions (it
      // counts them below), so a wave past the last piece repeats one
      constexpr int NI = C * L::UB / 1024, PU = VT / 8;
      static_assert(NI <= NL, "a wave loads one piece of u");
      const int ins = lw % NI, row = ins * (64 / PU) + lane / PU;
      copy16<AL>(ck.u + (bh0 + n) * (C * V) + v0 + row * V + (lane % PU) * 8, b + L::s_u + ins * 1024);
      if (lane < K / 4) copy16<AL>(ck.gcl + (bh0 + n) * K + lane * 4, b + L::s_gl);
    };
    // instructions of one chunk per wave: the wait that leaves only the newest chunk's outstanding
    constexpr int PER = (3 * C * L::RB + C * L::CB) / 1024 / NL + 2;
    static_assert(2 * PER <= 63, "two chunks' loads fit the wait counter");
    issue_ka(0);
    issue_wq(0);
    if (last > 0) {
      issue_ka(1);
      issue_wq(1);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(PER));
    } else {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    }
    loader_barrier<AL>();
    for (int n = 0; n < dm.NT; ++n) {
      const bool more = n + 2 <= last;
      if (more) issue_ka(n + 2);   // its buffer was read last before step n - 1's first barrier
      loader_barrier<AL>();
      if (more) {
        issue_wq(n + 2);           // its buffer was read last before this barrier
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(PER));
      } else {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
      }
      loader_barrier<AL>();
    }
    return;
  }

  if (wid < 4) {
    // ---------------- v_new and the state: h[d][v] with d = 16 (w RB + t) + r16, v = 16 u + 4 g4 + i
    f32x4 hs[RB][NTI];
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int u = 0; u < NTI; ++u) {
        const int d = 16 * (w * RB + t) + r16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float hv = h0 ? h0[((size_t)bh * K + d) * V + v0 + 16 * u + 4 * g4 + i] : 0.f;
          hs[t][u][i] = (mode & kStateSanitizeH0) ? sanitize(hv) : hv;
        }
        store4(reinterpret_cast<bf16*>(sH + seq_off<VT>(d, 16 * u + 4 * g4)), hs[t][u]);
      }
    __syncthreads();
    for (int n = 0; n < dm.NT; ++n) {
      const unsigned char* wq = lds + L::off_wq + (n & 1) * L::WQ;
      const unsigned char* ka = lds + L::off_ka + (n % 3) * L::KA;
      // v_new = u - w_pseudo h
      f32x4 x[NTI];
#pragma unroll
      for (int u = 0; u < NTI; ++u) x[u] = zero4();
#pragma unroll
      for (int s = 0; s < XK; ++s) {
        const bf16x8 wf = swz_rowfrag<PK>(wq + L::s_w, 16 * w, s);
#pragma unroll
        for (int u = 0; u < NTI; ++u) x[u] = M::mma(seq_colfrag<VT>(sH, u, 32 * s), wf, x[u]);
      }
      const int j = 16 * w + r16;
#pragma unroll
      for (int u = 0; u < NTI; ++u) {
        const bf16x4 uv = *reinterpret_cast<const bf16x4*>(wq + L::s_u + j * L::UB + (16 * u + 4 * g4) * 2);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[u][i] = (float)uv[i] - x[u][i];
        store4(reinterpret_cast<bf16*>(sVn + seq_off<VT>(j, 16 * u + 4 * g4)), x[u]);
      }
      // what does not need v_new: kg's fragments and h e^{gc_last}
      bf16x8 kt[RB][XC];
#pragma unroll
      for (int t = 0; t < RB; ++t) {
        const int d = 16 * (w * RB + t);
        const float e = __expf(*reinterpret_cast<const float*>(wq + L::s_gl + (d + r16) * 4));
#pragma unroll
        for (int s = 0; s < XC; ++s) kt[t][s] = swz_colfrag<PK>(ka + L::s_kg, d, 32 * s);
#pragma unroll
        for (int u = 0; u < NTI; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) hs[t][u][i] *= e;
      }
      __syncthreads();
      // h = sanitize(h e^{gc_last} + kg^T v_new)
#pragma unroll
      for (int s = 0; s < XC; ++s)
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
          const bf16x8 a = seq_colfrag<VT>(sVn, u, 32 * s);
#pragma unroll
          for (int t = 0; t < RB; ++t) hs[t][u] = M::mma(a, kt[t][s], hs[t][u]);
        }
#pragma unroll
      for (int t = 0; t < RB; ++t)
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
#pragma unroll
          for (int i = 0; i < 4; ++i) hs[t][u][i] = sanitize(hs[t][u][i]);
          store4(reinterpret_cast<bf16*>(sH + seq_off<VT>(16 * (w * RB + t) + r16, 16 * u + 4 * g4)), hs[t][u]);
        }
      __syncthreads();
    }
    if (h_final) {
#pragma unroll
      for (int t = 0; t < RB; ++t)
#pragma unroll
        for (int u = 0; u < NTI; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            h_final[((size_t)bh * K + 16 * (w * RB + t) + r16) * V + v0 + 16 * u + 4 * g4 + i] = hs[t][u][i];
    }
  } else {
    // ---------------- o = scale qg h + Aqk v_new (rows 16 w ...)
    const bool chunk_o = (mode & kStateChunkO) != 0;
    const size_t ors = chunk_o ? (size_t)V : (size_t)dm.H * V;  // o's row stride
    __syncthreads();
    for (int n = 0; n < dm.NT; ++n) {
      const size_t bhn = bh0 + n;
      const unsigned char* wq = lds + L::off_wq + (n & 1) * L::WQ;
      const unsigned char* ka = lds + L::off_ka + (n % 3) * L::KA;
      f32x4 x[NTI];
#pragma unroll
      for (int u = 0; u < NTI; ++u) x[u] = zero4();
#pragma unroll
      for (int s = 0; s < XK; ++s) {
        const bf16x8 qf = swz_rowfrag<PK>(wq + L::s_q, 16 * w, s);
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
          const bf16x8 a = seq_colfrag<VT>(sH, u, 32 * s);
          x[u] = M::mma(qf, a, x[u]);
          if (VT == 16 && save && s == w) store_frag_rows(ck.hT + bhn * V * K + (size_t)v0 * K + 32 * s, K, a);
        }
      }
#pragma unroll
      for (int u = 0; u < NTI; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) x[u][i] *= dm.scale;
      bf16x8 af[XC];
#pragma unroll
      for (int s = 0; s < XC; ++s) af[s] = swz_rowfrag<8>(ka + L::s_a, 16 * w, s);
      __syncthreads();
#pragma unroll
      for (int s = 0; s < XC; ++s)
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
          const bf16x8 a = seq_colfrag<VT>(sVn, u, 32 * s);
          if (32 * s <= 16 * w + 15) x[u] = M::mma(af[s], a, x[u]);  // Aqk is lower triangular
          if (VT == 16 && save && s == w) store_frag_rows(ck.vnT + bhn * V * C + (size_t)v0 * C + 32 * s, C, a);
        }
      if (o) {
        float* og = chunk_o ? o + bhn * C * V + v0 : o + (((size_t)bb * dm.T + (size_t)n * C) * dm.H + h) * V + v0;
#pragma unroll
        for (int u = 0; u < NTI; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) og[(size_t)(16 * w + 4 * g4 + i) * ors + 16 * u + r16] = n2n(x[u][i]);
      }
      __syncthreads();
    }
  }
}

// Sixteen bytes of an fp32 row per lane: row r16, elements k0 + 4 g4 + t; MFMA
// step t takes element t of every lane (k = k0 + 4 g4 + t), in both operands.
__device__ __forceinline__ f32x4 f32_col(const float* p, int ld, int i0, int k0) {
  const int l = lane_id();
  const float* q = p + (k0 + 4 * (l >> 4)) * ld + i0 + (l & 15);
  f32x4 v = {q[0], q[ld], q[2 * ld], q[3 * ld]};
  return v;
}
__device__ __forceinline__ f32x4 f32_mma(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int t = 0; t < 4; ++t) c = Mma<float>::mma(a[t], b[t], c);
  return c;
}

// fp32 state loop (two chunks of its operands do not fit the LDS): waves 0-3
// compute v_new and the state, 4-7 o and the saves, each holding the chunk's w
// / qg / Aqk row fragments in registers PD chunks ahead; kg passes through LDS
// (its fragments are columns).  K = 64 at B1 T512 H4: 0.037 -> 0.018 ms; B4
// T4096 H4 0.270 -> 0.117; K = 128, B4 T1024 H8 0.119 -> 0.065.  From more
// than one workgroup per CU of 16 columns on, 32 columns are faster (K = 64,
// 512 workgroups of 16: 0.040, 256 of 32: 0.029; K = 128: 0.155 and 0.116).
template <int C, int K, int V, int VT, int PD>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn2_fwd_state_f32(
    Gdn2Dims dm, Gdn2Chunks<float> ck, const float* __restrict__ h0, float* __restrict__ o,
    float* __restrict__ h_final, int mode) {
  constexpr int NVT = V / VT, NTI = VT / 16, RB = K / 64, XK = K / 16, XC = C / 16;
  constexpr int LK = K + 4, LV = VT + 4, KG = C * LK;
  static_assert(C == 64 && K % 64 == 0, "four row blocks");
  __shared__ __attribute__((aligned(16))) float lds[2 * KG + K * LV + C * LV];
  float* sH = lds + 2 * KG;
  float* sVn = sH + K * LV;
  int bh, vt;
  xcd_group_map(blockIdx.x, dm.B * dm.H, NVT, bh, vt);
  const int h = bh % dm.H, bb = bh / dm.H;
  const int v0 = vt * VT;
  const int w = wave_id() & 3, lane = lane_id(), r16 = lane & 15, g4 = lane >> 4;
  const size_t bh0 = (size_t)bh * dm.NT;
  const int last = dm.NT - 1;

  if (wave_id() < 4) {
    f32x4 hs[RB][NTI];
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int u = 0; u < NTI; ++u) {
        const int d = 16 * (w * RB + t) + r16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float hv = h0 ? h0[((size_t)bh * K + d) * V + v0 + 16 * u + 4 * g4 + i] : 0.f;
          hs[t][u][i] = (mode & kStateSanitizeH0) ? sanitize(hv) : hv;
        }
        store4(sH + d * LV + 16 * u + 4 * g4, hs[t][u]);
      }
    struct Set {
      f32x4 w[XK], u[NTI];
      float gl[RB];
    };
    Set S[PD];
    const int wo = (16 * w + r16) * K + 4 * g4, uo = (16 * w + r16) * V + v0 + 4 * g4;
    auto load = [&](Set& A, int n) {
      const float* wr = ck.wt + (bh0 + n) * (C * K);
      const float* ur = ck.u + (bh0 + n) * (C * V);
      const float* gr = ck.gcl + (bh0 + n) * K;
#pragma unroll
      for (int s = 0; s < XK; ++s) A.w[s] = *reinterpret_cast<const f32x4*>(wr + wo + s * 16);
#pragma unroll
      for (int u = 0; u < NTI; ++u) A.u[u] = *reinterpret_cast<const f32x4*>(ur + uo + 16 * u);
#pragma unroll
      for (int t = 0; t < RB; ++t) A.gl[t] = gr[16 * (w * RB + t) + r16];
    };
#pragma unroll
    for (int i = 0; i < PD; ++i) load(S[i], min(i, last));
    __syncthreads();
    auto step = [&](int n, Set& A) {
      const float* sKg = lds + (n & 1) * KG;
      f32x4 x[NTI];
#pragma unroll
      for (int u = 0; u < NTI; ++u) x[u] = zero4();
#pragma unroll
      for (int s = 0; s < XK; ++s)
#pragma unroll
        for (int u = 0; u < NTI; ++u) x[u] = f32_mma(f32_col(sH, LV, 16 * u, s * 16), A.w[s], x[u]);
#pragma unroll
      for (int u = 0; u < NTI; ++u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[u][i] = A.u[u][i] - x[u][i];
        store4(sVn + (16 * w + r16) * LV + 16 * u + 4 * g4, x[u]);
      }
      f32x4 kt[RB][XC];
#pragma unroll
      for (int t = 0; t < RB; ++t) {
#pragma unroll
        for (int s = 0; s < XC; ++s) kt[t][s] = f32_col(sKg, LK, 16 * (w * RB + t), s * 16);
        const float e = __expf(A.gl[t]);
#pragma unroll
        for (int u = 0; u < NTI; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) hs[t][u][i] *= e;
      }
      load(A, min(n + PD, last));
      __syncthreads();
#pragma unroll
      for (int s = 0; s < XC; ++s)
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
          const f32x4 a = f32_col(sVn, LV, 16 * u, s * 16);
#pragma unroll
          for (int t = 0; t < RB; ++t) hs[t][u] = f32_mma(a, kt[t][s], hs[t][u]);
        }
#pragma unroll
      for (int t = 0; t < RB; ++t)
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
#pragma unroll
          for (int i = 0; i < 4; ++i) hs[t][u][i] = sanitize(hs[t][u][i]);
          store4(sH + (16 * (w * RB + t) + r16) * LV + 16 * u + 4 * g4, hs[t][u]);
        }
      __syncthreads();
    };
    int n = 0;
    for (; n + PD <= dm.NT; n += PD) {
#pragma unroll
      for (int i = 0; i < PD; ++i) step(n + i, S[i]);
    }
#pragma unroll
    for (int i = 0; i < PD; ++i)
      if (n + i < dm.NT) step(n + i, S[i]);
    if (h_final) {
#pragma unroll
      for (int t = 0; t < RB; ++t)
#pragma unroll
        for (int u = 0; u < NTI; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            h_final[((size_t)bh * K + 16 * (w * RB + t) + r16) * V + v0 + 16 * u + 4 * g4 + i] = hs[t][u][i];
    }
  } else {
    constexpr int PIECES = C * K / 4 / 256, PER_ROW = K / 4;  // 16-byte kg pieces per thread
    struct Set { f32x4 q[XK], a[XC]; };
    struct KSet { f32x4 p[PIECES]; };
    Set S[PD];
    KSet G[PD];
    const int tid = threadIdx.x & 255;
    const int qo = (16 * w + r16) * K + 4 * g4, ao = (16 * w + r16) * C + 4 * g4;
    auto load = [&](Set& A, int n) {
      const float* qr = ck.qg + (bh0 + n) * (C * K);
      const float* ar = ck.aqk + (bh0 + n) * (C * C);
#pragma unroll
      for (int s = 0; s < XK; ++s) A.q[s] = *reinterpret_cast<const f32x4*>(qr + qo + s * 16);
#pragma unroll
      for (int s = 0; s < XC; ++s) A.a[s] = *reinterpret_cast<const f32x4*>(ar + ao + s * 16);
    };
    auto load_kg = [&](KSet& A, int n) {
      const float* kr = ck.kg + (bh0 + n) * (C * K);
#pragma unroll
      for (int i = 0; i < PIECES; ++i) A.p[i] = *reinterpret_cast<const f32x4*>(kr + (tid + 256 * i) * 4);
    };
    auto commit = [&](const KSet& A, int n) {
      float* d = lds + (n & 1) * KG;
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const int e = tid + 256 * i;
        *reinterpret_cast<f32x4*>(d + (e / PER_ROW) * LK + (e % PER_ROW) * 4) = A.p[i];
      }
    };
    const bool save = (mode & kStateSave) != 0;
    const bool chunk_o = (mode & kStateChunkO) != 0;
    const size_t ors = chunk_o ? (size_t)V : (size_t)dm.H * V;
    {
      KSet k0;
      load_kg(k0, 0);
#pragma unroll
      for (int i = 0; i < PD; ++i) {
        load(S[i], min(i, last));
        load_kg(G[i], min(i + 1, last));
      }
      commit(k0, 0);
    }
    __syncthreads();
    // B holds chunk n + 1's kg
    auto step = [&](int n, Set& A, KSet& B) {
      const size_t bhn = bh0 + n;
      f32x4 x[NTI];
#pragma unroll
      for (int u = 0; u < NTI; ++u) x[u] = zero4();
#pragma unroll
      for (int s = 0; s < XK; ++s)
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
          const f32x4 a = f32_col(sH, LV, 16 * u, s * 16);
          x[u] = f32_mma(A.q[s], a, x[u]);
          if (save && (s & 3) == w)
            *reinterpret_cast<f32x4*>(ck.hT + bhn * V * K + (size_t)(v0 + 16 * u + r16) * K + s * 16 + 4 * g4) = a;
        }
#pragma unroll
      for (int u = 0; u < NTI; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) x[u][i] *= dm.scale;
      commit(B, n + 1);   // past the last chunk: a copy nobody reads
      load_kg(B, min(n + PD + 1, last));
      __syncthreads();
#pragma unroll
      for (int s = 0; s < XC; ++s)
#pragma unroll
        for (int u = 0; u < NTI; ++u) {
          const f32x4 a = f32_col(sVn, LV, 16 * u, s * 16);
          if (s <= w) x[u] = f32_mma(A.a[s], a, x[u]);   // Aqk is lower triangular
          if (save && (s & 3) == w)
            *reinterpret_cast<f32x4*>(ck.vnT + bhn * V * C + (size_t)(v0 + 16 * u + r16) * C + s * 16 + 4 * g4) = a;
        }
      if (o) {
        float* og = chunk_o ? o + bhn * C * V + v0 : o + (((size_t)bb * dm.T + (size_t)n * C) * dm.H + h) * V + v0;
#pragma unroll
        for (int u = 0; u < NTI; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) og[(size_t)(16 * w + 4 * g4 + i) * ors + 16 * u + r16] = n2n(x[u][i]);
      }
      load(A, min(n + PD, last));
      __syncthreads();
    };
    int n = 0;
    for (; n + PD <= dm.NT; n += PD) {
#pragma unroll
      for (int i = 0; i < PD; ++i) step(n + i, S[i], G[i]);
    }
#pragma unroll
    for (int i = 0; i < PD; ++i)
      if (n + i < dm.NT) step(n + i, S[i], G[i]);
  }
}

}  // namespace ah
