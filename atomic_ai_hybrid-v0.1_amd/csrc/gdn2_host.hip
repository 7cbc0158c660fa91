// Host side of the GDN2 chunk pipeline: argument checks, workspace layout,
// template dispatch and the extern "C" entry points of include/atomic_hybrid.h.
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/atomic_hybrid.h"
#include "diag.hpp"
#include "gdn2_bwd.hip"
#include "launch.hpp"
#include "stage256.hpp"
#include "ws_tag.hpp"

namespace ah {

static size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// ------------------------------------------------ workspace records (ws_tag.hpp)
namespace {
struct WsEntry {
  const char *lo, *hi;
  WsTag t;
};
std::mutex g_ws_mu;
std::vector<WsEntry> g_ws_tags;
bool ws_same(const WsTag& a, const WsTag& b) {
  if (a.kind != b.kind) return false;
  for (int i = 0; i < 8; ++i)
    if (a.dims[i] != b.dims[i] || a.ptrs[i] != b.ptrs[i] || a.strides[i] != b.strides[i]) return false;
  return true;
}
void ws_erase_overlap(const char* lo, const char* hi) {
  size_t j = 0;
  for (size_t i = 0; i < g_ws_tags.size(); ++i)
    if (g_ws_tags[i].hi <= lo || g_ws_tags[i].lo >= hi) g_ws_tags[j++] = g_ws_tags[i];
  g_ws_tags.resize(j);
}
}  // namespace

void ws_tag_clobber(const void* ws, size_t bytes) {
  if (!ws) return;
  std::lock_guard<std::mutex> lk(g_ws_mu);
  const char* lo = static_cast<const char*>(ws);
  ws_erase_overlap(lo, lo + bytes);
}
void ws_tag_set(const void* ws, size_t bytes, const WsTag& t) {
  if (!ws) return;
  std::lock_guard<std::mutex> lk(g_ws_mu);
  const char* lo = static_cast<const char*>(ws);
  ws_erase_overlap(lo, lo + bytes);
  if (g_ws_tags.size() >= 1024) g_ws_tags.erase(g_ws_tags.begin());  // oldest record
  g_ws_tags.push_back(WsEntry{lo, lo + bytes, t});
}
bool ws_tag_matches(const void* ws, const WsTag& t) {
  std::lock_guard<std::mutex> lk(g_ws_mu);
  for (const WsEntry& e : g_ws_tags)
    if (e.lo == static_cast<const char*>(ws)) return ws_same(e.t, t);
  return false;
}

// the forward a GDN2 workspace holds: shapes, dtype, query scale (folded into
// the saved Aqk), whether h0 was sanitised, and the input pointers
static WsTag gdn2_tag(const atomic_gdn2_args* a, const void* q, const void* k, const void* v, const void* w,
                      const void* b, const void* g, const void* h0) {
  WsTag t{};
  t.kind = (a->flags & ATOMIC_GDN2_SANITIZE_H0) ? 0x101 : 1;
  int32_t scale_bits;
  static_assert(sizeof(scale_bits) == sizeof(a->scale), "scale is a 32-bit float");
  memcpy(&scale_bits, &a->scale, sizeof(scale_bits));
  const int32_t d[8] = {a->batch, a->seqlen, a->heads, a->dk, a->dv, a->chunk, a->dtype, scale_bits};
  const void* ptr[8] = {q, k, v, w, b, g, h0, nullptr};
  for (int i = 0; i < 8; ++i) { t.dims[i] = d[i]; t.ptrs[i] = ptr[i]; }
  const int64_t dK = (int64_t)a->heads * a->dk, dV = (int64_t)a->heads * a->dv;
  const int64_t dense[6] = {dK, dK, dV, dV, dK, dK};
  for (int i = 0; i < 6; ++i) t.strides[i] = a->row_stride[i] ? a->row_stride[i] : dense[i];  // the forward's inputs
  return t;
}

// The chunk length every GDN2 kernel runs at.
constexpr int kGdn2RunChunk = 64;

struct Gdn2Plan {
  Gdn2Dims dm;
  int es;        // operand element size
  bool sanitize_h0;  // ATOMIC_GDN2_SANITIZE_H0: the state loop clips / nan_to_nums h0 first
  size_t bhn;    // B * H * NT
  // forward intermediates
  size_t o_qg, o_kg, o_wt, o_u, o_aqk, o_ainv, o_gcl, o_ht, o_vnt, fwd_end;
  // backward scratch
  size_t o_dvn, o_dht, o_dqg, o_dwt, o_dkb, o_dkg, o_daqk, o_dakk, o_rlast, total;
};

static int gdn2_plan(const atomic_gdn2_args* a, Gdn2Plan* p) {
  if (!a) return ATOMIC_ERR_NULL;
  if (a->dtype != ATOMIC_F32 && a->dtype != ATOMIC_BF16) return ATOMIC_ERR_DTYPE;
  if (a->do_dtype != ATOMIC_F32 && a->do_dtype != ATOMIC_BF16) return ATOMIC_ERR_DTYPE;
  if (a->batch <= 0 || a->heads <= 0 || a->seqlen <= 0) return ATOMIC_ERR_SHAPE;
  if (a->chunk != 64 && a->chunk != 128 && a->chunk != 256) return ATOMIC_ERR_SHAPE;
  if (a->seqlen % a->chunk != 0) return ATOMIC_ERR_SHAPE;
  if (!((a->dk == 64 || a->dk == 128) && a->dv == a->dk)) return ATOMIC_ERR_SHAPE;
  Gdn2Dims d;
  // Chunks of 128 or 256 (the reference's Pallas path runs BT = 256,
  // kernel_a_scores.py:15-17; its oracle takes any chunk_size,
  // gdn2_wy_reference.py:105-112) run as 64-row chunks.  The chunked WY form
  // is exact for any chunk length; with every gate g <= 0 (the model's
  // g = -exp(a) softplus(f), model.py:606-610) the two differ only where the
  // reference's clip(+-20) floors a pair decay below exp(-20), and in the
  // +-1e4 state clip, applied at every 64 rows instead of every chunk.
  d.B = a->batch; d.T = a->seqlen; d.H = a->heads; d.K = a->dk; d.V = a->dv; d.C = kGdn2RunChunk;
  d.NT = a->seqlen / kGdn2RunChunk; d.scale = a->scale;
  {
    const long long dK = (long long)a->heads * a->dk, dV = (long long)a->heads * a->dv;
    const long long dense[7] = {dK, dK, dV, dV, dK, dK, dV};
    long long* out[7] = {&d.rq, &d.rk, &d.rv, &d.rw, &d.rb, &d.rg, &d.rdo};
    for (int i = 0; i < 7; ++i) {
      const long long s = a->row_stride[i];
      if (s != 0 && (s < dense[i] || s % 8 != 0)) return ATOMIC_ERR_SHAPE;
      *out[i] = s ? s : dense[i];
    }
  }
  p->dm = d;
  p->es = a->dtype == ATOMIC_BF16 ? 2 : 4;
  p->sanitize_h0 = (a->flags & ATOMIC_GDN2_SANITIZE_H0) != 0;
  const size_t N = (size_t)d.B * d.H * d.NT;
  p->bhn = N;
  const size_t es = p->es, C = d.C, K = d.K, V = d.V;
  size_t off = 0;
  auto take = [&](size_t bytes) { size_t o = off; off += align256(bytes); return o; };
  p->o_qg = take(N * C * K * es);
  p->o_kg = take(N * C * K * es);
  p->o_wt = take(N * C * K * es);
  p->o_u = take(N * C * V * es);
  p->o_aqk = take(N * C * C * es);
  p->o_ainv = take(N * C * C * es);
  p->o_gcl = take(N * K * 4);
  p->o_ht = take(N * V * K * es);
  p->o_vnt = take(N * V * C * es);
  p->fwd_end = off;
  p->o_dvn = take(N * C * V * es);
  p->o_dht = take(N * V * K * es);
  p->o_dqg = take(N * C * K * es);
  p->o_dwt = take(N * C * K * es);
  p->o_dkb = take(N * C * K * es);
  p->o_dkg = take(N * C * K * es);
  p->o_daqk = take(N * C * C * es);
  p->o_dakk = take(N * C * C * es);
  p->o_rlast = take(N * K * 4);
  p->total = off;
  return ATOMIC_OK;
}

template <typename T>
static Gdn2Chunks<T> gdn2_chunks(const Gdn2Plan& p, void* ws) {
  char* base = static_cast<char*>(ws);
  Gdn2Chunks<T> c;
  c.qg = reinterpret_cast<T*>(base + p.o_qg);
  c.kg = reinterpret_cast<T*>(base + p.o_kg);
  c.wt = reinterpret_cast<T*>(base + p.o_wt);
  c.u = reinterpret_cast<T*>(base + p.o_u);
  c.aqk = reinterpret_cast<T*>(base + p.o_aqk);
  c.ainv = reinterpret_cast<T*>(base + p.o_ainv);
  c.akk = nullptr;
  c.gcl = reinterpret_cast<float*>(base + p.o_gcl);
  c.hT = reinterpret_cast<T*>(base + p.o_ht);
  c.vnT = reinterpret_cast<T*>(base + p.o_vnt);
  return c;
}

// Whether the arrays that the chunk loops load straight to LDS lie on 16-byte addresses.
template <typename T>
static bool gdn2_aligned(const Gdn2Chunks<T>& c) {
  return aligned16({c.wt, c.qg, c.kg, c.aqk, c.u, c.gcl});
}

// Kernels A + B + C (gdn2_fwd_intra): the per-chunk intermediates into ck.
template <typename T, int K, int ST = kIntraAll>
static int gdn2_intra_launch(const Gdn2Plan& p, const void* q, const void* k, const void* v, const void* w,
                             const void* b, const float* g, const Gdn2Chunks<T>& ck, Launch& L) {
  constexpr int C = 64, V = K;
  hipStream_t st = L.st;
  static const char* const names[] = {"gdn2_fwd_intra", "gdn2_chunk_scores", "gdn2_wy_solve", "gdn2_recompute_wy"};
  return L(names[ST], [&] {
    hipLaunchKernelGGL((gdn2_fwd_intra<T, C, K, V, ST>), dim3((unsigned)p.bhn), dim3(512), 0, st, p.dm,
                       (const T*)q, (const T*)k, (const T*)v, (const T*)w, (const T*)b, g, ck);
  });
}

// Whether the chunk loops' V tiles of one head land on one XCD (xcd_group_map).
static bool gdn2_tiles_share_l2(int bh) { return bh % 8 == 0; }
// 16-column tiles in the bf16 chunk loops: up to a workgroup per CU, or three to
// every four CUs where the tiles of a head do not share an L2 and each fetches the
// chunk's operands for itself (T2048 K = 128 forward / with saves / dh: 20 heads
// 49 / 53 / 55 us against 45 / 64 / 56 with 32 columns, 25 heads 62 / 68 / 65
// against 46 / 65 / 57, 31 heads 79 / 90 / 84 against 45 / 76 / 59; K = 64, 41
// heads 33 / 36 / 40 against 30 / 39 / 40, 50 heads 41 / 46 / 43 against 31 / 44 / 41).
static bool gdn2_narrow(int bh, int V) { return bh * (V / 16) <= (gdn2_tiles_share_l2(bh) ? 256 : 192); }

// Kernels A + B + C (gdn2_fwd_intra): the) over the intermediates in ck; mode: kState* bits.
template <typename T, int K>
static int gdn2_state_launch(const Gdn2Plan& p, const Gdn2Chunks<T>& ck, const float* h0, float* o,
                             float* h_final, int mode, Launch& L) {
  constexpr int C = 64, V = K;
  hipStream_t st = L.st;
  const int bh = p.dm.B * p.dm.H;
  // V tiles of 16 columns while they fit one workgroup per CU (256 CUs): the
  // chunk step is shorter and twice the workgroups walk the chunks; every tile
  // re-reads the chunk's w, q, kg, which its XCD's L2 serves.  Past that, 32
  // (B4 T8192 H16 K = 128 without saves: 0.36 ms with 16, 0.25 with 32).
  const bool narrow = sizeof(T) == 2 ? gdn2_narrow(bh, V) : bh * (V / 16) <= 256;
  return L("gdn2_fwd_state", [&] {
    if constexpr (sizeof(T) == 2) {
      const int ns = mode & kStateSave ? 2 : 0;  // waves that store the saves (32 columns)
      // the loader waves' 16-byte loads to LDS need aligned arrays; a caller's own
      // (or its workspace) may not be, and go through registers
      if (!gdn2_aligned(ck)) {
        hipLaunchKernelGGL((gdn2_fwd_state<C, K, V, 32, 4, false>), dim3((unsigned)(bh * (V / 32))),
                           dim3(512 + 64 * (4 + ns)), 0, st, p.dm, ck, h0, o, h_final, mode);
        return;
      }
      // The prefetch wave where the tiles of a head share an L2 (elsewhere each
      // XCD gets only its share of the lines: B3 T4096 H21, 32 columns, 0.186 ms
      // with it, 0.173 without; T2048, 12 heads 0.035 and 0.033).  There it hides
      // latency with 16 columns (B1 T8192 H32: 0.156 ms with it, 0.208 without,
      // with saves 0.187 and 0.279; B1 T32768 H16: 0.51 and 0.66) and with 32 while
      // the workgroups leave CUs idle or store the saves (B8 T4096 H6 with saves
      // 0.150 and 0.168; B4 T8192 H16 with saves 0.297 and 0.321; B4 T4096 H16, 256
      // workgroups without saves and three chunks ahead, 0.132 and 0.131).
      const bool shared = gdn2_tiles_share_l2(bh);
      if (narrow) {
        const unsigned nwg = (unsigned)(bh * (V / 16));
        hipLaunchKernelGGL((gdn2_fwd_state<C, K, V, 16, 2>), dim3(nwg), dim3(512 + 64 * (2 + shared)), 0, st, p.dm, ck,
                           h0, o, h_final, mode);
      } else {
        const unsigned nwg = (unsigned)(bh * (V / 32));
        hipLaunchKernelGGL((gdn2_fwd_state<C, K, V, 32, 4>), dim3(nwg),
                           dim3(512 + 64 * (4 + ns + (shared && (nwg < 256 || ns)))), 0, st, p.dm, ck, h0, o, h_final, mode);
      }
    } else {
      if (narrow)
        hipLaunchKernelGGL((gdn2_fwd_state_f32<C, K, V, 16, K == 64 ? 2 : 1>), dim3((unsigned)(bh * (V / 16))),
                           dim3(512), 0, st, p.dm, ck, h0, o, h_final, mode);
      else
        hipLaunchKernelGGL((gdn2_fwd_state_f32<C, K, V, 32, 1>), dim3((unsigned)(bh * (V / 32))), dim3(512), 0, st,
                           p.dm, ck, h0, o, h_final, mode);
    }
  });
}

template <typename T, int K>
static int gdn2_forward_impl(const Gdn2Plan& p, const void* q, const void* k, const void* v,
                             const void* w, const void* b, const float* g, const float* h0,
                             float* o, float* h_final, void* ws, int save, Launch& L) {
  Gdn2Chunks<T> ck = gdn2_chunks<T>(p, ws);
  int rc = gdn2_intra_launch<T, K>(p, q, k, v, w, b, g, ck, L);
  if (rc) return rc;
  const int mode = (save ? kStateSave : 0) | (p.sanitize_h0 ? kStateSanitizeH0 : 0);
  return gdn2_state_launch<T, K>(p, ck, h0, o, h_final, mode, L);
}

template <typename T>
static Gdn2Grads<T> gdn2_grads(const Gdn2Plan& p, void* ws) {
  char* base = static_cast<char*>(ws);
  Gdn2Grads<T> g;
  g.dvn = reinterpret_cast<T*>(base + p.o_dvn);
  g.dhT = reinterpret_cast<T*>(base + p.o_dht);
  g.dqg = reinterpret_cast<T*>(base + p.o_dqg);
  g.dwt = reinterpret_cast<T*>(base + p.o_dwt);
  g.dkb = reinterpret_cast<T*>(base + p.o_dkb);
  g.dkg = reinterpret_cast<T*>(base + p.o_dkg);
  g.daqk = reinterpret_cast<T*>(base + p.o_daqk);
  g.dakk = reinterpret_cast<T*>(base + p.o_dakk);
  g.rlast = reinterpret_cast<float*>(base + p.o_rlast);
  return g;
}

template <typename T, typename TD, int K>
static int gdn2_backward_impl(const Gdn2Plan& p, const void* q, const void* k, const void* v,
                              const void* w, const void* b, const float* g, const float* h0,
                              const void* dO, const float* dh_final, void* dq, void* dk, void* dv,
                              void* dw, void* db, float* dg, float* dh0, void* ws, bool reuse,
                              Launch& L) {
  constexpr int C = 64, V = K, VT = 32;
  Gdn2Chunks<T> ck = gdn2_chunks<T>(p, ws);
  Gdn2Grads<T> gr = gdn2_grads<T>(p, ws);
  int rc;
  if (!reuse) {
    // recompute the forward intermediates (the reference's residuals are the
    // inputs only, kernel_trainable_B6.py:91-94,104-111)
    rc = gdn2_forward_impl<T, K>(p, q, k, v, w, b, g, h0, nullptr, nullptr, ws, 1, L);
    if (rc) return rc;
  }
  hipStream_t st = L.st;
  const int bh = p.dm.B * p.dm.H;
  const unsigned nblk = (unsigned)p.bhn;
  // 16-column V tiles under the same condition as the forward state loop (B4
  // T8192 H16 K = 128: 0.39 ms with 16, 0.30 with 32).  The prefetch wave where
  // tiles share an L2, with 16 columns (B1 T8192 H32: 0.170 ms with it, 0.231
  // without) and with 32 at K = 128 (B4 T8192 H16 0.246 and 0.281), where a chunk
  // is twice the bytes of K = 64 (B8 T4096 H12 0.103 and 0.096).
  rc = L("gdn2_bwd_dh", [&] {
    if constexpr (sizeof(T) == 2) {
      constexpr int NL = 2, NT0 = 512 + 64 * (NL + 2);
      const bool al = gdn2_aligned(ck), narrow = al && gdn2_narrow(bh, V);
      const unsigned nwg = (unsigned)(bh * (V / (narrow ? 16 : VT)));
      const unsigned nthr = NT0 + 64 * (gdn2_tiles_share_l2(bh) && (narrow || K == 128));
      if (!al)  // as in the forward state loop
        hipLaunchKernelGGL((gdn2_bwd_dh<TD, C, K, V, VT, NL, false>), dim3(nwg), dim3(NT0), 0, st, p.dm, ck, gr,
                           (const TD*)dO, dh_final, dh0);
      else if (narrow)
        hipLaunchKernelGGL((gdn2_bwd_dh<TD, C, K, V, 16, NL>), dim3(nwg), dim3(nthr), 0, st, p.dm, ck, gr,
                           (const TD*)dO, dh_final, dh0);
      else
        hipLaunchKernelGGL((gdn2_bwd_dh<TD, C, K, V, VT, NL>), dim3(nwg), dim3(nthr), 0, st, p.dm, ck, gr,
                           (const TD*)dO, dh_final, dh0);
    } else {
      hipLaunchKernelGGL((gdn2_bwd_dh_f32<T, TD, C, K, V, VT>), dim3((unsigned)(bh * (V / VT))), dim3(512), 0, st,
                         p.dm, ck, gr, (const TD*)dO, dh_final, dh0);
    }
  });
  if (rc) return rc;
  rc = L("gdn2_bwd_hgrad", [&] {
    hipLaunchKernelGGL((gdn2_bwd_hgrad<T, TD, C, K, V>), dim3(nblk), dim3(256), 0, st, p.dm, ck, gr,
                       (const TD*)dO);
  });
  if (rc) return rc;
  rc = L("gdn2_bwd_wy", [&] {
    hipLaunchKernelGGL((gdn2_bwd_wy<T, C, K, V>), dim3(nblk), dim3(256), 0, st, p.dm, ck, gr,
                       (const T*)k, (const T*)v, (const T*)w, (const T*)b, g, (T*)dw, (T*)dv);
  });
  if (rc) return rc;
  constexpr int KH = 64;  // column slice of the intra kernel
  return L("gdn2_bwd_intra", [&] {
    hipLaunchKernelGGL((gdn2_bwd_intra<T, C, K, V, KH>), dim3(nblk * (K / KH)), dim3(256), 0, st, p.dm, gr,
                       (const T*)q, (const T*)k, (const T*)b, g, (T*)dq, (T*)dk, (T*)db, dg);
  });
}

int gdn2_backward(const Gdn2Plan& p, int dtype, int do_dtype, const void* q, const void* k,
                  const void* v, const void* w, const void* b, const float* g, const float* h0,
                  const void* dO, const float* dh_final, void* dq, void* dk, void* dv, void* dw,
                  void* db, float* dg, float* dh0, void* ws, bool reuse, Launch& L) {
#define AH_GDN2_BWD(T, TD, KK) \
  return gdn2_backward_impl<T, TD, KK>(p, q, k, v, w, b, g, h0, dO, dh_final, dq, dk, dv, dw, db, dg, dh0, ws, reuse, L)
  if (dtype == ATOMIC_BF16) {
    if (p.dm.K == 128) {
      if (do_dtype == ATOMIC_BF16) AH_GDN2_BWD(bf16, bf16, 128);
      AH_GDN2_BWD(bf16, float, 128);
    }
    if (do_dtype == ATOMIC_BF16) AH_GDN2_BWD(bf16, bf16, 64);
    AH_GDN2_BWD(bf16, float, 64);
  }
  // fp32 operands: at K = 128 every backward kernel fits the LDS at one
  // workgroup per CU (gdn2_bwd_dh 160 KB, gdn2_bwd_hgrad 136 KB)
  if (p.dm.K == 128) {
    if (do_dtype == ATOMIC_BF16) AH_GDN2_BWD(float, bf16, 128);
    AH_GDN2_BWD(float, float, 128);
  }
  if (do_dtype == ATOMIC_BF16) AH_GDN2_BWD(float, bf16, 64);
  AH_GDN2_BWD(float, float, 64);
#undef AH_GDN2_BWD
}

int gdn2_forward(const Gdn2Plan& p, int dtype, const void* q, const void* k, const void* v,
                 const void* w, const void* b, const float* g, const float* h0, float* o,
                 float* h_final, void* ws, int save, Launch& L) {
  if (dtype == ATOMIC_BF16) {
    if (p.dm.K == 128) return gdn2_forward_impl<bf16, 128>(p, q, k, v, w, b, g, h0, o, h_final, ws, save, L);
    return gdn2_forward_impl<bf16, 64>(p, q, k, v, w, b, g, h0, o, h_final, ws, save, L);
  }
  if (p.dm.K == 128) return gdn2_forward_impl<float, 128>(p, q, k, v, w, b, g, h0, o, h_final, ws, save, L);
  return gdn2_forward_impl<float, 64>(p, q, k, v, w, b, g, h0, o, h_final, ws, save, L);
}

// ------------------------------------------------ stage reports
// Akk of one chunk (kernel A's second output, gdn2_wy_reference.py:80-81,87),
// recomputed pairwise from the inputs for its stage report: the fused intra
// kernel keeps it in LDS only.
//   Akk[i,j] = n2n(sum_d (b k)[i,d] k[j,d] exp(clip(gc[i,d] - gc[j,d], +-20))), i > j
template <typename T, int C, int K>
__global__ __launch_bounds__(256) void gdn2_diag_akk(Gdn2Dims dm, const T* __restrict__ k,
                                                     const T* __restrict__ b, const float* __restrict__ g,
                                                     atomic_stage_report* r) {
  constexpr int LD = K + 1;
  __shared__ float sgc[C * LD], sk[C * LD], sbk[C * LD];
  const int tid = threadIdx.x, bhn = blockIdx.x;
  const int n = bhn % dm.NT, bh = bhn / dm.NT, h = bh % dm.H, bb = bh / dm.H;
  const size_t t0 = (size_t)bb * dm.T + (size_t)n * C;
  for (int e = tid; e < C * K; e += 256) {
    const int i = e / K, d = e % K;
    const size_t hd = (size_t)h * K + d;
    const float kv = to_f(k[(t0 + i) * dm.rk + hd]);
    sgc[i * LD + d] = g[(t0 + i) * dm.rg + hd];
    sk[i * LD + d] = kv;
    sbk[i * LD + d] = to_f(b[(t0 + i) * dm.rb + hd]) * kv;
  }
  __syncthreads();
  for (int d = tid; d < K; d += 256)
    for (int i = 1; i < C; ++i) sgc[i * LD + d] += sgc[(i - 1) * LD + d];
  __syncthreads();
  uint32_t bad = 0;
  float mx = 0.f;
  for (int e = tid; e < C * C; e += 256) {
    const int i = e / C, j = e % C;
    if (i <= j) continue;
    float acc = 0.f;
    for (int d = 0; d < K; ++d) {
      const float dd = fminf(fmaxf(sgc[i * LD + d] - sgc[j * LD + d], -kClipDecay), kClipDecay);
      acc += sbk[i * LD + d] * sk[j * LD + d] * __expf(dd);
    }
    acc = n2n(acc);
    if (__builtin_isfinite(acc)) mx = fmaxf(mx, fabsf(acc));
    else ++bad;
  }
  stage_report_fold(bad, mx, r);
}

// Forward stage reports from the workspace of plan p (one window, for the
// no-allocation forward) and the outputs o / h_final (either may be NULL).
template <typename T, int K>
static int gdn2_forward_diag_t(const Gdn2Plan& p, StageDiag& D, const void* k, const void* b,
                               const float* g, const float* o, const float* h_final, void* ws) {
  constexpr int C = 64, V = K;
  const Gdn2Chunks<T> ck = gdn2_chunks<T>(p, ws);
  const size_t N = p.bhn;
  int rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_AQK, ck.aqk, N * C * C))) return rc;
  rc = D.L("gdn2_diag_akk", [&] {
    hipLaunchKernelGGL((gdn2_diag_akk<T, C, K>), dim3((unsigned)N), dim3(256), 0, D.L.st, p.dm, (const T*)k,
                       (const T*)b, g, D.r + ATOMIC_GDN2_DIAG_AKK);
  });
  if (rc) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_AINV, ck.ainv, N * C * C))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_W_PSEUDO, ck.wt, N * C * K))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_U, ck.u, N * C * V))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_KG, ck.kg, N * C * K))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_QG, ck.qg, N * C * K))) return rc;
  const size_t rows = (size_t)p.dm.B * p.dm.T * p.dm.H;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_O, o, rows * V))) return rc;
  return D.reduce(ATOMIC_GDN2_DIAG_H_FINAL, h_final, (size_t)p.dm.B * p.dm.H * K * V);
}

static int gdn2_forward_diag(const Gdn2Plan& p, int dtype, StageDiag& D, const void* k, const void* b,
                             const float* g, const float* o, const float* h_final, void* ws) {
  if (dtype == ATOMIC_BF16) {
    if (p.dm.K == 128) return gdn2_forward_diag_t<bf16, 128>(p, D, k, b, g, o, h_final, ws);
    return gdn2_forward_diag_t<bf16, 64>(p, D, k, b, g, o, h_final, ws);
  }
  if (p.dm.K == 128) return gdn2_forward_diag_t<float, 128>(p, D, k, b, g, o, h_final, ws);
  return gdn2_forward_diag_t<float, 64>(p, D, k, b, g, o, h_final, ws);
}

template <typename T>
static int gdn2_backward_diag_t(const Gdn2Plan& p, StageDiag& D, const void* dq, const void* dk,
                                const void* dv, const void* dw, const void* db, const float* dg,
                                const float* dh0, void* ws) {
  const Gdn2Grads<T> gr = gdn2_grads<T>(p, ws);
  const size_t N = p.bhn, C = p.dm.C, K = p.dm.K, V = p.dm.V;
  const size_t rows = (size_t)p.dm.B * p.dm.T * p.dm.H;
  int rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DV_NEW, gr.dvn, N * C * V))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DH, gr.dhT, N * V * K))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DAQK, gr.daqk, N * C * C))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DAKK, gr.dakk, N * C * C))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DQ, (const T*)dq, rows * K))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DK, (const T*)dk, rows * K))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DV, (const T*)dv, rows * V))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DW, (const T*)dw, rows * V))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DB, (const T*)db, rows * K))) return rc;
  if ((rc = D.reduce(ATOMIC_GDN2_DIAG_DG, dg, rows * K))) return rc;
  return D.reduce(ATOMIC_GDN2_DIAG_DH0, dh0, (size_t)p.dm.B * p.dm.H * K * V);
}

// ------------------------------------------------ no-allocation forward
// atomic_gdn2_fwd_noalloc runs the forward kernels out of a file-scope device
// array instead of a caller workspace.  Each device the library runs on holds
// its own copy of the array (64 MiB) from module load until the process ends.
// In host code the array's name is only a host-side stand-in: its device
// address is looked up once per device (hipGetSymbolAddress, with that device
// current) and only that address reaches the kernels.
constexpr size_t kNoallocScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kNoallocScratchBytes];

constexpr int kNoallocMaxDevices = 64;
static std::mutex g_noalloc_mu;
static void* g_noalloc_ptr[kNoallocMaxDevices];

// Device address of `scratch` on the current device (looked up on the first
// call on that device).
static int noalloc_scratch(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kNoallocMaxDevices) return ATOMIC_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (!g_noalloc_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr)
      return ATOMIC_ERR_LAUNCH;
    g_noalloc_ptr[dev] = ptr;
  }
  *out = g_noalloc_ptr[dev];
  return ATOMIC_OK;
}

// Plan of one window: batch 1, `nw` chunks, the call's heads and head dims.
static int gdn2_window_plan(const atomic_gdn2_args* a, int nw, Gdn2Plan* p) {
  atomic_gdn2_args w = *a;
  w.batch = 1;
  w.seqlen = nw * kGdn2RunChunk;
  w.chunk = kGdn2RunChunk;
  // every window but a batch row's first starts from a state the loop has
  // already clipped, so sanitising it again changes nothing
  w.flags = a->flags & ATOMIC_GDN2_SANITIZE_H0;
  return gdn2_plan(&w, p);
}

// The forward processes one batch row and a window of chunks at a time: the
// window's per-chunk intermediates fill the scratch after two fp32 state
// slots [H][K][V]; the state leaving a window goes to a slot (alternating,
// so a launch never reads the slot it writes) and enters the next window as
// its h0.  The last window of each batch row writes h_final.  Nothing in the
// scratch is read before the same call writes it.
static int gdn2_forward_noalloc(const atomic_gdn2_args* a, const void* q, const void* k, const void* v,
                                const void* w, const void* b, const float* g, const float* h0, float* o,
                                float* h_final, hipStream_t st) {
  const int NT = a->seqlen / kGdn2RunChunk, H = a->heads, K = a->dk, V = a->dv;
  const size_t es = a->dtype == ATOMIC_BF16 ? 2 : 4;
  const size_t state_elems = (size_t)H * K * V;
  const size_t slot = align256(state_elems * 4);
  if (2 * slot >= kNoallocScratchBytes) return ATOMIC_ERR_SCRATCH;
  const size_t room = kNoallocScratchBytes - 2 * slot;
  // largest window whose intermediates (the blocks before the saved-state
  // ones, which a forward without ATOMIC_GDN2_SAVE never touches) fit
  Gdn2Plan p1;
  int rc = gdn2_window_plan(a, 1, &p1);
  if (rc) return rc;
  if (p1.o_ht > room) return ATOMIC_ERR_SCRATCH;
  int W = (int)(room / p1.o_ht);
  if (W > NT) W = NT;
  Gdn2Plan pfull, ptail;  // full windows, and the shorter last window of a row
  for (;; --W) {
    rc = gdn2_window_plan(a, W, &pfull);
    if (rc) return rc;
    if (pfull.o_ht <= room) break;
  }
  const int tail = NT % W;
  if (tail) {
    rc = gdn2_window_plan(a, tail, &ptail);
    if (rc) return rc;
  }
  void* base = nullptr;
  rc = noalloc_scratch(&base);
  if (rc) return rc;
  float* slots[2] = {reinterpret_cast<float*>(base),
                     reinterpret_cast<float*>(static_cast<char*>(base) + slot)};
  void* ws = static_cast<char*>(base) + 2 * slot;
  Launch L{a->profile, st};
  StageDiag D{a->diag, L};
  if (D && (rc = D.clear(0, ATOMIC_GDN2_DIAG_DV_NEW))) return rc;
  const size_t T = (size_t)a->seqlen, rowV = (size_t)H * V;
  const Gdn2Dims& sd = p1.dm;  // the inputs' row strides
  for (int bb = 0; bb < a->batch; ++bb) {
    const float* hin = h0 ? h0 + (size_t)bb * state_elems : nullptr;
    int wi = 0;
    for (int n0 = 0; n0 < NT; n0 += W, ++wi) {
      const int nw = NT - n0 < W ? NT - n0 : W;
      const Gdn2Plan& pw = nw == W ? pfull : ptail;
      const size_t t0 = (size_t)bb * T + (size_t)n0 * kGdn2RunChunk;  // first row of the window
      const char* qp = static_cast<const char*>(q) + t0 * sd.rq * es;
      const char* kp = static_cast<const char*>(k) + t0 * sd.rk * es;
      const char* bp = static_cast<const char*>(b) + t0 * sd.rb * es;
      const char* vp = static_cast<const char*>(v) + t0 * sd.rv * es;
      const char* wp = static_cast<const char*>(w) + t0 * sd.rw * es;
      const float* gp = g + t0 * sd.rg;
      float* hout = n0 + nw == NT ? h_final + (size_t)bb * state_elems : slots[wi & 1];
      rc = gdn2_forward(pw, a->dtype, qp, kp, vp, wp, bp, gp, hin, o + t0 * rowV, hout, ws, 0, L);
      if (rc) return rc;
      if (D) {  // the reports accumulate over the windows
        rc = gdn2_forward_diag(pw, a->dtype, D, kp, bp, gp, o + t0 * rowV,
                               n0 + nw == NT ? hout : nullptr, ws);
        if (rc) return rc;
      }
      hin = hout;
    }
  }
  return ATOMIC_OK;
}

}  // namespace ah

using namespace ah;

extern "C" size_t atomic_gdn2_workspace_size(const atomic_gdn2_args* a) {
  Gdn2Plan p;
  if (gdn2_plan(a, &p) != ATOMIC_OK) return 0;
  return p.total;
}

extern "C" int atomic_gdn2_workspace_layout(const atomic_gdn2_args* a, atomic_gdn2_layout* out) {
  Gdn2Plan p;
  const int rc = gdn2_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!out) return ATOMIC_ERR_NULL;
  out->qg = p.o_qg; out->kg = p.o_kg; out->w_pseudo = p.o_wt; out->u = p.o_u;
  out->aqk = p.o_aqk; out->ainv = p.o_ainv; out->gc_last = p.o_gcl;
  out->h_pre_t = p.o_ht; out->v_new_t = p.o_vnt; out->total = p.total;
  return ATOMIC_OK;
}

extern "C" int atomic_gdn2_fwd(const atomic_gdn2_args* a, const void* q, const void* k, const void* v,
                               const void* w, const void* b, const float* g, const float* h0,
                               float* o, float* h_final, void* workspace, size_t workspace_bytes,
                               void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!q || !k || !v || !w || !b || !g || !o || !h_final) return ATOMIC_ERR_NULL;
  if (!workspace || workspace_bytes < p.total) return ATOMIC_ERR_WORKSPACE;
  Launch L{a->profile, (hipStream_t)stream};
  const bool save = (a->flags & ATOMIC_GDN2_SAVE) != 0;
  ws_tag_clobber(workspace, p.total);
  int r2 = gdn2_forward(p, a->dtype, q, k, v, w, b, g, h0, o, h_final, workspace, save ? 1 : 0, L);
  if (r2 == ATOMIC_OK && save) ws_tag_set(workspace, p.total, gdn2_tag(a, q, k, v, w, b, g, h0));
  if (r2 || !a->diag) return r2;
  StageDiag D{a->diag, L};
  if ((r2 = D.clear(0, ATOMIC_GDN2_DIAG_DV_NEW))) return r2;
  return gdn2_forward_diag(p, a->dtype, D, k, b, g, o, h_final, workspace);
}

extern "C" int atomic_gdn2_bwd(const atomic_gdn2_args* a, const void* q, const void* k, const void* v,
                               const void* w, const void* b, const float* g, const float* h0,
                               const void* dO, const float* dh_final, void* dq, void* dk, void* dv,
                               void* dw, void* db, float* dg, float* dh0, void* workspace,
                               size_t workspace_bytes, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!q || !k || !v || !w || !b || !g || !dO || !dq || !dk || !dv || !dw || !db || !dg)
    return ATOMIC_ERR_NULL;
  if (!workspace || workspace_bytes < p.total) return ATOMIC_ERR_WORKSPACE;
  const bool reuse = (a->flags & ATOMIC_GDN2_REUSE) != 0;
  const WsTag tag = gdn2_tag(a, q, k, v, w, b, g, h0);
  if (reuse && !ws_tag_matches(workspace, tag)) return ATOMIC_ERR_REUSE;
  Launch L{a->profile, (hipStream_t)stream};
  int r2 = gdn2_backward(p, a->dtype, a->do_dtype, q, k, v, w, b, g, h0, dO, dh_final, dq, dk, dv, dw,
                         db, dg, dh0, workspace, reuse, L);
  // the workspace now holds this forward (recomputed, or kept) and nothing else
  if (r2 == ATOMIC_OK) ws_tag_set(workspace, p.total, tag);
  else ws_tag_clobber(workspace, p.total);
  if (r2 || !a->diag) return r2;
  StageDiag D{a->diag, L};
  if ((r2 = D.clear(ATOMIC_GDN2_DIAG_DV_NEW, ATOMIC_GDN2_DIAG_COUNT - ATOMIC_GDN2_DIAG_DV_NEW))) return r2;
  if (a->dtype == ATOMIC_BF16)
    return gdn2_backward_diag_t<bf16>(p, D, dq, dk, dv, dw, db, dg, dh0, workspace);
  return gdn2_backward_diag_t<float>(p, D, dq, dk, dv, dw, db, dg, dh0, workspace);
}

// ------------------------------------------------ stage-level forward
// The forward's stages over caller-owned per-chunk arrays in the reference's
// layout ([B][H][NT][BT][D], gc_last [B][H][NT][K]): kernels A, B and C alone
// or in one pass, then kernel D.  Two blocks BT (args.chunk):
//   64   the chunk of this library's kernels, arrays in args.dtype (gc_last
//        and the outputs fp32);
//   256  the reference's Pallas block (kernel_a_scores.py:15-17), float32
//        arrays, by the kernels of stage256.hip (the one-pass A + B + C entry
//        takes 64 only).
static int gdn2_stage_plan(const atomic_gdn2_args* a, Gdn2Plan* p) {
  const int rc = gdn2_plan(a, p);
  if (rc != ATOMIC_OK) return rc;
  return a->chunk == kGdn2RunChunk || a->chunk == kStageBlock ? ATOMIC_OK : ATOMIC_ERR_SHAPE;
}

// The plan's dims over blocks of kStageBlock rows.
static Gdn2Dims gdn2_dims256(const Gdn2Plan& p) {
  Gdn2Dims d = p.dm;
  d.C = kStageBlock;
  d.NT = d.T / kStageBlock;
  return d;
}

template <typename T>
static Gdn2Chunks<T> gdn2_stage_chunks(void* aqk, void* ainv, void* wt, void* u, void* kg, void* qg, float* gcl,
                                       void* akk = nullptr) {
  Gdn2Chunks<T> c;
  c.akk = (T*)akk;
  c.qg = (T*)qg;
  c.kg = (T*)kg;
  c.wt = (T*)wt;
  c.u = (T*)u;
  c.aqk = (T*)aqk;
  c.ainv = (T*)ainv;
  c.gcl = gcl;
  c.hT = nullptr;
  c.vnT = nullptr;
  return c;
}

extern "C" int atomic_gdn2_chunk_wy(const atomic_gdn2_args* a, const void* q, const void* k, const void* v,
                                    const void* w, const void* b, const float* g, void* Aqk, void* A,
                                    void* w_pseudo, void* u, void* kg, void* qg, float* gc_last, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!q || !k || !v || !w || !b || !g || !Aqk || !A || !w_pseudo || !u || !kg || !qg || !gc_last)
    return ATOMIC_ERR_NULL;
  if (a->chunk != kGdn2RunChunk) return ATOMIC_ERR_SHAPE;  // Akk would need caller memory at 256
  Launch L{a->profile, (hipStream_t)stream};
  if (a->dtype == ATOMIC_BF16) {
    const Gdn2Chunks<bf16> ck = gdn2_stage_chunks<bf16>(Aqk, A, w_pseudo, u, kg, qg, gc_last);
    return p.dm.K == 128 ? gdn2_intra_launch<bf16, 128>(p, q, k, v, w, b, g, ck, L)
                         : gdn2_intra_launch<bf16, 64>(p, q, k, v, w, b, g, ck, L);
  }
  const Gdn2Chunks<float> ck = gdn2_stage_chunks<float>(Aqk, A, w_pseudo, u, kg, qg, gc_last);
  return p.dm.K == 128 ? gdn2_intra_launch<float, 128>(p, q, k, v, w, b, g, ck, L)
                       : gdn2_intra_launch<float, 64>(p, q, k, v, w, b, g, ck, L);
}

// One of kernels A, B, C alone (ST), bf16 or fp32, K = 64 or 128.
template <int ST>
static int gdn2_stage_launch(const atomic_gdn2_args* a, const Gdn2Plan& p, const void* q, const void* k,
                             const void* v, const void* w, const void* b, const float* g, void* aqk, void* akk,
                             void* ainv, void* wt, void* u, void* kg, void* qg, float* gcl, void* stream) {
  Launch L{a->profile, (hipStream_t)stream};
  if (a->dtype == ATOMIC_BF16) {
    const Gdn2Chunks<bf16> ck = gdn2_stage_chunks<bf16>(aqk, ainv, wt, u, kg, qg, gcl, akk);
    return p.dm.K == 128 ? gdn2_intra_launch<bf16, 128, ST>(p, q, k, v, w, b, g, ck, L)
                         : gdn2_intra_launch<bf16, 64, ST>(p, q, k, v, w, b, g, ck, L);
  }
  const Gdn2Chunks<float> ck = gdn2_stage_chunks<float>(aqk, ainv, wt, u, kg, qg, gcl, akk);
  return p.dm.K == 128 ? gdn2_intra_launch<float, 128, ST>(p, q, k, v, w, b, g, ck, L)
                       : gdn2_intra_launch<float, 64, ST>(p, q, k, v, w, b, g, ck, L);
}

extern "C" int atomic_gdn2_chunk_scores(const atomic_gdn2_args* a, const void* q, const void* k, const void* b,
                                        const float* g, void* Aqk, void* Akk, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!q || !k || !b || !g || !Aqk || !Akk) return ATOMIC_ERR_NULL;
  if (a->chunk == kStageBlock) {
    Launch L{a->profile, (hipStream_t)stream};
    return g256_scores(gdn2_dims256(p), a->dtype, q, k, b, g, (float*)Aqk, (float*)Akk, L);
  }
  return gdn2_stage_launch<kIntraScores>(a, p, q, k, nullptr, nullptr, b, g, Aqk, Akk, nullptr, nullptr, nullptr,
                                         nullptr, nullptr, nullptr, stream);
}

extern "C" int atomic_gdn2_wy_solve(const atomic_gdn2_args* a, const void* Akk, void* A, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!Akk || !A) return ATOMIC_ERR_NULL;
  if (a->chunk == kStageBlock) {
    Launch L{a->profile, (hipStream_t)stream};
    return g256_solve(gdn2_dims256(p), (const float*)Akk, (float*)A, L);
  }
  return gdn2_stage_launch<kIntraSolve>(a, p, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                                        const_cast<void*>(Akk), A, nullptr, nullptr, nullptr, nullptr, nullptr,
                                        stream);
}

extern "C" int atomic_gdn2_recompute_wy(const atomic_gdn2_args* a, const void* q, const void* k, const void* v,
                                        const void* w, const void* b, const float* g, const void* A,
                                        void* w_pseudo, void* u, void* kg, void* qg, float* gc_last, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!q || !k || !v || !w || !b || !g || !A || !w_pseudo || !u || !kg || !qg || !gc_last) return ATOMIC_ERR_NULL;
  if (a->chunk == kStageBlock) {
    Launch L{a->profile, (hipStream_t)stream};
    return g256_recompute(gdn2_dims256(p), a->dtype, q, k, v, w, b, g, (const float*)A, (float*)w_pseudo,
                          (float*)u, (float*)kg, (float*)qg, gc_last, L);
  }
  return gdn2_stage_launch<kIntraRecompute>(a, p, q, k, v, w, b, g, nullptr, nullptr, const_cast<void*>(A),
                                            w_pseudo, u, kg, qg, gc_last, stream);
}

extern "C" int atomic_gdn2_inter_chunk_combine(const atomic_gdn2_args* a, const void* Aqk, const void* w_pseudo,
                                               const void* u, const void* kg, const void* qg,
                                               const float* gc_last, const float* h0, float* o, float* h_final,
                                               void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!Aqk || !w_pseudo || !u || !kg || !qg || !gc_last || !o || !h_final) return ATOMIC_ERR_NULL;
  Launch L{a->profile, (hipStream_t)stream};
  if (a->chunk == kStageBlock)
    return g256_combine(gdn2_dims256(p), (const float*)Aqk, (const float*)w_pseudo, (const float*)u,
                        (const float*)kg, (const float*)qg, gc_last, h0, o, h_final, nullptr, nullptr, L);
  const int mode = kStateChunkO | kStateSanitizeH0;
  void* aq = const_cast<void*>(Aqk);
  void* wt = const_cast<void*>(w_pseudo);
  void* uu = const_cast<void*>(u);
  void* kk = const_cast<void*>(kg);
  void* qq = const_cast<void*>(qg);
  float* gl = const_cast<float*>(gc_last);
  if (a->dtype == ATOMIC_BF16) {
    const Gdn2Chunks<bf16> ck = gdn2_stage_chunks<bf16>(aq, nullptr, wt, uu, kk, qq, gl);
    return p.dm.K == 128 ? gdn2_state_launch<bf16, 128>(p, ck, h0, o, h_final, mode, L)
                         : gdn2_state_launch<bf16, 64>(p, ck, h0, o, h_final, mode, L);
  }
  const Gdn2Chunks<float> ck = gdn2_stage_chunks<float>(aq, nullptr, wt, uu, kk, qq, gl);
  return p.dm.K == 128 ? gdn2_state_launch<float, 128>(p, ck, h0, o, h_final, mode, L)
                       : gdn2_state_launch<float, 64>(p, ck, h0, o, h_final, mode, L);
}

extern "C" int atomic_gdn2_inter_chunk_combine_with_state(const atomic_gdn2_args* a, const void* Aqk,
                                                          const void* w_pseudo, const void* u, const void* kg,
                                                          const void* qg, const float* gc_last, const float* h0,
                                                          float* o, float* h_final, void* h_pre_t, void* v_new_t,
                                                          void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!Aqk || !w_pseudo || !u || !kg || !qg || !gc_last || !o || !h_final || !h_pre_t || !v_new_t)
    return ATOMIC_ERR_NULL;
  Launch L{a->profile, (hipStream_t)stream};
  if (a->chunk == kStageBlock)  // fp32, not transposed: h_pre [B][H][NT][K][V], v_new [B][H][NT][256][V]
    return g256_combine(gdn2_dims256(p), (const float*)Aqk, (const float*)w_pseudo, (const float*)u,
                        (const float*)kg, (const float*)qg, gc_last, h0, o, h_final, (float*)h_pre_t,
                        (float*)v_new_t, L);
  const int mode = kStateSave | kStateChunkO | kStateSanitizeH0;
  void* aq = const_cast<void*>(Aqk);
  void* wt = const_cast<void*>(w_pseudo);
  void* uu = const_cast<void*>(u);
  void* kk = const_cast<void*>(kg);
  void* qq = const_cast<void*>(qg);
  float* gl = const_cast<float*>(gc_last);
  if (a->dtype == ATOMIC_BF16) {
    Gdn2Chunks<bf16> ck = gdn2_stage_chunks<bf16>(aq, nullptr, wt, uu, kk, qq, gl);
    ck.hT = static_cast<bf16*>(h_pre_t);
    ck.vnT = static_cast<bf16*>(v_new_t);
    return p.dm.K == 128 ? gdn2_state_launch<bf16, 128>(p, ck, h0, o, h_final, mode, L)
                         : gdn2_state_launch<bf16, 64>(p, ck, h0, o, h_final, mode, L);
  }
  Gdn2Chunks<float> ck = gdn2_stage_chunks<float>(aq, nullptr, wt, uu, kk, qq, gl);
  ck.hT = static_cast<float*>(h_pre_t);
  ck.vnT = static_cast<float*>(v_new_t);
  return p.dm.K == 128 ? gdn2_state_launch<float, 128>(p, ck, h0, o, h_final, mode, L)
                       : gdn2_state_launch<float, 64>(p, ck, h0, o, h_final, mode, L);
}

extern "C" int atomic_gdn2_fwd_noalloc(const atomic_gdn2_args* a, const void* q, const void* k,
                                       const void* v, const void* w, const void* b, const float* g,
                                       const float* h0, float* o, float* h_final, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  // the shared scratch cannot keep intermediates for a later backward
  if (a->flags & (ATOMIC_GDN2_SAVE | ATOMIC_GDN2_REUSE)) return ATOMIC_ERR_SCRATCH;
  if (!q || !k || !v || !w || !b || !g || !o || !h_final) return ATOMIC_ERR_NULL;
  return gdn2_forward_noalloc(a, q, k, v, w, b, g, h0, o, h_final, (hipStream_t)stream);
}

// ------------------------------------------------------------------ backward stages (256-row blocks)
// The staged backward of kernel_trainable_B6.py:97-181 at the reference's
// block: chunk must be 256; every per-block array is float32.

static int gdn2_bwd_stage_plan(const atomic_gdn2_args* a, Gdn2Plan* p) {
  const int rc = gdn2_stage_plan(a, p);
  if (rc != ATOMIC_OK) return rc;
  return a->chunk == kStageBlock ? ATOMIC_OK : ATOMIC_ERR_SHAPE;
}

extern "C" int atomic_gdn2_dav_backward(const atomic_gdn2_args* a, const float* Aqk, const float* v_new,
                                        const void* dO, float* dAqk, float* dv_new, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_bwd_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!Aqk || !v_new || !dO || !dAqk || !dv_new) return ATOMIC_ERR_NULL;
  Launch L{a->profile, (hipStream_t)stream};
  return g256_dav_bwd(gdn2_dims256(p), a->do_dtype, Aqk, v_new, dO, dAqk, dv_new, L);
}

extern "C" int atomic_gdn2_dhu_backward(const atomic_gdn2_args* a, const void* dO, const float* dv_partial,
                                        const float* w_pseudo, const float* qg, const float* kg,
                                        const float* gc_last, const float* dht, float* dh_all, float* dh0,
                                        float* dv_all, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_bwd_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!dO || !dv_partial || !w_pseudo || !qg || !kg || !gc_last || !dh_all || !dh0 || !dv_all)
    return ATOMIC_ERR_NULL;
  Launch L{a->profile, (hipStream_t)stream};
  return g256_dhu_bwd(gdn2_dims256(p), a->do_dtype, dO, dv_partial, w_pseudo, qg, kg, gc_last, dht, dh_all, dh0,
                      dv_all, L);
}

extern "C" size_t atomic_gdn2_wy_dqkg_workspace_size(const atomic_gdn2_args* a) {
  Gdn2Plan p;
  if (gdn2_bwd_stage_plan(a, &p) != ATOMIC_OK) return 0;
  return g256_b3_ws(gdn2_dims256(p));
}

extern "C" int atomic_gdn2_wy_dqkg_backward(const atomic_gdn2_args* a, const void* q, const void* k, const void* b,
                                            const void* w, const void* v, const float* gc, const float* A,
                                            const float* h_pre, const float* v_new, const void* dO,
                                            const float* dv, const float* dh_next, float* dq, float* dk, float* db,
                                            float* dw, float* dv_raw, float* dgc, float* dAkk, void* workspace,
                                            size_t workspace_bytes, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_bwd_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!q || !k || !b || !w || !v || !gc || !A || !h_pre || !v_new || !dO || !dv || !dh_next || !dq || !dk || !db ||
      !dw || !dv_raw || !dgc || !dAkk)
    return ATOMIC_ERR_NULL;
  const Gdn2Dims d = gdn2_dims256(p);
  if (!workspace || workspace_bytes < g256_b3_ws(d)) return ATOMIC_ERR_WORKSPACE;
  Launch L{a->profile, (hipStream_t)stream};
  return g256_b3_bwd(d, a->dtype, a->do_dtype, q, k, b, w, v, gc, A, h_pre, v_new, dO, dv, dh_next, dq, dk, db, dw,
                     dv_raw, dgc, dAkk, static_cast<float*>(workspace), L);
}

extern "C" int atomic_gdn2_intra_backward(const atomic_gdn2_args* a, const float* dAqk, const float* dAkk,
                                          const void* q, const void* k, const void* b, const float* g, float* dq,
                                          float* dk, float* db, float* dgc, void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_bwd_stage_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!dAqk || !dAkk || !q || !k || !b || !g || !dq || !dk || !db || !dgc) return ATOMIC_ERR_NULL;
  Launch L{a->profile, (hipStream_t)stream};
  return g256_intra_bwd(gdn2_dims256(p), a->dtype, dAqk, dAkk, q, k, b, g, dq, dk, db, dgc, L);
}

extern "C" int atomic_gdn2_reverse_cumsum_bwd(const atomic_gdn2_args* a, const float* dgc, float* dg,
                                              void* stream) {
  Gdn2Plan p;
  const int rc = gdn2_plan(a, &p);
  if (rc != ATOMIC_OK) return rc;
  if (!dgc || !dg) return ATOMIC_ERR_NULL;
  Launch L{a->profile, (hipStream_t)stream};
  const long long blocks = (long long)a->batch * a->heads * (a->seqlen / a->chunk);
  return rev_cumsum_bwd(dgc, dg, blocks, a->chunk, a->dk, L);
}
