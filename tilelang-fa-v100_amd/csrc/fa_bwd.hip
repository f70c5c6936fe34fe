// Dense attention backward for gfx950 (FlashAttention-2, LSE recompute).
//
// Replaces tilelang_backward (tilelang_fa_v100/_kernels_backward.py:200-208):
// the PyTorch row_dot (:203), the dQ kernel (:10-85) and the dK/dV kernel
// (:88-176).  The reference recomputes QK^T and dO V^T in both kernels (7
// GEMMs per tile pair); here one KV-stationary kernel does the 5 GEMMs
//   S = Q K^T,  dP = dO V^T,  dV += P^T dO,  dK += dS^T Q,  dQ += dS K
// with P = exp(scale*S - lse), dS = P * (dP - rowdot(O, dO)) * scale
// (_kernels_backward.py:72-74,159-170).  dQ comes from a query-stationary
// kernel (fa_bwd_dq.h) that recomputes S and dP per query tile and builds
// each dQ row in one wave, like the reference's dQ kernel: no atomics, so
// dq, dk and dv repeat bit for bit (fp32 atomics into a dQ accumulator were
// measured slower at every head_dim: they are performed beyond the XCD's L2
// on this part).
//
// Kernels, in launch order:
//   bwd_dq_kernel       dQ (fa_bwd_dq.h); also writes the row statistics
//                       scale·rowdot(O, dO) and LSE*log2(e) of the rows it
//                       owns into one array [B*H][2][Sq] (LSE*log2(e)
//                       first, scale·rowdot second), so a lane of the dK / dV
//                       kernels addresses either with a 32-bit offset from a
//                       per-head base.
// Every kernel forms dS already multiplied by softmax_scale and rounds that
// to 16 bits before its products, as the reference does
// (_kernels_backward.py:74,160), so dS has fp16's full range.
//   bwd_main_mfma_kernel  dK / dV (fa_bwd_mfma.h); for small grids as several
//                       pieces per key tile, summed by bwd_reduce_kernel.
// At head_dim 128 / 256 with a workspace of bwd_workspace_bytes (causal or full
// attention) or bwd_preferred_workspace_bytes (window bands too), the order is
// instead bwd_stats_kernel (the row
// statistics), bwd_main_mfma_kernel<..., DS = true> (dK / dV, storing its dS
// tiles) and bwd_dq_ds_kernel (dQ = dS K from them), fa_bwd_ds.h.
#include "fa_bwd_dq.h"
#include "fa_bwd_ds.h"
#include "fa_bwd_mfma.h"
#include "fa_common.h"
#include "fa_internal.h"

namespace fa {

// ----------------------------------------------------------------- launchers

// Workspace: the row statistics [B*H][2][Sq] (LSE*log2(e), scale·rowdot), then,
// for the dS-store path, the dS tiles (fa_bwd_ds.h) from byte ds_offset(a).
static size_t stats_bytes(const fa_bwd_args& a) {
  const size_t rows = (size_t)a.batch * a.seqlen_q * a.num_heads;
  return 2 * rows * sizeof(float) + 256;
}
static size_t ds_offset(const fa_bwd_args& a) { return (stats_bytes(a) + 255) & ~(size_t)255; }

// Bytes of dS tiles for the dS-store path, or 0 where it does not apply:
// head_dim 128 / 256, below tiles::kBwdDsMaxBytes.
template <int MODE>
static size_t ds_bytes_of(const fa_bwd_args& a) {
  if ((a.head_dim != 128 && a.head_dim != 256) || a.seqlen_q <= 0 || a.seqlen_k <= 0) return 0;
  const Band band = make_band(a);
  const DsTiles<MODE> L = ds_tiles<MODE>(a.seqlen_q, a.seqlen_k, band.wl, band.wr);
  const size_t bytes = 2048 * (size_t)a.batch * a.num_heads * (size_t)L.per_head();
  // Strictly below the cap: a wave's dS reads go through one buffer resource
  // of count(qt) * 2 KB bytes (a 32-bit size), and count(qt) <= per_head.
  return bytes < tiles::kBwdDsMaxBytes ? bytes : 0;
}
// Causal and full attention: part of bwd_workspace_bytes.
static size_t ds_bytes(const fa_bwd_args& a) {
  const int mode = mask_mode(a);
  return mode == kMaskCausal ? ds_bytes_of<kMaskCausal>(a)
                             : (mode == kMaskNone ? ds_bytes_of<kMaskNone>(a) : 0);
}
// Window bands: part of bwd_preferred_workspace_bytes only.
static size_t band_ds_bytes(const fa_bwd_args& a) {
  return mask_mode(a) == kMaskBand && (int64_t)a.seqlen_q + a.seqlen_k < (1 << 29)
             ? ds_bytes_of<kMaskBand>(a)
             : 0;
}

size_t bwd_min_workspace_bytes(const fa_bwd_args& a) { return stats_bytes(a); }

size_t bwd_workspace_bytes(const fa_bwd_args& a) {
  const size_t ds = ds_bytes(a);
  return ds ? ds_offset(a) + ds : stats_bytes(a);
}

// Keys per workgroup of the dK / dV kernel, workgroups resident per CU, and
// the measured time of one 32-row query tile and of a workgroup's start and
// end (us, chip full), for the split rule below.
struct BwdMainCost {
  int bkv, per_cu;
  float tile_us, fixed_us;
};
static BwdMainCost bwd_main_cost(int head_dim) {
  switch (head_dim) {
    case 64: return {BwdShapeMfma<64>::BKV, tiles::kBwd64WavesPerSimd, 1.0f, 5.f};
    case 128: return {BwdShapeMfma<128>::BKV, 1, 2.0f, 6.f};
    default: return {BwdShapeMfma<256>::BKV, 1, 2.3f, 6.f};
  }
}

// Pieces the query tiles of every dK / dV workgroup are cut into.  One
// workgroup per (key tile, KV head) leaves CUs idle for small batches and few
// KV heads, and a causal problem ends with its longest workgroup; pieces cost
// fp32 partials written and read once.  The count is the one whose estimated
// time (rounds of equal pieces for full attention; the larger of the longest
// piece and the mean load for causal, whose pieces go out longest first) is
// smallest, no piece shorter than kBwdPieceTiles query tiles.  A window band
// is not split.
static int bwd_pieces(const fa_bwd_args& a) {
  const int mode = mask_mode(a);
  if (mode == kMaskBand || a.seqlen_q <= 0 || a.seqlen_k <= 0) return 1;
  if (a.head_dim != 64 && ds_bytes(a) == 0) return 1;
  const BwdMainCost c = bwd_main_cost(a.head_dim);
  const int64_t kvtiles = (a.seqlen_k + (int64_t)c.bkv - 1) / c.bkv;
  const int64_t heads = (int64_t)a.batch * a.num_heads_k, wgs = kvtiles * heads;
  const int64_t slots = (int64_t)device_cu_count() * c.per_cu;
  if (wgs >= 2 * slots) return 1;
  const int G = a.num_heads / a.num_heads_k;
  const int64_t nq = ((int64_t)a.seqlen_q + tiles::kBwdQueryRows - 1) / tiles::kBwdQueryRows;
  int64_t sum = 0, most = 0;  // query tiles of one KV head's workgroups
  for (int64_t t = 0; t < kvtiles; ++t) {
    int64_t first = 0;
    if (mode == kMaskCausal)
      first = std::max<int64_t>(0, t * c.bkv - ((int64_t)a.seqlen_k - a.seqlen_q)) /
              tiles::kBwdQueryRows;
    const int64_t n = G * std::max<int64_t>(0, nq - first);
    sum += n;
    most = std::max(most, n);
  }
  const double blocks = (double)wgs * c.bkv * a.head_dim * 8;  // bytes of one fp32 dK / dV
  double best = 0;
  int pieces = 1;
  for (int ns = 1; ns <= tiles::kBwdMaxPieces && (ns == 1 || most >= ns * tiles::kBwdPieceTiles);
       ++ns) {
    const double longest = (double)most / ns * c.tile_us + c.fixed_us;
    const double mean = ((double)sum * heads * c.tile_us + (double)wgs * ns * c.fixed_us) / slots;
    const double rounds = (double)((wgs * ns + slots - 1) / slots);
    double t = mode == kMaskCausal ? std::max(longest, mean + 0.25 * longest) : rounds * longest;
    if (ns > 1) t += 6.0 + 2.0 * ns * blocks / 4.0e6;  // us: launch, bytes at 4 TB/s
    if (ns == 1 || t < 0.97 * best) {
      best = t;
      pieces = ns;
    }
  }
  return pieces;
}

static size_t part_bytes(const fa_bwd_args& a, int pieces) {
  const BwdMainCost c = bwd_main_cost(a.head_dim);
  const size_t kvtiles = ((size_t)a.seqlen_k + c.bkv - 1) / c.bkv;
  return (size_t)pieces * a.batch * a.num_heads_k * kvtiles * c.bkv * a.head_dim * 8;
}
static size_t part_offset(const fa_bwd_args& a) { return (bwd_workspace_bytes(a) + 255) & ~(size_t)255; }

size_t bwd_preferred_workspace_bytes(const fa_bwd_args& a) {
  if (const size_t ds = band_ds_bytes(a)) return ds_offset(a) + ds;
  const int pieces = bwd_pieces(a);
  return pieces > 1 ? part_offset(a) + part_bytes(a, pieces) : bwd_workspace_bytes(a);
}

// Key-stationary dK / dV kernel for one mask mode; with ds, also stores the
// dS tiles (head_dim 128 / 256); with pieces > 1 (causal or full attention; at
// head_dim 128 / 256 only with ds), as that many pieces per workgroup whose sums
// land in `part`, then their reduction.
template <class T, int D, int MODE, bool DS, bool SPLIT>
static void launch_main(const fa_bwd_args& a, const float* stats, uint16_t* ds, float* part,
                        int pieces, hipStream_t st) {
  using S = BwdShapeMfma<D>;
  const int kvtiles = (a.seqlen_k + S::BKV - 1) / S::BKV;
  const unsigned wgs = (unsigned)kvtiles * a.num_heads_k * a.batch;
  hipLaunchKernelGGL((bwd_main_mfma_kernel<T, D, MODE, DS, SPLIT>), dim3(wgs * pieces),
                     dim3(64 * S::NW), 0, st, a, stats, ds, part, pieces);
  if constexpr (SPLIT) {
    const int nblk = kvtiles * S::NW;
    const int64_t items = (int64_t)a.batch * a.num_heads_k * nblk * 2 * (D / 32);
    hipLaunchKernelGGL((bwd_reduce_kernel<T, D>), dim3((unsigned)((items + 3) / 4)), dim3(256), 0,
                       st, a, part, pieces, nblk);
  }
}
template <class T, int D, int MODE>
static void launch_bwd_main(const fa_bwd_args& a, const float* stats, uint16_t* ds, float* part,
                            int pieces, hipStream_t st) {
  if (a.seqlen_k == 0) return;  // no keys: dK / dV are empty
  constexpr bool kDs = D >= 128;
  constexpr bool kSplit = MODE != kMaskBand;
  if constexpr (kDs) {
    if constexpr (kSplit)
      if (ds && pieces > 1)
        return launch_main<T, D, MODE, true, true>(a, stats, ds, part, pieces, st);
    if (ds) return launch_main<T, D, MODE, true, false>(a, stats, ds, nullptr, 1, st);
  } else if constexpr (kSplit) {
    if (pieces > 1) return launch_main<T, D, MODE, false, true>(a, stats, nullptr, part, pieces, st);
  }
  launch_main<T, D, MODE, false, false>(a, stats, nullptr, nullptr, 1, st);
}
template <class T, int D>
static void launch_bwd_main(const fa_bwd_args& a, int mode, const float* stats, uint16_t* ds,
                            float* part, int pieces, hipStream_t st) {
  if (mode == kMaskCausal)
    launch_bwd_main<T, D, kMaskCausal>(a, stats, ds, part, pieces, st);
  else if (mode == kMaskBand)
    launch_bwd_main<T, D, kMaskBand>(a, stats, ds, part, pieces, st);
  else
    launch_bwd_main<T, D, kMaskNone>(a, stats, ds, part, pieces, st);
}

// Query-stationary dQ kernel (also writes the row statistics).
template <class T, int D>
static void launch_bwd_dq(const fa_bwd_args& a, int mode, float* stats, hipStream_t st) {
  using S = BwdDqShape<D>;
  const int qtiles = (a.seqlen_q + S::BM - 1) / S::BM;
  const dim3 grid((unsigned)qtiles * a.num_heads * a.batch), block(64 * S::NW);
  if (mode == kMaskCausal)
    hipLaunchKernelGGL((bwd_dq_kernel<T, D, kMaskCausal>), grid, block, 0, st, a, stats);
  else if (mode == kMaskBand)
    hipLaunchKernelGGL((bwd_dq_kernel<T, D, kMaskBand>), grid, block, 0, st, a, stats);
  else
    hipLaunchKernelGGL((bwd_dq_kernel<T, D, kMaskNone>), grid, block, 0, st, a, stats);
}

// Waves per workgroup of the dQ-from-dS kernel.  Eight waves share each K tile
// (half the K traffic of four), but with at most one 8-wave workgroup per CU a
// causal problem runs as long as its longest one, and below half that a CU
// has waves to spare: four then, twice as many workgroups (two fit a CU at
// head_dim 128, one at 256).
// Measured (fa_bwd per call, us, 8 / 4 waves, same box; 8-wave workgroups in
// brackets): causal [2, 4096, 8, 256] 455 / 431 (256), [1, 2048, 16, 256] 198 /
// 180 (128), [1, 2048, 8, 128] 97 / 87 (64), [2, 2048, 16, 128] 173 / 170 (256),
// [2, 2000, 32/8, 128] 264 / 267 (512), [2, 8192, 8, 256] 1519 / 1557 (512);
// full [1, 4096, 8, 256] 423 / 399 (128), [1, 4096, 16, 128] 393 / 405 (256).
static int dq_ds_waves(const fa_bwd_args& a, int mode) {
  const int64_t wgs8 =
      ((int64_t)a.seqlen_q + 255) / 256 * a.num_heads * (int64_t)a.batch;
  const int cus = device_cu_count();
  return wgs8 <= (mode == kMaskCausal ? cus : cus / 2) ? 4 : 8;
}
template <class T, int D, int MODE, int NW>
static void launch_dq_ds(const fa_bwd_args& a, const uint16_t* ds, hipStream_t st) {
  const int nqb = ((a.seqlen_q + 31) / 32 + NW - 1) / NW;
  hipLaunchKernelGGL((bwd_dq_ds_kernel<T, D, MODE, NW>),
                     dim3((unsigned)nqb * a.num_heads * a.batch), dim3(64 * NW), 0, st, a, ds);
}

// dS-store path (head_dim 128 / 256): row statistics, dK / dV storing dS,
// then dQ = dS K (dS includes the scale).
template <class T, int D>
static hipError_t launch_bwd_ds(const fa_bwd_args& a, int mode, void* ws, float* part, int pieces,
                                hipStream_t st) {
  float* stats = static_cast<float*>(ws);
  uint16_t* ds = reinterpret_cast<uint16_t*>(static_cast<char*>(ws) + ds_offset(a));
  const int64_t blocks = (int64_t)a.batch * a.num_heads * ((a.seqlen_q + 31) / 32);
  constexpr int per_wg = 4 * StatsShape<D>::kTiles;  // 32-row blocks per workgroup
  hipLaunchKernelGGL((bwd_stats_kernel<T, D>), dim3((unsigned)((blocks + per_wg - 1) / per_wg)),
                     dim3(256), 0, st, a, stats);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  launch_bwd_main<T, D>(a, mode, stats, ds, part, pieces, st);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  const bool four = dq_ds_waves(a, mode) == 4;
  if (mode == kMaskBand)
    four ? launch_dq_ds<T, D, kMaskBand, 4>(a, ds, st) : launch_dq_ds<T, D, kMaskBand, 8>(a, ds, st);
  else if (mode == kMaskCausal)
    four ? launch_dq_ds<T, D, kMaskCausal, 4>(a, ds, st) : launch_dq_ds<T, D, kMaskCausal, 8>(a, ds, st);
  else
    four ? launch_dq_ds<T, D, kMaskNone, 4>(a, ds, st) : launch_dq_ds<T, D, kMaskNone, 8>(a, ds, st);
  return hipGetLastError();
}

// dQ (and the row statistics), then dK / dV.  Every output element is
// produced by one fixed sequence of operations.  A workspace of
// bwd_workspace_bytes selects the dS-store path where it applies; one of
// bwd_min_workspace_bytes, the recompute path; one of
// bwd_preferred_workspace_bytes also the dK / dV kernel in pieces.
template <class T, int D>
static hipError_t launch_bwd_d(const fa_bwd_args& a, void* ws, size_t ws_bytes, hipStream_t st) {
  const int mode = mask_mode(a);
  int pieces = bwd_pieces(a);
  if (pieces > 1 && ws_bytes < part_offset(a) + part_bytes(a, pieces)) pieces = 1;
  float* part = pieces > 1
                    ? reinterpret_cast<float*>(static_cast<char*>(ws) + part_offset(a))
                    : nullptr;
  if constexpr (D >= 128) {
    const size_t band_ds = band_ds_bytes(a);
    if (band_ds ? ws_bytes >= ds_offset(a) + band_ds
                : ds_bytes(a) && ws_bytes >= bwd_workspace_bytes(a))
      return launch_bwd_ds<T, D>(a, mode, ws, part, pieces, st);
  }
  float* stats = static_cast<float*>(ws);  // [B*H][2][Sq]
  launch_bwd_dq<T, D>(a, mode, stats, st);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  launch_bwd_main<T, D>(a, mode, stats, nullptr, part, pieces, st);
  return hipGetLastError();
}

template <class T>
static hipError_t launch_bwd_t(const fa_bwd_args& a, void* ws, size_t ws_bytes, hipStream_t st) {
  switch (a.head_dim) {
    case 64: return launch_bwd_d<T, 64>(a, ws, ws_bytes, st);
    case 128: return launch_bwd_d<T, 128>(a, ws, ws_bytes, st);
    case 256: return launch_bwd_d<T, 256>(a, ws, ws_bytes, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_bwd(const fa_bwd_args& a, void* ws, size_t ws_bytes, hipStream_t st) {
  return a.dtype == FA_DTYPE_BF16 ? launch_bwd_t<BFloat16>(a, ws, ws_bytes, st)
                                  : launch_bwd_t<Half>(a, ws, ws_bytes, st);
}

}  // namespace fa
