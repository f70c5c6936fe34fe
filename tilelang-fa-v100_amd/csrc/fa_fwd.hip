// Dense and paged (vLLM) attention forward kernels for gfx950.
//
// Dense:  replaces _forward_lse_kernel_func (tilelang_fa_v100/
//         _kernels_forward.py:94-172).  q/k/v/out are read and written in the
//         caller's [B, S, H, D] layout through strides, so the four layout
//         copies of interface.py:19-21,38 disappear.
// Paged:  replaces _paged_kernel_func (_kernels_paged.py:193-344).  The
//         grid is sized by total query rows, not rows x batch
//         (_paged_adapter.py:44), and each workgroup finds its sequence with a
//         scan over query_start_loc.  The Hq/Hkv query heads that share a KV
//         head are packed into one row space (row = token * G + g), so every
//         K/V tile fetched from the cache serves the whole GQA group.
#include <algorithm>

#include "fa_fwd_core.h"
#include "fa_fwd_d128.h"
#include "fa_fwd_1w.h"
#include "fa_fwd_split.h"
#include "fa_internal.h"

namespace fa {

struct DenseRows {
  const uint16_t* q;
  uint16_t* o;
  float* lse;
  const uint16_t* k;
  const uint16_t* v;
  int64_t qs, os, ks, vs;  // per-row (sequence) strides, elements
  int nrows, sk, off;      // off = seqlen_k - seqlen_q
  int wl, wr;              // window bounds (-1: unbounded); causal is wr = 0
  bool has_lse;
  // K / V rows are a base plus a row stride (below 2^24 elements, checked
  // by the launcher), so whole tiles can be DMA'd through buffer resources.
  static constexpr bool kF32Out = false;
  static constexpr bool kRowStrided = true;  // k_ptr(n + m) = k_ptr(n) + m * ks

  // Row r sees keys [r + off - wl, r + off + wr] within [0, sk).
  __device__ int kv_lo(int r) const { return wl >= 0 ? min(max(r + off - wl, 0), sk) : 0; }
  __device__ int kv_hi(int r) const {
    return wr >= 0 ? min(max(r + off + wr + 1, 0), sk) : sk;
  }
  __device__ const uint16_t* q_ptr(int r) const { return q + r * qs; }
  __device__ uint16_t* o_ptr(int r) const { return o + r * os; }
  __device__ float* lse_ptr(int r) const { return lse + r; }
  __device__ const uint16_t* k_ptr(int n) const { return k + n * ks; }
  __device__ const uint16_t* v_ptr(int n) const { return v + n * vs; }
  __device__ int64_t k_row_stride() const { return ks; }
  __device__ int64_t v_row_stride() const { return vs; }
};

// Tile geometry per head_dim and core: D = 128 (both schedules) uses the
// direct-to-LDS 8-wave cores, D = 256 with PP the direct-to-LDS one-pass
// 4-wave core, the rest the register-staged 4-wave core.
template <int D, bool PP>
struct FwdKernelCfg {
  static constexpr int BM = FwdShape<D>::BM;
  static constexpr int THREADS = 256;
  static constexpr int WAVES_PER_EU = FwdShape<D>::kWavesPerEU;
  static constexpr int WG_PER_CU = WAVES_PER_EU;  // 4 waves: one per SIMD each
  static constexpr int LDS_BYTES = FwdShape<D>::LDS_ELEMS * 2;
};
// One-wave-per-SIMD cores (fa_fwd_1w.h).
template <int D, int RB>
struct FwdKernelCfg1W {
  using S = FwdShape1W<D, RB>;
  static constexpr int BM = S::BM;
  static constexpr int THREADS = 64 * S::NW;
  static constexpr int WAVES_PER_EU = 1;
  static constexpr int WG_PER_CU = 1;
  static constexpr int LDS_BYTES = 5 * S::TILEB;
};
template <>
struct FwdKernelCfg<256, true> : FwdKernelCfg1W<256, 1> {};
template <bool PP>
struct FwdKernelCfg<128, PP> {
  static constexpr int BM = FwdShapeD128::BM;
  static constexpr int THREADS = 512;
  static constexpr int WAVES_PER_EU = 2;
  static constexpr int WG_PER_CU = 1;
  static constexpr int LDS_BYTES = FwdShapeD128::LDS_BYTES;
};

// LDS: one array for the 4-wave core; four regions for the D = 128 cores (see
// attn_fwd_tiles_d128).  PP: the ping-pong D = 128 core, which
// needs 16 consecutive keys at a fixed row stride (dense rows, or pages of
// at least 16 keys) with row strides below 2^24 elements; otherwise the
// one-phase core.
template <class T, int D, bool PP, class Prob>
__device__ __forceinline__ void run_fwd_tile(const Prob& P, int row0, float scale) {
  if constexpr (D == 128) {
    constexpr int B = FwdShapeD128::LDS_ARRAY_BYTES;
    __shared__ __attribute__((aligned(16))) char k0[B], v0[B], k1[B], v1[B];
    if constexpr (PP)
      attn_fwd_tile_d128<T>(P, row0, scale, k0, v0, k1, v1);
    else
      attn_fwd_tile_d128_plain<T>(P, row0, scale, k0, v0, k1, v1);
  } else if constexpr (D == 256 && PP) {
    __shared__ __attribute__((aligned(16))) char smem[FwdKernelCfg1W<256, 1>::LDS_BYTES];
    attn_fwd_tile_1w<T, 256, 1>(P, row0, scale, smem);
  } else {
    __shared__ __attribute__((aligned(16))) uint16_t smem[FwdShape<D>::LDS_ELEMS];
    attn_fwd_tile<T, D>(P, row0, scale, smem);
  }
}

// A sequence of row tiles on one workgroup: next(P, row0) rewrites the
// problem and first row for the next tile, false after the last one.  The
// D = 128 ping-pong core overlaps each tile's output stores with the next
// tile's first loads; the other cores run the tiles one after the other,
// with a barrier between them (their last LDS reads are not followed by a
// barrier of their own).
template <class T, int D, bool PP, class Prob, class Next>
__device__ __forceinline__ void run_fwd_tiles(Prob P, int row0, float scale, Next next) {
  if constexpr (D == 128 && PP) {
    constexpr int B = FwdShapeD128::LDS_ARRAY_BYTES;
    __shared__ __attribute__((aligned(16))) char k0[B], v0[B], k1[B], v1[B];
    attn_fwd_tiles_d128<T>(P, row0, scale, k0, v0, k1, v1, next);
  } else {
    for (;;) {
      run_fwd_tile<T, D, PP>(P, row0, scale);
      if (!next(P, row0)) break;
      __syncthreads();
    }
  }
}

// Row problem of query head bh % H of batch bh / H, its arguments read through
// `ap` (a pointer to fa_fwd_args in any address space).
template <int MODE, class ArgsPtr>
__device__ __forceinline__ void dense_rows(const ArgsPtr ap, int bh, DenseRows& P) {
  const int H = ap->num_heads;
  const int h = bh % H;
  const int b = bh / H;
  const int hk = h / (H / ap->num_heads_k);
  P.q = static_cast<const uint16_t*>(ap->q) + b * ap->q_stride[0] + h * ap->q_stride[2];
  P.o = static_cast<uint16_t*>(ap->out) + b * ap->o_stride[0] + h * ap->o_stride[2];
  P.lse = ap->lse ? ap->lse + ((int64_t)b * H + h) * ap->seqlen_q : nullptr;
  P.k = static_cast<const uint16_t*>(ap->k) + b * ap->k_stride[0] + hk * ap->k_stride[2];
  P.v = static_cast<const uint16_t*>(ap->v) + b * ap->v_stride[0] + hk * ap->v_stride[2];
  P.qs = ap->q_stride[1];
  P.os = ap->o_stride[1];
  P.ks = ap->k_stride[1];
  P.vs = ap->v_stride[1];
  P.nrows = ap->seqlen_q;
  P.sk = ap->seqlen_k;
  P.off = ap->seqlen_k - ap->seqlen_q;
  const Band band = mode_band<MODE>(*ap);
  P.wl = band.wl;
  P.wr = band.wr;
  P.has_lse = ap->lse != nullptr;
}

// MODE (MaskMode): full attention, causal, or a window band from the
// arguments.  The causal and full bands are compile-time constants.
template <class T, int D, int MODE>
__global__ __launch_bounds__((FwdKernelCfg<D, true>::THREADS),
                             (FwdKernelCfg<D, true>::WAVES_PER_EU))
void fwd_dense_kernel(fa_fwd_args a) {
  using C = FwdKernelCfg<D, true>;
  const int qtiles = (a.seqlen_q + C::BM - 1) / C::BM;
  const int nbh = a.batch * a.num_heads;
  // Persistent: this workgroup's tiles are rounds 0, 1, ... of
  // persistent_tile (one workgroup per tile when the grid covers them all).
  // Each tile's problem is set up from the arguments in the kernarg segment.
  auto setup = [qtiles, nbh](int vid, DenseRows& P, int& row0) {
    const auto* ap = kernel_args<fa_fwd_args>();
    const TileHead th = xcd_tile_order(vid, qtiles, nbh);
    // Heaviest causal tiles (largest query index) first.
    const int qt = MODE != kMaskNone ? qtiles - 1 - th.rank : th.rank;
    dense_rows<MODE>(ap, th.bh, P);
    row0 = qt * C::BM;
  };
  DenseRows P;
  int row0 = 0;
  if constexpr (MODE == kMaskBand) {
    // A band from the arguments costs the core registers (the tile loop
    // around it spilled inside the key loop): one workgroup per tile.
    if (blockIdx.x >= (unsigned)(qtiles * nbh)) return;
    setup(blockIdx.x, P, row0);
    run_fwd_tile<T, D, true>(P, row0, a.softmax_scale);
    return;
  }
  int r = 0;
  const int vid = persistent_tile(blockIdx.x, gridDim.x, r, qtiles * nbh, nbh);
  if (vid < 0) return;
  setup(vid, P, row0);
  run_fwd_tiles<T, D, true>(P, row0, a.softmax_scale, [&](DenseRows& Pn, int& rn) {
    const int v = persistent_tile(blockIdx.x, gridDim.x, ++r, qtiles * nbh, nbh);
    if (v < 0) return false;
    setup(v, Pn, rn);
    return true;
  });
}

// Keys split across the waves of a workgroup (fa_fwd_split.h), for grids too
// small for the kernel above: one workgroup per 32 query rows of a head.
constexpr int dense_split_waves(int D) {
  return D == 64 ? tiles::kFwdSplitWaves64 : tiles::kFwdSplitWaves128;
}
template <class T, int D, int MODE>
__global__ __launch_bounds__(64 * dense_split_waves(D)) void fwd_split_kernel(fa_fwd_args a) {
  constexpr int NW = dense_split_waves(D);
  __shared__ __attribute__((aligned(16))) char smem[FwdSplitShape<D, NW>::LDS];
  const TileHead th = xcd_tile_order(blockIdx.x, (a.seqlen_q + 31) / 32, a.batch * a.num_heads);
  DenseRows P;
  dense_rows<MODE>(&a, th.bh, P);
  attn_fwd_split_tile<T, D, NW>(P, 32 * th.rank, a.softmax_scale, smem);
}

struct PagedRows {
  const uint16_t* q;  // token 0 of the sequence, head hk*G
  uint16_t* o;
  float* lse;         // [Hq, num_tokens] at head hk*G, token 0 of the sequence
  int64_t q_tok, q_head, o_tok, o_head, lse_head;
  const uint16_t* kc;  // head hk
  const uint16_t* vc;
  int64_t k_page, k_slot, v_page, v_slot;
  const int32_t* bt;   // block_table row of the sequence
  int ps_log2, ps_mask, last_page;
  int G, nrows, seq_len, prefix, wq, wk;
  bool causal, has_lse;
  static constexpr bool kF32Out = false;
  static constexpr bool kRowStrided = false;

  __device__ int kv_lo(int r) const {
    if (!causal || wq <= 0) return 0;
    return max(0, r / G - wq + 1);
  }
  __device__ int kv_hi(int r) const {
    const int t = r / G;
    int hi = seq_len;
    if (causal) hi = min(hi, prefix + t + 1);
    if (causal && wk > 0) hi = min(hi, t + wk);
    return hi;
  }
  __device__ const uint16_t* q_ptr(int r) const {
    const int t = r / G;
    return q + t * q_tok + (r - t * G) * q_head;
  }
  __device__ uint16_t* o_ptr(int r) const {
    const int t = r / G;
    return o + t * o_tok + (r - t * G) * o_head;
  }
  __device__ float* lse_ptr(int r) const {
    const int t = r / G;
    return lse + (r - t * G) * lse_head + t;
  }
  __device__ int64_t page_of(int n) const {
    // The block table is read-only for the kernel's lifetime: through a
    // constant-address-space pointer a wave-uniform n reads it with a scalar
    // load (waited for on lgkmcnt).  A plain load compiled to a vector load
    // followed by vmcnt(0), which also waited for every K / V tile DMA in
    // flight, twice per tile.  The clamp guards against a corrupt table;
    // valid tables are unaffected.
    const auto* btc = (const __attribute__((address_space(4))) int32_t*)bt;
    return (int64_t)min((unsigned)btc[n >> ps_log2], (unsigned)last_page);
  }
  __device__ const uint16_t* k_ptr(int n) const {
    return kc + page_of(n) * k_page + (n & ps_mask) * k_slot;
  }
  __device__ const uint16_t* v_ptr(int n) const {
    return vc + page_of(n) * v_page + (n & ps_mask) * v_slot;
  }
  // Stride between consecutive keys of one page.
  __device__ int64_t k_row_stride() const { return k_slot; }
  __device__ int64_t v_row_stride() const { return v_slot; }
};

// One split of a split-KV paged prefill: the keys of the sequence are cut
// into nsplit ranges of a multiple of 128 keys; this problem sees only keys
// in [split_lo, split_hi) and writes its normalised partial O (fp32) and
// base-2 LSE into the workspace at [split][head][token].
struct PagedSplitRows : PagedRows {
  static constexpr bool kF32Out = true;
  int split_lo, split_hi;
  float* po;     // [nsplit][Hq][num_tokens][D] at (split, head hk*G, token 0 of the sequence)
  float* plse;   // [nsplit][Hq][num_tokens]    at the same origin
  int64_t p_head;  // num_tokens
  int D;

  __device__ int kv_lo(int r) const { return max(PagedRows::kv_lo(r), split_lo); }
  __device__ int kv_hi(int r) const { return min(PagedRows::kv_hi(r), split_hi); }
  __device__ float* o32_ptr(int r) const {
    const int t = r / G;
    return po + ((r - t * G) * p_head + t) * D;
  }
  __device__ float* lse2_ptr(int r) const {
    const int t = r / G;
    return plse + (r - t * G) * p_head + t;
  }
};

// Workgroup order of the paged kernels: `combos` (KV head, key range) pairs x
// row-tile slots, slot 0 the tile with the most keys (find_sequence).  The
// hardware deals workgroup ids to the 8 XCDs in turn and starts each XCD's in
// order, so every XCD gets whole combos where they divide evenly (its tiles
// share K / V in its L2), or shares a combo's slots with others in turn where
// there are fewer, and always walks the slots from the first: long tiles start
// first on every XCD and in every combo.  Ranges of ids that were contiguous
// per XCD (combo-major) started each combo's long tiles when the one before
// it ended, and with 1, 2 or 4 KV heads gave some XCDs only the long tiles and
// others the short ones (figures in fa_tiles.h).
struct SlotCombo {
  int slot, combo;
};
constexpr int kOrderXcds = 8;
__device__ __forceinline__ SlotCombo paged_order(int wg, int combos) {
  const int x = wg % kOrderXcds, l = wg / kOrderXcds;
  if (combos % kOrderXcds == 0) {
    const int per = combos / kOrderXcds;
    return {l / per, x * per + l % per};
  }
  if (kOrderXcds % combos == 0) {
    return {l * (kOrderXcds / combos) + x / combos, x % combos};
  }
  return {wg / combos, wg % combos};
}
// Workgroups that cover `slots` slots of `combos` combos (slots past the last
// tile find no sequence).
static int64_t paged_order_grid(int64_t slots, int64_t combos) {
  const int64_t f = kOrderXcds % combos == 0 ? kOrderXcds / combos : 1;
  return (slots + f - 1) / f * f * combos;
}

// Compute units, and the workgroups they hold at once, for find_sequence (figures
// in fa_tiles.h); slots of a key range where the ranges go one after the other, 0
// where they go side by side.
struct PagedOrder {
  int cus, one_round, range_slots;
};

// Finds the sequence owning slot `tile` in the varlen tile space where
// sequence b has ceil(qlen_b * G / BM) tiles.  Returns b (or -1) and the
// tile's index from the sequence's last (the one that sees most keys).
// Up to 64 sequences, one per lane of wave 0, in one of three orders; u_b is the
// history in units of a tile's rows, u_b + i + 1 the reach of tile i:
//  * by sequence, each from its longest tile: grids of no more workgroups (tiles x
//    combos) than CUs, a single sequence or two short prompts (the search below
//    costs 0.5-1 us a workgroup), and more rounds than the next item's without
//    histories to tell sequences apart;
//  * up to two rounds (kPagedTileOrderRounds; three where XCDs share combos): all
//    tiles by decreasing reach, ties by sequence.
//    Sequence b has n_b(K) = clamp(u_b + ntiles_b - K, 0, ntiles_b) tiles of
//    reach above K;
//  * more rounds: sequences by the reach of their last tile, longest
//    first (the tiles of one share its K / V in the L2), n_b(K) = all or none.
// For the last two a search for the smallest K with at most `tile` tiles above
// it, and the slot's rank among those at K, name the tile.  More sequences are
// scanned in their own order, 64 at a time.
__device__ int find_sequence(const int32_t* qsl, const int32_t* prefix, int batch, int G,
                             int BM, int combos, PagedOrder order, int tile, int* local) {
  __shared__ int found_b, found_local;
  if (wave_id() == 0) {
    const int lane = threadIdx.x & 63;
    int fb = -1, fl = 0;
    if (batch <= 64) {
      int n = 0, u = 0;
      if (lane < batch) {
        const int ql = qsl[lane + 1] - qsl[lane];
        n = ql > 0 ? (int)(((int64_t)ql * G + BM - 1) / BM) : 0;
        u = (int)min((int64_t)max(prefix[lane], 0) * G / BM, (int64_t)1 << 29);
      }
      int last = wave_scan(n);
      const int total = __builtin_amdgcn_readlane(last, 63);
      const int64_t wgs = (int64_t)total * combos;
      int here = n, before = 0, rank = tile;
      const int rounds = combos % kOrderXcds == 0 ? tiles::kPagedTileOrderRounds
                                                  : tiles::kPagedTileOrderRoundsShared;
      const bool by_tile = wgs <= rounds * (int64_t)order.one_round;
      const uint64_t some = __ballot(n > 0);
      if (wgs > order.cus && tile < total && __popcll(some) > 1) {
        const int u0 = __builtin_amdgcn_readlane(u, __ffsll((unsigned long long)some) - 1);
        auto reach = [&]() { return wave_max_nonneg(u + n); };
        if (__ballot(n > 0 && u != u0) != 0 ||
            (by_tile && (__popcll(some) > 2 ||
                         (int64_t)reach() * BM >= (int64_t)tiles::kPagedOrderPairKeys * G))) {
          auto above = [&](int K) {
            return by_tile ? min(max(u + n - K, 0), n) : (u + n > K ? n : 0);
          };
          // lo: all tiles lie above the least history; hi: none above the
          // longest reach.
          constexpr int kFar = 1 << 29;  // u's bound
          int lo = kFar - wave_max_nonneg(n > 0 ? kFar - u : 0), hi = reach();
          while (hi - lo > 1) {
            const int mid = (int)(((unsigned)lo + (unsigned)hi) >> 1);
            if (wave_total(above(mid)) > tile)
              lo = mid;
            else
              hi = mid;
          }
          before = above(hi);
          rank = tile - wave_total(before);  // among the tiles at K = hi
          here = above(hi - 1) - before;
          last = wave_scan(here);
        }
      }
      const uint64_t hit = __ballot(here > 0 && rank >= last - here && rank < last);
      if (hit) {
        fb = __ffsll((unsigned long long)hit) - 1;
        fl = __builtin_amdgcn_readlane(before + rank - (last - here), fb);
      }
    } else {
      int base = 0;
      for (int c0 = 0; c0 < batch; c0 += 64) {
        const int b = c0 + lane;
        int n = 0;
        if (b < batch) {
          const int ql = qsl[b + 1] - qsl[b];
          n = ql > 0 ? (int)(((int64_t)ql * G + BM - 1) / BM) : 0;
        }
        int incl = n;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int v = __shfl_up(incl, off);
          if (lane >= off) incl += v;
        }
        const int excl = incl - n;
        const bool hit = b < batch && n > 0 && tile >= base + excl && tile < base + incl;
        const uint64_t m = __ballot(hit);
        if (m) {
          const int src = __ffsll((unsigned long long)m) - 1;
          fb = c0 + src;
          fl = tile - base - __shfl(excl, src);
          break;
        }
        base += __shfl(incl, 63);
      }
    }
    if (lane == 0) {
      found_b = fb;
      found_local = fl;
    }
  }
  __syncthreads();
  *local = found_local;
  return found_b;
}

// Row problem of KV head hk of sequence b (query tokens qs .. qs+qlen-1).
template <class Args>
__device__ __forceinline__ void paged_rows(const Args& a, int hk, int b, int qs, int qlen,
                                           PagedRows& P) {
  const int G = a.num_heads / a.num_kv_heads;
  P.G = G;
  P.nrows = qlen * G;
  P.q = static_cast<const uint16_t*>(a.q) + (int64_t)qs * a.q_stride[0] +
        (int64_t)hk * G * a.q_stride[1];
  P.o = static_cast<uint16_t*>(a.out) + (int64_t)qs * a.o_stride[0] +
        (int64_t)hk * G * a.o_stride[1];
  P.q_tok = a.q_stride[0];
  P.q_head = a.q_stride[1];
  P.o_tok = a.o_stride[0];
  P.o_head = a.o_stride[1];
  P.has_lse = a.lse != nullptr;
  P.lse = a.lse ? a.lse + (int64_t)hk * G * a.num_tokens + qs : nullptr;
  P.lse_head = a.num_tokens;
  P.kc = static_cast<const uint16_t*>(a.k_cache) + (int64_t)hk * a.k_stride[2];
  P.vc = static_cast<const uint16_t*>(a.v_cache) + (int64_t)hk * a.v_stride[2];
  P.k_page = a.k_stride[0];
  P.k_slot = a.k_stride[1];
  P.v_page = a.v_stride[0];
  P.v_slot = a.v_stride[1];
  P.bt = a.block_table + (int64_t)b * a.block_table_stride;
  P.ps_log2 = __builtin_ctz(a.page_size);
  P.ps_mask = a.page_size - 1;
  P.last_page = a.num_pages - 1;
  // Keys beyond the block table's reach cannot be resolved; they are treated
  // as absent.
  P.seq_len = max(0, min(a.seq_lens[b], a.max_blocks * a.page_size));
  P.prefix = a.prefix_kv_lens[b];
  P.causal = a.causal != 0;
  P.wq = a.window_q;
  // (A bound of the sequence's length hides nothing; with one near 2^31, token
  // + bound would leave 32 bits.)
  P.wk = min(a.window_k, P.seq_len);
}

// One row tile of a paged problem, which sees up to keys() keys; setup(args, P)
// fills the problem from the kernel's arguments.  A tile of at most 32 rows (a
// decoding sequence in a prefill batch, or the last rows of a prompt) would
// keep one wave of the row-tile cores busy, serially over the keys; with FEW
// its keys, from kPagedFewMinKeys on, are split over the waves instead
// (fa_fwd_split.h).  Each branch sets up its own problem, the few-row one from
// arguments the compiler reloads: with one problem for both, its scalars stayed
// live across the ping-pong core and spilled in its loop (49 spilled SGPRs
// against 13, C5-size chunked prefill 0.7% slower).  The launcher leaves FEW out
// where tiles are mostly full (paged_few_rows): the branch costs the row-tile
// cores registers (head_dim 256 242 -> 256 VGPRs).
template <class T, int D, bool PP, bool FEW, class Prob, class Keys, class Setup>
__device__ __forceinline__ void run_paged_tile(const fa_paged_args& a, int rows, Keys keys,
                                               int row0, Setup setup) {
  using C = FwdKernelCfg<D, PP>;
  if constexpr (FEW) {
    constexpr int NW = C::THREADS / 64;
    constexpr int kSplitLds = FwdSplitShape<D, NW>::LDS;
    constexpr int kLds = kSplitLds > C::LDS_BYTES ? kSplitLds : C::LDS_BYTES;
    __shared__ __attribute__((aligned(16))) char smem[kLds];
    if (rows <= 32 && keys() >= (D == 256 ? tiles::kPagedFewMinKeys256 : tiles::kPagedFewMinKeys)) {
      const auto* ap = kernel_args<fa_paged_args>();
      Prob P;
      setup(*ap, P);
      attn_fwd_split_tile<T, D, NW>(P, row0, ap->softmax_scale, smem);
      return;
    }
    Prob P;
    setup(a, P);
    if constexpr (D == 128) {
      constexpr int B = FwdShapeD128::LDS_ARRAY_BYTES;
      attn_fwd_tile_d128<T>(P, row0, a.softmax_scale, smem, smem + B, smem + 2 * B, smem + 3 * B);
    } else if constexpr (D == 256) {
      attn_fwd_tile_1w<T, 256, 1>(P, row0, a.softmax_scale, smem);
    } else {
      attn_fwd_tile<T, D>(P, row0, a.softmax_scale, reinterpret_cast<uint16_t*>(smem));
    }
  } else {
    Prob P;
    setup(a, P);
    run_fwd_tile<T, D, PP>(P, row0, a.softmax_scale);
  }
}

template <class T, int D, bool PP, bool FEW>
__global__ __launch_bounds__((FwdKernelCfg<D, PP>::THREADS), (FwdKernelCfg<D, PP>::WAVES_PER_EU))
void fwd_paged_kernel(fa_paged_args a, PagedOrder order) {
  using S = FwdKernelCfg<D, PP>;
  const int G = a.num_heads / a.num_kv_heads;
  const SlotCombo sc = paged_order(blockIdx.x, a.num_kv_heads);
  const int hk = sc.combo, slot = sc.slot;

  int local = 0;
  const int b = find_sequence(a.query_start_loc, a.prefix_kv_lens, a.batch, G, S::BM,
                              a.num_kv_heads, order, slot, &local);
  if (b < 0) return;
  const int qs = a.query_start_loc[b];
  const int qlen = a.query_start_loc[b + 1] - qs;
  const int ntiles = (int)(((int64_t)qlen * G + S::BM - 1) / S::BM);
  // Later tiles of a causal sequence see more keys: run them first.
  const int tile = ntiles - 1 - local;
  const int row0 = tile * S::BM;
  run_paged_tile<T, D, PP, FEW, PagedRows>(
      a, qlen * G - row0, [&a, b] { return a.seq_lens[b]; }, row0,
      [=](const auto& args, PagedRows& P) { paged_rows(args, hk, b, qs, qlen, P); });
}

// Split-KV variant: workgroup (KV head, split, tile slot); the splits of a
// sequence cover its keys in ranges of ceil(seq_len / nsplit) rounded up to
// 128.
template <class T, int D, bool PP, bool FEW>
__global__ __launch_bounds__((FwdKernelCfg<D, PP>::THREADS), (FwdKernelCfg<D, PP>::WAVES_PER_EU))
void fwd_paged_split_kernel(fa_paged_args a, PagedOrder order, int nsplit, float* po,
                            float* plse) {
  using S = FwdKernelCfg<D, PP>;
  const int G = a.num_heads / a.num_kv_heads;
  // Ranges of a slot side by side, or (order.range_slots of them each) one range
  // after the other: see split_range_slots.
  const bool by_range = order.range_slots > 0;
  const SlotCombo sc = paged_order(blockIdx.x, by_range ? a.num_kv_heads : a.num_kv_heads * nsplit);
  const int hk = by_range ? sc.combo : sc.combo / nsplit;
  const int split = by_range ? sc.slot / order.range_slots : sc.combo % nsplit;
  const int slot = by_range ? sc.slot % order.range_slots : sc.slot;
  if (split >= nsplit) return;  // a grid rounded up to whole XCDs

  int local = 0;
  const int b = find_sequence(a.query_start_loc, a.prefix_kv_lens, a.batch, G, S::BM,
                              a.num_kv_heads * nsplit, order, slot, &local);
  if (b < 0) return;
  const int qs = a.query_start_loc[b];
  const int qlen = a.query_start_loc[b + 1] - qs;
  const int ntiles = (int)(((int64_t)qlen * G + S::BM - 1) / S::BM);
  const int tile = ntiles - 1 - local;
  const int row0 = tile * S::BM;
  run_paged_tile<T, D, PP, FEW, PagedSplitRows>(
      a, qlen * G - row0, [&a, b, nsplit] { return a.seq_lens[b] / nsplit; }, row0,
      [=](const auto& args, PagedSplitRows& P) {
        paged_rows(args, hk, b, qs, qlen, P);
        const int chunk = ((P.seq_len + nsplit - 1) / nsplit + 127) / 128 * 128;
        P.split_lo = split * chunk;
        P.split_hi = P.split_lo + chunk;
        const int64_t origin =
            ((int64_t)split * args.num_heads + (int64_t)hk * (args.num_heads / args.num_kv_heads)) *
                args.num_tokens + qs;
        P.po = po + origin * D;
        P.plse = plse + origin;
        P.p_head = args.num_tokens;
        P.D = D;
      });
}

// Merges the nsplit partials of each (query head, token): O = sum_s w_s O_s /
// sum_s w_s with w_s = 2^(lse_s - max); LSE = ln 2 (max + log2 sum_s w_s).
// One wave per (head, token); tokens outside query_start_loc[0] ..
// query_start_loc[batch] belong to no sequence and are left untouched, as
// the unsplit kernel leaves them.
template <class T, int D>
__global__ __launch_bounds__(256) void paged_combine_kernel(fa_paged_args a, int nsplit,
                                                            const float* po,
                                                            const float* plse) {
  constexpr int NP = (D + 127) / 128;  // d pairs per lane: 2 lane + 128 k
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;
  const int64_t NT = a.num_tokens;
  if (item >= (int64_t)a.num_heads * NT) return;
  const int h = (int)(item / NT);
  const int t = (int)(item % NT);
  if (t < a.query_start_loc[0] || t >= a.query_start_loc[a.batch]) return;
  const int64_t stride_s = (int64_t)a.num_heads * NT;  // rows per split
  const int64_t row = (int64_t)h * NT + t;
  float m = neg_inf();
  for (int s = lane; s < nsplit; s += 64) m = fmaxf(m, plse[s * stride_s + row]);
  m = wave_max(m);
  const float m_use = m == neg_inf() ? 0.f : m;
  float acc[NP][2];
#pragma unroll
  for (int k = 0; k < NP; ++k) acc[k][0] = acc[k][1] = 0.f;
  float wsum = 0.f;
  for (int s = 0; s < nsplit; ++s) {
    const float ls = plse[s * stride_s + row];
    const float w = ls == neg_inf() ? 0.f : fast_exp2(ls - m_use);
    wsum += w;
    const float* src = po + (s * stride_s + row) * D;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int d = 2 * lane + 128 * k;
      if (d < D) {
        const float2 pv = *reinterpret_cast<const float2*>(src + d);
        acc[k][0] = fmaf(w, pv.x, acc[k][0]);
        acc[k][1] = fmaf(w, pv.y, acc[k][1]);
      }
    }
  }
  const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
  uint16_t* op = static_cast<uint16_t*>(a.out) + (int64_t)t * a.o_stride[0] +
                 (int64_t)h * a.o_stride[1];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    const int d = 2 * lane + 128 * k;
    if (d < D)
      *reinterpret_cast<uint32_t*>(op + d) = T::pack(acc[k][0] * inv, acc[k][1] * inv);
  }
  if (a.lse && lane == 0) a.lse[row] = wsum > 0.f ? (m_use + log2f(wsum)) * kLn2 : neg_inf();
}

// ----------------------------------------------------------------- launchers

// Keys split across the waves of a workgroup (fa_fwd_split.h): one
// workgroup per 32 query rows of a head.
template <class T, int D>
static hipError_t launch_dense_split(const fa_fwd_args& a, int mode, hipStream_t st) {
  const dim3 grid((unsigned)((a.seqlen_q + 31) / 32) * a.num_heads * a.batch),
      block(64 * dense_split_waves(D));
  if (mode == kMaskCausal)
    hipLaunchKernelGGL((fwd_split_kernel<T, D, kMaskCausal>), grid, block, 0, st, a);
  else if (mode == kMaskBand)
    hipLaunchKernelGGL((fwd_split_kernel<T, D, kMaskBand>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((fwd_split_kernel<T, D, kMaskNone>), grid, block, 0, st, a);
  return hipGetLastError();
}

template <class T, int D>
static hipError_t launch_dense(const fa_fwd_args& a, hipStream_t st) {
  using C = FwdKernelCfg<D, true>;
  const int qtiles = (a.seqlen_q + C::BM - 1) / C::BM;
  const int mode = mask_mode(a);
  if constexpr (D == 64 || D == 128) {
    // Too few query tiles to give most CUs a workgroup: split the keys.
    const int64_t wgs = (int64_t)qtiles * a.num_heads * a.batch;
    if (wgs * tiles::kFwdSplitMaxFillDen < (int64_t)device_cu_count() * tiles::kFwdSplitMaxFillNum)
      return launch_dense_split<T, D>(a, mode, st);
  }
  // Band instances run one workgroup per tile (fwd_dense_kernel).
  const bool band = mode == kMaskBand;
  const dim3 grid((unsigned)(band ? qtiles * a.num_heads * a.batch
                                  : persistent_grid(qtiles, a.num_heads * a.batch,
                                                    C::WG_PER_CU)));
  if (mode == kMaskCausal)
    hipLaunchKernelGGL((fwd_dense_kernel<T, D, kMaskCausal>), grid, dim3(C::THREADS), 0, st, a);
  else if (band)
    hipLaunchKernelGGL((fwd_dense_kernel<T, D, kMaskBand>), grid, dim3(C::THREADS), 0, st, a);
  else
    hipLaunchKernelGGL((fwd_dense_kernel<T, D, kMaskNone>), grid, dim3(C::THREADS), 0, st, a);
  return hipGetLastError();
}

template <class T>
static hipError_t dispatch_dense_d(const fa_fwd_args& a, hipStream_t st) {
  switch (a.head_dim) {
    case 64: return launch_dense<T, 64>(a, st);
    case 128: return launch_dense<T, 128>(a, st);
    case 256: return launch_dense<T, 256>(a, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_fwd(const fa_fwd_args& a, hipStream_t st) {
  return a.dtype == FA_DTYPE_BF16 ? dispatch_dense_d<BFloat16>(a, st)
                                  : dispatch_dense_d<Half>(a, st);
}

// The D = 128 ping-pong core and the D = 256 core take K / V in runs of 16
// (D = 128) or 8 (D = 256) keys at a fixed row stride: pages of at least 16
// keys, token strides below 2^24 elements.
static bool paged_pingpong(const fa_paged_args& a) {
  const int64_t lim = int64_t(1) << 24;
  return (a.head_dim == 128 || a.head_dim == 256) && a.page_size >= 16 &&
         a.k_stride[1] < lim && a.v_stride[1] < lim;
}

int paged_block_rows(const fa_paged_args& a) {
  const bool pp = paged_pingpong(a);
  switch (a.head_dim) {
    case 64: return FwdKernelCfg<64, false>::BM;
    case 128: return FwdKernelCfg<128, false>::BM;
    case 256: return pp ? FwdKernelCfg<256, true>::BM : FwdKernelCfg<256, false>::BM;
    default: return FwdKernelCfg<512, false>::BM;
  }
}

int paged_grid_slots(const fa_paged_args& a) {
  const int G = a.num_heads / a.num_kv_heads;
  const int64_t rows = (int64_t)a.num_tokens * G;
  const int bm = paged_block_rows(a);
  // sum_b ceil(rows_b / BM) <= ceil(rows / BM) + batch
  return (int)((rows + bm - 1) / bm + a.batch);
}

// Workgroups of a paged problem before any split: the row tiles of all tokens
// together, but at least one per sequence (every sequence with tokens has a
// tile of its own), times the KV heads.
struct PagedTiles {
  int64_t rows, seqs, wgs;
};
static PagedTiles paged_tiles(const fa_paged_args& a) {
  const int64_t rows = (int64_t)a.num_tokens * (a.num_heads / a.num_kv_heads);
  const int64_t seqs = std::max(1, std::min(a.batch, a.num_tokens));
  const int bm = paged_block_rows(a);
  return {rows, seqs, std::max<int64_t>(seqs, (rows + bm - 1) / bm) * a.num_kv_heads};
}

// Whether few-row tiles get the key-split core, from sizes alone: pages and
// strides it can address (those of the ping-pong cores), and a batch in which
// such tiles can matter: at most kPagedFewMaxTiles full tiles per sequence,
// and more than the last rows of a single prompt.  Its workgroups at head_dim
// 256 have half the bytes in flight of the row-tile core's (one buffer in LDS),
// so once every CU has one, and with them the memory is busy, they lose
// (figures at kPagedFewMinKeys), except between tiles of more rows (half a tile's
// on average).
static bool paged_few_rows(const fa_paged_args& a, int nsplit) {
  const int64_t lim = int64_t(1) << 24;
  if (a.head_dim > 256 || a.page_size < 16 || a.k_stride[1] >= lim || a.v_stride[1] >= lim)
    return false;
  const PagedTiles t = paged_tiles(a);
  const int64_t bm = paged_block_rows(a);
  if (t.rows > tiles::kPagedFewMaxTiles * bm * t.seqs || (t.seqs == 1 && t.rows > 32)) return false;
  return a.head_dim != 256 || t.wgs * nsplit < device_cu_count() || 2 * t.rows > bm * t.seqs;
}

// Order of a split problem's key ranges.  Side by side, the long tiles of every
// range go first; but a range ends at a tile's causal limit, so of a long prompt
// the last range holds the short tiles and the others only whole ones, which
// then also went last: one range after the other there (kSplitByRangeTokens new
// tokens a sequence, an eighth of a range).
static int split_range_slots(const fa_paged_args& a, int nsplit) {
  if (nsplit <= 1) return 0;
  const int64_t seqs = paged_tiles(a).seqs, kv_cap = (int64_t)a.max_blocks * a.page_size;
  if (a.num_tokens < tiles::kSplitByRangeTokens * seqs ||
      8 * (int64_t)a.num_tokens * nsplit < kv_cap * seqs)
    return 0;
  return paged_grid_slots(a);
}

template <class T, int D, bool PP, bool FEW>
static hipError_t launch_paged_pp(const fa_paged_args& a, int nsplit, void* ws,
                                  hipStream_t st) {
  const int64_t slots = paged_grid_slots(a);
  const int range_slots = split_range_slots(a, nsplit);
  const unsigned grid = (unsigned)(range_slots > 0
      ? paged_order_grid(slots * nsplit, a.num_kv_heads)
      : paged_order_grid(slots, (int64_t)a.num_kv_heads * std::max(nsplit, 1)));
  const int cus = device_cu_count();
  const PagedOrder order{cus, cus * FwdKernelCfg<D, PP>::WG_PER_CU, range_slots};
  if (nsplit <= 1) {
    hipLaunchKernelGGL((fwd_paged_kernel<T, D, PP, FEW>), dim3(grid),
                       dim3(FwdKernelCfg<D, PP>::THREADS), 0, st, a, order);
    return hipGetLastError();
  }
  const size_t rows = (size_t)nsplit * a.num_heads * a.num_tokens;
  float* po = static_cast<float*>(ws);
  float* plse = po + rows * D;
  hipLaunchKernelGGL((fwd_paged_split_kernel<T, D, PP, FEW>), dim3(grid),
                     dim3(FwdKernelCfg<D, PP>::THREADS), 0, st, a, order, nsplit, po, plse);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t items = (int64_t)a.num_heads * a.num_tokens;
  hipLaunchKernelGGL((paged_combine_kernel<T, D>), dim3((unsigned)((items + 3) / 4)), dim3(256),
                     0, st, a, nsplit, po, plse);
  return hipGetLastError();
}

template <class T, int D>
static hipError_t launch_paged(const fa_paged_args& a, int nsplit, void* ws, hipStream_t st) {
  if constexpr (D == 128 || D == 256) {
    if (paged_pingpong(a))
      return paged_few_rows(a, nsplit) ? launch_paged_pp<T, D, true, true>(a, nsplit, ws, st)
                                       : launch_paged_pp<T, D, true, false>(a, nsplit, ws, st);
  }
  if constexpr (D == 64)
    if (paged_few_rows(a, nsplit)) return launch_paged_pp<T, D, false, true>(a, nsplit, ws, st);
  return launch_paged_pp<T, D, false, false>(a, nsplit, ws, st);
}

template <class T>
static hipError_t dispatch_paged_d(const fa_paged_args& a, int nsplit, void* ws,
                                   hipStream_t st) {
  switch (a.head_dim) {
    case 64: return launch_paged<T, 64>(a, nsplit, ws, st);
    case 128: return launch_paged<T, 128>(a, nsplit, ws, st);
    case 256: return launch_paged<T, 256>(a, nsplit, ws, st);
    case 512: return launch_paged<T, 512>(a, nsplit, ws, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_paged_prefill(const fa_paged_args& a, hipStream_t st) {
  return launch_paged_prefill_split(a, 1, nullptr, st);
}

hipError_t launch_paged_prefill_split(const fa_paged_args& a, int nsplit, void* ws,
                                      hipStream_t st) {
  return a.dtype == FA_DTYPE_BF16 ? dispatch_paged_d<BFloat16>(a, nsplit, ws, st)
                                  : dispatch_paged_d<Half>(a, nsplit, ws, st);
}

size_t paged_split_workspace_bytes(const fa_paged_args& a, int nsplit) {
  if (nsplit <= 1) return 0;
  const size_t rows = (size_t)nsplit * a.num_heads * a.num_tokens;
  return rows * a.head_dim * sizeof(float) + rows * sizeof(float) + 256;
}

// Split count from sizes alone (no device data).
int paged_num_splits(const fa_paged_args& a) {
  const auto [rows, seqs, wgs] = paged_tiles(a);
  const int64_t kv_cap = (int64_t)a.max_blocks * a.page_size;
  const int cus = device_cu_count();
  if (kv_cap < tiles::kSplitMinKeys) return 1;
  if (wgs >= cus) {
    // Every CU has a workgroup.  More ranges only shorten the last round, and
    // pay for it in partials of every row and a second launch: not for full
    // tiles.  Two ranges where one-token sequences have the longest tiles,
    // among chunks, in at most one and a half rounds.  At head_dim 64, whose
    // CUs hold two workgroups: three for batches of few rows a sequence, up to
    // four for full tiles after long histories.
    const bool mixed = a.num_tokens > seqs;
    const int64_t many = mixed && a.head_dim == 64 ? tiles::kSplitMinKeys : tiles::kSplitMaxRangeKeys;
    if (kv_cap <= many) return 1;
    const int bm = paged_block_rows(a);
    if (a.head_dim == 64) {
      if (2 * rows <= bm * seqs && wgs < 2 * (int64_t)cus) return 3;
      if (2 * wgs >= 3 * (int64_t)cus || kv_cap <= 2 * tiles::kSplitMaxRangeKeys) return 1;
      return (int)std::min<int64_t>(4, (kv_cap + tiles::kSplitMaxRangeKeys - 1) / tiles::kSplitMaxRangeKeys);
    }
    const int64_t full = (rows + bm - 1) / bm;
    return mixed && full <= seqs && 2 * (seqs + full) * a.num_kv_heads <= 3 * (int64_t)cus ? 2 : 1;
  }
  // No range is longer than kSplitMaxRangeKeys (a workgroup's serial length);
  // about one workgroup per CU, or two where the tiles hold few rows (tiles
  // bound by latency, whose partials are small); never shorter than
  // kSplitMinRangeKeys (each split adds a partial O per row to write and merge).
  const bool few = rows <= 32 * seqs;
  const int64_t want = few ? 2 * cus : cus;
  int64_t ns = std::max<int64_t>((kv_cap + tiles::kSplitMaxRangeKeys - 1) / tiles::kSplitMaxRangeKeys,
                                 (want + wgs - 1) / wgs);
  ns = std::min<int64_t>(ns, kv_cap / tiles::kSplitMinRangeKeys);
  return (int)std::max<int64_t>(1, std::min<int64_t>(ns, kMaxPagedSplits));
}

}  // namespace fa
