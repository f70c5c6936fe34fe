// Fixed gfx950 tile table.
//
// Replaces the reference's run-time autotuner (tilelang_fa_v100/_configs.py:5-79
// candidate generators, _utils.py:4-27 SM70 validity model, the fixed
// _BEST_CONFIGS / _DECODE_BEST_CONFIGS dicts in _kernels_paged.py:353-364,
// 495-499).  Every kernel takes its tile sizes from here; nothing is tuned at
// run time, so the first call of a shape costs no compilation or search.
// Each entry states the measurement (MI355X, rocprofv3 counters or event
// timing of T1 = causal fp16 B=2 S=8192 H=16 D=128, C2 = the same at B=4
// S=2048) that chose it over the alternatives tried.
#pragma once

namespace fa {
namespace tiles {

// ---- dense / paged forward, head_dim 128 (fa_fwd_d128.h)
// 256 query rows per workgroup = 8 waves x 32 rows (two waves per SIMD, 207
// VGPRs, no spills), 64-key K/V tiles double-buffered in LDS (64 KB).
// Evidence: T1 forward 0.545 ms, MFMA busy 52.5% (SQ_VALU_MFMA_BUSY_CYCLES);
// 4-wave / 128-row workgroups (two per CU) measured 0.673 ms against 0.640 ms
// for this shape under the same (one-phase) schedule; LDS bank conflicts 0
// (SQ_LDS_BANK_CONFLICT) with the 16-byte chunk swizzle.
constexpr int kFwd128Rows = 256;
constexpr int kFwd128Keys = 64;
constexpr int kFwd128Waves = 8;

// ---- dense / paged forward, head_dim 256 (fa_fwd_1w.h)
// 4 waves x 32 rows, one wave per SIMD, one pass over 32-key tiles with O in
// AGPRs (256 VGPRs + 155 AGPRs, no spills).  Evidence, T1 shape at head_dim
// 256 (B=2, S=8192, H=8, causal), same box: 0.638-0.649 ms against
// 0.760-0.763 ms for 8 waves x 32 rows at two waves per SIMD (230 VGPRs, O in
// two 128-column passes with the scores recomputed, 1.5x the products),
// bit-identical outputs; that schedule in turn took 0.844 ms against 1.204 ms
// for the one-pass register-staged 4-wave core (406 registers, accumulators
// shuffled between the register files).
constexpr int kFwd256Rows = 128;

// ---- forward, head_dim 64 / 256 / 512 (fa_fwd_core.h; head_dim 256 only for
// paged problems with pages of fewer than 16 keys)
// 128 query rows per workgroup (4 waves x 32 rows); keys per tile
// 8192 / D for D <= 256 (a 16 KB K tile), 32 for D = 512, whose O columns are
// accumulated in two 256-wide passes so Q, O and the staging fit one wave's
// 512 registers; 2 waves per SIMD for D <= 128, 1 above.
// Evidence (compiler resource usage): D = 64 takes 182 VGPRs and D = 256
// 254 VGPRs + 152 AGPRs (one wave per SIMD), both without spills; D = 512
// (two O passes) 253 VGPRs + 160 AGPRs in the VGPR MFMA form fa_fwd.hip is
// built in (35 spilled in the default form).  Dense problems too small to
// give half the CUs a 128-row tile (C1) take the key-split kernel below.
constexpr int kFwdCoreRows = 128;
constexpr int kFwdCoreTileElems = 8192;  // keys x head_dim per K tile (D <= 256)
constexpr int kFwdCoreKeys512 = 32;

// ---- dense forward with keys split across the waves of a workgroup
// (fa_fwd_split.h), head_dim 64 / 128: used when the standard cores' grid
// would give fewer than a kFwdSplitMaxFill share of the CUs a workgroup
// (configs[0], [1, 512, 16, 64]: 64 workgroups of 128 rows for 256 CUs).
// 32 query rows per workgroup; 8 waves (two per SIMD), each with a private
// pair of 32-key K / V tiles (double-buffered at head_dim 64, single at 128;
// 128 KB of LDS).  Evidence (event time per call, same box): C1 9.2 us
// against 13.5 us on the 128-row core (kernel trace 7.4 against 12.5 us) and
// 10.9 us with 16 waves (one tile each, single-buffered); [1, 2048, 8, 128]
// 43.0 / 33.2 us (full / causal) against 47.8 / 36.6 us with 4 waves and
// 57.4 / 55.0 us on the 256-row core; [4, 300, 8, 128] 18.6 us against 16.6
// (4 waves) and 18.9 (256-row core).
constexpr int kFwdSplitWaves64 = 8;
constexpr int kFwdSplitWaves128 = 8;
constexpr int kFwdSplitMaxFillNum = 1, kFwdSplitMaxFillDen = 2;  // one half

// ---- backward dK / dV kernel, head_dim 128 / 256 (fa_bwd_mfma.h)
// KV-stationary: head_dim 128 keeps 256 keys per workgroup (8 waves x 32 keys,
// dK / dV of a wave's 32 keys in 128 registers), head_dim 256 keeps 128 keys
// (4 waves); 32 query rows per iteration.  Evidence: every Q / dO tile read
// from LDS serves the whole key tile, so the largest key tile whose dK / dV fit
// the register file wins; 4 waves x 64 keys (512 registers each) measured
// 2.31 ms against 1.81 ms (T1 backward), and a two-group ping-pong schedule
// with three Q / dO buffers 1.115 against 1.105 ms for the kernel (it runs
// near the LDS read rate: five 1 KB operand reads per four MFMAs).
constexpr int kBwdQueryRows = 32;
// Measured again with the current kernel (same box, T1 backward, dK / dV /
// dQ bit-identical in every variant): 4 waves x 64 keys at one wave per SIMD
// (dK / dV of 64 keys pinned in the 256 AGPRs, every Q / dO / Qᵀ / dOᵀ read
// feeding two products) 1.85 ms against 1.69-1.77 ms for 8 waves x 32 keys,
// and C2 0.29 against 0.26-0.27 ms.  Counters (T1): the same MFMA busy
// cycles but co-execution of MFMA and VALU 10x lower (3.0e7 against 2.9e8
// cycles): a lone wave issues in order, so its softmax runs between its
// products instead of under the partner wave's.  Interleaving the element
// work into the chains (exponentials between the dP products, dS between the
// dV products, separate S / dP / dV / dK chains) compiled without spills
// only with the masked / unmasked branch confined to the element work, and
// still measured 1.81-1.93 ms (head_dim 256, same schedule: 1.76-1.87
// against 1.64-1.70 ms for the combined S / dP loop and dV / dK chain).

// ---- backward: dQ (fa_bwd_dq.h), query-stationary, no atomics.  Evidence
// (fa_bwd per call, ms, dQ by fp32 atomics from the key-stationary kernel /
// query-stationary kernel, fp16): D=64 B4 S2048 H16 causal 0.405 / 0.343,
// full 0.523 / 0.443; D=128 C2 causal 0.314 / 0.300, full 0.521 / 0.507, T1
// 1.811 / 1.814, GQA 32/8 B2 S4096 causal 1.283 / 1.224, full 1.733 / 1.772,
// B1 S16384 H8 1.767 / 1.777, B8 S1024 0.203 / 0.208; D=256 B2 S8192 H8 causal
// 3.474 / 2.409 (with fa_bwd.hip compiled for VGPR-form MFMA, see build.py).
// The atomics are performed beyond the XCD's L2 on this part, ~64 address
// cycles per instruction, a floor of ~1.17 ms for T1's backward.

// ---- backward: dQ from stored dS tiles (fa_bwd_ds.h), head_dim 128 / 256,
// while the tiles (2 bytes per visible (query, key) pair, 2.15 GB at T1; a
// window band takes its width in whole 32-key blocks per 32 rows) stay within
// this many bytes; larger problems recompute S and dP in bwd_dq_kernel.
// Evidence for bands (fa_bwd per call, us, recompute / dS, same box, both with
// the dK / dV kernel skipping the tiles outside a wave's band): causal,
// [2, 4096, 16, 128] window 1024 287 / 236, window 256 175 / 143, [2, 8192, 8,
// 128] window 4096 777 / 691, [2, 4096, 8, 256] window 1024 276 / 227, [1, 1024,
// 8, 128] window 200 60 / 48.
constexpr size_t kBwdDsMaxBytes = size_t(4) << 30;

// ---- backward dK / dV kernel, head_dim 64 (fa_bwd_mfma.h): 128 keys per
// workgroup (4 waves x 32 keys), three workgroups per CU (164-168 VGPRs, no
// spills).  Bound by the matrix cores and the VALU together (16 products
// against ~450 cycles of element work per 32 x 32 tile) and by the LDS operand
// reads.  Evidence (fa_bwd per call, us, same box, against the register-
// staged kernel this replaced, which transposed Q / dO with VALU and wrote
// both forms to LDS): [4, 2048, 16, 64] causal 237 -> 147, full 309 -> 265;
// [2, 8192, 16, 64] causal 1250 -> 990; [16, 512, 16, 64] causal 93 -> 69.  K
// in registers instead of LDS spills at three waves per SIMD and took 152 /
// 272 / 1000 / 71 us at two.
constexpr int kBwd64WavesPerSimd = 3;

// ---- backward dK / dV in pieces (fa_bwd.hip bwd_pieces): at most
// kBwdMaxPieces workgroups per (key tile, KV head), none with fewer than
// kBwdPieceTiles 32-row query tiles (a workgroup's start and end cost about
// three tiles, and the reduction another launch).  Evidence (fa_bwd per call,
// us, bf16, for 1 / 2 / 3 / 4 / 6 / 8 pieces; the rule's choice in brackets):
//   [1, 2048, 32/8, 128] causal   401 / 248 / 197 / 172 / 154 / 161  [5: 163]
//   [2, 2000, 32/8, 128] causal   434 / 297 / 253 / 256 / 287 / 313  [3]
//   [1, 8192, 8/2, 128] causal   1505 / 872 / 668 / 567 / 478 / 457  [6]
//   [1, 2048, 8, 128] full        140 / 114 / 103 / 103 / 120 / 125  [3]
//   [2, 2048, 16, 128] causal     162 / 178 / 204 / 244 / 316 / 378  [1]
//   [1, 4096, 32/8, 64] causal    438 / 314 / 286 / 266 / 274 / 279  [4]
//   [1, 8192, 8/2, 256] causal   1926 / 1175 / 914 / 832 / 897 / 875 [4]
constexpr int kBwdMaxPieces = 16;
constexpr int kBwdPieceTiles = 16;

// ---- decode, head_dim 64 / 128 / 256 / 512, pages of at least 16 keys or of
// at least one DMA instruction's 1024 / 2D rows (fa_decode_stream.h)
// Persistent waves; work item = a split of keys x one KV head x its query
// heads (up to 8, the 16x16x32 MFMA columns); 16-key tiles, two in flight
// per wave.  Keys per split: the largest of kDecSplitKeysMax, /2, /4 ..
// kDecSplitKeysMid whose item count, estimated from max_seq_len, is at least
// kDecItemsPerWave per resident wave (long items amortise each item's query
// load and partial-result store; enough items keep every wave streaming);
// the kernel doubles it when the actual lengths allow (T2 83%, C4 stays 80%).
// Evidence (C4 = 64 sequences of 1083-32645 keys, T2 = 64 x 32768; % of
// 8 TB/s, cache flushed by a read): split 256: 67.6 / 66.8; 512: 71.3 /
// 74.1; 1024: 75.3 / 76.3; 2048: 79.5 / 80.9; 4096: 66.2 / 83.4 (C4 then
// has ~1 item per wave, and max_seq_len cannot tell it from T2).  T2 reads
// 1.006x its algorithmic bytes (FETCH_SIZE).  Head_dim 64 and 256 run the same
// kernel with the ring depth and waves per workgroup scaled so that every CU
// keeps ~128 KB of K / V in flight (64: 4 tiles x 8 waves, 256: 2 tiles x 4
// waves, 512: 2 tiles x 2 waves): 64 x 16k keys at D = 64 76.0%, 64 x 8k at
// D = 256 83.2%, 64 x 4k at D = 512 79.2% of 8 TB/s, against 63-66% on the
// chunked kernel below.
// Below kDecSplitKeysMid, down to kDecSplitKeysMin, while there is less than one
// item per two waves (a wave walks its item's 16-key tiles serially, two in
// flight; ~1.3 us each), from max_seq_len on the host and from the actual
// lengths on the device (block tables are often far wider).  Evidence (us per
// call, 32 / 8 heads, D = 128, 512-key items / this rule): 4 sequences of
// 0.5-8k keys 49 / 20, 1 of 4k 45 / 12, 1 of 32k 53 / 30, 32 of 300-700 48 /
// 21, 16 of 0.5-8k (1100 items of 512) 61 / 57.  Halving until every wave has
// an item: 24 / 12 / 36 / 26 / 63 (more partials to write and merge); one per
// four waves: 22 / 12 / 31 / 31 / 57.
constexpr int kDecSplitKeysMax = 2048;
constexpr int kDecSplitKeysMid = 512;
constexpr int kDecSplitKeysMin = 64;
constexpr int kDecItemsPerWave = 2;
constexpr int kDecTileKeys = 16;
constexpr int kDecTilesInFlight = 2;

// ---- decode, pages of fewer than 1024 / 2D keys (fa_decode.hip): 32768
// elements (64 KB) of K per chunk, i.e. 32768 / D keys.  64 x 4k keys at
// D = 512 (16-key pages, before the streaming kernel took them): 63.8% of
// 8 TB/s; 64 x 16k keys at D = 128, pages of 1-8 keys: 65-67%.
constexpr int kDecChunkElems = 32768;

// ---- split-KV paged prefill (fa_fwd.hip paged_num_splits): no split when the
// block table holds fewer than kSplitMinKeys keys; with fewer workgroups (row
// tiles, at least one per sequence, x KV heads) than CUs
// max(ceil(keys / kSplitMaxRangeKeys), ceil(CUs / workgroups)) ranges (twice the
// CUs for tiles of few rows), but none shorter than kSplitMinRangeKeys and at
// most kMaxSplits; from one workgroup per CU on one range, or two (below).
// Evidence (2 sequences, 32 / 8 heads, D = 128, time per call in ms for
// 1 / 4 / 8 / 16 splits): 32k-key prefix + 128 tokens 0.955 / 0.277 / 0.171 /
// 0.192 (this rule: 8); 16k + 128: 0.487 / 0.153 / 0.104 / 0.128 (8);
// 32k + 512: 0.994 / 0.593 / 0.634 / 0.729 (5); 8k + 64: 0.252 / 0.087 /
// 0.062 / 0.080 (8).  The former rule (2 x CUs / workgroups ranges of at
// least 2048 keys) chose 16, 8, 4 and 4.
// Batches of one-token sequences, 1-8k keys (us for 1 / 2 / 4 / 8): 64 of them
// 224 / 235 / 248 / 295 (this rule 1; counting only the token rows' tiles it
// was 8), 16 of them 110 / 75 / 70 / 81 (4; was 8), 16 of four tokens after
// 2-16k keys 198 / 144 / 120 / 134 (4; was 16); 47 of them with a 512-token
// chunk, 64 heads 167 / 198 / 229 / 302 (1; was 2); 30 with two chunks, table
// of 16k keys 162 / 150 / 187 / 243 (2; was 3).
// From one workgroup per CU on (us for 1 / 2 / 3 ranges).  Full tiles: 16 chunks of
// 198-396 tokens, 16 / 16 heads 173 / 213 / 223; 6 of 352-704 after 3-12k keys, 32 / 8
// 437 / 458 / 458; 8 of 457-914, D = 256 190 / 218 / 225; 3 of 1378 after 6-25k, 16 / 2
// 608 / 657 / 636; none is faster split.  One-token sequences alone, 1-8k keys, D = 128:
// 20 of 16 / 16 heads 45 / 55 / 57 (1.1k keys), 142 / 130 / 127 (4.7k); 43 of 32 / 8
// 149 / 156 / 164.  With a chunk or two among them, tiles up to 1.5 per CU: 37, 32 / 8
// 192 / 137 / 138; 20, 16 / 16 172 / 140 / 136; 32, 32 / 8 157 / 119 / 126; 16 of 1.5k
// keys in a table of 4.5k 42 / 49 / 53; D = 256: 34, 32 / 8 525 / 435 / 427.  Above: 42,
// 64 / 8 (576) 312 / 378 / 389.  D = 64, two workgroups a CU: 35, 64 / 8, table of 4.1k 85 /
// 68 / 59; one-token sequences alone, 18 of 5.3k, 16 / 16 121 / 99 / 88; 46 of 7.8k, 64 / 8
// 187 / 172 / 165; 42 of 1.2k, 64 / 8 in a table of 32k 31 / 39 / 37; more rows, 52 and 26
// chunks, 32 / 8 (624 tiles) 68 / 87 / 92; full tiles, 7 chunks of 216 after 8-32k, 28 / 4
// 497, 396 in four ranges, 20 of 65 after 1-4k, 32 / 8 79 / 86.
constexpr int kSplitMinKeys = 4096;
constexpr int kSplitMinRangeKeys = 1024;
constexpr int kSplitMaxRangeKeys = 8192;
constexpr int kMaxSplits = 64;
// Key ranges one after the other instead of side by side (fa_fwd.hip
// split_range_slots) from this many new tokens a sequence on (us, side by side / in
// turn, 2 ranges unless noted): one of 2146 tokens after 2k keys, 16 / 2 heads
// 136 / 85; one of 1213, D = 256 158 / 106; one of 1051 after 13k, 32 / 8 218 / 189;
// two of 1517 after 1.5k, 28 / 4 216 / 176; three of 703, 16 / 2 125 / 110; with fewer or
// in longer ranges, two of 808 after 5-22k, 16 / 2, 3 ranges 263 / 292; seven of 579 after
// 7-29k, 4 ranges 600 / 656; one of 507 after 15k, 28 / 4, D = 64, 6 112 / 122; three of 344 after 28k,
// 16 / 16, D = 64, 4 ranges 197 / 221; 12 of 210, 16 / 16, D = 64 159 / 175; 21 of 35
// after 10k, 28 / 4, 4 ranges 156 / 193.
constexpr int64_t kSplitByRangeTokens = 512;

// ---- workgroup order of the paged kernels (fa_fwd.hip paged_order,
// find_sequence).  Up to kPagedTileOrderRounds rounds of (tile, KV head, key range)
// workgroups (CUs x workgroups per CU is one) every tile goes by its own reach, up
// to kPagedTileOrderRoundsShared where (KV head, key range) pairs are no multiple
// of the 8 XCDs, which then share them and their K / V anyway; above, whole
// sequences by their reach where histories differ, else in their own order.
// Evidence (us, same box, D = 128 unless noted, against combo-major ranges of ids
// with sequences by history): 8 prompts of 512-4096 tokens, 16 / 2 heads 281 -> 262;
// 8 of 300-2048, 16 / 16 heads 110 -> 105; 8 of 512-2048, 28 / 4 heads, D = 64
// 149 -> 143; the same after up to 4k keys, 16 / 2 heads, D = 256 988 -> 680; 2
// chunks + 30 one-token sequences, 2 ranges 158 -> 150.  The tile order loses the
// K / V reuse in the L2, so it stops at two rounds: 27 prompts of 356-712 tokens,
// 32 / 8 heads (1900 workgroups) 140 by sequence, 153 by tile; 8 of 512-4096 (2400)
// 467 and 474.  Between two and 3.3 rounds, over 69 drawn batches with 2 or 4 KV heads
// the tile order up to three rounds is 2.5% faster than up to two (three prompts of
// 1491-1884 tokens, 28 / 4 90.4 -> 87.0, where combo-major took 84; 23 of 313-626, 16 / 2
// 57.7 -> 49.8; the most it loses is 8%, four chunks of 614-1228 among 25 one-token
// sequences, 28 / 4).  Over 70 with 8 or 16 it gains nothing and costs up to 19% (four of
// 183-366, 64 / 8, D = 256 37.9 by sequence, 45.2 by tile).
// The search for a workgroup's tile takes 0.5-1 us, so a single sequence and two
// prompts below kPagedOrderPairKeys go without it (searched / by sequence: one of
// 535-1070 tokens, 64 / 8 heads, D = 256 47.3 / 45.4; two of 434-868, 64 / 8 37.4 /
// 35.8), while two longer ones or three and more gain by it (two of 941-1882, 16 / 16,
// D = 64 41.5 / 47.2; 11 of 411-822, 16 / 2 41.2 / 48.0; 5 of 169-338, 64 / 8, D = 64
// 21.5 / 24.5), as do two histories (two of 100-200 after 8-31k keys, 28 / 4, 6 ranges
// 117 / 144).  Two rounds are 1024 workgroups at D = 64, which runs two a CU (14 of
// 185-370, 28 / 4 27.1 by tile, 29.0 by sequence; 4 of 736-1472, 16 / 16 33.9, 40.4).
constexpr int kPagedOrderPairKeys = 1024;
constexpr int kPagedTileOrderRounds = 2;
constexpr int kPagedTileOrderRoundsShared = 3;

// ---- paged tiles of at most 32 rows (fa_fwd.hip run_paged_tile, paged_few_rows):
// their keys are split over the workgroup's waves from kPagedFewMinKeys keys (of
// the tile's range; head_dim 256 kPagedFewMinKeys256) on, in batches of at most kPagedFewMaxTiles full tiles per
// sequence.  Evidence (us, one-token sequences, row-tile / key-split core, one
// range): D = 128, 32 / 8 heads, 16 sequences of 512 / 2048 / 8192 keys 19.7 / 18.1,
// 48.7 / 31.1, 190 / 125; 128 of 128 / 256 / 512 / 2048 keys 33.2 / 38.5, 45.1 / 47.0,
// 67.5 / 58.5, 228 / 196.  D = 64, 16 of 1024 / 8192 23.8 / 17.3, 122 / 65; 128 of 256 /
// 512 24.3 / 24.3, 34.0 / 31.8.  D = 256 (fewer workgroups than CUs only): 16 of 1024 /
// 8192 45.5 / 32.3, 288 / 210; 32 (256 workgroups) 48.7 / 49.5, 347 / 381; 64 101 / 105,
// 682 / 747.  Mixed with chunks, D = 128: 3 sequences, one of a token, 32 / 8 heads, 644
// rows a sequence, 7k keys 75 / 65; D = 256: 39 of 3-9k keys, 20 of them chunks of 116
// tokens 767 / 687; 19 of 8-16k, 16 / 16 heads, 109 rows a sequence 888 / 816; 18, 63
// rows a sequence 610 / 643.
constexpr int kPagedFewMinKeys = 384;
constexpr int kPagedFewMinKeys256 = 128;  // 16 sequences of 128 / 256 keys 15.3 / 14.6, 20.0 / 16.8
constexpr int kPagedFewMaxTiles = 8;

}  // namespace tiles
}  // namespace fa
