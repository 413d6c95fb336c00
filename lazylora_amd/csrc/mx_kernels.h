// Kernel argument blocks and launch helpers shared by the .hip translation units.
// Host-visible; no torch types.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mx {

// ---------------------------------------------------------------- forward products
enum FwdMode : int {
  kFwdPlain = 0,   // y[row, n] = A[row] . W[n]
  kFwdGateUp = 1,  // act = GLU(A . W1^T, A . W3^T) -> two-term e4m3 act (+ optional fp32 gate|up)
  kFwdDown = 2,    // y_pair[p, n] = tw[p] * (act[p] . W2[n])
};

struct FwdArgs {
  const uint8_t* wp0;  // packed W (or W1 for kFwdGateUp), expert-major
  const uint8_t* ws0;
  const uint8_t* wp1;  // W3 for kFwdGateUp
  const uint8_t* ws1;
  long long wp_estride;  // bytes between experts in wp*
  long long ws_estride;  // bytes between experts in ws*
  int R, K;              // each W is [R, K]
  // A operand: two-term e4m3 activations in the AT layout, one block of at_tile_bytes(K)
  // per work tile (tile t of the list below)
  const uint8_t* a_tiles;
  // kFwdGateUp, one-tile work-groups: A in the XT layout instead; pair row p reads row
  // row_token[p] of a_rows (rows a_row_bytes apart), a tile's unused slots row a_zero_row. Its
  // grouped work-groups read a_tiles, of which only the large buckets' tiles need be written.
  const uint8_t* a_rows;
  long long a_row_bytes;
  int a_zero_row;
  // work: tiles[t] = {expert, first row, row count <= 16, 0}; null = dense, rows 16t.. of M
  const int4* tiles;
  const int* n_tiles;
  int M;  // rows: all of them, or with a tile list at most
  int n_ct;  // column tiles per row tile
  // outputs
  float* y;
  long long ldy;
  const int* y_rows;     // output row of each row (null: the row itself; top-1 routing writes tokens)
  const float* row_w;    // kFwdDown: combine weight per row
  uint8_t* q_tiles;      // kFwdGateUp: act in the AT layout with K = R (= F), same tiles
  float* save;           // kFwdGateUp: [rows, 2R] gate | up in fp32, or null
  int act_kind;
  // token of each pair row (XT gather); with LoRA, gate|up of row p gain
  // lora_delta[row_token[p], 0:2R) before the GLU
  const int* row_token;
  const float* lora_delta;  // [tokens, 2R] fp32, or null
  // kFwdGateUp: the third term of x (X3 layout, rows as a_rows, x3_row_bytes apart), or null, and
  // the call-wide flag (non-zero: some block has a third term; zero: the products skip it all)
  const uint8_t* x3;
  long long x3_row_bytes;
  const int* x3_any;
  // Bucket split (with a tile list and K a multiple of 512): the tiles of small buckets
  // (indices into `tiles`) take the one-row-tile work-groups; the large buckets' tiles, in groups
  // ({expert, first tile, tiles, 0}), work-groups that share each column tile's weights over the
  // group's row tiles. Null small_tiles: every tile takes the first shape.
  const int* small_tiles;
  const int* n_small;
  const int4* wgroups;
  const int* n_wgroups;
  bool all_wide;  // every bucket is a large one (routed with wide_min 1): no one-tile items
  int* wcounter;  // the wide-group launch's work queue: 2 ints, zero before the first launch (queue_next)
  // Forward layout (launch_forward_layout) of W (W1 for kFwdGateUp) and W3, or null: the
  // one-tile fast path's work-groups then read their weight codes and scales from it in whole
  // lines, the wide large-bucket work-groups their codes (the general path, the wide groups'
  // scales and the rare third-term pass always read wp* / ws*).
  const uint8_t* fl0;
  const uint8_t* fl1;
  long long fl_estride;  // bytes between experts in fl*
};

// Forward layout of E stacked packed [R, K] matrices (K a multiple of 512) and their E8M0 scales
// [R, K / 32], per expert forward_layout_bytes(R, K) bytes, nrg = ceil(R / 16) row groups and
// nsc = K / 512 super-chunks: codes, the 4 KiB at (rg * nsc + c) * 4096 hold super-chunk c of the
// 16 rows 16 rg .., MFMA q's operand block at q * 1024, lane l's 16 bytes (MX block
// 4 (l / 16) + q of row 16 rg + l % 16) at l * 16; then scales, the 256 B at
// nrg * nsc * 4096 + (rg * nsc + c) * 256 hold lane l's scale dword (blocks 4 (l / 16) .. + 3 of
// super-chunk c of row 16 rg + l % 16) at 4 l. Rows past R repeat row R - 1.
long long forward_layout_bytes(int R, int K);
hipError_t launch_forward_layout(const uint8_t* packed, const uint8_t* scales, uint8_t* out, int E, int R, int K,
                                 hipStream_t s);

// ---------------------------------------------------------------- transposed products
enum BwdMode : int {
  kBwdPlain = 0,   // y[row, c] (+)= sum_r A[row, r] W[r, c]
  kBwdDownT = 1,   // h = g . W2 -> grad_w partials, GLU backward -> bf16 d_gate | d_up
  kBwdGateUpT = 2, // y_pair[p, c] = [d_gate | d_up] . [W1 ; W3]
};

struct BwdArgs {
  const uint8_t* wp0;
  const uint8_t* ws0;
  const uint8_t* wp1;  // second row segment (W3), or null
  const uint8_t* ws1;
  long long wp_estride;
  long long ws_estride;
  int nseg;      // 1 or 2 row segments
  int R, C;      // each segment is [R, C]
  const uint16_t* a_hi;  // bf16 [rows, lda], contraction index in [0, nseg*R), zero padded
  const uint16_t* a_lo;
  long long lda;
  const int* a_row_map;
  const int4* tiles;
  const int* n_tiles;
  int M;  // rows: all of them, or with a tile list at most
  int n_ct;  // column tiles of kBwdColsPerTile
  float* y;
  long long ldy;
  int accumulate;
  // kBwdDownT
  const float* row_w;
  const float* saved;  // [rows, 2C] gate | up
  int act_kind;
  uint16_t* d_hi;      // [rows, 2C]
  uint16_t* d_lo;
  float* gw_part;      // [rows, n_ct]
  // kBwdDownT with LoRA: h = g . W2 of row p gains lora_rq[a_row_map[p], 0:C) (the down
  // adapter's A^T q of the row's token), so both the GLU backward and grad_w see it
  const float* lora_rq;  // [tokens, C] fp32, or null
  // Bucket split, as in FwdArgs: small-bucket tiles take one-tile work-groups, large-bucket
  // groups work-groups that reuse each decoded weight slab for all of the group's tiles.
  const int* small_tiles;
  const int* n_small;
  const int4* groups;
  const int* n_groups;
  // Backward layout (launch_backward_layout) of each row segment (W; W1 and W3 for two), or
  // null: the work-groups of kBwdDownT / kBwdGateUpT then read it instead of wp / ws. Needs
  // backward_layout_ok(R, C).
  const uint8_t* bl0;
  const uint8_t* bl1;
  long long bl_estride;  // bytes per expert: backward_layout_bytes(R, C)
};

constexpr int kFwdRowsPerTile = 16;
constexpr int kGroupTiles = 4;     // row tiles of one large-bucket group
constexpr int kWideGroupTiles = 8;  // row tiles of one wide group (the large-bucket forward)
// Experts with at least this many tiles take the large-bucket path: usually four; where the buckets average
// kFewerMinRows rows, two in the forward (a wide item of two tiles reads the weights once and takes little
// longer than a one-tile item) and three in the transposed products (whose items always compute four
// tiles). From the checkpoint layout the forward then has no one-tile items at all: a launch
// of their own for the few short buckets costs more than their wide items (3584 / 3072, 64 experts, top-8,
// whole forward, us, with them then without: 20 rows per bucket 375 / 314, 64 rows 419 / 412; Zipf 20 rows
// 363 / 349, 64 rows 538 / 506; 7168 / 2048, 128 experts, 16 rows 748 / 699). With a forward layout both
// kinds share one launch, and the one-tile items stay (Zipf 64 rows 430 / 440). 128 tokens, top-16 of 64
// experts (32 rows on average, 3584 / 3072, checkpoint layout), four everywhere, then this: gate/up 0.33 ->
// 0.24 ms, down 0.18 -> 0.13, W1 | W3 transposed 0.38 -> 0.29, W2 0.20 -> 0.20.
constexpr int kLargeMinTiles = 4, kWideMinTiles = 2, kGroupMinTiles = 3;
constexpr int kFewerMinRows = 12;
constexpr long long kFewerMinWeights = 1 << 20;  // elements per matrix: below, both shapes are a launch's latency
// Short buckets (none of kLargeMinTiles tiles) are another matter: a wide item waits out the same serial
// quarters whether it has one tile or three, while one-tile items of one expert run side by side. Wide items
// pay only from a number of weight readings saved: the tiles past each expert's first x the eight-column
// items of a tile (both products) above kJudgeItems, with a forward layout kJudgeItemsLayout (one and a
// half to two for each CU). Whole forward, us, as one-tile items / wide, uniform routing: 7168 / 2048 from the
// checkpoint layout, 16 experts of 16 rows (158 items saved) 143 / 156, of 32 (510) 193 / 167, 32 of 20 (563)
// 270 / 218; forward layout, 16 of 16 121 / 140, of 32 187 / 148; 3584 / 3072, checkpoint layout, 16 of 24 (304)
// 119 / 137, 64 of 12 (152) 264 / 290, of 16 (547) 329 / 297; 2048 / 1024, 32 of 24 (256) 64 / 83, 128 of 20
// (820) 178 / 158. The routing's counts decide it on the device unless some bucket must be of four tiles (P >
// 48 E). From the checkpoint layout, where leaving both kinds possible costs an empty launch of each
// product (5 us), the wide items are taken for sure where uniform routing would save more than kSureItems,
// its tiles past the first being about (P - 11 E) / 12.
constexpr int kJudgeItems = 480, kJudgeItemsLayout = 390;
constexpr int kSureItems = 420;
// The transposed products likewise: a group item of three tiles decodes once but takes longer than a one-tile
// item, so a few of them only lengthen a launch whose other items are done after one round. They pay where
// some bucket has such items anyway, or from that many experts of three tiles x the items above. Both
// products, us, as one-tile items / groups, 7168 / 2048, checkpoint layout, uniform routing: 64 experts of 24
// rows (3 of three tiles) 556 / 702, of 32 (29) 759 / 698; 32 of 32 (14) 436 / 436, 16 of 32 (7) 330 / 415;
// 3584 / 3072: 32 of 32 338 / 435, 64 of 32 566 / 461; 2048 / 1024: 64 of 32 147 / 177, 128 of 32 (58) 250 / 234.
constexpr int kJudgeGroupItems = 400;
constexpr int kFwdColsPerTile = 64;  // kFwdPlain / kFwdDown; kFwdGateUp covers 32 features
constexpr int kBwdColsPerTile = 256;  // output columns of one transposed-product wave

// Whether launch_fwd splits a routed product over W [R, K] into small-bucket and large-bucket
// work-groups: the large-bucket shape needs the fast path (K a multiple of 512, one buffer
// resource addressing the whole matrix). Without the split every tile takes the one-tile
// work-groups, whose gate/up product reads the token-major (XT) rows of x for every tile.
bool fwd_bucket_split(int R, int K);
// Whether the routed product `a` (of max_tiles tiles at most) runs as split-K items of one tile x 64
// weight rows, whatever its buckets. Its gate/up product then reads the token-major (XT) rows of x for
// every tile. The line: while its eight-column-tile items (at most rows * ceil(n_ct / 8)) would leave
// half of the 256 CUs without one and, from the checkpoint layout, while the split work-groups are at
// most three per CU: the one-tile items take one pass over the weights whatever the rows, the split ones
// a round more every 256. Measured (us, the product with x's quantisation, as one-tile items / split, pairs
// of distinct experts), gate/up of 7168 / 2048 from the checkpoint layout: 8 pairs (two rounds) 55 / 44, 9 to
// 12 (three) 56 / 57 to 58 / 59, 14 (four) 59 / 72, 16 62 / 75; its down product: 8 pairs 20 / 22, 10 30 / 30;
// gate/up of 3584 / 3072: 8 (three) 39 / 40, 10 (four) 40 / 48; its down product: 9 (two) 24 / 19, 13 (three)
// 25 / 25, 16 (four) 26 / 31. From the forward layout, whose one-tile items are eight waves: gate/up of 7168 / 2048
// 8 pairs 63 / 39, 16 68 / 64, 17 68 / 66.
bool fwd_few_rows(const FwdArgs& a, int mode, int max_tiles);
hipError_t launch_fwd(const FwdArgs& a, int mode, int max_tiles, hipStream_t s);
hipError_t launch_bwd(const BwdArgs& a, int mode, int max_tiles, hipStream_t s);
// The dense transposed product (kBwdPlain) straight from the fp32 rows x [M, R] (4-byte aligned),
// the contraction split over the waves of a work-group: for up to kBwdFewRows rows. a_hi, a_lo and
// lda are not used.
constexpr int kBwdFewRows = 256;
hipError_t launch_bwd_few(const BwdArgs& a, const float* x, hipStream_t s);

// Backward layout: a load-time copy of E stacked MXFP4 matrices [R, C] (codes [R, C/2], E8M0
// scales [R, C/32]) for the one-tile transposed products. Per expert, blocks (32-row step st,
// 256-column stripe c) in order st * (C / 256) + c: each block's 4 KiB of codes in the order the
// lanes of the stripe's wave load them (lane 16g + n, load u: bytes 8n .. 8n + 7 of rows 8g + 2u
// and 8g + 2u + 1), then, after every block's codes, 256 B of scales per block (8 bytes per lane
// pair: the scale bytes of rows 8g .. 8g + 7 for the pair's MX block). R % 32 == 0, C % 256 == 0.
bool backward_layout_ok(int R, int C);
long long backward_layout_bytes(int R, int C);  // per expert; 0 unless backward_layout_ok(R, C)
hipError_t launch_backward_layout(const uint8_t* packed, const uint8_t* scales, uint8_t* out, int E, int R, int C,
                                  hipStream_t s);

// ---------------------------------------------------------------- elementwise / routing
// Two-term quantisation of activation rows into the AT layout of the work tiles. Tile t slot i
// holds row tiles[t].y + i (through row_map when given: the token of a (token, slot) pair);
// with tiles == null the tiles are dense: tile t holds rows 16t.. of `rows`. Unused slots get
// zeros. max_tiles bounds the grid; the live tile count is read from n_tiles on the device.
// xt (with row_map): the XT rows of x written by launch_quant_rows on the same stream; when that
// call wrote them (it got no meta, or meta says some bucket is small) the tiles are copied from
// them instead of quantising x again (the same bytes). x3 (with row_map): where the tiles are quantised
// from x, also the X3 rows of their tokens (launch_quant_rows writes them otherwise). x3_any
// (with x3): set to non-zero when some block has a third term (it must be zero before the call).
// groups (the routing's wide groups; n_groups on the device): only their tiles, found through the
// list by a resident grid instead of one work-group per tile and chunk; the others are left untouched.
hipError_t launch_quant_tiles(const void* x, int x_bf16, long long ldx, int rows, int K, const int4* tiles,
                              const int* n_tiles, int max_tiles, const int* row_map, const uint8_t* xt,
                              const int* meta, uint8_t* out, uint8_t* x3, int* x3_any, hipStream_t s,
                              const int4* groups = nullptr, const int* n_groups = nullptr);
// Rows 0 .. rows - 1 of x into the XT layout (xt_row_bytes(K) per row), followed by zero rows
// up to xt_rows(rows): row `rows` is the all-zero row a tile's unused slots gather. x3 (or null):
// the third term of the flagged blocks in the X3 layout (x3_row_bytes(K) per row; rows < rows).
// With meta saying every bucket is large the call writes nothing (launch_quant_tiles writes X3).
inline long long xt_rows(int rows) { return ((long long)rows + 16) / 16 * 16; }
hipError_t launch_quant_rows(const void* x, int x_bf16, long long ldx, int rows, int K, const int* meta, uint8_t* out,
                             uint8_t* x3, int* x3_any, hipStream_t s);
hipError_t launch_split_bf16(const float* x, long long ldx, int rows, int K, int Kpad, uint16_t* hi,
                             uint16_t* lo, hipStream_t s);
hipError_t launch_dequant(void* out, int out_bf16, const uint8_t* packed, const uint8_t* scales, int K, int R,
                          hipStream_t s);
// Routing: per-expert counts, scan, the tile list (tiles[t] = {expert, first pair row, rows, 0}),
// the forward's large buckets (experts with at least wide_min tiles) as wide groups of up to
// kWideGroupTiles tiles ({expert, first tile, tiles, 0}, the full ones first) and its other tiles'
// indices (small_tiles), the transposed products' large buckets (at least group_min tiles) as groups
// of up to kGroupTiles and their other tiles' indices (bsmall_tiles), meta = {tiles, flags (bit 0:
// an id outside [0, E)), small tiles (forward), groups, wide groups, full wide groups, third term
// present (set by the quantisers), small tiles (transposed), then the work queues (2 ints each) of
// the wide-group launches of the forward gate/up and down products, the runs of the partial wide groups
// when each is cut into two or four (at most its tiles), -, -} (16 ints, all zeroed or written
// here), and the pair maps. judge (>= 0): where no expert has kLargeMinTiles tiles and no more than `judge`
// tiles lie past an expert's first, kLargeMinTiles stands for wide_min; judge_groups (>= 0): where no expert
// has kLargeMinTiles tiles and no more than that many have kGroupMinTiles, kLargeMinTiles stands for group_min.
hipError_t launch_route(const void* topk_idx, int idx64, const float* topk_w, int N, int k, int E, int* counts,
                        int* offsets, int* cursor, int4* tiles, int* small_tiles, int* bsmall_tiles, int4* groups,
                        int4* wgroups, int* meta, int wide_min, int group_min, int judge, int judge_groups,
                        int* pair_token, float* pair_w, int* pair_of, hipStream_t s);
hipError_t launch_combine(float* out, const float* ypair, long long ldy, const int* pair_of, int N, int k,
                          int D, hipStream_t s);
// Top-1 routing (the down product writes token rows itself): zeros into the rows of tokens with no
// pair (pair_of[t] < 0, an id outside [0, E)).
hipError_t launch_zero_unrouted(float* out, long long ldo, int D, const int* pair_of, int N, hipStream_t s);
hipError_t launch_combine_bwd(float* grad_h, float* grad_w, const float* dxpair, long long ldy,
                              const float* gw_part, int n_ct, const int* pair_of, int N, int k, int D,
                              hipStream_t s);
hipError_t launch_zero(void* p, size_t bytes, hipStream_t s);
// ---------------------------------------------------------------- LoRA coupling
// Encodings of the row-major matrices the LoRA kernels read.
enum LoraSrc : int {
  kLoraF32 = 0,   // p0: fp32 [rows, ld]
  kLoraBF16 = 1,  // p0: bf16 [rows, ld]
  kLoraGLU = 2,   // p0: saved fp32 gate | up [rows, 2F]; element (row, c) = GLU(gate[c], up[c])
  kLoraHiLo = 3,  // p0 / p1: bf16 hi and lo [rows, ld]; element = hi + lo
};
struct LoraMat {
  int kind;
  const void* p0;
  const void* p1;
  long long ld;
  int F, act_kind;  // kLoraGLU
};
// Small dense factor M of a LoRA adapter, addressed as M(j, k) (j < rank): j-major means
// M[j * ld + k] (lora_A [r, in]), k-major means M[k * ld + j] (lora_B [out, r]).
struct LoraFactor {
  const float* m;
  long long ld;
  int kmajor;
  float scale;
};

constexpr int kLoraMaxRank = 32;

// Destination of an outer-product gradient: element (j, c) of segment s goes to
// p[s][kmajor[s] ? c * ld[s] + j : j * ld[s] + c] times scale[s].
struct LoraOuterDst {
  float* p[2];
  long long ld[2];
  int kmajor[2];
  float scale[2];
  int split_j;  // coefficients j >= split_j go to p[1] (index minus split_j), or 0
};

// One job of a LoRA pass (launch_lora_pass), over a source of `rows` rows (tokens, or pairs in
// bucket order; rows at or past *rows_dev, when given, are skipped) in nseg <= 2 segments of K
// columns (a multiple of 32), segment s starting at source column koff[s]:
//   kLoraRowDot: partial row dots of out[row, s*r + j] = sum_k src(row, koff_s + k) f_s(j, k)
//     (nseg 2), or of out[row, n*r + j] with factor f_n on the one segment (nseg 1, n < nfac <= 2);
//   kLoraOuter: partial column sums of G[j, s*K + c] = sum over q < rows of
//     row_w[q] * coef[crow(q), coff_s + j] * src(row(q), koff_s + c), j < m <= 64: with row_of,
//     q runs over (token, slot) pairs in token order, row(q) = row_of[q] (skipped when negative)
//     and crow(q) = q / k, so the sums do not depend on the bucket order; else row(q) = crow(q)
//     = q. row_w null: 1.
// Factor scales are not applied here (the finish applies them).
//   kLoraRowOuter: both, over one two-term (hi + lo) pair source with row_of (nseg segments, m = r <=
//     16 coefficients per segment, factor f_s on segment s): each element is read once.
enum LoraJobType : int { kLoraRowDot = 0, kLoraOuter = 1, kLoraRowOuter = 2 };
struct LoraPassJob {
  int type;
  LoraMat src;
  int rows;
  const int* rows_dev;
  int nseg, K;
  int koff[2];
  int r;
  int nfac;
  LoraFactor f[2];
  const float* coef;
  long long ldc;
  int coff[2];
  const int* row_of;
  int k;
  const float* row_w;
  int m;
};
// Partials a pass job leaves for its finish: `count` slices (row dots: [count, rows, m_out]) or
// row chunks (outer products: [count, m, nseg * K]); a fused job leaves its outer-product
// partials in p and its row-dot partials in p2 (count2 slices of [rows, nseg * r]).
struct LoraPartial {
  const float* p;
  int count;
  const float* p2;
  int count2;
};
size_t lora_pass_partial_floats(const LoraPassJob* jobs, int n);
// Up to 4 jobs in one launch; parts[i] receives job i's partials (inside `partial`, which holds
// lora_pass_partial_floats(jobs, n) floats).
hipError_t launch_lora_pass(const LoraPassJob* jobs, int n, float* partial, LoraPartial* parts, hipStream_t s);

// One job of launch_lora_finish: the partials added in a fixed order.
//   kLoraFinCoef: value (row, j) = scale[j / r] * sum over slices of the row-dot partials
//     ([count, prow, m]); with pair_of, rows are pairs and out[t, j] = sum over token t's slots, in
//     slot order, of (topk_w[t, s] or 1) * value(pair_of[t, s], j); else out[t, j] = value(t, j);
//     out is [ntok, m].
//   kLoraFinOuter: G[j, c] = sum over chunks of the outer partials ([count, om, Ctot]), written
//     through dst; segments by column (Kseg > 0: s = c / Kseg) or by j (dst.split_j).
enum LoraFinType : int { kLoraFinCoef = 0, kLoraFinOuter = 1 };
struct LoraFinishJob {
  int type;
  LoraPartial part;
  int prow, m, r;
  float scale[2];
  const int* pair_of;
  const float* topk_w;
  int k, ntok;
  float* out;
  int om, Ctot, Kseg;
  LoraOuterDst dst;
};
hipError_t launch_lora_finish(const LoraFinishJob* jobs, int n, hipStream_t s);

// out[t, c] = ef_s.scale * sum_{j < r} coef[t, ecoff_s + j] * ef_s(j, c - s*Cseg) for t < ntok,
// c < Cexp (multiples of 4), segment s = c / Cseg (Cseg 0 or >= Cexp: one segment; two segments
// share the factor layout); coef rows hold m floats, out rows are ldo apart. With part (row-dot
// partials [count, ntok, m] of tokens), the coefficient rows are first reduced from them
// (coef[t, j] = part_scale[j / r] * the slices' sum, added in slice order) and written to coef.
hipError_t launch_lora_expand(float* coef, int m, int ntok, int r, float* out, long long ldo, int Cexp,
                              int Cseg, const LoraFactor* ef, const int* ecoff, hipStream_t s,
                              const LoraPartial* part = nullptr, const float* part_scale = nullptr);

// out[t, c] = sum over token t's slots, in slot order, of rows[pair_of[t, s], c] (skipped when
// negative) + sum over segments s < nseg of f_s.scale * sum_{j < r} coef[t, s*r + j] f_s(j, c);
// with grad_w, also grad_w[t, s] = sum over ct < n_ct of gw_part[pair, ct] (the backward combine).
hipError_t launch_lora_combine(float* out, const float* rows, long long ldy, const int* pair_of, int N, int k, int D,
                               const float* coef, int r, int nseg, const LoraFactor* f, float* grad_w,
                               const float* gw_part, int n_ct, hipStream_t s);

// Router selection (sigmoid, bias, top-k, renormalise, scale), one wave per token.
hipError_t launch_router_topk(long long* topk_idx, float* topk_w, const float* logits, const float* bias, int N,
                              int E, int top_k, float scale, int renormalize, hipStream_t s);
hipError_t launch_router_topk_bwd(float* grad_logits, const long long* topk_idx, const float* grad_w,
                                  const float* logits, int N, int E, int top_k, float scale, int renormalize,
                                  hipStream_t s);


}  // namespace mx
