// Internal launch interface between the kernel files (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace qlin {

struct W8GemvArgs {
  const int8_t* w;     // [n, k] int8
  const uint16_t* s;   // [n, k / 64] BF16 scales
  const uint16_t* bias;  // [n] BF16 or nullptr
  const uint16_t* x;   // [k] BF16
  uint16_t* y;         // [n] BF16
  int n;
  int k;
};

// One GEMV of a grouped launch; block_begin is the first block index of the
// launch that works on it (descriptors sorted by block_begin) and each of its
// blocks covers rows_per_block rows (a multiple of 4 waves x 8-row tasks).
struct W8GroupDesc {
  const int8_t* w;
  const uint16_t* s;
  const uint16_t* bias;
  const uint16_t* x;
  uint16_t* y;
  int n;
  int k;
  int block_begin;
  int rows_per_block;
};

// A small grouped launch: descriptors passed by value as kernel arguments.
constexpr int kSmallGroupMax = 8;
struct W8SmallGroup {
  W8GroupDesc d[kSmallGroupMax];
  int count;
};

struct Bf16GemvArgs {
  const uint16_t* w;     // [n, k] BF16
  const uint16_t* bias;  // [n] BF16 or nullptr
  const uint16_t* x;     // [k] BF16
  uint16_t* y;           // [n] BF16
  int n;
  int k;
};

// One GEMM Y[m, n] = bf16(sum_k X[m, k] W[n, k] + bias[n]); W is int8 with
// BF16 group-64 scales s (W8A16) or BF16 with s unused.
struct GemmArgs {
  const void* w;         // [n, k] int8 or BF16
  const uint16_t* s;     // [n, k / 64] BF16 scales (W8A16 only)
  const uint16_t* bias;  // [n] BF16 or nullptr
  const uint16_t* x;     // [m, k] BF16
  uint16_t* y;           // [m, n] BF16
  int m;
  int n;
  int k;
};

// Skinny GEMM for a few tokens (m <= kSkinnyMaxTokens) and long K: each
// workgroup streams 32 weight rows of one GEMM for 32 tokens, its waves
// splitting K.  Up to kSkinnyMaxDescs GEMMs per launch (each on its own x and
// y); block_begin is set by layout_skinny.
constexpr int kSkinnyMaxTokens = 128;
constexpr int kSkinnyMaxDescs = 8;
struct SkinnyDesc {
  const void* w;         // [n, k] int8 or BF16
  const uint16_t* s;     // [n, k / 64] BF16 scales (W8A16 only)
  const uint16_t* bias;  // [n] BF16 or nullptr
  const uint16_t* x;     // [m, k] BF16
  uint16_t* y;           // [m, n] BF16
  int n;
  int k;
  int block_begin;
};
struct SkinnyArgs {
  SkinnyDesc d[kSkinnyMaxDescs];
  int count;
  int m;
};
bool gemm_skinny_supported(const void* w, const uint16_t* x, int m, int n, int k);
// Where the skinny kernel's unsplit launch beats the ring tiles, which may
// split (may_split) or not.
bool gemm_skinny_preferred(bool w8, int m, int n, int k, bool may_split);
// Sets block_begin; returns the workgroups.
int layout_skinny(SkinnyArgs& a);
void launch_gemm_skinny(bool w8, const SkinnyArgs& a, int blocks, int cus, hipStream_t stream);

// MFMA GEMM workgroup tiles (rows x columns of Y).
enum GemmTile {
  kGemmTile128x128 = 0,
  kGemmTile128x64 = 1,
  kGemmTile64x128 = 2,
  kGemmTile64x64 = 3,
  kGemmTile32x128 = 4,
  kGemmTile256x128 = 5,  // 8 waves; grouped plans at M >= 256
  kGemmTileCount = 6,
};

// One GEMM of a grouped launch: its blocks are block_begin ..
// block_begin + tiles_m * tiles_n * splits - 1, each one part (of
// `splits`, split_stages K stages of 64 each) of one output tile of the
// plan's tile size (gemm_grouped_tile_rows x gemm_grouped_tile_cols).  Split tiles hand off through partial (splits FP32 tiles per
// output tile) and counters (one per output tile, zero between launches).
struct GemmGroupDesc {
  const void* w;
  const uint16_t* s;
  const uint16_t* bias;
  const uint16_t* x;
  uint16_t* y;
  int m;
  int n;
  int k;
  int tiles_m;
  int block_begin;
  int splits;
  int split_stages;
  float* partial;
  int* counters;
  // A gate|up pair (never split): w, s, bias are gate_proj, w2, s2, bias2
  // up_proj, both [n / 2, k]; each tile computes half its columns of both and
  // writes bf16(silu(bf16(gate)) * bf16(up)), y being [m, n / 2] (exact_silu,
  // ring only: by silu_mul, as a launch of its own does it, else
  // silu_mul_fast).  Null w2: a plain GEMM.
  const void* w2 = nullptr;
  const uint16_t* s2 = nullptr;
  const uint16_t* bias2 = nullptr;
  // The prefill's q|k|v epilogue (ring tiles of 64 columns, one head of 64 per
  // tile; rope_kind 0: the plain epilogue).  The tile's BF16 rows (bias
  // added, rounded) are, for kind 1, rotated by RoPE (pairs (i, i + 32),
  // the (cos, sin) of position rope_start + row at rope[position * 32 + i])
  // and written to y; kind 2, rotated and written to row rope_start + row of
  // kv_cache ([n / 64 heads][max_seq][64]); kind 3, written to kv_cache
  // unrotated.  Rows at or past max_seq are not written.
  const float2* rope = nullptr;
  uint16_t* kv_cache = nullptr;
  int rope_kind = 0;
  int rope_start = 0;
  int max_seq = 0;
  int exact_silu = 0;
};
// Split-K in the wide-tile grouped launch.  A GEMM whose wide tiles are
// split over K in `parts` parts writes each part's FP32 tile, row-major
// 256 x 128, to partial + (tile * parts + part) * 256 * 128 (tile = m_tile
// + tiles_m * n_tile); a second, reduction launch sums the parts in index
// order, adds the bias and writes BF16 Y.  Its blocks block_begin ..
// block_begin + tiles * 16 - 1 cover the GEMM, 16 rows of a tile each.
struct SplitReduceDesc {
  const float* partial;
  const uint16_t* bias;
  uint16_t* y;
  int m;
  int n;
  int tiles_m;
  int parts;
  int block_begin;
};
constexpr int kSplitReduceRows = 16;  // rows of a tile per reduction block

// XCD placement of a wide-tile plan.  Workgroup b of a launch runs on XCD
// b % 8, and each XCD has its own L2, so a split tile's parts are kept on one
// XCD and its reduction blocks on the same one: the FP32 parts are then
// written to and read back from that XCD's L2.  Both maps are permutations
// of the launches' logical blocks (any permutation gives the same results).
//
// Build options (measured alternatives, off by default; `make EXTRA_DEFS=...`):
// QLIN_WIDE_INKERNEL=1 sums a wide split tile's parts inside the GEMM launch
// (gemm.hip, wide_split_handoff) instead of in the reduction launch, with
// device-coherent (sc1) partial stores and loads, or with QLIN_HANDOFF_FENCE=1
// with plain accesses between agent-scope release and acquire fences, or
// with QLIN_HANDOFF_L2=1 (launches whose map keeps a tile's parts on one
// XCD) with plain accesses through that XCD's L2.
// QLIN_WIDE_DIRECT_A=1 (gemm.hip): the wide tile's X tiles go straight into
// LDS (buffer_load ... lds, two stages ahead into three swizzled buffers).
// QLIN_WIDE_HELP=1: on a mapped launch, every workgroup on an XCD that holds
// split tiles sums their slices once its own unit is done (gemm.hip,
// wide_split_help), so no reduction launch runs.
// QLIN_XCD_MAP=0 places workgroups in logical order.
#ifndef QLIN_XCD_MAP
#define QLIN_XCD_MAP 1
#endif
#ifndef QLIN_WIDE_INKERNEL
#define QLIN_WIDE_INKERNEL 0
#endif
#ifndef QLIN_WIDE_HELP
#define QLIN_WIDE_HELP 0
#endif
// The in-launch hand-off: 4 ints of counters per split tile, at most 32 parts.
constexpr int kWideSplitCounterInts = 4;
constexpr int kWideMaxParts = 32;
constexpr int kXcds = 8;
constexpr int kWideMapBlocks = 256;  // plans with more blocks run unmapped
// The in-launch reduction by the XCD's workgroups: a 128-byte line of
// counters per split tile (arrived parts, next slice, departed workgroups),
// at most kHelpTiles split tiles per XCD.
constexpr int kHelpCounterInts = 32;
constexpr int kHelpTiles = 8;
struct WideBlockMap {
  int mapped = 0;                       // 0: workgroup b runs logical block b
  int help = 0;                         // 1: the launch sums its split tiles itself
  uint8_t logical[kWideMapBlocks] = {};  // workgroup -> logical block
  // help: split tiles (numbered over the launch's split descriptors in
  // order) whose parts run on XCD x, 0xFF: none
  uint8_t help_tiles[kXcds][kHelpTiles] = {};
  // help: workgroup -> its rank among the whole-tile workgroups of its XCD
  // (0xFF: a split part), and their number on each XCD
  uint8_t help_rank[kWideMapBlocks] = {};
  uint8_t help_members[kXcds] = {};
};
constexpr int kReduceSlots = 16;
struct ReduceBlockMap {
  // split tiles per XCD: the reduction launch has kXcds * slots *
  // (256 / kSplitReduceRows) workgroups; 0: unmapped
  int slots = 0;
  uint8_t tile[kXcds][kReduceSlots] = {};  // split tile of slot s on XCD x, 0xFF: none
};
// Places a wide-tile layout (after layout_gemm_group and bind_gemm_group) on
// the XCDs: each split tile's parts on the XCD with the most free workgroups,
// the whole tiles in the rest.  Leaves both maps unmapped when the launch has
// more than kWideMapBlocks blocks, no split tile, or a split tile that fits
// no XCD; *reducers receives the reduction launch's workgroups.
void map_wide_group_to_xcds(const GemmGroupDesc* descs, int count, int blocks, WideBlockMap* gmap,
                            ReduceBlockMap* rmap, int* reducers);

// A grouped launch laid out on the host and passed by value as kernel
// arguments, for callers whose shapes change from call to call (the model's
// prefill at the prompt's length): no descriptor table in device memory.
constexpr int kInlineGroupMax = 8;
struct GemmGroupArgs {
  GemmGroupDesc d[kInlineGroupMax];
  int count;
};
struct SplitReduceArgs {
  SplitReduceDesc d[kInlineGroupMax];
  int count;
};
struct GemmGroupLaunch {
  int tile;
  bool w8;
  int blocks;    // workgroups of the GEMM launch
  int reducers;  // workgroups of the split-K reduction launch (wide tile only)
  GemmGroupArgs g;
  SplitReduceArgs r;
  WideBlockMap gmap;   // wide tile: workgroup -> unit (map_wide_group_to_xcds)
  ReduceBlockMap rmap;
};

// plan.cpp: the layout shared by grouped plans and inline launches.  Sets
// every descriptor's tiles_m, splits, split_stages and block_begin (and
// sorts them, longest units first) for one launch on a device with `cus`
// CUs.  The tile is 256 x 128 once every GEMM has 256 rows or more (with
// `fill`, also only when the group has wide tiles for half the CUs), else
// 64 x 64.  K is split so that no unit is much longer than the group's
// shortest reduction (at least 8 stages), with parts lengthened until the
// units fit the device at once (one per CU on the wide tile, two on 64 x 64);
// with `fill`, for a lone or long-K group of one launch, into at most 4
// parts of at least 14 stages instead.
// Returns the tile; *blocks, *partial_floats and *counters receive the
// launch size and its split-K scratch needs.
// (Only its wide-tile layouts are launched; what it gives 64 x 64 tiles runs on
// the ring, and its parts there are what a lone call's workspace must hold.)
int layout_gemm_group(GemmGroupDesc* descs, int count, int cus, bool fill, int* blocks,
                      size_t* partial_floats, size_t* counters);
// Points the split descriptors at `partial` / `counters` (sizes from
// layout_gemm_group) and writes the wide tile's reduction descriptors to
// reduce (at most count); returns the number of reduction descriptors and
// sets *reducers to the reduction launch's workgroups.
int bind_gemm_group(GemmGroupDesc* descs, int count, int tile, float* partial, int* counters,
                    SplitReduceDesc* reduce, int* reducers);
void launch_gemm_group_inline(const GemmGroupLaunch& l, hipStream_t stream);

// Timeline slots of one workgroup (a plan's timeline launch), in
// 100 MHz s_memrealtime ticks unless noted.
enum PlanStamp {
  kStampEntry = 0,      // first instruction
  kStampLoop = 1,       // first stage in LDS (end of the prologue)
  kStampEpilogue = 2,   // last stage's MFMAs issued (start of the epilogue)
  kStampEnd = 3,        // every thread's stores done
  kStampXcc = 4,        // XCC_ID hardware register (the XCD)
  kStampHwId = 5,       // HW_ID hardware register (CU, SIMD, shader engine)
  kStampUnit = 6,       // logical block | stages << 16 | kind << 24 (0 whole, 1 part, 2 pair)
  kStampCycles = 7,     // s_memtime (shader clock) from entry to end
  kStampStored = 8,     // split part: its FP32 tile stored (in-launch hand-off)
  kStampArrived = 9,    // split part: every part has arrived (or the wait ended)
  kStampReduced = 10,   // split part: its slices summed and stored
  kStampHelp = 11,      // own unit done, the in-launch reduction (map.help) begins
  kStampSlots = 16
};

// gemm_ring.hip: GEMMs whose operands are loaded straight into an LDS ring.
enum RingTile {
  kRingSmall = 0,      // 64 x 32
  kRingSmallLong = 1,  // 64 x 32, K > 1024
  kRingMid2 = 2,       // 64 x 64, two K groups
  kRingMid2Long = 3,   // 64 x 64, two K groups, K > 1024
  kRingMid = 4,        // 64 x 64
  kRingLarge = 5,      // 128 x 64
  kRingPair = 6,       // 64 x 64, pairs only: BF16 two K groups, W8A16 four
  kRingMidDeep = 7,    // 64 x 64, BF16 only: four slots
};
constexpr int kRingMaxParts = 16;
constexpr int kRingMaxSplitTiles = 1024;  // split tiles of a launch (their counters)
struct RingArgs {
  GemmGroupDesc d[kInlineGroupMax];
  const GemmGroupDesc* table;  // device memory, for more than kInlineGroupMax; else null
  int count;
  int blocks;  // units (the grid is rounded up to whole XCD rounds)
};
// Tile, K parts and block_begin of a group (or of one gate|up pair: w2 set, n
// counting both weights) of GEMMs the MFMA path supports; sorts the
// descriptors, longest units first.  heads: the tiles must hold whole heads
// (64 columns, never split: the rope epilogue).  With may_split the group
// needs *partial_floats and *counters (zero between launches) of scratch,
// bound by ring_bind.  Returns the tile; *blocks < 0: too many units.
int ring_layout(bool w8, GemmGroupDesc* d, int count, int cus, bool heads, bool may_split,
                int* blocks, size_t* partial_floats, size_t* counters);
void ring_bind(GemmGroupDesc* d, int count, int tile, float* partial, int* counters);
void launch_gemm_ring(bool w8, const RingArgs& a, int tile, hipStream_t stream);
// The same for a.table's GEMMs (no pair), unit u writing the PlanStamp words
// stamps[u * kStampSlots ..]; those of a hand-off inside the launch stay as they
// are.
void launch_gemm_ring_timeline(bool w8, const RingArgs& a, int tile, unsigned long long* stamps,
                               hipStream_t stream);
// The token counts at which layouts may change, in order (start with 0): every
// tile and limit is in multiples of 32 tokens, so the counts of tiles change
// behind one and the kernel may change at one.
inline int next_layout_tokens(int m, int max_tokens) {
  if (m >= max_tokens) return max_tokens + 1;
  return std::min(m % 32 == 31 ? m + 1 : m + 31, max_tokens);
}
// One GEMM, K whole, on the wide tile or the ring kernel.
void launch_gemm_lone(bool w8, const GemmArgs& a, int cus, hipStream_t stream);

// gemm.hip: gate_proj and up_proj of the same input, then SiLU-mul, as one
// launch of gate|up pair tiles (wide or ring tiles, half their columns of
// each; never split): y[m, n] = bf16(silu(bf16(x gate^T + gate_b)) *
// bf16(x up^T + up_b)), y [m, inter].  Supported when both GEMMs take the MFMA
// path.  exact: the SiLU by silu_mul (the ring tiles), not silu_mul_fast.
bool gate_up_silu_supported(const void* gate_w, const void* up_w, const uint16_t* x, int m,
                            int inter, int hidden);
void launch_gate_up_silu(bool w8, const void* gate_w, const uint16_t* gate_s,
                         const uint16_t* gate_b, const void* up_w, const uint16_t* up_s,
                         const uint16_t* up_b, const uint16_t* x, uint16_t* y, int m, int inter,
                         int hidden, bool exact, int cus, hipStream_t stream);

// The wide-tile grouped launch (`units` blocks over descs) and, when some
// GEMM is split, its reduction launch (`reducers` blocks over rdescs).
void launch_gemm_wide_grouped(bool w8, const GemmGroupDesc* descs, int count, int units,
                              const WideBlockMap& gmap, const SplitReduceDesc* rdescs, int rcount,
                              int reducers, const ReduceBlockMap& rmap, hipStream_t stream);
// The same, each workgroup of the GEMM launch writing 16 timeline words
// (entry, first stage, epilogue, end, XCD, hardware id, unit, shader cycles,
// and a split part's hand-off times) to stamps[16 b ..].
void launch_gemm_wide_grouped_timeline(bool w8, const GemmGroupDesc* descs, int count, int units,
                                       const WideBlockMap& gmap, unsigned long long* stamps,
                                       const SplitReduceDesc* rdescs, int rcount, int reducers,
                                       const ReduceBlockMap& rmap, hipStream_t stream);
// The same for launch_gemm_group_inline's wide-tile launches.
void launch_gemm_wide_grouped_timeline(const GemmGroupLaunch& l, unsigned long long* stamps,
                                       hipStream_t stream);

// gemm.hip (grouped launches use kGemmTile256x128; the others are lone calls')
int gemm_tile_rows(int tile);
int gemm_tile_cols(int tile);
bool gemm_mfma_supported(const void* w, const uint16_t* x, int m, int n, int k);
// Lone GEMMs: the wide tile, not the ring's.
bool gemm_wide_preferred(bool w8, int m, int n, int k, int cus);
void launch_gemm_mfma(int tile, bool w8, const GemmArgs& a, hipStream_t stream);

// gemv.hip
bool w8a16_gemv_fast_supported(const int8_t* w, const uint16_t* x, int k);
void launch_w8a16_gemv_fast(const W8GemvArgs& a, hipStream_t stream);
void launch_w8a16_linear_generic(const int8_t* w, const uint16_t* s, int group_size,
                                 const uint16_t* bias, const uint16_t* x, uint16_t* y,
                                 int tokens, int n, int k, hipStream_t stream);
bool bf16_gemv_fast_supported(const uint16_t* w, const uint16_t* x, int k);
void launch_bf16_gemv_fast(const Bf16GemvArgs& a, hipStream_t stream);
void launch_bf16_linear_generic(const uint16_t* w, const uint16_t* bias, const uint16_t* x,
                                uint16_t* y, int tokens, int n, int k, hipStream_t stream);
size_t lm_head_blocks(int vocab, int in_features, bool fast);

// Grouped W8A16 GEMV: rows per block for a descriptor of in_features k, and
// the launch of a descriptor table (any mix of K) resident on the device.
int w8a16_grouped_rows_per_block(int k);
void launch_w8a16_gemv_grouped(const W8GroupDesc* device_descs, int count, int total_blocks,
                               hipStream_t stream);

// Plans that move few bytes: one round of loads per wave, rows per block by
// w8a16_small_rows_per_block, the descriptors in the kernel arguments
// (launch_w8a16_gemv_small) or, past kSmallGroupMax, in a device table
// (launch_w8a16_gemv_rows).
bool w8a16_gemv_plan_small(double bytes);
int w8a16_small_rows_per_block(int k);
void launch_w8a16_gemv_rows(const W8GroupDesc* descs, int count, int total_blocks,
                            hipStream_t stream);
void launch_w8a16_gemv_small(const W8SmallGroup& g, int total_blocks, hipStream_t stream);

}  // namespace qlin
