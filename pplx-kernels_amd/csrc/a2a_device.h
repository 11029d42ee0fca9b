// Device-visible records shared by the host layer and the kernels.
//
// One DispatchRank / CombineRank row per simulated EP rank lives in a table in
// HBM; kernels index it by rank.  They carry what the reference passes as
// Strided1D/2D/3D views (csrc/core/buffer.h:116-161) in the kernel argument
// lists of csrc/all_to_all/intranode_dispatch.cu:15-53 and
// csrc/all_to_all/intranode_combine.cu:16-47.
#pragma once

#include <cstddef>
#include <cstdint>

namespace pplx_amd {

constexpr uint32_t kWave = 64;            // gfx950 wavefront
constexpr uint32_t kInvalidSlot = 0xffffffffu;

constexpr uint32_t kFaultRowDropped = 1u;   // slot >= out_expert_x rows
constexpr uint32_t kFaultBadExpert = 2u;    // index >= num_experts
constexpr uint32_t kFaultBadSlot = 4u;      // combine slot >= expert_y rows
constexpr uint32_t kFaultDuplicateExpert = 8u;   // an expert id repeated inside one token was dropped
constexpr uint32_t kFaultTooManyTokens = 16u;    // bound_m > max_num_tokens (or > rows) was clamped

// Division by a number that is fixed for a launch (tokens per group, experts per rank ...):
// a multiply-high, a subtract, an add and two shifts instead of the thirty-odd instructions of
// a 32-bit hardware-less division (Granlund & Montgomery, "Division by invariant integers using
// multiplication", figure 4.1, N = 32).  Exact for every 32-bit numerator and divisor >= 1.
struct FastDiv {
  uint32_t mul;
  uint32_t shifts;  // sh1 (0 or 1) in bit 0, sh2 from bit 8 up: q = (t + ((n - t) >> sh1)) >> sh2
};
inline FastDiv make_fast_div(uint32_t d) {
  FastDiv f{1u, 0u};
  if (d <= 1) return f;  // l = 0: q = n
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;  // ceil(log2 d)
  f.mul = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
  f.shifts = 1u | ((l - 1) << 8);
  return f;
}
#ifdef __HIPCC__
__host__ __device__
#endif
inline uint32_t fast_div(uint32_t n, const FastDiv &f) {
  const uint32_t t = (uint32_t)(((uint64_t)f.mul * n) >> 32);
  return (t + ((n - t) >> (f.shifts & 1u))) >> (f.shifts >> 8);
}

// (The buffers of a rank's experts come first, together: every pick of a token looks its expert's up, in three loads out of
// two lines before, in two out of mostly one now.  Combine with the tables in the arguments, us: 1 rank, 32 tokens 3.30 /
// 2.93, 4 ranks in groups of two, 20 tokens 3.29 / 3.13.)
struct alignas(16) DispatchRank {
  uint8_t *expert_x;
  int64_t x_stride_row;     // bytes
  int64_t x_stride_expert;  // bytes
  float *expert_xs;
  int64_t xs_stride_elem;   // floats
  int64_t xs_stride_row;
  int64_t xs_stride_expert;
  uint32_t x_rows;
  uint32_t m;
  const uint8_t *dp_x;
  int64_t dp_x_stride_row;  // bytes
  const float *dp_xs;
  int64_t dp_xs_stride_elem;
  int64_t dp_xs_stride_row;
  const uint32_t *indices;
  const uint32_t *bound_m;
  int32_t *out_num_tokens;
  int64_t out_num_tokens_stride;
  uint64_t pad_;
};
static_assert(sizeof(DispatchRank) == 144, "DispatchRank layout");

struct alignas(16) CombineRank {
  const void *expert_y;
  int64_t y_stride_row;     // elements
  int64_t y_stride_expert;
  uint32_t y_rows;
  uint32_t m;
  const uint32_t *bound_m;
  const uint32_t *indices;
  const float *weights;
  int64_t w_stride_row;
  void *out_tokens;
  int64_t out_stride_row;   // elements
};
static_assert(sizeof(CombineRank) == 80, "CombineRank layout");

// Geometry + scratch of a world; passed to every kernel by value, and kept short: in some processes a launch with more
// than kShortArguments bytes of arguments costs the host 3.4 to 3.95 us instead of 2.55 (in the others 2.2, 9 KiB 2.7).  Beside a
// table in HBM the one-launch dispatch, the scatters and the gather of combine stay within them; the routing kernels, whose
// RouteSpan alone is 56 bytes, do not.
constexpr size_t kShortArguments = 112;
struct WorldDev {
  uint32_t M;        // max tokens per DP group
  uint32_t H;        // elements per row
  uint32_t Hb;       // bytes per dispatched row
  uint32_t S;        // fp32 scales per row
  uint32_t num_tiles;    // ceil(G * M / (64 * tile_chunks))
  // (bits of words, which scalar loads fetch, and not shorter integers, which they do not)
  uint32_t R : 16;   // simulated ranks (no more than experts)
  uint32_t dp : 16;  // ranks per DP group
  uint32_t G : 16;   // DP groups = R / dp
  uint32_t E : 16;   // experts (check_config: up to 5461)
  uint32_t L : 16;   // experts per rank
  uint32_t K : 8;    // experts per token (up to 64)
  uint32_t tile_chunks : 8;  // 64-token chunks per routing tile of a whole-step dispatch (up to 16)
  FastDiv by_M, by_dp, by_L, by_K;  // fast_div(n, by_X) == n / X
  uint32_t *tile_cnt;    // tokens routed to each expert inside each tile, and behind them
                         // (route_tables) [num_tiles * tile_chunks][E] 64-bit masks, one bit per
                         // token of a chunk
  uint32_t *slot_map;    // [G * M][K] row of (token, pick) inside its expert
  uint32_t *faults;      // [1] sticky fault bits
};
static_assert(sizeof(WorldDev) == 88, "WorldDev layout");

// ... and what only the host needs of it.
struct WorldHost : WorldDev {
  uint32_t lds_per_cu;   // bytes of LDS a CU has (0 = unknown): caps residency, and rows in LDS have to fit it
  DispatchRank *drank;   // [R]
  CombineRank *crank;    // [R]
};

// The routing scratch of a world is one block: the tiles' counts, the chunks' masks, and for each
// chunk the rows of its tile's earlier chunks.  The counts have one of two forms.  Steps of up to
// kScanFreeTiles tiles keep them expert-major, 16 bits each (a tile holds at most 1024 tokens):
// the kScanFreeTiles counts of an expert are one 128-byte line, short enough for whoever wants a
// prefix of it to add it up.  Longer steps keep [num_tiles][E] 32-bit counts, which route_scan
// turns into prefixes.
constexpr uint32_t kScanFreeTiles = 64;
struct RouteTables {
  uint64_t mask_offset, base_offset, bytes;
};
#ifdef __HIPCC__
__host__ __device__
#endif
inline RouteTables route_tables(uint32_t num_tiles, uint32_t tile_chunks, uint32_t experts) {
  RouteTables t;
  const uint64_t chunks = (uint64_t)num_tiles * tile_chunks;
  const uint64_t scanned = (uint64_t)num_tiles * experts * 4u, rows = (uint64_t)experts * kScanFreeTiles * 2u;
  t.mask_offset = ((scanned > rows ? scanned : rows) + 127u) & ~127ull;
  t.base_offset = t.mask_offset + chunks * experts * 8u;
  t.bytes = t.base_offset + chunks * experts * 2u;
  return t;
}

// Which virtual tokens a routing launch covers and where its results go.
struct RouteSpan {
  uint32_t v_begin;       // first virtual token (tiles are counted from here)
  uint32_t v_count;       // virtual tokens covered
  uint32_t tile_chunks;   // 64-token chunks per tile (one workgroup)
  uint32_t pick_vector;   // expert ids one load may fetch (4, 2 or 1)
  uint32_t *tile_cnt;     // [tiles][E], scanned form
  uint16_t *tile_row;     // [E][kScanFreeTiles], the form that needs no scan; NULL: the counts go to tile_cnt
  unsigned long long *tile_mask;  // [tiles * tile_chunks][E] route_count keeps the chunks' masks
                                  // here (and reports the faults) when set: the scatter that
                                  // follows works the slots out by itself
  uint16_t *chunk_base;   // [tiles * tile_chunks][E], beside tile_mask: rows of the tile's earlier chunks
  uint32_t *slot_out;     // [G * M][K], indexed by absolute virtual token
};

// Device state of split send / recv mode: two hops through staging that the world owns.
// The reference's SEND puts one copy of a row per pick into the inbox of the rank that owns the
// pick's expert, because that copy has to cross a link (csrc/all_to_all/intranode_dispatch.cu:
// 146-180); with every rank in one HBM the staging area is the wire, and one copy per TOKEN is
// all SEND has to leave behind:
//   dispatch SEND   copies what the call may not keep -- every present token's row, scales and
//                   picks, and the number of tokens present in each DP group -- into stage_x /
//                   stage_idx / stage_n (row | fp32 scales, padded to 16 bytes: the reference's
//                   wire row, csrc/all_to_all/intranode.cpp:41-47, without the source-token tag,
//                   which the position in the staging area stands for)
//   dispatch RECV   is the one-call dispatch reading the staged copies and writing the outputs
//                   named by the RECV calls
//   combine SEND    is the one-call combine writing into stage_y, one row per (rank, token)
//   combine RECV    copies each present token's combined row to the caller's out_tokens
struct SplitDev {
  uint8_t *stage_x;        // [G * M][token_stride]
  uint32_t token_stride;   // round_up(Hb + 4 S, 16)
  uint32_t pad_;
  uint32_t *stage_idx;     // [G * M][K] the staged tokens' picks
  uint32_t *stage_n;       // [G] tokens present in each DP group at SEND
  uint8_t *stage_y;        // [R * M][H] combined rows, 2-byte elements
};

// stage_x, stage_idx and stage_n are one allocation, in this order.
struct StageLayout {
  uint32_t token_stride;
  uint64_t idx_offset, n_offset, bytes;
};
#ifdef __HIPCC__
__host__ __device__
#endif
inline StageLayout stage_layout(uint32_t row_bytes, uint32_t scales, uint64_t tokens, uint32_t picks,
                                uint32_t groups) {
  StageLayout l;
  l.token_stride = (row_bytes + 4u * scales + 15u) & ~15u;
  l.idx_offset = tokens * l.token_stride;
  l.n_offset = (l.idx_offset + tokens * picks * 4u + 15u) & ~15ull;
  l.bytes = l.n_offset + ((4ull * groups + 15u) & ~15ull);
  return l;
}

// A step's rank tables reach the kernels in one of two ways.  Worlds of up to kInlineRanks ranks pass them as
// kernel arguments (up to 9 KiB for dispatch and 5 KiB for combine; HIP on gfx950 takes kernel
// arguments well beyond 4 KiB, eagerly and as graph nodes).  Larger worlds (drank / crank), and steps that were bound
// beforehand (pplx_a2a_bound_create), go through tables in HBM, written by bind kernels that take up to kBindBatch rows as
// arguments each.  Kernels read those faster than their arguments, which no cache holds from one launch to the next.  Us,
// tables in the arguments / in HBM, dispatch and combine of one buffer set: 1 rank, 32 tokens of 2 KiB 3.77 / 3.50 and
// 3.27 / 2.87; 64 x 1 DSv3 tokens 5.53 / 5.26 and 4.01 / 3.58; 8 x 128 12.69 / 12.51 and 22.12 / 21.90.
constexpr uint32_t kInlineRanks = 64;
// A table of up to this many ranks goes in an argument of that size (1152 bytes for dispatch, 640 for combine) and not in
// one for kInlineRanks, which is filled and copied at each launch and costs more to launch in processes where that grows
// with the arguments (2.24 us at 1240 bytes, 2.70 at 9304; in the others both take 3.9).  Steps, us, 64 ranks' room / this:
// 8 x 4 tokens, per-rank calls 18.2 / 17.2; 4 ranks in groups of two, 20 tokens, one call 9.2 / 8.5; 8 x 128, split
// 37.6 / 35.1.  Eight is what a node holds.  (A third kind of table makes the library 8.1 MB instead of 5.5.)
constexpr uint32_t kShortInlineRanks = 8;
constexpr uint32_t kBindBatch = 64;
// A one-launch dispatch whose rows (all picks of all tokens) stay within this many bytes and go through registers
// stores them write-through into the 256 MB last-level cache instead of streaming them past it.  That pays where
// a step's buffers come back soon: 14 KiB rows, top-8, 1024 tokens (112 MiB), one buffer set, dispatch alone 25.9
// us written through / 30.4 streamed.  With three sets in turn the two are level from about 108 MiB on (step,
// 112 MiB 55.1 / 53.2; 8 KiB rows 112 MiB 51.1 / 51.2, 140 65.0 / 63.8; 7 KiB fp8 rows 56 MiB 37.3 / 40.2,
// 95 66.7 / 67.3, 112 78.5 / 77.0), and with sixteen streaming is ahead from 8 MiB on (7 KiB fp8 rows,
// 32 MiB 30.3 / 28.6, 64 51.5 / 49.7).
constexpr uint64_t kWriteThroughMaxBytes = 192ull << 20;
// The same for rows that go through LDS, whose whole lines stream well: up to where the two are level on three sets.
// Us, written through / streamed, 8 ranks, top-8, at the MiB of rows stored; one set: dispatch alone, others: step:
//                one set                              three sets                           sixteen sets
//                66          80          95           66          80          95           66          80
//   2576 bytes   16.5 18.0   18.1 20.6                35.2 35.4   41.5 40.9                42.5 36.1   48.8 42.7
//   4240 bytes   15.3 17.4   18.2 21.8   20.2 23.2    33.8 35.0   41.8 42.5   48.2 46.7    40.5 35.4   48.1 43.1
//   5264 bytes   15.3 17.6   17.3 21.4   20.3 23.6    33.1 34.8   42.0 43.7   49.7 46.8    39.5 34.9   48.4 44.0
//   8176 bytes   15.3 17.8   17.1 20.0   19.1 24.5    35.8 37.0   40.4 40.6   47.1 46.4    41.0 37.4   44.9 40.9
// (2648 steps of 64 to 80 MiB, one to four ranks to a DP group, full and ragged, three sets: 1.6 % ahead of streaming on
// average, 0.91 to 1.15 of its time; groups of four 1 % behind.)
constexpr uint64_t kLdsWriteThroughMaxBytes = 80ull << 20;

// Device memory that pplx_a2a_static_step works in instead of a world's allocations: a fixed
// array inside the library's code object (a2a_static.hip), one copy per GPU.  The chunks' bases
// beside the masks take up to 1.25 times what masks and counts take by themselves: every step whose
// slot map, masks and counts fit 8 MiB has its room.
constexpr size_t kStaticScratchBytes = 10u << 20;
// Address of the calling thread's current device's copy (looked up once per device).
int static_scratch_address(int device, void **out);
// True once static_scratch_address has succeeded for `device`.
bool static_scratch_known(int device);

struct BindDispatchBatch {
  uint32_t first, count;
  uint64_t pad_;
  DispatchRank rows[kBindBatch];
};
struct BindCombineBatch {
  uint32_t first, count;
  uint64_t pad_;
  CombineRank rows[kBindBatch];
};

// Launchers implemented in a2a_dispatch.hip, a2a_combine.hip and a2a_split.hip; they return a
// hipError_t as int.
// `inline_rows` (world_size rows, host memory) selects the inline-table kernels;
// NULL selects the HBM tables (w.drank / w.crank), which must have been bound.
int launch_bind_dispatch(DispatchRank *table, const BindDispatchBatch &b, void *stream);
int launch_bind_combine(CombineRank *table, const BindCombineBatch &b, void *stream);
// pick_vector: how many expert ids one load may fetch from any rank's indices (4, 2 or 1):
// K must be a multiple of it and every indices pointer aligned to 4 * pick_vector bytes.
int launch_dispatch(const WorldHost &w, const DispatchRank *inline_rows, uint32_t pick_vector,
                    void *stream);
int launch_combine(const WorldHost &w, const CombineRank *inline_rows, int in_dtype, int out_dtype,
                   void *stream);
// Split mode's own launches, each for all ranks at once (`inline_rows` as above): dispatch SEND
// stages the tokens, combine RECV delivers the combined rows (`elem_bytes` of out_tokens).
// dispatch RECV and combine SEND are launch_dispatch / launch_combine on rows that point into
// the staging area.
int launch_split_stage_tokens(const WorldHost &w, const SplitDev &sp, const DispatchRank *inline_rows,
                              void *stream);
int launch_split_deliver(const WorldHost &w, const SplitDev &sp, const CombineRank *inline_rows, void *stream);
// True when dispatch runs as the single fused launch for this geometry.
bool dispatch_is_fused(const WorldHost &w);
// What launch_dispatch does with this geometry (the values of pplx_a2a_plan_t).
enum class DispatchForm : uint32_t { kOneLaunch = 0, kSlotMap = 1, kTables = 2, kScannedTables = 3 };
struct DispatchPlan {
  DispatchForm form;
  uint32_t scatter_waves_per_cu;
  bool scatter_in_turn;
  bool rows_in_lds;
};
DispatchPlan dispatch_plan(const WorldHost &w);
// What launch_combine does with this geometry (in_dtype: pplx_a2a_dtype): the picks that a wave takes at a time, the
// pieces of 64 x 8 elements that it reads of each, and whether it gathers once for the ranks of a DP group.
struct CombineForm {
  uint32_t picks, pieces;
  bool per_group;
};
CombineForm combine_form(const WorldHost &w, int in_dtype);
// Whether it stores the combined rows plainly, not past the caches.
bool combine_stores_plainly(const WorldHost &w);
// LDS bytes the routing kernels need for a given geometry.
uint32_t route_lds_bytes(uint32_t num_experts, uint32_t tile_chunks);

}  // namespace pplx_amd
