// gfx950 kernels of the MoE dispatch / combine path (single-GPU loopback).
//
// The reference moves every token through a per-peer inbox with atomically
// assigned slots and grid-wide syncs (csrc/all_to_all/intranode_dispatch.cu:15-284,
// csrc/all_to_all/intranode_combine.cu:16-187).  With all simulated ranks in one
// HBM the same results come from a count -> scan -> scatter pipeline whose
// placement is the canonical (expert, DP group, token) order that the
// reference's tests enumerate (tests/test_all_to_all.py:113-120):
//
//   route_count      per routing tile: 64-token bitmasks per expert in LDS -> rows per
//                    expert of the tile, and the masks themselves          (only if > 1 tile)
//   route_scan       per expert: prefix of the tiles' rows, totals         (only if > 64 tiles)
//   dispatch_scatter_slots  one wave per token (or per share of its K picks): the row is
//                    read once into registers, lane k works the slot of pick k out of the
//                    tiles' rows and the masks, the row is stored K times, 16 B / lane
//                    (dispatch_scatter_scanned behind route_scan)
//   route_slots + dispatch_scatter  the same with the slots written by a launch of their
//                    own (single tile, rows beyond the register variants)
//   dispatch_fused   small steps: routing and scatter in one launch; every
//                    workgroup recounts the picks of the tokens before its own
//                    (rows that cut 64-byte half lines go through LDS instead of registers in
//                    both, and so do those that no register variant of dispatch_fused fits)
//   combine_gather   one wave per 1 KiB of an output row: K rows gathered through
//                    the slot map, fp32 accumulate in pick order, 16 B stores
//
// No atomics on global memory (fault flags aside), no spin waits, no
// cooperative launch: phase boundaries are kernel boundaries on one stream, so a
// step captures into a hipGraph as is.  Wavefronts are 64 wide throughout.
//
// Rank tables reach the kernels either inline, as kernel arguments (worlds of
// up to kInlineRanks ranks: nothing to bind, nothing to go stale), or through
// HBM tables written by bind_rows (larger worlds, and steps bound beforehand).
#include "a2a_route.h"
#include "a2a_rows.h"

// Built with -DPPLX_A2A_TIMELINE (make TIMELINE=1), dispatch_fused records when thread 0 of every
// workgroup passes its phase boundaries (the GPU's 100 MHz wall clock) into a table that
// pplx_a2a_debug_timeline copies out; `bench.py --timeline` prints the summary.  The waits that
// the stamps need (for the row, for the stores) are not in the regular build.
#ifdef PPLX_A2A_TIMELINE
__device__ unsigned long long g_timeline[1024 * 16];
extern "C" int pplx_a2a_debug_timeline(unsigned long long *host, int words) {
  return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(g_timeline), sizeof(unsigned long long) * (size_t)words);
}
#endif

namespace pplx_amd {
namespace {

struct Timeline {
#ifdef PPLX_A2A_TIMELINE
  unsigned long long at[9];
  __device__ __forceinline__ void mark(int i) { at[i] = wall_clock64(); }
  __device__ __forceinline__ void wait_for_memory() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }
  __device__ __forceinline__ void flush() {
    if (threadIdx.x != 0 || blockIdx.x >= 1024) return;
    for (int i = 0; i < 9; ++i) g_timeline[blockIdx.x * 16 + i] = at[i];
    g_timeline[blockIdx.x * 16 + 9] = __builtin_amdgcn_s_getreg((20 << 0) | (0 << 6) | (3 << 11)) & 0xf;  // XCC id
  }
#else
  __device__ __forceinline__ void mark(int) {}
  __device__ __forceinline__ void wait_for_memory() {}
  __device__ __forceinline__ void flush() {}
#endif
};

// ---------------------------------------------------------------------------
// Table binding: rows arrive as kernel arguments and are stored with vector
// stores, so a captured graph carries its own pointers.
// ---------------------------------------------------------------------------
template <typename Batch, typename Row>
__global__ __launch_bounds__(256) void bind_rows(Row *table, Batch b) {
  constexpr uint32_t kWords = sizeof(Row) / 8;
  const uint64_t *src = reinterpret_cast<const uint64_t *>(b.rows);
  uint64_t *dst = reinterpret_cast<uint64_t *>(table + b.first);
  for (uint32_t i = threadIdx.x; i < b.count * kWords; i += blockDim.x) {
    dst[i] = src[i];
  }
}

// Where a scatter wave gets its token's slots from.
enum class Slots {
  kMap,      // the slot map, which route_slots wrote
  kScanned,  // the routing tables behind route_scan (the wave writes the slot map)
  kTables,   // the routing tables as route_count left them (the same)
};

// One wave per token (or per share of its picks).  It needs the row, the picks' slots and their experts'
// buffers.  IN_TURN fetches them one behind the other; otherwise the picks go out first (loads return
// in order) and what depends on them, the buffers and the routing tables, is fetched while the row is
// still on its way.  Which steps want which: scatter_plan.
template <int NV, bool EXACT, class DT, Slots SLOTS, bool IN_TURN>
__device__ __forceinline__ void scatter_token(const WorldDev &w, const DT &tab, uint32_t wave, uint32_t ksplit,
                                              uint32_t kper) {
  const uint32_t lane = lane_id();
  const uint32_t v = wave >> __builtin_ctz(ksplit);  // (ksplit is a power of two)
  const uint32_t part = wave - v * ksplit;
  const uint32_t g = group_of(w, v);
  const uint32_t t = v - g * w.M;
  if (g >= w.G) return;
  if (t >= dispatch_group_tokens(w, tab, g)) return;
  const DispatchRank &src = tab.at(sender_of(w, g, t));
  constexpr bool kStaged = NV == 0;  // the row goes through LDS
  extern __shared__ u32x4 lds_row[];
  RowRegs<kStaged ? 1 : NV> regs;
  auto fetch_row = [&]() {
    if constexpr (kStaged) {
      regs.sc = load_scale(w, src, t, lane);
      stage_row(w, src, t, lane, 0, 1, lds_row);
    } else {
      load_row<NV, EXACT>(w, src, t, lane, regs);
    }
  };
  if constexpr (IN_TURN) fetch_row();
  const uint32_t e = lane < w.K ? as_global(src.indices)[(size_t)t * w.K + lane] : w.E;
  if constexpr (!IN_TURN) fetch_row();
  ExpertBuffer buffer;
  if constexpr (!IN_TURN) buffer = expert_buffer(w, tab, e);
  uint32_t slot = kInvalidSlot;
  if constexpr (SLOTS == Slots::kMap) {
    if (lane < w.K && e < w.E) slot = as_global(w.slot_map)[(size_t)v * w.K + lane];
  } else {
    slot = slots_from_tables<SLOTS == Slots::kScanned>(w, v, lane, e);
    if (lane < w.K && part == 0) as_global(w.slot_map)[(size_t)v * w.K + lane] = slot;
  }
  if constexpr (IN_TURN) {
    settle(slot);
    buffer = expert_buffer(w, tab, e);
  }
  const Destination dst = destination_of(w, buffer, slot, part == 0);
  const uint32_t k0 = part * kper;
  const uint32_t k1 = (k0 + kper < w.K) ? k0 + kper : w.K;
  // Rows stream past the caches; the 4-byte-per-lane scale rows are written through into the
  // last-level cache instead, where the partial lines of neighbouring rows meet before they go
  // to HBM (3-4 % of the kernel's time at 224-byte scale rows).
  if constexpr (kStaged) {
    row_staged();
    store_staged_row<RowStore::kStream, RowStore::kKeep, RowStore::kKeep>(w, src, t, lane, dst, k0, k1, regs.sc, lds_row);
  } else {
    store_row<NV, EXACT, RowStore::kStreamThrough, RowStore::kKeep>(w, src, t, lane, dst, k0, k1, regs);
  }
}

// Launched as one-wave workgroups whose dynamic LDS size caps how many of them a CU holds at a
// time (scatter_lds); only the variants for rows that go through LDS (NV = 0) use it, for the row.
template <int NV, bool EXACT, class DT>
__global__ __launch_bounds__(kWave) void dispatch_scatter(WorldDev w, DT tab, uint32_t ksplit, uint32_t kper) {
  scatter_token<NV, EXACT, DT, Slots::kMap, false>(w, tab, blockIdx.x, ksplit, kper);
}

template <int NV, bool EXACT, class DT, bool IN_TURN>
__global__ __launch_bounds__(kWave) void dispatch_scatter_scanned(WorldDev w, DT tab, uint32_t ksplit, uint32_t kper) {
  scatter_token<NV, EXACT, DT, Slots::kScanned, IN_TURN>(w, tab, blockIdx.x, ksplit, kper);
}

// The first ceil(E / 8) workgroups write the experts' totals.
template <int NV, bool EXACT, class DT, bool IN_TURN>
__global__ __launch_bounds__(kWave) void dispatch_scatter_slots(WorldDev w, DT tab, uint32_t ksplit, uint32_t kper) {
  const uint32_t totals = (w.E + 7) / 8;
  if (blockIdx.x < totals) {
    write_totals(w, tab, blockIdx.x, lane_id());
    return;
  }
  scatter_token<NV, EXACT, DT, Slots::kTables, IN_TURN>(w, tab, blockIdx.x - totals, ksplit, kper);
}

// Threads of a dispatch_fused workgroup: 16 waves (fewer, larger workgroups repeat less
// counting) while the row fits 8 registers of 16 bytes per lane, 8 waves for the 14- and
// 16-register rows, which would spill under the 128-register limit of a 1024-thread workgroup.
// A compile-time size also keeps the kernel's first loads free of any wait.
constexpr uint32_t fused_threads(int nv) { return nv > 8 ? 512u : 1024u; }

// How a launch of dispatch_fused goes about its tokens.
struct FusedShape {
  uint32_t ksplit : 8, kper : 8;  // waves that share a token's picks, picks of each
  uint32_t tokens_per_block : 8;
  uint32_t pick_vector : 4;       // expert ids one load may fetch
  uint32_t write_through : 1;
};
static_assert(sizeof(WorldDev) + sizeof(HbmDispatch) + sizeof(FusedShape) <= kShortArguments, "arguments of dispatch_fused");
static_assert(sizeof(WorldDev) + sizeof(HbmDispatch) + 2 * sizeof(uint32_t) <= kShortArguments, "arguments of the scatters");

// A rank table that dispatch_fused has copied into LDS.
struct LdsDispatch {
  const DispatchRank *rows;
  __device__ __forceinline__ const DispatchRank &at(uint32_t i) const { return rows[i]; }
};

// Picks first, ..., first + NP - 1 of a token in registers, fetched PV at a time by loads that are issued
// together.  Positions beyond the token's K picks hold copies of others; FULL: K == NP.
template <int PV, int NP, bool FULL> struct PickBlock {
  typedef PickVector<PV> Vec;
  typename Vec::type v[NP / PV];
  __device__ __forceinline__ void load(const PPLX_GLOBAL typename Vec::type *idx, uint32_t first, uint32_t K) {
    const uint32_t from = first / PV;
    if constexpr (FULL) {
#pragma unroll
      for (uint32_t i = 0; i < NP / PV; ++i) v[i] = idx[i];
      return;
    }
    uint32_t last = K / PV - 1;
    settle(last);  // (a vector register: sixteen clamped offsets do not fit beside the scalars)
#pragma unroll
    for (uint32_t i = 0; i < NP / PV; ++i) v[i] = idx[from + i < last ? from + i : last];
  }
  __device__ __forceinline__ uint32_t at(int u) const { return Vec::at(v[u / PV], u % PV); }
};

// Counts, per expert, the tokens before virtual token v_end that are routed to it, into the LDS
// histogram `hist`: one thread per token and pass, PV picks per load (K % PV == 0 and every
// indices pointer aligned to the vector: the host checks both), NP picks of a token in registers at a time.
// Every expert a token names counts once (a repeat inside the token takes no row).
//
// The loads of a token (its group's token count and its first NP picks) are
// unconditional, from a harmless address when the thread has no token, and sit in
// straight-line code: they are issued together and cost one trip to memory, and the count is
// applied afterwards.  The loads of the next pass are issued before the picks of this one are
// counted, so a step of several passes pays one trip, not one per pass.
template <int PV, int NP, bool FULL, uint32_t THREADS, class Table>
__device__ __forceinline__ void count_earlier_picks(const WorldDev &w, const Table &rows, uint32_t v_end,
                                                    uint32_t *hist) {
  typedef typename PickVector<PV>::type vec_t;
  struct Fetch {
    PickBlock<PV, NP, FULL> picks;
    uint32_t n;           // tokens present in the group
    uint32_t t;           // token inside its group
    const PPLX_GLOBAL vec_t *idx;
    bool valid;
  };
  auto issue = [&](uint32_t v) {
    Fetch f;
    const bool in_range = v < v_end;
    const uint32_t g = in_range ? group_of(w, v) : 0;
    f.t = in_range ? v - g * w.M : 0;
    const DispatchRank &head = rows.at(g * w.dp);
    const DispatchRank &src = w.dp == 1 ? head : rows.at(sender_of(w, g, f.t));
    f.valid = in_range && f.t < src.m && f.t < head.m;
    const bool bounded = f.valid && head.bound_m != nullptr;
    const uint32_t loaded_n = *as_global(bounded ? head.bound_m : w.faults);
    f.idx = as_global(reinterpret_cast<const vec_t *>(f.valid ? src.indices + (size_t)f.t * w.K : w.slot_map));
    f.picks.load(f.idx, 0, w.K);
    f.n = bounded ? loaded_n : head.m;
    return f;
  };
  // Picks first, ... of the token, of which the earlier ones have been counted.
  auto count = [&](const PickBlock<PV, NP, FULL> &picks, uint32_t first, const PPLX_GLOBAL vec_t *idx) {
    if constexpr (FULL) {
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        bool counts = picks.at(u) < w.E;
#pragma unroll
        for (int p = 0; p < u; ++p) counts = counts && picks.at(p) != picks.at(u);
        if (counts) atomicAdd(&hist[picks.at(u)], 1u);
      }
      return;
    }
    // bit u: pick first + u does not exist, or repeats an earlier one
    unsigned skip = w.K - first < NP ? ~0u << (w.K - first) : 0u;
    settle(skip);
    if (NP > 8 && first != 0) {
      const PPLX_GLOBAL uint32_t *before = reinterpret_cast<const PPLX_GLOBAL uint32_t *>(idx);
      for (uint32_t p = 0; p < first; ++p) {
        const uint32_t earlier = before[p];
#pragma unroll
        for (int u = 0; u < NP; ++u) skip |= (unsigned)(earlier == picks.at(u)) << u;
      }
    }
#pragma unroll
    for (int u = 1; u < NP; ++u) {
      bool repeats = false;
#pragma unroll
      for (int p = 0; p < u; ++p) repeats = repeats || picks.at(p) == picks.at(u);
      skip |= (unsigned)repeats << u;
      settle(skip);  // (bits in a register, not a condition mask per comparison)
    }
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      if (picks.at(u) < w.E && !((skip >> u) & 1u)) atomicAdd(&hist[picks.at(u)], 1u);
    }
  };
  auto consume = [&](const Fetch &f) {
    if (!f.valid || f.t >= f.n) return;
    PickBlock<PV, NP, FULL> picks = f.picks;
    for (uint32_t first = 0;;) {
      count(picks, first, f.idx);
      first += NP;
      if (NP <= 8 || first >= w.K) break;
      picks.load(f.idx, first, w.K);
    }
  };

  Fetch current = issue(threadIdx.x);
  for (uint32_t v = threadIdx.x + THREADS; v < v_end; v += THREADS) {
    const Fetch next = issue(v);
    consume(current);
    current = next;
  }
  consume(current);
}

// Small steps: one launch does routing and scatter.  A workgroup owns tokens_per_block
// consecutive virtual tokens; each of them belongs to one wave (or to ksplit waves that share
// its picks), and lane k of such a row wave is the token's pick k.
//   0. the rank table (world_size rows of it) is copied from the kernel arguments, or from HBM, into LDS with
//      loads that depend on nothing, so every later lookup is an LDS read and not another trip
//      to memory behind the one that fetches the geometry (tables of more than 64 ranks too, up to 56 KiB for 384:
//      dispatch, us, looked up in HBM / copied: 72 ranks x 1 token, top-8, 2 KiB fp8 rows 4.96 / 4.51, 256 x 1 5.65 / 5.23, 384 x
//      10, 512 wide, top-2 7.50 / 6.11; 60 shapes of 72 to 384 ranks 0.94 of the time, at worst, 384 x 4 rows of 14 KiB, 1.03);
//   1. one batch of small loads: every thread fetches the picks of one token before the
//      workgroup's own (and its group's token count), the row waves their own picks;
//   2. the picks of the earlier tokens are counted per expert in an LDS histogram (every
//      workgroup repeats this over the indices, which are a few KiB in L2); the row waves mark
//      their token in a per-expert bit mask of the workgroup's own tokens and issue the loads of
//      their rows (where exactly the row loads go -- with the picks' loads, behind their
//      arrival, or behind the counting as written here -- changes nothing that can be measured:
//      8 x 128 DSv3 tokens take 13.5-13.7 us and 64 x 1 tokens 5.6-6.3 us in every order, the
//      first bound by the rate of their stores, the second by the chain of cold trips);
//   3. behind one barrier a pick's slot is the histogram's count plus the own tokens before
//      its own that go to the same expert (a popcount of the mask below the token's bit); the
//      lane resolves its destination row and keeps it in registers;
//   4. the waves fan their rows out.  The last workgroup has counted everything and writes
//      out_expert_num_tokens.
// NV = 0: the rows go through LDS; the waves that share a token fetch its row together (fused_rows_in_lds).
// MANY: more than eight picks.  Counting them takes 70 registers, in a kernel of its own so that the others do not pay
// for them: rows of 1, 2 and 3 KiB get by with 42, 45 and 55, and two workgroups fit a CU (kernel alone, us, all
// numbers of picks in one kernel / apart, medians of two runs of 360 launches: 512-byte rows, 8 x 128 tokens, top-8 6.28 6.36 /
// 6.12 6.24, 8 x 512, top-4 7.64 7.72 / 7.44 7.64; 1 KiB rows, 8 x 128, top-8 level at 6.20 - 6.32).
template <int NV, bool EXACT, class DT, bool MANY>
__device__ __forceinline__ void dispatch_in_one(const WorldDev &w, const DT &tab, const FusedShape &shape) {
  const uint32_t ksplit = shape.ksplit, kper = shape.kper, tokens_per_block = shape.tokens_per_block;
  const uint32_t pick_vector = shape.pick_vector, write_through = shape.write_through;
  constexpr uint32_t kFusedThreads = fused_threads(NV);
  extern __shared__ unsigned long long lds_u64[];
  Timeline timeline;
  timeline.mark(0);
  constexpr uint32_t kRowWords = sizeof(DispatchRank) / 8;
  const uint32_t table_words = w.R * kRowWords;
  {
    const unsigned long long *table = reinterpret_cast<const unsigned long long *>(&tab.at(0));
    for (uint32_t i = threadIdx.x; i < table_words; i += kFusedThreads) lds_u64[i] = table[i];
  }
  uint32_t *hist = reinterpret_cast<uint32_t *>(lds_u64 + table_words);  // [E] tokens before the workgroup's own
  uint32_t *own_mask = hist + w.E;                                       // [E] bit j: own token j goes to e
  // NV = 0: the workgroup's rows, one behind the other
  u32x4 *own_rows = reinterpret_cast<u32x4 *>(lds_u64 + ((table_words + w.E + 1) & ~1u));
  for (uint32_t e = threadIdx.x; e < 2 * w.E; e += kFusedThreads) hist[e] = 0;
  // Orders the zeroing (and the staged table) before the first counter update of any wave.
  __syncthreads();
  timeline.mark(1);
  const LdsDispatch rows{reinterpret_cast<const DispatchRank *>(lds_u64)};

  const uint32_t total = w.G * w.M;
  const uint32_t v0 = blockIdx.x * tokens_per_block;

  // 1. this wave's token; lane k is its pick k
  const uint32_t lane = lane_id();
  const uint32_t my_wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t my_j = my_wave >> __builtin_ctz(ksplit);  // (ksplit is a power of two)
  const uint32_t my_part = my_wave - my_j * ksplit;
  const uint32_t my_v = v0 + my_j;
  const bool my_in_range = my_j < tokens_per_block && my_v < total;
  const uint32_t my_g = my_in_range ? group_of(w, my_v) : 0;
  const uint32_t my_t = my_in_range ? my_v - my_g * w.M : 0;
  const DispatchRank &my_head = rows.at(my_g * w.dp);
  const DispatchRank &my_src = w.dp == 1 ? my_head : rows.at(sender_of(w, my_g, my_t));
  const bool my_row_exists = my_in_range && my_t < my_src.m && my_t < my_head.m;
  const bool my_bounded = my_row_exists && my_head.bound_m != nullptr;
  const uint32_t my_loaded_n = *as_global(my_bounded ? my_head.bound_m : w.faults);
  const bool has_pick = my_row_exists && lane < w.K;
  const uint32_t my_loaded_e = *as_global(has_pick ? my_src.indices + (size_t)my_t * w.K + lane : w.faults);

  // 2. picks of all earlier tokens
  if constexpr (MANY) {
    if (pick_vector > 1) count_earlier_picks<2, 16, false, kFusedThreads>(w, rows, v0, hist);
    else count_earlier_picks<1, 16, false, kFusedThreads>(w, rows, v0, hist);
  } else if (w.K > 4) {
    if (pick_vector == 4) count_earlier_picks<4, 8, true, kFusedThreads>(w, rows, v0, hist);
    else if (pick_vector == 2) count_earlier_picks<2, 8, false, kFusedThreads>(w, rows, v0, hist);
    else count_earlier_picks<1, 8, false, kFusedThreads>(w, rows, v0, hist);
  } else if (w.K > 2) {
    if (pick_vector == 4) count_earlier_picks<4, 4, true, kFusedThreads>(w, rows, v0, hist);
    else count_earlier_picks<1, 4, false, kFusedThreads>(w, rows, v0, hist);
  } else {
    if (pick_vector == 2) count_earlier_picks<2, 2, true, kFusedThreads>(w, rows, v0, hist);
    else count_earlier_picks<1, 2, false, kFusedThreads>(w, rows, v0, hist);
  }
  timeline.mark(2);
  // ... and the workgroup's own: a pick that names no expert, or repeats an earlier pick of its
  // token, has no row.
  uint32_t my_n = my_bounded ? my_loaded_n : my_head.m;
  my_n = my_n < w.M ? my_n : w.M;
  const bool my_live = my_row_exists && my_t < my_n;
  const uint32_t my_e = has_pick ? my_loaded_e : w.E;
  bool my_repeats = false;
  for (uint32_t k = 0; k + 1 < w.K; ++k) {
    const uint32_t earlier = (uint32_t)__builtin_amdgcn_readlane((int)my_e, (int)k);
    if (lane > k && earlier == my_e) my_repeats = true;
  }
  const bool my_pick_has_row = my_live && my_e < w.E && !my_repeats;
  if (my_pick_has_row && my_part == 0) atomicOr(&own_mask[my_e], 1u << my_j);
  timeline.mark(3);
  constexpr bool kRowInLds = NV == 0;
  RowRegs<kRowInLds ? 1 : NV> regs;
  u32x4 *my_row = own_rows + (size_t)my_j * (w.Hb / 16);
  if constexpr (kRowInLds) {
    regs.sc = 0.f;
    if (my_live) {
      regs.sc = load_scale(w, my_src, my_t, lane);
      stage_row(w, my_src, my_t, lane, my_part, ksplit, my_row);
    }
    row_staged();
  } else {
    if (my_live) load_row<NV, EXACT>(w, my_src, my_t, lane, regs);
  }
  __syncthreads();
  timeline.mark(4);

  // 3. own slots and destinations
  uint32_t my_slot = kInvalidSlot;
  if (my_pick_has_row) my_slot = hist[my_e] + __popc(own_mask[my_e] & ((1u << my_j) - 1u));
  Destination dst;
  if (my_in_range && lane < w.K) {
    const size_t pair = (size_t)my_v * w.K + lane;
    if (my_live) dst = destination_of(w, expert_buffer(w, rows, my_e), my_slot, my_part == 0);
    if (my_live && my_part == 0) {
      as_global(w.slot_map)[pair] = my_slot;
      if (my_e >= w.E) {
        atomicOr(w.faults, kFaultBadExpert);
      } else if (my_repeats) {
        atomicOr(w.faults, kFaultDuplicateExpert);
      }
    }
  }
  if (v0 + tokens_per_block >= total) {  // (and not by gridDim, which is an argument of its own)
    for (uint32_t e = threadIdx.x; e < w.E; e += kFusedThreads) {
      const uint32_t rows_of_e = hist[e] + __popc(own_mask[e]);
      const DispatchRank &owner = rows.at(owner_of(w, e));
      as_global(owner.out_num_tokens)[(int64_t)local_of(w, e) * owner.out_num_tokens_stride] = (int32_t)rows_of_e;
    }
  }

  timeline.mark(5);
  // 4. fan out
  if (my_live) {
    timeline.wait_for_memory();
    timeline.mark(6);
    const uint32_t k0 = my_part * kper;
    const uint32_t k1 = (k0 + kper < w.K) ? k0 + kper : w.K;
    if constexpr (kRowInLds) {
      if (write_through) {
        store_staged_row<RowStore::kKeep, RowStore::kKeep, RowStore::kKeep>(w, my_src, my_t, lane, dst, k0, k1, regs.sc, my_row);
      } else {
        store_staged_row<RowStore::kStream, RowStore::kKeep, RowStore::kKeep>(w, my_src, my_t, lane, dst, k0, k1, regs.sc, my_row);
      }
    } else if (write_through) {
      store_row<NV, EXACT, RowStore::kKeep>(w, my_src, my_t, lane, dst, k0, k1, regs);
    } else {
      store_row<NV, EXACT, RowStore::kStream>(w, my_src, my_t, lane, dst, k0, k1, regs);
    }
  }
  timeline.mark(7);
  timeline.wait_for_memory();
  timeline.mark(8);
  timeline.flush();
  // A bound_m beyond the limit is reported once, behind the stores (it costs a trip to memory).
  if (blockIdx.x == 0) {
    for (uint32_t g = threadIdx.x; g < w.G; g += kFusedThreads) {
      if (dispatch_group_overflows(w, rows, g)) atomicOr(w.faults, kFaultTooManyTokens);
    }
  }
}

template <int NV, bool EXACT, class DT, bool MANY>
__global__ __launch_bounds__(fused_threads(NV)) void dispatch_fused(WorldDev w, DT tab, FusedShape shape) {
  dispatch_in_one<NV, EXACT, DT, MANY>(w, tab, shape);
}
// ... with a table of few ranks among the arguments.  The same code, which the table's type alone would tell apart: the name of
// its own is for what counts the built library's kernels by name (the registers of the short rows' forms).
template <int NV, bool EXACT, class DT, bool MANY>
__global__ __launch_bounds__(fused_threads(NV)) void dispatch_fused_few(WorldDev w, DT tab, FusedShape shape) {
  dispatch_in_one<NV, EXACT, DT, MANY>(w, tab, shape);
}
template <int NV, bool EXACT, class DT, bool MANY> constexpr auto fused_kernel() {
  if constexpr (std::is_same_v<DT, InlineDispatch<kShortInlineRanks>>) return dispatch_fused_few<NV, EXACT, DT, MANY>;
  else return dispatch_fused<NV, EXACT, DT, MANY>;
}

// Rows longer than the register variants cover: stream each vector K times.
template <class DT>
__global__ __launch_bounds__(256) void dispatch_scatter_long(WorldDev w, DT tab) {
  __shared__ uint64_t s_row[kWave];
  __shared__ uint64_t s_scale[kWave];
  __shared__ int64_t s_step[kWave];
  const uint32_t v = blockIdx.x;
  const uint32_t g = group_of(w, v);
  const uint32_t t = v - g * w.M;
  if (g >= w.G) return;
  if (t >= dispatch_group_tokens(w, tab, g)) return;
  const DispatchRank &src = tab.at(sender_of(w, g, t));
  if (threadIdx.x < w.K) {
    uint64_t dst_row = 0, dst_scale = 0;
    int64_t step = 0;
    const uint32_t e = as_global(src.indices)[(size_t)t * w.K + threadIdx.x];
    const uint32_t slot = as_global(w.slot_map)[(size_t)v * w.K + threadIdx.x];
    if (e < w.E && slot != kInvalidSlot) {
      const DispatchRank &dst = tab.at(owner_of(w, e));
      const uint32_t el = local_of(w, e);
      if (slot < dst.x_rows) {
        dst_row = reinterpret_cast<uint64_t>(dst.expert_x + (int64_t)el * dst.x_stride_expert +
                                             (int64_t)slot * dst.x_stride_row);
        if (w.S) {
          dst_scale = reinterpret_cast<uint64_t>(dst.expert_xs + (int64_t)el * dst.xs_stride_expert +
                                                 (int64_t)slot * dst.xs_stride_row);
          step = dst.xs_stride_elem;
        }
      } else {
        atomicOr(w.faults, kFaultRowDropped);
      }
    }
    s_row[threadIdx.x] = dst_row;
    s_scale[threadIdx.x] = dst_scale;
    s_step[threadIdx.x] = step;
  }
  __syncthreads();
  const uint32_t nvec = w.Hb / 16;
  const PPLX_GLOBAL u32x4 *row =
      as_global(reinterpret_cast<const u32x4 *>(src.dp_x + (int64_t)t * src.dp_x_stride_row));
  for (uint32_t j = threadIdx.x; j < nvec; j += blockDim.x) {
    const u32x4 x = row[j];
    for (uint32_t k = 0; k < w.K; ++k) {
      if (s_row[k]) global_ptr<u32x4>(s_row[k])[j] = x;
    }
  }
  if (w.S) {
    const PPLX_GLOBAL float *srow = as_global(src.dp_xs) + (int64_t)t * src.dp_xs_stride_row;
    for (uint32_t j = threadIdx.x; j < w.S; j += blockDim.x) {
      const float sc = srow[(int64_t)j * src.dp_xs_stride_elem];
      for (uint32_t k = 0; k < w.K; ++k) {
        if (s_scale[k]) global_ptr<float>(s_scale[k])[(int64_t)j * s_step[k]] = sc;
      }
    }
  }
}

// LDS of a dispatch_fused workgroup: the rank table, the histogram and the mask of the workgroup's own tokens.
uint32_t fused_lds_bytes(const WorldHost &w) {
  return (w.R * (uint32_t)sizeof(DispatchRank) + 2u * w.E * (uint32_t)sizeof(uint32_t) + 15u) & ~15u;
}
// Tokens of a dispatch_fused workgroup: as few as still give every CU a workgroup (all of a workgroup's
// waves help with the counting; only the waves that own a token, or a share of one, load and store
// rows, and few storing waves per CU suit the memory system better than sixteen: 8 x 128 DSv3
// tokens take 14.7 us with 4 row waves per workgroup against 15.1 us with 16).
uint32_t fused_tokens_per_block(uint32_t tokens, uint32_t waves) {
  const uint32_t n = (tokens + 255) / 256;
  return n > waves ? waves : n < 1 ? 1 : n;
}
// Whether dispatch_fused keeps its rows in LDS: those that no register variant fits, and those that cut half lines once a
// step stores enough for whole lines to matter (the way through LDS costs 0.3-0.8 us in front of the first store, and
// every copy reads the row from there again).  How much that is depends on where a step's buffers are: the lines lie
// where little is lost while the last-level cache still holds them, although cold buffers gain from far smaller steps
// on.  Dispatch + combine, top-8, us, registers / LDS as stored here, at the MiB of rows stored, on three buffer sets in
// turn and on sixteen, nothing of which is cached:
//                  three sets                                          sixteen sets
//                  24          40          56          66          80          24          40          56          66
//   2064 bytes *   16.9 17.2   24.2 25.2   31.2 31.8                           23.3 21.8   34.0 31.6   43.8 39.9
//   2576 bytes *   16.4 16.7   23.0 23.6   30.0 30.7   34.8 35.1   42.3 40.5   23.1 21.0   32.5 29.7   42.9 37.8   48.8 42.7
//   3088 bytes     15.9 16.2   22.4 23.1   29.6 30.6   35.0 35.1   42.4 40.4   21.9 20.3   32.4 29.1   42.5 37.1   48.1 41.5
//   3600 bytes     16.0 16.2   22.5 22.9   29.7 29.5   34.1 34.0   42.8 40.5   22.5 20.7   32.4 28.5   41.5 35.9
//   4240 bytes     16.0 16.2   22.8 22.9   29.4 29.8   34.4 33.8   45.3 41.8   22.5 20.2   32.4 28.0   42.6 36.1   48.2 40.5
//   5264 bytes     16.1 16.3   22.2 22.5   29.6 29.3   33.5 33.2   44.3 41.4   22.7 20.5   31.6 27.0   42.9 35.6   48.5 39.8
//   8176 bytes     15.6 15.7   23.3 23.5   27.0 27.2   37.0 35.8   48.1 40.4   22.4 20.3   32.8 27.9   40.0 32.8   49.8 41.0
// (* below 64 MiB these two stay in registers.)  Rows without a register variant took two launches; dispatch, two
// launches / one: 12016 bytes, top-8 0.7 MiB 8.8 / 6.4, 46 27.6 / 13.5, 93 41.5 / 23.6; 13312 bytes, top-5 32 23.8 / 10.8;
// 9216 bytes, top-4 18 12.8 / 7.7.
bool fused_rows_in_lds(const WorldHost &w) {
  if (!row_has_register_variant(w)) return true;
  if (!row_cuts_half_lines(w)) return false;
  const uint64_t stored = (uint64_t)w.G * w.M * w.K * (w.Hb + 4ull * w.S);
  return w.Hb >= 3072 ? stored > 16ull << 20 : w.Hb >= 2048 && stored > 64ull << 20;
}
uint32_t fused_waves(const WorldHost &w) {
  const uint32_t per_lane = (w.Hb / 16 + kWave - 1) / kWave;
  return fused_threads(fused_rows_in_lds(w) ? 0 : (int)per_lane) / kWave;
}

// Number of waves a row's K copies are spread over (the row's re-reads hit L2).  Steps of one
// routing tile need them to cover the 256 CUs.  Larger ones split only what leaves each wave long
// runs of stores (8 ranks, us in this form at one / two / four waves per token: 14 KiB rows, top-8, 1280 tokens
// 38.8 / 36.4 / 38.6; 7 KiB rows, top-8, 2048 tokens 29.9 / 29.8 / 35.2; 4 KiB rows, top-8, 3072 tokens
// 25.1 / 28.3 / 30.6; 8 KiB rows, top-2, 3072 tokens 18.1 / 20.4 / 30.6).
uint32_t pick_ksplit(const WorldHost &w, uint32_t max_split) {
  const uint64_t tokens = (uint64_t)w.G * w.M;
  const uint64_t stored = w.K * (w.Hb + 4ull * w.S);
  uint32_t ksplit = 1;
  while (ksplit < max_split && ksplit < w.K && tokens * ksplit < 4096 &&
         (w.num_tiles == 1 || stored / (2 * ksplit) >= 48 * 1024)) ksplit *= 2;
  return ksplit;
}

// Whether the scatter takes rows that cut half lines through LDS.  A row costs a trip to LDS in front of its
// first store and another read of it per copy there, which short rows of small steps, bound by the chain of a wave and
// not by the memory, do not get back.  Dispatch on three buffer sets, experts 64, LDS : registers at 4200, 8000 and
// 20000 tokens
//               top-4              top-8              top-10             top-16             top-64
//   112 bytes   1.02 1.02 1.01     1.07 1.04 1.00     1.10 1.03 0.98     1.12 1.03 0.93     0.91 0.76 0.83
//   144 bytes   1.04 1.01 1.01     1.09 1.02 0.97     1.12 1.00 0.99     1.09 0.97 0.87     0.92 0.77 0.80
//   272 bytes   1.02 0.99 0.95     1.08 0.96 0.89     1.07 0.94 0.81     1.06 0.88 0.76     1.00 0.90 0.96
//   400 bytes   1.01 0.96 0.90     1.04 0.91 0.81     1.01 0.86 0.77     0.91 0.71 0.68     0.90 0.83 0.90
//   528 bytes   1.00 0.97 0.83     0.99 0.83 0.71     0.97 0.79 0.66     0.81 0.63 0.63     0.87 0.95 0.88
// The two are level where the step's rows, read once, come to 2 MiB, or what it stores to 24.  Rows of 96 bytes and
// less lose (16 bytes 1.03 - 1.44, 48 bytes 1.0 - 1.26, 64 bytes, which cut no line, 1.20 - 1.44, 96 bytes 1.0 - 1.12)
// except for some steps of 64 picks (80 and 96 bytes 0.85 - 0.91).
bool scatter_rows_in_lds(const WorldHost &w) {
  if (!row_cuts_half_lines(w) || w.Hb < 112) return false;
  const uint64_t read = (uint64_t)w.G * w.M * w.Hb;
  return w.Hb >= 1024 || read >= 2u << 20 || read * w.K >= 24u << 20;
}

// How the scatter's waves go about their stores: how many of them a CU holds at a time (0 = as many
// as fit), and whether they take the row, the slots and the experts' buffers one behind the other
// (scatter_token).  A wave's launch, its loads and its slot arithmetic are dead time for the stores, so
// the less a wave stores the more of them it takes to keep the CU's stores going; where it stores much,
// few waves keep the stores in longer runs, and large steps do best with three whose stores start
// later.  Dispatch on 8 ranks, us, all forms alternating in one process on the same buffers (whose
// place in memory moves all of them by up to 15 % from one process to the next); side by side at 4 and
// 9 waves / one behind the other at 3:
//   59 KiB stored per wave (DSv3 fp8 rows, top-8 of 256)
//     8 x 509    52.7 /  -  / 53.0     8 x 1024  97.8 /  -  / 98.4    8 x 2048  184 / 189 / 185
//     8 x 4096    432 / 431 / 430      8 x 6000   645 / 626 / 610     8 x 8192  859 / 843 / 826
//     8 x 10000  1070 / 1038 / 1010    8 x 8192, half of the tokens absent  430 / 430 / 424
//   48 KiB (6 KiB fp8 rows, top-8)     8 x 4096   338 / 337 / 325     8 x 8192  744 / 730 / 710
//   64 KiB (8 KiB rows, top-8 of 64)   8 x 4096   428 / 442 / 431     8 x 8192   -  / 974 / 941
//  112 KiB (14 KiB rows, top-8)        8 x 4096   852 /  -  / 845     8 x 8192 1682 /  -  / 1679
//   40 KiB (10 KiB rows, top-4 of 32)  8 x 4096   328 / 332 / 311     8 x 8192   -  / 672 / 620
//   32 KiB (8 KiB rows, top-4 of 32)   8 x 4096    -  / 225 / 208     8 x 8192   -  / 531 / 472
//   32 KiB (4 KiB fp8 rows, top-8)     8 x 509   33.6 /  -  / 37.1    8 x 2048  108 / 109 / 107
//     8 x 4096    209 / 212 / 206      8 x 6000   320 / 330 / 367     8 x 8192  458 / 478 / 584
//   25 KiB (4 KiB rows, top-6 of 64)   8 x 4096   155 / 159 /  -      8 x 1024 43.7 / 45.8 / -
//   24 KiB (3 KiB fp8 rows, top-8)     8 x 4096   157 / 162 / 172     8 x 8192  351 / 340 / 450
// and whole steps of 8 x 4096 tokens at 3 / 4 / 6 / 8 / 12 / 16 waves / full occupancy, side by side:
//   16 KiB (8 KiB rows, top-2)                         283 /  285 /  291 /  292 /  294 /  295 /  294
//   17 KiB (2 KiB fp8 rows with scales, top-8)         357 /  337 /  316 /  311 /  312 /  314 /  315
//   14 KiB (DSv3 fp8 rows, top-2)                      382 /  373 /  377 /  378 /  378 /  379 /  379
//    8 KiB (1 KiB fp8 rows with scales, top-8)         226 /  202 /  179 /  169 /  159 /  159 /  160
//    4 KiB (2 KiB fp8 rows with scales, top-2)         162 /  143 /  125 /  118 /  112 /  110 /  109
// (8 / 9 / 10 / 12: 8 x 4096 tokens, 16 KiB 106.7 / 107.2 / 107.6 / 108.6, 24 KiB 212.5 / 213.5 / 213.5 / 215.2; 8 x 1024,
// 13 KiB, step 67.9 at nine, 68.3 at ten)
// What a wave stores between 12 and 24 KiB of in rows of 4 KiB and more depends on the rows: those with scales, whose short
// stores hold a wave up, want nine waves from 8192 tokens on, the others four (steps on three buffer sets, four / nine: 4608-byte
// rows with scales, top-3, 46000 tokens 247.9 / 224.2, 20000 203.2 / 184.2, top-4, 39000 263.8 / 238.7; drawn ones with
// scales of more than 16384 tokens 0.965, of more than 8192 0.984, of up to 8192 0.998 of the time; 8 KiB rows without, top-2, 8 x
// 4096 tokens, skewed 266 / 278; rows of 7 KiB and more with scales beyond 16384 tokens, which in dispatches back to back are up
// to 8 % ahead with four, are level in steps: 1.00 over 59 drawn ones, 1.02 where tokens are absent).
// (one behind the other they lose: 8 x 4096 tokens of 8 KiB, top-2, skewed: 123 and 130; 2 KiB rows,
// top-6, 8 x 1024: 26.2 and 27.5).
// Rows in LDS (a2a_rows.h) spend more time in front of and between their stores and want more waves.  Us at 6 / 8 / 12 /
// 16 waves / as many as fit, side by side unless it says otherwise:
//   66 KiB (8656-byte rows, top-10 of 128)  2 x 1252  54.1 / 56.6 / 55.4 / 55.8 /  -
//   41 KiB (5264-byte rows, top-8 of 256)   8 x 513   42.0 / 44.1 / 43.3 /  -        8 x 2048  139 / 140 / 143 / 143
//     8 x 5000   339 / 339 / 342 (in turn 348 / 343 / 343; four waves 404, three 455)
//   48 KiB (8176-byte rows, top-6 of 64)    8 x 4097   347 / 348 / 359
//   40 KiB (8208-byte rows, top-5 of 40)    8 x 2100   137 / 138 / 139 (in turn 140)  8 x 6100  449 / 466 / 461 (in turn 443)
//   23 KiB (2976-byte rows, top-8 of 16)    4 x 4903   95.1 / 92.1 / 94.4 / 96.6
//   17 KiB (4240-byte rows, top-4 of 4)     4 x 6712   59.7 / 54.2 / 52.6 / 53.0
//    5 KiB (2528-byte rows, top-2 of 64)    8 x 8000    -  / 143 / 109 / 101 / 97.6
// and on two buffer sets in turn, at 12 / 16 / 25 waves / as many as fit:
//    9 KiB (3088-byte rows, top-3 of 64)    8 x 5000  110 / 106 / 105 / 106
//    8 KiB (1040-byte rows, top-8 of 64)    8 x 8000  175 / 161 / 158 / 153
//    8 KiB (2064-byte rows, top-4 of 64)    8 x 8000  152 / 139 / 136 / 138    8 x 1000  22.8 / 22.1 / 21.3 / 21.9
//    7 KiB (784-byte rows, top-10 of 64)    8 x 6000  108 / 95.1 / 83.9 / 80.9
//    6 KiB (3088-byte rows, top-2 of 64)    8 x 2000  34.4 / 31.6 / 30.0 / 29.8
struct ScatterPlan {
  uint32_t waves_per_cu;
  bool in_turn;
};

ScatterPlan scatter_plan(const WorldHost &w, uint32_t picks_per_wave) {
  if (w.lds_per_cu == 0) return {0, false};
  const uint64_t tokens = (uint64_t)w.G * w.M;
  const uint64_t row = w.Hb + 4ull * w.S;
  const uint64_t stored = (uint64_t)picks_per_wave * row;
  if (scatter_rows_in_lds(w)) {
    if (stored >= 32 * 1024) {
      if (tokens > 16384 && row >= 8192) return {6, true};
      return {tokens > 32768 ? 8u : 6u, false};
    }
    if (stored >= 20 * 1024) return {8, false};
    return {stored >= 12 * 1024 ? 12u : 0u, false};
  }
  if (stored >= 24 * 1024) {
    if (tokens <= 16384) return {4, false};
    if (stored >= 48 * 1024 || (stored >= 32 * 1024 && (row >= 8192 || tokens <= 32768))) return {3, true};
    return {stored >= 32 * 1024 || tokens <= 32768 ? 4u : 9u, false};
  }
  if (stored >= 12 * 1024) return {row >= 4096 && (w.S == 0 || tokens <= 8192) ? 4u : 9u, false};
  return {stored >= 6 * 1024 ? 12u : 0u, false};
}

// Dynamic LDS of a scatter workgroup (one wave): the row if it goes through LDS, and the share of a CU's LDS of which as
// many fit as the plan wants.  LDS is handed out in blocks of 1280 bytes, 128 to a CU (one-wave workgroups that hold 16384
// bytes run nine to a CU, with 15360 ten; 12288 and 12800 twelve).
constexpr uint32_t kLdsBlock = 1280;
uint32_t scatter_lds(const WorldHost &w, const ScatterPlan &plan) {
  const uint32_t share = plan.waves_per_cu ? w.lds_per_cu / kLdsBlock / plan.waves_per_cu * kLdsBlock : 0;
  return scatter_rows_in_lds(w) && share < w.Hb ? w.Hb : share;
}

// Rows that dispatch_scatter holds in registers (longer ones stream through dispatch_scatter_long).
bool scatter_has_register_rows(const WorldHost &w) { return (w.Hb / 16 + kWave - 1) / kWave <= 32; }

template <class DT>
int launch_scatter_t(const WorldHost &w, const DT &tab, Slots slots, hipStream_t s) {
  const uint32_t tokens = w.G * w.M;
  if (!scatter_has_register_rows(w)) {
    return launch_kernel(dispatch_scatter_long<DT>, dim3(tokens), dim3(256), 0, s, w, tab);
  }
  const uint32_t ksplit = pick_ksplit(w, kWave);
  const uint32_t kper = (w.K + ksplit - 1) / ksplit;
  const uint64_t waves = (uint64_t)tokens * ksplit;
  // One wave per workgroup, and few of them per CU at a time.  A wave reads one row and then
  // has up to K rows of stores to issue; HBM takes those stores best when a CU sends the rows of
  // a few waves at a time (three or four where each stores much) rather than those of thirty-two
  // interleaved (figures at scatter_plan).  The hardware has no such knob, so each workgroup asks for a share of
  // the CU's LDS that only that many fit into.
  const ScatterPlan plan = scatter_plan(w, kper);
  const bool staged = scatter_rows_in_lds(w);
  const uint32_t lds = scatter_lds(w, plan);
  const dim3 grid((uint32_t)waves + (slots == Slots::kTables ? (w.E + 7) / 8 : 0u)), block(kWave);
#define PPLX_ROW_KERNEL_ARGS ksplit, kper
#define PPLX_LAUNCH_LARGE_ROW_VARIANT(KERNEL)                                                    \
  do {                                                                                           \
    if (per_lane <= 16) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 16, false);                              \
    else PPLX_LAUNCH_ROW_VARIANT(KERNEL, 32, false);                                             \
  } while (0)
  if (slots == Slots::kMap) {
    if (staged) PPLX_LAUNCH_ROW_VARIANT(dispatch_scatter, 0, false);
    else PPLX_DISPATCH_ROW_VARIANTS(dispatch_scatter);
  }
#undef PPLX_LAUNCH_LARGE_ROW_VARIANT
  // (rows beyond 16 KiB leave no registers for the slot arithmetic: slots_of() sends them through
  // route_slots and the kernel above)
#define PPLX_LAUNCH_LARGE_ROW_VARIANT(KERNEL)                                                    \
  do {                                                                                           \
    if (per_lane <= 16) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 16, false);                              \
    else return (int)hipErrorInvalidValue;                                                       \
  } while (0)
#undef PPLX_LAUNCH_ROW_VARIANT
#define PPLX_LAUNCH_ROW_VARIANT(KERNEL, NV, EXACT)                                               \
  do {                                                                                           \
    if (plan.in_turn) return launch_kernel(KERNEL<NV, EXACT, DT, true>, grid, block, lds, s, w, tab, ksplit, kper); \
    return launch_kernel(KERNEL<NV, EXACT, DT, false>, grid, block, lds, s, w, tab, ksplit, kper); \
  } while (0)
  if (slots == Slots::kScanned) {
    if (staged) PPLX_LAUNCH_ROW_VARIANT(dispatch_scatter_scanned, 0, false);
    else PPLX_DISPATCH_ROW_VARIANTS(dispatch_scatter_scanned);
  } else if (slots == Slots::kTables) {
    if (staged) PPLX_LAUNCH_ROW_VARIANT(dispatch_scatter_slots, 0, false);
    else PPLX_DISPATCH_ROW_VARIANTS(dispatch_scatter_slots);
  }
#undef PPLX_LAUNCH_ROW_VARIANT
#undef PPLX_LAUNCH_LARGE_ROW_VARIANT
#undef PPLX_ROW_KERNEL_ARGS
  return (int)hipErrorInvalidValue;
}

template <class DT>
int launch_fused_t(const WorldHost &w, const DT &tab, uint32_t pick_vector, hipStream_t s) {
  const uint32_t tokens = w.G * w.M;
  const uint32_t kWaves = fused_waves(w);
  const uint32_t tokens_per_block = fused_tokens_per_block(tokens, kWaves);
  // Steps of fewer than 1024 tokens spread each token's picks over several waves; rows in LDS, which the waves
  // share, up to 4096 (4240-byte rows, top-4, 1024 tokens 8.0 us at one wave per token, 7.7 at all of a
  // workgroup's; 15984-byte rows, top-4 17.8 and 17.2; 5264-byte rows, top-8, 2048 tokens 21.3 and 21.2).
  const bool staged = fused_rows_in_lds(w);
  const uint64_t spread_below = staged ? 4096 : 1024;
  uint32_t ksplit = 1;
  while (ksplit * 2 <= w.K && tokens_per_block * ksplit * 2 <= kWaves && (uint64_t)tokens * ksplit < spread_below) ksplit *= 2;
  const uint32_t kper = (w.K + ksplit - 1) / ksplit;
  const dim3 grid((tokens + tokens_per_block - 1) / tokens_per_block), block(kWaves * kWave);
  const uint32_t lds = fused_lds_bytes(w) + (staged ? tokens_per_block * w.Hb : 0u);
  // Rows that fit the last-level cache with room to spare are written through into it.
  const uint64_t row_bytes = (uint64_t)tokens * w.K * (w.Hb + 4ull * w.S);
  const uint32_t write_through = row_bytes <= (staged ? kLdsWriteThroughMaxBytes : kWriteThroughMaxBytes) ? 1u : 0u;
  const FusedShape shape{ksplit, kper, tokens_per_block, pick_vector, write_through};
#define PPLX_ROW_KERNEL_ARGS shape
#define PPLX_LAUNCH_ROW_VARIANT(KERNEL, NV, EXACT)                                                              \
  do {                                                                                                          \
    if (w.K > 8) return launch_kernel(KERNEL<NV, EXACT, DT, true>(), grid, block, lds, s, w, tab, PPLX_ROW_KERNEL_ARGS); \
    return launch_kernel(KERNEL<NV, EXACT, DT, false>(), grid, block, lds, s, w, tab, PPLX_ROW_KERNEL_ARGS);    \
  } while (0)
#define PPLX_LAUNCH_LARGE_ROW_VARIANT(KERNEL) return (int)hipErrorInvalidValue
  if (staged) PPLX_LAUNCH_ROW_VARIANT(fused_kernel, 0, false);
  else PPLX_DISPATCH_ROW_VARIANTS(fused_kernel);
#undef PPLX_LAUNCH_LARGE_ROW_VARIANT
#undef PPLX_LAUNCH_ROW_VARIANT
#undef PPLX_ROW_KERNEL_ARGS
  return (int)hipErrorInvalidValue;
}

// Steps of several tiles leave the last routing launch out (the scatter's waves work their own
// slots out of the tiles' tables), and the scan too as long as an expert's counts are one line.
Slots slots_of(const WorldHost &w) {
  if (w.num_tiles == 1 || (w.Hb / 16 + kWave - 1) / kWave > 16) return Slots::kMap;
  return w.num_tiles <= kScanFreeTiles ? Slots::kTables : Slots::kScanned;
}

template <class DT>
int launch_dispatch_t(const WorldHost &w, const DT &tab, uint32_t pick_vector, hipStream_t s) {
  if (dispatch_is_fused(w)) return launch_fused_t(w, tab, pick_vector, s);
  RouteSpan span{};
  span.v_begin = 0;
  span.v_count = w.G * w.M;
  span.tile_chunks = w.tile_chunks;
  span.pick_vector = pick_vector;
  span.tile_cnt = w.tile_cnt;
  span.slot_out = w.slot_map;
  const Slots slots = slots_of(w);
  if (slots != Slots::kMap) {
    const RouteTables tables = route_tables(w.num_tiles, w.tile_chunks, w.E);
    uint8_t *base = reinterpret_cast<uint8_t *>(w.tile_cnt);
    span.tile_mask = reinterpret_cast<unsigned long long *>(base + tables.mask_offset);
    span.chunk_base = reinterpret_cast<uint16_t *>(base + tables.base_offset);
    if (slots == Slots::kTables) span.tile_row = reinterpret_cast<uint16_t *>(base);
  }
  int err = launch_route_t(w, tab, span, s);
  if (err) return err;
  return launch_scatter_t(w, tab, slots, s);
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
uint32_t route_lds_bytes(uint32_t num_experts, uint32_t tile_chunks) {
  return tile_chunks * num_experts * (uint32_t)(sizeof(unsigned long long) + sizeof(uint32_t));
}

bool dispatch_is_fused(const WorldHost &w) {
  if (fused_lds_bytes(w) > 60 * 1024) return false;
  const bool in_lds = fused_rows_in_lds(w);
  if (in_lds && w.Hb > 16 * 1024) return false;
  // One launch while a workgroup per CU can own all tokens, one wave each: 4096 tokens, or 2048 of
  // rows that take 512-thread workgroups (beyond that a second round of workgroups recounts
  // everything: 8 ranks, 2 KiB rows, top-6 of 64: 4096 tokens 15.0 us against 15.9 with the routing
  // in a launch of its own, 5120 tokens 24.2 against 20.0; 14 KiB rows, top-8: 2048 tokens 53.0 / 54.6,
  // 2560 65.8 / 61.3).  All of a workgroup's row waves store at once, though, where the scatter keeps few
  // storing waves per CU, and that costs more than the routing launch once the rows fill the last-level
  // cache.  Where that is depends on the rows; on 8 ranks, top-8 (us, one launch / routing + scatter; MiB of
  // rows stored):
  //   fp8 rows with scales, 7 KiB: 108 29.5 / 30.4, 116 31.1 / 31.8, 130 34.1 / 33.8, 144 37.3 / 36.5,
  //     159 42.1 / 40.9; 6 KiB: 111 29.0 / 31.2, 148 36.4 / 36.7; 5 KiB: 124 33.2 / 31.1, 144 37.2 / 36.0;
  //     4 KiB: 107 26.9 / 29.1, 116 28.8 / 33.8, 132 32.0 / 32.7
  //   whole lines only (no scales), 8 KiB: 116 28.6 / 30.5, 144 34.5 / 36.9, 160 37.8 / 42.2, 176 40.7 /
  //     42.8, 192 45.2 / 45.8; 7 KiB: 126 30.8 / 33.4, 140 33.9 / 35.8, 154 36.5 / 38.7; the same with half of
  //     the tokens absent (8 KiB, 144: 21.3 / 23.2), and for 8 KiB rows with scales (148 35.5 / 37.9,
  //     182 42.8 / 44.2): these run up to 176
  // Picks that are not counted four at a time, or more than eight, run up to 112 (120 in steps of up to 1024 tokens).
  // That is safe for all of them, and short of where the forms come level for most: 8 KiB rows, top-5 80 21.3 / 23.4,
  // 160 39.8 / 38.3; top-9 144 35.5 / 36.2; top-10 160 38.4 / 38.7; top-12 192 45.1 / 44.9; up to 1024 tokens the slots
  // take a launch of a single workgroup, and one launch is ahead beyond 120 too (top-16 128 31.1 / 43.6).
  const uint64_t tokens = (uint64_t)w.G * w.M;
  const uint32_t waves = fused_waves(w);
  const uint64_t stored = tokens * w.K * (w.Hb + 4ull * w.S);
  if (tokens > 256u * waves) return false;
  // Picks beyond eight weigh more, the most where they can only be fetched one by one or do not fit the registers
  // (us, one launch / routing + scatter): 2 KiB rows, top-9 1024 tokens 9.8 / 16.6, 2048 16.9 / 14.9, 4096 31.0 / 21.9;
  // 8 KiB rows, top-9 2048 35.5 / 36.2; 4720-byte rows, top-9 2048 29.9 / 30.2, 4096 54.3 / 45.2; 2 KiB rows, top-24 1024
  // 21.4 / 32.2, 2048 40.0 / 28.4; top-32 1024 28.5 / 45.2.  (2 KiB rows, top-10 2048 14.3 / 15.9, 4096 23.8 / 24.6; top-16
  // 2048 19.3 / 21.5.)
  if (tokens > 1024 && w.K > 16) return false;
  if (tokens > 1024 && w.K > 8 && w.K % 2 != 0 && (w.Hb < 4096 || tokens > 2048)) return false;
  // Rows in LDS, dispatch + combine on three buffer sets, us, one launch / two:
  //   cutting half lines, MiB     150           169           180           192           205
  //     5264 bytes, top-10         71.5 / 72.6   81.6 / 83.7                 88.4 / 88.7   94.7 / 94.5
  //     6160 bytes, top-8          71.1 / 75.6   80.2 / 82.8   83.3 / 84.8   88.6 / 89.8
  //     8176 bytes, top-6          74.2 / 78.0   80.3 / 83.0   85.0 / 86.2   90.3 / 90.7
  //     12016 bytes, top-8         70.6 / 79.4   75.5 / 82.1   81.4 / 85.9   89.1 / 92.6
  //     4240 bytes, top-12         69.0 / 70.8   78.1 / 81.6   83.2 / 84.8   88.3 / 87.9
  //   whole half lines: 13312 bytes, top-5 102 52.6 / 53.6, 130 62.6 / 63.0, 169 82.0 / 81.0, top-3 107 57.1 / 57.6, 117 61.0 /
  //     60.6; 9216 bytes, top-4 72 38.0 / 40.4, 99 51.0 / 51.6, 117 59.2 / 59.1, top-1, 4096 tokens 32.8 / 34.2; 9280 bytes, top-4
  //     85 44.6 / 45.8; 11264 bytes, top-8 129 59.5 / 62.3, 146 68.6 / 70.0; 10304 bytes, top-4 156 77.0 / 74.1
  if (in_lds) {
    const uint64_t rows = (uint64_t)fused_tokens_per_block((uint32_t)tokens, waves) * w.Hb;
    const uint64_t limit = row_cuts_half_lines(w) ? 180ull << 20 : 128ull << 20;
    // (a device that does not say how much LDS it has is taken to have the 64 KiB of any)
    const uint32_t lds = w.lds_per_cu ? w.lds_per_cu : 64u << 10;
    return fused_lds_bytes(w) + rows <= lds && stored <= limit;
  }
  if (waves < 16) return true;
  const bool quick_count = w.K % 4 == 0 && w.K <= 8;
  const bool whole_lines = w.S == 0 || w.Hb >= 8192;
  uint64_t limit = 112ull << 20;
  if (quick_count || (tokens <= 1024 && w.K <= 16)) limit = 120ull << 20;
  if (quick_count && whole_lines && tokens <= 3072) limit = 176ull << 20;
  return stored <= limit;
}

DispatchPlan dispatch_plan(const WorldHost &w) {
  if (dispatch_is_fused(w)) return {DispatchForm::kOneLaunch, 0, false, fused_rows_in_lds(w)};
  const Slots slots = slots_of(w);
  const DispatchForm form = slots == Slots::kMap      ? DispatchForm::kSlotMap
                            : slots == Slots::kTables ? DispatchForm::kTables
                                                      : DispatchForm::kScannedTables;
  if (!scatter_has_register_rows(w)) return {form, 0, false, false};
  const uint32_t ksplit = pick_ksplit(w, kWave);
  const ScatterPlan plan = scatter_plan(w, (w.K + ksplit - 1) / ksplit);
  uint32_t waves = plan.waves_per_cu;
  if (waves) {  // (fewer where the rows take more than their share)
    const uint32_t blocks = (scatter_lds(w, plan) + kLdsBlock - 1) / kLdsBlock;
    const uint32_t fit = w.lds_per_cu / kLdsBlock / (blocks ? blocks : 1);
    if (waves > fit) waves = fit;
  }
  return {form, waves, plan.in_turn && slots != Slots::kMap, scatter_rows_in_lds(w)};
}

int launch_bind_dispatch(DispatchRank *table, const BindDispatchBatch &b, void *stream) {
  return launch_kernel(bind_rows<BindDispatchBatch, DispatchRank>, dim3(1), dim3(256), 0, (hipStream_t)stream, table, b);
}

int launch_bind_combine(CombineRank *table, const BindCombineBatch &b, void *stream) {
  return launch_kernel(bind_rows<BindCombineBatch, CombineRank>, dim3(1), dim3(256), 0, (hipStream_t)stream, table, b);
}

int launch_dispatch(const WorldHost &w, const DispatchRank *inline_rows, uint32_t pick_vector, void *stream) {
  if (pick_vector != 4 && pick_vector != 2) pick_vector = 1;
  return with_table<InlineDispatch>(w, inline_rows, HbmDispatch{w.drank}, [&](const auto &tab) {
    return launch_dispatch_t(w, tab, pick_vector, (hipStream_t)stream);
  });
}

}  // namespace pplx_amd
