// gfx950 combine kernel of the MoE dispatch / combine path: the top-k weighted
// gather-reduce (also the SEND phase of a split combine, with its output rows in the staging area).
#include "a2a_common.h"

namespace pplx_amd {
namespace {

// ---------------------------------------------------------------------------
// Combine: out[t, :] = (U) sum_k w[t, k] * (float) expert_y[e_k][slot(t, k), :]
// with k ascending and fp32 accumulation
// (csrc/all_to_all/intranode_combine.cu:141-168).
// ---------------------------------------------------------------------------
// What a lane has of a piece of a row (64 x 8 elements): where it lies, how it is fetched and stored.  In 16-bit rows that
// is one vector of 8 elements.  In fp32 rows it is two vectors of 4 elements that lie 1 KiB apart, so that every load of
// the wave covers whole lines: with the 32 bytes of 8 elements in one lane each of the two loads touches all lines of 2 KiB
// and takes half of each.  Combine alone on three buffer sets, us, 8 elements in one lane / two vectors apart: 7168 wide, top-8,
// 8 x 128 tokens 46.0 / 41.5, 8 x 1024 381.8 / 347.4; 512 wide, top-8, 8 x 2048 56.7 / 47.8; 4096 wide, top-2, 8 x 2048
// 118.1 / 110.0, top-1 72.5 / 66.1; 520 wide, top-6, 8 x 1024 25.7 / 21.4; 2880 wide, top-5, groups of four, 3001 tokens
// 50.6 / 46.1 (242 MB: 4.8 -> 5.25 TB/s).  The stores, 8 bytes a lane, still cover whole lines: lanes that swap halves in
// pairs to store 16 bytes each measured the same (4200 steps: 1.000).
template <typename U> struct OutVectors;
template <> struct OutVectors<__bf16> {
  typedef __bf16 by4 __attribute__((ext_vector_type(4)));
  typedef bf16x8 by8;
};
template <> struct OutVectors<_Float16> {
  typedef _Float16 by4 __attribute__((ext_vector_type(4)));
  typedef f16x8 by8;
};

// Streaming or plain.  (By the compiler's own stores: it sees to what may follow a 16-byte store, which it does not know in
// inline asm to be one, before the registers stored are written again.)
template <RowStore POLICY, typename V> __device__ __forceinline__ void out_store(V v, PPLX_GLOBAL V *p) {
  static_assert(POLICY == RowStore::kStream || POLICY == RowStore::kPlain, "out_store");
  if constexpr (POLICY == RowStore::kStream) __builtin_nontemporal_store(v, p);
  else *p = v;
}

template <typename T> struct Row8;
template <> struct Row8<float> {
  struct Raw {
    f32x4 a, b;
  };
  struct Place {
    uint32_t a, b;  // in vectors of 4 elements
  };
  static __device__ __forceinline__ Place place(uint32_t piece, uint32_t lane) {
    return Place{2 * piece * kWave + lane, (2 * piece + 1) * kWave + lane};
  }
  // (beyond the row its last vector is fetched: loads stay unconditional)
  static __device__ __forceinline__ Place clamped(Place p, uint32_t H) {
    const uint32_t last = H / 4 - 1;
    return Place{p.a < last ? p.a : last, p.b < last ? p.b : last};
  }
  static __device__ __forceinline__ Raw load(uint64_t row, Place p) {
    const PPLX_GLOBAL f32x4 *x = global_cptr<f32x4>(row);
    return Raw{__builtin_nontemporal_load(x + p.a), __builtin_nontemporal_load(x + p.b)};
  }
  static __device__ __forceinline__ f32x8 widen(const Raw &r) {
    return __builtin_shufflevector(r.a, r.b, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  // N rows held as 2 N registers of 16 bytes
  template <int N> static __device__ __forceinline__ void settle(Raw *raw) {
    SettleAll<2 * N>::of(reinterpret_cast<f32x4 *>(raw));
  }
  template <typename U, RowStore POLICY>
  static __device__ __forceinline__ void store(uint64_t row, Place p, uint32_t H, const f32x8 &acc) {
    typedef typename OutVectors<U>::by4 vec_t;
    PPLX_GLOBAL vec_t *out = global_ptr<vec_t>(row);
    const f32x4 a = __builtin_shufflevector(acc, acc, 0, 1, 2, 3), b = __builtin_shufflevector(acc, acc, 4, 5, 6, 7);
    if (p.a < H / 4) out_store<POLICY>(__builtin_convertvector(a, vec_t), out + p.a);
    if (p.b < H / 4) out_store<POLICY>(__builtin_convertvector(b, vec_t), out + p.b);
  }
};
// The 16-bit types.
template <typename V> struct Row8By16 {
  typedef V Raw;
  typedef uint32_t Place;  // in vectors of 8 elements
  static __device__ __forceinline__ Place place(uint32_t piece, uint32_t lane) { return piece * kWave + lane; }
  static __device__ __forceinline__ Place clamped(Place p, uint32_t H) {
    const uint32_t last = H / 8 - 1;
    return p < last ? p : last;
  }
  static __device__ __forceinline__ Raw load(uint64_t row, Place p) {
    return __builtin_nontemporal_load(global_cptr<V>(row) + p);
  }
  template <int N> static __device__ __forceinline__ void settle(Raw *raw) { SettleAll<N>::of(raw); }
  template <typename U, RowStore POLICY>
  static __device__ __forceinline__ void store(uint64_t row, Place p, uint32_t H, const f32x8 &acc) {
    typedef typename OutVectors<U>::by8 vec_t;
    if (p < H / 8) out_store<POLICY>(__builtin_convertvector(acc, vec_t), global_ptr<vec_t>(row) + p);
  }
};
template <> struct Row8<__bf16> : Row8By16<u32x4> {
  static __device__ __forceinline__ f32x8 widen(const Raw &raw) {
    f32x8 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      out[2 * i] = __uint_as_float(raw[i] << 16);
      out[2 * i + 1] = __uint_as_float(raw[i] & 0xffff0000u);
    }
    return out;
  }
};
template <> struct Row8<_Float16> : Row8By16<f16x8> {
  static __device__ __forceinline__ f32x8 widen(const Raw &raw) { return __builtin_convertvector(raw, f32x8); }
};

// N picks starting at k, VPL vectors of each: all N * VPL loads are issued before the first is used.
template <typename T, int N, int VPL>
__device__ __forceinline__ void gather_group(f32x8 (&acc)[VPL], uint64_t row_of_lane, float weight_of_lane,
                                             uint32_t k, const typename Row8<T>::Place (&at)[VPL]) {
  typename Row8<T>::Raw raw[VPL][N];
#pragma unroll
  for (int v = 0; v < VPL; ++v) {
#pragma unroll
    for (int i = 0; i < N; ++i) raw[v][i] = Row8<T>::load(read_lane64(row_of_lane, k + i), at[v]);
  }
  Row8<T>::template settle<VPL * N>(&raw[0][0]);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float wk = __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight_of_lane), (int)(k + i)));
#pragma unroll
    for (int v = 0; v < VPL; ++v) acc[v] += wk * Row8<T>::widen(raw[v][i]);
  }
}

constexpr uint32_t kWavesPerBlock = 4;

// The sum of one output row's piece: lane `base + k` holds the row and the weight of pick k.
template <typename T, int KB, int VPL>
__device__ __forceinline__ void reduce_picks(f32x8 (&acc)[VPL], uint32_t K, uint64_t row, float weight, uint32_t base,
                                             bool all_rows, const typename Row8<T>::Place (&at)[VPL]) {
#pragma unroll
  for (int v = 0; v < VPL; ++v) acc[v] = f32x8{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (!all_rows) {
    // A pick without a row (bad expert id or slot) contributes nothing.
    for (uint32_t k = 0; k < K; ++k) {
      if (read_lane64(row, base + k) != 0) gather_group<T, 1, VPL>(acc, row, weight, base + k, at);
    }
    return;
  }
  uint32_t k = 0;
  for (; k + KB <= K; k += KB) gather_group<T, KB, VPL>(acc, row, weight, base + k, at);
  if constexpr (KB > 4) {
    if ((K - k) & 4) { gather_group<T, 4, VPL>(acc, row, weight, base + k, at); k += 4; }
  }
  if constexpr (KB > 2) {
    if ((K - k) & 2) { gather_group<T, 2, VPL>(acc, row, weight, base + k, at); k += 2; }
  }
  if constexpr (KB > 1) {
    if ((K - k) & 1) { gather_group<T, 1, VPL>(acc, row, weight, base + k, at); }
  }
}

// One wave owns VPL * 64 consecutive 8-element vectors of one output row (VPL KiB of a bf16
// row) and takes the picks KB at a time, so KB * VPL row loads per lane are in flight
// (which of the two: launch_combine_k).
//
// GROUPED (DP groups of several ranks, dp * K <= 64): the members of a group hold the same
// tokens, so the rows they gather are the same ones.  A wave then serves the token for all
// members: lane i * K + k resolves pick k of member i, and members whose rows and weights agree
// with those of the first present member (compared bit for bit, token by token: the operator
// takes every rank's own indices and weights) share one gather and only store apart.  What is
// bound by the gathered bytes moves up to dp times fewer of them: 8 ranks in groups of four, 3001
// tokens of fp32 rows, 2880 wide, top-5: 150 us with a gather per rank, 54 us with one per
// group (242 MB at 4.5 TB/s); groups of two, 4 x 128 bf16 tokens, 7168 wide, top-8: 16.5 and 15.0
// us (the second gather of a step this small hits the last-level cache).  Members that do not agree are
// gathered for one after the other by the same wave: if every token's weights differ, a step of 4 x 128
// tokens takes 41 us where a gather per rank takes 33 (groups of four, 2 x 128: 36 and 25), one of 4 x
// 1024 tokens 267 and 275.  Copies of a token carry the same weights, so nothing is made of that case.
template <typename T, typename U, class CT, int KB, int VPL, bool GROUPED>
__global__ __launch_bounds__(kWavesPerBlock * kWave) void combine_gather(WorldDev w, CT tab, uint32_t segments,
                                                                         FastDiv by_segments, uint32_t plain_stores) {
  const uint32_t lane = lane_id();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave);
  const uint32_t token = fast_div(wave, by_segments);
  const uint32_t segment = wave - token * segments;
  const uint32_t owner_index = group_of(w, token);  // the rank, or the DP group when GROUPED
  const uint32_t t = token - owner_index * w.M;
  if (owner_index >= (GROUPED ? w.G : w.R)) return;
  const uint32_t member = GROUPED ? fast_div(lane, w.by_K) : 0;
  const uint32_t pick = lane - member * w.K;
  const bool has_pick = GROUPED ? member < w.dp : lane < w.K;
  const uint32_t g = GROUPED ? owner_index : fast_div(owner_index, w.by_dp);
  const CombineRank &c = tab.at(GROUPED ? g * w.dp + (has_pick ? member : 0) : owner_index);
  bool present = t < combine_rank_tokens(w, c);
  if constexpr (!GROUPED) {
    if (!present) return;
  }
  present = present && has_pick;
  if (GROUPED && __builtin_amdgcn_ballot_w64(present) == 0) return;

  // Lane k (of its member) resolves pick k: no LDS, no barrier.
  uint64_t row = 0;
  float weight = 0.f;
  if (present) {
    const uint32_t e = as_global(c.indices)[(size_t)t * w.K + pick];
    const uint32_t slot = as_global(w.slot_map)[((size_t)g * w.M + t) * w.K + pick];
    weight = as_global(c.weights)[(int64_t)t * c.w_stride_row + pick];
    if (e < w.E && slot != kInvalidSlot) {
      // (the buffer and its length in one trip, not the one behind the other)
      const CombineRank &owner = tab.at(owner_of(w, e));
      const uint32_t y_rows = owner.y_rows;
      uint64_t address = reinterpret_cast<uint64_t>(reinterpret_cast<const T *>(owner.expert_y) +
                                                    (int64_t)local_of(w, e) * owner.y_stride_expert +
                                                    (int64_t)slot * owner.y_stride_row);
      settle(address);
      if (slot < y_rows) {
        row = address;
      } else if (segment == 0) {
        atomicOr(w.faults, kFaultBadSlot);
      }
    }
  }
  const uint64_t no_row = __builtin_amdgcn_ballot_w64(present && row == 0);

  const uint64_t out = reinterpret_cast<uint64_t>(reinterpret_cast<U *>(c.out_tokens) + (int64_t)t * c.out_stride_row);
  typedef Row8<T> Row;
  typename Row::Place at[VPL];
#pragma unroll
  for (int v = 0; v < VPL; ++v) at[v] = Row::clamped(Row::place(segment * VPL + v, lane), w.H);
  f32x8 acc[VPL];
  auto store = [&](uint64_t out) {
    if (plain_stores) {
      // (fenced: stores of two branches that differ in their hint alone would be made one, without the hint)
      asm volatile("" ::: "memory");
#pragma unroll
      for (int v = 0; v < VPL; ++v)
        Row::template store<U, RowStore::kPlain>(out, Row::place(segment * VPL + v, lane), w.H, acc[v]);
      asm volatile("" ::: "memory");
      return;
    }
#pragma unroll
    for (int v = 0; v < VPL; ++v)
      Row::template store<U, RowStore::kStream>(out, Row::place(segment * VPL + v, lane), w.H, acc[v]);
  };
  if constexpr (!GROUPED) {
    reduce_picks<T, KB, VPL>(acc, w.K, row, weight, 0, no_row == 0, at);
    store(out);
  } else {
    const uint64_t picks = w.K == kWave ? ~0ull : (1ull << w.K) - 1;
    // one lane per present member
    for (uint64_t todo = __builtin_amdgcn_ballot_w64(present && pick == 0); todo != 0;) {
      const uint32_t base = (uint32_t)__builtin_ctzll(todo);
      // members that want the same sum: every pick's row and weight as this member's
      const int src = (int)((base + pick) & (kWave - 1));
      const bool same = __shfl((uint32_t)row, src, kWave) == (uint32_t)row &&
                        __shfl((uint32_t)(row >> 32), src, kWave) == (uint32_t)(row >> 32) &&
                        __shfl(__float_as_uint(weight), src, kWave) == __float_as_uint(weight);
      const uint64_t differs = __builtin_amdgcn_ballot_w64(present && !same);
      reduce_picks<T, KB, VPL>(acc, w.K, row, weight, base, ((no_row >> base) & picks) == 0, at);
      for (uint64_t rest = todo; rest != 0; rest &= rest - 1) {
        const uint32_t head = (uint32_t)__builtin_ctzll(rest);
        if (((differs >> head) & picks) != 0) continue;
        store(read_lane64(out, head));
        todo &= ~(1ull << head);
      }
    }
  }
}

// DP groups of several ranks gather once per group as long as a wave has a lane for every member's
// pick; beyond that (no routing in use comes near) every rank gathers for itself.  So it does in steps
// whose ranks gather up to 10 MiB together: there the bytes cost less than the longer chain in front of
// them (dispatch + combine, us, per rank / per group, at the MiB that all ranks gather): 8 ranks in groups
// of two, 7168-wide bf16, top-8: 14 12.5 / 12.8, 19 14.4 / 13.8, 64 28.2 / 22.9; 2048 wide, top-6: 3 10.8 / 11.3,
// 14 14.0 / 13.7; 4096 wide, top-2: 8 10.7 / 11.4, 14 12.9 / 13.3, 32 20.6 / 19.3; groups of four, 7168 wide:
// 3.5 10.3 / 10.7, 19 14.3 / 12.8; 1024-wide f16, top-4: 8 10.2 / 11.1, 14 11.5 / 11.8, 32 14.6 / 13.9; 2880-wide
// fp32, top-5: 7 11.0 / 11.8, 14 13.9 / 12.6; 64 ranks in groups of four, 10 13.8 / 12.6.
constexpr uint64_t kGroupGatherMinBytes = 10ull << 20;
bool combine_per_group(const WorldHost &w, size_t elem_bytes) {
  return w.dp > 1 && w.dp * w.K <= kWave &&
         (uint64_t)w.R * w.M * w.K * w.H * elem_bytes > kGroupGatherMinBytes;
}

// Combined rows whose length is no multiple of half a 128-byte line, the unit in which memory takes writes, begin anywhere:
// stores that stream past the caches cut half lines there, and a small step's kernel ends waiting for those partial writes.
// Plain stores meet in the caches first.  Dispatch + combine on three buffer sets, 8 ranks, top-2 of 32, us, streaming /
// plain: 2968 wide, 8 x 16 tokens 7.3 / 7.0, 8 x 64 8.6 / 8.3, 8 x 128 (5.8 MiB) 11.3 / 10.8; 5384 wide, 8 x 64 (5.3 MiB) 10.9 / 10.4;
// 2008 wide, top-4, 8 x 128 12.2 / 11.8; groups of two, top-3, 2968 wide, 8 x 100 9.9 / 9.6 (45 shapes of groups of two 0.97).
// Beyond, the lines that stay behind cost what follows more than that: plain stores for 5384 wide, top-4, 8 x 200 34.5 / 37.8, 7176
// wide, top-2, 8 x 256 35.2 / 40.8.  Both kinds of store over 488 to 7176 wide rows, top-1 to top-8, groups of one, two and four, plain
// over streaming, mean (lowest to highest): 252 steps of 1 to 5.9 MiB 0.977 (0.943 to 1.019; top-8 0.98), 48 of 6.2 and 7 MiB 0.985 (to
// 1.016), 60 of 8 MiB 0.999 (0.969 to 1.043), 24 of 10 MiB 1.002 (to 1.058), 60 of 12 MiB 1.007 (to 1.084), 48 of 16 and 24 MiB 1.013
// (to 1.116): 6 MiB is where the worst of them begin to lose.  Rows are counted for every rank, present or not, as in all
// rules here.  Rows of whole half lines are level in small steps.  (The same in dispatch, plain instead of
// written-through stores, gives 2 % of the smallest steps and costs 6 % at 8 x 128 tokens; pieces that begin at half lines of the
// output instead of the row's start gave nothing in large steps.)
constexpr uint64_t kPlainStoresMaxBytes = 6ull << 20;
bool plain_stores(const WorldDev &w) {
  const uint64_t row = 2ull * w.H;
  return row % 64 != 0 && (uint64_t)w.R * w.M * row <= kPlainStoresMaxBytes;
}

template <typename T, typename U, class CT, int KB, int VPL>
int launch_combine_v(const WorldHost &w, const CT &tab, bool grouped, hipStream_t s) {
  static_assert(sizeof(WorldDev) + sizeof(HbmCombine) + 2 * sizeof(uint32_t) + sizeof(FastDiv) <= kShortArguments,
                "arguments of combine_gather");
  const uint32_t nvec_segments = (w.H / 8 + kWave - 1) / kWave;
  const uint32_t segments = (nvec_segments + VPL - 1) / VPL;
  const uint64_t waves = (uint64_t)(grouped ? w.G : w.R) * w.M * segments;
  const dim3 grid((uint32_t)((waves + kWavesPerBlock - 1) / kWavesPerBlock)), block(kWavesPerBlock * kWave);
  const FastDiv by_segments = make_fast_div(segments);
  const uint32_t plain = plain_stores(w) ? 1 : 0;
  if (grouped)
    return launch_kernel(combine_gather<T, U, CT, KB, VPL, true>, grid, block, 0, s, w, tab, segments, by_segments, plain);
  return launch_kernel(combine_gather<T, U, CT, KB, VPL, false>, grid, block, 0, s, w, tab, segments, by_segments, plain);
}

// Whether 8 KiB pieces of a 16-bit row make workgroups that come out even, two to four of them to each of the 256 CUs,
// with at most 1 KiB of padding to a piece.
bool even_pieces(uint64_t tokens, uint32_t segments) {
  const uint32_t pieces = (segments + 7) / 8;
  if (pieces * 8 - segments > pieces) return false;
  const uint64_t workgroups = (tokens * pieces + kWavesPerBlock - 1) / kWavesPerBlock;
  const uint64_t per_cu = (workgroups + 255) / 256;
  return per_cu >= 2 && per_cu <= 4 && 256 * per_cu - workgroups <= 16;
}

// How pieces of 7 KiB (whole rows of them) or 8 KiB of a 16-bit row fall on the 256 CUs: the most workgroups that one
// gets, and whether those of all CUs and the padding of the pieces leave less than a quarter of it idle.
struct LongPieces {
  uint64_t per_cu;
  bool even;
};
LongPieces long_pieces(uint64_t tokens, uint32_t segments) {
  const uint32_t length = segments % 7 == 0 ? 7 : 8;
  const uint32_t pieces = (segments + length - 1) / length;
  const uint64_t workgroups = (tokens * pieces + kWavesPerBlock - 1) / kWavesPerBlock;
  const uint64_t per_cu = (workgroups + 255) / 256;
  return {per_cu, 4 * workgroups * segments >= 3 * 256 * per_cu * pieces * length};
}

// The form of combine_gather that a step takes, for rows of `elem_bytes` (2 or 4) an element: form(picks, pieces).  A piece is
// 512 elements, 1 KiB of a 16-bit row and 2 KiB of an fp32 one; KiB are those of the rows that are read.
CombineForm combine_form_of(const WorldHost &w, uint32_t elem_bytes) {
  const bool grouped = combine_per_group(w, elem_bytes);
  auto form = [grouped](uint32_t picks, uint32_t pieces) { return CombineForm{picks, pieces, grouped}; };
  const uint32_t nvec_segments = (w.H / 8 + kWave - 1) / kWave;
  const uint64_t tokens = (uint64_t)(grouped ? w.G : w.R) * w.M;
  const uint64_t gathered = tokens * w.K * w.H * elem_bytes;
  const bool whole_pieces = w.H % (8 * kWave) == 0;
  // Steps of a few hundred to two thousand tokens have all their waves resident at the same moment.  More than four picks in rows
  // of seven pieces and more are best taken one after the other in 7 or 8 KiB pieces there, by a quarter as many waves, but
  // only where the workgroups of such pieces come out even over the CUs (long_pieces): the CUs that get one more of them
  // take that much longer.  Dispatch + combine on three buffer sets, top-8, 8 ranks, us, long pieces / three picks in 1
  // KiB: 7168 wide, 1024 tokens 38.4 / 39.0, 544 25.0 / 23.7, 7136 wide, 528 30.2 / 28.4, 7656 wide, 1048 61.8 / 57.6; 4096 wide, 388
  // 19.7 / 15.4, 448 20.4 / 17.0, 680 23.7 / 22.7, 784 24.8 / 25.0, 1024 29.9 / 30.3.  (653 steps of that range drawn
  // at random, against long pieces for all of them: 0.946 of the time, 0.73 to 1.03.)  DP groups, whose waves compare the
  // members first, take two picks in 2 KiB pieces or, beyond a workgroup to a CU, one in 3 KiB instead (5120 wide, 386
  // tokens of all groups 20.2 / 17.9; 3696 wide, 596 23.5 / 21.2), fp32 rows two picks in 2 KiB (4608 wide, top-6, 1256
  // tokens 49.3 / 44.4; 3584 wide, 1152 40.7 / 35.5; their long pieces are 14 and 16 KiB).
  const bool middle = tokens > 384 && tokens <= 2048;
  if (w.K > 4 && middle && nvec_segments >= 7) {
    const LongPieces pieces = long_pieces(tokens, nvec_segments);
    if (pieces.even && (grouped || pieces.per_cu > 1)) {
      if (nvec_segments % 7 == 0) return form(1, 7);
      return form(1, 8);
    }
    if (elem_bytes == 2) {
      if (!grouped) return form(3, 1);
      if (pieces.per_cu == 1) return form(2, 2);
      return form(1, 3);
    }
  }
  // fp32 rows of three pieces (6 KiB) and more.  Two picks at a time beside the above (2048 wide, top-8, 464 tokens
  // 13.0 / 12.8; 1536 wide, 808 16.3 / 15.6; 2560 wide, 1040 29.8 / 28.7, eight / two).  Larger steps take eight at a time, whose
  // registers leave room for fewer waves: against two picks of 8 KiB or three of 4 KiB 6656 wide, top-8, 2095 tokens 130.4 / 126.2,
  // 3588 180.4 / 173.7; 4096 wide, 7168 221.2 / 215.7; top-6, 7680 wide, 5232 279.4 / 271.2; seven pieces and more also with four
  // picks (6144 wide, 2156 tokens 56.0 / 55.3; 4096 wide, 8 x 1024, combine alone 103.2 / 98.1).  DP groups of that size take three
  // (2048 wide, 2136 tokens 43.1 / 40.5), rows of two pieces three of both (eight 1.0 to 1.1 of their time).
  if (elem_bytes == 4) {
    if (w.K > 4 && middle && nvec_segments >= 3) return form(2, 1);
    if (tokens > 2048) {
      if (!grouped && w.K > 3 && nvec_segments >= 7) return form(8, 1);
      if (w.K > 4 && nvec_segments == 2) return form(3, 2);
      if (w.K > 4 && nvec_segments >= 3) {
        if (grouped) return form(3, 1);
        return form(8, 1);
      }
    }
  } else if (grouped && nvec_segments > 1) {
    // Steps of DP groups, 16-bit rows, eight picks / three in pieces of 2 KiB: 5120 wide, top-6, 2888 tokens 86.8 / 84.0;
    // 1024 wide, top-8, 12268 88.1 / 87.1 (541 steps: 0.983, 0.90 to 1.05).  Eight and more are eight at a time again where the
    // rows are more than 1 GiB of whole KiB (combine, eight / three: 6144 wide, top-8, 25012 tokens 611 / 640, 5120 wide, 25104 423 /
    // 445; 4608 wide, top-10, 19340 419 / 439; 28 steps of that size 0.99 of the time, 65 smaller ones 1.01, 31 of rows with a
    // partial KiB 1.02: 3784 wide, top-8, 29830 537 / 491; dispatch + combine 0.98, 1.01 where tokens are absent).  Three and
    // four picks, all at once / two: 1536 wide, top-4, 3260 25.0 / 23.5; 5120 wide, 856 23.5 / 22.9.
    if (w.K > 4 && tokens > 2048 && (w.K < 8 || !whole_pieces || gathered <= 1ull << 30)) return form(3, 2);
    if ((w.K == 3 || w.K == 4) && tokens > 600 && nvec_segments > 2) return form(2, 2);
  }
  // Of what is left, up to five picks are taken all at once, six in two goes of three, nine and ten in two of five, others
  // up to eight at a time.  One or two leave a wave of 1 KiB with little in flight, so they read longer pieces: up to 3
  // KiB of one pick and 2 KiB of two, which is ahead of 8 and of 4 KiB nearly everywhere (dispatch + combine, 8 ranks, us,
  // long / short pieces: one pick of 16-bit rows, 512 tokens, 2048 wide 8.3 / 7.8, 4096 wide 9.2 /
  // 8.8, 8192 wide 12.0 / 11.4; 8192 tokens, 52.3 / 51.0 and 105.9 / 103.6; two picks, 512 tokens, 8.7 / 8.3, 10.0 /
  // 10.0 and 14.1 / 13.9; 8192 tokens, 71.6 / 70.5 and 151.8 / 150.2; not one pick, 1024 tokens, 2560 wide 9.2 / 9.6, 3072
  // 9.6 / 10.1), except
  //  - where the workgroups of the long pieces come out even over the CUs (even_pieces): one pick, 2048 tokens, 3584 wide
  //    15.1 / 15.7, 4096 wide 16.0 / 16.7, 8192 wide 28.9 / 29.5; 4096 tokens of 4096 29.5 / 30.2; 1536 of 7168 19.6 / 20.5 (but
  //    uneven, 4096 wide, 1536 tokens 15.1 / 14.3, 2560 19.8 / 19.8, 3584 25.1 / 24.6);
  //  - for DP groups, whose waves compare the members first.  They keep the long pieces for rows that are longer than half
  //    of one (groups of two, 4 x 512 tokens, one pick, 4096 wide 18.8 / 20.6, 7168 wide 32.1 / 31.4; groups of four, 2 x 512,
  //    15.0 / 15.1 and 22.1 / 24.0; two picks, 25.2 / 25.9 and 44.3 / 44.4, 17.3 / 19.2 and 28.3 / 28.9), one pick also unless
  //    the last piece would be all but empty (4608 wide, nine KiB, 23.3 / 22.4), but not of fp32 rows (combine, 16 / 6 KiB: 6880 wide,
  //    17562 tokens 295 / 265, 6600 wide, 20950 345 / 322; 2560 wide, 1198 10.6 / 9.1; 30 steps 0.96 of the time, 30 of
  //    dispatch + combine 0.97);
  //  - fp32 rows, which have twice the bytes, outside DP groups: 4 KiB of one pick (2 KiB up to 384 tokens, unless the row
  //    has two pieces), 2 KiB of two (one pick, 7168 wide, 208 tokens 9.0 / 8.4, 4096 wide, 2428 20.4 / 19.6; two picks of
  //    8 KiB / 2 KiB, 7680 wide, 4928 91.6 / 89.2).
  // Picks of one go, against eight places of 1 KiB: top-3 (two picks and then one), 8192 tokens, 2048 wide 57.0 / 52.4, 4096
  // wide 99.5 / 90.4; top-5 (four and one), 16000 tokens, 512 wide 43.4 / 41.6, 4096 tokens, 7168 wide 124.6 / 122.5.  Four picks
  // in 2 KiB / 1 KiB: 5120 wide, 88 tokens 8.7 / 8.2, 3584 wide, 2048 25.0 / 24.4, 7680 wide, 1388 43.4 / 42.5 (995 steps: 0.987).
  // Six, four and two / three and three: 2560 wide, 2792 tokens 32.6 / 31.5, 3072 wide, 3914 50.0 / 48.8 (1 KiB to 6 KiB
  // wide, beyond 2048 tokens: 0.975; up to 2048 0.99).  Ten, eight and two / five and five: 512 wide, 1160 14.6 / 14.0, 3584
  // wide, 352 15.5 / 15.2.  Of 16-bit rows neither in large steps of 7 KiB and more (six 0.97 to 1.04, ten 1.012), nor where the
  // rows are more than 512 MiB (combine, six, 2560 wide, 50368 tokens 298 / 312, 2048 wide, 52608 252 / 263; ten, 2048 wide, 50224
  // 364 / 384; 35 steps of that size 0.98 of the time, 69 smaller ones 1.03; dispatch + combine 0.98), but six also there if the
  // last KiB is partial (1048 wide, 46064 tokens 131 / 117, 1544 wide, 38208 151 / 141), nor for DP groups.
  const bool large = gathered > 512ull << 20 && (w.K > 6 || whole_pieces);
  const bool halves = elem_bytes == 4 || (!grouped && (tokens <= 2048 || (nvec_segments < 7 && !large)));
  switch (w.K) {
    case 1:
      if (nvec_segments == 1) return form(1, 1);
      if (nvec_segments == 2) return form(1, 2);
      if (!grouped && elem_bytes == 4) {
        if (tokens <= 384) return form(1, 1);
        return form(1, 2);
      }
      if (nvec_segments == 4) return form(1, 4);
      if (grouped && elem_bytes == 2 && nvec_segments > 4 && 8 * ((8 - nvec_segments % 8) % 8) <= 5 * nvec_segments)
        return form(1, 8);
      if (!grouped && elem_bytes == 2 && even_pieces(tokens, nvec_segments)) return form(1, 8);
      return form(1, 3);
    case 2:
      if (nvec_segments == 1 || (elem_bytes == 4 && (!grouped || tokens <= 384))) return form(2, 1);
      if (grouped && elem_bytes == 2 && nvec_segments > 2) return form(2, 4);
      return form(2, 2);
    case 3: return form(3, 1);
    case 4:
      if (elem_bytes == 2 && nvec_segments > 1 && (grouped || (nvec_segments == 2 && tokens > 600))) return form(4, 2);
      return form(4, 1);
    case 5: return form(5, 1);
    case 6:
      if (halves) return form(3, 1);
      return form(8, 1);
    case 9:
    case 10:
      if (halves) return form(5, 1);
      return form(8, 1);
    default: return form(8, 1);
  }
}

template <typename T, typename U, class CT>
int launch_combine_k(const WorldHost &w, const CT &tab, hipStream_t s) {
  const CombineForm form = combine_form_of(w, sizeof(T));
  switch (form.picks * 16 + form.pieces) {
#define PPLX_COMBINE(KB, VPL) \
  case KB * 16 + VPL: return launch_combine_v<T, U, CT, KB, VPL>(w, tab, form.per_group, s)
    PPLX_COMBINE(1, 1);
    PPLX_COMBINE(1, 2);
    PPLX_COMBINE(1, 3);
    PPLX_COMBINE(1, 4);
    PPLX_COMBINE(1, 7);
    PPLX_COMBINE(1, 8);
    PPLX_COMBINE(2, 1);
    PPLX_COMBINE(2, 2);
    PPLX_COMBINE(2, 4);
    PPLX_COMBINE(3, 1);
    PPLX_COMBINE(3, 2);
    PPLX_COMBINE(4, 1);
    PPLX_COMBINE(4, 2);
    PPLX_COMBINE(5, 1);
    PPLX_COMBINE(8, 1);
#undef PPLX_COMBINE
    default: return (int)hipErrorInvalidValue;
  }
}

template <class CT>
int launch_combine_t(const WorldHost &w, const CT &tab, int in_dtype, int out_dtype, hipStream_t s) {
  // dtype codes follow pplx_a2a_dtype: 0 = f32, 1 = bf16, 2 = f16.
  switch (in_dtype * 4 + out_dtype) {
    case 0 * 4 + 1: return launch_combine_k<float, __bf16>(w, tab, s);
    case 0 * 4 + 2: return launch_combine_k<float, _Float16>(w, tab, s);
    case 1 * 4 + 1: return launch_combine_k<__bf16, __bf16>(w, tab, s);
    case 1 * 4 + 2: return launch_combine_k<__bf16, _Float16>(w, tab, s);
    case 2 * 4 + 1: return launch_combine_k<_Float16, __bf16>(w, tab, s);
    case 2 * 4 + 2: return launch_combine_k<_Float16, _Float16>(w, tab, s);
    default: return (int)hipErrorInvalidValue;
  }
}

}  // namespace

CombineForm combine_form(const WorldHost &w, int in_dtype) { return combine_form_of(w, in_dtype == 0 ? 4 : 2); }
bool combine_stores_plainly(const WorldHost &w) { return plain_stores(w); }

int launch_combine(const WorldHost &w, const CombineRank *inline_rows, int in_dtype, int out_dtype,
                   void *stream) {
  return with_table<InlineCombine>(w, inline_rows, HbmCombine{w.crank}, [&](const auto &tab) {
    return launch_combine_t(w, tab, in_dtype, out_dtype, (hipStream_t)stream);
  });
}

}  // namespace pplx_amd
