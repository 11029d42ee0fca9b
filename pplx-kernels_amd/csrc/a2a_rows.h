// Row fan-out in registers and through LDS, shared by the dispatch kernels, and the macro that picks the register variant
// for a row size.
#pragma once
#include "a2a_common.h"

namespace pplx_amd {
namespace {

// ---------------------------------------------------------------------------
// Row fan-out shared by dispatch_scatter and dispatch_fused.  The calling wave
// owns one token; the row is read once into NV 16-byte registers per lane
// (load_row) and stored for picks [k0, k1) (store_row), lane k passing the slot of
// pick k.  EXACT: the row is exactly NV * 64 vectors, so nothing is predicated.
// ---------------------------------------------------------------------------
template <int NV>
struct RowRegs {
  u32x4 x[NV];   // the row, 16 bytes per lane per register
  float sc;      // scale `lane` of the row (lanes >= S hold a copy of the last one)
};

// Scale `lane` of row t (0 when there are none).
__device__ __forceinline__ float load_scale(const WorldDev &w, const DispatchRank &src, uint32_t t, uint32_t lane) {
  if (w.S == 0) return 0.f;
  const uint32_t j = lane < w.S ? lane : w.S - 1;
  return as_global(src.dp_xs)[(int64_t)t * src.dp_xs_stride_row + (int64_t)j * src.dp_xs_stride_elem];
}

// First half: issues the loads of row t of `src`; needs t < src.m only.
template <int NV, bool EXACT>
__device__ __forceinline__ void load_row(const WorldDev &w, const DispatchRank &src, uint32_t t,
                                         uint32_t lane, RowRegs<NV> &regs) {
  const uint32_t nvec = w.Hb / 16;
  const PPLX_GLOBAL u32x4 *row =
      as_global(reinterpret_cast<const u32x4 *>(src.dp_x + (int64_t)t * src.dp_x_stride_row));
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    uint32_t j = lane + i * kWave;
    if (!EXACT) j = j < nvec ? j : nvec - 1;  // clamp: loads stay unconditional
    regs.x[i] = row[j];
  }
  regs.sc = load_scale(w, src, t, lane);
}

// Where pick (expert e, row `slot`) of a token lands: row address, scale-row address and the
// element stride of the scale row; all zero when the pick has no destination.
struct Destination {
  uint64_t row = 0, scale = 0;
  int64_t scale_step = 0;
};

// The buffers of one expert, out of its owner's row of the rank table.  Fetched whole and without
// conditions, so that it costs one trip to memory which can overlap with whatever finds the slot.
struct ExpertBuffer {
  uint64_t row, scale;
  int64_t row_step, scale_step, scale_elem_step;
  uint32_t rows;
};

template <class DT>
__device__ __forceinline__ ExpertBuffer expert_buffer(const WorldDev &w, const DT &tab, uint32_t e) {
  const uint32_t known = e < w.E ? e : 0;
  const DispatchRank &owner = tab.at(owner_of(w, known));
  const uint32_t el = local_of(w, known);
  ExpertBuffer b;
  b.row = reinterpret_cast<uint64_t>(owner.expert_x + (int64_t)el * owner.x_stride_expert);
  b.row_step = owner.x_stride_row;
  b.scale = reinterpret_cast<uint64_t>(owner.expert_xs + (int64_t)el * owner.xs_stride_expert);
  b.scale_step = owner.xs_stride_row;
  b.scale_elem_step = owner.xs_stride_elem;
  b.rows = owner.x_rows;
  return b;
}

__device__ __forceinline__ Destination destination_of(const WorldDev &w, const ExpertBuffer &b, uint32_t slot,
                                                      bool report) {
  Destination d;
  if (slot != kInvalidSlot) {
    if (slot < b.rows) {
      d.row = b.row + (uint64_t)((int64_t)slot * b.row_step);
      if (w.S) {
        d.scale = b.scale + 4u * (uint64_t)((int64_t)slot * b.scale_step);
        d.scale_step = b.scale_elem_step;
      }
    } else if (report) {
      atomicOr(w.faults, kFaultRowDropped);
    }
  }
  return d;
}

// The scale row of pick k; `scale` is scale `lane` of the token.
template <RowStore POLICY>
__device__ __forceinline__ void store_scales(const WorldDev &w, const DispatchRank &src, uint32_t t, uint32_t lane,
                                             const Destination &dst, uint32_t k, float scale) {
  const uint32_t S = w.S;
  if (S == 0) return;
  PPLX_GLOBAL float *sout = global_ptr<float>(read_lane64(dst.scale, k));
  const int64_t step = (int64_t)read_lane64((uint64_t)dst.scale_step, k);
  if (lane < S) row_store<POLICY>(scale, sout + (int64_t)lane * step);
  if (S > kWave) {
    const PPLX_GLOBAL float *srow = as_global(src.dp_xs) + (int64_t)t * src.dp_xs_stride_row;
    for (uint32_t j = lane + kWave; j < S; j += kWave) {
      sout[(int64_t)j * step] = srow[(int64_t)j * src.dp_xs_stride_elem];
    }
  }
}

// Second half: lane k holds the destination of pick k; the row is stored for picks [k0, k1).
template <int NV, bool EXACT, RowStore POLICY = RowStore::kStream, RowStore SCALE_POLICY = POLICY>
__device__ __forceinline__ void store_row(const WorldDev &w, const DispatchRank &src, uint32_t t,
                                          uint32_t lane, Destination dst, uint32_t k0, uint32_t k1,
                                          RowRegs<NV> &regs) {
  const uint32_t nvec = w.Hb / 16;
#pragma unroll
  for (int i = 0; i < NV; ++i) settle(regs.x[i]);
  settle(regs.sc);
  settle(dst.row);
  settle(dst.scale);
  settle(dst.scale_step);

  for (uint32_t k = k0; k < k1; ++k) {
    const uint64_t p = read_lane64(dst.row, k);
    if (p == 0) continue;
    PPLX_GLOBAL u32x4 *out = global_ptr<u32x4>(p);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const uint32_t j = lane + i * kWave;
      if (EXACT || j < nvec) row_store<POLICY>(regs.x[i], out + j);
    }
    store_scales<SCALE_POLICY>(w, src, t, lane, dst, k, regs.sc);
  }
}

// ---------------------------------------------------------------------------
// Rows through LDS.  They are for rows whose length is no multiple of half a 128-byte line, the unit in which memory
// takes writes.  Every copy of such a row begins somewhere else inside a line, so a wave that stores 64 vectors from the
// row's start at a time cuts a half line in two at each of its stores, and the parts reach the memory as partial
// writes.  Such a row is kept in LDS instead of registers (fetched with loads that write LDS directly), and for every
// pick the lanes take it from there shifted by the copy's offset in its line: all stores but the ends of the row cover
// whole lines.  The lines that two rows share are written through into the last-level cache ("sc1"), where their parts
// meet; the others stream.  Dispatch, us, registers streamed through ("sc1 nt") / registers non-temporal / LDS
// non-temporal / LDS with shared lines written through:
//   5264-byte rows, top-8 of 256, 8 x 2048 tokens  210 / 175 / 160 / 139
//   2976-byte rows, top-8 of 16, 4 x 4903          125 / 116 / 105 / 92
//   8656-byte rows, top-10 of 128, 2 x 1252        74 / 61 / 58 / 54
//   3296-byte rows, top-3 of 16, 25979             79 / 65 / 62 / 59
//   2528-byte rows, top-1 of 64, 2 x 16358         43 / 38 / 39 / 39
// Rows of whole half lines stay in registers.  Dispatch on three buffer sets, top-8, registers / LDS: 192 bytes, 8000 tokens
// 11.4 / 14.4; 320 bytes, top-10, 20000 20.5 / 27.4; 1856 bytes, top-6, 42394 97 / 117; 3264 bytes, 4712 29.9 / 32.0; 8256
// bytes, top-6, 9408 94 / 101; 14400 bytes, 3124 73.6 / 79.5; with half a KiB left over 4608 bytes with scales, 8 x 2048
// 120 / 124; 5760 bytes, top-5, 8 x 3001 71 / 73; 512 bytes 61 / 89.  Which of the
// others take it: scatter_rows_in_lds, and fused_rows_in_lds for the one-launch dispatch, which also holds rows of whole
// half lines there that no register variant fits.
// ---------------------------------------------------------------------------
constexpr uint32_t kLineBytes = 128;
inline bool row_cuts_half_lines(const WorldDev &w) { return w.Hb % (kLineBytes / 2) != 0; }

// Vectors first, first + step, ... (64 each) of row t go to the same place in `lds`, which the calling wave
// may read once its loads have returned (row_staged).
__device__ __forceinline__ void stage_row(const WorldDev &w, const DispatchRank &src, uint32_t t, uint32_t lane,
                                          uint32_t first, uint32_t step, u32x4 *lds) {
  const uint32_t nvec = w.Hb / 16;
  const PPLX_GLOBAL u32x4 *row =
      as_global(reinterpret_cast<const u32x4 *>(src.dp_x + (int64_t)t * src.dp_x_stride_row));
  for (uint32_t j = first * kWave; j < nvec; j += step * kWave) {
    if (j + lane < nvec) {
      __builtin_amdgcn_global_load_lds((const PPLX_GLOBAL void *)(row + j + lane),
                                       (__attribute__((address_space(3))) void *)(lds + j), 16, 0, 0);
    }
  }
}

// All loads of the wave have returned.  (The builtin, which the compiler counts, and not inline asm:
// it would otherwise wait for the stores of one pick before it reads LDS for the next.)
__device__ __forceinline__ void row_staged() {
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  asm volatile("" ::: "memory");
}

// store_row for a row in LDS.
template <RowStore POLICY, RowStore EDGE_POLICY, RowStore SCALE_POLICY>
__device__ __forceinline__ void store_staged_row(const WorldDev &w, const DispatchRank &src, uint32_t t, uint32_t lane,
                                                 Destination dst, uint32_t k0, uint32_t k1, float scale,
                                                 const u32x4 *lds) {
  constexpr uint32_t kLineVecs = kLineBytes / 16;
  const uint32_t nvec = w.Hb / 16;
  settle(scale);
  settle(dst.row);
  settle(dst.scale);
  settle(dst.scale_step);
  for (uint32_t k = k0; k < k1; ++k) {
    const uint64_t p = read_lane64(dst.row, k);
    if (p == 0) continue;
    PPLX_GLOBAL u32x4 *out = global_ptr<u32x4>(p);
    // vector j of the row is vector j + shift of the lines it covers
    const uint32_t shift = (uint32_t)(p / 16) % kLineVecs;
    const uint32_t end = nvec + shift;
    // (64 vectors a trip: two, four and eight times as many with their LDS reads in front measured the same
    // for long rows and up to 25 % more for rows of a few hundred vectors)
    for (uint32_t first = 0; first < end; first += kWave) {
      const uint32_t at = first + lane, j = at - shift;  // (j wraps beyond nvec in front of the row)
      if (j >= nvec) continue;
      const u32x4 x = lds[j];
      if ((shift != 0 && at < kLineVecs) || at / kLineVecs == end / kLineVecs) {
        row_store<EDGE_POLICY>(x, out + j);
      } else {
        row_store<POLICY>(x, out + j);
      }
    }
    store_scales<SCALE_POLICY>(w, src, t, lane, dst, k, scale);
  }
}

}  // namespace
}  // namespace pplx_amd

namespace pplx_amd {
namespace {
// Rows of up to 8 KiB and rows of exactly 10, 12, 14 or 16 KiB (5120-, 6144-, 7168- and 8192-wide
// bf16) have a register variant in every row kernel; other sizes beyond 8 KiB go through LDS (the one-launch
// dispatch; the scatter too where they cut half lines), take the scatter's padded variants or the streaming kernels.
inline bool row_has_register_variant(const WorldDev &w) {
  const uint32_t nvec = w.Hb / 16;
  const uint32_t per_lane = (nvec + kWave - 1) / kWave;
  const bool exact = nvec % kWave == 0;
  return per_lane <= 8 || (exact && (per_lane == 10 || per_lane == 12 || per_lane == 14 || per_lane == 16));
}
}  // namespace
}  // namespace pplx_amd

// Picks the register variant for the row size, launches KERNEL<NV, EXACT, DT> and returns what launch_kernel says.
// Rows beyond 8 KiB exist only for dispatch_scatter (PPLX_LAUNCH_LARGE_ROW_VARIANT).
#define PPLX_LAUNCH_ROW_VARIANT(KERNEL, NV, EXACT)                                               \
  return launch_kernel(KERNEL<NV, EXACT, DT>, grid, block, lds, s, w, tab, PPLX_ROW_KERNEL_ARGS)

#define PPLX_DISPATCH_ROW_VARIANTS(KERNEL)                                                       \
  do {                                                                                           \
    const uint32_t nvec = w.Hb / 16;                                                             \
    const uint32_t per_lane = (nvec + kWave - 1) / kWave;                                        \
    const bool exact = nvec % kWave == 0;                                                        \
    if (exact && per_lane == 1) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 1, true);                        \
    else if (exact && per_lane == 2) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 2, true);                   \
    else if (exact && per_lane == 3) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 3, true);                   \
    else if (exact && per_lane == 4) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 4, true);                   \
    else if (exact && per_lane == 5) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 5, true);                   \
    else if (exact && per_lane == 6) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 6, true);                   \
    else if (exact && per_lane == 7) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 7, true);                   \
    else if (exact && per_lane == 8) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 8, true);                   \
    else if (exact && per_lane == 10) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 10, true);                 \
    else if (exact && per_lane == 12) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 12, true);                 \
    else if (exact && per_lane == 14) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 14, true);                 \
    else if (exact && per_lane == 16) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 16, true);                 \
    else if (per_lane <= 1) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 1, false);                           \
    else if (per_lane <= 2) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 2, false);                           \
    else if (per_lane <= 4) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 4, false);                           \
    else if (per_lane <= 8) PPLX_LAUNCH_ROW_VARIANT(KERNEL, 8, false);                           \
    else PPLX_LAUNCH_LARGE_ROW_VARIANT(KERNEL);                                                  \
  } while (0)
