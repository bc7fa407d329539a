// Rows of CSR slots by fixed shares: a wave takes kWaveSlots consecutive edge
// slots whatever the rows' lengths, so no degree bins are needed.
#pragma once

#include "kc_common.h"

namespace kc {

constexpr int kWaveSlots = 512;
constexpr uint32_t kLaneSlots = kWaveSlots / kWave;

// The last row r with off[r] <= e (off[0] <= e < off[n]), 64 probes a step.
__device__ __forceinline__ uint64_t row_of_slot(const uint64_t *off, uint64_t n, uint64_t e) {
  uint64_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint64_t step = (hi - lo + kWave - 1) / kWave;
    const uint64_t p = lo + (lane_id() + 1) * step;
    const uint64_t below = __popcll(__ballot(p < hi && off[p] <= e));
    lo += below * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo;
}

// Calls f(j, row, target) for the wave's slots [c0, c1): lane l's j-th slot is
// c0 + j * kWave + l, j < kLaneSlots (slots past c1 give no call).  The wave
// searches its first and last row, marks the rows' first slots in LDS (row:
// kWaveSlots words of the wave's own) and spreads the marks by a running
// maximum; where the range spans many empty rows, each lane searches its
// slot's row instead.
template <class F>
__device__ __forceinline__ void for_wave_slots(uint64_t n, const uint64_t *off, const uint32_t *col, uint64_t c0,
                                               uint64_t c1, uint32_t *row, F f) {
  const uint32_t ln = lane_id();
  const uint64_t r0 = row_of_slot(off, n, c0), r1 = row_of_slot(off, n, c1 - 1);
  const bool marked = r1 - r0 <= 4 * kWaveSlots;
  if (marked) {
    for (uint32_t j = ln; j < kWaveSlots; j += kWave) row[j] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (uint64_t r = r0 + 1 + ln; r <= r1; r += kWave) {  // non-empty rows start at distinct slots
      const uint64_t s = off[r];
      if (off[r + 1] > s) row[s - c0] = static_cast<uint32_t>(r - r0);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t m[kLaneSlots], run = 0;
#pragma unroll
    for (uint32_t j = 0; j < kLaneSlots; ++j) {
      const uint32_t x = row[ln * kLaneSlots + j];
      run = x > run ? x : run;
      m[j] = run;
    }
    uint32_t inc = run;
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t t = static_cast<uint32_t>(__shfl_up(static_cast<int>(inc), o));
      if (ln >= static_cast<uint32_t>(o) && t > inc) inc = t;
    }
    uint32_t before = static_cast<uint32_t>(__shfl_up(static_cast<int>(inc), 1));
    if (ln == 0) before = 0;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (uint32_t j = 0; j < kLaneSlots; ++j) row[ln * kLaneSlots + j] = m[j] > before ? m[j] : before;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  uint32_t w[kLaneSlots];
#pragma unroll
  for (uint32_t j = 0; j < kLaneSlots; ++j) {
    const uint64_t e = c0 + j * kWave + ln;
    w[j] = e < c1 ? col[e] : kNone;
  }
#pragma unroll
  for (uint32_t j = 0; j < kLaneSlots; ++j) {
    const uint64_t e = c0 + j * kWave + ln;
    if (e >= c1) continue;
    uint64_t u;
    if (marked) {
      u = r0 + row[j * kWave + ln];
    } else {
      uint64_t lo = r0, hi = r1 + 1;
      while (hi - lo > 1) {
        const uint64_t mid = lo + (hi - lo) / 2;
        if (off[mid] <= e)
          lo = mid;
        else
          hi = mid;
      }
      u = lo;
    }
    f(j, static_cast<uint32_t>(u), w[j]);
  }
}

}  // namespace kc
