// The last levels of a contraction in one workgroup: once a level has at most
// kTailVertices vertices and kTailSlots edge slots, its remaining levels, the
// base case and the way back up to this level run in two launches and without
// a word to the host, where the general path takes about 30 launches and four
// synchronisations for each level, most of them far too short to fill the
// chip (a level of 2283 vertices and 51 K slots: about 0.3 ms).
//
// Keys are packed (distance << 15 | label) in LDS; the edges, each undirected
// one once as a pair of 16-bit indices, stay in a global buffer that one CU
// streams from its L2 (64 bytes a clock).  What bounds it: the LDS accesses of
// the key passes and, on few vertices, the barriers between the phases.
//
// Same decisions as the general path: deviates, fixed point (or the local
// variant's two synchronous passes), stall rule, next level in label order,
// cut-off on the exact number of distinct edges.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "deviates.h"
#include "kc_common.h"
#include "kernels.h"
#include "slot_rows.h"

namespace kc {

namespace {

constexpr int kTailBlock = 1024;
constexpr uint32_t kLabelBits = 15, kLabelMask = (1u << kLabelBits) - 1, kHop = 1u << kLabelBits;
static_assert(kTailVertices <= kHop && kTailMaxDeviate + 2 < 1u << (32 - kLabelBits), "key packing");
constexpr uint32_t kTable = 1u << kLabelBits;  // hash slots over the LDS of the keys (and their copy)
constexpr uint32_t kTableLoad = 20000;     // edges of one hash part (load 0.61)
constexpr uint32_t kNoIndex = 0xFFFF;

__device__ __forceinline__ uint32_t first_key(const TailArgs &a, uint32_t v, uint32_t id, uint32_t iteration) {
  const uint32_t dev = a.local ? uniform_deviate_100(id, a.d.seed, iteration)
                               : exp_deviate(id, a.d.seed, iteration, a.d.rng_offset, a.d.fused != 0, a.d.stream,
                                             a.d.table, a.d.k_max);
  return (dev << kLabelBits) | v;
}

// What the whole chip does for the one workgroup: the first level's ids and
// keys, and its edges, each once (from its larger end's row) as
// (row | target << 16) in no particular order; *count (zeroed) = their number.
__global__ __launch_bounds__(kBlock) void k_tail_edges(TailArgs a, uint64_t m2, const uint64_t *off,
                                                      const uint32_t *col) {
  const uint32_t n = a.n;
  uint32_t *edge = a.edge, *count = a.count;
  for (uint32_t v = blockIdx.x * kBlock + threadIdx.x; v < n; v += gridDim.x * kBlock) {
    const uint32_t id = a.gid_in ? a.gid_in[v] : v;
    a.cur[v] = v;
    a.gid[v] = id;
    a.key0[v] = first_key(a, v, id, a.iteration);
  }
  __shared__ uint32_t row_lds[kBlock / kWave][kWaveSlots];
  const uint64_t c0 = (blockIdx.x * static_cast<uint64_t>(kBlock / kWave) + threadIdx.x / kWave) * kWaveSlots;
  if (c0 >= m2) return;
  const uint64_t c1 = c0 + kWaveSlots < m2 ? c0 + kWaveSlots : m2;
  uint32_t x[kLaneSlots], kept = 0;
#pragma unroll
  for (uint32_t j = 0; j < kLaneSlots; ++j) x[j] = kNone;
  for_wave_slots(n, off, col, c0, c1, row_lds[threadIdx.x / kWave], [&](uint32_t j, uint32_t v, uint32_t w) {
    if (w < v) {
      x[j] = v | (w << 16);
      ++kept;
    }
  });
  uint32_t inc = kept;
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t t = static_cast<uint32_t>(__shfl_up(static_cast<int>(inc), o));
    if (lane_id() >= static_cast<uint32_t>(o)) inc += t;
  }
  uint32_t at = 0;
  if (lane_id() == kWave - 1 && inc) at = atomicAdd(count, inc);
  at = static_cast<uint32_t>(__shfl(static_cast<int>(at), kWave - 1)) + inc - kept;
#pragma unroll
  for (uint32_t j = 0; j < kLaneSlots; ++j)
    if (x[j] != kNone) edge[at++] = x[j];
}

// Exclusive scan over the workgroup; total = the sum.
__device__ __forceinline__ uint32_t tail_scan(uint32_t x, uint32_t *wave, uint32_t &total) {
  const uint32_t ln = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t inc = x;
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t t = static_cast<uint32_t>(__shfl_up(static_cast<int>(inc), o));
    if (ln >= static_cast<uint32_t>(o)) inc += t;
  }
  if (ln == 63) wave[w] = inc;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
  for (uint32_t i = 0; i < kTailBlock / kWave; ++i) {
    const uint32_t t = wave[i];
    before += i < w ? t : 0u;
    total += t;
  }
  __syncthreads();  // wave is free again
  return before + inc - x;
}

__device__ __forceinline__ uint32_t edge_hash(uint32_t x) {
  x ^= x >> 15;
  x *= 0x2c1b3c6du;
  x ^= x >> 12;
  x *= 0x297a2d39u;
  return x ^ (x >> 15);
}

// Edges 4i .. 4i + 3 (the buffer ends in zeros, an edge (0, 0) changes nothing).
__device__ __forceinline__ uint4 load4(const uint32_t *edge, uint32_t i, uint32_t n4) {
  return i < n4 ? reinterpret_cast<const uint4 *>(edge)[i] : make_uint4(0u, 0u, 0u, 0u);
}

// The next level's index of a label is its rank among the marked ones: a bit
// and a count per 32 labels in LDS, where an index per label had to be written
// for all of them, above kTailSmall vertices to global memory: 32 008 vertices 300
// -> 232 us, 26 157 with 16 levels that hardly contract 4.5 -> 3.4 ms.
__global__ __launch_bounds__(kTailBlock) void k_tail(TailArgs a) {
  static_assert(kTailVertices == 32 * kTailBlock, "a thread per word of marks");
  __shared__ __align__(16) uint32_t lds[kTable];  // the keys, up to kTailSmall of them with a copy; all of it the edge table
  __shared__ uint2 rank[kTailBlock];              // 32 labels: those of clusters with an edge, and their number before
  __shared__ uint32_t wave[kTailBlock / kWave];
  __shared__ uint32_t s_radius, s_full;
  uint32_t *key = lds, *key2 = lds + kTable / 2;
  const auto set_mark = [&](uint32_t l) {
    if (!(rank[l >> 5].x >> (l & 31) & 1u)) atomicOr(&rank[l >> 5].x, 1u << (l & 31));
  };
  const auto index_of = [&](uint32_t l) -> uint32_t {
    const uint2 w = rank[l >> 5];
    const uint32_t bit = 1u << (l & 31);
    return w.x & bit ? w.y + static_cast<uint32_t>(__popc(w.x & (bit - 1))) : kNoIndex;
  };
  const auto marked_index = [&](uint32_t l) -> uint32_t {  // of a marked label
    const uint2 w = rank[l >> 5];
    return w.y + static_cast<uint32_t>(__popc(w.x & ((1u << (l & 31)) - 1)));
  };
  const auto clear_table = [&] {
    for (uint32_t j = threadIdx.x; j < kTable / 4; j += kTailBlock)
      reinterpret_cast<uint4 *>(lds)[j] = make_uint4(kNone, kNone, kNone, kNone);
  };
  const uint32_t tid = threadIdx.x;
  const uint32_t n0 = a.n;
  uint32_t nl = n0, ne = *a.count;
  uint64_t m = a.m;  // distinct undirected edges of the level
  uint32_t iteration = a.iteration, levels = 0, sweeps = 0, radius_sum = 0, status = kTailDone;
  if (tid == 0) s_full = 0;
  // the level's ids, and the next level's (the first keys are read before it is written)
  uint32_t *gid = a.gid, *gid_next = a.key0;
  if (tid < 3) a.edge[ne + tid] = 0;
  __syncthreads();
  while (true) {
    const bool base = a.seq_limit > 0 && m <= a.seq_limit;
    if (!base && levels >= a.max_levels) {
      status = kTailLevels;
      break;
    }
    if (tid == 0) s_radius = 0;
    const uint32_t n4 = (ne + 3) / 4;
    uint4 *edge4 = reinterpret_cast<uint4 *>(a.edge);
    for (uint32_t v = tid; v < nl; v += kTailBlock)
      key[v] = base ? v : iteration == a.iteration ? a.key0[v] : first_key(a, v, gid[v], iteration);
    __syncthreads();
    bool first_change = true;
    if (base || !a.local) {
      // passes over the edges until no key changes (base case: labels alone
      // flow, each pass followed by a pointer jump)
      const uint32_t hop = base ? 0u : kHop;
      for (uint32_t pass = 0;; ++pass) {
        bool changed = false;
        // eight edges in two 16-byte loads per step, the next step's loads in
        // flight meanwhile
        uint4 c0 = load4(a.edge, tid, n4), c1 = load4(a.edge, tid + kTailBlock, n4);
        for (uint32_t i = tid; i < n4; i += 2 * kTailBlock) {
          const uint32_t e[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
          c0 = load4(a.edge, i + 2 * kTailBlock, n4);
          c1 = load4(a.edge, i + 3 * kTailBlock, n4);
          uint32_t ku[8], kw[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            ku[j] = key[e[j] & 0xFFFFu];
            kw[j] = key[e[j] >> 16];
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (ku[j] + hop < kw[j]) {
              atomicMin(&key[e[j] >> 16], ku[j] + hop);
              changed = true;
            } else if (kw[j] + hop < ku[j]) {
              atomicMin(&key[e[j] & 0xFFFFu], kw[j] + hop);
              changed = true;
            }
          }
        }
        if (base) {
          __syncthreads();
          for (uint32_t v = tid; v < nl; v += kTailBlock) {
            const uint32_t k = key[v], k2 = key[k];
            if (k2 < k) {
              key[v] = k2;  // (a key only falls; a neighbour's jump read early costs a pass)
              changed = true;
            }
          }
        }
        ++sweeps;
        const bool any = __syncthreads_or(changed) != 0;
        if (pass == 0) first_change = any;
        if (!any) break;
      }
    } else {
      // two synchronous passes over the closed neighbourhood, hop 0
      for (int pass = 0; pass < 2; ++pass) {
        uint32_t *in = pass ? key2 : key, *out = pass ? key : key2;
        for (uint32_t v = tid; v < nl; v += kTailBlock) out[v] = in[v];
        __syncthreads();
        for (uint32_t i = tid; i < n4; i += kTailBlock) {
          const uint4 c = edge4[i];
          const uint32_t e[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t u = e[j] & 0xFFFFu, w = e[j] >> 16, ku = in[u], kw = in[w];
            if (ku < kw)
              atomicMin(&out[w], ku);
            else if (kw < ku)
              atomicMin(&out[u], kw);
          }
        }
        __syncthreads();
      }
      sweeps += 2;
    }
    if (base) {
      for (uint32_t v = tid; v < n0; v += kTailBlock) {
        const uint32_t c = a.cur[v];
        if (c != kNone) a.rep[v] = gid[key[c]];
      }
      break;
    }
    ++levels;
    if (a.stall_rule && !first_change) {
      // every vertex is its own centre and keeps an edge: the contraction is
      // the identity; the next iteration draws again on the same graph
      ++iteration;
      continue;
    }
    uint32_t r = 0;
    for (uint32_t v = tid; v < nl; v += kTailBlock) {
      const uint32_t k = key[v];
      const uint32_t h = a.local ? 0u : (k >> kLabelBits) - (key[k & kLabelMask] >> kLabelBits);
      r = h > r ? h : r;
    }
    rank[tid].x = 0;
    for (int o = 32; o > 0; o >>= 1) {
      const uint32_t t = static_cast<uint32_t>(__shfl_xor(static_cast<int>(r), o));
      r = t > r ? t : r;
    }
    if ((tid & 63) == 0 && r) atomicMax(&s_radius, r);
    __syncthreads();
    radius_sum += s_radius;
    // the edges between clusters as label pairs, smaller label first; their clusters marked
    for (uint32_t i0 = tid; i0 < n4; i0 += 2 * kTailBlock) {
      const uint4 c0 = load4(a.edge, i0, n4), c1 = load4(a.edge, i0 + kTailBlock, n4);
      uint32_t e[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {  // (the zeros past the end become kNone too)
        const uint32_t x = key[e[j] & 0xFFFFu] & kLabelMask, y = key[e[j] >> 16] & kLabelMask;
        if (x != y) {
          set_mark(x);
          set_mark(y);
        }
        e[j] = x == y ? kNone : x < y ? x | (y << 16) : y | (x << 16);
      }
      edge4[i0] = make_uint4(e[0], e[1], e[2], e[3]);
      if (i0 + kTailBlock < n4) edge4[i0 + kTailBlock] = make_uint4(e[4], e[5], e[6], e[7]);
    }
    __syncthreads();
    // next-level indices in label order
    uint32_t n_next = 0;
    rank[tid].y = tail_scan(static_cast<uint32_t>(__popc(rank[tid].x)), wave, n_next);
    __syncthreads();
#pragma unroll 4
    for (uint32_t v = tid; v < nl; v += kTailBlock) {
      const uint32_t x = index_of(v);
      if (x != kNoIndex) gid_next[x] = gid[v];
    }
    for (uint32_t v = tid; v < n0; v += kTailBlock) {
      const uint32_t c = a.cur[v];
      if (c == kNone) continue;
      const uint32_t l = key[c] & kLabelMask;
      const uint32_t x = index_of(l);
      if (x != kNoIndex) {
        a.cur[v] = x;
      } else {
        a.cur[v] = kNone;
        a.rep[v] = gid[l];
      }
    }
    __syncthreads();
    if (n_next == 0) break;
    // The pairs renumbered and moved to the front, repeats dropped where the
    // filter meets them: of equal edges the first to reach their slot is kept
    // (a repeat that stays changes no key).
    clear_table();
    __syncthreads();
    uint32_t out = 0;
    const uint4 none = make_uint4(kNone, kNone, kNone, kNone);
    uint4 c0 = tid < n4 ? edge4[tid] : none, c1 = kTailBlock + tid < n4 ? edge4[kTailBlock + tid] : none;
    for (uint32_t b = 0; b < n4; b += 2 * kTailBlock) {
      uint32_t x[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w}, kept = 0;
      const uint32_t ahead = b + 2 * kTailBlock + tid;
      c0 = ahead < n4 ? edge4[ahead] : none;
      c1 = ahead + kTailBlock < n4 ? edge4[ahead + kTailBlock] : none;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (x[j] != kNone) x[j] = marked_index(x[j] & 0xFFFFu) | (marked_index(x[j] >> 16) << 16);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (x[j] != kNone && atomicExch(&lds[edge_hash(x[j]) & (kTable - 1)], x[j]) == x[j]) x[j] = kNone;
      // places by wave, then by edge: the lanes of one store write consecutive words
#pragma unroll
      for (int j = 0; j < 8; ++j) kept += static_cast<uint32_t>(__popcll(__ballot(x[j] != kNone)));
      if ((tid & 63) == 0) wave[tid >> 6] = kept;
      __syncthreads();  // this step's edges are in registers, the next step's too
      uint32_t at = out;
      for (uint32_t w = 0; w < kTailBlock / kWave; ++w) {
        at += w < tid >> 6 ? wave[w] : 0u;
        out += wave[w];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint64_t m64 = __ballot(x[j] != kNone);
        if (x[j] != kNone) a.edge[at + static_cast<uint32_t>(__popcll(m64 & lanes_below()))] = x[j];
        at += static_cast<uint32_t>(__popcll(m64));
      }
      __syncthreads();  // wave is free again
    }
    ne = out;
    m = ne;
    if (a.seq_limit > 0 && ne > a.seq_limit) {
      // The cut-off compares the distinct edges: they are counted by hash
      // parts, each in a table of its own, until there are more than the
      // bound; where a table of one part holds the bound and the steps between
      // two looks at the count, one part does whatever their number.
      constexpr uint32_t step_edges = 4 * kTailBlock, look_steps = 2;
      static_assert(kTailCountOnce + look_steps * step_edges == kTableLoad, "cut-offs of one part");
      const uint32_t parts = a.seq_limit <= kTailCountOnce ? 1 : (ne + kTableLoad - 1) / kTableLoad;
      uint64_t distinct = 0;
      for (uint32_t part = 0; part < parts && distinct <= a.seq_limit; ++part) {
        clear_table();
        __syncthreads();
        uint32_t added = 0, steps = 0, total = 0;
        for (uint32_t b = 0; b < ne && distinct <= a.seq_limit; b += step_edges) {
          uint32_t e[4], slot[4], jump[4], open = 0;  // bit j of open: edge j still probing
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t i = b + j * kTailBlock + tid;
            e[j] = i < ne ? a.edge[i] : kNone;
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t h = edge_hash(e[j]);
            // (the part takes the hash's high bits, the slot its low ones, the step between slots both)
            slot[j] = h & (kTable - 1);
            jump[j] = (h >> 12) | 1u;
            const bool mine = parts == 1 || static_cast<uint32_t>((static_cast<uint64_t>(h) * parts) >> 32) == part;
            open |= (e[j] != kNone && mine ? 1u : 0u) << j;
          }
          // the four edges probe together, so their LDS round trips overlap
          for (uint32_t probe = 0; open; ++probe) {
            uint32_t seen[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) seen[j] = open >> j & 1u ? lds[slot[j]] : 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if ((open >> j & 1u) && seen[j] == kNone) {
                seen[j] = atomicCAS(&lds[slot[j]], kNone, e[j]);
                if (seen[j] == kNone) {  // claimed
                  open &= ~(1u << j);
                  ++added;
                }
              }
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (open >> j & 1u) {
                if (seen[j] == e[j]) open &= ~(1u << j);
                slot[j] = (slot[j] + jump[j]) & (kTable - 1);
              }
            if (probe >= kTable) {  // the part's table is full: its hash took more than kTable of the edges
              s_full = 1;
              break;
            }
          }
          if (parts == 1 && ++steps % look_steps == 0) {
            tail_scan(added, wave, total);
            distinct += total;
            added = 0;
          }
        }
        tail_scan(added, wave, total);
        distinct += total;
      }
      if (s_full) {
        status = kTailFull;
        break;
      }
      m = distinct;  // exact up to the bound
    }
    if (tid < 3) a.edge[ne + tid] = 0;  // (within the old list's padding)
    __syncthreads();
    nl = n_next;
    uint32_t *swap = gid;
    gid = gid_next;
    gid_next = swap;
    ++iteration;
  }
  if (tid == 0) {
    a.info[0] = status;
    a.info[1] = levels;
    a.info[2] = sweeps;
    a.info[3] = radius_sum;
  }
}

}  // namespace

void tail_levels(const TailArgs &a, uint64_t m2, const uint64_t *off, const uint32_t *col, hipStream_t s) {
  const uint64_t g = std::max(ceil_div(m2, static_cast<uint64_t>(kWaveSlots) * (kBlock / kWave)),
                              ceil_div(a.n, static_cast<uint64_t>(kBlock)));
  hipLaunchKernelGGL(k_tail_edges, dim3(static_cast<unsigned>(g)), dim3(kBlock), 0, s, a, m2, off, col);
  KC_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_tail, dim3(1), dim3(kTailBlock), 0, s, a);
  KC_LAUNCH_CHECK();
}

}  // namespace kc
