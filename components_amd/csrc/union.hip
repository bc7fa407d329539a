// Connected components by lock-free union-find: the base case of the
// contraction (RunSequentialCC, lib/components/exponential_contraction.h:
// 908-922), the shortcuts variant and the components inside the blocks of the
// pre-contraction.
//
// parent[v] <= v always, so the forest has no cycles, and a root is its own parent.
// The last pass over the edges (link) hooks roots alone, each under a smaller root
// by compare-and-swap as in Anderson and Woll 1991, so that a finished tree's
// root is its component's smallest index.  Any parent value ever read in that
// pass stays an ancestor, so loads may be stale (the chiplets' L2s are
// not coherent within a launch): a hook with a stale root fails and returns
// the current parent, from which the search goes on downward.  The passes
// ahead of it only have to keep parents within the component and below their
// children: they start every vertex at a neighbour, as in the connected-components
// code ECL-CC (Jaiganesh and Burtscher 2018), and replace the links of
// vertices that may be no roots any more (hook); the last pass links every edge again.
//
// A few passes over the edges replace min-label sweeps with a pointer jump
// after each, whose number grows with the diameter (2D grid 1500 x 1100, p =
// 0.6: 62 sweeps and jumps, 2.0 ms; now 0.21 ms).  What bounds it: the random
// parent reads and one device atomic per successful hook.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kc_common.h"
#include "kernels.h"
#include "slot_rows.h"

namespace kc {

namespace {

constexpr uint32_t kFirstNeighbours = 4;
constexpr int kShortenHops = 32;
constexpr uint64_t kShortenTwiceMin = 1u << 16;
constexpr uint32_t kUnionCountBlocks = 2048;

// Indices [lo, hi) whose edges count for v: its block of consecutive indices,
// or everything.
__device__ __forceinline__ bool same_block(uint32_t u, uint32_t v, uint64_t block) {
  return block == 0 || u / block == v / block;
}

// parent[v] = the smallest of v and its first few neighbours: no cycle (every
// parent is at most its child) and no atomic, and it leaves far fewer trees.
__global__ __launch_bounds__(kBlock) void k_union_init(uint64_t n, const uint64_t *off, const uint32_t *col,
                                                      uint64_t block, uint32_t *parent) {
  const uint64_t v = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x;
  if (v >= n) return;
  const uint32_t self = static_cast<uint32_t>(v);
  const uint64_t e0 = off[v], len = off[v + 1] - e0;
  uint32_t p = self;
  uint32_t c[kFirstNeighbours];
#pragma unroll
  for (uint32_t j = 0; j < kFirstNeighbours; ++j) c[j] = j < len ? col[e0 + j] : self;
#pragma unroll
  for (uint32_t j = 0; j < kFirstNeighbours; ++j)
    if (c[j] < p && same_block(c[j], self, block)) p = c[j];
  parent[v] = p;
}

// Every vertex jumps up to kShortenHops ancestors: a chain of d edges shrinks
// to about d / kShortenHops, or less where other vertices' jumps are seen.
__global__ __launch_bounds__(kBlock) void k_union_shorten(uint64_t n, uint32_t *parent) {
  const uint64_t v = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x;
  if (v >= n) return;
  const uint32_t first = parent[v];
  uint32_t p = first;
  for (int h = 0; h < kShortenHops; ++h) {
    const uint32_t q = parent[p];
    if (q == p) break;
    p = q;
  }
  if (p != first) parent[v] = p;
}

// Root of v, by path splitting (Tarjan and van Leeuwen 1984): every vertex on the
// way gets its parent's parent for its own.  The store needs no atomic: it goes to
// a vertex that has been hooked already, so no compare-and-swap on it can succeed
// any more, and leaves it an ancestor.  (Path halving, a store every other
// vertex: a path of 10 000 in index order 180 -> 130 us, G(1000, 2000) 34 -> 37,
// G(10 000, 10 000) 60 -> 64.)
__device__ __forceinline__ uint32_t find_root(uint32_t *parent, uint32_t v) {
  uint32_t p = parent[v];
  if (p == v) return v;
  for (uint32_t above = parent[p]; above != p; above = parent[p]) {
    parent[v] = above;
    v = p;
    p = above;
  }
  return p;
}

// Joins the trees of u and w.  A large tree whose root hi was hooked a moment
// ago still looks a root to the other chiplets, and each of its edges to another
// tree would send its own compare-and-swap there, 4 ns apart: 1 ms where two large
// trees were left (the base case of a contracted R-MAT 25, some seeds, of 70 us).  So
// where many of a wave's lanes share the first one's hi, that lane's swap serves them.
constexpr int kCrowd = 8;
__device__ __forceinline__ void link(uint32_t *parent, uint32_t u, uint32_t w) {
  uint32_t a = find_root(parent, u), b = find_root(parent, w);
  while (a != b) {
    const uint32_t hi = a > b ? a : b, lo = a > b ? b : a;
    const bool like_first = hi == static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(hi)));
    const uint64_t crowd = __ballot(like_first);
    const bool served = like_first && __popcll(crowd) >= kCrowd;
    const uint32_t first_lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(lo)));
    const uint32_t under = served ? first_lo : lo;
    uint32_t old = 0;
    if (!served || lane_id() == static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(crowd)) - 1))
      old = atomicCAS(&parent[hi], hi, under);
    const uint32_t firsts = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(old)));
    if (served) old = firsts;
    a = old == hi ? under : find_root(parent, old);  // hi is hooked now, by this swap or another: under < hi
    b = lo;
  }
}

// Hooks the larger of two ends' parents, a and b, under the smaller one without a
// search: trees that are stars (or nearly) merge in one step each.  Where the
// larger is no root any more its link is replaced; every edge is linked again
// by the last pass, so nothing is lost.
__device__ __forceinline__ void hook(uint32_t *parent, uint32_t a, uint32_t b) {
  if (a == b) return;
  const uint32_t hi = a > b ? a : b, lo = a > b ? b : a;
  if (parent[hi] > lo) atomicMin(&parent[hi], lo);
}

// Hooks along four edges of every row, other ones in either round (a shorter row:
// all).
__global__ __launch_bounds__(kBlock) void k_union_hook_rows(uint64_t n, const uint64_t *off, const uint32_t *col,
                                                           uint64_t block, uint32_t *parent, uint32_t round) {
  constexpr uint64_t kSamples = 4;
  const uint64_t v = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x;
  if (v >= n) return;
  const uint32_t self = static_cast<uint32_t>(v);
  const uint64_t e0 = off[v], len = off[v + 1] - e0;
  uint32_t c[kSamples], p[kSamples];
#pragma unroll
  for (uint64_t j = 0; j < kSamples; ++j) {
    const uint64_t i = len <= kSamples ? j : len * (2 * j + 1 + round) / (2 * kSamples + 2);
    c[j] = i < len ? col[e0 + i] : self;
  }
  const uint32_t own = parent[v];
#pragma unroll
  for (uint64_t j = 0; j < kSamples; ++j) p[j] = same_block(c[j], self, block) ? parent[c[j]] : own;
#pragma unroll
  for (uint64_t j = 0; j < kSamples; ++j) hook(parent, own, p[j]);
}

// Links (or, with kHook, hooks) the two ends of every edge, from its larger
// end's row; with every > 1, of the edges in each every-th share of a wave's slots,
// from share `first` on.
template <bool kHook>
__global__ __launch_bounds__(kBlock) void k_union_link(uint64_t n, uint64_t m2, const uint64_t *off,
                                                      const uint32_t *col, uint64_t block, uint32_t *parent,
                                                      uint32_t every, uint32_t first) {
  __shared__ uint32_t row_lds[kBlock / kWave][kWaveSlots];
  const uint64_t share = blockIdx.x * static_cast<uint64_t>(kBlock / kWave) + threadIdx.x / kWave;
  const uint64_t c0 = (share * every + first) * kWaveSlots;
  if (c0 >= m2) return;
  const uint64_t c1 = c0 + kWaveSlots < m2 ? c0 + kWaveSlots : m2;
  for_wave_slots(n, off, col, c0, c1, row_lds[threadIdx.x / kWave], [&](uint32_t, uint32_t v, uint32_t w) {
    if (w < v && same_block(w, v, block)) {
      if (kHook)
        hook(parent, parent[v], parent[w]);
      else
        link(parent, v, w);
    }
  });
}

__device__ __forceinline__ uint32_t root_of(const uint32_t *parent, uint64_t v) {
  uint32_t p = parent[v], q;
  while ((q = parent[p]) != p) p = q;
  return p;
}

__global__ __launch_bounds__(kBlock) void k_union_reps(uint64_t n, const uint32_t *parent, const uint32_t *gid,
                                                      uint32_t *rep) {
  const uint64_t v = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x;
  if (v >= n) return;
  const uint32_t r = root_of(parent, v);
  rep[v] = gid ? gid[r] : r;
}

__global__ __launch_bounds__(kBlock) void k_union_keys(uint64_t n, const uint32_t *parent, uint64_t *key) {
  const uint64_t v = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x;
  if (v < n) key[v] = root_of(parent, v);
}

__global__ __launch_bounds__(kBlock) void k_union_labels(uint64_t n, const uint32_t *parent, uint32_t *labels,
                                                        uint32_t *partial) {
  __shared__ uint32_t wc[kBlock / kWave];
  uint32_t roots = 0;
  for (uint64_t v = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x; v < n;
       v += static_cast<uint64_t>(gridDim.x) * kBlock) {
    const uint32_t r = root_of(parent, v);
    labels[v] = r;
    roots += r == static_cast<uint32_t>(v);
  }
  roots = group_sum_u32(roots, kWave);
  if (lane_id() == 0) wc[threadIdx.x / kWave] = roots;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = wc[0] + wc[1] + wc[2] + wc[3];
}

unsigned blocks_for(uint64_t n) { return static_cast<unsigned>(ceil_div(n, static_cast<uint64_t>(kBlock))); }

void shorten(uint64_t n, uint32_t *parent, hipStream_t s, bool again = true) {
  // (a path of 2^20 vertices in index order is the worst case: two passes
  // before the links and two after leave about a thousand hops to the search)
  for (int pass = 0; pass < (again && n >= kShortenTwiceMin ? 2 : 1); ++pass) {
    hipLaunchKernelGGL(k_union_shorten, dim3(blocks_for(n)), dim3(kBlock), 0, s, n, parent);
    KC_LAUNCH_CHECK();
  }
}

// Rounds of hooks before the links: along four edges of every row (rows), or
// along the edges of each every-th share (shares).  The links of many
// neighbouring trees wait for one another along chains of roots, so the hooks
// have to leave few trees; and a round costs its launches, which counts on small
// graphs.  Shortcuts calls on the device in us:
//   below 2^14 vertices, with no round and with two of rows (two full ones take
//   as long or longer): G(16 000, 10 n) 168 -> 64, G(4000, 4 n) 54 -> 51, a path of
//   16 000 in index order 222 -> 46, 2D grid 60^2 49 -> 45, R-MAT 13 31 -> 34, a clique
//   of 1500 21 -> 29;
//   above 16 slots a vertex, with no round, one and two full ones, and two of an
//   eighth: G(n, 10 n) of 60 000 vertices 413, 81, 84, 89; of 200 000 1468, 146, 157,
//   122; G(n, 20 n) of 10^6 940, 528, 677, 441; R-MAT 20 328, 394, 526, 322; random
//   geometric 10^6 328, 201, -, 172;
//   elsewhere by the number of full rounds, from none: 2D grid 1500 x 1100, p = 0.6:
//   940, 641, 692, 214, 236; G(n, 3n) of 200 000 vertices 787, 970, 143, 156.
struct HookRounds {
  int rows, shares;
  uint32_t every;
};
HookRounds hook_rounds(uint64_t n, uint64_t m2) {
  if (n < (1u << 14)) return {2, 0, 1};
  if (m2 > 16 * n) return {0, 2, 8};
  return {0, n < (1u << 19) ? 2 : 3, 1};
}

}  // namespace

void union_components(uint64_t n, uint64_t m2, const uint64_t *off, const uint32_t *col, uint64_t block,
                      uint32_t *parent, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_union_init, dim3(blocks_for(n)), dim3(kBlock), 0, s, n, off, col, block, parent);
  KC_LAUNCH_CHECK();
  if (!m2) return;
  const auto share_blocks = [&](uint32_t every) {
    return dim3(static_cast<unsigned>(ceil_div(m2, static_cast<uint64_t>(kWaveSlots) * (kBlock / kWave) * every)));
  };
  const HookRounds rounds = hook_rounds(n, m2);
  shorten(n, parent, s);
  for (int r = 0; r < rounds.rows; ++r) {
    hipLaunchKernelGGL(k_union_hook_rows, dim3(blocks_for(n)), dim3(kBlock), 0, s, n, off, col, block, parent,
                       static_cast<uint32_t>(r));
    KC_LAUNCH_CHECK();
    shorten(n, parent, s);
  }
  for (int r = 0; r < rounds.shares; ++r) {
    hipLaunchKernelGGL(k_union_link<true>, share_blocks(rounds.every), dim3(kBlock), 0, s, n, m2, off, col, block,
                       parent, rounds.every, rounds.every > 1 ? static_cast<uint32_t>(r) : 0u);
    KC_LAUNCH_CHECK();
    shorten(n, parent, s, rounds.every == 1);  // (dense graphs' trees are shallow)
  }
  hipLaunchKernelGGL(k_union_link<false>, share_blocks(1), dim3(kBlock), 0, s, n, m2, off, col, block, parent, 1u, 0u);
  KC_LAUNCH_CHECK();
  shorten(n, parent, s);
}

void union_reps(uint64_t n, const uint32_t *parent, const uint32_t *gid, uint32_t *rep, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_union_reps, dim3(blocks_for(n)), dim3(kBlock), 0, s, n, parent, gid, rep);
  KC_LAUNCH_CHECK();
}

void union_keys(uint64_t n, const uint32_t *parent, uint64_t *key, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_union_keys, dim3(blocks_for(n)), dim3(kBlock), 0, s, n, parent, key);
  KC_LAUNCH_CHECK();
}

void union_labels(uint64_t n, const uint32_t *parent, uint32_t *labels, uint32_t *roots, uint32_t *partial,
                  hipStream_t s) {
  if (!n) return;
  const unsigned g = std::min(blocks_for(n), kUnionCountBlocks);
  hipLaunchKernelGGL(k_union_labels, dim3(g), dim3(kBlock), 0, s, n, parent, labels, partial);
  KC_LAUNCH_CHECK();
  sum_partials_u32(partial, g, roots, s);
}

}  // namespace kc
