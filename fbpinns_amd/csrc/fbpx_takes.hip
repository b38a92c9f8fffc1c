// Take and work-list builder on the device: the reference's get_inputs
// (trainers.py:332-419) -- inside test, active remap, all_ims = [active;
// fixed], m_take re-index, the (point, pou) unique of jnp.unique
// (trainers.py:380-388) -- followed by this library's kernel layout (tile
// order, segments and slots, chunks and launch bins; fbpx_worklist).
//
// Everything is integer work over the pair list.  The stages:
//   count    per point, the boxes holding it (inside_kernel) -> exclusive scan
//            -> offsets; the host reads the pair count s (one sync).
//   fill     point-major pairs (n_take, global model), ascending box id per
//            point: the row-major nonzero of the inside matrix
//            (decompositions_base.py:50-68).
//   used     models holding at least one point (LDS flags per workgroup).
//   remap    one workgroup: active 0 -> 1, times used (trainers.py:351-357),
//            all_ims = ascending active ids then ascending fixed ids, its
//            inverse, and the number of distinct pou values.
//   segments per point, the distinct pou values of its pairs (a 32-bit mask:
//            pou values lie in [0, 32)); segment = (point, pou) in ascending
//            order, so its index is jnp.unique's inverse p_take; the pairs
//            of a segment keep the point-major (reference) order, which
//            gives each pair its slot.
//   tiles    pairs grouped by model position, ascending point within: a
//            stable counting sort of the point-major pairs by model position.
//            Each workgroup takes the pairs of tile_points(m) points, counts
//            them per model in LDS, one exclusive scan in (model, block) order gives
//            every block's place in every model, and a fill pass writes the
//            pairs there in order (tile_sort_kernel).
//   chunks   cut flags at every model start, every `chunk` pairs inside a
//            model and at both kernels' bin edges (round(linspace) over the
//            pairs, numpy's half-to-even rounding), compacted by a scan.
// All sums are exclusive scans with a fixed order; the only atomics are
// order-independent (the "used" flags, the sort's integer counts in LDS), so the
// result is a function of the input alone.
#include <algorithm>

#include "fbpx_common.hpp"

namespace fbpx {
namespace {

constexpr int kThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kThreads * kScanItems;   // elements per scan workgroup
constexpr int kXcds = 8;                            // dies with an L2 each, workgroups dealt in turn
constexpr int kSortWaves = 8;                       // waves of a tile workgroup
constexpr int kSortAhead = 8;                       // 64-pair steps whose pairs are read at once
constexpr int kSortModels = 1536;                   // models counted at a time (48 KB of LDS counters)
// Points per tile workgroup: 512, or 1,024 where several windows of models are
// counted (the counts, one per model and workgroup, are then the larger part).
// 864 models, 524,288 points, 3.6 M pairs: count and place 9.4 + 102 us with
// 2,048 or 1,024 points, 8.8 + 61.6 with 512; a build with 6,400 models and
// 200,000 points 1,320 us with 1,024, 1,340 with 512.
constexpr int tile_points(int m) { return m <= kSortModels ? 512 : 1024; }
constexpr int kUsedLds = 32768;                     // models flagged in LDS
constexpr int64_t kUsedPairs = 4096;                // pairs per "used" workgroup
constexpr int kMaxPou = 32;

// ------------------------------------------------------------------ scan

template <class T>
__device__ inline T wave_incl_scan(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T u = __shfl_up(v, d, 64);
    if (lane >= d) v += u;
  }
  return v;
}

// Exclusive scan over the NT threads of the workgroup (thread order); total
// is the sum over all threads.  Every thread must call it.
template <class T, int NT = kThreads>
__device__ inline T block_excl_scan(T v, T& total) {
  __shared__ T wsum[NT / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const T inc = wave_incl_scan(v);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  T base = 0;
  total = 0;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) {
    if (i < w) base += wsum[i];
    total += wsum[i];
  }
  __syncthreads();
  return base + inc - v;
}

// tsum[tile] = sum of in[i] over the tile's elements i < n.
template <class In>
__global__ void __launch_bounds__(kThreads) scan_tile_sums(const In* __restrict__ in, int64_t n,
                                                           int64_t* __restrict__ tsum) {
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int64_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k)
    if (base + k < n) s += (int64_t)in[base + k];
  int64_t tot;
  block_excl_scan<int64_t>(s, tot);
  if (threadIdx.x == 0) tsum[blockIdx.x] = tot;
}

// Exclusive scan of tsum[0 .. nt) in place, one workgroup.
__global__ void __launch_bounds__(kThreads) scan_tile_prefix(int64_t* __restrict__ tsum, int64_t nt) {
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < nt; b0 += kScanTile) {
    const int64_t base = b0 + (int64_t)threadIdx.x * kScanItems;
    int64_t v[kScanItems], s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      v[k] = base + k < nt ? tsum[base + k] : 0;
      s += v[k];
    }
    int64_t tot;
    int64_t run = carry + block_excl_scan<int64_t>(s, tot);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      if (base + k < nt) tsum[base + k] = run;
      run += v[k];
    }
    carry += tot;
  }
}

// out[i] = sum of in[j] for j < i, for i <= n (out[n] = total).  in and out
// may be the same array (each workgroup reads its elements before writing).
template <class In, class Out>
__global__ void __launch_bounds__(kThreads) scan_apply(const In* in, int64_t n, const int64_t* __restrict__ tsum,
                                                       Out* out) {
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int64_t v[kScanItems], s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = base + k < n ? (int64_t)in[base + k] : 0;
    s += v[k];
  }
  int64_t tot;
  int64_t run = tsum[blockIdx.x] + block_excl_scan<int64_t>(s, tot);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    if (base + k <= n) out[base + k] = (Out)run;
    run += v[k];
  }
}

int64_t scan_tiles(int64_t n) { return (n + 1 + kScanTile - 1) / kScanTile; }

// Exclusive scan of n elements into n + 1 outputs; tsum: scan_tiles(n) int64.
template <class In, class Out>
void scan(hipStream_t s, const In* in, int64_t n, Out* out, int64_t* tsum) {
  const int64_t nt = scan_tiles(n);
  hipLaunchKernelGGL(scan_tile_sums<In>, dim3((unsigned)nt), dim3(kThreads), 0, s, in, n, tsum);
  hipLaunchKernelGGL(scan_tile_prefix, dim3(1), dim3(kThreads), 0, s, tsum, nt);
  hipLaunchKernelGGL((scan_apply<In, Out>), dim3((unsigned)nt), dim3(kThreads), 0, s, in, n, tsum, out);
}

// ------------------------------------------------------------------ helpers

template <class T>
__global__ void __launch_bounds__(kThreads) fill_kernel(T* __restrict__ p, int64_t n, T v) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) p[i] = v;
}

template <class T>
void fill(hipStream_t s, T* p, int64_t n, T v) {
  if (n <= 0) return;
  const int64_t nb = (n + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(fill_kernel<T>, dim3((unsigned)(nb < 65536 ? nb : 65536)), dim3(kThreads), 0, s, p, n, v);
}

unsigned grid_for(int64_t n) { return (unsigned)((n + kThreads - 1) / kThreads); }

// used[j] = 1 for every model j holding a pair.  Each workgroup flags its
// pairs' models in LDS (when m fits) and writes each flag once.
__global__ void __launch_bounds__(kThreads) used_kernel(const int32_t* __restrict__ mg, int64_t s, int m,
                                                        uint8_t* __restrict__ used) {
  __shared__ uint8_t f[kUsedLds];
  const bool lds = m <= kUsedLds;
  if (lds) {
    for (int j = threadIdx.x; j < m; j += kThreads) f[j] = 0;
    __syncthreads();
  }
  const int64_t b0 = (int64_t)blockIdx.x * kUsedPairs;
  const int64_t b1 = b0 + kUsedPairs < s ? b0 + kUsedPairs : s;
  for (int64_t q = b0 + threadIdx.x; q < b1; q += kThreads) {
    const int j = mg[q];
    if (lds)
      f[j] = 1;
    else
      used[j] = 1;
  }
  if (lds) {
    __syncthreads();
    for (int j = threadIdx.x; j < m; j += kThreads)
      if (f[j]) used[j] = 1;
  }
}

// info slots (device int32, read back by the host at the end)
enum { kInfoActive = 0, kInfoUsed, kInfoNpou, kInfoBadActive, kInfoBadPou, kInfoBadOffsets,
       kInfoSegs, kInfoCuts, kInfoPlaced, kInfoLen = 16 };

// One workgroup: the active remap of trainers.py:347-357 and all_ims.
constexpr int kRemapThreads = 1024;
__global__ void __launch_bounds__(kRemapThreads) remap_kernel(const int32_t* __restrict__ active,
                                                              const uint8_t* __restrict__ used,
                                                              const int32_t* __restrict__ pou, int m,
                                                              int32_t* __restrict__ act_out,
                                                              int32_t* __restrict__ all_ims,
                                                              int32_t* __restrict__ inv, int32_t* __restrict__ info) {
  __shared__ uint32_t pmask;
  __shared__ int bad;   // bit 0: active, bit 1: pou
  if (threadIdx.x == 0) {
    pmask = 0;
    bad = 0;
  }
  uint32_t my_pou = 0;
  int my_bad = 0;
  int carry = 0;
  for (int j0 = 0; j0 < m; j0 += kRemapThreads) {
    const int j = j0 + threadIdx.x;
    int a = 0;
    if (j < m) {
      a = active[j];
      if (a < 0 || a > 2) my_bad |= 1;
      const int pv = pou[j];
      if (pv < 0 || pv >= kMaxPou)
        my_bad |= 2;
      else
        my_pou |= 1u << pv;
      if (a == 0) a = 1;
      if (!used[j]) a = 0;
      act_out[j] = a;
      inv[j] = -1;
    }
    int tot;
    const int ex = block_excl_scan<int, kRemapThreads>(a == 1, tot);
    if (a == 1) {
      all_ims[carry + ex] = j;
      inv[j] = carry + ex;
    }
    carry += tot;
  }
  const int n_active = carry;
  for (int j0 = 0; j0 < m; j0 += kRemapThreads) {
    const int j = j0 + threadIdx.x;
    const int a = j < m ? act_out[j] : 0;
    int tot;
    const int ex = block_excl_scan<int, kRemapThreads>(a == 2, tot);
    if (a == 2) {
      all_ims[carry + ex] = j;
      inv[j] = carry + ex;
    }
    carry += tot;
  }
  __syncthreads();
  if (my_pou) atomicOr(&pmask, my_pou);
  if (my_bad) atomicOr(&bad, my_bad);
  __syncthreads();
  if (threadIdx.x == 0) {
    info[kInfoActive] = n_active;
    info[kInfoUsed] = carry;
    info[kInfoNpou] = __popc(pmask);
    info[kInfoBadActive] = bad & 1;
    info[kInfoBadPou] = bad >> 1;
  }
}

// Per point: the mask of pou values among its pairs (pmask) and the number
// of distinct values (its segment count, written to nseg for the scan).
__global__ void __launch_bounds__(kThreads) seg_count_kernel(int n, const int64_t* __restrict__ off,
                                                             const int32_t* __restrict__ mg,
                                                             const int32_t* __restrict__ pou,
                                                             uint32_t* __restrict__ pmask, int32_t* __restrict__ nseg) {
  const int p = blockIdx.x * kThreads + threadIdx.x;
  if (p >= n) return;
  uint32_t mask = 0;
  for (int64_t q = off[p]; q < off[p + 1]; ++q) {
    const int v = pou[mg[q]];
    if ((unsigned)v < (unsigned)kMaxPou) mask |= 1u << v;   // others: reported by remap_kernel
  }
  pmask[p] = mask;
  nseg[p] = __popc(mask);
}

// Per point: the pair count of each of its segments (ascending pou).
__global__ void __launch_bounds__(kThreads) seg_size_kernel(int n, const int64_t* __restrict__ off,
                                                            const int32_t* __restrict__ mg,
                                                            const int32_t* __restrict__ pou,
                                                            const uint32_t* __restrict__ pmask,
                                                            const int32_t* __restrict__ point_seg_start,
                                                            int32_t* __restrict__ segcnt) {
  const int p = blockIdx.x * kThreads + threadIdx.x;
  if (p >= n) return;
  int seg = point_seg_start[p];
  const int64_t q0 = off[p], q1 = off[p + 1];
  for (uint32_t mm = pmask[p]; mm; mm &= mm - 1, ++seg) {
    const int v = __ffs(mm) - 1;
    int c = 0;
    for (int64_t q = q0; q < q1; ++q) c += pou[mg[q]] == v;
    segcnt[seg] = c;
  }
}

// Per pair: p_take, the slot (segment start + its rank among the segment's
// pairs in point-major order), the re-indexed m_take and, at a segment's first
// pair, np_take.  A thread per pair keeps the three output streams coalesced
// (a thread per point took 65 us for 3.6 M pairs).
__global__ void __launch_bounds__(kThreads) seg_fill_kernel(int64_t s, const int64_t* __restrict__ off,
                                                            const int32_t* __restrict__ n_take,
                                                            const int32_t* __restrict__ mg,
                                                            const int32_t* __restrict__ pou,
                                                            const uint32_t* __restrict__ pmask,
                                                            const int32_t* __restrict__ point_seg_start,
                                                            const int32_t* __restrict__ seg_pair_start,
                                                            const int32_t* __restrict__ inv,
                                                            int32_t* __restrict__ p_take, int32_t* __restrict__ slot_pm,
                                                            int32_t* __restrict__ np_take,
                                                            int32_t* __restrict__ m_take) {
  const int64_t q = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (q >= s) return;
  const int p = n_take[q], j = mg[q];
  m_take[q] = inv[j];
  const int v = pou[j];
  if ((unsigned)v >= (unsigned)kMaxPou) return;   // reported by remap_kernel
  const uint32_t mm = pmask[p];
  const int64_t q0 = off[p];
  const int seg = point_seg_start[p] + __popc(mm & ((1u << v) - 1));
  int rank = (int)(q - q0);
  if (mm & (mm - 1)) {   // several levels: count the point's earlier pairs of this one
    rank = 0;
    for (int64_t r = q0; r < q; ++r) rank += pou[mg[r]] == v;
  }
  p_take[q] = seg;
  slot_pm[q] = seg_pair_start[seg] + rank;
  if (rank == 0) np_take[seg] = p;
}

// Stable counting sort of the point-major pairs by model position, one
// workgroup per block of tile_points(m) points, wave w over its share of them
// in order, kSortModels models at a time.
// FILL = false: blkcnt[k * nblk + b] = the block's pairs of model position k
// (0 for k >= n_used).  FILL = true: blkcnt holds the scanned bases; each
// wave turns its counts into its own bases and places its pairs 64 at a time,
// a pair's place being its model's base plus its rank among the 64 lanes
// (equal models found by one ballot per bit of the position), so pairs of a
// model stay in point-major order.  Bound by partial-line writes: a block's run
// of a model is a few pairs, and its neighbours in memory come from the next
// blocks.  Workgroups are dealt to the dies in turn, so each die takes a run of
// consecutive blocks (and blocks are small enough to be in flight together):
// the lines fill in its L2 before they leave it.  Placing 3.6 M pairs of 864
// models took 131 us with blocks dealt in order, 102 with this mapping, 61.6
// with 512 points per block as well.  (Testing every point of a block against
// every box and searching each pair's twin in its point's list took 1.85 ms.)
template <bool FILL>
__global__ void __launch_bounds__(64 * kSortWaves) tile_sort_kernel(
    int n, int nblk, int m, int win, const int64_t* __restrict__ off, const int32_t* __restrict__ info,
    const int32_t* __restrict__ m_take, const int32_t* __restrict__ n_take, const int32_t* __restrict__ p_take,
    const int32_t* __restrict__ slot_pm, int32_t* __restrict__ blkcnt, int32_t* __restrict__ pair_point,
    int32_t* __restrict__ pair_seg, int32_t* __restrict__ pair_slot) {
  extern __shared__ int32_t sort_cnt[];   // [kSortWaves][win]
  const int tp = tile_points(m), wave_points = tp / kSortWaves;
  const int per = gridDim.x / kXcds;   // the grid is kXcds times as many as a die's blocks
  const int b = (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (b >= nblk) return;
  int32_t* cnt = sort_cnt + w * win;
  const int n_used = info[kInfoUsed];
  const int p0 = (int)min((int64_t)n, (int64_t)b * tp + w * wave_points), p1 = (int)min((int64_t)n, (int64_t)p0 + wave_points);
  const int64_t q0 = off[p0], q1 = off[p1];
  for (int k0 = 0; k0 < (FILL ? n_used : m); k0 += win) {
    for (int k = lane; k < win; k += 64) cnt[k] = 0;
    if (k0 < n_used) {
      for (int64_t q = q0 + lane; q < q1; q += 64 * kSortAhead) {
        int k[kSortAhead];
#pragma unroll
        for (int j = 0; j < kSortAhead; ++j) k[j] = m_take[min(q + 64 * j, q1 - 1)] - k0;
#pragma unroll
        for (int j = 0; j < kSortAhead; ++j)
          if (q + 64 * j < q1 && k[j] >= 0 && k[j] < win) atomicAdd(&cnt[k[j]], 1);
      }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < win && k0 + k < m; k += 64 * kSortWaves) {
      const int64_t slot = (int64_t)(k0 + k) * nblk + b;
      int32_t base = FILL ? blkcnt[slot] : 0;
      for (int v = 0; v < kSortWaves; ++v) {
        const int32_t c = sort_cnt[v * win + k];
        if (FILL) sort_cnt[v * win + k] = base;
        base += c;
      }
      if (!FILL) blkcnt[slot] = base;
    }
    __syncthreads();
    if (FILL) {
      // kSortAhead steps' pairs are read at once
      for (int64_t qb = q0; qb < q1; qb += 64 * kSortAhead) {   // wave-uniform trip count
        int ka[kSortAhead], pp[kSortAhead], ps[kSortAhead], pt[kSortAhead];
#pragma unroll
        for (int j = 0; j < kSortAhead; ++j) {
          const int64_t q = min(qb + 64 * j + lane, q1 - 1);
          ka[j] = m_take[q];
          pp[j] = n_take[q];
          ps[j] = p_take[q];
          pt[j] = slot_pm[q];
        }
#pragma unroll
        for (int j = 0; j < kSortAhead; ++j) {
          const int k = qb + 64 * j + lane < q1 ? ka[j] - k0 : -1;
          const bool in = k >= 0 && k < win;
          uint64_t same = __ballot(in);
          if (same == 0) continue;
#pragma unroll
          for (int bit = 0; bit < 11; ++bit) {
            const bool one = (k >> bit) & 1;
            const uint64_t v = __ballot(one);
            same &= one ? v : ~v;
          }
          if (in) {
            const int64_t t = cnt[k] + __popcll(same & ((1ull << lane) - 1));
            // the model's highest lane moves its base past the 64 pairs, after
            // every lane has read it (a wave's LDS operations are in order)
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if ((same >> lane) == 1) cnt[k] += __popcll(same);
            pair_point[t] = pp[j];
            pair_seg[t] = ps[j];
            pair_slot[t] = pt[j];
          }
          __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
      }
      __syncthreads();
    }
  }
}
static_assert(kSortModels <= 1 << 11, "a model position within a window is matched on 11 bits");

// model_start[k] = base[k * nblk] for k <= n_used (base[n_used * nblk] = s).
__global__ void __launch_bounds__(kThreads) model_start_kernel(const int32_t* __restrict__ base, int nblk, int m,
                                                               const int32_t* __restrict__ info,
                                                               int32_t* __restrict__ model_start) {
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if (k <= info[kInfoUsed] && k <= m) model_start[k] = base[(int64_t)k * nblk];
}

// Cut flags at model starts and every `chunk` pairs inside a model.
__global__ void __launch_bounds__(kThreads) cut_models_kernel(const int32_t* __restrict__ model_start, int m,
                                                              const int32_t* __restrict__ info, int chunk,
                                                              uint8_t* __restrict__ flags) {
  const int k = blockIdx.x * kThreads + threadIdx.x;
  const int n_used = info[kInfoUsed];
  if (k > n_used || k > m) return;
  const int t0 = model_start[k];
  flags[t0] = 1;
  if (chunk > 0 && k < n_used) {
    const int cnt = model_start[k + 1] - t0;
    for (int t = chunk; t < cnt; t += chunk) flags[t0 + t] = 1;
  }
}

// Cut flags at round(linspace(0, S, nb + 1)) (numpy: i * (S / nb) in float64,
// the last point exactly S, rounded half to even), S = s or the trained
// prefix model_start[n_active].
__global__ void __launch_bounds__(kThreads) cut_bins_kernel(int nb, int64_t s, const int32_t* __restrict__ model_start,
                                                            const int32_t* __restrict__ info, bool trained,
                                                            uint8_t* __restrict__ flags, int32_t* __restrict__ edges) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i > nb) return;
  const int64_t S = trained ? (int64_t)model_start[info[kInfoActive]] : s;
  const double step = (double)S / (double)nb;
  const int64_t t = i == nb ? S : (int64_t)rint((double)i * step);
  flags[t] = 1;
  edges[i] = (int32_t)t;
}

// chunk_start[cut[t]] = t for every flagged position t <= s.
__global__ void __launch_bounds__(kThreads) chunk_start_kernel(const uint8_t* __restrict__ flags,
                                                               const int32_t* __restrict__ cut, int64_t s,
                                                               int32_t* __restrict__ chunk_start) {
  const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (t <= s && flags[t]) chunk_start[cut[t]] = (int32_t)t;
}

// Per chunk: its model position (the last model start <= its start), model
// id and trained flag.
__global__ void __launch_bounds__(kThreads) chunk_info_kernel(const int32_t* __restrict__ chunk_start,
                                                              const int32_t* __restrict__ cut, int64_t s,
                                                              const int32_t* __restrict__ model_start,
                                                              const int32_t* __restrict__ all_ims,
                                                              const int32_t* __restrict__ info,
                                                              int32_t* __restrict__ chunk_model,
                                                              uint8_t* __restrict__ chunk_train) {
  const int c = blockIdx.x * kThreads + threadIdx.x;
  const int n_chunks = cut[s + 1] - 1;
  if (c >= n_chunks) return;
  const int t = chunk_start[c];
  int a = 0, e = info[kInfoUsed] + 1;   // upper bound of t in model_start[0 .. n_used]
  while (a < e) {
    const int mid = (a + e) >> 1;
    if (model_start[mid] <= t)
      a = mid + 1;
    else
      e = mid;
  }
  const int pos = a - 1;
  chunk_model[c] = all_ims[pos];
  chunk_train[c] = pos < info[kInfoActive] ? 1 : 0;
}

// row_chunk_start[k] = the chunk starting at model k's first pair (k <= n_active).
__global__ void __launch_bounds__(kThreads) rows_kernel(const int32_t* __restrict__ model_start,
                                                        const int32_t* __restrict__ cut,
                                                        const int32_t* __restrict__ info, int m,
                                                        int32_t* __restrict__ row_chunk_start) {
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if (k <= info[kInfoActive] && k <= m) row_chunk_start[k] = cut[model_start[k]];
}

// bin_chunk_start[i] = the chunk starting at bin edge i (nb > 0), or i for
// every chunk (nb == 0: one bin per chunk).
__global__ void __launch_bounds__(kThreads) bins_kernel(int nb, const int32_t* __restrict__ edges,
                                                        const int32_t* __restrict__ cut, int64_t s, int max_chunks,
                                                        int32_t* __restrict__ bin_chunk_start) {
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (nb > 0) {
    if (i <= nb) bin_chunk_start[i] = cut[edges[i]];
  } else if (i <= cut[s + 1] - 1 && i <= max_chunks) {
    bin_chunk_start[i] = i;
  }
}

// The sizes found on the way, next to the other info slots (one read-back).
__global__ void sizes_kernel(const int32_t* __restrict__ n_segs, const int32_t* __restrict__ cuts,
                             const int32_t* __restrict__ placed, int32_t* __restrict__ info) {
  info[kInfoSegs] = *n_segs;
  info[kInfoCuts] = *cuts;
  info[kInfoPlaced] = *placed;
}

// ------------------------------------------------------------------ work space

size_t align_up(size_t v) { return (v + 255) & ~size_t(255); }

struct Carve {
  char* base;
  size_t off, cap;
  template <class T>
  T* take(int64_t count) {
    T* p = reinterpret_cast<T*>(base ? base + off : nullptr);
    off += align_up((size_t)(count > 0 ? count : 1) * sizeof(T));
    return p;
  }
};

int64_t nblocks(int n, int m) { return ((int64_t)n + tile_points(m) - 1) / tile_points(m); }

struct Work {
  int32_t* counts;
  int64_t* tsum;
  int32_t* mg;
  uint8_t* used;
  int32_t* inv;
  int32_t* info;
  uint32_t* pmask;
  int32_t* slot_pm;
  int32_t* blkcnt;
  int32_t* model_start;
  uint8_t* flags;
  int32_t* cut;
  int32_t* fedges;
  int32_t* bedges;
};

Work carve(void* base, int n, int xd, int m, int64_t s, int fbins, int bbins, size_t* bytes) {
  Carve c{static_cast<char*>(base), 0, 0};
  Work w;
  const int64_t nb = nblocks(n, m);
  const int64_t nmax = std::max<int64_t>(std::max<int64_t>(n, s + 1), (int64_t)m * nb + 1);
  w.counts = c.take<int32_t>(n);
  w.tsum = c.take<int64_t>(scan_tiles(nmax) + 1);
  w.mg = c.take<int32_t>(s);
  w.used = c.take<uint8_t>(m);
  w.inv = c.take<int32_t>(m);
  w.info = c.take<int32_t>(kInfoLen);
  w.pmask = c.take<uint32_t>(n);
  w.slot_pm = c.take<int32_t>(s);
  w.blkcnt = c.take<int32_t>((int64_t)m * nb + 1);
  w.model_start = c.take<int32_t>((int64_t)m + 1);
  w.flags = c.take<uint8_t>(s + 1);
  w.cut = c.take<int32_t>(s + 2);
  w.fedges = c.take<int32_t>((int64_t)fbins + 1);
  w.bedges = c.take<int32_t>((int64_t)bbins + 1);
  *bytes = c.off;
  return w;
}

void launch_tiles(hipStream_t st, bool fill_pass, int n, int nblk, int m, const Work& w, const int64_t* off,
                  const fbpx_takes_out& o) {
  const int win = std::min(m, kSortModels);
  const size_t lds = sizeof(int32_t) * kSortWaves * win;
  const unsigned grid = (unsigned)((nblk + kXcds - 1) / kXcds * kXcds);
  hipLaunchKernelGGL(fill_pass ? tile_sort_kernel<true> : tile_sort_kernel<false>, dim3(grid),
                     dim3(64 * kSortWaves), lds, st, n, nblk, m, win, off, w.info, o.m_take, o.n_take, o.p_take,
                     w.slot_pm, w.blkcnt, o.pair_point, o.pair_seg, o.pair_slot);
}

int check_sizes(const char* what, const float* x, int32_t n, int32_t xd, const float* xmin, const float* xmax,
                int32_t m) {
  if (n < 0 || m < 1 || xd < 1 || xd > FBPX_MAX_XD || (n > 0 && !x) || !xmin || !xmax) {
    set_error("%s: bad arguments n=%d m=%d xd=%d", what, n, m, xd);
    return FBPX_EINVAL;
  }
  return FBPX_OK;
}

}  // namespace
}  // namespace fbpx

using namespace fbpx;

extern "C" {

int64_t fbpx_takes_max_chunks(int32_t m, int64_t n_pairs, int32_t chunk, int32_t fbins, int32_t bbins) {
  return (chunk > 0 ? n_pairs / chunk : 0) + 2 * (int64_t)m + (int64_t)fbins + (int64_t)bbins + 3;
}

int64_t fbpx_takes_work_bytes(int32_t n, int32_t xd, int32_t m, int64_t n_pairs, int32_t fbins, int32_t bbins) {
  if (n < 0 || m < 1 || xd < 1 || xd > FBPX_MAX_XD || n_pairs < 0 || fbins < 0 || bbins < 0) return -1;
  size_t bytes = 0;
  carve(nullptr, n, xd, m, n_pairs, fbins, bbins, &bytes);
  return (int64_t)bytes;
}

int fbpx_takes_count(void* stream, const float* x, int32_t n, int32_t xd, const float* xmin, const float* xmax,
                     int32_t m, int64_t* offsets, void* work, int64_t work_bytes, int64_t* n_pairs) {
  int rc = check_sizes("takes_count", x, n, xd, xmin, xmax, m);
  if (rc) return rc;
  size_t need = 0;
  carve(nullptr, n, xd, m, 0, 0, 0, &need);
  if (!offsets || !n_pairs || !work || work_bytes < (int64_t)need) {
    set_error("takes_count: null output or work space of %lld bytes (need %zu)", (long long)work_bytes, need);
    return FBPX_EINVAL;
  }
  hipStream_t s = (hipStream_t)stream;
  Work w = carve(work, n, xd, m, 0, 0, 0, &need);
  if (n > 0 && (rc = fbpx_inside_count(stream, x, n, xd, xmin, xmax, m, nullptr, w.counts))) return rc;
  scan<int32_t, int64_t>(s, w.counts, n, offsets, w.tsum);
  if ((rc = hip_check(hipGetLastError(), "takes_count"))) return rc;
  int64_t total = 0;
  if ((rc = hip_check(hipMemcpyAsync(&total, offsets + n, sizeof(int64_t), hipMemcpyDeviceToHost, s),
                      "takes_count: copy")))
    return rc;
  if ((rc = hip_check(hipStreamSynchronize(s), "takes_count: sync"))) return rc;
  if (total > INT32_MAX - 2) {
    set_error("takes_count: %lld (point, subdomain) pairs exceed the int32 work-list indices", (long long)total);
    return FBPX_EUNSUPPORTED;
  }
  *n_pairs = total;
  return FBPX_OK;
}

int fbpx_build_worklist(void* stream, const float* x, int32_t n, int32_t xd, const float* xmin, const float* xmax,
                        int32_t m, const int32_t* active, const int32_t* pou, const int64_t* offsets, int64_t n_pairs,
                        int32_t chunk, int32_t fbins, int32_t bbins, int64_t max_chunks, void* work,
                        int64_t work_bytes, const fbpx_takes_out* out, fbpx_takes_info* info) {
  int rc = check_sizes("build_worklist", x, n, xd, xmin, xmax, m);
  if (rc) return rc;
  if (!active || !pou || !offsets || !out || !info || n_pairs < 0 || n_pairs > INT32_MAX - 2 || chunk < 0 ||
      fbins < 0 || bbins < 0) {
    set_error("build_worklist: bad arguments (n_pairs=%lld chunk=%d fbins=%d bbins=%d)", (long long)n_pairs, chunk,
              fbins, bbins);
    return FBPX_EINVAL;
  }
  const int64_t s = n_pairs;
  const int64_t need_chunks = fbpx_takes_max_chunks(m, s, chunk, fbins, bbins);
  if (max_chunks < need_chunks || max_chunks > INT32_MAX - 2) {
    set_error("build_worklist: chunk arrays for %lld chunks, need %lld (fbpx_takes_max_chunks)",
              (long long)max_chunks, (long long)need_chunks);
    return FBPX_EINVAL;
  }
  size_t need = 0;
  carve(nullptr, n, xd, m, s, fbins, bbins, &need);
  if (!work || work_bytes < (int64_t)need) {
    set_error("build_worklist: work space of %lld bytes, need %zu", (long long)work_bytes, need);
    return FBPX_EINVAL;
  }
  const fbpx_takes_out& o = *out;
  if ((s > 0 && (!o.m_take || !o.n_take || !o.p_take || !o.np_take || !o.pair_point || !o.pair_seg ||
                 !o.pair_slot)) ||
      !o.active || !o.all_ims || !o.point_seg_start || !o.seg_pair_start || !o.chunk_model || !o.chunk_start ||
      !o.chunk_train || !o.row_chunk_start || !o.fbin_chunk_start || !o.bbin_chunk_start) {
    set_error("build_worklist: null output array");
    return FBPX_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  Work w = carve(work, n, xd, m, s, fbins, bbins, &need);
  const int64_t nblk = nblocks(n, m);

  // point-major pairs and the models they use
  fill<uint8_t>(st, w.used, m, 0);
  fill<int32_t>(st, w.info, kInfoLen, 0);
  if (s > 0) {
    if ((rc = inside_fill_checked(st, x, n, xd, xmin, xmax, m, offsets, s, o.n_take, w.mg, w.info + kInfoBadOffsets)))
      return rc;
    hipLaunchKernelGGL(used_kernel, dim3((unsigned)((s + kUsedPairs - 1) / kUsedPairs)), dim3(kThreads), 0, st, w.mg,
                       s, m, w.used);
  }
  hipLaunchKernelGGL(remap_kernel, dim3(1), dim3(kRemapThreads), 0, st, active, w.used, pou, m, o.active, o.all_ims, w.inv,
                     w.info);

  // segments: (point, pou) rows in ascending order and each pair's slot
  if (n > 0) {
    hipLaunchKernelGGL(seg_count_kernel, dim3(grid_for(n)), dim3(kThreads), 0, st, n, offsets, w.mg, pou, w.pmask,
                       o.point_seg_start);
  }
  scan<int32_t, int32_t>(st, o.point_seg_start, n, o.point_seg_start, w.tsum);
  fill<int32_t>(st, o.seg_pair_start, s, 0);
  if (n > 0)
    hipLaunchKernelGGL(seg_size_kernel, dim3(grid_for(n)), dim3(kThreads), 0, st, n, offsets, w.mg, pou, w.pmask,
                       o.point_seg_start, o.seg_pair_start);
  scan<int32_t, int32_t>(st, o.seg_pair_start, s, o.seg_pair_start, w.tsum);
  if (s > 0)
    hipLaunchKernelGGL(seg_fill_kernel, dim3(grid_for(s)), dim3(kThreads), 0, st, s, offsets, o.n_take, w.mg, pou,
                       w.pmask, o.point_seg_start, o.seg_pair_start, w.inv, o.p_take, w.slot_pm, o.np_take, o.m_take);

  // tile order: count per (model position, point block), scan, fill
  const int64_t nwg = (int64_t)m * nblk;
  if (nwg > 0) {
    launch_tiles(st, false, n, (int)nblk, m, w, offsets, o);
    scan<int32_t, int32_t>(st, w.blkcnt, nwg, w.blkcnt, w.tsum);
    launch_tiles(st, true, n, (int)nblk, m, w, offsets, o);
  } else {
    fill<int32_t>(st, w.blkcnt, 1, 0);
  }
  hipLaunchKernelGGL(model_start_kernel, dim3(grid_for((int64_t)m + 1)), dim3(kThreads), 0, st, w.blkcnt,
                     (int)(nblk > 0 ? nblk : 1), m, w.info, w.model_start);

  // chunks and bins
  fill<uint8_t>(st, w.flags, s + 1, 0);
  hipLaunchKernelGGL(cut_models_kernel, dim3(grid_for((int64_t)m + 1)), dim3(kThreads), 0, st, w.model_start, m, w.info,
                     chunk, w.flags);
  if (fbins > 0)
    hipLaunchKernelGGL(cut_bins_kernel, dim3(grid_for((int64_t)fbins + 1)), dim3(kThreads), 0, st, fbins, s,
                       w.model_start, w.info, false, w.flags, w.fedges);
  if (bbins > 0)
    hipLaunchKernelGGL(cut_bins_kernel, dim3(grid_for((int64_t)bbins + 1)), dim3(kThreads), 0, st, bbins, s,
                       w.model_start, w.info, true, w.flags, w.bedges);
  scan<uint8_t, int32_t>(st, w.flags, s + 1, w.cut, w.tsum);
  hipLaunchKernelGGL(chunk_start_kernel, dim3(grid_for(s + 1)), dim3(kThreads), 0, st, w.flags, w.cut, s,
                     o.chunk_start);
  hipLaunchKernelGGL(chunk_info_kernel, dim3(grid_for(max_chunks)), dim3(kThreads), 0, st, o.chunk_start, w.cut, s,
                     w.model_start, o.all_ims, w.info, o.chunk_model, o.chunk_train);
  hipLaunchKernelGGL(rows_kernel, dim3(grid_for((int64_t)m + 1)), dim3(kThreads), 0, st, w.model_start, w.cut, w.info,
                     m, o.row_chunk_start);
  hipLaunchKernelGGL(bins_kernel, dim3(grid_for((fbins > 0 ? fbins : max_chunks) + 1)), dim3(kThreads), 0, st, fbins,
                     w.fedges, w.cut, s, (int)max_chunks, o.fbin_chunk_start);
  hipLaunchKernelGGL(bins_kernel, dim3(grid_for((bbins > 0 ? bbins : max_chunks) + 1)), dim3(kThreads), 0, st, bbins,
                     w.bedges, w.cut, s, (int)max_chunks, o.bbin_chunk_start);
  // sizes back to the host
  hipLaunchKernelGGL(sizes_kernel, dim3(1), dim3(1), 0, st, o.point_seg_start + n, w.cut + s + 1, w.blkcnt + nwg,
                     w.info);
  if ((rc = hip_check(hipGetLastError(), "build_worklist"))) return rc;
  int32_t h_info[kInfoLen] = {};
  if ((rc = hip_check(hipMemcpyAsync(h_info, w.info, sizeof(h_info), hipMemcpyDeviceToHost, st), "copy info")) ||
      (rc = hip_check(hipStreamSynchronize(st), "build_worklist: sync")))
    return rc;
  if (h_info[kInfoBadActive]) {
    set_error("build_worklist: active values must be 0, 1 or 2 (trainers.py:348)");
    return FBPX_EINVAL;
  }
  if (h_info[kInfoBadPou]) {
    set_error("build_worklist: pou values must lie in [0, %d)", kMaxPou);
    return FBPX_EUNSUPPORTED;
  }
  if ((int64_t)h_info[kInfoPlaced] != s || h_info[kInfoBadOffsets]) {
    set_error("build_worklist: tile pass placed %d pairs of %lld (offsets not from fbpx_takes_count on these inputs?)",
              h_info[kInfoPlaced], (long long)s);
    return FBPX_EINVAL;
  }
  info->n_pairs = s;
  info->n_segs = h_info[kInfoSegs];
  info->n_used = h_info[kInfoUsed];
  info->n_active = h_info[kInfoActive];
  info->n_chunks = h_info[kInfoCuts] - 1;
  info->n_fbins = fbins > 0 ? fbins : h_info[kInfoCuts] - 1;
  info->n_bbins = bbins > 0 ? bbins : h_info[kInfoCuts] - 1;
  info->npou = h_info[kInfoNpou];
  return FBPX_OK;
}

}  // extern "C"
