// Counting sort of the particles by (scene, grid cell) (GridHash::construct,
// Framework/Topology/GridHash.cu:298-323, for a batch of independent scenes),
// the exclusive scans it needs (Core/Utility/Scan.cu), the fused integrator and
// the scatter back to the caller's order.
//
// HBM layout: caller arrays x, v are packed xyz float triples in original order
// (scenes concatenated); the sorted arrays xn, x0, xa, xb, vs are float4 in
// (scene, cell) order (w of the position buffers carries lambda between
// passes). Cells are compact: each scene owns the window of cells spanned by
// its in-grid particles plus one bucket for its out-of-grid particles.
// Between the steps of one call the state stays in the previous step's cell
// order (float4 x and v plus each particle's original index): the sort then
// reads nearly in order, and the order within a cell is still by original
// index, so the result is the same as from the caller's order.
#include <climits>

#include "pbf_device.h"

namespace pbf {

// ---------------------------------------------------------------------------
// Exclusive scan with a host-known length: blocks of 1024 threads x 4 elements
// scanned with wave64 shuffles, recursion over the block sums.

constexpr int kScanPerBlock = 4096;

// Exclusive scan of a 4096-element tile held 4 per thread; returns this
// thread's exclusive prefix of its first element and the tile total.
__device__ __forceinline__ int block_scan4(int a0, int a1, int a2, int a3, int& total) {
  __shared__ int wsum[16];
  const int tsum = a0 + a1 + a2 + a3;
  const int incl = wave_inclusive_scan(tsum);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  if (wave == 0) {
    int t = lane < 16 ? wsum[lane] : 0;
    t = wave_inclusive_scan(t);
    if (lane < 16) wsum[lane] = t;
  }
  __syncthreads();
  const int e = (wave > 0 ? wsum[wave - 1] : 0) + incl - tsum;
  total = wsum[15];
  __syncthreads();  // wsum is reused by the next call
  return e;
}

__device__ __forceinline__ void store4(int* out, int base, int n, int e, int a0, int a1, int a2) {
  if (base < n) out[base] = e;
  e += a0;
  if (base + 1 < n) out[base + 1] = e;
  e += a1;
  if (base + 2 < n) out[base + 2] = e;
  e += a2;
  if (base + 3 < n) out[base + 3] = e;
}

__global__ __launch_bounds__(1024) void k_scan_block(const int* in, int* out, int n, int* block_sums) {
  const int base = blockIdx.x * kScanPerBlock + threadIdx.x * 4;
  const int a0 = base < n ? in[base] : 0;
  const int a1 = base + 1 < n ? in[base + 1] : 0;
  const int a2 = base + 2 < n ? in[base + 2] : 0;
  const int a3 = base + 3 < n ? in[base + 3] : 0;
  int total;
  const int e = block_scan4(a0, a1, a2, a3, total);
  store4(out, base, n, e, a0, a1, a2);
  if (threadIdx.x == 0) {
    block_sums[blockIdx.x] = total;
    if (gridDim.x == 1) out[n] = total;
  }
}

__global__ __launch_bounds__(1024) void k_scan_add(int* out, int n, const int* block_offsets, int nb) {
  const int add = block_offsets[blockIdx.x];
  const int base = blockIdx.x * kScanPerBlock + threadIdx.x * 4;
#pragma unroll
  for (int t = 0; t < 4; ++t)
    if (base + t < n) out[base + t] += add;
  if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = block_offsets[nb];
}

size_t scan_scratch_ints(long long n) {
  long long nb = (n + kScanPerBlock - 1) / kScanPerBlock;
  if (nb <= 1) return 4;
  size_t here = (size_t)((nb + 3) / 4 * 4) + (size_t)((nb + 1 + 3) / 4 * 4);
  return here + scan_scratch_ints(nb);
}

void scan_exclusive(const int* in, int* out, int n, int* scratch, hipStream_t st) {
  const int nb = (n + kScanPerBlock - 1) / kScanPerBlock;
  if (nb <= 1) {
    k_scan_block<<<1, 1024, 0, st>>>(in, out, n, scratch);
    return;
  }
  int* sums = scratch;
  int* offs = scratch + (nb + 3) / 4 * 4;
  int* rest = offs + (nb + 1 + 3) / 4 * 4;
  k_scan_block<<<nb, 1024, 0, st>>>(in, out, n, sums);
  scan_exclusive(sums, offs, nb, rest, st);
  k_scan_add<<<nb, 1024, 0, st>>>(out, n, offs, nb);
}

// ---------------------------------------------------------------------------
// Exclusive scan with a device-resident length (reduce, scan the block sums,
// rescan): kScanDevBlocks blocks, each owning a contiguous chunk of tiles.

__device__ __forceinline__ void dev_chunk(int n, int& lo, int& hi) {
  const int tiles = (n + kScanPerBlock - 1) / kScanPerBlock;
  const int per = (tiles + gridDim.x - 1) / gridDim.x;
  lo = min(n, (int)blockIdx.x * per * kScanPerBlock);
  hi = min(n, lo + per * kScanPerBlock);
}

// One scan of a launch: length min(*n_ptr, n_max), n_max without n_ptr; gate
// (may be null): the scan runs only when *gate != 0. Row y of the grid runs
// scan y.
struct ScanJob {
  int* in;
  int* out;
  const int* n_ptr;
  int n_max;
  int* part;
  const unsigned long long* gate;
};

__global__ __launch_bounds__(1024) void k_scan_dev_reduce(ScanJob j0, ScanJob j1) {
  __shared__ int wsum[16];
  const ScanJob& job = blockIdx.y == 0 ? j0 : j1;
  if (job.gate && *job.gate == 0) return;
  const int* in = job.in;
  int* part = job.part;
  const int n = job.n_ptr ? min(*job.n_ptr, job.n_max) : job.n_max;
  int lo, hi;
  dev_chunk(n, lo, hi);
  int acc = 0;
  for (int t = lo + threadIdx.x; t < hi; t += 1024) acc += in[t];
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    int s = 0;
    for (int w = 0; w < 16; ++w) s += wsum[w];
    part[blockIdx.x] = s;
  }
}

// Each block first sums the block totals before its own (gridDim.x <= 1024)
// and the last block writes the grand total. The counts are zeroed once read,
// so the next sort starts from zero counts without a clearing pass (the array
// is zeroed when allocated).
__global__ __launch_bounds__(1024) void k_scan_dev_down(ScanJob j0, ScanJob j1) {
  const ScanJob& job = blockIdx.y == 0 ? j0 : j1;
  if (job.gate && *job.gate == 0) return;
  int* in = job.in;
  int* out = job.out;
  const int* part = job.part;
  const int n = job.n_ptr ? min(*job.n_ptr, job.n_max) : job.n_max;
  int lo, hi;
  dev_chunk(n, lo, hi);
  int before;
  {
    const int i = threadIdx.x;
    const int v = i < (int)gridDim.x ? part[i] : 0;
    int total;
    const int e = block_scan4(v, 0, 0, 0, total);
    __shared__ int off;
    if (i == (int)blockIdx.x) off = e;
    if (blockIdx.x == gridDim.x - 1 && i == 0) out[n] = total;
    __syncthreads();
    before = off;
  }
  int running = before;
  for (int t0 = lo; t0 < hi; t0 += kScanPerBlock) {
    const int base = t0 + threadIdx.x * 4;
    const int a0 = base < hi ? in[base] : 0;
    const int a1 = base + 1 < hi ? in[base + 1] : 0;
    const int a2 = base + 2 < hi ? in[base + 2] : 0;
    const int a3 = base + 3 < hi ? in[base + 3] : 0;
    int total;
    const int e = block_scan4(a0, a1, a2, a3, total);
    store4(out, base, hi, running + e, a0, a1, a2);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (base + t < hi) in[base + t] = 0;
    running += total;
  }
}

// ---------------------------------------------------------------------------
// Scene windows

// A scene's box: min i j k, max i j k of its in-grid particles' cells, its
// out-of-grid particles (kBoxInts ints per scene). Empty boxes hold INT_MAX,
// INT_MIN and 0: set once when the boxes are allocated; the windows empty each
// box again once it is read.
__host__ __device__ constexpr int empty_box(int a) { return a < 3 ? INT_MAX : (a < 6 ? INT_MIN : 0); }

__global__ void k_scene_reset(int* minmax, int nscenes) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < kBoxInts * nscenes) minmax[t] = empty_box(t % kBoxInts);
}

void launch_scene_reset(int* minmax, int nscenes, hipStream_t st) {
  if (nscenes > 0) k_scene_reset<<<(kBoxInts * nscenes + kBlock - 1) / kBlock, kBlock, 0, st>>>(minmax, nscenes);
}

__device__ __forceinline__ int scene_of(const int* __restrict__ off, int nscenes, int i) {
  int lo = 0, hi = nscenes;  // off[lo] <= i < off[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= i)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Position and velocity of input particle i (caller order or cell order).
template <bool kCellOrder>
__device__ __forceinline__ float3 in_pos(const SortIn& in, int i) {
  if (kCellOrder) {
    const float4 p = in.x4[i];
    return make_float3(p.x, p.y, p.z);
  }
  return make_float3(in.x[3 * (size_t)i], in.x[3 * (size_t)i + 1], in.x[3 * (size_t)i + 2]);
}
template <bool kCellOrder>
__device__ __forceinline__ float3 in_vel(const SortIn& in, int i) {
  if (kCellOrder) {
    const float4 p = in.v4[i];
    return make_float3(p.x, p.y, p.z);
  }
  return make_float3(in.v[3 * (size_t)i], in.v[3 * (size_t)i + 1], in.v[3 * (size_t)i + 2]);
}

__device__ __forceinline__ bool grid_cell(const GridDev& g, float3 p, int& ci, int& cj, int& ck, bool& nonfinite) {
  nonfinite = !(isfinite(p.x) && isfinite(p.y) && isfinite(p.z));
  cell_of(g, p.x, p.y, p.z, ci, cj, ck);
  return !nonfinite && in_grid(g, ci, cj, ck);
}

// The scene of particle i by one wave, 64 offsets at a time (every lane active).
__device__ __forceinline__ int scene_of_wave(const int* __restrict__ off, int nscenes, int i) {
  int lo = 0, hi = nscenes;  // off[lo] <= i < off[hi]
  while (hi - lo > 1) {
    const int step = (hi - lo + 63) >> 6;
    const int at = lo + (int)(threadIdx.x & 63) * step;
    const bool below = at < hi && (at == lo || off[at] <= i);
    const int last = 63 - __clzll(__ballot(below));  // the offsets never decrease
    lo += last * step;
    hi = min(hi, lo + step);
  }
  return lo;
}

// A word that another workgroup of the same kernel reads after the ticket below
// (written through to memory, read past the caches that other XCDs' writes do
// not reach).
__device__ __forceinline__ void share_store(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int share_load(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What the bounds pass leaves for the windows.
struct WindowOut {
  int* minmax;  // the scenes' boxes
  int nscenes;
  SceneWin* win;
  int* total_cells;
  const int* bpart;
  int nbounds;
  unsigned long long* counters;
  int* cell_cnt;
};

// Windows and compact cell bases of all scenes, by one workgroup of kWaves
// waves; each scene's box is emptied again for the next sort, and each
// out-of-grid bucket gets its count. With one scene the workgroup also reduces
// the bounds blocks' boxes (read as bload reads them). It also sets the search's
// counters: the out-of-grid and non-finite totals of the bounds pass, the cell
// total, and zero for the counters the neighbor pass accumulates.
template <int kWaves, class BLoad>
__device__ __forceinline__ void scene_windows(const WindowOut& o, BLoad&& bload) {
  __shared__ int box[kWaves][8];
  __shared__ int wsum[kWaves], base;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool one = o.nscenes == 1;
  int r[6] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN};
  int oog = 0, nonfinite = 0;
#pragma unroll 4
  for (int b = tid; b < o.nbounds; b += 64 * kWaves) {
    const int* e = o.bpart + 8 * (size_t)b;
    const unsigned v = (unsigned)bload(e + 7);
    oog += v & 0xffffu;
    nonfinite += v >> 16;
    if (one) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        r[a] = min(r[a], bload(e + 1 + a));
        r[3 + a] = max(r[3 + a], bload(e + 4 + a));
      }
    }
  }
  // every lane of the workgroup is active
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    r[a] = wave_min_full(r[a]);
    r[3 + a] = wave_max_full(r[3 + a]);
  }
  oog = wave_sum_full(oog);
  nonfinite = wave_sum_full(nonfinite);
  if (lane == 0) {
#pragma unroll
    for (int a = 0; a < 6; ++a) box[wave][a] = r[a];
    box[wave][6] = oog;
    box[wave][7] = nonfinite;
  }
  if (tid == 0) base = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w == 0) oog = nonfinite = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      r[a] = min(r[a], box[w][a]);
      r[3 + a] = max(r[3 + a], box[w][3 + a]);
    }
    oog += box[w][6];
    nonfinite += box[w][7];
  }
  for (int s0 = 0; s0 < o.nscenes; s0 += 64 * kWaves) {
    const int s = s0 + tid;
    SceneWin w{};
    int cells = 0, out = 0;
    if (s < o.nscenes) {
      int m[7];
      if (one) {
#pragma unroll
        for (int a = 0; a < 6; ++a) m[a] = r[a];
        m[6] = oog;
      } else {
        int* p = o.minmax + kBoxInts * (size_t)s;
#pragma unroll
        for (int a = 0; a < 7; ++a) {
          m[a] = bload(p + a);
          p[a] = empty_box(a);
        }
      }
      if (m[3] >= m[0]) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          w.lo[a] = m[a];
          w.dim[a] = m[a + 3] - m[a] + 1;
        }
      }
      w.ncell = w.dim[0] * w.dim[1] * w.dim[2];
      cells = w.ncell + 1;  // + out-of-grid bucket
      out = m[6];
    }
    const int incl = wave_inclusive_scan(cells);
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int before = base, all = 0;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
      before += k < wave ? wsum[k] : 0;
      all += wsum[k];
    }
    if (s < o.nscenes) {
      w.cell_base = before + incl - cells;
      o.win[s] = w;
      if (out > 0) o.cell_cnt[w.cell_base + w.ncell] = out;
    }
    __syncthreads();
    if (tid == 0) base += all;
    __syncthreads();
  }
  if (tid == 0) {
    *o.total_cells = base;
    o.counters[C_CELLS] = (unsigned long long)base;
    o.counters[C_OOG] = (unsigned long long)oog;
    o.counters[C_NONFINITE] = (unsigned long long)nonfinite;
    o.counters[C_MASK_WORDS] = 0;
    o.counters[C_FALLBACK] = 0;
    for (int k = 0; k < 8; ++k) o.counters[C_EIGHTH + k] = 0;
  }
}

// Whether this workgroup is the last of the launch to get here (each of them
// calls this once, with all its threads): the words that every workgroup's
// thread 0 wrote before with share_store are then there for share_load. The
// order is this chip's, not the language's: agent-scope stores are written through
// the L2, the wait holds the ticket back until they are acknowledged, and
// agent-scope loads pass the caches by. A release on the ticket would also write
// the rest of the L2 back, which nothing here needs.
__device__ __forceinline__ bool last_block(int* ticket) {
  __shared__ int mine;
  if (threadIdx.x == 0) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);  // the stores have reached memory
    asm volatile("" ::: "memory");
    mine = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const bool last = mine == (int)gridDim.x - 1;
  if (last && threadIdx.x == 0) *ticket = 0;  // for the next launch
  return last;
}

// Scene of every particle and the cell bounding box of each scene's in-grid
// particles. Each block covers kBoundsSpan particles (kBoundsPer per thread,
// coalesced). A block whose particles all belong to one scene writes its
// box to bpart (8 ints: scene, min i j k, max i j k, and its out-of-grid and
// non-finite counts packed as o | f << 16); blocks that straddle
// scenes mark bpart -1 and update the scenes' boxes with atomics (per wave,
// per lane where a wave straddles). Same-address atomics from every block
// would serialize in L2, so the single-scene blocks are reduced per scene by
// k_scene_reduce (for one scene by scene_windows: with kWindows the last block
// to end makes the window, otherwise k_scene_windows).
//
// A particle's scene: the block's first and last particle are looked up once
// each, 64 offsets at a time; threads search between the two only where they
// differ. A binary search per particle, six dependent loads deep, took 22 us for
// 40,009 particles in 8 scenes and 40 us for 1.3M in 64.
constexpr int kBoundsBlock = 256, kBoundsPer = 4, kBoundsSpan = kBoundsBlock * kBoundsPer;

size_t bounds_part_ints(long long n) { return 8 * (size_t)((n + kBoundsSpan - 1) / kBoundsSpan + 1); }

template <bool kCellOrder, bool kWindows>
__global__ __launch_bounds__(kBoundsBlock) void k_scene_bounds(SortIn in, int n, GridDev g,
                                                               const int* __restrict__ off, int nscenes,
                                                               int* __restrict__ sid, int* __restrict__ minmax,
                                                               int* __restrict__ bpart, int* __restrict__ oog_flag,
                                                               WindowOut windows, int* __restrict__ ticket) {
  __shared__ int red[kBoundsBlock / 64][7];
  __shared__ int ends[2];
  const int base = blockIdx.x * kBoundsSpan;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int s_first = 0, s_last = 0;
  if (nscenes > 1) {
    if (wave < 2) {
      const int s = scene_of_wave(off, nscenes, wave == 0 ? base : min(n, base + kBoundsSpan) - 1);
      if (lane == 0) ends[wave] = s;
    }
    __syncthreads();
    s_first = ends[0];
    s_last = ends[1];
  }
  const bool one_scene = s_first == s_last;  // block-uniform
  int sq[kBoundsPer], cq[kBoundsPer][3];
  bool inq[kBoundsPer];
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
  int counts = 0;  // out-of-grid | non-finite << 16
#pragma unroll
  for (int q = 0; q < kBoundsPer; ++q) {
    const int i = base + q * kBoundsBlock + (int)threadIdx.x;
    int sc = -1, c[3] = {0, 0, 0};
    bool nonfinite = false, inside = false;
    if (i < n) {
      sc = one_scene ? s_first : s_first + scene_of(off + s_first, s_last - s_first + 1, i);
      sid[i] = sc;
      inside = grid_cell(g, in_pos<kCellOrder>(in, i), c[0], c[1], c[2], nonfinite);
      counts += (inside ? 0 : 1) + (nonfinite ? 1 << 16 : 0);
      if (!inside) oog_flag[kCellOrder ? in.id[i] : i] = 1;
    }
    sq[q] = sc;
    inq[q] = inside;
    for (int a = 0; a < 3; ++a) {
      cq[q][a] = c[a];
      if (inside) {
        lo[a] = min(lo[a], c[a]);
        hi[a] = max(hi[a], c[a]);
      }
    }
  }
  // every lane of the block is active (no early exit)
  for (int a = 0; a < 3; ++a) {
    lo[a] = wave_min_full(lo[a]);
    hi[a] = wave_max_full(hi[a]);
  }
  counts = wave_sum_full(counts);
  if (lane == 0) {
    for (int a = 0; a < 3; ++a) {
      red[wave][a] = lo[a];
      red[wave][3 + a] = hi[a];
    }
    red[wave][6] = counts;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int r[6] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN};
    int tot = 0;
    for (int w = 0; w < kBoundsBlock / 64; ++w) {
      for (int a = 0; a < 3; ++a) r[a] = min(r[a], red[w][a]);
      for (int a = 3; a < 6; ++a) r[a] = max(r[a], red[w][a]);
      tot += red[w][6];
    }
    int* bp = bpart + 8 * (size_t)blockIdx.x;
    if (kWindows) {
      for (int a = 0; a < 6; ++a) share_store(bp + 1 + a, r[a]);
      share_store(bp + 7, tot);
    } else {
      bp[0] = one_scene ? s_first : -1;
      for (int a = 0; a < 6; ++a) bp[1 + a] = r[a];
      bp[7] = tot;
    }
  }
  if (kWindows) {
    if (last_block(ticket)) scene_windows<kBoundsBlock / 64>(windows, [](const int* p) { return share_load(p); });
    return;
  }
  if (one_scene) return;  // block-uniform
  // a block that straddles scenes: a few scenes one after the other, one set of
  // atomics each (an atomic per wave and slot took 20 us where the scenes'
  // boundaries meet); many scenes per particle slot q, per wave where the wave's
  // particles share a scene, else per lane
  if (s_last - s_first < 8) {
    for (int s = s_first; s <= s_last; ++s) {
      int m[7] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN, 0};
#pragma unroll
      for (int q = 0; q < kBoundsPer; ++q) {
        if (sq[q] != s) continue;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          m[a] = min(m[a], inq[q] ? cq[q][a] : INT_MAX);
          m[3 + a] = max(m[3 + a], inq[q] ? cq[q][a] : INT_MIN);
        }
        m[6] += inq[q] ? 0 : 1;
      }
#pragma unroll
      for (int a = 0; a < 7; ++a) m[a] = a < 3 ? wave_min_full(m[a]) : (a < 6 ? wave_max_full(m[a]) : wave_sum_full(m[a]));
      __syncthreads();  // red is free
      if (lane == 0) {
#pragma unroll
        for (int a = 0; a < 7; ++a) red[wave][a] = m[a];
      }
      __syncthreads();
      if (threadIdx.x < 7) {
        const int a = threadIdx.x;
        int v = red[0][a];
        for (int w = 1; w < kBoundsBlock / 64; ++w)
          v = a < 3 ? min(v, red[w][a]) : (a < 6 ? max(v, red[w][a]) : v + red[w][a]);
        int* box = minmax + kBoxInts * (size_t)s + a;
        if (v != empty_box(a)) {
          if (a < 3)
            atomicMin(box, v);
          else if (a < 6)
            atomicMax(box, v);
          else
            atomicAdd(box, v);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < kBoundsPer; ++q) {
    const int i = base + q * kBoundsBlock + (int)threadIdx.x;
    const bool valid = i < n;
    const int s0 = __shfl(sq[q], 0);  // lane 0 is valid whenever any lane is
    if (__all(!valid || sq[q] == s0)) {
      int m[6];
      for (int a = 0; a < 3; ++a) {
        m[a] = wave_min_full(inq[q] ? cq[q][a] : INT_MAX);
        m[3 + a] = wave_max_full(inq[q] ? cq[q][a] : INT_MIN);
      }
      const int out = __popcll(__ballot(valid && !inq[q]));
      if (lane == 0 && s0 >= 0) {
        int* box = minmax + kBoxInts * (size_t)s0;
        if (m[3] >= m[0]) {
          for (int a = 0; a < 3; ++a) atomicMin(box + a, m[a]);
          for (int a = 3; a < 6; ++a) atomicMax(box + a, m[a]);
        }
        if (out) atomicAdd(box + 6, out);
      }
    } else if (valid) {
      int* box = minmax + kBoxInts * (size_t)sq[q];
      if (inq[q]) {
        for (int a = 0; a < 3; ++a) atomicMin(box + a, cq[q][a]);
        for (int a = 0; a < 3; ++a) atomicMax(box + 3 + a, cq[q][a]);
      } else {
        atomicAdd(box + 6, 1);
      }
    }
  }
}

// One block per scene: reduce the boxes of the single-scene blocks of the
// scene's particle range and merge them into the scene's box. Each entry is
// read as two 16-byte loads, four entries per thread in flight.
constexpr int kReduceBlock = 1024;

__device__ __forceinline__ void merge_box(int r[7], const int* __restrict__ bpart, int b, int s) {
  const int4 u = reinterpret_cast<const int4*>(bpart)[2 * (size_t)b];
  const int4 w = reinterpret_cast<const int4*>(bpart)[2 * (size_t)b + 1];
  if (u.x != s) return;
  r[0] = min(r[0], u.y);
  r[1] = min(r[1], u.z);
  r[2] = min(r[2], u.w);
  r[3] = max(r[3], w.x);
  r[4] = max(r[4], w.y);
  r[5] = max(r[5], w.z);
  r[6] += w.w & 0xffff;
}

__global__ __launch_bounds__(kReduceBlock) void k_scene_reduce(const int* __restrict__ off, int nscenes,
                                                               const int* __restrict__ bpart,
                                                               int* __restrict__ minmax) {
  __shared__ int red[kReduceBlock / 64][7];
  const int s = blockIdx.x;
  const int b0 = off[s] / kBoundsSpan;
  const int b1 = off[s + 1] > off[s] ? (off[s + 1] - 1) / kBoundsSpan + 1 : b0;
  int r[7] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN, 0};
  int b = b0 + (int)threadIdx.x;
  for (; b + 3 * kReduceBlock < b1; b += 4 * kReduceBlock) {
#pragma unroll
    for (int q = 0; q < 4; ++q) merge_box(r, bpart, b + q * kReduceBlock, s);
  }
  for (; b < b1; b += kReduceBlock) merge_box(r, bpart, b, s);
  // every lane of the block is active
  for (int a = 0; a < 3; ++a) r[a] = wave_min_full(r[a]);
  for (int a = 3; a < 6; ++a) r[a] = wave_max_full(r[a]);
  r[6] = wave_sum_full(r[6]);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0)
    for (int a = 0; a < 7; ++a) red[wave][a] = r[a];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kReduceBlock / 64; ++w) {
      for (int a = 0; a < 3; ++a) r[a] = min(r[a], red[w][a]);
      for (int a = 3; a < 6; ++a) r[a] = max(r[a], red[w][a]);
      r[6] += red[w][6];
    }
    // the only block that writes this scene's box now
    int* m = minmax + kBoxInts * (size_t)s;
    for (int a = 0; a < 3; ++a) m[a] = min(m[a], r[a]);
    for (int a = 3; a < 6; ++a) m[a] = max(m[a], r[a]);
    m[6] += r[6];
  }
}

__global__ __launch_bounds__(1024) void k_scene_windows(WindowOut o) {
  scene_windows<16>(o, [](const int* p) { return *p; });
}

// K_CalculateParticleNumber (GridHash.cu:78-87): key = compact cell or the
// scene's out-of-grid bucket (whose count the windows set); slot = arrival order
// inside a cell, -1 in a bucket.
template <bool kCellOrder>
__global__ __launch_bounds__(kBlock) void k_bin(SortIn in, int n, GridDev g,
                                                const int* __restrict__ sid, const SceneWin* __restrict__ win,
                                                int* __restrict__ key, int* __restrict__ slot,
                                                int* __restrict__ cell_cnt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int ci, cj, ck;
  bool nonfinite;
  const bool inside = grid_cell(g, in_pos<kCellOrder>(in, i), ci, cj, ck, nonfinite);
  const SceneWin w = win[sid[i]];
  int k = w.cell_base + w.ncell;
  if (inside) k = w.cell_base + (ci - w.lo[0]) + w.dim[0] * ((cj - w.lo[1]) + w.dim[1] * (ck - w.lo[2]));
  key[i] = k;
  const int lane = threadIdx.x & 63;
  int sl = 0;
  if (kCellOrder) {
    // Input in the previous step's cell order: in-grid lanes of one cell are
    // mostly adjacent. One atomic per run of equal keys, at the run's first
    // lane (a key split over several runs of the wave counts once per run);
    // out-of-grid lanes end runs and count below. Active lanes are the low
    // lanes of the wave.
    const int prev = __shfl_up(k, 1);
    const bool cut = !inside || lane == 0 || prev != k;
    const unsigned long long cuts = __ballot(cut), act = __ballot(true);
    const unsigned long long upto = (2ull << lane) - 1ull;  // lanes 0..lane
    const int hl = 63 - __clzll(cuts & upto);               // first lane of this run
    const unsigned long long after = cuts & ~upto;
    const int end = after ? __ffsll((long long)after) - 1 : 64 - __clzll(act);
    int base = 0;
    if (inside && cut) base = atomicAdd(&cell_cnt[k], end - lane);
    const int b = __shfl(base, hl);
    if (inside) sl = b + (lane - hl);
  } else if (inside) {
    sl = atomicAdd(&cell_cnt[k], 1);
  }
  slot[i] = inside ? sl : -1;
}

// K_ConstructHashTable (GridHash.cu:187-198): ids into their cell's slots. An
// out-of-grid particle's place in its bucket is the rank of its original index
// among the scene's out-of-grid particles (oog_pre, the scan of the bounds
// pass's flags), so a bucket is in original-index order at any size without
// atomics. Input in cell order: tid receives the original index beside each
// input index.
template <bool kCellOrder>
__global__ __launch_bounds__(kBlock) void k_scatter(const int* __restrict__ key, const int* __restrict__ slot,
                                                    const int* __restrict__ cell_start, int* __restrict__ tmp,
                                                    const int* __restrict__ id, int* __restrict__ tid, int n,
                                                    const int* __restrict__ sid, const int* __restrict__ scene_off,
                                                    const int* __restrict__ oog_pre) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int sl = slot[i];
  if (sl < 0) sl = oog_pre[kCellOrder ? id[i] : i] - oog_pre[scene_off ? min(scene_off[sid[i]], n) : 0];
  const int p = cell_start[key[i]] + sl;
  tmp[p] = i;
  if (kCellOrder) tid[p] = id[i];
}

// Final position inside the cell = rank of the particle id among the cell's
// ids (deterministic order, independent of atomic arrival). Cells holding more
// than kRankMax particles keep arrival order (still a valid cell sort); a
// scene's out-of-grid bucket is in original-index order already (k_bin). One
// thread per slot of the scattered order: slot t's particle lands inside its
// own cell's range, so the sorted arrays are written nearly in order and only
// the inputs are read scattered.
// The integrator (ParticleIntegrator.cu:60-70,103-112, force zeroed by begin)
// is fused here: x^n goes to xn (the neighbor sets are built on it,
// PositionBasedFluidModel.cpp:93-94), the integrated state to x0 / vs.
constexpr int kRankMax = 1024;

template <bool kCellOrder>
__global__ __launch_bounds__(kBlock) void k_reorder(const int* __restrict__ key, const int* __restrict__ cell_start,
                                                    const int* __restrict__ tmp, const int* __restrict__ tid,
                                                    const int* __restrict__ sid, SortIn in, int n,
                                                    int* __restrict__ perm, int* __restrict__ ssid,
                                                    float4* __restrict__ xn,
                                                    float4* __restrict__ x0, float4* __restrict__ vs, PhysConst pc,
                                                    int integrate, float* __restrict__ xc, int xc_stride,
                                                    int* __restrict__ oog_rcnt, const SceneWin* __restrict__ win) {
#pragma clang fp contract(off)
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t == 0) x0[n] = make_float4(kPadCoord, kPadCoord, kPadCoord, 0.0f);  // the padding particle
  if (t >= n) return;
  const int i = tmp[t];  // input index
  const int id = kCellOrder ? tid[t] : i;  // original index
  const int k = key[i];
  const int a = cell_start[k], b = cell_start[k + 1];
  int s = t;
  const SceneWin w = win[sid[i]];
  if (k != w.cell_base + w.ncell && b - a <= kRankMax) {
    int rank = 0;
    const int* ids = kCellOrder ? tid : tmp;
    int u = a;
    for (; u + 4 <= b; u += 4) {  // four loads in flight
      const int c0 = ids[u], c1 = ids[u + 1], c2 = ids[u + 2], c3 = ids[u + 3];
      rank += (c0 < id) + (c1 < id) + (c2 < id) + (c3 < id);
    }
    for (; u < b; ++u) rank += ids[u] < id;
    s = a + rank;
  }
  perm[s] = id;
  ssid[s] = sid[i];
  oog_rcnt[s] = 0;
  const float3 p = in_pos<kCellOrder>(in, i);
  const float px = p.x, py = p.y, pz = p.z;
  xn[s] = make_float4(px, py, pz, 0.0f);
  xc[s] = px;
  xc[xc_stride + s] = py;
  xc[2 * (size_t)xc_stride + s] = pz;
  if (integrate) {
    const float3 v = in_vel<kCellOrder>(in, i);
    const float vx = v.x + pc.gdt[0];
    const float vy = v.y + pc.gdt[1];
    const float vz = v.z + pc.gdt[2];
    x0[s] = make_float4(px + vx * pc.dt, py + vy * pc.dt, pz + vz * pc.dt, 0.0f);
    vs[s] = make_float4(vx, vy, vz, 0.0f);
  } else {
    x0[s] = make_float4(px, py, pz, 0.0f);
  }
}

// ---------------------------------------------------------------------------
// The whole sort of a one-scene search of at most kSortOneMax particles in one
// workgroup: nine launches of 1.5 to 5 us each, most of it launch and memory
// latency, become one (and one that returns at once unless the window is
// large). The in-grid particles go to LDS buckets of consecutive cells, and a
// particle's place is its bucket's start plus the number of its bucket's
// particles before it by (cell, original index): the order of the sort above,
// for cells of any size. The out-of-grid particles, of which there may be
// thousands, follow in the order of their original indices, ranked in a bit set.
// The starts of the window's cells are found in the sorted keys.
constexpr int kSortOneMax = 4096, kSortOneBlock = 1024, kSortOnePer = kSortOneMax / kSortOneBlock;
constexpr int kSortBuckets = 8192, kBucketsPer = kSortBuckets / kSortOneBlock;
constexpr int kSortIdBits = 12, kSortIdWords = kSortOneMax / 32;
static_assert(1 << kSortIdBits == kSortOneMax, "an index and its cell inside a bucket share a word");

// First position of keys[lo..hi) whose key is at least c.
__device__ __forceinline__ int lower_key(const int* keys, int lo, int hi, int c) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (keys[mid] < c)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

template <bool kCellOrder>
__global__ __launch_bounds__(kSortOneBlock) void k_sort_one(SortIn in, int n, GridDev g, SceneWin* __restrict__ win,
                                                            int* __restrict__ total_cells,
                                                            unsigned long long* __restrict__ counters,
                                                            int* __restrict__ cell_start, int* __restrict__ keys,
                                                            int* __restrict__ perm, int* __restrict__ ssid,
                                                            float4* __restrict__ xn, float4* __restrict__ x0,
                                                            float4* __restrict__ vs, PhysConst pc, int integrate,
                                                            float* __restrict__ xc, int xc_stride,
                                                            int* __restrict__ oog_rcnt) {
#pragma clang fp contract(off)
  __shared__ int start[kSortBuckets + 1];
  // entries in bucket order: the cell, the cell inside the bucket with the
  // original index, the input index
  __shared__ int skey[kSortOneMax], src[kSortOneMax];
  __shared__ unsigned sord[kSortOneMax];
  __shared__ unsigned out_bit[kSortIdWords];  // out-of-grid original indices
  __shared__ int out_pre[kSortIdWords], out_half;
  __shared__ int red[kSortOneBlock / 64][8];
  __shared__ SceneWin sw;
  __shared__ int nout;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int b = tid; b <= kSortBuckets; b += kSortOneBlock) start[b] = 0;
  if (tid < kSortIdWords) out_bit[tid] = 0;
  // cells and their box
  int c[kSortOnePer][3];
  bool inside[kSortOnePer];
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
  int counts = 0;  // out-of-grid | non-finite << 16
#pragma unroll
  for (int q = 0; q < kSortOnePer; ++q) {
    const int i = tid + q * kSortOneBlock;
    bool nonfinite = false;
    inside[q] = false;
    if (i < n) {
      inside[q] = grid_cell(g, in_pos<kCellOrder>(in, i), c[q][0], c[q][1], c[q][2], nonfinite);
      counts += (inside[q] ? 0 : 1) + (nonfinite ? 1 << 16 : 0);
    }
    if (inside[q]) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        lo[a] = min(lo[a], c[q][a]);
        hi[a] = max(hi[a], c[q][a]);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    lo[a] = wave_min_full(lo[a]);
    hi[a] = wave_max_full(hi[a]);
  }
  counts = wave_sum_full(counts);
  if (lane == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      red[wave][a] = lo[a];
      red[wave][3 + a] = hi[a];
    }
    red[wave][6] = counts & 0xffff;
    red[wave][7] = counts >> 16;
  }
  __syncthreads();
  if (wave == 0) {
    int r[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int id = k < 3 ? INT_MAX : (k < 6 ? INT_MIN : 0);
      const int v = lane < kSortOneBlock / 64 ? red[lane][k] : id;
      r[k] = k < 3 ? wave_min_full(v) : (k < 6 ? wave_max_full(v) : wave_sum_full(v));
    }
    if (lane == 0) {
      SceneWin w{};
      const bool any = r[3] >= r[0];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        w.lo[a] = any ? r[a] : 0;
        w.dim[a] = any ? r[3 + a] - r[a] + 1 : 0;
      }
      w.cell_base = 0;
      w.ncell = w.dim[0] * w.dim[1] * w.dim[2];
      sw = w;
      nout = r[6];
      win[0] = w;
      *total_cells = w.ncell + 1;
      counters[C_CELLS] = (unsigned long long)w.ncell + 1;
      counters[C_OOG] = (unsigned long long)r[6];
      counters[C_NONFINITE] = (unsigned long long)r[7];
      counters[C_MASK_WORDS] = 0;
      counters[C_FALLBACK] = 0;
    }
  }
  __syncthreads();
  const SceneWin w = sw;
  const int nin = n - nout;  // in-grid particles
  // buckets of 2^shift consecutive cells
  const int shift = max(0, 32 - __clz(w.ncell) - 13);
  int key[kSortOnePer], slot[kSortOnePer];
#pragma unroll
  for (int q = 0; q < kSortOnePer; ++q) {
    key[q] = inside[q] ? window_cell(w, c[q][0], c[q][1], c[q][2]) : w.ncell;
    slot[q] = inside[q] ? atomicAdd(&start[key[q] >> shift], 1) : 0;
  }
  if (nout > 0) {
#pragma unroll
    for (int q = 0; q < kSortOnePer; ++q) {
      const int i = tid + q * kSortOneBlock;
      if (i < n && !inside[q]) {
        const int id = kCellOrder ? in.id[i] : i;
        atomicOr(&out_bit[id >> 5], 1u << (id & 31));
      }
    }
  }
  __syncthreads();
  if (nout > 0 && tid < kSortIdWords) {
    const int v = __popc(out_bit[tid]);
    const int incl = wave_inclusive_scan(v);
    out_pre[tid] = incl - v;
    if (tid == 63) out_half = incl;
  }
  {  // exclusive scan of the bucket counts, kBucketsPer per thread
    int v[kBucketsPer], sum = 0;
#pragma unroll
    for (int k = 0; k < kBucketsPer; ++k) {
      v[k] = start[tid * kBucketsPer + k];
      sum += v[k];
    }
    int total;
    int e = block_scan4(sum, 0, 0, 0, total);
#pragma unroll
    for (int k = 0; k < kBucketsPer; ++k) {
      start[tid * kBucketsPer + k] = e;
      e += v[k];
    }
    if (tid == 0) start[kSortBuckets] = nin;
  }
  __syncthreads();
  // input i with original index id and cell k to its sorted place s
  auto put = [&](int s, int i, int id, int k) {
    perm[s] = id;
    ssid[s] = 0;
    oog_rcnt[s] = 0;
    keys[s] = k;
    const float3 p = in_pos<kCellOrder>(in, i);
    xn[s] = make_float4(p.x, p.y, p.z, 0.0f);
    xc[s] = p.x;
    xc[xc_stride + s] = p.y;
    xc[2 * (size_t)xc_stride + s] = p.z;
    if (integrate) {
      const float3 v = in_vel<kCellOrder>(in, i);
      const float vx = v.x + pc.gdt[0];
      const float vy = v.y + pc.gdt[1];
      const float vz = v.z + pc.gdt[2];
      x0[s] = make_float4(p.x + vx * pc.dt, p.y + vy * pc.dt, p.z + vz * pc.dt, 0.0f);
      vs[s] = make_float4(vx, vy, vz, 0.0f);
    } else {
      x0[s] = make_float4(p.x, p.y, p.z, 0.0f);
    }
  };
#pragma unroll
  for (int q = 0; q < kSortOnePer; ++q) {
    const int i = tid + q * kSortOneBlock;
    if (i >= n) continue;
    const int id = kCellOrder ? in.id[i] : i;
    if (inside[q]) {
      const int p = start[key[q] >> shift] + slot[q];
      skey[p] = key[q];
      sord[p] = (unsigned)(key[q] & ((1 << shift) - 1)) << kSortIdBits | (unsigned)id;
      src[p] = i;
    } else {
      const int at = id >> 5;
      put(nin + out_pre[at] + (at >= 64 ? out_half : 0) + __popc(out_bit[at] & ((1u << (id & 31)) - 1u)), i, id,
          w.ncell);
    }
  }
  __syncthreads();
  // the place of each in-grid entry
#pragma unroll
  for (int q = 0; q < kSortOnePer; ++q) {
    const int t = tid + q * kSortOneBlock;
    if (t >= nin) continue;
    const int k = skey[t], b = k >> shift;
    const unsigned o = sord[t];
    const int a = start[b], e = start[b + 1];
    int rank = 0;
#pragma unroll 4
    for (int u = a; u < e; ++u) rank += sord[u] < o ? 1 : 0;
    put(a + rank, src[t], (int)(o & (kSortOneMax - 1)), k);
  }
  if (tid == 0) x0[n] = make_float4(kPadCoord, kPadCoord, kPadCoord, 0.0f);  // the padding particle
  if (w.ncell >= kSortBuckets) return;  // k_cell_starts
  // a bucket is one cell: its start is the cell's
  for (int b = tid; b <= w.ncell + 1; b += kSortOneBlock) cell_start[b] = b <= w.ncell ? start[b] : n;
}

// Starts of the cells of a window too large for k_sort_one's buckets, from the
// sorted keys in LDS. The window is as large as the particles are spread (a stray
// one is enough), up to the whole grid: a workgroup narrows the keys down to its
// contiguous range of cells first, so that most cells, which are empty, cost
// their share of a 16-byte store.
constexpr int kStartsBlock = 256, kStartsBlocks = 512;

__global__ __launch_bounds__(kStartsBlock) void k_cell_starts(const SceneWin* __restrict__ win,
                                                              const int* __restrict__ keys, int n,
                                                              int* __restrict__ cell_start) {
  const int ncell = win[0].ncell;
  if (ncell < kSortBuckets) return;
  __shared__ int key[kSortOneMax];
  for (int t = threadIdx.x; t < n; t += kStartsBlock) key[t] = keys[t];
  __syncthreads();
  const int cells = ncell + 2;  // one past the out-of-grid bucket: n
  const int per = (cells + kStartsBlocks * 4 - 1) / (kStartsBlocks * 4) * 4;
  const int c0 = blockIdx.x * per, c1 = min(c0 + per, cells);
  if (c0 >= c1) return;
  const int lo = lower_key(key, 0, n, c0), hi = lower_key(key, lo, n, c1);
  for (int c = c0 + 4 * (int)threadIdx.x; c < c1; c += 4 * kStartsBlock) {
    int4 s;
    s.x = lower_key(key, lo, hi, c);
    s.w = lower_key(key, s.x, hi, c + 3);
    s.y = lower_key(key, s.x, s.w, c + 1);
    s.z = lower_key(key, s.y, s.w, c + 2);
    if (c + 4 <= c1) {
      *reinterpret_cast<int4*>(cell_start + c) = s;
    } else {
      cell_start[c] = s.x;
      if (c + 1 < c1) cell_start[c + 1] = s.y;
      if (c + 2 < c1) cell_start[c + 2] = s.z;
    }
  }
}

template <bool kCellOrder>
void sort_one(const SortBufs& sb, const GridDev& g, const SortIn& in, int n, float4* xn, float4* x0, float4* vs,
              const PhysConst* integrate, unsigned long long* counters, hipStream_t st) {
  PhysConst pc{};
  if (integrate) pc = *integrate;
  k_sort_one<kCellOrder><<<1, kSortOneBlock, 0, st>>>(in, n, g, sb.win, sb.total_cells, counters, sb.cell_start,
                                                      sb.key, sb.perm, sb.ssid, xn, x0, vs, pc, integrate ? 1 : 0,
                                                      sb.xc, sb.xc_stride, sb.oog_rcnt);
  k_cell_starts<<<kStartsBlocks, kStartsBlock, 0, st>>>(sb.win, sb.key, n, sb.cell_start);
}

// Bounds blocks of a launch whose last one makes the window: their tickets are
// same-address atomics, about 9 ns each (256 blocks: 262,144 particles).
constexpr int kTicketBlocks = 256;

template <bool kCellOrder>
void sort_in(const SortBufs& sb, const GridDev& g, const SortIn& in, int n, float4* xn, float4* x0, float4* vs,
             const PhysConst* integrate, unsigned long long* counters, hipStream_t st) {
  const int nb = (n + kBlock - 1) / kBlock;
  const int nbounds = (n + kBoundsSpan - 1) / kBoundsSpan;
  const WindowOut windows{sb.scene_minmax, sb.nscenes, sb.win, sb.total_cells, sb.bpart, nbounds, counters, sb.cell_cnt};
  if (sb.nscenes == 1 && nbounds <= kTicketBlocks) {
    k_scene_bounds<kCellOrder, true><<<nbounds, kBoundsBlock, 0, st>>>(in, n, g, sb.scene_off, 1, sb.sid,
                                                                       sb.scene_minmax, sb.bpart, sb.oog_flag,
                                                                       windows, sb.ticket);
  } else {
    k_scene_bounds<kCellOrder, false><<<nbounds, kBoundsBlock, 0, st>>>(in, n, g, sb.scene_off, sb.nscenes, sb.sid,
                                                                        sb.scene_minmax, sb.bpart, sb.oog_flag,
                                                                        windows, nullptr);
    if (sb.nscenes > 1)
      k_scene_reduce<<<sb.nscenes, kReduceBlock, 0, st>>>(sb.scene_off, sb.nscenes, sb.bpart, sb.scene_minmax);
    k_scene_windows<<<1, 1024, 0, st>>>(windows);
  }
  k_bin<kCellOrder><<<nb, kBlock, 0, st>>>(in, n, g, sb.sid, sb.win, sb.key, sb.slot, sb.cell_cnt);
  // the cell counts, and the out-of-grid ranks by original index (only when the
  // bounds pass found any; the last scene offset is n)
  const ScanJob cells{sb.cell_cnt, sb.cell_start, sb.total_cells, INT_MAX, sb.scan_part, nullptr};
  const ScanJob flags{sb.oog_flag, sb.oog_pre, sb.scene_off ? sb.scene_off + sb.nscenes : nullptr, n,
                      sb.scan_part + kScanDevBlocks, counters + C_OOG};
  k_scan_dev_reduce<<<dim3(kScanDevBlocks, 2), 1024, 0, st>>>(cells, flags);
  k_scan_dev_down<<<dim3(kScanDevBlocks, 2), 1024, 0, st>>>(cells, flags);
  k_scatter<kCellOrder><<<nb, kBlock, 0, st>>>(sb.key, sb.slot, sb.cell_start, sb.tmp, in.id, sb.tid, n, sb.sid,
                                               sb.scene_off, sb.oog_pre);
  PhysConst pc{};
  if (integrate) pc = *integrate;
  k_reorder<kCellOrder><<<nb, kBlock, 0, st>>>(sb.key, sb.cell_start, sb.tmp, sb.tid, sb.sid, in, n, sb.perm,
                                               sb.ssid, xn, x0, vs, pc, integrate ? 1 : 0, sb.xc, sb.xc_stride,
                                               sb.oog_rcnt, sb.win);
}

void launch_sort(const SortBufs& sb, const GridDev& g, const SortIn& in, int n, float4* xn, float4* x0, float4* vs,
                 const PhysConst* integrate, unsigned long long* counters, hipStream_t st) {
  if (sb.nscenes == 1 && n <= kSortOneMax) {
    if (in.x4)
      sort_one<true>(sb, g, in, n, xn, x0, vs, integrate, counters, st);
    else
      sort_one<false>(sb, g, in, n, xn, x0, vs, integrate, counters, st);
  } else if (in.x4)
    sort_in<true>(sb, g, in, n, xn, x0, vs, integrate, counters, st);
  else
    sort_in<false>(sb, g, in, n, xn, x0, vs, integrate, counters, st);
}

// Copy of cell_start[0..total] (the device-side cell count of the last sort).
__global__ void k_copy_cells(const int* __restrict__ src, int* __restrict__ dst, const int* __restrict__ total_cells) {
  const int total = *total_cells + 1;
  const int stride = gridDim.x * blockDim.x;
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < total; c += stride) dst[c] = src[c];
}

void launch_copy_cells(const int* src, int* dst, const int* total_cells, long long cap, hipStream_t st) {
  const int blocks = (int)std::min<long long>((cap + 2 + kBlock - 1) / kBlock, 1024);
  k_copy_cells<<<blocks, kBlock, 0, st>>>(src, dst, total_cells);
}

__global__ void k_set_offsets(int* off, int n) {
  if (threadIdx.x == 0) {
    off[0] = 0;
    off[1] = n;
  }
}

void launch_set_offsets(int* off, int n, hipStream_t st) { k_set_offsets<<<1, 64, 0, st>>>(off, n); }

__global__ __launch_bounds__(kBlock) void k_write_back(const float4* __restrict__ xs, const float4* __restrict__ vs,
                                                       const int* __restrict__ perm, int n, float* __restrict__ x_out,
                                                       float* __restrict__ v_out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const size_t i = (size_t)perm[s];
  const float4 a = xs[s], b = vs[s];
  x_out[3 * i] = a.x;
  x_out[3 * i + 1] = a.y;
  x_out[3 * i + 2] = a.z;
  v_out[3 * i] = b.x;
  v_out[3 * i + 1] = b.y;
  v_out[3 * i + 2] = b.z;
}

void launch_write_back(const float4* xs, const float4* vs, const int* perm, int n, float* x_out, float* v_out,
                       hipStream_t st) {
  k_write_back<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(xs, vs, perm, n, x_out, v_out);
}

// inv[perm[s]] = s (the CSR export needs the sorted slot of every particle).
__global__ __launch_bounds__(kBlock) void k_invert(const int* __restrict__ perm, int* __restrict__ inv, int n) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) inv[perm[s]] = s;
}

void launch_invert(const int* perm, int* inv, int n, hipStream_t st) {
  if (n > 0) k_invert<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(perm, inv, n);
}

__global__ __launch_bounds__(kBlock) void k_csr_count(const int* __restrict__ nbr_cnt, const int* __restrict__ inv,
                                                      int n, int* __restrict__ cnt_orig) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cnt_orig[i] = nbr_cnt[inv[i]];
}

void launch_csr_count(const int* nbr_cnt, const int* inv, int n, int* cnt_orig, hipStream_t st) {
  k_csr_count<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(nbr_cnt, inv, n, cnt_orig);
}

}  // namespace pbf
