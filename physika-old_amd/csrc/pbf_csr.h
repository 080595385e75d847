// Traversal of a caller's CSR list by the module-granular passes.
//
// Four lanes share a row (one where rows are short: row_lanes): per step they read sixteen consecutive elements (one
// 16-byte load per lane), so a wave covers sixteen rows and a launch has four
// times the waves of a thread per row, whose 64 rows each touch a line of their
// own with every load. Measured at 262,144 particles (18.9M listed pairs):
// density and lambda 393 -> 37 us per pass; viscosity at 131,072 particles 94 ->
// 33 us. Eight lanes per row, one element per load each, took 39 us (33 us for
// the viscosity).
#pragma once
#include "pbf_device.h"

namespace pbf {

constexpr int kRowLanes = 4;
constexpr int kRowUnroll = 4;  // consecutive elements of a lane

// Lanes per row of a pass over a list: one where the rows have kShortRows elements
// or fewer in the mean (a spray, a list cut short), whose four lanes would be a
// wave's worth of reading for one lane's work. One and four lanes at 262,144 rows,
// five iterations, us: 7 elements a row, both ways, 109 and 145 (viscosity 70 and 85),
// 8 one way, 1,343 and 1,299; at 1,000,000 rows viscosity over 1 element a row 94 and
// 151, over 8 208 and 212, over 12 288 and 250, the constraint over 7 239 and 335.
constexpr int kShortRows = 7;
inline int row_lanes(const Csr& nb) {
  return (long long)nb.nelems <= kShortRows * (long long)nb.n ? 1 : kRowLanes;
}

// kL: lanes per row.
template <int kL> struct CsrRow {
  int i;     // the row (n or more: none)
  int lane;  // 0..kL-1
};

// The row of this thread in a launch over the rows from `first` on; blocks of
// neighboring rows run on one XCD.
template <int kL, int kThreads = kBlock>
__device__ __forceinline__ CsrRow<kL> csr_row(const Csr& nb, int first = 0) {
  const long long g = (long long)xcd_block(blockIdx.x, gridDim.x) * kThreads + threadIdx.x;
  const long long i = first + g / kL;
  return CsrRow<kL>{i < nb.n ? (int)i : nb.n, (int)(g % kL)};
}

// Blocks of a launch over `rows` rows, at most kRowsPerLaunch (a grid holds
// fewer than 2^32 threads).
constexpr int kRowsPerLaunch = 1 << 28;
inline int csr_blocks(int rows, int lanes, int block = kBlock) {
  return (int)(((long long)rows * lanes + block - 1) / block);
}

typedef int i4u __attribute__((ext_vector_type(4), aligned(4)));

// body(u, j, gather(j)) for the up to kRowUnroll elements u of the lane in each
// step of sixteen, then step(); before the last step, which may reach past the
// row's end, clear(). The four lanes of a row run the same steps. The address
// unit takes a gather's lanes at 32 cycles per 64 and is what these passes wait
// for (87% busy), so the last step leaves the lanes past the row's end out (an
// 81-neighbor row would otherwise gather 96), its elements come with one load,
// and the next step's elements are on their way while this step's neighbors are
// gathered. Against a last step that repeats the row's last element: five
// iterations on 262,144 rows 373 -> 357 us.
template <int kL, class GatherFn, class Body, class Clear, class Step>
__device__ __forceinline__ void csr_each(const Csr& nb, const CsrRow<kL>& r, GatherFn&& gather, Body&& body,
                                         Clear&& clear, Step&& step) {
  constexpr int kStep = kL * kRowUnroll;
  const int b = nb.begin(r.i);
  const unsigned cnt = (unsigned)max(nb.end(r.i) - b, 0);
  if (cnt == 0) return;
  const int* __restrict__ e = nb.elems + b;
  const unsigned at = kRowUnroll * r.lane, full = cnt & ~(kStep - 1u);
  // the last step's elements: a load may reach into the next row, not past the list
  const unsigned tail = full + at;
  i4u jt = {0, 0, 0, 0};
  if (tail < cnt) {
    if ((unsigned)b + tail + kRowUnroll <= (unsigned)nb.nelems) {
      jt = *reinterpret_cast<const i4u*>(e + tail);
    } else {
#pragma unroll
      for (int u = 0; u < kRowUnroll; ++u) jt[u] = e[min(tail + u, cnt - 1)];
    }
  }
  if (full > 0) {
    i4u j = *reinterpret_cast<const i4u*>(e + at);
    for (unsigned t0 = 0; t0 < full; t0 += kStep) {
      decltype(gather(0)) q[kRowUnroll];
#pragma unroll
      for (int u = 0; u < kRowUnroll; ++u) q[u] = gather(j[u]);
      const i4u next = *reinterpret_cast<const i4u*>(e + (t0 + kStep < full ? t0 + kStep + at : at));
      asm volatile("" ::: "memory");  // keep the loads above in this step
#pragma unroll
      for (int u = 0; u < kRowUnroll; ++u) body(u, (int)j[u], q[u]);
      step();
      j = next;
    }
  }
  if (full < cnt) {
    clear();
    decltype(gather(0)) q[kRowUnroll];
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u)
      if (tail + u < cnt) q[u] = gather(jt[u]);
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u)
      if (tail + u < cnt) body(u, (int)jt[u], q[u]);
    step();
  }
}

// Sum over the lanes of a row, in every one of them.
template <int kL>
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
  for (int d = 1; d < kL; d <<= 1) v += __shfl_xor(v, d);
  return v;
}

__device__ __forceinline__ void row_clear(float (&t)[kRowUnroll]) {
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) t[u] = 0.0f;
}

// v of lane kLane of the row (a quad of the wave).
template <int kL, int kLane>
__device__ __forceinline__ float row_lane(float v) {
  if constexpr (kL == 1) return v;
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kLane * 0x55, 0xf, 0xf, true));
}

// acc + sum of t^3 over the step's elements, added one by one in the row's
// order on every lane: lambda is a small difference of this sum and the rest
// density, and the order of a thread per row keeps its rounding.
template <int kL, int kLane>
__device__ __forceinline__ float row_cubes_of(float acc, const float (&t)[kRowUnroll]) {
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) {
    const float tu = row_lane<kL, kLane>(t[u]);
    acc = fmaf(tu * tu, tu, acc);
  }
  return acc;
}
template <int kL>
__device__ __forceinline__ float row_cubes(float acc, const float (&t)[kRowUnroll]) {
  static_assert(kL == 1 || kL == 4, "one lane or a quad");
  acc = row_cubes_of<kL, 0>(acc, t);
  if constexpr (kL == 1) return acc;
  acc = row_cubes_of<kL, 1>(acc, t);
  acc = row_cubes_of<kL, 2>(acc, t);
  return row_cubes_of<kL, 3>(acc, t);
}

}  // namespace pbf
