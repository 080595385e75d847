// Traversal of a caller's CSR list by the module-granular passes.
//
// Four lanes share a row: per step they read sixteen consecutive elements (one
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
constexpr int kRowStep = kRowLanes * kRowUnroll;

struct CsrRow {
  int i;     // the row (n or more: none)
  int lane;  // 0..kRowLanes-1
};

// The row of this thread in a launch over the rows from `first` on; blocks of
// neighboring rows run on one XCD.
__device__ __forceinline__ CsrRow csr_row(const Csr& nb, int first = 0) {
  const long long g = (long long)xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const long long i = first + g / kRowLanes;
  return CsrRow{i < nb.n ? (int)i : nb.n, (int)(g % kRowLanes)};
}

// Blocks of a launch over `rows` rows, at most kRowsPerLaunch (a grid holds
// fewer than 2^32 threads).
constexpr int kRowsPerLaunch = 1 << 28;
inline int csr_blocks(int rows) { return (int)(((long long)rows * kRowLanes + kBlock - 1) / kBlock); }

typedef int i4u __attribute__((ext_vector_type(4), aligned(4)));

// The lane's elements t .. t + 3 of a row of cnt; past the row's end its last.
__device__ __forceinline__ i4u row_elements(const int* __restrict__ e, unsigned t, unsigned cnt) {
  if (t + kRowUnroll <= cnt) return *reinterpret_cast<const i4u*>(e + t);
  i4u j;
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) j[u] = e[min(t + u, cnt - 1)];
  return j;
}

// body(u, j, gather(j), on) for the kRowUnroll elements u of the lane in each
// step of sixteen, then step(). The last step may reach past the row's end:
// those elements repeat the row's last one with on false, and a body adds
// nothing for them. The four lanes of a row run the same steps. The next step's
// elements are on their way while this step's neighbors are gathered.
template <class GatherFn, class Body, class Step>
__device__ __forceinline__ void csr_each(const Csr& nb, const CsrRow& r, GatherFn&& gather, Body&& body,
                                         Step&& step) {
  const int b = nb.begin(r.i);
  const unsigned cnt = (unsigned)max(nb.end(r.i) - b, 0);
  if (cnt == 0) return;
  const int* __restrict__ e = nb.elems + b;
  i4u j = row_elements(e, kRowUnroll * r.lane, cnt);
  for (unsigned t0 = 0; t0 < cnt; t0 += kRowStep) {
    const unsigned t = t0 + kRowUnroll * r.lane;
    decltype(gather(0)) q[kRowUnroll];
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) q[u] = gather(j[u]);
    const i4u next = t0 + kRowStep < cnt ? row_elements(e, t + kRowStep, cnt) : j;
    asm volatile("" ::: "memory");  // keep the loads above in this step
#pragma unroll
    for (int u = 0; u < kRowUnroll; ++u) body(u, (int)j[u], q[u], t + u < cnt);
    step();
    j = next;
  }
}

// Sum over the lanes of a row, in every one of them.
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
  for (int d = 1; d < kRowLanes; d <<= 1) v += __shfl_xor(v, d);
  return v;
}

// v of lane kLane of the row (a quad of the wave).
template <int kLane>
__device__ __forceinline__ float row_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kLane * 0x55, 0xf, 0xf, true));
}

// acc + sum of t^3 over the step's elements, added one by one in the row's
// order on every lane: lambda is a small difference of this sum and the rest
// density, and the order of a thread per row keeps its rounding.
template <int kLane>
__device__ __forceinline__ float row_cubes_of(float acc, const float (&t)[kRowUnroll]) {
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) {
    const float tu = row_lane<kLane>(t[u]);
    acc = fmaf(tu * tu, tu, acc);
  }
  return acc;
}
__device__ __forceinline__ float row_cubes(float acc, const float (&t)[kRowUnroll]) {
  acc = row_cubes_of<0>(acc, t);
  acc = row_cubes_of<1>(acc, t);
  acc = row_cubes_of<2>(acc, t);
  return row_cubes_of<3>(acc, t);
}

}  // namespace pbf
