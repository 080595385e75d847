// Module-granular kernels: the reference modules' passes over a caller CSR
// list, in original particle order (ParticleIntegrator, SummationDensity,
// DensityPBD with its pairwise atomic scatter).
#include <algorithm>

#include "pbf_csr.h"

namespace pbf {

// ParticleIntegrator::integrate: K_UpdateVelocity then K_UpdatePosition
// (ParticleIntegrator.cu:60-70,103-112), each multiply and add rounded
// separately as the source writes them.
__global__ __launch_bounds__(kBlock) void k_integrate(float* __restrict__ x, float* __restrict__ v,
                                                      const float* __restrict__ f, int n, PhysConst pc) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t b = 3 * (size_t)i;
  float vx, vy, vz;
  if (f) {
    vx = v[b] + (f[b] + pc.g[0]) * pc.dt;
    vy = v[b + 1] + (f[b + 1] + pc.g[1]) * pc.dt;
    vz = v[b + 2] + (f[b + 2] + pc.g[2]) * pc.dt;
  } else {
    vx = v[b] + pc.gdt[0];
    vy = v[b + 1] + pc.gdt[1];
    vz = v[b + 2] + pc.gdt[2];
  }
  v[b] = vx;
  v[b + 1] = vy;
  v[b + 2] = vz;
  x[b] = x[b] + vx * pc.dt;
  x[b + 1] = x[b + 1] + vy * pc.dt;
  x[b + 2] = x[b + 2] + vz * pc.dt;
}

void launch_integrate(float* x, float* v, const float* f, int n, const PhysConst& pc, hipStream_t st) {
  k_integrate<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(x, v, f, n, pc);
}

// ---------------------------------------------------------------------------
// Passes over a caller CSR list.

// A neighbor's position with its inverse mass (1 without masses).
struct MassPos {
  float4 x;
  float m;
};

// DP_UpdateVelocity (DensityPBD.cu:368-378) of particle i with x_old = the
// caller's x, then x := the constrained position p.
__device__ __forceinline__ void csr_finish(int i, float4 p, float* __restrict__ x, float* __restrict__ v, float dt) {
  const size_t b = 3 * (size_t)i;
  v[b] += (p.x - x[b]) / dt;
  v[b + 1] += (p.y - x[b + 1]) / dt;
  v[b + 2] += (p.z - x[b + 2]) / dt;
  x[b] = p.x;
  x[b + 1] = p.y;
  x[b + 2] = p.z;
}

// K_ComputeDensity (SummationDensity.cu:13-36) over a CSR list.
template <int kL>
__global__ __launch_bounds__(kBlock) void k_csr_density(const float* __restrict__ x, Csr nb,
                                                        float* __restrict__ rho, PhysConst pc, int first) {
  const CsrRow<kL> row = csr_row<kL>(nb, first);
  if (row.i >= nb.n) return;
  const float4 xi = load3(x, row.i);
  float acc = 0.f, t[kRowUnroll];
  csr_each(
      nb, row, [&](int j) { return load3(x, j); },
      [&](int u, int, float4 xj) { t[u] = pair_geom(xi, xj, pc.inv_h).t; },
      [&] { row_clear(t); }, [&] { acc = row_cubes<kL>(acc, t); });
  if (row.lane == 0) rho[row.i] = acc * pc.cW;
}

void launch_csr_density(const float* x, const Csr& nb, float* rho, const PhysConst& pc, hipStream_t st) {
  for (long long first = 0; first < nb.n; first += kRowsPerLaunch) {
    const int rows = (int)std::min<long long>(nb.n - first, kRowsPerLaunch);
    const int lanes = row_lanes(nb), blocks = csr_blocks(rows, lanes);
    if (lanes == 1)
      k_csr_density<1><<<blocks, kBlock, 0, st>>>(x, nb, rho, pc, (int)first);
    else
      k_csr_density<kRowLanes><<<blocks, kBlock, 0, st>>>(x, nb, rho, pc, (int)first);
  }
}

__global__ __launch_bounds__(kBlock) void k_aos_to_f4(const float* __restrict__ x, float4* __restrict__ xa, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) xa[i] = load3(x, i);
}

void launch_aos_to_f4(const float* x, float4* xa, int n, hipStream_t st) {
  k_aos_to_f4<<<(n + kBlock - 1) / kBlock, kBlock, 0, st>>>(x, xa, n);
}

// The positions as the constraint's first iterate, its second buffer cleared
// (the displacement sums of a one-sided list start from zero,
// m_deltaPos.reset(), DensityPBD.cu:315), and the list's pairing sums.
__global__ __launch_bounds__(kBlock) void k_csr_begin(const float* __restrict__ x, float4* __restrict__ xa,
                                                      float4* __restrict__ xb, int n,
                                                      unsigned long long* __restrict__ pairing) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kPairingWords) pairing[i] = 0ull;
  if (i >= n) return;
  xa[i] = load3(x, i);
  xb[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Whether every listed pair is listed both ways, with equal multiplicity: the
// matrix A of the list (A_ij: how often row i lists j) is symmetric exactly
// when the bilinear form sum_ij (A_ij - A_ji) r_i s_j vanishes for all r, s.
// Row i adds r_i sum_j s_j - s_i sum_j r_j with r a 64-bit SplitMix64 value per
// particle and s another xorshift-multiply mix of it (Freivalds' check of a matrix
// identity, modulo 2^64): a
// symmetric list gives 0, another one does with probability of order 2^-60.
// Only integers are added, so the sum depends on no order.
__device__ __forceinline__ unsigned long long pairing_r(int j) {
  unsigned long long z = (unsigned long long)(unsigned)j * 0x9E3779B97F4A7C15ull + 0xD1B54A32D192ED03ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ unsigned long long pairing_s(unsigned long long r) {
  r = (r ^ (r >> 32)) * 0xD6E8FEB86659FD93ull;
  return r ^ (r >> 29);
}

// True when the sums of the list's rows add up to zero (uniform loads).
__device__ __forceinline__ bool csr_paired(const unsigned long long* __restrict__ pairing) {
  unsigned long long v = 0;
#pragma unroll
  for (int k = 0; k < kPairingSlots; ++k) v += pairing[k * kPairingStride];
  return v == 0ull;
}

// The iterate that iteration `it` reads: a list that lists every pair both
// ways moves the particles from one buffer to the other, any other one keeps
// them in xa and sums the displacements in xb.
__device__ __forceinline__ float4* csr_iterate(float4* xa, float4* xb, bool paired, int it) {
  return paired && (it & 1) ? xb : xa;
}

// The displacement sums of particle j of any other list: three floats each, packed.
// The atomics of neighboring particles fall into fewer lines than with a float4
// each: five iterations at 262,144 rows of 3 elements 575 -> 522 us, of 72 9,970 ->
// 8,990.
__device__ __forceinline__ float* csr_sums(float4* xb, int j) {
  return reinterpret_cast<float*>(xb) + 3 * (size_t)j;
}

// Density and K_ComputeLambdas (DensityPBD.cu:46-90) over a CSR list; lambda
// goes to w of the iterate. With minv (inverse masses) the massInv variant
// (DensityPBD.cu:93-131): S = sum_j |g|^2 m_j^-1 + |sum g|^2 m_i^-1. The first
// iteration (kFirst) also adds up the pairing sums of the rows.
template <bool kFirst, bool kMass, int kL>
__global__ __launch_bounds__(kBlock) void k_csr_lambda(float4* xa, float4* xb, int it, Csr nb,
                                                       float* __restrict__ rho, PhysConst pc,
                                                       const float* __restrict__ minv,
                                                       unsigned long long* __restrict__ pairing) {
  float4* xs = kFirst ? xa : csr_iterate(xa, xb, csr_paired(pairing), it);
  const CsrRow<kL> row = csr_row<kL>(nb);
  const bool active = row.i < nb.n;
  unsigned long long sum_r = 0, sum_s = 0;
  if (active) {
    const int i = row.i;
    const float4 xi = xs[i];
    float acc = 0.f, sgx = 0.f, sgy = 0.f, sgz = 0.f, sgg = 0.f, t[kRowUnroll];
    csr_each(
        nb, row, [&](int j) { return MassPos{xs[j], kMass ? minv[j] : 1.0f}; },
        [&](int u, int j, const MassPos& q) {
          const PairGeom p = pair_geom(xi, q.x, pc.inv_h);
          t[u] = p.t;
          const float t2 = p.t * p.t;
          const float gq = p.r > pc.pair_eps ? t2 * p.rinv : 0.0f;
          const float gx = gq * p.dx, gy = gq * p.dy, gz = gq * p.dz;
          sgx += gx;
          sgy += gy;
          sgz += gz;
          const float gg = gx * gx + gy * gy + gz * gz;
          sgg += kMass ? gg * q.m : gg;
          if (kFirst) {
            const unsigned long long r = pairing_r(j);
            sum_r += r;
            sum_s += pairing_s(r);
          }
        },
        [&] { row_clear(t); }, [&] { acc = row_cubes<kL>(acc, t); });
    acc *= pc.cW;
    sgx = row_sum<kL>(sgx);
    sgy = row_sum<kL>(sgy);
    sgz = row_sum<kL>(sgz);
    sgg = row_sum<kL>(sgg);
    if (row.lane == 0) {
      const float G2 = sgx * sgx + sgy * sgy + sgz * sgz;
      const float S = (pc.cG * pc.cG) * (sgg + (kMass ? G2 * minv[i] : G2));
      float lam = -(acc - pc.lam_rest) / (S + pc.lam_eps);
      lam = lam > 0.0f ? 0.0f : lam;
      reinterpret_cast<float*>(xs + i)[3] = lam;
      if (rho) rho[i] = acc;
    }
  }
  if (kFirst) {
    // every lane of the block is here; one atomic per block, over a few slots
    __shared__ unsigned long long part[kBlock / 64];
    const unsigned long long r = active ? pairing_r(row.i) : 0ull;
    unsigned long long v = r * sum_s - (active ? pairing_s(r) : 0ull) * sum_r;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < kBlock / 64; ++w) v += part[w];
      atomicAdd(&pairing[blockIdx.x % kPairingSlots * kPairingStride], v);
    }
  }
}

// K_ComputeDisplacement and K_UpdatePosition (DensityPBD.cu:135-179,227-237)
// over any list. The reference adds dp_ij to i and -dp_ij to j from row i. In
// a list with every pair listed both ways (what NeighborQuery gives for
// particles inside the grid) the two rows of a pair add the same to i, since
// dp_ji = -dp_ij: row i alone gives 2 sum_j dp_ij, with no atomics and in a
// fixed order. Any other list takes float atomics on the displacement sums (in
// xb), as the reference, applied by k_csr_apply. The atomics are what the
// general form costs: 1,747 us per pass at 262,144 particles (18.9M pairs, about
// 32 G atomics/s), against 36 us without. With minv the massInv variant
// (DensityPBD.cu:182-224): dp_ij m_i^-1 to i, -dp_ij m_j^-1 to j. The last
// iteration of a paired list also makes the velocity update
// (DensityPBD.cu:368-378) and writes the caller's arrays.
template <bool kMass, int kL>
__global__ __launch_bounds__(kBlock) void k_csr_displacement(float4* xa, float4* xb, int it, int last, Csr nb,
                                                             PhysConst pc, const float* __restrict__ minv,
                                                             const unsigned long long* __restrict__ pairing,
                                                             float* __restrict__ x, float* __restrict__ v) {
  const bool paired = csr_paired(pairing);
  const float4* xs = csr_iterate(xa, xb, paired, it);
  const CsrRow<kL> row = csr_row<kL>(nb);
  if (row.i >= nb.n) return;
  const int i = row.i;
  const float4 xi = xs[i];
  const float scale = pc.corr * pc.cG;
  const float mi = kMass ? minv[i] : 1.0f;
  float ax = 0.f, ay = 0.f, az = 0.f;
  if (paired) {
    csr_each(
        nb, row, [&](int j) { return xs[j]; },
        [&](int, int, float4 xj) {
          const PairGeom p = pair_geom(xi, xj, pc.inv_h);
          const bool use = p.r > pc.pair_eps;
          const float c = scale * (xi.w + xj.w) * (p.t * p.t) * p.rinv;
          ax += use ? c * p.dx : 0.0f;
          ay += use ? c * p.dy : 0.0f;
          az += use ? c * p.dz : 0.0f;
        },
        [] {}, [] {});
    const float k = 2.0f * mi;
    ax = row_sum<kL>(ax);
    ay = row_sum<kL>(ay);
    az = row_sum<kL>(az);
    if (row.lane != 0) return;
    const float nx = fmaf(k, ax, xi.x), ny = fmaf(k, ay, xi.y), nz = fmaf(k, az, xi.z);
    if (last)
      csr_finish(i, make_float4(nx, ny, nz, 0.0f), x, v, pc.dt);
    else
      (it & 1 ? xa : xb)[i] = make_float4(nx, ny, nz, 0.0f);
    return;
  }
  csr_each(
      nb, row, [&](int j) { return MassPos{xs[j], kMass ? minv[j] : 1.0f}; },
      [&](int, int j, const MassPos& q) {
        const PairGeom p = pair_geom(xi, q.x, pc.inv_h);
        if (!(p.r > pc.pair_eps)) return;
        const float c = scale * (xi.w + q.x.w) * (p.t * p.t) * p.rinv;
        const float px = c * p.dx, py = c * p.dy, pz = c * p.dz;
        ax += px * mi;
        ay += py * mi;
        az += pz * mi;
        float* d = csr_sums(xb, j);
        atomicAdd(d, -px * q.m);
        atomicAdd(d + 1, -py * q.m);
        atomicAdd(d + 2, -pz * q.m);
      },
      [] {}, [] {});
  ax = row_sum<kL>(ax);
  ay = row_sum<kL>(ay);
  az = row_sum<kL>(az);
  if (row.lane != 0) return;
  float* d = csr_sums(xb, i);
  atomicAdd(d, ax);
  atomicAdd(d + 1, ay);
  atomicAdd(d + 2, az);
}

// K_UpdatePosition (DensityPBD.cu:227-237) of a list with one-sided pairs;
// clears the displacement sums for the next round (m_deltaPos.reset(),
// DensityPBD.cu:315). The last iteration makes the velocity update.
__global__ __launch_bounds__(kBlock) void k_csr_apply(float4* __restrict__ xa, float4* __restrict__ xb, int n,
                                                      int last, const unsigned long long* __restrict__ pairing,
                                                      float* __restrict__ x, float* __restrict__ v, float dt) {
  if (csr_paired(pairing)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float4 p = xa[i];
  float* d = csr_sums(xb, i);
  p.x += d[0];
  p.y += d[1];
  p.z += d[2];
  if (last) {
    csr_finish(i, p, x, v, dt);
    return;
  }
  xa[i] = p;
  d[0] = d[1] = d[2] = 0.f;
}

// x := x + 0 and v := v + 0/dt of a constraint without iterations
// (DP_UpdateVelocity alone, DensityPBD.cu:368-388).
__global__ __launch_bounds__(kBlock) void k_csr_finish(const float4* __restrict__ xa, float* __restrict__ x,
                                                       float* __restrict__ v, int n, float dt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) csr_finish(i, xa[i], x, v, dt);
}

template <bool kMass, int kL>
void csr_rounds(float4* xa, float4* xb, unsigned long long* pairing, const Csr& nb, float* x, float* v, float* rho,
                const PhysConst& pc, int K, const float* minv, hipStream_t st) {
  const int nb1 = (nb.n + kBlock - 1) / kBlock, nbr = csr_blocks(nb.n, kL);
  for (int it = 0; it < K; ++it) {
    const int last = it + 1 == K;
    float* r = last ? rho : nullptr;
    if (it == 0)
      k_csr_lambda<true, kMass, kL><<<nbr, kBlock, 0, st>>>(xa, xb, it, nb, r, pc, minv, pairing);
    else
      k_csr_lambda<false, kMass, kL><<<nbr, kBlock, 0, st>>>(xa, xb, it, nb, r, pc, minv, pairing);
    k_csr_displacement<kMass, kL><<<nbr, kBlock, 0, st>>>(xa, xb, it, last, nb, pc, minv, pairing, x, v);
    k_csr_apply<<<nb1, kBlock, 0, st>>>(xa, xb, nb.n, last, pairing, x, v, pc.dt);
  }
  if (K == 0) k_csr_finish<<<nb1, kBlock, 0, st>>>(xa, x, v, nb.n, pc.dt);
}

void launch_csr_constrain(float4* xa, float4* xb, unsigned long long* pairing, const Csr& nb, float* x, float* v,
                          float* rho, const PhysConst& pc, int K, const float* minv, hipStream_t st) {
  const int blocks = (std::max(nb.n, kPairingWords) + kBlock - 1) / kBlock;
  k_csr_begin<<<blocks, kBlock, 0, st>>>(x, xa, xb, nb.n, pairing);
  auto run = [&](auto* rounds) { rounds(xa, xb, pairing, nb, x, v, rho, pc, K, minv, st); };
  if (row_lanes(nb) == 1)
    run(minv ? csr_rounds<true, 1> : csr_rounds<false, 1>);
  else
    run(minv ? csr_rounds<true, kRowLanes> : csr_rounds<false, kRowLanes>);
}

}  // namespace pbf
