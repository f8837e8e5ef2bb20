// Protein potential grids built on the device from the protein's atoms.
//
// Channel p < nprobe (soft-core Lennard-Jones for a probe of radius r_p):
//   sum_i sqrt(eps_i) * ((R/d)^12 - 2 (R/d)^6),  R = r_i + r_p,
// over atoms with d <= lj_cutoff, then capped at +lj_cap.
// Channel nprobe (Coulomb with a distance-dependent dielectric 4d):
//   sum_i 332.0636 q_i / (4 d^2) over atoms with d <= elec_cutoff, clamped
// to [-elec_cap, elec_cap].  d^2 is floored at 1e-4 A^2.
// Grid point (i, j, k) sits at gmin + (i, j, k) * h.  Each point sums its
// atoms in ascending index order in FP64 with no contraction, so the result
// is fixed by the inputs (independent of the launch shape).
#include <hip/hip_runtime.h>

#include "gridbuild.hpp"

namespace cdk {

namespace {

constexpr int kTile = 256;     // atoms staged in LDS per pass
constexpr int kMaxProbe = 15;  // probe channels

// One wavefront per 4 x 4 x 4 cube of grid points, four (2 x 2 x 1) per
// workgroup; grid edges are multiples of 8.  Per tile of staged atoms, each
// lane tests one atom against the wavefront's cube and the wavefront takes
// only the atoms whose cutoff sphere reaches it, in ascending order.
//
// What bounds it: FP64 vector instructions.  A wavefront along a z row (64
// points, 32 A) had some lane inside the cutoffs of 44% (elec) and 20% (LJ) of
// 3 000 atoms in a 32 A box and evaluated their divisions and probe terms for
// all lanes, after a distance to every atom; a 2 A cube meets 17% and 7%.
// The squared contact distances (r_i + r_p)^2 are staged per atom and probe,
// and s^12 - 2 s^6 is one fma (2 s^6 is exact), so a probe term is 7
// instructions instead of 10.  Same terms in the same order: bit-identical.
// Measured, 3 000 atoms onto 64^3 x 9: 1.12 ms -> 0.42 ms.  (Two atoms'
// divisions side by side, and workgroups in a scattered order so that every
// CU gets inner and outer cubes, changed nothing.)
//
// NPC: probe channels computed, the next multiple of 4 (zero radius past
// nprobe, not written).
template <int NPC>
__global__ __launch_bounds__(256) void k_build_grids(int natom, const double* __restrict__ atoms, int nprobe,
                                                     const double* __restrict__ probe, int n, double g0, double g1,
                                                     double g2, double h, double rc_lj2, double rc_el2,
                                                     double lj_cap, double el_cap, float* __restrict__ out) {
#pragma clang fp contract(off)
  __shared__ double sx[kTile], sy[kTile], sz[kTile], sc[kTile], se[kTile];
  __shared__ __align__(16) double sr2[kTile][NPC];  // (r_i + r_p)^2
  const size_t G = (size_t)n * n * n;
  const int nb = n / 8;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int bz = (int)(blockIdx.x % (2 * nb)), by = (int)(blockIdx.x / (2 * nb)) % nb, bx = (int)(blockIdx.x / (2 * nb * nb));
  const int x0 = 8 * bx + 4 * (wave >> 1), y0 = 8 * by + 4 * (wave & 1), z0 = 4 * bz;
  const int ix = x0 + (lane >> 4), iy = y0 + ((lane >> 2) & 3), iz = z0 + (lane & 3);
  const double gx = g0 + ix * h, gy = g1 + iy * h, gz = g2 + iz * h;
  // the wavefront's cube
  const double lx = g0 + x0 * h, ly = g1 + y0 * h, lz = g2 + z0 * h;
  const double hx = g0 + (x0 + 3) * h, hy = g1 + (y0 + 3) * h, hz = g2 + (z0 + 3) * h;
  // far above the rounding of the distances, so no atom that some point of
  // the cube has within the cutoff is left out
  const double reach2 = rc_el2 * (1.0 + 1e-9) + 1e-9;
  double lj[NPC];
#pragma unroll
  for (int p = 0; p < NPC; ++p) lj[p] = 0.0;
  double el = 0.0;
  for (int t0 = 0; t0 < natom; t0 += kTile) {
    const int m = min(kTile, natom - t0);
    __syncthreads();
    if ((int)threadIdx.x < m) {
      const int t = threadIdx.x;
      const double* a = atoms + (size_t)(t0 + t) * 6;
      sx[t] = a[0];
      sy[t] = a[1];
      sz[t] = a[2];
      sc[t] = 332.0636 * a[3];
      se[t] = sqrt(a[5]);
#pragma unroll
      for (int p = 0; p < NPC; ++p) {
        const double R = a[4] + (p < nprobe ? probe[p] : 0.0);
        sr2[t][p] = R * R;
      }
    }
    __syncthreads();
    for (int b = 0; b < m; b += 64) {
      const int t = b + lane;
      bool near = false;
      if (t < m) {
        // distance from the atom to the cube; + 0 x keeps a NaN coordinate in
        const double x = sx[t], y = sy[t], z = sz[t];
        const double dx = fmax(fmax(lx - x, x - hx), 0.0) + 0.0 * x;
        const double dy = fmax(fmax(ly - y, y - hy), 0.0) + 0.0 * y;
        const double dz = fmax(fmax(lz - z, z - hz), 0.0) + 0.0 * z;
        near = !(dx * dx + dy * dy + dz * dz > reach2);
      }
      for (unsigned long long mask = __ballot(near); mask; mask &= mask - 1) {
        const int k = b + __builtin_ctzll(mask);
        const double dx = sx[k] - gx, dy = sy[k] - gy, dz = sz[k] - gz;
        double d2 = dx * dx + dy * dy + dz * dz;
        if (d2 > rc_el2) continue;
        d2 = fmax(d2, 1e-4);
        el += sc[k] / (4.0 * d2);
        if (d2 > rc_lj2) continue;
        const double inv2 = 1.0 / d2;
        const double w = se[k];
#pragma unroll
        for (int p = 0; p < NPC; ++p) {
          const double s2 = sr2[k][p] * inv2;
          const double s6 = s2 * s2 * s2;
          lj[p] += w * fma(-2.0, s6, s6 * s6);
        }
      }
    }
  }
  const size_t g = ((size_t)ix * n + iy) * n + iz;
#pragma unroll
  for (int p = 0; p < NPC; ++p)
    if (p < nprobe) out[(size_t)p * G + g] = (float)fmin(lj[p], lj_cap);
  out[(size_t)nprobe * G + g] = (float)fmax(-el_cap, fmin(el, el_cap));
}

}  // namespace

int grid_build_max_probes() { return kMaxProbe; }

hipError_t launch_build_grids(hipStream_t st, int natom, const double* atoms, int nprobe, const double* probe, int n,
                              const double* gmin, double h, double lj_cutoff, double elec_cutoff, double lj_cap,
                              double elec_cap, float* out) {
  if (nprobe < 0 || nprobe > kMaxProbe) return hipErrorInvalidValue;
  if (n <= 0 || n % 8 != 0) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(n / 8) * (unsigned)(n / 8) * (unsigned)(n / 4));
  auto* k = nprobe <= 4 ? k_build_grids<4> : nprobe <= 8 ? k_build_grids<8> : nprobe <= 12 ? k_build_grids<12>
                                                                                        : k_build_grids<16>;
  hipLaunchKernelGGL(k, grid, dim3(256), 0, st, natom, atoms, nprobe, probe, n, gmin[0], gmin[1], gmin[2], h,
                     lj_cutoff * lj_cutoff, elec_cutoff * elec_cutoff, lj_cap, elec_cap, out);
  return hipGetLastError();
}

}  // namespace cdk
