// Random-torsion conformers on the device.
//
// GeneRandomConformations.cpp:36-47 sets every rotatable bond of each of
// 2000 copies of the ligand to an angle drawn uniformly in [-pi, pi), then
// minimises each copy with OpenMM and keeps those under an energy cap
// (:49-109).  Here each trial sets the rotors in order to angles from a
// counter-based stream (seed, trial, rotor), keeps the trial when no
// non-excluded atom pair comes closer than clash_dist (a steric filter in
// place of the force-field energy, which needs OpenMM), and reports one flag
// per trial; the host keeps the first survivors in trial order.
//
// Setting a rotor (a, b, c, d) to angle theta: phi = the current (IUPAC)
// dihedral of a-b-c-d; the atoms on the d side of bond b-c turn about the
// axis b->c through c by theta - phi (Rodrigues, right-handed).  All in FP64,
// every fused multiply-add written out.
#include <hip/hip_runtime.h>

#include "conformers.hpp"

namespace cdk {

// splitmix64 finaliser on a (seed, trial, rotor) counter -> U[0, 1), 53 bits.
__host__ __device__ double torsion_uniform(unsigned long long seed, int trial, int rotor) {
  unsigned long long z = seed + 0x9E3779B97F4A7C15ull * ((unsigned long long)trial * 0x100000001ull +
                                                          (unsigned long long)rotor + 1ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

namespace {

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Value of v on lane `lane` (uniform).
__device__ __forceinline__ double lane_value(double v, int lane) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// a b - c d and a . b, each product but the first rounded with its sum.
__device__ __forceinline__ double cross(double a, double b, double c, double d) {
#pragma clang fp contract(off)
  return fma(a, b, -(c * d));
}
__device__ __forceinline__ double dot(double ax, double ay, double az, double bx, double by, double bz) {
#pragma clang fp contract(off)
  return fma(az, bz, fma(ay, by, ax * bx));
}

// One 64-thread workgroup per trial; the trial's coordinates live in LDS.
//
// What bounds it: a serial chain of nrotor rotations per trial, each a
// dihedral of four moving atoms and a turn of the atoms behind it.  Per 64
// rotors, lane r holds rotor r's atoms and the cosine and sine of its target
// angle theta, so the chain itself has no transcendental function and no
// global load: the turn by theta - phi comes from the angle sums, with cos phi
// and sin phi the dihedral's two components over their length.  Which atoms a
// rotor moves, and which partners the clash test of an atom skips, are bits in
// one 64-bit word per atom.  Measured, 20 000 trials of a 40-atom chain: 575 us
// with atan2, cos and sin per rotor and byte masks -> 353 us; a first set of
// 4 096 takes 86 us.  The components' rounding would stretch the turned
// atoms a little with every rotor, so the turn is brought to unit length and
// sums of products are fused.  Error against quadruple precision over 2 000
// trials of 40-atom chains, r.m.s. / mean largest of a chain, in A: 4.2e-14 /
// 3.5e-13 (with atan2, cos and sin 5.3e-14 / 5.2e-13; with neither 5.2e-14 /
// 4.9e-13).
//
// moving [ceil(nrotor / 64)][natom]: bit r % 64 of word r / 64 of an atom set
// when rotor r moves it.  exclude [natom][ceil(natom / 64)]: bits of the
// partners an atom is not tested against.
__global__ __launch_bounds__(64) void k_conformers(int natom, const double* __restrict__ coords, int nrotor,
                                                   const int4* __restrict__ rotors,
                                                   const unsigned long long* __restrict__ moving,
                                                   const unsigned long long* __restrict__ exclude, int first,
                                                   int ntrial, unsigned long long seed, double clash2,
                                                   double* __restrict__ out, int* __restrict__ ok) {
#pragma clang fp contract(off)
  extern __shared__ double sm[];
  const int lane = threadIdx.x;
  if ((int)blockIdx.x >= ntrial) return;
  const int t = first + blockIdx.x;
  double* x = sm;
  for (int i = lane; i < natom * 3; i += 64) x[i] = coords[i];
  const double kPi = 3.14159265358979323846;
  for (int r0 = 0; r0 < nrotor; r0 += 64) {
    const int nr = min(64, nrotor - r0);
    int4 rot = make_int4(0, 0, 0, 0);
    double ct = 1.0, st = 0.0;
    if (lane < nr) {
      rot = rotors[r0 + lane];
      sincos(-kPi + 2.0 * kPi * torsion_uniform(seed, t, r0 + lane), &st, &ct);
    }
    const unsigned long long* mvw = moving + (size_t)(r0 >> 6) * natom;
    const unsigned long long mv0 = lane < natom ? mvw[lane] : 0ull;
    for (int r = 0; r < nr; ++r) {
      const int a = __builtin_amdgcn_readlane(rot.x, r), b = __builtin_amdgcn_readlane(rot.y, r),
                c = __builtin_amdgcn_readlane(rot.z, r), d = __builtin_amdgcn_readlane(rot.w, r);
      wave_sync();  // the previous rotor's moves
      // current dihedral (every lane computes the same value)
      const double ax = x[a * 3 + 0], ay = x[a * 3 + 1], az = x[a * 3 + 2];
      const double bx = x[b * 3 + 0], by = x[b * 3 + 1], bz = x[b * 3 + 2];
      const double cx = x[c * 3 + 0], cy = x[c * 3 + 1], cz = x[c * 3 + 2];
      const double ex = x[d * 3 + 0], ey = x[d * 3 + 1], ez = x[d * 3 + 2];
      const double b1x = bx - ax, b1y = by - ay, b1z = bz - az;
      const double b2x = cx - bx, b2y = cy - by, b2z = cz - bz;
      const double b3x = ex - cx, b3y = ey - cy, b3z = ez - cz;
      const double n1x = cross(b1y, b2z, b1z, b2y), n1y = cross(b1z, b2x, b1x, b2z), n1z = cross(b1x, b2y, b1y, b2x);
      const double n2x = cross(b2y, b3z, b2z, b3y), n2y = cross(b2z, b3x, b2x, b3z), n2z = cross(b2x, b3y, b2y, b3x);
      const double l2 = sqrt(dot(b2x, b2y, b2z, b2x, b2y, b2z));
      // (xv, yv) = rho (cos phi, sin phi): xv = n1 . n2, yv = b2^ . (n1 x n2),
      // phi the IUPAC dihedral (0 for a collinear rotor)
      const double qx = cross(n1y, n2z, n1z, n2y), qy = cross(n1z, n2x, n1x, n2z), qz = cross(n1x, n2y, n1y, n2x);
      const double yv = dot(qx, qy, qz, b2x, b2y, b2z) / l2;
      const double xv = dot(n1x, n1y, n1z, n2x, n2y, n2z);
      const double rho = sqrt(fma(xv, xv, yv * yv));
      const double cp = rho == 0.0 ? 1.0 : xv / rho, sp = rho == 0.0 ? 0.0 : yv / rho;
      const double cth = lane_value(ct, r), sth = lane_value(st, r);
      double ca = fma(cth, cp, sth * sp), sa = fma(sth, cp, -(cth * sp));
      // one Newton step to unit length, so bond lengths do not drift
      const double dn = -0.5 * fma(ca, ca, fma(sa, sa, -1.0));
      ca = fma(dn, ca, ca);
      sa = fma(dn, sa, sa);
      const double ux = b2x / l2, uy = b2y / l2, uz = b2z / l2;
      wave_sync();  // every lane has read the rotor's atoms
      for (int i = lane; i < natom; i += 64) {
        if (!(((i == lane ? mv0 : mvw[i]) >> r) & 1)) continue;
        const double vx = x[i * 3 + 0] - cx, vy = x[i * 3 + 1] - cy, vz = x[i * 3 + 2] - cz;
        const double kd = dot(ux, uy, uz, vx, vy, vz);
        const double kx = cross(uy, vz, uz, vy), ky = cross(uz, vx, ux, vz), kz = cross(ux, vy, uy, vx);
        x[i * 3 + 0] = cx + fma(ux * kd, 1.0 - ca, fma(kx, sa, vx * ca));
        x[i * 3 + 1] = cy + fma(uy * kd, 1.0 - ca, fma(ky, sa, vy * ca));
        x[i * 3 + 2] = cz + fma(uz * kd, 1.0 - ca, fma(kz, sa, vz * ca));
      }
    }
  }
  wave_sync();
  // steric filter over the non-excluded pairs i < j
  const int ew = (natom + 63) >> 6;
  int bad = 0;
  for (int i = lane; i < natom; i += 64) {
    const double px = x[i * 3 + 0], py = x[i * 3 + 1], pz = x[i * 3 + 2];
    for (int j0 = (i & ~63); j0 < natom; j0 += 64) {
      unsigned long long skip = exclude[(size_t)i * ew + (j0 >> 6)];
      if (j0 <= i) skip |= ~0ull >> (63 - (i - j0));  // j <= i
      const int nj = min(64, natom - j0);
      for (int j = 0; j < nj; ++j) {
        const double dx = px - x[(j0 + j) * 3 + 0], dy = py - x[(j0 + j) * 3 + 1], dz = pz - x[(j0 + j) * 3 + 2];
        if (!((skip >> j) & 1) && dx * dx + dy * dy + dz * dz < clash2) bad = 1;
      }
    }
  }
  const unsigned long long anybad = __ballot(bad);
  double* o = out + (size_t)blockIdx.x * natom * 3;
  if (!anybad)
    for (int i = lane; i < natom * 3; i += 64) o[i] = x[i];
  if (lane == 0) ok[blockIdx.x] = anybad ? 0 : 1;
}

// The first max_keep set flags of ok[0, n): their indices to list, in order,
// and their number to *count.  One workgroup.
__global__ __launch_bounds__(1024) void k_kept(int n, const int* __restrict__ ok, int max_keep,
                                               int* __restrict__ list, int* __restrict__ count) {
  __shared__ int wsum[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int base = 0;
  for (int t0 = 0; t0 < n && base < max_keep; t0 += 1024) {
    const int t = t0 + threadIdx.x;
    const bool f = t < n && ok[t] != 0;
    const unsigned long long m = __ballot(f);
    if (lane == 0) wsum[wave] = __popcll(m);
    __syncthreads();
    int before = base, total = 0;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) before += wsum[w];
      total += wsum[w];
    }
    const int k = before + __popcll(m & ((1ull << lane) - 1));
    if (f && k < max_keep) list[k] = t;
    base += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) *count = min(base, max_keep);
}

// Kept trials' coordinates, packed: kept[k] = all[list[k]], k < *count; their
// trial numbers to trial.
__global__ __launch_bounds__(256) void k_pack(int per, int first, const double* __restrict__ all,
                                              const int* __restrict__ list, const int* __restrict__ count,
                                              double* __restrict__ kept, int* __restrict__ trial) {
  const int k = blockIdx.x;
  if (k >= *count) return;
  const double* s = all + (size_t)list[k] * per;
  double* d = kept + (size_t)k * per;
  for (int i = threadIdx.x; i < per; i += 256) d[i] = s[i];
  if (threadIdx.x == 0) trial[k] = first + list[k];
}

}  // namespace

hipError_t launch_conformers(hipStream_t st, int natom, const double* coords, int nrotor, const int* rotors,
                             const unsigned long long* moving, const unsigned long long* exclude, int first,
                             int ntrial, unsigned long long seed, double clash_dist, double* out, int* ok) {
  if (ntrial <= 0) return hipSuccess;
  const size_t lds = (size_t)natom * 3 * sizeof(double);
  hipLaunchKernelGGL(k_conformers, dim3((unsigned)ntrial), dim3(64), lds, st, natom, coords, nrotor,
                     reinterpret_cast<const int4*>(rotors), moving, exclude, first, ntrial, seed,
                     clash_dist * clash_dist, out, ok);
  return hipGetLastError();
}

hipError_t launch_keep_conformers(hipStream_t st, int natom, int first, int ntrial, const int* ok, const double* all,
                                  int max_keep, int* list, int* count, double* kept, int* trial) {
  if (ntrial <= 0 || max_keep <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_kept, dim3(1), dim3(1024), 0, st, ntrial, ok, max_keep, list, count);
  hipLaunchKernelGGL(k_pack, dim3((unsigned)min(max_keep, ntrial)), dim3(256), 0, st, natom * 3, first, all, list,
                     count, kept, trial);
  return hipGetLastError();
}

}  // namespace cdk
