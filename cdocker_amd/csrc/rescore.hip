// Grid-energy rescoring and rigid-body refinement of retained poses.
//
// The score of a pose with atoms at r_a (absolute coordinates, A) is
//   E = sum_a  sqrt(eps_a) * P_probe(a)(r_a) + q_a * P_elec(r_a),
// with P(r) the trilinear interpolation of a protein potential grid at
// u = (r - gridMin) / h.  Spreading an atom onto the 8 corners of its cell
// with the same weights and correlating (what the FFT search does,
// FillLigandGrid.cpp:41-66 and TranRotaConfSearchNoMini.cu:376-464) gives
// exactly this sum, so at a pose the search returns (pose rebuild of
// NoMini:468-487) the score equals the search's energy up to FP32 rounding.
// These kernels evaluate it in FP64, with its gradient, for poses handed to a
// minimiser (the grid forces of AddGridForcesToOpenMMSystem.cpp:54,100 use a
// spline interpolant instead, so they differ from this score by the
// interpolation).
#include <hip/hip_runtime.h>

#include <cmath>

#include "rescore.hpp"

namespace cdk {

namespace {

struct AtomTerm {
  double e;
  double g[3];
  int inside;
};

// Energy and gradient of one atom.  grid: [nch][N][N][N], z fastest.
__device__ __forceinline__ AtomTerm atom_term(const float* __restrict__ grid, int N, int pch, int ech, double wv,
                                              double wq, double x, double y, double z, double g0, double g1,
                                              double g2, double inv_h) {
  AtomTerm t{0.0, {0.0, 0.0, 0.0}, 0};
  const double u[3] = {(x - g0) * inv_h, (y - g1) * inv_h, (z - g2) * inv_h};
  int i[3];
  double f[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double fl = floor(u[k]);
    i[k] = (int)fl;
    f[k] = u[k] - fl;
    if (!(fl >= 0.0) || i[k] > N - 2) return t;  // outside (or NaN): no term
  }
  t.inside = 1;
  const size_t G = (size_t)N * N * N;
  const size_t base = ((size_t)i[0] * N + i[1]) * N + i[2];
  const float* pv = pch >= 0 ? grid + (size_t)pch * G + base : nullptr;
  const float* pe = grid + (size_t)ech * G + base;
  double e = 0.0, d0 = 0.0, d1 = 0.0, d2 = 0.0;
  // The corners' grid values, the two of a z edge in one load (4-byte aligned):
  // each lane's cell lies in lines of its own, so a load instruction costs its
  // lanes one by one and half the instructions take half the time.
  float fe[8], fv[8];
#pragma unroll
  for (int c = 0; c < 8; c += 2) {
    const size_t off = ((size_t)(c >> 2) * N + ((c >> 1) & 1)) * N;
    __builtin_memcpy(fe + c, pe + off, 8);
    if (pv) __builtin_memcpy(fv + c, pv + off, 8);
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int dx = c >> 2, dy = (c >> 1) & 1, dz = c & 1;
    const double X = dx ? f[0] : 1.0 - f[0], Y = dy ? f[1] : 1.0 - f[1], Z = dz ? f[2] : 1.0 - f[2];
    const double sx = dx ? 1.0 : -1.0, sy = dy ? 1.0 : -1.0, sz = dz ? 1.0 : -1.0;
    double v = wq * (double)fe[c];
    if (pv) v += wv * (double)fv[c];
    e += X * Y * Z * v;
    d0 += sx * Y * Z * v;
    d1 += X * sy * Z * v;
    d2 += X * Y * sz * v;
  }
  t.e = e;
  t.g[0] = d0 * inv_h;
  t.g[1] = d1 * inv_h;
  t.g[2] = d2 * inv_h;
  return t;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// One wavefront per pose, four poses per workgroup; lanes stride over atoms,
// then a fixed-order butterfly reduction (the same for every launch, so results
// are reproducible).  The caller's arrays may be pinned host memory: the
// workgroup takes its poses in, and puts their gradients out, as whole 16-byte
// pieces through LDS, so the host link carries each byte once.  Measured, 1 000
// poses of 40 atoms with the gradient, host arrays in and out: the call 191 ->
// 92 us (copies to and from device arrays before); the kernel itself, which
// carries those bytes now, 38 us (26 without the gradient; 7 on device arrays).
__global__ __launch_bounds__(256) void k_rescore(int npose, int natom, const double* __restrict__ coords,
                                                 const int* __restrict__ pch, const float* __restrict__ wv,
                                                 const float* __restrict__ wq, const float* __restrict__ grid, int N,
                                                 int ech, double g0, double g1, double g2, double inv_h,
                                                 double* __restrict__ energy, double* __restrict__ grad,
                                                 int* __restrict__ inside) {
  extern __shared__ double xs[];  // [4][natom][3], then the channels and weights
  const int p0 = blockIdx.x * 4;
  const int np = min(4, npose - p0), per = natom * 3, n = np * per;
  int* spch = reinterpret_cast<int*>(xs + 4 * per);
  float* swv = reinterpret_cast<float*>(spch + natom);
  float* swq = swv + natom;
  // p0 * per doubles is a multiple of 16 bytes
  const double2* src = reinterpret_cast<const double2*>(coords + (size_t)p0 * per);
  for (int i = threadIdx.x; i < n / 2; i += 256) reinterpret_cast<double2*>(xs)[i] = src[i];
  if ((n & 1) && threadIdx.x == 0) xs[n - 1] = coords[(size_t)p0 * per + n - 1];
  for (int a = threadIdx.x; a < natom; a += 256) {
    spch[a] = pch[a];
    swv[a] = wv[a];
    swq[a] = wq[a];
  }
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double e = 0.0;
  int n_in = 0;
  if (w < np) {
    double* r = xs + w * per;
    for (int a = lane; a < natom; a += 64) {
      const AtomTerm t = atom_term(grid, N, spch[a], ech, (double)swv[a], (double)swq[a], r[a * 3 + 0], r[a * 3 + 1],
                                   r[a * 3 + 2], g0, g1, g2, inv_h);
      e += t.e;
      n_in += t.inside;
      if (grad) {
        r[a * 3 + 0] = t.g[0];
        r[a * 3 + 1] = t.g[1];
        r[a * 3 + 2] = t.g[2];
      }
    }
    e = wave_sum(e);
    n_in = wave_sum_i(n_in);
    if (lane == 0) {
      energy[p0 + w] = e;
      if (inside) inside[p0 + w] = n_in;
    }
  }
  if (!grad) return;
  __syncthreads();
  double2* dst = reinterpret_cast<double2*>(grad + (size_t)p0 * per);
  for (int i = threadIdx.x; i < n / 2; i += 256) dst[i] = reinterpret_cast<const double2*>(xs)[i];
  if ((n & 1) && threadIdx.x == 0) grad[(size_t)p0 * per + n - 1] = xs[n - 1];
}

// ---- sums over the wavefront, several at a time -----------------------------
// Eight lane values v[0..7] -> their eight wavefront sums, sum k on the lanes
// whose bits 5, 4, 3 spell k: at each of the first three halvings a lane keeps
// half of the values and takes its partner's, so the eight sums cost 10 adds
// and exchanges instead of 48.  Every sum adds the same pairs as wave_sum's
// butterfly (lanes 32 apart, then 16, 8, 4, 2, 1): the same bits.
struct F64Pair {
  double a, b;
};
__device__ __forceinline__ F64Pair swap32(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return {__longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])),
          __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]))};
}
__device__ __forceinline__ F64Pair swap16(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return {__longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])),
          __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]))};
}
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// v of the lane 4 away (lane ^ 4): half-row mirror (^ 7), then quad reversal (^ 3).
__device__ __forceinline__ double xor4(double v) { return dpp64<0x1B>(dpp64<0x141>(v)); }

__device__ __forceinline__ double wave_sum8(const double (&v)[8]) {
  double h[4], q[2];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const F64Pair p = swap32(v[k], v[k + 4]);
    h[k] = p.a + p.b;
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const F64Pair p = swap16(h[k], h[k + 2]);
    q[k] = p.a + p.b;
  }
  const bool up = (threadIdx.x & 8) != 0;
  const double keep = up ? q[1] : q[0], give = up ? q[0] : q[1];
  double s = keep + dpp64<0x128>(give);  // row rotation by 8: lane ^ 8
  s += xor4(s);
  s += dpp64<0x4E>(s);  // quad permutation 2 3 0 1: lane ^ 2
  s += dpp64<0xB1>(s);  // quad permutation 1 0 3 2: lane ^ 1
  return s;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Lane sums of the force, the torque and the score of one pose: v[0..2] F,
// v[3..5] tau, v[6] E (penalty for an atom off the grid), v[7] = 0.
struct PoseTerm {
  double x, y, z;  // position
  double wv, wq;
  int pch;
};
__device__ __forceinline__ void add_terms(const PoseTerm& p, const float* __restrict__ grid, int N, int ech, double g0,
                                          double g1, double g2, double inv_h, double penalty, const double (&c)[3],
                                          double (&v)[8]) {
  const AtomTerm at = atom_term(grid, N, p.pch, ech, p.wv, p.wq, p.x, p.y, p.z, g0, g1, g2, inv_h);
  v[6] += at.inside ? at.e : penalty;
  const double fx = -at.g[0], fy = -at.g[1], fz = -at.g[2];
  v[0] += fx;
  v[1] += fy;
  v[2] += fz;
  const double dx = p.x - c[0], dy = p.y - c[1], dz = p.z - c[2];
  v[3] += dy * fz - dz * fy;
  v[4] += dz * fx - dx * fz;
  v[5] += dx * fy - dy * fx;
}

// Rigid-body descent on the grid score, one wavefront per pose.  Each step
// evaluates E, the force F = -sum g_a and the torque about the centroid
// tau = sum (r_a - c) x (-g_a); the trial move translates by st along F and
// rotates by sr about tau (Rodrigues).  A trial that lowers E + penalty is
// kept and both steps grow by 1.2 (capped), otherwise they halve.  Atoms off
// the grid add `penalty` each, so a pose cannot lower its score by leaving.
//
// One 64-thread workgroup per pose, atoms strided over the lanes (AL per lane,
// in registers).
//
// What bounds it: one wavefront per pose and a serial chain of `steps` score
// evaluations, so time is the chain's latency.  Keeping each lane's atoms,
// channels and weights in registers takes the LDS round trips and their
// global reloads out of it; the seven sums of an evaluation cost ten adds
// (wave_sum8) instead of 42 rounds through the LDS crossbar; the two norms and
// the six quotients that follow are each one square root and one division,
// on the lanes that hold the sums.  What is left per step is the latency of
// the grid gather and of the FP64 terms.  Measured, 1 000 poses of 40 atoms,
// 50 steps: 251 -> 194 us, and 117 us with the corner pairs of atom_term.
template <int AL>
__global__ __launch_bounds__(64) void k_refine(int npose, int natom, double* __restrict__ coords,
                                               const int* __restrict__ pch, const float* __restrict__ wv,
                                               const float* __restrict__ wq, const float* __restrict__ grid, int N,
                                               int ech, double g0, double g1, double g2, double inv_h, int steps,
                                               double penalty, double* __restrict__ energy) {
  const int pose = blockIdx.x;
  const int lane = threadIdx.x;
  if (pose >= npose) return;
  double* gr = coords + (size_t)pose * natom * 3;
  PoseTerm r[AL], q[AL];
#pragma unroll
  for (int u = 0; u < AL; ++u) {
    const int a = lane + 64 * u;
    r[u] = PoseTerm{0.0, 0.0, 0.0, 0.0, 0.0, -1};
    if (a < natom) r[u] = PoseTerm{gr[a * 3 + 0], gr[a * 3 + 1], gr[a * 3 + 2], (double)wv[a], (double)wq[a], pch[a]};
    q[u] = r[u];
  }
  double c[3];
  {
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < AL; ++u)
      if (lane + 64 * u < natom) {
        v[0] += r[u].x;
        v[1] += r[u].y;
        v[2] += r[u].z;
      }
    const double s = wave_sum8(v);
    for (int k = 0; k < 3; ++k) c[k] = lane_value(s, 8 * k) / (double)natom;
  }
  // this lane's sum among F (0..2), tau (3..5) and E (6), and all of them
  auto score = [&](const PoseTerm (&p)[AL], const double (&cc)[3]) {
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < AL; ++u)
      if (lane + 64 * u < natom) add_terms(p[u], grid, N, ech, g0, g1, g2, inv_h, penalty, cc, v);
    return wave_sum8(v);
  };
  const int mine = lane >> 3;  // which sum this lane holds
  double s = score(r, c);
  double e = lane_value(s, 48);
  double st = 0.1, sr = 0.02;
  const double st_max = 0.5, sr_max = 0.1;
  for (int it = 0; it < steps; ++it) {
    // |F| on the lanes of F, |tau| on the others
    const bool rot = mine >= 3;
    const double n0 = lane_value(s, 0), n1 = lane_value(s, 8), n2 = lane_value(s, 16);
    const double m0 = lane_value(s, 24), m1 = lane_value(s, 32), m2 = lane_value(s, 40);
    const double v0 = rot ? m0 : n0, v1 = rot ? m1 : n1, v2 = rot ? m2 : n2;
    const double norm = sqrt(v0 * v0 + v1 * v1 + v2 * v2);
    const double fn = lane_value(norm, 0), tn = lane_value(norm, 24);
    if (fn == 0.0 && tn == 0.0) break;
    // d = st F / |F|, axis = tau / |tau|
    const double num = rot ? s : st * s;
    const double quo = norm > 0.0 ? num / norm : 0.0;
    const double d[3] = {lane_value(quo, 0), lane_value(quo, 8), lane_value(quo, 16)};
    const double ax[3] = {lane_value(quo, 24), lane_value(quo, 32), lane_value(quo, 40)};
    const double th = tn > 0.0 ? sr : 0.0;
    double ct, sn;
    sincos(th, &sn, &ct);
#pragma unroll
    for (int u = 0; u < AL; ++u) {
      const double v0 = r[u].x - c[0], v1 = r[u].y - c[1], v2 = r[u].z - c[2];
      const double kd = ax[0] * v0 + ax[1] * v1 + ax[2] * v2;
      const double cx = ax[1] * v2 - ax[2] * v1, cy = ax[2] * v0 - ax[0] * v2, cz = ax[0] * v1 - ax[1] * v0;
      q[u].x = c[0] + d[0] + v0 * ct + cx * sn + ax[0] * kd * (1.0 - ct);
      q[u].y = c[1] + d[1] + v1 * ct + cy * sn + ax[1] * kd * (1.0 - ct);
      q[u].z = c[2] + d[2] + v2 * ct + cz * sn + ax[2] * kd * (1.0 - ct);
    }
    const double cn[3] = {c[0] + d[0], c[1] + d[1], c[2] + d[2]};
    const double s2 = score(q, cn);
    const double e2 = lane_value(s2, 48);
    if (e2 < e) {  // wave-uniform
#pragma unroll
      for (int u = 0; u < AL; ++u) r[u] = q[u];
      e = e2;
      s = s2;
      for (int k = 0; k < 3; ++k) c[k] = cn[k];
      st = fmin(st * 1.2, st_max);
      sr = fmin(sr * 1.2, sr_max);
    } else {
      st *= 0.5;
      sr *= 0.5;
    }
  }
#pragma unroll
  for (int u = 0; u < AL; ++u) {
    const int a = lane + 64 * u;
    if (a < natom) {
      gr[a * 3 + 0] = r[u].x;
      gr[a * 3 + 1] = r[u].y;
      gr[a * 3 + 2] = r[u].z;
    }
  }
  if (lane == 0) energy[pose] = e;
}

// CHARMM grid order (z fastest) to OpenMM's Continuous3DFunction order
// (x fastest), widened to double (AddGridForcesToOpenMMSystem.cpp:30-41).
__global__ __launch_bounds__(256) void k_grid_xfast(const float* __restrict__ in, int X, int Y, int Z,
                                                    double* __restrict__ out) {
  const size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t n = (size_t)X * Y * Z;
  if (o >= n) return;
  const int i = (int)(o % X);
  const int j = (int)((o / X) % Y);
  const int k = (int)(o / ((size_t)X * Y));
  out[o] = (double)in[((size_t)i * Y + j) * Z + k];
}

}  // namespace

hipError_t launch_grid_xfast(hipStream_t st, const float* in, int X, int Y, int Z, double* out) {
  const size_t n = (size_t)X * Y * Z;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_grid_xfast, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in, X, Y, Z, out);
  return hipGetLastError();
}

hipError_t launch_rescore(hipStream_t st, int npose, int natom, const double* coords, const int* pch,
                          const float* wv, const float* wq, const float* grid, int N, int ech, const double* gmin,
                          double h, double* energy, double* grad, int* inside) {
  if (npose <= 0) return hipSuccess;
  const unsigned blocks = (unsigned)((npose + 3) / 4);
  const size_t lds = (size_t)natom * (4 * 3 * sizeof(double) + sizeof(int) + 2 * sizeof(float));
  hipLaunchKernelGGL(k_rescore, dim3(blocks), dim3(256), lds, st, npose, natom, coords, pch, wv, wq, grid, N, ech,
                     gmin[0], gmin[1], gmin[2], 1.0 / h, energy, grad, inside);
  return hipGetLastError();
}

hipError_t launch_refine(hipStream_t st, int npose, int natom, double* coords, const int* pch, const float* wv,
                         const float* wq, const float* grid, int N, int ech, const double* gmin, double h, int steps,
                         double penalty, double* energy) {
  if (npose <= 0) return hipSuccess;
  if (natom <= 0 || natom > 64 * 8) return hipErrorInvalidValue;
  auto* k = natom <= 64 ? k_refine<1> : natom <= 128 ? k_refine<2> : natom <= 256 ? k_refine<4> : k_refine<8>;
  hipLaunchKernelGGL(k, dim3((unsigned)npose), dim3(64), 0, st, npose, natom, coords, pch, wv, wq, grid, N, ech,
                     gmin[0], gmin[1], gmin[2], 1.0 / h, steps, penalty, energy);
  return hipGetLastError();
}

}  // namespace cdk
