// Batched NVT molecular dynamics on the device: the step of ASE's
// NVTBerendsen (ASE 3.18.1, the version the reference pins), which the
// reference's MD driver runs one structure per process
// (gappy/example/ASE-GAPPY/run_md.py:10-21: NVTBerendsen with
// timestep = POTIM fs, temperature = TEBEG K, taut = 500 fs):
//
//   T      = 2 Ekin / (3 N kB),  Ekin = sum p^2 / 2m
//   s      = sqrt(1 + (T0 / T - 1) dt / taut), clipped to [0.9, 1.1]
//   p     <- s p + dt/2 F
//   p     <- p - sum(p) / N            (fixcm: total momentum removed)
//   x     <- x + dt p / m
//   F     <- forces at x               (a GAP evaluation of the batch)
//   p     <- p + dt/2 F
//
// with every structure of the batch advanced together.  taut <= 0 turns the
// scaling off (plain velocity Verlet).  Units are ASE's: positions A,
// momenta amu A / t, masses amu, forces eV/A, dt in ASE time units
// (1 fs = 0.09822694788464063 t).
#include <cmath>

#include "../../include/gapx.h"
#include "gapx_internal.h"

namespace gapx {

namespace {

__device__ __forceinline__ double wave_sum_md(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// One workgroup per structure: 2 Ekin, sum p, sum F over its atoms, summed in
// a fixed order (lanes, then the four waves).  With kick the momenta first get
// half a step of the forces (p <- p + half_dt F).
template <bool KICK>
__device__ void struct_sums(const StructParams &P, const double *__restrict__ mass, double *__restrict__ p,
                            const double *__restrict__ f, double half_dt, double out[7]) {
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  double v[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int a = t; a < P.natoms; a += 256) {
    const size_t i = (size_t)(P.atom_base + a);
    const double m = mass[i];
    for (int c = 0; c < 3; ++c) {
      double pc = p[3 * i + c];
      const double fc = f[3 * i + c];
      if (KICK) {
        pc += half_dt * fc;
        p[3 * i + c] = pc;
      }
      v[0] += pc * pc / m;
      v[1 + c] += pc;
      v[4 + c] += fc;
    }
  }
  __shared__ double red[4][7];
  for (int k = 0; k < 7; ++k) {
    const double s = wave_sum_md(v[k]);
    if (lane == 0) red[wv][k] = s;
  }
  __syncthreads();
  for (int k = 0; k < 7; ++k) out[k] = (red[0][k] + red[1][k]) + (red[2][k] + red[3][k]);
  __syncthreads();
}

// Velocity scale and momentum shift per atom of a structure of n atoms.
__device__ __forceinline__ void step_coef(const MdParams &mp, int n, const double sum[7], double cf[4]) {
  double scale = 1.0;
  if (mp.taut > 0.0) {
    const double T = sum[0] / (3.0 * n * mp.kB);  // 2 Ekin / (3 N kB)
    scale = sqrt(1.0 + (mp.temperature / T - 1.0) * (mp.dt / mp.taut));
    // T = 0 gives +inf here and the clip to 1.1, as the division does in ASE
    if (!(scale <= 1.1)) scale = 1.1;
    if (scale < 0.9) scale = 0.9;
  }
  cf[0] = scale;
  for (int c = 0; c < 3; ++c)
    cf[1 + c] = mp.fixcm ? (scale * sum[1 + c] + 0.5 * mp.dt * sum[4 + c]) / n : 0.0;
}

__device__ __forceinline__ void drift_atom(size_t i, const double *__restrict__ mass, const double *__restrict__ f,
                                           const double cf[4], double dt, double *__restrict__ p,
                                           double *__restrict__ x) {
  const double m = mass[i];
  for (int c = 0; c < 3; ++c) {
    const double pc = cf[0] * p[3 * i + c] + 0.5 * dt * f[3 * i + c] - cf[1 + c];
    p[3 * i + c] = pc;
    x[3 * i + c] += dt * pc / m;
  }
}

__device__ __forceinline__ void write_log(const MdParams &mp, int n, const double sum[7], double ene, double *log) {
  log[0] = ene;
  log[1] = 0.5 * sum[0];
  log[2] = sum[0] / (3.0 * n * mp.kB);
}

// All that lies between two evaluations, in one launch: the second half kick of
// the step that ends (kick), its log entry (log != null) and the first half of
// the next step (drift).  One workgroup per structure, thread t on atoms t,
// t + 256, ..: no thread reads what another one wrote.  Bound by the launch
// itself for small structures: one instead of four takes 9 us of a step.
__global__ __launch_bounds__(256) void k_md_turn(int nstruct, const StructParams *__restrict__ sp,
                                                 const double *__restrict__ mass, const double *__restrict__ f,
                                                 MdParams mp, int kick, int drift, const double *__restrict__ ene,
                                                 double *__restrict__ p, double *__restrict__ x,
                                                 double *__restrict__ log) {
  const int s = blockIdx.x;
  if (s >= nstruct) return;
  const StructParams &P = sp[s];
  double sum[7];
  if (kick)
    struct_sums<true>(P, mass, p, f, 0.5 * mp.dt, sum);
  else
    struct_sums<false>(P, mass, p, f, 0.0, sum);
  if (log && threadIdx.x == 0) write_log(mp, P.natoms, sum, ene[s], log + 3 * (size_t)s);
  if (!drift) return;
  double cf[4];
  step_coef(mp, P.natoms, sum, cf);
  for (int a = threadIdx.x; a < P.natoms; a += 256) drift_atom((size_t)(P.atom_base + a), mass, f, cf, mp.dt, p, x);
}

__global__ __launch_bounds__(256) void k_md_prepare(int nstruct, const StructParams *__restrict__ sp,
                                                    const double *__restrict__ mass, double *__restrict__ p,
                                                    const double *__restrict__ f, MdParams mp,
                                                    double *__restrict__ coef) {
  const int s = blockIdx.x;
  if (s >= nstruct) return;
  const StructParams &P = sp[s];
  double sum[7];
  struct_sums<false>(P, mass, p, f, 0.0, sum);
  if (threadIdx.x == 0) step_coef(mp, P.natoms, sum, coef + 4 * (size_t)s);
}

__global__ void k_md_drift(int N, const int *__restrict__ atom_struct, const double *__restrict__ mass,
                           const double *__restrict__ f, const double *__restrict__ coef, double dt,
                           double *__restrict__ p, double *__restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  drift_atom((size_t)i, mass, f, coef + 4 * (size_t)atom_struct[i], dt, p, x);
}

__global__ void k_md_kick(int N, const double *__restrict__ f, double half_dt, double *__restrict__ p) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 3 * N) p[i] += half_dt * f[i];
}

}  // namespace

hipError_t launch_md_turn(hipStream_t s, int nstruct, const StructParams *sp, const double *mass, const double *f,
                          const MdParams &mp, bool kick, bool drift, const double *ene, double *p, double *x,
                          double *log) {
  k_md_turn<<<nstruct, 256, 0, s>>>(nstruct, sp, mass, f, mp, kick, drift, ene, p, x, log);
  return hipGetLastError();
}

hipError_t launch_md_prepare(hipStream_t s, int nstruct, const StructParams *sp, const double *mass, double *p,
                             const double *f, const MdParams &mp, double *coef) {
  k_md_prepare<<<nstruct, 256, 0, s>>>(nstruct, sp, mass, p, f, mp, coef);
  return hipGetLastError();
}

hipError_t launch_md_drift(hipStream_t s, int N, const int *atom_struct, const double *mass, const double *f,
                           const double *coef, double dt, double *p, double *x) {
  k_md_drift<<<(N + 255) / 256, 256, 0, s>>>(N, atom_struct, mass, f, coef, dt, p, x);
  return hipGetLastError();
}

hipError_t launch_md_kick(hipStream_t s, int N, const double *f, double half_dt, double *p) {
  k_md_kick<<<(3 * N + 255) / 256, 256, 0, s>>>(N, f, half_dt, p);
  return hipGetLastError();
}

}  // namespace gapx
