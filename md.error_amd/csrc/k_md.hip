// k_md.hip -- the MD step either side of the force path: velocity Verlet
// (H/src/Integrator.cu:273-347, velocityVerlet_part1/part2), the two-link
// Nose-Hoover chain thermostat (H/src/Thermostat.cu:255-276, NoseHoover_Chains2::
// operator_L) and the centre-of-mass velocity removal
// (H/src/Integrator_interface.cu:40-68, TranslationalFreedomRemover::remove),
// in the order of the reference driver (H/app/lj.nhc-xtc.cu:158-196):
//   remove COM -> NHC(dt/2) -> kick(dt/2) + drift(dt) -> force -> kick(dt/2)
//   -> NHC(dt/2).
// GPU-side formulation: one reduction of (kinetic energy, momentum) per step,
// taken in the kick kernel; the chain variables live on the device and one
// single-block kernel (or, in small systems, every block of the next drift)
// turns the reduced sums into the velocity factors of the next step
// (v <- a2 (a1 v - v_com)), using that scaling all velocities by a multiplies K
// by a^2 and that removing the COM velocity lowers K by |P|^2 / 2M.  The drift is
// also the position refresh.  No host synchronisation: the whole step is
// graph-capturable.
#include "sre_internal.h"

namespace sre {

constexpr int kMDBlock = 256;
constexpr int kStateWords = sizeof(MDState) / 4;
static_assert(sizeof(MDState) % 4 == 0 && kStateWords <= kMDBlock, "one word per thread");

// one NHC half step of length h on the chain variables, given the current
// kinetic energy K; returns the velocity scale factor (operator_L order)
__device__ double nhc_operator(MDState &m, double h, double K) {
  const double T = m.refT;
  m.vxi2 += (m.Q1 * m.vxi1 * m.vxi1 - T) / m.Q2 * (0.5 * h);   // G2
  m.vxi1 *= exp(-m.vxi2 * 0.25 * h);                             // vxi1
  m.vxi1 += (2.0 * K - m.LL * T) / m.Q1 * (0.5 * h);             // G1
  m.vxi1 *= exp(-m.vxi2 * 0.25 * h);                             // vxi1
  const double a = exp(-m.vxi1 * h);                             // Cv
  K *= a * a;
  m.xi1 += m.vxi1 * h;                                           // xi
  m.xi2 += m.vxi2 * h;
  m.vxi1 *= exp(-m.vxi2 * 0.25 * h);                             // vxi1
  m.vxi1 += (2.0 * K - m.LL * T) / m.Q1 * (0.5 * h);             // G1
  m.vxi1 *= exp(-m.vxi2 * 0.25 * h);                             // vxi1
  m.vxi2 += (m.Q1 * m.vxi1 * m.vxi1 - T) / m.Q2 * (0.5 * h);     // G2
  return a;
}

// Kick v += F dt/(2m) (caller order; forces read from the sorted slot) and
// save the force in caller order for the next step's first kick (a rebuild
// in between reorders the sorted arrays).  Per-block partial sums of
// (K = sum m v^2 / 2, P = sum m v) in a fixed order -> part[block][4].
__global__ __launch_bounds__(kMDBlock) void k_md_kick(
    int n, const uint32_t *__restrict__ inv_perm, const int *__restrict__ types,
    const int64_t *__restrict__ fx, const int64_t *__restrict__ fy,
    const int64_t *__restrict__ fz, const double *__restrict__ fxd,
    const double *__restrict__ fyd, const double *__restrict__ fzd,
    const float *__restrict__ mass, float hdt, float *__restrict__ vel,
    float *__restrict__ fcall, double *__restrict__ part, MDState *state,
    const MDState *next) {
  __shared__ double red[kMDBlock / kWave][4];
  const bool store = next && blockIdx.x == 0 && threadIdx.x < kStateWords;
  const uint32_t word = store ? reinterpret_cast<const uint32_t *>(next)[threadIdx.x] : 0u;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double k = 0.0, px = 0.0, py = 0.0, pz = 0.0;
  if (i < n) {
    const int s = (int)inv_perm[i];
    float Fx, Fy, Fz;
    if (fx) {
      Fx = (float)((double)fx[s] * kFixInv);
      Fy = (float)((double)fy[s] * kFixInv);
      Fz = (float)((double)fz[s] * kFixInv);
    } else {
      Fx = (float)fxd[s];
      Fy = (float)fyd[s];
      Fz = (float)fzd[s];
    }
    const float m = mass[types[i]];
    const float c = hdt / m;
    float *v = vel + (size_t)i * 3;
    const float vx = v[0] + c * Fx, vy = v[1] + c * Fy, vz = v[2] + c * Fz;
    v[0] = vx;
    v[1] = vy;
    v[2] = vz;
    float *f = fcall + (size_t)i * 3;
    f[0] = Fx;
    f[1] = Fy;
    f[2] = Fz;
    k = 0.5 * (double)m * ((double)vx * vx + (double)vy * vy + (double)vz * vz);
    px = (double)m * vx;
    py = (double)m * vy;
    pz = (double)m * vz;
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    k += __shfl_xor(k, o, kWave);
    px += __shfl_xor(px, o, kWave);
    py += __shfl_xor(py, o, kWave);
    pz += __shfl_xor(pz, o, kWave);
  }
  const int w = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) {
    red[w][0] = k; red[w][1] = px; red[w][2] = py; red[w][3] = pz;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < kMDBlock / kWave; ++q) {
      k += red[q][0]; px += red[q][1]; py += red[q][2]; pz += red[q][3];
    }
    double *d = part + (size_t)blockIdx.x * 4;
    d[0] = k; d[1] = px; d[2] = py; d[3] = pz;
  }
  if (store) reinterpret_cast<uint32_t *>(state)[threadIdx.x] = word;
}

// fixed-order sum of the kick partials by one block
__device__ void reduce_parts(int nparts, const double *part, double out[4]) {
  __shared__ double red[kMDBlock / kWave][4];
  double a[4] = {0, 0, 0, 0};
  for (int b = threadIdx.x; b < nparts; b += blockDim.x)
    for (int c = 0; c < 4; ++c) a[c] += part[(size_t)b * 4 + c];
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) a[c] += __shfl_xor(a[c], o, kWave);
  const int w = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0)
    for (int c = 0; c < 4; ++c) red[w][c] = a[c];
  __syncthreads();
  if (threadIdx.x == 0)
    for (int q = 1; q < kMDBlock / kWave; ++q)
      for (int c = 0; c < 4; ++c) a[c] += red[q][c];
  for (int c = 0; c < 4; ++c) out[c] = a[c];  // valid on thread 0
}

// Start of a step: the pending end-of-step NHC half step of the previous
// step, the COM velocity removal and this step's first NHC half step, all
// from the kinetic energy and momentum s after the previous kick.
__device__ void md_factors(MDState &m, const double s[4]) {
  const double h = 0.5 * m.dt;
  double K = s[0], P[3] = {s[1], s[2], s[3]};
  double a1 = 1.0, a2 = 1.0;
  if (m.thermostat && m.have_end) {
    a1 = nhc_operator(m, h, K);
    K *= a1 * a1;
    for (int c = 0; c < 3; ++c) P[c] *= a1;
  }
  for (int c = 0; c < 3; ++c) m.vcom[c] = 0.0;
  if (m.remove_com) {
    for (int c = 0; c < 3; ++c) m.vcom[c] = P[c] / m.total_mass;
    K -= 0.5 * (P[0] * P[0] + P[1] * P[1] + P[2] * P[2]) / m.total_mass;
  }
  if (m.thermostat) {
    a2 = nhc_operator(m, h, K);
    K *= a2 * a2;
  }
  m.a1 = a1;
  m.a2 = a2;
  m.have_end = 1;
  m.K = K;
}

__global__ __launch_bounds__(kMDBlock) void k_md_factors(int nparts,
                                                         const double *part,
                                                         MDState *st) {
  double s[4];
  reduce_parts(nparts, part, s);
  if (threadIdx.x != 0) return;
  MDState m = *st;
  md_factors(m, s);
  *st = m;
}

// The first half of a velocity Verlet step (H/src/Integrator.cu:273-324,
// velocityVerlet_part1) and the position refresh with its skin test (as in
// k_update_positions, one atom per thread in caller order):
// v <- a2 (a1 v - vcom) + F dt/(2m), x <- x + v dt, then x is wrapped back into
// [0, L) by one add or subtract of L (the reference wraps at each rebuild,
// H/src/MDSystem_interface.cu:19-36).
// With FOLD every block works out the factors itself, all from the same sums
// in the same order, behind its atoms' loads; block 0 leaves the advanced
// state in d.next, since others may still read d.state, and the kick that
// ends the step stores it.  What bounds it: latency, the loads' and the
// chain's (ten exponentials one after the other).
template <bool FOLD>
__global__ __launch_bounds__(kMDBlock) void k_md_drift(
    int n, const uint32_t *__restrict__ inv_perm, float *__restrict__ pos, int stride,
    const RepInfo *__restrict__ reps, Geom g1, int one_rep, uint4 *__restrict__ pos4,
    const uint4 *__restrict__ backup, float4 *__restrict__ res4,
    float *__restrict__ skin_part, int nparts, DriftArgs d) {
  __shared__ float fac[5];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int w = i / kWave;  // slots exist for the waves holding atoms
  const bool wslot = w * kWave < n;
  const int k = i < n ? i : n - 1;
  // issued first: this wave's running maximum, compared at the end, and all
  // that the atom needs
  const float prev = ((threadIdx.x & (kWave - 1)) == 0 && wslot) ? skin_part[w] : 0.f;
  const uint4 b = backup[k];
  const uint32_t s = inv_perm[k];
  float *p = pos + (size_t)k * stride;
  float *v = d.vel + (size_t)k * 3;
  const float *f = d.fcall + (size_t)k * 3;
  const float v0 = v[0], v1 = v[1], v2 = v[2];
  const float f0 = f[0], f1 = f[1], f2 = f[2];
  const float p0 = p[0], p1 = p[1], p2 = p[2];
  const float m = d.mass[d.types[k]];
  if (FOLD) {
    MDState ms;
    if (threadIdx.x == 0) ms = *d.state;
    double sum[4];
    reduce_parts(nparts, d.part, sum);
    if (threadIdx.x == 0) {
      md_factors(ms, sum);
      fac[0] = (float)ms.a1;
      fac[1] = (float)ms.a2;
      for (int c = 0; c < 3; ++c) fac[2 + c] = (float)ms.vcom[c];
      if (blockIdx.x == 0) *d.next = ms;
    }
    __syncthreads();
  }
  const float a1 = FOLD ? fac[0] : (float)d.state->a1;
  const float a2 = FOLD ? fac[1] : (float)d.state->a2;
  const float c0 = FOLD ? fac[2] : (float)d.state->vcom[0];
  const float c1 = FOLD ? fac[3] : (float)d.state->vcom[1];
  const float c2 = FOLD ? fac[4] : (float)d.state->vcom[2];
  float d2 = 0.f;
  if (i < n) {
    const float c = 0.5f * d.dt / m;
    const float vx = a2 * (a1 * v0 - c0) + c * f0;
    const float vy = a2 * (a1 * v1 - c1) + c * f1;
    const float vz = a2 * (a1 * v2 - c2) + c * f2;
    v[0] = vx;
    v[1] = vy;
    v[2] = vz;
    // with one replica its geometry is an argument
    const Geom G = one_rep ? g1 : geom_of(reps[b.w >> 8]);
    float x = p0 + vx * d.dt, y = p1 + vy * d.dt, z = p2 + vz * d.dt;
    x = x < 0.f ? x + G.L[0] : (x >= G.L[0] ? x - G.L[0] : x);
    y = y < 0.f ? y + G.L[1] : (y >= G.L[1] ? y - G.L[1] : y);
    z = z < 0.f ? z + G.L[2] : (z >= G.L[2] ? z - G.L[2] : z);
    p[0] = x;
    p[1] = y;
    p[2] = z;
    const uint32_t ux = quantize(x, G.invq[0]);
    const uint32_t uy = quantize(y, G.invq[1]);
    const uint32_t uz = quantize(z, G.invq[2]);
    pos4[s] = make_uint4(ux, uy, uz, b.w);
    if (res4)
      res4[s] = make_float4(quant_residual(x, G.invq[0], G.qd[0]),
                            quant_residual(y, G.invq[1], G.qd[1]),
                            quant_residual(z, G.invq[2], G.qd[2]), 0.f);
    d2 = dist2(disp(ux, b.x, G.q[0]), disp(uy, b.y, G.q[1]), disp(uz, b.z, G.q[2]));
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1)
    d2 = fmaxf(d2, __shfl_xor(d2, o, kWave));
  if ((threadIdx.x & (kWave - 1)) == 0 && wslot && d2 > prev) skin_part[w] = d2;
}

__global__ __launch_bounds__(kMDBlock) void k_md_store(MDState *state, const MDState *next) {
  if (threadIdx.x < kStateWords)
    reinterpret_cast<uint32_t *>(state)[threadIdx.x] =
        reinterpret_cast<const uint32_t *>(next)[threadIdx.x];
}

void launch_md_store(MDState *state, const MDState *next, hipStream_t st) {
  hipLaunchKernelGGL(k_md_store, dim3(1), dim3(kMDBlock), 0, st, state, next);
}

// End of a run: the pending end-of-step NHC half step; v <- a1 v follows
// (k_md_scale).  K is the kinetic energy after it.
__global__ __launch_bounds__(kMDBlock) void k_md_finish(int nparts,
                                                        const double *part,
                                                        MDState *st) {
  double s[4];
  reduce_parts(nparts, part, s);
  if (threadIdx.x != 0) return;
  MDState m = *st;
  double K = s[0], a1 = 1.0;
  if (m.thermostat && m.have_end) {
    a1 = nhc_operator(m, 0.5 * m.dt, K);
    K *= a1 * a1;
  }
  m.a1 = a1;
  m.a2 = 1.0;
  for (int c = 0; c < 3; ++c) m.vcom[c] = 0.0;
  m.have_end = 0;
  m.K = K;
  *st = m;
}

__global__ __launch_bounds__(kMDBlock) void k_md_scale(int n, const MDState *st,
                                                       float *vel) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * n) return;
  vel[i] = (float)(st->a1 * (double)vel[i]);
}

// Copies up to kCopySegs buffers (whole 4-byte words) in one launch: the
// snapshot / restore of an adaptive MD stretch.
__global__ __launch_bounds__(kMDBlock) void k_md_copy(CopySegs c) {
  size_t w = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int k = 0; k < c.count; ++k) {
    if (w < c.words[k]) {
      c.dst[k][w] = c.src[k][w];
      return;
    }
    w -= c.words[k];
  }
}

void launch_md_copy(const CopySegs &c, hipStream_t st) {
  size_t total = 0;
  for (int k = 0; k < c.count; ++k) total += c.words[k];
  if (total == 0) return;
  hipLaunchKernelGGL(k_md_copy, dim3((unsigned)((total + kMDBlock - 1) / kMDBlock)),
                     dim3(kMDBlock), 0, st, c);
}

int md_part_count(int n) { return (n + kMDBlock - 1) / kMDBlock; }

void launch_md_kick(int n, const uint32_t *inv_perm, const int *types,
                    const int64_t *fx, const int64_t *fy, const int64_t *fz,
                    const double *fxd, const double *fyd, const double *fzd,
                    const float *mass, float hdt, float *vel, float *fcall,
                    double *part, MDState *state, const MDState *next, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_md_kick, dim3(md_part_count(n)), dim3(kMDBlock), 0, st,
                     n, inv_perm, types, fx, fy, fz, fxd, fyd, fzd, mass, hdt,
                     vel, fcall, part, state, next);
}

// Each block adds up all sums of the kick, one per 256 atoms: with few, that
// hides behind the loads, and the launch of one block saved gives (100 MD steps
// of a slab with their rebuilds, a launch for the factors / folded) 2904 /
// 2786 us at 4 000 atoms, 4392 / 4290 at 64 000, 6178 / 6128 at 120 000, the
// same at 250 000 and 16460 / 16556 at 500 000
bool md_fold_factors(int n) { return n <= 131072; }

void launch_md_drift(int n, const uint32_t *inv_perm, float *pos, int stride,
                     const RepInfo *reps, const RepInfo *host_rep0, uint4 *pos4,
                     const uint4 *backup, float4 *res4, float *skin_part,
                     const DriftArgs &drift, hipStream_t st) {
  if (n <= 0) return;
  const Geom g = host_rep0 ? geom_of(*host_rep0) : Geom{};
  const dim3 grid((n + kMDBlock - 1) / kMDBlock), block(kMDBlock);
  const int parts = md_part_count(n), one = host_rep0 ? 1 : 0;
  if (drift.next) {
    hipLaunchKernelGGL(k_md_drift<true>, grid, block, 0, st, n, inv_perm, pos, stride, reps, g,
                       one, pos4, backup, res4, skin_part, parts, drift);
    return;
  }
  hipLaunchKernelGGL(k_md_factors, dim3(1), block, 0, st, parts, drift.part, drift.state);
  hipLaunchKernelGGL(k_md_drift<false>, grid, block, 0, st, n, inv_perm, pos, stride, reps, g,
                     one, pos4, backup, res4, skin_part, parts, drift);
}

void launch_md_finish(int n, const double *part, MDState *state, float *vel,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_md_finish, dim3(1), dim3(kMDBlock), 0, st,
                     md_part_count(n), part, state);
  hipLaunchKernelGGL(k_md_scale, dim3((3 * n + kMDBlock - 1) / kMDBlock),
                     dim3(kMDBlock), 0, st, n, state, vel);
}

}  // namespace sre
