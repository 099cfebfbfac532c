// step.hip -- CDNA4 kernels of one AlgoGas hydro sub-step
// (src/SourceEuler.c:398-716 and its callees).
//
// Storage type T is double or float; arithmetic is double throughout, with
// the reference's operation order, so that the FP64 build reproduces the
// reference pointwise (the library is compiled without contraction).
// Every kernel of a sub-step reads dfargo_ctrl::active and returns at once
// when the host's DT is already covered, so that a fixed batch of sub-steps
// can be launched (or replayed from a HIP graph) without a host round trip.
#include <hip/hip_runtime.h>
#include <math.h>

#include "kernels.h"

const char *kKernelNames[KID_COUNT] = {
    "sg_rows_fwd", "sg_cols", "sg_rows_inv",
    "cfl_ring",    "control",        "source",  "energy",
    "transport_azi", "finish",      "dust_move",      "dust_scan",  "dust_scatter",
    "dust_rank",     "dust_deposit", "evanescent", "nonreflecting",
    "sgz_mean",      "sgz_conv",     "sgz_fill",     "eos_step",      "visc1d",
    "df_cfl",        "df_axisg",      "df_source",    "df_stress",    "df_visc",       "df_substep2",
    "df_transport_azi", "df_finish"};

// ------------------------------------------------------------------------
// helpers
// ------------------------------------------------------------------------

// The dust fluid runs with FP64 storage only: its branches in the shared
// kernels are compiled out of the FP32 instantiations.
#define DF_ON(T, a) (sizeof(T) == sizeof(double) && (a).df_on)

template <typename T> __device__ __forceinline__ double ld(const void *p, long i) {
  return (double)((const T *)p)[i];
}
template <typename T> __device__ __forceinline__ void st(void *p, long i, double v) {
  ((T *)p)[i] = (T)v;
}
// Unbiased stochastic rounding of the state to FP32 storage.  A value
// between two floats is stored as the upper one with probability equal to
// its distance from the lower one, in ulps; the draw is a hash of the cell,
// the sub-step count and a per-field salt, so the result is deterministic
// (a graph replay and an eager run agree).  Round-to-nearest would drop the
// same sub-ulp increment of a slowly evolving field every sub-step and let
// the error grow linearly; with unbiased rounding it grows as a random
// walk.  FP64 storage stores the value as it is.
__device__ __forceinline__ unsigned mix32(unsigned x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}
// (the part of the key that is the same in every cell, and a cell's key from it)
__device__ __forceinline__ unsigned sr_field(const dfargo_ctrl *c, unsigned salt) {
  return mix32((unsigned)c->substeps_total * 0x85EBCA6BU + salt);
}
__device__ __forceinline__ unsigned sr_cell(long l, unsigned field) { return mix32((unsigned)l * 0x9E3779B9U ^ field); }
__device__ __forceinline__ unsigned sr_key(const dfargo_ctrl *c, long l, unsigned salt) {
  return sr_cell(l, sr_field(c, salt));
}
template <typename T> __device__ __forceinline__ T sr_round(double v, unsigned key);
template <> __device__ __forceinline__ double sr_round<double>(double v, unsigned) { return v; }
// The 29 mantissa bits of the double below the float's last bit are the
// distance to the float of smaller magnitude, in units of 2^-29 ulp: adding
// 29 random bits (the top bits of the key) and clearing them carries into
// the float's last bit with exactly that probability, and the remaining
// double converts to float exactly (for normal floats; exact floats, zeros,
// infinities and NaNs come out unchanged).
template <> __device__ __forceinline__ float sr_round<float>(double v, unsigned key) {
  const long long b = __double_as_longlong(v);
  const long long t = (b + (long long)(key >> 3)) & ~0x1FFFFFFFLL;
  return (float)__longlong_as_double(t);
}
template <typename T> __device__ __forceinline__ void st_sr(void *p, long i, double v, unsigned key) {
  ((T *)p)[i] = sr_round<T>(v, key);
}
// salts of the stochastically rounded stores
enum { SR_VR = 1, SR_VT, SR_E, SR_EN, SR_RAD = 8, SR_AZI = 16, SR_EVA = 24, SR_ACC = 32, SR_FIN = 40 };

// a / b from the hardware reciprocal, two Newton steps and one correction of
// the quotient: the compiler's IEEE sequence without its scaling of operands
// near the ends of the exponent range (three of eleven instructions and the
// waits on their carry).  For the transport's operands, slopes and densities
// far from 1e-154 and 1e154, that is the IEEE quotient; with a zero or
// infinite divisor it is a NaN.
__device__ __forceinline__ double div_nr(double a, double b) {
  double r = __builtin_amdgcn_rcp(b);
  double e = fma(-b, r, 1.0);
  r = fma(r, e, r);
  e = fma(-b, r, 1.0);
  r = fma(r, e, r);
  const double q = a * r;
  return fma(r, fma(-b, q, a), q);
}

__device__ __forceinline__ double dmin2(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double dmax2(double a, double b) { return (b > a) ? b : a; }

// Sum and minimum over a wavefront, the same in every lane, in a fixed order, by
// VALU moves: a shuffle butterfly goes through the LDS crossbar twelve times for
// a double, each step waiting for the one before.
//
// The sum adds the halves, then quarters, ... then neighbours, a shuffle tree's
// order (32, 16, 8, 4, 2, 1): a sum of the ring (the cooling time's mean
// vtheta) enters every cell of it, so its last bit decides how single FP32 values
// are stored, and self-gravitating discs let those grow (128x512 with cooling: 4e-5
// after forty calls).  Halves and rows meet by gfx950's lane swaps, which given
// one value twice leave both partners' in every lane; lanes within a row by
// rotations (row_ror 8, 4, 2, 1 = 0x128, 0x124, 0x122, 0x121).
template <int CTRL> __device__ __forceinline__ double row_rotate(double v) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ double wave_sum(double v) {
  const unsigned l0 = (unsigned)__double2loint(v), h0 = (unsigned)__double2hiint(v);
  const auto l1 = __builtin_amdgcn_permlane32_swap(l0, l0, false, false);
  const auto h1 = __builtin_amdgcn_permlane32_swap(h0, h0, false, false);
  v = __hiloint2double((int)h1[0], (int)l1[0]) + __hiloint2double((int)h1[1], (int)l1[1]);
  const unsigned l2 = (unsigned)__double2loint(v), h2 = (unsigned)__double2hiint(v);
  const auto l3 = __builtin_amdgcn_permlane16_swap(l2, l2, false, false);
  const auto h3 = __builtin_amdgcn_permlane16_swap(h2, h2, false, false);
  v = __hiloint2double((int)h3[0], (int)l3[0]) + __hiloint2double((int)h3[1], (int)l3[1]);
  v += row_rotate<0x128>(v);
  v += row_rotate<0x124>(v);
  v += row_rotate<0x122>(v);
  v += row_rotate<0x121>(v);
  return v;
}
// row_shr:1, 2, 4, 8 = 0x111, 0x112, 0x114, 0x118; row_bcast:15, :31 = 0x142,
// 0x143 (into the rows 1 and 3, then 2 and 3); lanes without a source keep their
// own value; the total is in lane 63
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_row(double v, double other) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(__double2hiint(other), hi, CTRL, ROWS, 0xf, false),
                          __builtin_amdgcn_update_dpp(__double2loint(other), lo, CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ double lane63(double v) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}
__device__ __forceinline__ double wave_min(double v) {
  v = dmin2(v, dpp_row<0x111, 0xf>(v, v));
  v = dmin2(v, dpp_row<0x112, 0xf>(v, v));
  v = dmin2(v, dpp_row<0x114, 0xf>(v, v));
  v = dmin2(v, dpp_row<0x118, 0xf>(v, v));
  v = dmin2(v, dpp_row<0x142, 0xa>(v, v));
  v = dmin2(v, dpp_row<0x143, 0xc>(v, v));
  return lane63(v);
}

// The same over a block of whole wavefronts, the wavefronts' values in
// wavefront order; every thread gets the results.  sh holds 16 N doubles and
// may be used again after the return.
template <int N> __device__ __forceinline__ void block_sum_n(double (&v)[N], double *sh) {
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const double s = wave_sum(v[k]);
    if ((threadIdx.x & 63) == 0) sh[wave * N + k] = s;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; k++) {
    double s = 0.0;
    for (int w = 0; w < nw; w++) s += sh[w * N + k];
    v[k] = s;
  }
  __syncthreads();
}
__device__ __forceinline__ double block_sum(double v, double *sh) {
  double w[1] = {v};
  block_sum_n<1>(w, sh);
  return w[0];
}
__device__ __forceinline__ double block_min(double v, double *sh) {
  const int nw = blockDim.x >> 6;
  v = wave_min(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double m = sh[0];
  for (int w = 1; w < nw; w++) m = dmin2(m, sh[w]);
  __syncthreads();
  return m;
}

// Neumaier-compensated running sum
struct CSum {
  double s, c;
  __device__ void add(double x) {
    double t = s + x;
    if (fabs(s) >= fabs(x)) c += (s - t) + x;
    else c += (x - t) + s;
    s = t;
  }
  __device__ double value() const { return s + c; }
};

// Ring kernels hold K cells of a ring per thread.  With K = 1 a block may
// have 1024 threads (128 VGPRs per lane), with K = 2 768 threads (168
// VGPRs), from K = 3 on 512 threads (256 VGPRs), so that the K-wide working
// set stays in registers.
#define RING_LB(K) ((K) == 1 ? 1024 : ((K) == 2 ? 768 : 512))

// AspectRatio (src/Viscosity.c:107-122) and compute_smoothing
// (src/Force.c:255-263), LAMBDADOUBLING = 0
__device__ double d_aspect_ratio(const KArgs &a, double rad) {
  double ar = a.aspect_ratio;
  double rmin = a.transition_radius - a.transition_width * a.aspect_ratio;
  double rmax = a.transition_radius + a.transition_width * a.aspect_ratio;
  if (rad < rmin) ar *= a.transition_ratio;
  if ((rad >= rmin) && (rad <= rmax))
    ar *= exp((rmax - rad) / (rmax - rmin) * log(a.transition_ratio));
  return ar;
}
__device__ double d_smoothing(const KArgs &a, double r) {
  // pow(r, 1) is r
  return a.thickness_smoothing * d_aspect_ratio(a, r) * (a.flaring == 0.0 ? r : pow(r, 1.0 + a.flaring));
}

// gravitational potential at cell (i, j): FillForcesArrays
// (src/Pframeforce.c:44-129) with the parameters the control kernel stored
__device__ double pot_at(const KArgs &a, const dfargo_ctrl *c, int i, int j) {
  double x = a.Rmed[i] * a.CosAz[j], y = a.Rmed[i] * a.SinAz[j];
  double pot = 0.0;
  for (int k = 0; k < c->nb; k++) {
    double xp = c->pot_x[k], yp = c->pot_y[k], mp = c->pot_m[k];
    double distance = (x - xp) * (x - xp) + (y - yp) * (y - yp);
    double distancesmooth = sqrt(distance + c->pot_smooth[k]);
    double pk = -DF_G * mp / distancesmooth;
    if (a.indirect_term) pk += DF_G * mp * c->pot_invd3[k] * (x * xp + y * yp);
    pot += pk;
  }
  double ps = -DF_G * 1.0 * a.InvRmed[i];
  if (a.gas_indirect) ps -= c->ind_x * x + c->ind_y * y;
  pot += ps;
  return pot;
}

// ------------------------------------------------------------------------
// per-call and per-sub-step control
// ------------------------------------------------------------------------

// GetPsysInfo (src/Psys.c:233-350), actions MARK (get = 0) and GET
// (get = 1).  The frame's centre is planet 0 (the outermost planet with
// COROTATEWITHOUTERPLANET) or, with FRAME B, the barycentre of planets 0 and
// 1, moved with FRAME G to the guiding centre of its orbit unless e < 1e-8.
// GET returns the angle the centre turned through since the mark.  The
// orbital frequency the reference also forms (with its self-gravity
// correction) serves only the FREQUENCY action and the guiding centre's
// velocity, which MARK and GET do not use.
__device__ double psys_info(const KArgs &a, dfargo_ctrl *c, int get) {
  const int k = a.frame_outer ? c->nb - 1 : 0;
  double x = c->pl_x[k], y = c->pl_y[k], vx = c->pl_vx[k], vy = c->pl_vy[k], m = c->pl_m[k] + 1.;
  if (a.frame == DFARGO_FRAME_BINARY_CENTER) {
    double m0 = c->pl_m[0], m1 = c->pl_m[1];
    if (m0 == 0.0) m0 = c->pl_m1[0];
    if (m1 == 0.0) m1 = c->pl_m1[1];
    x = (m0 * c->pl_x[0] + m1 * c->pl_x[1]) / (m0 + m1);
    y = (m0 * c->pl_y[0] + m1 * c->pl_y[1]) / (m0 + m1);
    vx = (m0 * c->pl_vx[0] + m1 * c->pl_vx[1]) / (m0 + m1);
    vy = (m0 * c->pl_vy[0] + m1 * c->pl_vy[1]) / (m0 + m1);
    m = m0 + m1 + 1.;
  }
  double xc = x, yc = y;
  if (a.frame == DFARGO_FRAME_GUIDING_CENTER) {
    const double h = x * vy - y * vx, d = sqrt(x * x + y * y);
    const double Ax = x * vy * vy - y * vx * vy - DF_G * m * x / d;
    const double Ay = y * vx * vx - x * vx * vy - DF_G * m * y / d;
    const double e = sqrt(Ax * Ax + Ay * Ay) / m, sa = h * h / DF_G / m / (1. - e * e);
    const double arg = (e == 0.0) ? 1.0 : (1.0 - d / sa) / e;
    double E = (fabs(arg) >= 1.0) ? DF_PI * (1. - arg / fabs(arg)) / 2. : acos((1.0 - d / sa) / e);
    if ((x * y * (vy * vy - vx * vx) + vx * vy * (x * x - y * y)) < 0) E = -E;
    const double M = E - e * sin(E), pa = atan2(Ay, Ax);
    if (!(e < 1e-8)) {
      xc = sa * cos(M + pa);
      yc = sa * sin(M + pa);
    }
  }
  if (!get) {
    c->mark_x = xc;
    c->mark_y = yc;
    return 0.0;
  }
  const double d2 = sqrt(xc * xc + yc * yc), d1 = sqrt(c->mark_x * c->mark_x + c->mark_y * c->mark_y);
  const double cross = c->mark_x * yc - xc * c->mark_y;
  c->mark_x = xc;
  c->mark_y = yc;
  return asin(cross / (d1 * d2));
}

// The planets as the control wavefront holds them: planet k in lane k
// (k < nb; the other lanes hold zeros), other planets' values by lane moves.
struct Body {
  double x, y, vx, vy, m;
};
__device__ __forceinline__ Body load_body(const dfargo_ctrl *c, int lane) {
  Body b = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (lane < c->nb) b = {c->pl_x[lane], c->pl_y[lane], c->pl_vx[lane], c->pl_vy[lane], c->pl_m[lane]};
  return b;
}

// start of a sub-step: mass taper, n-body limit and the force-sum targets
// (src/SourceEuler.c:398-440, src/Pframeforce.c:131-161); one wavefront, run
// once the loop condition holds.  c lies in LDS.
__device__ void begin_substep(const KArgs &a, dfargo_ctrl *c, Body b, double time, int lane) {
  const int nb = c->nb;
  const bool planet = lane < nb;
  double pmass = c->particles_mass0;
  if (a.mass_taper_param > 1e-2) {
    double mt = (time - c->time0) / (a.mass_taper_param * 2.0 * DF_PI);
    mt = (mt > 1.0 ? 1.0 : pow(sin(mt * DF_PI / 2.0), 2.0));
    if (planet && mt < 1.0) b.m = c->pl_m0[lane] + (c->pl_m1[lane] - c->pl_m0[lane]) * mt;
    pmass = pmass * mt;
    if (lane == 0) c->mass_taper = mt;
  } else if (planet && c->pl_acc[lane] < 1e-10) {
    b.m = c->pl_m1[lane];
  }
  if (planet) c->pl_m[lane] = b.m;
  double dtnbody = 100.0;
  if (nb > 1) {
    dtnbody = 1e5;
    for (int j = 1; j < nb; j++) {
      const double dx = b.x - __shfl(b.x, j, 64), dy = b.y - __shfl(b.y, j, 64), mj = __shfl(b.m, j, 64);
      const double dist = sqrt(dx * dx + dy * dy);
      const double buf = 2.0 * DF_PI * sqrt(dist * dist * dist / (b.m + mj + 1e-8)) / 100.0;
      if (lane < j) dtnbody = dmin2(dtnbody, buf);
    }
    dtnbody = wave_min(dtnbody);
  }
  // target 0: the star (ComputeAccel at 0,0, src/SourceEuler.c:482); then
  // the planets that feel the disc, in order
  const bool feels = planet && c->pl_feel_disk[lane];
  const unsigned long long who = __ballot(feels);
  if (lane == 0) {
    c->particles_mass = pmass;
    c->dtnbody = dtnbody;
    c->tg_x[0] = 0.0;
    c->tg_y[0] = 0.0;
    c->tg_rsm[0] = a.indirect_smoothing;
    c->tg_a[0] = 0.0;
    c->tg_rh[0] = 1e-15;
    c->tg_planet[0] = -1;
    c->ntarget = 1 + __popcll(who);
  }
  if (feels) {
    const int nt = 1 + __popcll(who & ((1ull << lane) - 1ull));
    const double r = sqrt(b.x * b.x + b.y * b.y);
    c->tg_x[nt] = b.x;
    c->tg_y[nt] = b.y;
    c->tg_rsm[nt] = a.roche ? r * pow(b.m / 3., 1. / 3.) * a.roche_smoothing : d_smoothing(a, r);
    c->tg_a[nt] = r;
    // the Hill radius enters only the cut of EXCLUDEHILL
    c->tg_rh[nt] = a.exclude_hill ? pow(b.m / 3., 1. / 3.) * r + 1e-15 : 0.0;
    c->tg_planet[nt] = lane;
  }
}

// AlgoGas entry: loop variables, and the first sub-step's start.  The
// sub-step kernels read three flags of the control block: `go` (the loop
// condition of the current sub-step: read by the kernels that may run
// before or beside the control kernel, the CFL and self-gravity kernels),
// `active` (set by the control kernel from `go`, read by every kernel after
// it) and `go_next` (the condition of the next sub-step, set by the control
// kernel, which also prepares that sub-step's start; it tells the kernels
// after the control kernel whether theirs is the last sub-step of the
// call).  The last kernel of a sub-step copies go_next into go, so no flag
// changes under a kernel that reads it, even with the self-gravity kernels
// running concurrently with the control kernel.
__global__ void __launch_bounds__(64) k_algogas_begin(KArgs a, double DT) {
  __shared__ dfargo_ctrl cs;
  constexpr int NW = (int)(sizeof(dfargo_ctrl) / 8);
  const int t = threadIdx.x;
  for (int w = t; w < NW; w += 64) ((unsigned long long *)&cs)[w] = ((const unsigned long long *)a.ctrl)[w];
  __syncthreads();
  if (t == 0) {
    cs.DT = DT;
    cs.dtemp = 0.0;
    cs.substeps = 0;
    cs.gas_timesteps_cfl = 1;
    cs.active = 0;
    cs.go = 0.0 < 0.999999999 * DT;
    cs.go_next = cs.go;
    cs.fargo_margin_bits = 0x3FE0000000000000ULL; // 0.5
  }
  __syncthreads();
  if (cs.go) begin_substep(a, &cs, load_body(&cs, t), cs.time, t);
  __syncthreads();
  for (int w = t; w < NW; w += 64) ((unsigned long long *)a.ctrl)[w] = ((const unsigned long long *)&cs)[w];
}

// ConditionCFL per ring (src/SourceEuler.c:1340-1484) fused with the
// per-ring partial sums of ComputeForce (src/Force.c:155-214), GasTotalMass
// and the barycentre (src/SideEuler.c:15-77) and DetectCrash
// (src/SourceEuler.c:51-69): one read of rho, vr, vt (and cs, e).
//
// Bound by the chain load - sum of vt - CFL terms - minimum, a few
// microseconds on its own whatever the grid, so everything the ring mean of
// vt does not enter shares the first reduction with it and the fields are
// loaded before that reduction waits (up to six cells per thread; beyond, the
// registers do not hold them).  The star's force needs no sum of its own: the
// ring's cells lie at one distance from it, so it is the barycentre sum times a
// factor of the ring.  SG: with self-gravity it is summed cell by cell all the
// same.  The two differ in the last bits, which through the indirect term enter
// the potential of every cell; a cell whose vr passes zero then stores another
// FP32 value, and gravity spreads it (128x384 and 128x512 with cooling: 4e-5 after
// forty calls).  1024x3072 FP32 374 -> 381 us a sub-step, 512x1536 154.6 -> 155.6.
template <typename T, int K, bool SG> __device__ __forceinline__ void cfl_ring(const KArgs &a) {
  constexpr int M = SG ? 9 : 7;
  __shared__ double sh[16 * M];
  __shared__ double shmin[16], shf[16 * 4];
  const dfargo_ctrl *c = a.ctrl;
  if (!c->go) return;
  const int i = ring_of_block(a), ns = a.ns, nr = a.nr, t = threadIdx.x, TB = ns / K, nw = blockDim.x >> 6;
  const bool on = t < TB; // the block is the ring's threads rounded up to whole wavefronts
  const int t0 = on ? t : 0;
  const long base = (long)i * ns;
  // the CFL arithmetic is FP64 whatever the storage type: the sub-step
  // count ceil(DT / dt_min) then follows the FP64 run's, and FP32 storage
  // changes the solution, not the time discretisation
  const T *vt = (const T *)a.vt + base, *vr = (const T *)a.vr + base, *rho = (const T *)a.rho + base;
  constexpr bool AHEAD = K <= 6;
  constexpr int KA = AHEAD ? K : 1;
  T vt_own[K], vt_next[KA], vr_in[KA], vr_out[KA], cs_prev[KA];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int j = t0 + k * TB;
    vt_own[k] = vt[j];
    if constexpr (AHEAD) {
      vt_next[k] = vt[(j == ns - 1) ? 0 : j + 1];
      vr_in[k] = vr[j];
      vr_out[k] = vr[j + ns];
      cs_prev[k] = a.energy ? ((const T *)a.cs)[base + j] : (T)0;
    }
  }
  // per-ring partials, stored partial-major (ring_part[p * nr + i]):
  // negative-density and negative-energy counts, disc mass, barycentre.
  // With the energy equation the same pass is ComputeSoundSpeed
  // (src/SourceEuler.c:2340; the CFL below reads the previous cs) and
  // the ring mean of cs that mpi_make1Dprofile feeds to FViscosity
  // (src/Viscosity.c:30-35) for the kernels after this one.
  double *part = a.ring_part + i;
  T cs_new[K];
  {
    CSum m = {0, 0}, xb = {0, 0}, yb = {0, 0}, fx = {0, 0}, fy = {0, 0};
    double s = 0.0, css = 0.0;
    int crd = 0, cre = 0;
    const double rsm = c->tg_rsm[0];
    const double g = a.gamma;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int j = t0 + k * TB;
      const double dens = (double)rho[j];
      s += (double)vt_own[k];
      crd += dens < 0.0;
      cs_new[k] = (T)0;
      if (a.energy) {
        const double en = ld<T>(a.en, base + j);
        cre += en < 0.0;
        cs_new[k] = (T)sqrt(g * (g - 1.0) * en / dens);
        css += (double)cs_new[k];
      }
      const double cm = a.Surf[i] * dens;
      const double xc = a.Rmed[i] * a.CosAz[j], yc = a.Rmed[i] * a.SinAz[j];
      m.add(cm);
      xb.add(cm * xc);
      yb.add(cm * yc);
      if (SG) {
        const double dist2 = (xc * xc + yc * yc) + rsm * rsm, inv3 = 1.0 / dist2 / sqrt(dist2);
        fx.add(DF_G * cm * xc * inv3);
        fy.add(DF_G * cm * yc * inv3);
      }
    }
    const double v[9] = {s, (double)crd, (double)cre, m.value(), xb.value(), yb.value(), css, fx.value(), fy.value()};
#pragma unroll
    for (int q = 0; q < M; q++) {
      if ((q == 2 || q == 6) && !a.energy) continue;
      const double w = wave_sum(on ? v[q] : 0.0);
      if ((t & 63) == 0) sh[(t >> 6) * M + q] = w;
    }
  }
  __syncthreads();
  double vsum = 0.0;
  for (int w = 0; w < nw; w++) vsum += sh[w * M];
  const double vmoy = vsum / (double)ns;
  // The threads past the ring take no part in the minimum: beyond six cells a
  // thread cs is read here, and the thread that owns a cell replaces it below
  // with no barrier between, so each thread may only read its own cells.
  double dtmin = 1e30;
  if (i >= 1 && on) {
    const double viscosity = a.nu_ring[i];
    const double dxrad = a.Rsup[i] - a.Rinf[i];
    const double dxtheta = a.Rmed[i] * a.pm / (double)ns;
    const double dxmin = (dxrad < dxtheta) ? dxrad : dxtheta;
    const double invdt5 = (viscosity != 0.0) ? viscosity * 4.0 / a.powmin2[i] : 1e-10;
    // the ring's cell sizes divide every cell's terms: one reciprocal each
    // (within an ulp of the quotients, which only moves dt by as much)
    const double idxmin = 1.0 / dxmin, idxrad = 1.0 / dxrad, idxtheta = 1.0 / dxtheta;
    double smax = 0.0;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int j = t0 + k * TB;
      double vtn, vrl, vro, cs;
      if constexpr (AHEAD) {
        vtn = (double)vt_next[k];
        vrl = (double)vr_in[k];
        vro = (double)vr_out[k];
        cs = a.energy ? (double)cs_prev[k] : a.cs_iso[i];
      } else {
        vtn = (double)vt[(j == ns - 1) ? 0 : j + 1];
        vrl = (double)vr[j];
        vro = (double)vr[j + ns];
        cs = a.energy ? ld<T>(a.cs, base + j) : a.cs_iso[i];
      }
      const double vtl = (double)vt_own[k];
      const double vres = a.fast ? vtl - vmoy : vtl;
      const double invdt1 = cs * idxmin;
      const double invdt2 = fabs(vrl) * idxrad;
      const double invdt3 = fabs(vres) * idxtheta;
      double dvr = vro - vrl, dvt = vtn - vtl;
      if (dvr >= 0.0) dvr = 1e-10; else dvr = -dvr;
      if (dvt >= 0.0) dvt = 1e-10; else dvt = -dvt;
      const double q4 = dvr * idxrad, q5 = dvt * idxtheta;
      double invdt4 = (q5 > q4) ? q5 : q4;
      invdt4 *= 4.0 * DF_CVNR * DF_CVNR;
      const double invdt6 = 1e-10;
      // dt = CFLSECURITY / sqrt(S) decreases with S, and rounding keeps
      // that order: the smallest dt of the ring is that of its largest S
      const double S = invdt1 * invdt1 + invdt2 * invdt2 + invdt3 * invdt3 + invdt4 * invdt4 + invdt5 * invdt5 +
                       invdt6 * invdt6;
      smax = (S > smax) ? S : smax;
    }
    dtmin = DF_CFLSECURITY / sqrt(smax);
  }
  dtmin = wave_min(dtmin);
  if ((t & 63) == 0) shmin[t >> 6] = dtmin;
  if (on) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      const long l = base + t + k * TB;
      if (a.energy) {
        // the particles of this sub-step still read the previous cs
        if (a.d_on) ((T *)a.cs_old)[l] = ((const T *)a.cs)[l];
        ((T *)a.cs)[l] = cs_new[k];
      }
      // the particle buckets of this sub-step start empty
      if (a.d_on) a.cell_count[l] = 0;
    }
  }
  __syncthreads();
  const bool hill = a.exclude_hill;
  if (t < M && !((t == 2 || t == 6) && !a.energy)) {
    double s = 0.0;
    for (int w = 0; w < nw; w++) s += sh[w * M + t];
    if (t == 0) {
      a.vmoy[i] = vmoy;
      double d = shmin[0];
      for (int w = 1; w < nw; w++) d = dmin2(d, shmin[w]);
      a.ring_dt[i] = d;
    } else if (t < 6) {
      part[(long)(t - 1) * nr] = s;
      if (t >= 4 && !SG) {
        // target 0, the star: G cellmass dx / d^3 with d one value on the ring
        // (no cell lies in its Hill radius, 1e-15)
        const double rsm = c->tg_rsm[0], dist2 = a.Rmed[i] * a.Rmed[i] + rsm * rsm;
        const double f = DF_G * s * (1.0 / dist2 / sqrt(dist2));
        double *g = part + (long)(5 + 2 * (t - 4)) * nr;
        g[0] = f;
        if (hill) g[nr] = f;
      }
    } else if (SG && t >= 7) {
      double *g = part + (long)(5 + 2 * (t - 7)) * nr;
      g[0] = s;
      if (hill) g[nr] = s;
    } else {
      const double gcs = s / (double)ns;
      a.gcs[i] = gcs;
      double nu = a.visc_const;
      if (a.alpha_on) nu = a.alpha * gcs * gcs * a.r15[i];
      a.nu_ring[i] = a.visc_on ? nu * a.visc_mult[i] : 0.0;
    }
  }
  // then fx, fx (Hill-cut), fy, fy (Hill-cut) per planet that feels the disc;
  // the inner/outer split of GlobalForce is only ever summed, so it is not kept
  for (int tg = 1; tg < c->ntarget; tg++) {
    const double x = c->tg_x[tg], y = c->tg_y[tg], rsm = c->tg_rsm[tg];
    const double rh = c->tg_rh[tg];
    CSum fx[2] = {{0, 0}, {0, 0}}, fy[2] = {{0, 0}, {0, 0}};
    if (on)
#pragma unroll
      for (int k = 0; k < K; k++) {
        const int j = t + k * TB;
        double xc = a.Rmed[i] * a.CosAz[j], yc = a.Rmed[i] * a.SinAz[j];
        double cellmass = a.Surf[i] * (double)rho[j];
        double dx = xc - x, dy = yc - y;
        double d2 = dx * dx + dy * dy;
        double dist2 = d2 + rsm * rsm;
        double distance = sqrt(dist2);
        double InvDist3 = 1.0 / dist2 / distance;
        fx[0].add(DF_G * cellmass * dx * InvDist3 * 1.0);
        fy[0].add(DF_G * cellmass * dy * InvDist3 * 1.0);
        if (hill) {
          double planet_distance = sqrt(d2);
          double cutoff = a.exclude_hill_factor * rh, hill_cut;
          if (planet_distance / cutoff < 0.5) hill_cut = 0.0;
          else if (planet_distance > cutoff) hill_cut = 1.0;
          else hill_cut = pow(sin((planet_distance / cutoff - .5) * DF_PI), 2.);
          fx[1].add(DF_G * cellmass * dx * InvDist3 * hill_cut);
          fy[1].add(DF_G * cellmass * dy * InvDist3 * hill_cut);
        }
      }
    double *g = part + (long)(5 + 4 * tg) * nr;
    if (hill) {
      double v[4] = {fx[0].value(), fx[1].value(), fy[0].value(), fy[1].value()};
      block_sum_n<4>(v, shf);
      if (t == 0)
#pragma unroll
        for (int k = 0; k < 4; k++) g[(long)k * nr] = v[k];
    } else {
      double v[2] = {fx[0].value(), fy[0].value()};
      block_sum_n<2>(v, shf);
      if (t == 0) { g[0] = v[0]; g[2 * (long)nr] = v[1]; }
    }
  }
}
template <typename T, int K> __global__ void __launch_bounds__(RING_LB(K)) k_cfl_ring(KArgs a) {
  cfl_ring<T, K, false>(a);
}
template <typename T, int K> __global__ void __launch_bounds__(RING_LB(K)) k_cfl_ring_sg(KArgs a) {
  cfl_ring<T, K, true>(a);
}

// Cash-Karp RK5 of the star+planet problem (src/RungeKunta.c:14-91), a planet
// per lane with its six stages in registers
__device__ __forceinline__ Body d_deriv_rk5(const Body &q, double dt, int n, int lane, bool feels_others,
                                            int indirect) {
  const double Di = sqrt(q.x * q.x + q.y * q.y);
  const double self = -DF_G * 1.0 / Di / Di / Di;
  Body d = {q.vx, q.vy, self * q.x, self * q.y, 0.0};
  for (int j = 0; j < n; j++) {
    const double xj = __shfl(q.x, j, 64), yj = __shfl(q.y, j, 64), mj = __shfl(q.m, j, 64);
    if (indirect) {
      const double Dj = __shfl(Di, j, 64), w = DF_G * mj / Dj / Dj / Dj;
      d.vx -= w * xj;
      d.vy -= w * yj;
    }
    if (n > 1 && j != lane && feels_others) {
      const double dist = sqrt((q.x - xj) * (q.x - xj) + (q.y - yj) * (q.y - yj));
      const double w = DF_G * mj / dist / dist / dist;
      d.vx += w * (xj - q.x);
      d.vy += w * (yj - q.y);
    }
  }
  return {d.x * dt, d.y * dt, d.vx * dt, d.vy * dt, 0.0};
}
template <int N> __device__ __forceinline__ Body d_translate(const Body &q, const Body (&k)[6], const double (&c)[N]) {
  Body r = q;
#pragma unroll
  for (int s = 0; s < N; s++) {
    if (c[s] == 0.0) continue;
    r.x += c[s] * k[s].x;
    r.y += c[s] * k[s].y;
    r.vx += c[s] * k[s].vx;
    r.vy += c[s] * k[s].vy;
  }
  return r;
}
__device__ Body d_rk5(const Body &q, double dt, int n, int lane, bool fo, int ind) {
  Body k[6];
  k[0] = d_deriv_rk5(q, dt, n, lane, fo, ind);
  const double c1[1] = {0.2};
  k[1] = d_deriv_rk5(d_translate<1>(q, k, c1), dt, n, lane, fo, ind);
  const double c2[2] = {0.075, 0.225};
  k[2] = d_deriv_rk5(d_translate<2>(q, k, c2), dt, n, lane, fo, ind);
  const double c3[3] = {0.3, -0.9, 1.2};
  k[3] = d_deriv_rk5(d_translate<3>(q, k, c3), dt, n, lane, fo, ind);
  const double c4[4] = {-11.0 / 54.0, 2.5, -70.0 / 27.0, 35.0 / 27.0};
  k[4] = d_deriv_rk5(d_translate<4>(q, k, c4), dt, n, lane, fo, ind);
  const double c5[5] = {1631.0 / 55296.0, 175.0 / 512.0, 575.0 / 13824.0, 44275.0 / 110592.0, 253.0 / 4096.0};
  k[5] = d_deriv_rk5(d_translate<5>(q, k, c5), dt, n, lane, fo, ind);
  const double c6[6] = {37.0 / 378.0, 0.0, 250.0 / 621.0, 125.0 / 594.0, 0.0, 512.0 / 1771.0};
  return d_translate<6>(q, k, c6);
}

// Scalar part of a sub-step, one block: the CFL reduction and sub-step dt
// (src/SourceEuler.c:443-470, 1485-1551), the gas indirect term and the
// barycentre acceleration (src/SideEuler.c:91-112), the potential
// parameters of FillForcesArrays (src/Pframeforce.c:44-90), and the planet
// update (AdvanceSystemFromDisk, AdvanceSystemRK5, RotatePsys).
// AccreteOntoPlanets (src/Planet.c:11-126) by the whole control workgroup
// once dt is known.  Each cell of a planet's window belongs to one thread,
// which updates its density in place.  The planet's mass and momentum gains
// are block sums over the accreted cells, and so are the changes of the
// disc's mass, barycentre and force sums: the CFL kernel formed those
// partials before the accretion, the reference forms them after it, and
// they are linear in the density.  At most one planet accretes (checked on
// the host), so no cell is accreted by two threads.  red holds 16 doubles
// per reduced value.
template <typename T>
__device__ void accrete_planets(const KArgs &a, dfargo_ctrl *c, double dt, double *sums, double *red) {
  const int t = threadIdx.x, TB = blockDim.x, lane = t & 63, wv = t >> 6, nw = TB >> 6;
  const int nr = a.nr, ns = a.ns, ntg = c->ntarget;
  constexpr int NV = 6 + 2 * DF_MAXTG;
  for (int k = 0; k < c->nb; k++) {
    if (!(c->pl_acc[k] > 1e-10)) continue;
    const double facc = dt * c->pl_acc[k], facc1 = 1.0 / 3.0 * facc, facc2 = 2.0 / 3.0 * facc;
    const double Xp = c->pl_x[k], Yp = c->pl_y[k], Mp = c->pl_m[k];
    const double Rp = sqrt(Xp * Xp + Yp * Yp), RRoche = pow((1.0 / 3.0 * Mp), (1.0 / 3.0)) * Rp;
    int i_min = 0, i_max = nr - 1;
    while ((i_min < nr) && (a.Rsup[i_min] < Rp - RRoche)) i_min++;
    while ((i_max > 0) && (a.Rinf[i_max] > Rp + RRoche)) i_max--;
    const double angle = atan2(Yp, Xp);
    const int j_min = (int)((double)ns / a.pm * (angle - 2.0 * RRoche / Rp - a.pmin));
    const int j_max = (int)((double)ns / a.pm * (angle + 2.0 * RRoche / Rp - a.pmin));
    const int wj = j_max - j_min + 1;
    const int ncell = (i_max >= i_min && wj > 0) ? (i_max - i_min + 1) * wj : 0;
    // 0-2: the planet's mass and momentum gains; 3-5: the disc's mass and
    // barycentre changes (per thread); then fx, fy per force target, summed
    // per wavefront after each chunk of TB cells into the wave's own slots
    // of red (few live registers: no spills in the control kernel)
    for (int q = t; q < NV * 16; q += TB) red[q] = 0.0;
    __syncthreads();
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int base = 0; base < ncell; base += TB) {
      const int idx = base + t;
      double dcm = 0.0, xc = 0.0, yc = 0.0;
      if (idx < ncell) {
        const int i = i_min + idx / wj, j = j_min + idx % wj;
        int jf = j % ns;
        jf = (jf < 0) ? jf + ns : jf;
        const long l = (long)i * ns + jf, lip = l + ns, ljp = (jf == ns - 1) ? (long)i * ns : l + 1;
        xc = a.Rmed[i] * a.CosAz[jf];
        yc = a.Rmed[i] * a.SinAz[jf];
        const double dx = Xp - xc, dy = Yp - yc, distance = sqrt(dx * dx + dy * dy);
        // the inner radius (0.45) lies inside the outer one (0.75)
        if (distance < 0.75 * RRoche) {
          const double vtcell = 0.5 * (ld<T>(a.vt, l) + ld<T>(a.vt, ljp)) + a.Rmed[i] * c->omega_frame;
          const double vrcell = 0.5 * (ld<T>(a.vr, l) + ld<T>(a.vr, lip));
          const double vxcell = (vrcell * xc - vtcell * yc) / a.Rmed[i];
          const double vycell = (vrcell * yc + vtcell * xc) / a.Rmed[i];
          const double d0 = ld<T>(a.rho, l);
          double dens = d0;
          double deltaM = facc1 * dens * a.Surf[i];
          dens *= (1.0 - facc1);
          v[0] += deltaM;
          v[1] += deltaM * vxcell;
          v[2] += deltaM * vycell;
          if (distance < 0.45 * RRoche) {
            deltaM = facc2 * dens * a.Surf[i];
            dens *= (1.0 - facc2);
            v[0] += deltaM;
            v[1] += deltaM * vxcell;
            v[2] += deltaM * vycell;
          }
          const T dstored = sr_round<T>(dens, sr_key(c, l, SR_ACC));
          ((T *)a.rho)[l] = dstored;
          // the change of the cell's mass as stored, in the partials' terms
          dcm = a.Surf[i] * ((double)dstored - d0);
          v[3] += dcm;
          v[4] += dcm * xc;
          v[5] += dcm * yc;
        }
      }
      for (int tg = 0; tg < ntg; tg++) {
        double fx = 0.0, fy = 0.0;
        if (dcm != 0.0) {
          const double ddx = xc - c->tg_x[tg], ddy = yc - c->tg_y[tg], rsm = c->tg_rsm[tg];
          const double dist2 = ddx * ddx + ddy * ddy + rsm * rsm, dd = sqrt(dist2);
          const double InvDist3 = 1.0 / dist2 / dd;
          fx = DF_G * dcm * ddx * InvDist3 * 1.0;
          fy = DF_G * dcm * ddy * InvDist3 * 1.0;
        }
        fx = wave_sum(fx);
        fy = wave_sum(fy);
        if (lane == 0) {
          red[(6 + 2 * tg) * 16 + wv] += fx;
          red[(7 + 2 * tg) * 16 + wv] += fy;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 6; q++) {
      const double w = wave_sum(v[q]);
      if (lane == 0) red[q * 16 + wv] = w;
    }
    __syncthreads();
    if (t == 0) {
      // the wavefronts' sums of value q, in wavefront order
      auto total = [&](int q) {
        double x = 0.0;
        for (int w = 0; w < nw; w++) x += red[q * 16 + w];
        return x;
      };
      double Px = Mp * c->pl_vx[k], Py = Mp * c->pl_vy[k], M = Mp;
      Px += total(1);
      Py += total(2);
      M += total(0);
      if (c->pl_feel_disk[k]) {
        c->pl_vx[k] = Px / M;
        c->pl_vy[k] = Py / M;
      }
      c->pl_m[k] = M;
      sums[2] += total(3);
      sums[3] += total(4);
      sums[4] += total(5);
      for (int tg = 0; tg < ntg; tg++) {
        sums[5 + 4 * tg] += total(6 + 2 * tg);
        sums[5 + 4 * tg + 2] += total(7 + 2 * tg);
      }
    }
    __syncthreads();
  }
}

__device__ void control_wave(const KArgs &a, dfargo_ctrl *c, const double *sums, double dt, double dtemp, int lane);

// Two builds: without accretion, 1024 threads; with it, 512, whose larger
// register budget keeps the accretion path and the n-body code free of spills.
//
// One workgroup between two grids: bound by its own latency.  All of its
// global reads (the control block, the rings' limits, the partials in batches
// of eight per lane) are issued before the loop condition is looked at, they
// meet in one barrier, and one wavefront does the rest with a planet per lane
// and its n-body stages in registers.  One thread with the stages in LDS and a
// load, an add and a wait per ring took 24 us at 200x400 with a free planet
// and 23 us at 1024 rings.
template <bool ACC> struct CtrlBlock { static constexpr int n = 1024; };
template <> struct CtrlBlock<true> { static constexpr int n = 512; };
template <typename T, bool ACC> __global__ void __launch_bounds__(CtrlBlock<ACC>::n) k_control(KArgs a) {
  constexpr int TB = CtrlBlock<ACC>::n, NWV = TB / 64;
  __shared__ double sums[DF_NPART(DF_MAXTG)];
  __shared__ double smin[NWV];
  __shared__ unsigned long long tsw[NWV];
  // The control block is staged in LDS for the kernel's run: the part below
  // reads and writes dozens of its fields in dependent order, which from
  // global memory costs a memory latency each.  It is copied in and back by
  // all threads; no kernel that may run beside this one writes the block
  // (the self-gravity transforms only read its go flag, which this kernel
  // leaves as it is).
  __shared__ dfargo_ctrl cs;
  constexpr int NW = (int)(sizeof(dfargo_ctrl) / 8);
  static_assert(sizeof(dfargo_ctrl) % 8 == 0 && NW <= TB, "the control block is copied as 8-byte words, one a thread");
  dfargo_ctrl *const cg = a.ctrl;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nr = a.nr, ns = a.ns;
  const int go = cg->go, NP = DF_NPART(cg->ntarget);
  const unsigned long long word = t < NW ? ((const unsigned long long *)cg)[t] : 0ull;
  double nd = 1e30;
  for (int i = t; i < nr; i += TB) {
    double v = i > 0 ? a.ring_dt[i] : 1e30;
    // with the dust fluid each cell's limit is max2(min2(dtg, dtd), 1e-10)
    // (src/SourceEuler.c:1462-1465); both maps are monotone, so per ring
    if (a.df_on && i > 0) v = dmax2(dmin2(v, a.df_ring_dt[i]), 1.e-10);
    nd = dmin2(nd, v);
    if (i < nr - 1) {
      const double w0 = a.InvRmed[i], w1 = a.InvRmed[i + 1];
      v = a.pm * DF_CFLSECURITY / (double)ns / fabs(a.vmoy[i] * w0 - a.vmoy[i + 1] * w1);
      nd = dmin2(nd, v);
      // the dust fluid's shear limit (src/SourceEuler.c:1486-1491)
      if (a.df_on && !a.df_sfta) {
        v = a.pm * DF_CFLSECURITY / (double)ns / fabs(a.dvmoy[i] * w0 - a.dvmoy[i + 1] * w1);
        nd = dmin2(nd, v);
      }
    }
  }
  // minimum stopping time of the last particle interpolation (reset to 1e6
  // at each interpolation, src/Dsys.c:300): the minimum of the per-block
  // minima, compared as bit patterns of positive doubles
  const bool ts_limit = a.d_on && a.d_np > 0 && a.d_feedback;
  unsigned long long ts = (unsigned long long)__double_as_longlong(1e6);
  if (ts_limit) {
    const int nblk = (a.d_np + 255) / 256;
    for (int b = t; b < nblk; b += TB) ts = (a.p_tsmin[b] < ts) ? a.p_tsmin[b] : ts;
  }
  // each wavefront sums whole partials: lanes stride the rings with a
  // compensated sum, then a fixed tree (deterministic)
  double psum[(DF_NPART(DF_MAXTG) + NWV - 1) / NWV];
#pragma unroll
  for (int r = 0; r < (DF_NPART(DF_MAXTG) + NWV - 1) / NWV; r++) {
    const int p = wave + r * NWV;
    psum[r] = 0.0;
    if (p >= NP) continue;
    const double *src = a.ring_part + (long)p * nr;
    CSum s = {0, 0};
    for (int i0 = 0; i0 < nr; i0 += 8 * 64) {
      double x[8];
#pragma unroll
      for (int q = 0; q < 8; q++) x[q] = (i0 + q * 64 + lane < nr) ? src[i0 + q * 64 + lane] : 0.0;
#pragma unroll
      for (int q = 0; q < 8; q++) s.add(x[q]);
    }
    psum[r] = s.value();
  }
  if (!go) {
    if (t == 0) cg->active = 0;
    return;
  }
  if (t < NW) ((unsigned long long *)&cs)[t] = word;
  nd = wave_min(nd);
  if (lane == 0) smin[wave] = nd;
  if (ts_limit) {
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned long long o = (unsigned long long)__shfl_xor((long)ts, off, 64);
      ts = (o < ts) ? o : ts;
    }
    if (lane == 0) tsw[wave] = ts;
  }
#pragma unroll
  for (int r = 0; r < (DF_NPART(DF_MAXTG) + NWV - 1) / NWV; r++) {
    const int p = wave + r * NWV;
    if (p >= NP) continue;
    const double v = wave_sum(psum[r]);
    if (lane == 0) sums[p] = v;
  }
  __syncthreads();
  dfargo_ctrl *const c = &cs;
  __shared__ double s_dt;
  if (wave == 0) {
    // sub-step dt
    double dt;
    int gts = c->gas_timesteps_cfl;
    if (!a.d_fixed_dt) {
      nd = wave_min(lane < NWV ? smin[lane] : 1e30);
      const double deltaT = c->DT - c->dtemp;
      // the minimum stopping time of the last interpolation, resolved by two
      // steps (src/SourceEuler.c:1501-1507)
      if (ts_limit) {
        unsigned long long m = tsw[0];
        for (int w = 1; w < NWV; w++) m = (tsw[w] < m) ? tsw[w] : m;
        double dt_fb = 0.5 * __longlong_as_double((long long)m);
        if (dt_fb == 0.0) dt_fb = 1e10;
        if (dt_fb < nd) nd = dt_fb;
      }
      if (deltaT < nd) nd = deltaT;
      gts = (int)(ceil(deltaT / nd));
      const double dthydro = deltaT / (double)gts;
      dt = dmin2(dthydro, c->dtnbody);
    } else {
      // the particles' fixed time step (src/SourceEuler.c:457-463)
      dt = a.d_dust_timestep;
    }
    const double dtemp = c->dtemp + dt;
    if (lane == 0) {
      c->gas_timesteps_cfl = gts;
      if (a.d_fixed_dt) c->mindt = c->maxdt = dt;
      c->dtemp = dtemp;
      if (dt < c->mindt) c->mindt = dt;
      if (dt > c->maxdt) c->maxdt = dt;
      c->dt = dt;
      s_dt = dt;
    }
    if constexpr (!ACC) control_wave(a, c, sums, dt, dtemp, lane);
  }
  if constexpr (ACC) {
    // AccreteOntoPlanets right after dt (src/SourceEuler.c:454)
    __shared__ double red[(6 + 2 * DF_MAXTG) * 16];
    __syncthreads();
    accrete_planets<T>(a, c, s_dt, sums, red);
    __syncthreads();
    if (wave == 0) control_wave(a, c, sums, s_dt, c->dtemp, lane);
  }
  __syncthreads();
  if (t < NW) ((unsigned long long *)cg)[t] = ((const unsigned long long *)&cs)[t];
}

// The part of the control kernel one wavefront does on the LDS copy c of the
// control block, a planet per lane: crash flags, indirect terms, barycentre,
// FillForcesArrays' parameters, AdvanceSystemFromDisk, AdvanceSystemRK5, the
// frame and the loop condition.  What is not a planet's is formed by every
// lane and stored by lane 0.
// The call's time dtemp after this sub-step comes as an argument: a lane must
// not read back what lane 0 stores here.
__device__ void control_wave(const KArgs &a, dfargo_ctrl *c, const double *sums, double dt, double dtemp, int lane) {
  const int nb = c->nb;
  const bool planet = lane < nb;
  const double time = c->time;
  // gas indirect term: ComputeAccel(star), src/SideEuler.c:282-298
  const double *g0 = sums + 5;
  const double dop_x = a.exclude_hill ? g0[1] : g0[0], dop_y = a.exclude_hill ? g0[3] : g0[2];
  // barycentre (src/SideEuler.c:42-112)
  const double total = sums[2];
  const double bx = sums[3] / (1.0 + total), by = sums[4] / (1.0 + total);
  const double dopalt_x = -(bx - 2.0 * c->barx[1] + c->barx[0]) / (dt * dt);
  const double dopalt_y = -(by - 2.0 * c->bary[1] + c->bary[0]) / (dt * dt);
  double ind_x = -dop_x, ind_y = -dop_y;
  if (a.alt_indirect) {
    ind_x = -dopalt_x;
    ind_y = -dopalt_y;
  }
  if (!a.indirect_term) {
    ind_x = 0.0;
    ind_y = 0.0;
  }
  if (lane == 0) {
    c->omega_prev = c->omega_frame;
    c->crashed_d = sums[0] > 0.0;
    // an isothermal disc has no energy to scan (its partials are not formed)
    c->crashed_e = a.energy && sums[1] > 0.0;
    c->dop_x = dop_x;
    c->dop_y = dop_y;
    c->dopalt_x = dopalt_x;
    c->dopalt_y = dopalt_y;
    c->barx[0] = c->barx[1]; c->barx[1] = bx; c->barx[2] = bx;
    c->bary[0] = c->bary[1]; c->bary[1] = by; c->bary[2] = by;
    c->ind_x = ind_x;
    c->ind_y = ind_y;
  }
  // FillForcesArrays parameters
  double planetmass_taper = 1.0;
  if (a.mass_taper_param > 1e-2) {
    const double mt = (time - c->time0) / (a.mass_taper_param * 2.0 * DF_PI);
    planetmass_taper = (mt > 1.0 ? 1.0 : .5 * (1.0 - cos(DF_PI * mt)));
  }
  Body b = load_body(c, lane);
  if (planet) {
    const double mp = b.m * planetmass_taper, PlanetDistance = sqrt(b.x * b.x + b.y * b.y);
    const double sm = a.roche ? PlanetDistance * pow((1.0 / 3.0 * mp), 1.0 / 3.0) * a.roche_smoothing
                              : d_smoothing(a, PlanetDistance);
    c->pot_x[lane] = b.x;
    c->pot_y[lane] = b.y;
    c->pot_m[lane] = mp;
    c->pot_invd3[lane] = 1.0 / PlanetDistance / PlanetDistance / PlanetDistance;
    c->pot_smooth[lane] = sm * sm;
  }
  // the corotating frame's mark (src/SourceEuler.c:476), before the
  // disc's kick changes the velocities
  if (a.frame && lane == 0) psys_info(a, c, 0);
  double omega_frame = c->omega_frame;
  // AdvanceSystemFromDisk (src/Pframeforce.c:131-161)
  for (int tg = 1; tg < c->ntarget; tg++) {
    if (c->tg_planet[tg] != lane) continue;
    const double *g = sums + 5 + 4 * tg;
    const double gx = a.exclude_hill ? g[1] : g[0], gy = a.exclude_hill ? g[3] : g[2];
    b.vx += dt * gx;
    b.vy += dt * gy;
    b.vx += dt * ind_x;
    b.vy += dt * ind_y;
  }
  // AdvanceSystemRK5 (src/Pframeforce.c:163-266)
  if (nb > 0) {
    const bool moves = planet && lane >= 1 - (time >= a.release_date);
    if (!a.forced_circular) {
      const Body q = d_rk5(b, dt, nb, lane, planet && c->pl_feel_others[lane], a.indirect_term);
      if (moves) b = q;
    } else if (moves) {
      const double theta = atan2(b.y, b.x);
      const double r = sqrt(b.x * b.x + b.y * b.y), v = sqrt(b.vx * b.vx + b.vy * b.vy);
      const double omega = (-b.y * b.vx + b.x * b.vy) / r / r, dtheta = omega * dt;
      double sn, cn;
      sincos(theta + dtheta, &sn, &cn);
      b.x = r * cn;
      b.y = r * sn;
      b.vx = -v * sn;
      b.vy = v * cn;
    }
    if (lane == 0 && time < a.release_date) {
      const double x = b.x, y = b.y, r = sqrt(x * x + y * y), theta = atan2(y, x);
      const double rdot = (a.release_radius - r) / (a.release_date - time);
      const double omega = sqrt((1. + b.m) / r / r / r), new_r = r + rdot * dt, denom = r - new_r;
      const double dtheta = (denom != 0.0) ? 2. * dt * r * omega / denom * (sqrt(r / new_r) - 1.) : omega * dt;
      const double vx = rdot, vy = new_r * sqrt((1. + b.m) / new_r / new_r / new_r);
      const double cn = cos(dtheta + theta), sn = sin(dtheta + theta);
      b.x = new_r * cn;
      b.y = new_r * sn;
      b.vx = vx * cn - vy * sn;
      b.vy = vx * sn + vy * cn;
    }
    // the frame follows its centre (src/SourceEuler.c:516-524); the
    // source kernel applies CorrectVtheta (vt -= domega Rmed) where it
    // reads vt
    if (a.frame) {
      if (planet) {
        c->pl_x[lane] = b.x; c->pl_y[lane] = b.y;
        c->pl_vx[lane] = b.vx; c->pl_vy[lane] = b.vy;
      }
      __threadfence_block();
      double omega_new = 0.0;
      if (lane == 0) {
        omega_new = psys_info(a, c, 1) / dt;
        c->domega = omega_new - omega_frame;
        c->omega_frame = omega_new;
      }
      omega_frame = __shfl(omega_new, 0, 64);
    }
    if (planet) {
      // the particles of this sub-step feel the planets where the n-body
      // step left them (src/SourceEuler.c:504-513 come before RotatePsys)
      if (a.d_on) {
        // distance, azimuth and smoothing length, once for all particles
        const double rpl = sqrt(b.x * b.x + b.y * b.y);
        c->dust_pl_r[lane] = rpl;
        c->dust_pl_t[lane] = atan2(b.y, b.x);
        c->dust_pl_eps[lane] = a.thickness_smoothing * a.aspect_ratio * pow(0.5 * rpl, 1.0 + a.flaring) *
                               pow(2.0, 1.0 + a.flaring);
      }
      // RotatePsys (src/Psys.c:352-370)
      const double angle = omega_frame * dt;
      if (angle != 0.0) {
        double sint, cost;
        sincos(angle, &sint, &cost);
        double xt = b.x, yt = b.y;
        b.x = xt * cost + yt * sint;
        b.y = -xt * sint + yt * cost;
        xt = b.vx;
        yt = b.vy;
        b.vx = xt * cost + yt * sint;
        b.vy = -xt * sint + yt * cost;
      }
      c->pl_x[lane] = b.x; c->pl_y[lane] = b.y;
      c->pl_vx[lane] = b.vx; c->pl_vy[lane] = b.vy;
      // masses of this sub-step for the particle kernels
      if (a.d_on) c->dust_pl_m[lane] = b.m;
    }
  }
  // PhysicalTime += dt closes the sub-step (src/SourceEuler.c:714); every
  // other use of PhysicalTime in the sub-step is above
  const int go_next = dtemp < 0.999999999 * c->DT;
  if (lane == 0) {
    c->time = time + dt;
    c->substeps += 1;
    c->substeps_total += 1;
    c->active = 1;
    if (a.d_on) {
      // ... and a fresh minimum for their interpolation (src/Dsys.c:300)
      c->dust_mp = c->particles_mass;
      c->out_count = 0;
    }
    // loop condition and start of the next sub-step
    c->go_next = go_next;
  }
  if (go_next) begin_substep(a, c, b, time + dt, lane);
}

// ComputeSoundSpeed at the start of AlgoGas (src/SourceEuler.c:2340); in
// the sub-steps the CFL kernel recomputes cs with its ring means
template <typename T, int K> __global__ void __launch_bounds__(RING_LB(K)) k_eos(KArgs a) {
  const int i = ring_of_block(a), ns = a.ns, t = threadIdx.x, TB = ns / K;
  if (t >= TB) return;
  const long base = (long)i * ns;
  const double g = a.gamma;
#pragma unroll
  for (int k = 0; k < K; k++) {
    const long l = base + t + k * TB;
    st<T>(a.cs, l, sqrt(g * (g - 1.0) * ld<T>(a.en, l) / ld<T>(a.rho, l)));
  }
}

// ComputeViscousTerms stresses (src/Viscosity.c:159-300) on (vr, vt)
template <typename T>
__device__ void visc_stress_cell(const KArgs &a, const void *vr, const void *vt, int i, int j,
                                 double *Trr, double *Tpp, double *Trp, double *divv) {
  const int ns = a.ns;
  const long l = (long)i * ns + j, lip = l + ns, ljp = (j == ns - 1) ? (long)i * ns : l + 1;
  const double onethird = 1.0 / 3.0, nu = a.nu_ring[i];
  double vrl = ld<T>(vr, l), vrp = ld<T>(vr, lip), vtl = ld<T>(vt, l), vtp = ld<T>(vt, ljp);
  double dv = (vrp * a.Rsup[i] - vrl * a.Rinf[i]) * a.InvDiffRsup[i] * a.InvRmed[i];
  dv += (vtp - vtl) * a.invdphi * a.InvRmed[i];
  double Drr = (vrp - vrl) * a.InvDiffRsup[i];
  double Dpp = (vtp - vtl) * a.invdphi * a.InvRmed[i] + 0.5 * (vrp + vrl) * a.InvRmed[i];
  double rho = ld<T>(a.rho, l);
  *Trr = 2.0 * rho * nu * (Drr - onethird * dv);
  *Tpp = 2.0 * rho * nu * (Dpp - onethird * dv);
  *divv = dv;
  if (i >= 1) {
    const long lim = l - ns, ljm = (j == 0) ? (long)i * ns + ns - 1 : l - 1, ljmim = ljm - ns;
    double Drp = 0.5 * (a.Rinf[i] * (vtl * a.InvRmed[i] - ld<T>(vt, lim) * a.InvRmed[i - 1]) *
                            a.InvDiffRmed[i] +
                        (vrl - ld<T>(vr, ljm)) * a.invdphi * a.InvRinf[i]);
    *Trp = 2.0 * 0.25 * (rho + ld<T>(a.rho, lim) + ld<T>(a.rho, ljm) + ld<T>(a.rho, ljmim)) * nu * Drp;
  } else {
    *Trp = 0.0;
  }
}

// stresses of the current state, for the diagnostics outside a sub-step
template <typename T> __global__ void __launch_bounds__(256) k_visc_stress(KArgs a, int from_state) {
  const int i = blockIdx.y, ns = a.ns, j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ns) return;
  const long l = (long)i * ns + j;
  double Trr, Tpp, Trp, dv;
  visc_stress_cell<T>(a, from_state ? a.vr : a.vri, from_state ? a.vt : a.vti, i, j, &Trr, &Tpp, &Trp, &dv);
  st<T>(a.trr, l, Trr);
  st<T>(a.tpp, l, Tpp);
  st<T>(a.trp, l, Trp);
}

// The source and transport kernels hold a ring's cells in wavefronts: 64
// consecutive cells a wavefront, one a lane.  The values of neighbouring cells
// are neighbouring lanes', so each step that reads them leaves fewer valid
// cells at either end; after the source terms (SubStep1, the stresses, the
// viscous update, SubStep2: one cell each) and after the transport's two
// azimuthal passes (two cells each) the middle 56 are complete, which the
// wavefront owns.
#define AZ_LANES 64
#define AZ_HALO 4
#define AZ_OWN (AZ_LANES - 2 * AZ_HALO)
static_assert(AZ_OWN == DF_SRC_COLS, "the source kernel leaves one partial sum per wavefront");

// The neighbouring lanes' values: lane L receives lane L - 1's (prev) or
// lane L + 1's (next); the end lanes receive zeros, which only feed cells
// outside the valid range.  CDNA's whole-wavefront DPP shifts (wave_shr:1,
// wave_shl:1) move each 32-bit half in one VALU operation, without the LDS
// crossbar of a general lane permute; with zeros for the end lanes the move
// needs no copy of its destination first.
template <int CTRL> __device__ __forceinline__ double dpp_shift(double v) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true));
}
#define DPP_WAVE_SHL1 0x130
#define DPP_WAVE_SHR1 0x138
__device__ __forceinline__ double lane_prev(double v) { return dpp_shift<DPP_WAVE_SHR1>(v); }
__device__ __forceinline__ double lane_next(double v) { return dpp_shift<DPP_WAVE_SHL1>(v); }

// The operations' order is that of the reference, whatever the storage type.
// Over thousands of sub-steps of a nearly steady flow another order of the
// products and sums drifts from it by more than 1e-12; and particles that read
// the nearest cell turn a single FP32 cell that rounds the other way into a
// different run (a grain by an edge reads another cell, and its drag acts on
// that one).  Three groups of operations are not the reference's own: a Work
// value is Q times 1 / (rho + 1e-20), an elongation (vt dt) (1 / dt), an
// azimuthal slope a product with 1 / dxtheta; and a division is div_nr.

// 1 / b to within an ulp, and with it the quotients a / b of that divisor:
// div_nr's steps, shared where several quotients have one divisor
__device__ __forceinline__ double rcp_nr(double b) {
  double r = __builtin_amdgcn_rcp(b);
  r = fma(r, fma(-b, r, 1.0), r);
  return fma(r, fma(-b, r, 1.0), r);
}
__device__ __forceinline__ double quotient(double a, double b, double r) {
  const double q = a * r;
  return fma(r, fma(-b, q, a), q);
}

// lane k's value (k uniform); only where every lane is active
__device__ __forceinline__ double lane_value(double v, int k) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), k),
                          __builtin_amdgcn_readlane(__double2loint(v), k));
}
// Source terms of one sub-step: SubStep1 (src/SourceEuler.c:865-994, with the
// self-gravity kick of update_sgvelocity, src/sgupdate.c:30-72), the viscous
// stresses and velocity update (ComputeViscousTerms +
// UpdateVelocitiesWithViscosity, src/Viscosity.c:159-378) and SubStep2
// (src/SourceEuler.c:1012-1116), in that order.  A wavefront walks outwards
// through a strip of S rings with one column a lane: having read ring r it forms
// VradInt / VthetaInt of ring r, the stresses and the viscous update of VradInt
// of ring r - 1, and the viscous update of VthetaInt and SubStep2 of ring r - 2,
// whose inputs are then complete.  Every value is formed once per column, is
// kept in registers as long as the rings above need it, and comes from the
// neighbouring columns by lane moves.  The state is read only; the
// post-SubStep2 velocities go to vri / vti and the energy to e_int (the
// ActualiseGas copies of src/SourceEuler.c:598-630 are deferred to the end of
// the sub-step), so no wavefront overwrites what another one still reads.
//
// VALU issue bounds it first (66-76 % of the time at 1024x3072), then the latency
// that three or four wavefronts a SIMD leave uncovered.  As tiles in LDS with a
// halo per stage the potential was formed 1.9 times a cell (8 rings, FP64) and
// every operand went through LDS behind a barrier: 121 us at 1024x3072 FP64, 98 us
// FP32 with self-gravity; now 64 and 71 us.  The quotients by the sums of
// neighbouring densities (six a cell) share two reciprocals.
//
// Rings at a strip's ends take only the stages that its own rings need.
//
// X: the less used terms, SRC_FRAME a corotating frame and the dust fluid's drag
// on the gas, SRC_DUST particles (and a frame), whose switches and grids
// otherwise take the scalar registers of every disc's loop; E: the energy
// equation.
enum { SRC_PLAIN = 0, SRC_FRAME = 1, SRC_DUST = 2 };
#define SRC_STRIP_MAX 32
// wavefronts per SIMD: the registers of all but the plainest kernel exceed a
// fourth wavefront's budget of 128
constexpr int src_occupancy(bool fp64, bool E, int X) { return (fp64 || E || X != SRC_PLAIN) ? 3 : 4; }

// the state of one cell of the newest ring, as stored; x: the particles'
// feedback accelerations, or the dust fluid's Stokes number, density and
// velocities where it drags the gas
template <typename T> struct SrcRaw {
  T rho, vt, vr, en, sgr, sgt, x[4];
};
template <typename T, bool E, int X> __device__ __forceinline__ SrcRaw<T> src_load(const KArgs &a, int r, int j) {
  const long l = (long)r * a.ns + j;
  SrcRaw<T> q;
  q.rho = ((const T *)a.rho)[l];
  q.vt = ((const T *)a.vt)[l];
  q.vr = ((const T *)a.vr)[l];
  q.en = E ? ((const T *)a.en)[l] : (T)0;
  q.sgr = q.sgt = (T)0;
  if (a.sg) {
    q.sgr = ((const T *)a.sgr)[l];
    q.sgt = ((const T *)a.sgt)[l];
  }
  q.x[0] = q.x[1] = q.x[2] = q.x[3] = (T)0;
  if constexpr (X == SRC_DUST) {
    if (a.d_feedback) {
      q.x[0] = ((const T *)a.radfbacc)[l];
      q.x[1] = ((const T *)a.azifbacc)[l];
    }
  }
  if constexpr (X == SRC_FRAME) {
    if (DF_ON(T, a) && a.df_feedback) {
      q.x[0] = (T)a.dstokes[l];
      q.x[1] = (T)a.drho[l];
      q.x[2] = (T)a.dvr[l];
      q.x[3] = (T)a.dvt[l];
    }
  }
  return q;
}
// the ring tables: ring rb + k in lane k (zero outside the grid), and one ring's
struct SrcTab {
  double idrm, rinf, irinf, rmed, supp, idxt, nu, rsup, idrs, irmed, cs, r15;
};
__device__ __forceinline__ SrcTab src_tables(const KArgs &a, int i, bool in) {
  const int k = in ? i : 0;
  SrcTab t = {a.InvDiffRmed[k], a.Rinf[k], a.InvRinf[k],      a.Rmed[k],    a.supp_torque[k], a.InvDxTheta[k],
              a.nu_ring[k],     a.Rsup[k], a.InvDiffRsup[k], a.InvRmed[k], a.cs_iso[k],      a.r15[k]};
  if (!in) t = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  return t;
}
__device__ __forceinline__ SrcTab src_table_of(const SrcTab &t, int k) {
  return {lane_value(t.idrm, k), lane_value(t.rinf, k), lane_value(t.irinf, k), lane_value(t.rmed, k),
          lane_value(t.supp, k), lane_value(t.idxt, k), lane_value(t.nu, k),    lane_value(t.rsup, k),
          lane_value(t.idrs, k), lane_value(t.irmed, k), lane_value(t.cs, k),   lane_value(t.r15, k)};
}

template <typename T, bool E, int X>
__global__ void __launch_bounds__(256, src_occupancy(sizeof(T) == 8, E, X)) k_source(KArgs a, int S) {
  const dfargo_ctrl *c = a.ctrl;
  if (!c->active) return;
  const int ns = a.ns, nr = a.nr, lane = threadIdx.x & (AZ_LANES - 1), per = blockDim.x / AZ_LANES;
  // the particles of this sub-step were re-sorted into the other set
  if (X == SRC_DUST && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) a.ctrl->pset ^= 1;
  // the blocks of one XCD take neighbouring segments and strips (ring_of_block)
  const int nb = gridDim.x * gridDim.y, b0 = blockIdx.y * gridDim.x + blockIdx.x;
  const int b = (a.xcd_remap && nb % 8 == 0) ? (b0 % 8) * (nb / 8) + b0 / 8 : b0;
  const int seg = __builtin_amdgcn_readfirstlane((b % gridDim.x) * per + threadIdx.x / AZ_LANES);
  const int i0 = (b / gridDim.x) * S, i1 = (i0 + S < nr) ? i0 + S : nr;
  if (seg * AZ_OWN >= ns) return; // a whole wavefront
  int j = (seg * AZ_OWN - AZ_HALO + lane) % ns;
  if (j < 0) j += ns;
  const int own = lane - AZ_HALO;
  const bool store = own >= 0 && own < AZ_OWN && seg * AZ_OWN + own < ns;
  const int rb = (i0 - 3 > 0) ? i0 - 3 : 0;
  SrcRaw<T> next = src_load<T, E, X>(a, rb, j);
  const SrcTab tabs = src_tables(a, rb + lane, rb + lane < nr);
  const double cosj = a.CosAz[j], sinj = a.SinAz[j];
  // the planets, planet k in lane k
  const int npl = c->nb, lp = lane < npl ? lane : 0;
  const double pX = c->pot_x[lp], pY = c->pot_y[lp], pM = c->pot_m[lp], pS = c->pot_smooth[lp], pI = c->pot_invd3[lp];
  const double dt = c->dt, invdt = 1.0 / dt, Of = c->omega_frame, ind_x = c->ind_x, ind_y = c->ind_y;
  const double invdphi = a.invdphi, g1 = a.gamma - 1.0, C2 = DF_CVNR * DF_CVNR, onethird = 1.0 / 3.0;
  const bool frame_trip = X == SRC_DUST && a.d_np > 0 && c->omega_prev != 0.0;
  // the change of the corotating frame's rate this sub-step
  const bool frame = X != SRC_PLAIN && a.frame;
  const double omega_prev = c->omega_prev, dom = frame ? c->domega : 0.0;
  const int ntile = (ns + DF_SRC_COLS - 1) / DF_SRC_COLS;
  const unsigned f_vr = sr_field(c, SR_VR), f_vt = sr_field(c, SR_VT), f_e = sr_field(c, SR_E);
  const SrcTab zero_tab = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  // ring s = r - 1: the state, its density to the left, the reciprocals of the
  // density sums across its inner and left face, VradInt, VthetaInt
  double s_rho = 1.0, s_rhojm = 1.0, s_rr = 0.0, s_rt = 0.0, s_vr = 0.0, s_vt = 0.0, s_en = 0.0;
  double s_p = 0.0, s_pot = 0.0, s_ip = 0.0, s_vt0 = 0.0, s_vtn0 = 0.0, s_sgr = 0.0;
  SrcTab ts = zero_tab;
  // ring t = r - 2: the same, VradInt after viscosity, the stresses, SubStep2's
  // radial pressure of ring t - 1
  double t_rho = 1.0, t_rhojm = 1.0, t_rr = 0.0, t_rt = 0.0, t_vr = 0.0, t_vt = 0.0, t_en = 0.0;
  double t_trr = 0.0, t_tpp = 0.0, t_trp = 0.0, u_rho = 1.0, u_qr = 0.0;
  SrcTab tt = zero_tab;
  for (int r = rb; r <= i1 + 1; r++) {
    const SrcRaw<T> raw = next;
    if (r + 1 < nr && r <= i1) next = src_load<T, E, X>(a, r + 1, j);
    const SrcTab tr = src_table_of(tabs, r - rb);
    const int s = r - 1, t = r - 2;
    // SubStep1 at ring r (VradInt and VthetaInt of ring nrad are zero, as in
    // the reference where they are never set)
    const double rho = (double)raw.rho, rhojm = lane_prev(rho), en = (double)raw.en;
    const double sum_r = rho + s_rho, sum_t = rho + rhojm;
    const double rr = rcp_nr(sum_r), rt = rcp_nr(sum_t);
    double vt0 = (double)raw.vt;
    if (frame_trip) {
      // the particles' interpolation holds vt + Rmed OmegaFrame in the gas
      // grid and subtracts it again (src/Dsys.c:316,1082): SubStep1 reads
      // the round trip's result
      const double rw = tr.rmed * omega_prev;
      vt0 = (double)(T)((vt0 + rw) - rw);
    }
    const double vtn0 = lane_next(vt0), sgr = (double)raw.sgr;
    const double cs = (double)(T)tr.cs, p = E ? g1 * en : rho * cs * cs;
    // the potential (pot_at)
    double pot = 0.0, ip = 0.0;
    {
      const double x = tr.rmed * cosj, y = tr.rmed * sinj;
      for (int k = 0; k < npl; k++) {
        const double xp = lane_value(pX, k), yp = lane_value(pY, k), mp = lane_value(pM, k);
        const double distance = (x - xp) * (x - xp) + (y - yp) * (y - yp);
        double pk = div_nr(-DF_G * mp, sqrt(distance + lane_value(pS, k)));
        if (a.indirect_term) pk += DF_G * mp * lane_value(pI, k) * (x * xp + y * yp);
        pot += pk;
      }
      double ps = -DF_G * 1.0 * tr.irmed;
      const double gi = ind_x * x + ind_y * y;
      if (a.gas_indirect) ps -= gi;
      pot += ps;
      // its indirect part as the particles feel it (the IndPot grid of
      // FillForcesArrays, src/Pframeforce.c:60-88): the planets' term is
      // assigned, not summed, so the last planet's stands, as in the reference
      if (X == SRC_DUST) {
        if (a.indirect_term && a.d_feel_planets && npl > 0)
          ip = DF_G * lane_value(pM, npl - 1) * lane_value(pI, npl - 1) *
               (x * lane_value(pX, npl - 1) + y * lane_value(pY, npl - 1));
        if (a.gas_indirect && a.d_feel_disk) ip -= gi;
      }
    }
    const double ipjm = X == SRC_DUST ? lane_prev(ip) : 0.0;
    double vr1 = 0.0, vt1 = 0.0;
    const double pljm = lane_prev(p), potjm = lane_prev(pot), sgtjm = a.sg ? lane_prev((double)raw.sgt) : 0.0;
    if (r < nr && r >= i0 - 2) {
      const long l = (long)r * ns + j;
      // the particles' grids (pressure gradients, indirect and self-gravity
      // accelerations, src/SourceEuler.c:893-948) on the wavefront's own cells
      const bool dgrid = X == SRC_DUST && store && r >= i0 && r < i1;
      if (r >= 1) {
        const double gradp = quotient((p - s_p) * 2.0, sum_r, rr) * tr.idrm;
        const double gradphi = (pot - s_pot) * tr.idrm;
        double vt2;
        if (frame) {
          // CorrectVtheta (src/SideEuler.c:1133-1148) on the values read
          const double ci = dom * tr.rmed, cim = dom * ts.rmed;
          vt2 = (vt0 - ci) + (vtn0 - ci) + (s_vt0 - cim) + (s_vtn0 - cim);
        } else {
          vt2 = vt0 + vtn0 + s_vt0 + s_vtn0;
        }
        vt2 = vt2 / 4.0 + tr.rinf * Of;
        vt2 = vt2 * vt2;
        vr1 = (double)raw.vr + dt * (-gradp - gradphi + vt2 * tr.irinf);
        if (X == SRC_DUST && a.d_feedback) vr1 += dt * (double)raw.x[0];
        if (X == SRC_FRAME && DF_ON(T, a) && a.df_feedback) {
          // the dust fluid's drag on the gas, implicit (src/SourceEuler.c:915-921)
          const double st = (double)raw.x[0] * tr.r15, eps = div_nr((double)raw.x[1], rho);
          vr1 = div_nr(vr1 * st + eps * (double)raw.x[2] * dt, st + dt * eps);
        }
        if (dgrid) {
          st<T>(a.radgradp, l, (p - s_p) * tr.idrm);
          if (a.indirect_term)
            st<T>(a.radindacc, l, -(ip - s_ip) * tr.idrm);
        }
        if (a.sg) {
          const double radsgacc = ((tr.rinf - ts.rmed) * sgr + (tr.rmed - tr.rinf) * s_sgr) * tr.idrm;
          if (dgrid) st<T>(a.radsgacc, l, radsgacc);
          vr1 = vr1 + dt * radsgacc;
        }
      }
      const double gradp = quotient((p - pljm) * 2.0, sum_t, rt) * tr.idxt;
      const double gradphi = (pot - potjm) * tr.idxt;
      vt1 = vt0;
      if (frame) vt1 = vt1 - dom * tr.rmed;
      vt1 = vt1 - dt * (gradp + gradphi);
      vt1 += dt * tr.supp;
      if (X == SRC_DUST && a.d_feedback) vt1 += dt * (double)raw.x[1];
      if (X == SRC_FRAME && DF_ON(T, a) && a.df_feedback) {
        // src/SourceEuler.c:991-997, with the dust's vtheta after CorrectVtheta
        const double st = (double)raw.x[0] * tr.r15, eps = div_nr((double)raw.x[1], rho);
        const double dvtl = frame ? (double)raw.x[3] - dom * tr.rmed : (double)raw.x[3];
        vt1 = div_nr(vt1 * st + eps * dvtl * dt, st + dt * eps);
      }
      if (dgrid) {
        st<T>(a.azigradp, l, (p - pljm) * tr.idxt);
        if (a.indirect_term)
          st<T>(a.aziindacc, l, -(ip - ipjm) * tr.idxt);
      }
      if (a.sg) {
        const double azisgacc = 0.5 * ((double)raw.sgt + sgtjm);
        if (dgrid) st<T>(a.azisgacc, l, azisgacc);
        vt1 = vt1 + dt * azisgacc;
      }
    }
    // the stresses of ring s, then VradInt of ring s and VthetaInt of ring t
    double trr = 0.0, tpp = 0.0, trp = 0.0, vs = s_vr, vtt = t_vt;
    if (a.visc_on) {
      if (s >= 0 && s >= i0 - 2 && s < nr) {
        const double vtnx = lane_next(s_vt);
        double dv = (vr1 * ts.rsup - s_vr * ts.rinf) * ts.idrs * ts.irmed;
        dv += (vtnx - s_vt) * invdphi * ts.irmed;
        const double Drr = (vr1 - s_vr) * ts.idrs;
        const double Dpp = (vtnx - s_vt) * invdphi * ts.irmed + 0.5 * (vr1 + s_vr) * ts.irmed;
        // the stresses round to storage, as the grids of them that are read
        // between sub-steps do
        trr = (double)(T)(2.0 * s_rho * ts.nu * (Drr - onethird * dv));
        tpp = (double)(T)(2.0 * s_rho * ts.nu * (Dpp - onethird * dv));
        if (s >= 1) {
          const double Drp = 0.5 * (ts.rinf * (s_vt * ts.irmed - t_vt * tt.irmed) * ts.idrm +
                                    (s_vr - lane_prev(s_vr)) * invdphi * ts.irinf);
          trp = (double)(T)(2.0 * 0.25 * (s_rho + t_rho + s_rhojm + t_rhojm) * ts.nu * Drp);
        }
      }
      if (s >= 1 && s >= i0 - 1 && s < nr) {
        const double trpn = lane_next(trp);
        const double num = dt * ts.irinf *
                           ((ts.rmed * trr - tt.rmed * t_trr) * ts.idrm + (trpn - trp) * invdphi - 0.5 * (tpp + t_tpp));
        vs += 2.0 * quotient(num, s_rho + t_rho, s_rr);
      }
      if (t >= 1 && t >= i0 && t < nr - 1) {
        const double tppjm = lane_prev(t_tpp);
        const double num = dt * tt.irmed *
                           ((tt.rsup * trp - tt.rinf * t_trp) * tt.idrs + (t_tpp - tppjm) * invdphi + 0.5 * (t_trp + trp));
        vtt += 2.0 * quotient(num, t_rho + t_rhojm, t_rt);
      }
    }
    // SubStep2 at ring t, and the wavefront's sum of the elongation rates
    // vt dt / dt of the stored vtheta (ComputeThetaElongations and
    // ComputeAverageThetaVelocities, src/TransportEuler.c:249-290), from which
    // the transport forms the ring mean
    double dv = vs - t_vr;
    const double qr = (dv < 0.0) ? C2 * t_rho * dv * dv : 0.0;
    if (t >= i0 && t < i1) {
      const double dvt = lane_next(vtt) - vtt;
      const double qt = (dvt < 0.0) ? C2 * t_rho * dvt * dvt : 0.0, qtm = lane_prev(qt);
      const double step = dt * 2.0;
      double rate = 0.0;
      if (store) {
        const long l = (long)t * ns + j;
        double vrn = 0.0;
        if (t >= 1) vrn = t_vr - quotient(step, t_rho + u_rho, t_rr) * (qr - u_qr) * tt.idrm;
        const double vtn = vtt - quotient(step, t_rho + t_rhojm, t_rt) * (qt - qtm) * tt.idxt;
        ((T *)a.vri)[l] = sr_round<T>(vrn, sr_cell(l, f_vr));
        const T vts = sr_round<T>(vtn, sr_cell(l, f_vt));
        ((T *)a.vti)[l] = vts;
        rate = ((double)vts * dt) * invdt;
        if (E) {
          const double e = t_en - dt * qr * dv * tt.idrs - dt * qt * dvt * tt.idxt;
          ((T *)a.e_int)[l] = sr_round<T>(e, sr_cell(l, f_e));
        }
        if (t == nr - 1) {
          // vr and vt of ring nrad are zero after ActualiseGas
          st<T>(a.vr, l + ns, 0.0);
          st<T>(a.vt, l + ns, 0.0);
        }
      }
      rate = wave_sum(rate);
      if (lane == 0) a.vt_part[(long)t * ntile + seg] = rate;
    }
    u_rho = t_rho; u_qr = qr;
    t_rho = s_rho; t_rhojm = s_rhojm; t_rr = s_rr; t_rt = s_rt; t_vr = vs; t_vt = s_vt; t_en = s_en;
    t_trr = trr; t_tpp = tpp; t_trp = trp;
    tt = ts;
    s_rho = rho; s_rhojm = rhojm; s_rr = rr; s_rt = rt; s_vr = vr1; s_vt = vt1; s_en = en;
    s_p = p; s_pot = pot; s_ip = ip; s_vt0 = vt0; s_vtn0 = vtn0; s_sgr = sgr;
    ts = tr;
  }
}

// Rings per strip of a walk of S + extra rings' time, for `columns` wavefronts a
// ring and a kernel of which `occupancy` wavefronts share a SIMD.  On a small
// grid a SIMD has at most one wavefront, which is alone with its own latency:
// the shortest strips for which that holds, up to four rings (64x192 FP32
// transport: 1 ring 8.8 us, 2 rings 10.3; 200x400 FP64: 2 rings, 800 wavefronts,
// 12.2, 1 ring, 1600, 13.3).  On larger ones the shortest walk times rounds of
// wavefronts, since a last round that is nearly empty costs as much as a full
// one (1024x3072 FP32 transport: 19 rings, 2970 wavefronts on 3072 places, 109 us;
// 16 rings, 3520, 121; 28 rings, two wavefronts a SIMD on average but not
// evenly, 127).
static int strip_rings(const KArgs &a, int columns, int occupancy, int extra, int most) {
  const long simds = 4L * a.num_cu;
  for (int S = 1; S <= 4; S++)
    if ((long)columns * ((a.nr + S - 1) / S) <= simds) return S;
  int best = 2;
  long cost = -1;
  for (int S = 2; S <= most; S++) {
    const long t = ((long)columns * ((a.nr + S - 1) / S) + occupancy * simds - 1) / (occupancy * simds) * (S + extra);
    if (cost < 0 || t < cost) {
      cost = t;
      best = S;
    }
  }
  return best;
}
template <typename T> static void launch_source(const KArgs &a, hipStream_t s) {
  const int nseg = (a.ns + AZ_OWN - 1) / AZ_OWN, per = 4, bx = (nseg + per - 1) / per;
  // a strip of S rings walks S + 5, plus its start
  const int x = a.d_on ? SRC_DUST : (a.frame || (DF_ON(T, a) && a.df_feedback)) ? SRC_FRAME : SRC_PLAIN;
  const int S = strip_rings(a, nseg, src_occupancy(sizeof(T) == 8, a.energy, x), 7, SRC_STRIP_MAX);
  const dim3 g(bx, (a.nr + S - 1) / S), b(per * AZ_LANES);
#define SRC_LAUNCH(X)                                                                        \
  if (a.energy) hipLaunchKernelGGL((k_source<T, true, X>), g, b, 0, s, a, S);                \
  else hipLaunchKernelGGL((k_source<T, false, X>), g, b, 0, s, a, S)
  if (x == SRC_DUST) {
    SRC_LAUNCH(SRC_DUST);
  } else if (x == SRC_FRAME) {
    SRC_LAUNCH(SRC_FRAME);
  } else {
    SRC_LAUNCH(SRC_PLAIN);
  }
#undef SRC_LAUNCH
}

// Energy source terms, per ring: ComputeDivergenceVelocity
// (src/SourceEuler.c:2373-2411), the stresses and ComputeViscousHeating
// (src/SourceEuler.c:1554-1606) on the post-SubStep2 velocities, then
// SubStep3 (src/SourceEuler.c:1147-1198) with beta cooling
template <typename T>
__device__ double vischeat_cell(const KArgs &a, int i, int j, double *trr, double *tpp,
                                double *trp, double *divv) {
  visc_stress_cell<T>(a, a.vri, a.vti, i, j, trr, tpp, trp, divv);
  const double viscosity = a.nu_ring[i];
  if (viscosity == 0.0) return 0.0;
  const double dens = ld<T>(a.rho, (long)i * a.ns + j);
  double vh = 0.5 / viscosity / dens * (*trr * *trr + 2.0 * *trp * *trp + *tpp * *tpp);
  vh += (2.0 / 9.0) * viscosity * dens * *divv * *divv;
  return vh;
}

template <typename T, int K> __global__ void __launch_bounds__(RING_LB(K)) k_energy(KArgs a) {
  __shared__ double sh[16];
  const dfargo_ctrl *c = a.ctrl;
  if (!c->active) return;
  const int i = ring_of_block(a), ns = a.ns, nr = a.nr, TB = ns / K;
  // threads past the ring (the block is whole wavefronts) repeat its first
  // cells, outside the sum, and store nothing
  const bool on = (int)threadIdx.x < TB;
  const int t = on ? threadIdx.x : 0;
  const long base = (long)i * ns;
  const double dt = c->dt;
  // the stresses, divergence and heating are diagnostics read between
  // AlgoGas calls: stored on the last sub-step of a call only
  const bool last = !c->go_next;
  double vh[K], dv[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int j = t + k * TB;
    double trr, tpp, trp, d;
    if (a.viscous_heating && i >= 1) {
      vh[k] = vischeat_cell<T>(a, i, j, &trr, &tpp, &trp, &d);
    } else {
      visc_stress_cell<T>(a, a.vri, a.vti, i, j, &trr, &tpp, &trp, &d);
      vh[k] = 0.0;
    }
    if (a.viscous_heating && i == 0) {
      // power-law extrapolation from rings 1 and 2; the test reads the
      // viscosity left by the ring loop, i.e. that of ring nrad-1
      double t1, t2, t3, d1;
      double q1 = vischeat_cell<T>(a, 1, j, &t1, &t2, &t3, &d1);
      double q2 = vischeat_cell<T>(a, 2, j, &t1, &t2, &t3, &d1);
      vh[k] = (a.nu_ring[nr - 1] != 0.0) ? q1 * exp(log(q1 / q2) * a.vh_lr1 / a.vh_lr2) : 0.0;
    }
    dv[k] = d;
    if (last && on) {
      st<T>(a.trr, base + j, trr);
      st<T>(a.tpp, base + j, tpp);
      st<T>(a.trp, base + j, trp);
      st<T>(a.divv, base + j, d);
      st<T>(a.vh, base + j, vh[k]);
    }
  }
  double enew[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const long l = base + t + k * TB;
    double num = ld<T>(a.e_int, l) + (a.viscous_heating ? 1 : 0) * vh[k] * dt;
    double den = 1.0 + (a.gamma - 1.0) * dt * dv[k];
    enew[k] = num / den;
  }
  if (a.beta_cooling) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < K; k++) s += (ld<T>(a.vti, base + t + k * TB) + a.Rmed[i] * c->omega_frame);
    s = block_sum(on ? s : 0.0, sh);
    double omega = s / (double)ns;
    omega /= a.Rmed[i];
    double coolingtime = a.beta[i] / omega;
#pragma unroll
    for (int k = 0; k < K; k++) {
      double num = enew[k], den = 1.0 + dt / coolingtime;
      enew[k] = num / den;
    }
  }
  // heating by the dust feedback (src/SourceEuler.c:1291-1299)
  if (a.d_on && a.d_feedback) {
#pragma unroll
    for (int k = 0; k < K; k++) enew[k] += ld<T>(a.fbedot, base + t + k * TB) * dt;
  }
  if (on)
#pragma unroll
    for (int k = 0; k < K; k++) st_sr<T>(a.en, base + t + k * TB, enew[k], sr_key(c, base + t + k * TB, SR_EN));
}

// ------------------------------------------------------------------------
// transport
// ------------------------------------------------------------------------

// Transport (ComputeLRMomenta, OneWindRad and OneWindTheta,
// src/TransportEuler.c:89-465): a wavefront holds 64 consecutive columns, one a
// lane, and walks outwards through a strip of S rings.  At each ring the radial
// pass completes the ring before, which then takes the residual and the uniform
// azimuthal pass and the integer shift while it is still in registers.
//
// Radial and azimuthal pass as kernels of their own took 87 + 76 us at 1024x3072
// with FP64 storage (five quantities written by one and read by the other, 250
// MB) and 78 + 75 us with FP32 storage.  Together they take 104 and 113 us: they
// read the state and write the transported quantities once.  VALU issue bounds
// them first (75 and 81 % of the time), then the latency that three wavefronts a
// SIMD leave uncovered.  With FP32 storage the radially transported quantities
// still round to it between the passes, each by its own draw, as where a grid
// held them (97 us without that rounding and with products shared across the
// quantities, but other values: see the operations' order above).  What is
// counted beyond the memory's traffic is instructions: each Work value
// Q / (rho + 1e-20), difference, slope, face value and flux is formed once (tiles
// in LDS formed every radial face twice and 10/8 of the slopes: 90 us for the
// radial pass alone).  A strip repeats the Work of four rings and the slopes of
// two at its ends, a wavefront eight of its 64 columns; strip_rings picks S.
// FP64 whatever the storage type.
//
// The ring quantities of the FARGO scheme come first, from the per-tile sums
// k_source leaves of the velocity before transport: the mean VMed
// (ComputeAverageThetaVelocities), the integer shift Nshift and the constant
// residual (ComputeConstantResidual, src/TransportEuler.c:292-348), two lanes
// per ring of the strip.  Every wavefront of a ring forms them from the same
// sums in the same order, so all agree on the shift.

// What an azimuthal pass shares over its quantities, for the velocity v of this
// lane's face (between the previous cell and this one): the upwind side, and
// the weights with which a cell's slope enters the values at its two faces
// (ComputeStarTheta, src/TransportEuler.c:419-444): dxtheta - v dt at its right
// face, which is the next lane's, when that one is left by this cell, and
// -(dxtheta + v dt) at its left.
struct AziFace {
  bool up;
  double wl, wr;
};
struct AziRing {
  double dx, invdx, dxrad, invsurf;
};
__device__ __forceinline__ AziFace azi_face(double v, double dt, const AziRing &g) {
  const double ksi = v * dt;
  return {ksi > 0.0, -(g.dx + ksi), lane_next(g.dx - ksi)};
}
// the value at this lane's face for the cell values x; one difference per
// face (a cell's second one is its neighbour's)
__device__ __forceinline__ double azi_star_lane(double x, const AziFace &f, const AziRing &g) {
  const double dqp = lane_next(x) - x, dqm = lane_prev(dqp);
  // the quotient is formed on every lane and selected (where it is not used
  // it may be a NaN of a zero sum, which the select discards)
  const double prod = dqp * dqm;
  const double d = div_nr(prod, dqp + dqm) * g.invdx, dq = prod > 0.0 ? d : 0.0;
  const double left = lane_prev(x + f.wr * dq), right = x + f.wl * dq;
  return f.up ? left : right;
}

// QuantitiesAdvection (src/TransportEuler.c:375-400) with velocity v: the
// density star first, then every quantity's star, flux and update.  Q[5]
// is the density.  The flux through this lane's face is dxrad S RS v; the
// cell's update is its own face's flux minus the next lane's, over the surface.
template <typename T, bool E>
__device__ __forceinline__ void azi_pass_lane(const KArgs &a, double (&Q)[6], double v, double dt, const AziRing &g) {
  const double RI = Q[5];
  const AziFace f = azi_face(v, dt, g);
  const double rs = azi_star_lane(RI, f, g);
  // the Work values Q / (rho + 1e-20) share one reciprocal
  const double inv = div_nr(1.0, RI + 1e-20);
#pragma unroll
  for (int q = 0; q < 6; q++) {
    if (q == 4 && !E) continue;
    if (q < 4 && DF_ON(T, a) && a.tr_skip_mom) continue;
    const double star = azi_star_lane(Q[q] * inv, f, g);
    const double flux = g.dxrad * star * rs * v;
    Q[q] += (flux - lane_next(flux)) * g.invsurf;
  }
}

// the state of one cell of the newest ring, as stored, and vr at its outer face
template <typename T> struct RadRaw {
  T rho, vt, vtp, en, vr_out;
};
template <typename T, bool E>
__device__ __forceinline__ RadRaw<T> rad_load(const KArgs &a, int r, int j, int jp) {
  const long l = (long)r * a.ns;
  RadRaw<T> q;
  q.rho = ((const T *)a.rho)[l + j];
  q.vt = ((const T *)a.vti)[l + j];
  q.vtp = ((const T *)a.vti)[l + jp];
  q.vr_out = ((const T *)a.vri)[l + a.ns + j];
  q.en = E ? ((const T *)a.en)[l + j] : (T)0;
  return q;
}
// v plus the value of the other lane of its pair (quad_perm 1,0,3,2)
__device__ __forceinline__ double pair_sum(double v) {
  return v + __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), 0xB1, 0xf, 0xf, true),
                              __builtin_amdgcn_update_dpp(0, __double2loint(v), 0xB1, 0xf, 0xf, true));
}
// rings per strip, at most (two lanes per ring hold its FARGO values)
#define TR_STRIP_MAX 32
// wavefronts per SIMD the registers allow: 166 of them without the energy
// equation; with it 188, which three wavefronts' budget of 168 would spill
// (256x768 FP64: 24 us against 21)
constexpr int tr_occupancy(bool energy) { return energy ? 2 : 3; }

// Quantity slots: 0 rp, 1 rm, 2 tp, 3 tm, 4 e (E: the energy equation), 5 rho
// (the Work of the density itself); slot 6 of the radial pass's values is rho
// as its own base for RhoStar.
template <typename T, bool E> __global__ void __launch_bounds__(256, tr_occupancy(E)) k_transport_azi(KArgs a, int S) {
  const dfargo_ctrl *c = a.ctrl;
  if (!c->active) return;
  const int ns = a.ns, nr = a.nr, lane = threadIdx.x & (AZ_LANES - 1), per = blockDim.x / AZ_LANES;
  // the blocks of one XCD take neighbouring segments and strips (ring_of_block)
  const int nb = gridDim.x * gridDim.y, b0 = blockIdx.y * gridDim.x + blockIdx.x;
  const int b = (a.xcd_remap && nb % 8 == 0) ? (b0 % 8) * (nb / 8) + b0 / 8 : b0;
  const int seg = __builtin_amdgcn_readfirstlane((b % gridDim.x) * per + threadIdx.x / AZ_LANES);
  const int i0 = (b / gridDim.x) * S, i1 = (i0 + S < nr) ? i0 + S : nr;
  if (seg * AZ_OWN >= ns) return; // a whole wavefront
  int j = (seg * AZ_OWN - AZ_HALO + lane) % ns;
  if (j < 0) j += ns;
  const int jp = (j == ns - 1) ? 0 : j + 1;
  const double dt = c->dt, invdt = 1.0 / dt, Of = c->omega_frame, dtheta = a.pm / (double)ns;
  const bool skip_mom = DF_ON(T, a) && a.tr_skip_mom;
  const int rb = (i0 - 2 > 0) ? i0 - 2 : 0;
  double v_r = (double)((const T *)a.vri)[(long)rb * ns + j]; // vr at face r
  RadRaw<T> next = rad_load<T, E>(a, rb, j, jp);
  // ring tables of the walk, ring rb + k in lane k: read once, ahead (a scalar
  // load per ring would make the walk wait for each)
  const int rt = (rb + lane < nr + 1) ? rb + lane : nr + 1;
  const double tRmed = a.Rmed[rt], tIdr = a.InvDiffRmed[rt], tRinf = a.Rinf[rt], tInvS = a.InvSurf[rt];
  // the FARGO scheme's ring values, ring i0 + k in the lanes 2 k and 2 k + 1
  double gV, gU, gDx, gInvDx, gDxrad;
  int gShift;
  {
    const int ntile = (ns + DF_SRC_COLS - 1) / DF_SRC_COLS;
    const int i = (i0 + (lane >> 1) < i1) ? i0 + (lane >> 1) : i1 - 1;
    double sum = 0.0;
    for (int t0 = 0; t0 < ntile; t0 += 16) {
      double x[8]; // in flight together
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const int t = t0 + 2 * q + (lane & 1);
        x[q] = t < ntile ? a.vt_part[(long)i * ntile + t] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < 8; q++) sum += x[q];
    }
    gV = pair_sum(sum) / (double)ns;
    const double Ntilde = gV * a.InvRmed[i] * dt * (double)ns / a.pm;
    const double Nround = floor(Ntilde + 0.5);
    const long nshift = (long)Nround;
    gU = (Ntilde - Nround) * a.Rmed[i] * invdt * (a.pm / (double)ns);
    gDx = a.pm / (double)ns * a.Rmed[i];
    gInvDx = 1.0 / gDx;
    gDxrad = (a.Rsup[i] - a.Rinf[i]) * dt;
    long sh = nshift % ns;
    if (sh < 0) sh += ns;
    gShift = (int)sh;
    if (seg == 0) {
      // distance of Ntilde from the nearest rounding tie, min over the call
      // (the gas's shift)
      double margin = 0.5 - fabs(Ntilde - Nround);
      margin = wave_min(margin > 0.0 ? margin : 0.0);
      if ((lane & 1) == 0 && i0 + (lane >> 1) < i1) {
        a.vmed[i] = gV;
        a.nshift[i] = nshift;
      }
      if (lane == 0 && !(DF_ON(T, a) && a.tr_dust))
        atomicMin(&a.ctrl->fargo_margin_bits, (unsigned long long)__double_as_longlong(margin));
    }
  }
  const int own = lane - AZ_HALO;
  const bool store = own >= 0 && own < AZ_OWN && seg * AZ_OWN + own < ns;
  void *zp[6] = {a.z_rp, a.z_rm, a.z_tp, a.z_tm, a.z_en, a.z_rho};
  unsigned f_rad[6], f_azi[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    f_rad[k] = sr_field(c, SR_RAD + k);
    f_azi[k] = sr_field(c, SR_AZI + k);
  }
  // Entering step r (the newest ring read is r, q = r - 1 the one before):
  // Qq, Wq, vtq: ring q; Qp, vtp: ring q - 1; diff: the scaled differences
  // across face q (between rings q - 1 and q); right: the values of ring q - 1
  // at face q; flux: through face q - 1; v: the velocity at face q.
  double Qp[6], Qq[6], Wq[7], diff[7], right[7], flux[6], v = 0.0, vtq = 0.0, vtp = 0.0;
#pragma unroll
  for (int k = 0; k < 7; k++) Wq[k] = diff[k] = right[k] = 0.0;
#pragma unroll
  for (int k = 0; k < 6; k++) Qp[k] = Qq[k] = flux[k] = 0.0;
  for (int r = rb; r <= i1 + 1; r++) {
    const RadRaw<T> raw = next;
    if (r + 1 < nr && r <= i1) next = rad_load<T, E>(a, r + 1, j, jp);
    const int tr = r - rb; // table lane of ring r
    // (beyond the last ring the walk repeats it, with differences of weight 0)
    const double d = (double)raw.rho, Rm = lane_value(tRmed, tr), RO = Rm * Of, v_out = (double)raw.vr_out;
    const double Q[6] = {d * v_out,
                         d * v_r,
                         d * ((double)raw.vtp + RO) * Rm,
                         d * ((double)raw.vt + RO) * Rm,
                         E ? (double)raw.en : 0.0,
                         d};
    // the Work values share one reciprocal per cell
    const double inv = div_nr(1.0, d + 1e-20);
    double W[7];
#pragma unroll
    for (int k = 0; k < 6; k++) W[k] = Q[k] * inv;
    W[6] = d;
    const int q = r - 1;
    if (q >= 0) {
      // ComputeStarRad: the slopes of ring q (zero on the first and last), the
      // values of ring q at its lower face q and its upper face r, and with
      // them the values at face q from the upwind side; the faces 0 and nr are
      // closed
      const double idr = r < nr ? lane_value(tIdr, tr) : 0.0;
      const bool inner = q > 0 && q < nr - 1, open = q > 0 && q < nr;
      const double gap = (inner && tr > 0) ? lane_value(tRmed, tr) - lane_value(tRmed, tr - 1) : 0.0; // q to r
      const double wl = -0.5 * (gap + v * dt), wr = 0.5 * (gap - v_r * dt);
      double star[7];
#pragma unroll
      for (int k = 0; k < 7; k++) {
        if (k == 4 && !E) continue;
        const double dm = diff[k];
        const double dp = (W[k] - Wq[k]) * idr;
        diff[k] = dp;
        // the quotient is formed on every lane and selected (where it is not
        // used it may be a NaN of a zero sum, which the select discards)
        const double prod = dp * dm, x = div_nr(2.0 * prod, dp + dm);
        const double slope = (inner && prod > 0.0) ? x : 0.0;
        star[k] = v > 0.0 ? right[k] : Wq[k] + wl * slope;
        right[k] = Wq[k] + wr * slope;
      }
      // VanLeerRadial (src/TransportEuler.c:205-217): the flux through face q,
      // then ring q - 1's update
      const double f0 = (open && tr > 0) ? dt * dtheta * lane_value(tRinf, tr - 1) : 0.0;
      const int i = q - 1;
      const bool mine = i >= i0 && i < i1;
      const double invs = mine ? lane_value(tInvS, tr - 2) : 0.0;
#pragma unroll
      for (int k = 0; k < 6; k++) {
        if (k == 4 && !E) continue;
        const double f = f0 * star[k] * star[6] * v, varq = flux[k] - f;
        flux[k] = f;
        if (!(k < 4 && skip_mom)) Qp[k] = Qp[k] + varq * invs;
        if (k == 5 && i == 0 && mine && store) a.lost_col[j] = varq;
        // the radially transported quantities round to storage
        if (!(k < 4 && skip_mom)) Qp[k] = (double)sr_round<T>(Qp[k], sr_cell((long)i * ns + j, f_rad[k]));
      }
      if (mine) {
        // the residual velocity of the cell (src/TransportEuler.c:280-290),
        // the residual pass (the only pass of the standard transport) and the
        // uniform pass with the constant residual
        const int g = 2 * (i - i0);
        const double vmed = lane_value(gV, g), u = lane_value(gU, g);
        const AziRing ring = {lane_value(gDx, g), lane_value(gInvDx, g), lane_value(gDxrad, g), invs};
        double vres = (vtp * dt) * invdt - vmed;
        if (!a.fast) vres = u + vres;
        azi_pass_lane<T, E>(a, Qp, vres, dt, ring);
        if (a.fast) azi_pass_lane<T, E>(a, Qp, u, dt, ring);
        // AdvectSHIFT (src/TransportEuler.c:350-373): new[j] = old[j - Nshift]
        // (the shift is read while every lane is active: lane g may be one that
        // stores nothing, and a register reloaded for the storing lanes alone
        // would not hold its value)
        const int shift = __builtin_amdgcn_readlane(gShift, g);
        if (store) {
          int jn = j + shift;
          if (jn >= ns) jn -= ns;
          const long l = (long)i * ns + jn;
#pragma unroll
          for (int k = 0; k < 6; k++) {
            if (k == 4 && !E) continue;
            ((T *)zp[k])[l] = sr_round<T>(Qp[k], sr_cell(l, f_azi[k]));
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 6; k++) {
      Qp[k] = Qq[k];
      Qq[k] = Q[k];
    }
#pragma unroll
    for (int k = 0; k < 7; k++) Wq[k] = W[k];
    vtp = vtq;
    vtq = (double)raw.vt;
    v = v_r;
    v_r = v_out;
  }
}

template <typename T> static void launch_transport(const KArgs &a, hipStream_t s) {
  const int per = (a.tune_azi_waves == 1 || a.tune_azi_waves == 2) ? a.tune_azi_waves : 4;
  const int nseg = (a.ns + AZ_OWN - 1) / AZ_OWN, bx = (nseg + per - 1) / per;
  // a strip of S rings walks S + 4, plus its start
  const int S = strip_rings(a, nseg, tr_occupancy(a.energy), 6, TR_STRIP_MAX);
  const dim3 g(bx, (a.nr + S - 1) / S), b(per * AZ_LANES);
  if (a.energy) hipLaunchKernelGGL((k_transport_azi<T, true>), g, b, 0, s, a, S);
  else hipLaunchKernelGGL((k_transport_azi<T, false>), g, b, 0, s, a, S);
}

// The mass through the inner edge (VanLeerRadial's LostByDisk, ring 0;
// LostMassd for the dust fluid) from the columns' fluxes the transport left:
// one wavefront of the kernel that ends the sub-step for that fluid.
__device__ __forceinline__ void add_lost_mass(const KArgs &a, const double *col, double *total) {
  double lost = 0.0;
  for (int j = threadIdx.x; j < a.ns; j += 8 * 64) {
    double x[8]; // in flight together
#pragma unroll
    for (int q = 0; q < 8; q++) x[q] = j + q * 64 < a.ns ? col[j + q * 64] : 0.0;
#pragma unroll
    for (int q = 0; q < 8; q++) lost += x[q];
  }
  lost = wave_sum(lost);
  if (threadIdx.x == 0) *total += lost;
}

// ComputeVelocities (src/TransportEuler.c:515-547) and the floors
// (src/SourceEuler.c:2506-2541) of one cell from the transported momenta,
// rounded to the storage type as the stored state would be.  The
// velocities are quotients formed here, so with FP32 storage they are
// rounded stochastically like every other state store (keyed by the cell,
// so an edge ring that copies a neighbour's value recomputes exactly the
// value stored there); density and energy are already stored values.
struct CellState {
  double rho, vr, vt, e;
};
template <typename T> __device__ CellState vel_cell(const KArgs &a, const dfargo_ctrl *c, int i, int j) {
  const int ns = a.ns;
  const long l = (long)i * ns + j, lim = l - ns, ljm = (j == 0) ? (long)i * ns + ns - 1 : l - 1;
  const double rho = ld<T>(a.z_rho, l);
  CellState s;
  s.vr = 0.0;
  if (i != 0) s.vr = (ld<T>(a.z_rp, lim) + ld<T>(a.z_rm, l)) / (rho + ld<T>(a.z_rho, lim) + 1e-20);
  s.vt = (ld<T>(a.z_tp, ljm) + ld<T>(a.z_tm, l)) / (rho + ld<T>(a.z_rho, ljm) + 1e-20) / a.Rmed[i] -
         a.Rmed[i] * c->omega_frame;
  s.rho = rho;
  if (a.floors && s.rho < a.floor_dens) s.rho = a.floor_dens;
  s.e = 0.0;
  if (a.energy) {
    s.e = ld<T>(a.z_en, l);
    const double e_bottom = 1e-3 * a.EnergyMed[i];
    if (a.floors && s.e < e_bottom) s.e = e_bottom;
  }
  s.rho = (double)(T)s.rho;
  s.vr = (double)sr_round<T>(s.vr, sr_key(c, l, SR_FIN));
  s.vt = (double)sr_round<T>(s.vt, sr_key(c, l, SR_FIN + 1));
  s.e = (double)(T)s.e;
  return s;
}

// End of the sub-step: ComputeVelocities and the floors, then
// ApplyBoundaryCondition (src/SideEuler.c:1102-1131) -- wall or open edges
// and the sub-Keplerian reset of vt in rings 0 and nrad-1, which runs for
// every boundary type (src/SideEuler.c:1110-1112).  Each cell of the edge
// rings takes the values the boundary routines would copy into it from the
// rings they read (2, 3 and nrad-2), recomputed here from the momenta.
// Stores cell (i, j) of rings 0 .. nrad-1.
template <typename T> __device__ __forceinline__ void finish_cell(const KArgs &a, const dfargo_ctrl *c, int i, int j) {
  const int nr = a.nr;
  const long l = (long)i * a.ns + j;
  CellState s = vel_cell<T>(a, c, i, j);
  if (a.bc == DFARGO_BC_WALL) {
    if (i == 0) {
      s.vr = -vel_cell<T>(a, c, 2, j).vr;
      s.rho = a.SigmaMed[0];
    } else if (i == 1) {
      s.vr = 0.0;
      s.rho = a.SigmaMed[1];
    }
    if (i == nr - 2) s.rho = a.SigmaMed[nr - 2];
    if (i == nr - 1) {
      s.vr = 0.0;
      s.rho = a.SigmaMed[nr - 1];
    }
  }
  if (i == 0) s.vt = a.VthetaMed[0] - a.Rmed[0] * c->omega_frame;
  if (i == nr - 1) s.vt = a.VthetaMed[nr - 1] - a.Rmed[nr - 1] * c->omega_frame;
  if (a.bc == DFARGO_BC_OPEN) {
    // OpenBoundary (src/SideEuler.c:300-408), standard prescription
    if (i <= 2) {
      const CellState s2 = (i == 2) ? s : vel_cell<T>(a, c, 2, j);
      const double vrp = vel_cell<T>(a, c, 3, j).vr;
      const double vr2 = ((vrp >= 0.0) || (s2.rho < a.SigmaMed[0])) ? 0.0 : vrp;
      if (i == 2) s.vr = vr2;
      if (i == 1) {
        s.rho = s2.rho;
        s.e = s2.e;
        s.vt = s2.vt * a.open_vt_in1[0];
        s.vr = vr2;
      }
      if (i == 0) {
        s.rho = s2.rho;
        s.e = s2.e;
        s.vt = s2.vt * a.open_vt_in2[0];
      }
    }
    if (i == nr - 1) {
      const CellState sm = vel_cell<T>(a, c, nr - 2, j);
      s.rho = sm.rho;
      s.e = sm.e;
      s.vt = sm.vt * a.open_vt_out[0];
      s.vr = ((sm.vr < 0.0) || (sm.rho < a.SigmaMed[nr - 2])) ? 0.0 : sm.vr;
    }
  }
  st<T>(a.rho, l, s.rho);
  st<T>(a.vr, l, s.vr);
  st<T>(a.vt, l, s.vt);
  if (a.energy) st<T>(a.en, l, s.e);
}
// the wall's radial velocity at the outer face (ring nrad)
template <typename T> __device__ __forceinline__ void finish_outer_face(const KArgs &a, const dfargo_ctrl *c, int j) {
  if (a.bc == DFARGO_BC_WALL) st<T>(a.vr, (long)a.nr * a.ns + j, -vel_cell<T>(a, c, a.nr - 2, j).vr);
}

// One row of blocks for the mass through the inner edge, then rings 0 .. nrad,
// the last only for the wall's vr at the outer face.  The mass comes first since
// it is a chain of loads and lane sums: in the last ring's row that was the
// launch's tail (512x1536 FP32 9.7 us, now 9.0; 1024x3072 20.8 and 19.9).
template <typename T> __global__ void __launch_bounds__(256) k_finish(KArgs a) {
  const dfargo_ctrl *c = a.ctrl;
  if (!c->active) return;
  // the sub-step ends here: the next one's loop condition takes effect
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) a.ctrl->go = c->go_next;
  const int i = (int)blockIdx.y - 1, ns = a.ns, nr = a.nr, j = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 0) {
    if (blockIdx.x == 0 && threadIdx.x < 64) add_lost_mass(a, a.lost_col, &a.ctrl->lost_mass);
    return;
  }
  if (j >= ns) return;
  if (i == nr) {
    finish_outer_face<T>(a, c, j);
    return;
  }
  finish_cell<T>(a, c, i, j);
}

// EvanescentBoundary (src/SideEuler.c:796-950) for the gas, after the
// boundary conditions: in the wave-killing zones Rmed < WKZRMIN and
// Rmed > WKZRMAX each ring relaxes as q <- (q + lambda q0) / (1 + lambda)
// towards its azimuthal mean (DampToAxi, FP64 sums) or the initial profile
// (DampToIni), lambda = x^2 dt / (ratio Rmed^1.5) with x rising from 0 at
// the zone's edge to 1 at the grid's edge.  With ZEROVRADBC the two
// innermost and the outermost ring take vr = 0 and the target density and
// vtheta.  One 256-thread workgroup per ring of the zones; each thread
// reads and rewrites the same cells, so the update is in place.
enum { EV_TB = 256 };

// SolveOneDViscousEvolution (src/SideEuler.c:1518-1565): one explicit step
// of the 1-D viscous disc the DAMPTOVISCOUS zones relax towards -- the
// diffusion dSigma/dt = 3[(nu Sigma)'' + 3/(2R)(nu Sigma)'] on the
// non-uniform 1-D grid, its radial velocity, then the boundary rule.  One
// workgroup; the profile is staged in LDS, updated there, written back.
enum { V1D_MAX = 1024, V1D_TB = 256 };
__global__ void __launch_bounds__(V1D_TB) k_visc1d(KArgs a) {
  const dfargo_ctrl *c = a.ctrl;
  if (!c->active) return;
  __shared__ double sS[V1D_MAX], sV[V1D_MAX], sN[V1D_MAX], sR[V1D_MAX], sT[V1D_MAX];
  const int n = a.n1d, tid = threadIdx.x;
  const double dt = c->dt;
  for (int i = tid; i < n; i += V1D_TB) {
    sS[i] = a.v1d_sigma[i];
    sV[i] = a.v1d_vrad[i];
    sN[i] = a.v1d_nu[i];
    sR[i] = a.v1d_rmed[i];
  }
  __syncthreads();
  for (int i = 1 + tid; i <= n - 2; i += V1D_TB) {
    const double drm = sR[i] - sR[i - 1], drp = sR[i + 1] - sR[i];
    const double drnu = (drm * drm * sN[i + 1] - drp * drp * sN[i - 1] + (drp * drp - drm * drm) * sN[i]) /
                        (drm * drm * drp + drp * drp * drm);
    const double drsigma = (drm * drm * sS[i + 1] - drp * drp * sS[i - 1] + (drp * drp - drm * drm) * sS[i]) /
                           (drm * drm * drp + drp * drp * drm);
    const double d2rnu = (drm * sN[i + 1] + drp * sN[i - 1] - (drm + drp) * sN[i]) /
                         (0.5 * drm * drp * drp + 0.5 * drp * drm * drm);
    const double d2rsigma = (drm * sS[i + 1] + drp * sS[i - 1] - (drm + drp) * sS[i]) /
                            (0.5 * drm * drp * drp + 0.5 * drp * drm * drm);
    const double term1 = 3.0 * sS[i] * (1.5 * drnu / sR[i] + d2rnu);
    const double term2 = 3.0 * drsigma * (1.5 * sN[i] / sR[i] + 2.0 * drnu);
    const double term3 = 3.0 * sN[i] * d2rsigma;
    sT[i] = term1 + term2 + term3;
    sV[i] = -1.5 * sN[i] / sR[i] - 3.0 * drnu - 1.5 * (sN[i] / sS[i]) * drsigma;
  }
  __syncthreads();
  for (int i = 1 + tid; i <= n - 2; i += V1D_TB) sS[i] += dt * sT[i];
  __syncthreads();
  if (tid == 0) {
    if (a.bc1d == 1) {
      sS[0] = sS[1] * (sN[1] / sN[0]) * sqrt(sR[1] / sR[0]);
      sS[n - 1] = sS[n - 2] * (sN[n - 2] / sN[n - 1]) * sqrt(sR[n - 2] / sR[n - 1]);
    } else if (a.bc1d == 2) {
      sS[0] = sS[1] * (sN[1] / sN[0]);
      sS[n - 1] = sS[n - 2] * (sN[n - 2] / sN[n - 1]);
    } else {
      sS[0] = 1e-9;
      sS[n - 1] = 1e-9;
    }
    sV[0] = sV[1];
    sV[n - 1] = sV[n - 2];
  }
  __syncthreads();
  for (int i = tid; i < n; i += V1D_TB) {
    a.v1d_sigma[i] = sS[i];
    a.v1d_vrad[i] = sV[i];
  }
}
template <typename T> __global__ void __launch_bounds__(EV_TB) k_evanescent(KArgs a) {
  const dfargo_ctrl *c = a.ctrl;
  if (!c->active) return;
  const int b = blockIdx.x, nr = a.nr, ns = a.ns, tid = threadIdx.x;
  const int i = (b < a.wkz_n_in) ? b : a.wkz_i_out + (b - a.wkz_n_in);
  const long base = (long)i * ns;
  const double R = a.Rmed[i];
  const bool in_zone = R < a.wkz_rmin;
  const double damping = in_zone ? (R - a.wkz_rmin) / (a.Rmed[0] - a.wkz_rmin)
                                 : (R - a.wkz_rmax) / (a.Rmed[nr - 1] - a.wkz_rmax);
  const double Tz = a.damp_ratio * pow(R, 1.5);
  const double lambda = damping * damping * c->dt / Tz;
  double q0[4];
  if (a.damp_visc) {
    // the ring means of vtheta and e, Sigma and vr interpolated linearly in
    // the 1-D disc (src/SideEuler.c:868-887)
    __shared__ double partv[EV_TB / 64][2];
    double s[2] = {0.0, 0.0};
    for (int j = tid; j < ns; j += EV_TB) {
      s[0] += ld<T>(a.vt, base + j);
      if (a.energy) s[1] += ld<T>(a.en, base + j);
    }
#pragma unroll
    for (int k = 0; k < 2; k++) s[k] = wave_sum(s[k]);
    if ((tid & 63) == 0) {
      partv[tid >> 6][0] = s[0];
      partv[tid >> 6][1] = s[1];
    }
    __syncthreads();
    double sv = 0.0, se = 0.0;
    for (int w = 0; w < EV_TB / 64; w++) {
      sv += partv[w][0];
      se += partv[w][1];
    }
    q0[1] = sv / (double)ns;
    q0[3] = se / (double)ns;
    int m = 0;
    while (a.v1d_rmed[m] < R) m++;
    m--;
    const double r0 = a.v1d_rmed[m], r1 = a.v1d_rmed[m + 1];
    q0[2] = ((r1 - R) * a.v1d_sigma[m] + (R - r0) * a.v1d_sigma[m + 1]) / (r1 - r0);
    q0[0] = ((r1 - R) * a.v1d_vrad[m] + (R - r0) * a.v1d_vrad[m + 1]) / (r1 - r0);
  } else if (a.damp_ini) {
    q0[0] = a.VradMed[i];
    q0[1] = a.VthetaMed[i] - R * c->omega_frame;
    q0[2] = a.SigmaMed[i];
    q0[3] = a.EnergyMed[i];
  } else {
    __shared__ double part[EV_TB / 64][4];
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int j = tid; j < ns; j += EV_TB) {
      s[0] += ld<T>(a.vr, base + j);
      s[1] += ld<T>(a.vt, base + j);
      s[2] += ld<T>(a.rho, base + j);
      if (a.energy) s[3] += ld<T>(a.en, base + j);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) s[k] = wave_sum(s[k]);
    if ((tid & 63) == 0)
#pragma unroll
      for (int k = 0; k < 4; k++) part[tid >> 6][k] = s[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; k++) {
      double t = 0.0;
      for (int w = 0; w < EV_TB / 64; w++) t += part[w][k];
      q0[k] = t / (double)ns;
    }
  }
  // the dust fluid's targets (src/SideEuler.c:844-848,887-926): its
  // initial profiles, or with DampToAxi its ring means; with the open dust
  // edge the fluid is not damped
  double dq0[3] = {0.0, 0.0, 0.0};
  const bool ddamp = DF_ON(T, a) && !a.df_open;
  if (ddamp) {
    if (!a.damp_ini && !a.damp_visc) {
      __shared__ double dpart[EV_TB / 64][3];
      double s[3] = {0.0, 0.0, 0.0};
      for (int j = tid; j < ns; j += EV_TB) {
        s[0] += a.dvr[base + j];
        s[1] += a.dvt[base + j];
        s[2] += a.drho[base + j];
      }
#pragma unroll
      for (int k = 0; k < 3; k++) s[k] = wave_sum(s[k]);
      if ((tid & 63) == 0)
#pragma unroll
        for (int k = 0; k < 3; k++) dpart[tid >> 6][k] = s[k];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 3; k++) {
        double t = 0.0;
        for (int w = 0; w < EV_TB / 64; w++) t += dpart[w][k];
        dq0[k] = t / (double)ns;
      }
    } else {
      dq0[0] = a.DVradMed[i];
      dq0[1] = a.DVthetaMed[i] - R * c->omega_frame;
      dq0[2] = a.DSigmaMed[i];
    }
  }
  const bool edge = a.zero_vrad && ((in_zone && (i == 0 || i == 1)) || (!in_zone && i == nr - 1));
  for (int j = tid; j < ns; j += EV_TB) {
    const long l = base + j;
    if (ddamp) {
      a.dvr[l] = (a.dvr[l] + lambda * dq0[0]) / (1.0 + lambda);
      a.dvt[l] = (a.dvt[l] + lambda * dq0[1]) / (1.0 + lambda);
      a.drho[l] = (a.drho[l] + lambda * dq0[2]) / (1.0 + lambda);
    }
    double vr = (ld<T>(a.vr, l) + lambda * q0[0]) / (1.0 + lambda);
    double vt = (ld<T>(a.vt, l) + lambda * q0[1]) / (1.0 + lambda);
    double rho = (ld<T>(a.rho, l) + lambda * q0[2]) / (1.0 + lambda);
    if (edge) {
      vr = 0.0;
      rho = q0[2];
      vt = q0[1];
    }
    st_sr<T>(a.vr, l, vr, sr_key(c, l, SR_EVA));
    st_sr<T>(a.vt, l, vt, sr_key(c, l, SR_EVA + 1));
    st_sr<T>(a.rho, l, rho, sr_key(c, l, SR_EVA + 2));
    if (a.energy) st_sr<T>(a.en, l, (ld<T>(a.en, l) + lambda * q0[3]) / (1.0 + lambda), sr_key(c, l, SR_EVA + 3));
  }
}

// NonReflectingBoundary (src/SideEuler.c:569-794), barotropic case without
// the accreting variant, after the sub-Keplerian reset (which it leaves
// alone).  Workgroup 0 does the inner edge, workgroup 1 the outer one.
// Each edge takes a pattern speed from the innermost (outermost) planet
// inside the grid, turns it into an integer azimuthal shift i_angle over the
// first (last) ring spacing at the mean sound speed, and
//   inner: rho(0, j + i_angle) = rho(1, j), shifted by a constant so that
//          ring 0's mean is SigmaMed[0]; vr(1, j) = 2 vr_med - vr(2, j) with
//          vr_med = -cs1 (rho(1, j) - <rho(1)>) / <rho(1)>;
//   outer: rho(nr-1, j) = rho(nr-2, j - i_angle) + SigmaMed[nr-1] - <...>;
//          vr(nr-1, j) = 2 vr_med - vr(nr-2, j), vr_med = +cs (...).
// The new edge ring is a cyclic shift of its neighbour, so its mean is the
// neighbour's: the constant is formed from that mean.  The sound speed is
// the isothermal ring value, the mean of its identical cells.
enum { NR_TB = 256 };

// block sums of N values per thread, in a fixed order (wavefront tree, then
// the wavefronts in order); every thread gets the totals
template <int N> __device__ void nr_block_sums(double (&v)[N], double (*part)[NR_TB / 64]) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < N; q++) {
    const double w = wave_sum(v[q]);
    if ((tid & 63) == 0) part[q][tid >> 6] = w;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < N; q++) {
    double s = 0.0;
    for (int w = 0; w < NR_TB / 64; w++) s += part[q][w];
    v[q] = s;
  }
}

// the pattern speed: the innermost (outermost) planet inside the grid (the
// loops of src/SideEuler.c:590-600 and 702-712; the reference leaves r
// undefined when planet 0 is outside the grid, here the grid's edge stands
// in)
__device__ double nr_pattern_omega(const KArgs &a, const dfargo_ctrl *c, bool inner) {
  const double r0 = a.Rinf[0], r1 = a.Rsup[a.nr - 1];
  double buf = inner ? r1 : r0, rp_sel = buf, omega = pow(buf, -1.5);
  for (int k = 0; k < c->nb; k++) {
    const double xp = c->pl_x[k], yp = c->pl_y[k], rp = sqrt(xp * xp + yp * yp);
    if (inner ? ((rp < buf) && (rp >= r0)) : ((rp > buf) && (rp <= r1))) {
      rp_sel = rp;
      omega = pow(rp, -1.5);
    }
    buf = rp_sel;
  }
  return omega;
}

__device__ __forceinline__ int nr_wrap(int j, int ns) {
  int jp = j % ns;
  return (jp < 0) ? jp + ns : jp;
}

// NonReflectingBoundary (src/SideEuler.c:569-794) without the accreting
// variant, after the sub-Keplerian reset (which it leaves alone).
// Workgroup 0 does the inner edge, workgroup 1 the outer one.  Each edge
// takes a pattern speed from the innermost (outermost) planet inside the
// grid and turns it into an integer azimuthal shift i_angle over the first
// (last) ring spacing at a mean sound speed.
//   barotropic: rho(0, j + i_angle) = rho(1, j) and
//     rho(nr-1, j) = rho(nr-2, j - i_angle), each shifted by a constant so
//     that the edge ring's mean is SigmaMed; vr at the faces 1 and nr-1 is
//     2 vr_med - vr of the next face in, vr_med = -/+ cs drho / <rho>;
//   adiabatic (inner edge): the energy is copied with the shift, the
//     density follows it acoustically, SigmaMed[0] + (gamma-1)(e -
//     EnergyMed[0]) / csinit0^2, and both are shifted to the initial means;
//     vr_med uses the initial profiles; the outer edge is the barotropic one
//     with the energy copied and shifted to EnergyMed too and vr_med from the
//     cell's own sound speed.
// A shifted edge ring is a cyclic copy of its neighbour, so its mean is the
// neighbour's: the constants are formed from that mean.  The sound speed is
// the isothermal ring value (the mean of its identical cells), or, with the
// energy equation, the grid k_eos_step has just formed from the state the
// boundary sees (src/SideEuler.c:1121-1122).
template <typename T> __global__ void __launch_bounds__(NR_TB) k_nonreflecting(KArgs a) {
  const dfargo_ctrl *c = a.ctrl;
  if (!c->active) return;
  const bool inner = blockIdx.x == 0;
  const int nr = a.nr, ns = a.ns, tid = threadIdx.x;
  // the ring the edge copies from, and the edge ring
  const int src = inner ? 1 : nr - 2, dst = inner ? 0 : nr - 1;
  const long bs = (long)src * ns, bd = (long)dst * ns;
  __shared__ double part[4][NR_TB / 64];
  const double omega = nr_pattern_omega(a, c, inner);
  const double g = a.gamma;
  if (a.energy && inner) {
    const double csinit0 = sqrt(g) * a.aspect_ratio * pow(a.Rmed[0], -0.5 + a.flaring);
    const double csinit1 = sqrt(g) * a.aspect_ratio * pow(a.Rmed[1], -0.5 + a.flaring);
    double dangle = (pow(a.Rinf[1], -1.5) - omega) / (.5 * (csinit0 + csinit1));
    dangle *= (a.Rmed[1] - a.Rmed[0]);
    const int i_angle = (int)(dangle / a.pm * (double)ns + .5);
    double s[2] = {0.0, 0.0};
    for (int j = tid; j < ns; j += NR_TB) {
      const double e = ld<T>(a.en, bs + j);
      s[0] += e;
      s[1] += a.SigmaMed[0] + (g - 1.0) * (e - a.EnergyMed[0]) / csinit0 / csinit0;
    }
    nr_block_sums<2>(s, part);
    const double mean_e = s[0] / (double)ns, mean_rho = s[1] / (double)ns;
    for (int j = tid; j < ns; j += NR_TB) {
      const double e = ld<T>(a.en, bs + j);
      const double rho = a.SigmaMed[0] + (g - 1.0) * (e - a.EnergyMed[0]) / csinit0 / csinit0;
      const int jp = nr_wrap(j + i_angle, ns);
      st<T>(a.en, jp, e + (a.EnergyMed[0] - mean_e));
      st<T>(a.rho, jp, rho + (a.SigmaMed[0] - mean_rho));
      const double vr_med = -csinit1 * (ld<T>(a.rho, bs + j) - a.SigmaMed[1]) / a.SigmaMed[1];
      st<T>(a.vr, bs + j, 2. * vr_med - ld<T>(a.vr, bs + j + ns));
    }
    return;
  }
  // ring means: rho of the source ring; the sound speed of both rings
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  for (int j = tid; j < ns; j += NR_TB) {
    s[0] += ld<T>(a.rho, bs + j);
    if (a.energy) {
      s[1] += ld<T>(a.cs, bd + j);
      s[2] += ld<T>(a.cs, bs + j);
      s[3] += ld<T>(a.en, bs + j);
    }
  }
  nr_block_sums<4>(s, part);
  const double mean = s[0] / (double)ns;
  // isothermal: the ring value, the mean of the ring's identical cells
  const double cs_a = a.energy ? s[1] / (double)ns : a.cs_iso[dst];
  const double cs_b = a.energy ? s[2] / (double)ns : a.cs_iso[src];
  double dangle = (pow(a.Rinf[inner ? 1 : nr - 2], -1.5) - omega) / (.5 * (cs_a + cs_b));
  dangle *= inner ? (a.Rmed[1] - a.Rmed[0]) : (a.Rmed[nr - 1] - a.Rmed[nr - 2]);
  const int i_angle = (int)(dangle / a.pm * (double)ns + .5);
  const double shift = a.SigmaMed[dst] - mean;
  const double eshift = a.EnergyMed[nr - 1] - s[3] / (double)ns;
  for (int j = tid; j < ns; j += NR_TB) {
    const long ls = bs + j;
    const double rs = ld<T>(a.rho, ls);
    if (inner) {
      const double vr_med = -a.cs_iso[1] * (rs - mean) / mean;
      st<T>(a.rho, nr_wrap(j + i_angle, ns), rs + shift);
      st<T>(a.vr, ls, 2. * vr_med - ld<T>(a.vr, ls + ns));
    } else {
      const long l = bd + j;
      const long lp = bs + nr_wrap(j - i_angle, ns);
      // the outer face's own sound speed with the energy equation
      const double csv = a.energy ? ld<T>(a.cs, l) : a.cs_iso[nr - 1];
      const double vr_med = csv * (rs - mean) / mean;
      st<T>(a.rho, l, ld<T>(a.rho, lp) + shift);
      if (a.energy) st<T>(a.en, l, ld<T>(a.en, lp) + eshift);
      st<T>(a.vr, l, 2. * vr_med - ld<T>(a.vr, ls));
    }
  }
}

// ComputeSoundSpeed inside ApplyBoundaryCondition (src/SideEuler.c:
// 1121-1122), for the non-reflecting boundary with the energy equation: cs
// of the state after transport and floors, which the boundary and the next
// sub-step's CFL condition read
template <typename T, int K> __global__ void __launch_bounds__(RING_LB(K)) k_eos_step(KArgs a) {
  if (!a.ctrl->active) return;
  const int i = ring_of_block(a), ns = a.ns, t = threadIdx.x, TB = ns / K;
  if (t >= TB) return;
  const long base = (long)i * ns;
  const double g = a.gamma;
#pragma unroll
  for (int k = 0; k < K; k++) {
    const long l = base + t + k * TB;
    st<T>(a.cs, l, sqrt(g * (g - 1.0) * ld<T>(a.en, l) / ld<T>(a.rho, l)));
  }
}

// Potential grid on demand (the field of FillForcesArrays)
template <typename T> __global__ void k_potential(KArgs a) {
  const int i = blockIdx.y, ns = a.ns, j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ns) return;
  st<T>(a.pot, (long)i * ns + j, pot_at(a, a.ctrl, i, j));
}

// ------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------

static int ring_k(int ns) {
  static const int ks[] = {1, 2, 3, 4, 6, 8, 12, 16};
  for (int k : ks)
    if (ns % k == 0 && ns / k <= RING_LB(k)) return k;
  return -1;
}

int ring_kcheck(int ns) { return ring_k(ns); }

// Six cells per thread (four waves per ring) for the ring reductions of
// the CFL kernel: its block reductions then run over fewer waves, measured
// faster than two or three cells per thread at more waves.  Rings of fewer
// than 1536 cells keep the smallest K.
static int wide_k(int ns) {
  if (ns % 6 == 0 && ns / 6 >= 256 && ns / 6 <= RING_LB(6)) return 6;
  return ring_k(ns);
}

#define RING_DISPATCH(KERNEL, T, a, s, lds, ...) RING_DISPATCH_K(ring_k((a).ns), KERNEL, T, a, s, lds, ##__VA_ARGS__)
#define RING_DISPATCH_K(KSEL, KERNEL, T, a, s, lds, ...)                                    \
  do {                                                                                      \
    int K_ = (KSEL);                                                                        \
    /* whole wavefronts: the reductions need them */                                        \
    dim3 g_((a).nr), b_(((a).ns / K_ + 63) / 64 * 64);                                      \
    switch (K_) {                                                                           \
      case 1: hipLaunchKernelGGL((KERNEL<T, 1>), g_, b_, lds, s, a, ##__VA_ARGS__); break;  \
      case 2: hipLaunchKernelGGL((KERNEL<T, 2>), g_, b_, lds, s, a, ##__VA_ARGS__); break;  \
      case 3: hipLaunchKernelGGL((KERNEL<T, 3>), g_, b_, lds, s, a, ##__VA_ARGS__); break;  \
      case 4: hipLaunchKernelGGL((KERNEL<T, 4>), g_, b_, lds, s, a, ##__VA_ARGS__); break;  \
      case 6: hipLaunchKernelGGL((KERNEL<T, 6>), g_, b_, lds, s, a, ##__VA_ARGS__); break;  \
      case 8: hipLaunchKernelGGL((KERNEL<T, 8>), g_, b_, lds, s, a, ##__VA_ARGS__); break;  \
      case 12: hipLaunchKernelGGL((KERNEL<T, 12>), g_, b_, lds, s, a, ##__VA_ARGS__); break; \
      case 16: hipLaunchKernelGGL((KERNEL<T, 16>), g_, b_, lds, s, a, ##__VA_ARGS__); break; \
    }                                                                                       \
  } while (0)

template <typename T> __device__ __forceinline__ double src_press(const KArgs &a, long l, int i) {
  if (!a.energy) {
    const double cs = (double)(T)a.cs_iso[i];
    return ld<T>(a.rho, l) * cs * cs;
  }
  return (a.gamma - 1.0) * ld<T>(a.en, l);
}

#include "dust_fluid.h"

static dim3 cell_grid(const KArgs &a, int rings) {
  int bx = a.ns < 256 ? a.ns : 256;
  return dim3((a.ns + bx - 1) / bx, rings);
}
static dim3 cell_block(const KArgs &a) { return dim3(a.ns < 256 ? a.ns : 256); }
// the velocity/boundary kernel's workgroup: the tuned width, at most a ring
// in whole wavefronts
static int finish_bx(const KArgs &a) {
  const int w = (a.tune_finish_block == 64 || a.tune_finish_block == 128) ? a.tune_finish_block : 256;
  return a.ns < w ? (a.ns + 63) / 64 * 64 : w;
}

template <typename T> void launch_kernel(int id, const KArgs &a, hipStream_t s) {
  switch (id) {
    case KID_CFL:
      if (a.sg) RING_DISPATCH_K(wide_k(a.ns), k_cfl_ring_sg, T, a, s, 0);
      else RING_DISPATCH_K(wide_k(a.ns), k_cfl_ring, T, a, s, 0);
      break;
    case KID_CONTROL:
      if (a.accrete) hipLaunchKernelGGL((k_control<T, true>), dim3(1), dim3(CtrlBlock<true>::n), 0, s, a);
      else hipLaunchKernelGGL((k_control<T, false>), dim3(1), dim3(CtrlBlock<false>::n), 0, s, a);
      break;
    case KID_EOS_STEP: RING_DISPATCH(k_eos_step, T, a, s, 0); break;
    case KID_VISC1D: hipLaunchKernelGGL(k_visc1d, dim3(1), dim3(V1D_TB), 0, s, a); break;
    case KID_NONREFLECTING:
      hipLaunchKernelGGL(k_nonreflecting<T>, dim3(2), dim3(NR_TB), 0, s, a);
      break;
    case KID_EVANESCENT:
      hipLaunchKernelGGL(k_evanescent<T>, dim3(a.wkz_n_in + (a.nr - a.wkz_i_out)), dim3(EV_TB), 0, s, a);
      break;
    case KID_SOURCE:
      launch_source<T>(a, s);
      break;
    case KID_ENERGY: RING_DISPATCH(k_energy, T, a, s, 0); break;
    case KID_TRANSPORT_AZI: launch_transport<T>(a, s); break;
    case KID_FINISH: {
      const int bx = finish_bx(a);
      hipLaunchKernelGGL(k_finish<T>, dim3((a.ns + bx - 1) / bx, a.nr + 2), dim3(bx), 0, s, a);
      break;
    }
    case KID_DUST_MOVE:
    case KID_DUST_SCAN:
    case KID_DUST_SCATTER:
    case KID_DUST_RANK:
    case KID_DUST_DEPOSIT: launch_dust_kernel<T>(id, a, s); break;
    case KID_DF_CFL:
    case KID_DF_AXISG:
    case KID_DF_SOURCE:
    case KID_DF_STRESS:
    case KID_DF_VISC:
    case KID_DF_SUBSTEP2:
    case KID_DF_TRANSPORT_AZI:
    case KID_DF_FINISH:
      // the dust fluid runs with FP64 storage only (the context refuses it
      // otherwise)
      if (sizeof(T) == sizeof(double)) launch_df_kernel(id, a, s);
      break;
    default: launch_sg_kernel<T>(id, a, s); break;
  }
}

template <typename T> void launch_eos_pre(const KArgs &a, hipStream_t s) {
  RING_DISPATCH(k_eos, T, a, s, 0);
}
template <typename T> void launch_potential(const KArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_potential<T>, cell_grid(a, a.nr), cell_block(a), 0, s, a);
}
template <typename T> void launch_visc_stress_state(const KArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_visc_stress<T>, cell_grid(a, a.nr), cell_block(a), 0, s, a, 1);
}
void launch_algogas_begin(const KArgs &a, double DT, hipStream_t s) {
  hipLaunchKernelGGL(k_algogas_begin, dim3(1), dim3(64), 0, s, a, DT);
}

template <typename T> void prepare_kernels(const KArgs &a) {
  if (a.sg && !a.sg_zero) sg_prepare<T>(a);
}
template void prepare_kernels<double>(const KArgs &);
template void prepare_kernels<float>(const KArgs &);
template void launch_kernel<double>(int, const KArgs &, hipStream_t);
template void launch_kernel<float>(int, const KArgs &, hipStream_t);
template void launch_eos_pre<double>(const KArgs &, hipStream_t);
template void launch_eos_pre<float>(const KArgs &, hipStream_t);
template void launch_potential<double>(const KArgs &, hipStream_t);
template void launch_potential<float>(const KArgs &, hipStream_t);
template void launch_visc_stress_state<double>(const KArgs &, hipStream_t);
template void launch_visc_stress_state<float>(const KArgs &, hipStream_t);

// ------------------------------------------------------------------------
// per-DT diagnostics (src/main.c:291-394): outside AlgoGas, on the state
// the last call left
// ------------------------------------------------------------------------

// Per ring i, part[q * nr + i] for q = 0 GasTotalMass (src/SideEuler.c:
// 15-36), 1 GasMomentum (src/SideEuler.c:114-146), 2 GasTotalEnergy
// (src/SideEuler.c:149-180; the energy grid of an isothermal run holds
// zeros), then for body k, 3 + 4k + {0 fx, 1 fx Hill-cut, 2 fy, 3 fy
// Hill-cut} of ComputeForce (src/Force.c:155-214); the ring's inner/outer
// side is decided in k_diag_reduce.  Compensated FP64 sums, fixed block
// reduction order.
template <typename T, int K> __global__ void __launch_bounds__(RING_LB(K)) k_diag_ring(KArgs a, DiagBodies b,
                                                                                       double *part) {
  __shared__ double sh[16 * 4];
  const dfargo_ctrl *c = a.ctrl;
  const int i = blockIdx.x, ns = a.ns, nr = a.nr, t = threadIdx.x, TB = ns / K;
  const bool on = t < TB; // the block is whole wavefronts
  const long base = (long)i * ns;
  const double Rm = a.Rmed[i], S = a.Surf[i], Of = c->omega_frame;
  const double wr = (a.Rsup[i] - a.Rinf[i]);
  CSum m = {0, 0}, mom = {0, 0}, en = {0, 0};
  for (int k = 0; on && k < K; k++) {
    const int j = t + k * TB;
    const long l = base + j;
    const double d = ld<T>(a.rho, l);
    const double vtl = ld<T>(a.vt, l), vtp = ld<T>(a.vt, (j < ns - 1) ? l + 1 : base);
    const double vt_cent = 0.5 * (vtl + vtp) + Rm * Of;
    double vr_cent = (Rm - a.Rinf[i]) * ld<T>(a.vr, l + ns) + (a.Rsup[i] - Rm) * ld<T>(a.vr, l);
    vr_cent /= wr;
    const double e = a.energy ? ld<T>(a.en, l) : 0.0;
    m.add(S * d);
    mom.add(S * d * Rm * vt_cent);
    en.add(0.5 * S * d * (vr_cent * vr_cent + vt_cent * vt_cent) + S * e - S * d * pot_at(a, c, i, j));
  }
  double v[3] = {m.value(), mom.value(), en.value()};
  block_sum_n<3>(v, sh);
  if (t == 0)
    for (int q = 0; q < 3; q++) part[(long)q * nr + i] = v[q];
  for (int bd = 0; bd < b.n; bd++) {
    const double x = b.x[bd], y = b.y[bd], rsm = b.rsm[bd], cutoff = a.exclude_hill_factor * b.rh[bd];
    CSum f[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    for (int k = 0; on && k < K; k++) {
      const int j = t + k * TB;
      const double xc = Rm * a.CosAz[j], yc = Rm * a.SinAz[j];
      const double cellmass = S * ld<T>(a.rho, base + j);
      const double dx = xc - x, dy = yc - y;
      const double d2 = dx * dx + dy * dy;
      const double planet_distance = sqrt(d2);
      const double dist2 = d2 + rsm * rsm;
      const double distance = sqrt(dist2);
      const double InvDist3 = 1.0 / dist2 / distance;
      double hill_cut;
      if (planet_distance / cutoff < 0.5) hill_cut = 0.0;
      else if (planet_distance > cutoff) hill_cut = 1.0;
      else hill_cut = pow(sin((planet_distance / cutoff - .5) * DF_PI), 2.);
      f[0].add(DF_G * cellmass * dx * InvDist3 * 1.0);
      f[1].add(DF_G * cellmass * dx * InvDist3 * hill_cut);
      f[2].add(DF_G * cellmass * dy * InvDist3 * 1.0);
      f[3].add(DF_G * cellmass * dy * InvDist3 * hill_cut);
    }
    double w[4] = {f[0].value(), f[1].value(), f[2].value(), f[3].value()};
    block_sum_n<4>(w, sh);
    if (t == 0)
      for (int q = 0; q < 4; q++) part[(long)(3 + 4 * bd + q) * nr + i] = w[q];
  }
}

// Ring sums in ring order (compensated): out[0..2] the budgets, then for
// body k out[3 + 8k ..] = fx inner, fx Hill-cut inner, fx outer, fx
// Hill-cut outer, fy inner, fy Hill-cut inner, fy outer, fy Hill-cut outer
// (GlobalForce's order; a ring is inner when Rmed < a_k).
__global__ void __launch_bounds__(64) k_diag_reduce(KArgs a, DiagBodies b, const double *part, double *out) {
  const int q = threadIdx.x, nr = a.nr;
  if (q < 3) {
    CSum s = {0, 0};
    for (int i = 0; i < nr; i++) s.add(part[(long)q * nr + i]);
    out[q] = s.value();
  }
  const int bd = q / 4, comp = q % 4;
  if (bd < b.n) {
    CSum in = {0, 0}, outer = {0, 0};
    const double *pp = part + (long)(3 + 4 * bd + comp) * nr;
    for (int i = 0; i < nr; i++) {
      if (a.Rmed[i] < b.a[bd]) in.add(pp[i]);
      else outer.add(pp[i]);
    }
    // comp: 0 fx, 1 fx Hill-cut, 2 fy, 3 fy Hill-cut -> GlobalForce slots
    const int axis = comp / 2, hill = comp % 2;
    out[3 + 8 * bd + 4 * axis + hill] = in.value();
    out[3 + 8 * bd + 4 * axis + 2 + hill] = outer.value();
  }
}

template <typename T> void launch_diagnostics(const KArgs &a, const DiagBodies &b, double *part, double *out,
                                              hipStream_t s) {
  RING_DISPATCH(k_diag_ring, T, a, s, 0, b, part);
  hipLaunchKernelGGL(k_diag_reduce, dim3(1), dim3(64), 0, s, a, b, (const double *)part, out);
}
template void launch_diagnostics<double>(const KArgs &, const DiagBodies &, double *, double *, hipStream_t);
template void launch_diagnostics<float>(const KArgs &, const DiagBodies &, double *, double *, hipStream_t);

