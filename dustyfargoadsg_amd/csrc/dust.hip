// dust.hip -- Lagrangian dust particles of one sub-step on CDNA4
// (SemiUpdateDustPositions, src/DustUpdate.c:6-138; UpdateDustVelocities,
// src/DustUpdate.c:267-435; interpolation, src/Dsys.c:265-1149; the
// start-up interpolation of src/main.c:287).
//
// One thread per particle moves it, finds its cell, gathers the gas
// quantities of its three stencils (unrolled per interpolation scheme),
// computes its Stokes number and drag, updates its velocity, stores its
// stencil weights and takes a slot in its cell's bucket.  The feedback
// deposit (the scatter half of interpolation) is turned into a gather so
// that no float atomics decide the summation order: the bucket counts are
// scanned ring by ring, the particles scattered to their slots, each
// particle ranked in its bucket by its id, and wavefronts that walk outwards
// pass over each bucket once and add it to the cells its stencils reach, in a
// fixed order.  Every sum is thus deterministic; against the reference's
// particle-index order only its rounding differs.  With its rank a particle is also copied, in
// bucket order, into the other of two particle sets: the next sub-step finds
// neighbouring particles in neighbouring memory, and its gathers and
// deposit read few cache lines per wavefront.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace {

template <typename T> __device__ __forceinline__ double ldd(const void *p, long i) {
  return (double)((const T *)p)[i];
}

// AspectRatio (src/Viscosity.c:107-122)
__device__ double d_aspect(const KArgs &a, double rad) {
  double ar = a.aspect_ratio;
  const double rmin = a.transition_radius - a.transition_width * a.aspect_ratio;
  const double rmax = a.transition_radius + a.transition_width * a.aspect_ratio;
  if (rad < rmin) ar *= a.transition_ratio;
  if ((rad >= rmin) && (rad <= rmax)) ar *= exp((rmax - rad) / (rmax - rmin) * log(a.transition_ratio));
  return ar;
}

// reference azimuth of column j of a stencil: AziInf for the vtheta one,
// the cell centre otherwise; columns past either end continue the grid
// (src/Dsys.c:411-425).  Returns the wrapped column.  Branch-free: the
// table load does not wait on the column's case.
__device__ __forceinline__ int d_col(const KArgs &a, int kind, int j, double &az) {
  const int ns = a.ns;
  const double half = 0.5 * (a.pm) / (double)ns;
  const int jc = j < 0 ? 0 : (j >= ns ? ns - 1 : j);
  const double a0 = (kind == 1) ? a.Azimuth[jc] - half : a.Azimuth[jc];
  az = (j >= 0 && j < ns) ? a0 : (j < 0 ? a0 + j * a.delta_phi : a0 + (j + 1 - ns) * a.delta_phi);
  return (j < 0) ? j + ns : (j >= ns ? j - ns : j);
}

// radial distance of a stencil node: to Rinf for the vr stencil, to Rmed
// otherwise, logarithmic on a logarithmic grid
// (0 outside the grid; computed branch-free so that the table loads of a
// stencil issue together)
__device__ __forceinline__ double d_dr(const KArgs &a, int kind, int i, double rp) {
  const bool inr = (i >= 0) && (i <= a.nr - 1);
  const int ic = i < 0 ? 0 : (i > a.nr - 1 ? a.nr - 1 : i);
  const double ref = (kind == 0) ? a.Rinf[ic] : a.Rmed[ic];
  const double d = a.log_grid ? fabs(log(rp / ref)) : fabs(rp - ref);
  return inr ? d : 0.0;
}

__device__ __forceinline__ bool d_in_grid(const KArgs &a, double r) {
  return (r >= a.Rinf[0]) && (r < a.Rsup[a.nr - 1]);
}

// keep an azimuth in [AziInf[0], AziSup[ns-1]] (src/DustUpdate.c:38-45)
__device__ __forceinline__ double d_wrap(const KArgs &a, double th) {
  if (th < a.aziinf0) th += (a.azisup_last - a.aziinf0);
  if (th > a.azisup_last) th -= (a.azisup_last - a.aziinf0);
  return th;
}

// cell of a particle inside the grid: ip is the last ring with
// Rinf[ip] <= r (the linear search of src/Dsys.c:363-365), found from the
// grid's spacing and corrected against the table, jp from the azimuth.
// False when jp falls outside the grid, which only an azimuth outside
// [AziInf[0], AziSup[ns-1]] can produce.
__device__ bool d_cell(const KArgs &a, double rp, double tp, int &ip, int &jp) {
  const int nr = a.nr;
  double g = a.log_grid ? log(rp / a.Rinf[0]) / a.d_ring_step : (rp - a.Rinf[0]) / a.d_ring_step;
  int i = (int)g;
  i = i < 0 ? 0 : (i > nr - 1 ? nr - 1 : i);
  while (i > 0 && rp < a.Rinf[i]) i--;
  while (i < nr - 1 && rp >= a.Rinf[i + 1]) i++;
  ip = i;
  jp = (int)floor(a.ns * (tp - a.aziinf0) / (a.azisup_last - a.aziinf0));
  if (jp == a.ns) jp = 0;
  return jp >= 0 && jp < a.ns;
}

// ------------------------------------------------------------------------
// stencils, specialised per interpolation scheme S: node counts, first
// node and the separable weights (wr depends on the radial distance only,
// wt on the azimuthal one)

__host__ __device__ constexpr int nodes_r(int S, int kind) {
  return S == DFARGO_INTERP_NGP ? (kind == 0 ? 2 : 1) : (S == DFARGO_INTERP_CIC ? 2 : 3);
}
__host__ __device__ constexpr int nodes_t(int S, int kind) {
  return S == DFARGO_INTERP_NGP ? (kind == 1 ? 2 : 1) : (S == DFARGO_INTERP_CIC ? 2 : 3);
}

// first ring and column of stencil `kind` (0 vr, 1 vtheta, 2 cell-centred)
// for a particle in cell (ip, jp) (src/Dsys.c:371-406,456-488,620-639): the
// rings stay within ip-1 .. ip+1 and the columns within jp-1 .. jp+2, the
// neighbourhood the deposit gathers from
// (az_jp = Azimuth[jp], rmed_ip = Rmed[ip])
template <int S> __device__ __forceinline__ int first_ring(int kind, int ip, double rp, double rmed_ip) {
  if (S == DFARGO_INTERP_NGP) return ip;
  if (S == DFARGO_INTERP_CIC) return (kind != 0 && rp < rmed_ip) ? ip - 1 : ip;
  return ip - 1;
}
template <int S> __device__ __forceinline__ int first_col(int kind, int jp, double tp, double az_jp) {
  if (S == DFARGO_INTERP_NGP) return jp;
  if (S == DFARGO_INTERP_CIC) return (kind != 1 && tp < az_jp) ? jp - 1 : jp;
  return ((kind == 1 && tp > az_jp) ? jp + 1 : jp) - 1;
}

// the weights of src/Dsys.c:407-441,490-524,640-665, one factor at a time
template <int S> __device__ __forceinline__ double w_rad(int kind, double dr, double delta) {
  if (S == DFARGO_INTERP_NGP) return (kind == 0) ? ((dr < 0.5 * delta) ? 1.0 : 0.0) : 1.0;
  if (S == DFARGO_INTERP_CIC) return 1.0 - dr / delta;
  double w = 0.0;
  if (dr < 0.5 * delta) w = 0.75 - dr * dr / delta / delta;
  if ((dr >= 0.5 * delta) && (dr <= 1.5 * delta)) w = 0.5 * (1.5 - dr / delta) * (1.5 - dr / delta);
  if (dr > 1.5 * delta) w = 0.0;
  return w;
}
template <int S> __device__ __forceinline__ double w_azi(int kind, double dphi, double delta) {
  if (S == DFARGO_INTERP_NGP) return (kind == 1) ? ((dphi < 0.5 * delta) ? 1.0 : 0.0) : 1.0;
  if (S == DFARGO_INTERP_CIC) return 1.0 - dphi / delta;
  double w = 0.0;
  if (dphi < 0.5 * delta) w = 0.75 - dphi * dphi / delta / delta;
  if ((dphi >= 0.5 * delta) && (dphi <= 1.5 * delta)) w = 0.5 * (1.5 - dphi / delta) * (1.5 - dphi / delta);
  if (dphi > 1.5 * delta) w = 0.0;
  return w;
}

// The weights of a stencil are products of a radial factor, the vr stencil's
// own or the one the other two share (they stand on the same rings), and an
// azimuthal one, the vtheta stencil's own or the one the other two share: four
// sets of three, at 3 w .. 3 w + 2 of p_w, stored for the deposit when asked.
enum { W_RAD_VR = 0, W_AZI_CENTRE = 1, W_RAD_CENTRE = 2, W_AZI_VT = 3 };
__host__ __device__ constexpr int w_rad_set(int kind) { return kind == 0 ? W_RAD_VR : W_RAD_CENTRE; }
__host__ __device__ constexpr int w_azi_set(int kind) { return kind == 1 ? W_AZI_VT : W_AZI_CENTRE; }
template <int S, int KIND>
__device__ __forceinline__ int rad_weights(const KArgs &a, int ip, double rp, double rmed_ip, double (&wr)[3],
                                           bool store, int k) {
  constexpr int NI = nodes_r(S, KIND);
  const int imin = first_ring<S>(KIND, ip, rp, rmed_ip);
#pragma unroll
  for (int q = 0; q < NI; q++) wr[q] = w_rad<S>(KIND, d_dr(a, KIND, imin + q, rp), a.delta_r);
  if (store)
#pragma unroll
    for (int q = 0; q < NI; q++) a.p_w[(3 * w_rad_set(KIND) + q) * (long)a.d_np + k] = wr[q];
  return imin;
}
template <int S, int KIND>
__device__ __forceinline__ int azi_weights(const KArgs &a, int jp, double tp, double az_jp, double (&wt)[3],
                                           int (&col)[3], bool store, int k) {
  constexpr int NJ = nodes_t(S, KIND);
  const int jmin = first_col<S>(KIND, jp, tp, az_jp);
#pragma unroll
  for (int q = 0; q < NJ; q++) {
    double az;
    col[q] = d_col(a, KIND, jmin + q, az);
    wt[q] = w_azi<S>(KIND, fabs(tp - az), a.delta_phi);
  }
  if (store)
#pragma unroll
    for (int q = 0; q < NJ; q++) a.p_w[(3 * w_azi_set(KIND) + q) * (long)a.d_np + k] = wt[q];
  return jmin;
}

// Gathers of stencil KIND: up to four grids at its nodes, all loads issued
// before the sums, which then run in the reference's order (columns outer,
// rings inner) over the nodes inside the grid.  Grid g1 of the
// cell-centred stencil may be the per-ring isothermal sound speed; g2 and
// g3 are read always (a valid grid stands in for an unused one) and summed
// only when use2 / use3.  With a frame rate, g0 is vtheta and is read as
// vt + Rmed frame at each node.
template <typename T, int S, int KIND>
__device__ __forceinline__ void stencil_gather(const KArgs &a, const double (&wr)[3], const double (&wt)[3],
                                               const int (&col)[3], int imin, const void *g0, const void *g1,
                                               const void *g2, const void *g3, bool iso1, bool use2, bool use3,
                                               double &s0, double &s1, double &s2, double &s3,
                                               double frame = 0.0) {
  constexpr int NI = nodes_r(S, KIND), NJ = nodes_t(S, KIND);
  const int nr = a.nr, ns = a.ns;
  bool inr[NI];
  int ic[NI];
#pragma unroll
  for (int p = 0; p < NI; p++) {
    const int i = imin + p;
    inr[p] = (i >= 0) && (i <= nr - 1);
    ic[p] = i < 0 ? 0 : (i > nr - 1 ? nr - 1 : i);
  }
  double x0[NJ][NI], x1[NJ][NI], x2[NJ][NI], x3[NJ][NI];
#pragma unroll
  for (int q = 0; q < NJ; q++)
#pragma unroll
    for (int p = 0; p < NI; p++) {
      const long l = (long)ic[p] * ns + col[q];
      x0[q][p] = ldd<T>(g0, l);
      if (frame != 0.0) x0[q][p] = x0[q][p] + a.Rmed[ic[p]] * frame;
      x1[q][p] = iso1 ? (double)(T)((const double *)g1)[ic[p]] : ldd<T>(g1, l);
      x2[q][p] = ldd<T>(g2, l);
      x3[q][p] = ldd<T>(g3, l);
    }
#pragma unroll
  for (int q = 0; q < NJ; q++)
#pragma unroll
    for (int p = 0; p < NI; p++) {
      const double w = wr[p] * wt[q];
      s0 = inr[p] ? s0 + (w * x0[q][p]) : s0;
      s1 = inr[p] ? s1 + (w * x1[q][p]) : s1;
      if (use2) s2 = inr[p] ? s2 + (w * x2[q][p]) : s2;
      if (use3) s3 = inr[p] ? s3 + (w * x3[q][p]) : s3;
    }
}

// does this sub-step (or the start-up) need the buckets and the deposit?
__device__ __forceinline__ bool dust_deposit_needed(const KArgs &a, const dfargo_ctrl *c, int force) {
  return force || a.d_feedback || !c->go_next;
}

// One particle per thread.  In a sub-step: SemiUpdateDustPositions over
// 2 dt, interpolation (gathers, Stokes number, drag), UpdateDustVelocities
// and RotateDsys by OmegaFrame dt; the particle is counted into its cell's
// bucket at the position before the rotation, where the reference's
// interpolation deposits it.  At start-up: the interpolation only, with the
// given time step.  The gas vtheta is read in the fixed frame, vt + Rmed
// OmegaFrame per cell (src/Dsys.c:316), with the frame rate before this
// sub-step's frame update.  A particle outside the grid keeps its state
// and has no cell (p_cell = -1).  Bound by the latency of its gathers (VALU busy
// 40 %) at the four wavefronts a SIMD that 126 registers allow (10^6 particles,
// CIC: 118 us; 176 us when each stencil formed both its factors, in 213
// registers, and each particle the planet's azimuth and smoothing length).
template <typename T, int S>
__global__ void __launch_bounds__(256) k_dust_move(KArgs a, int startup, double timestep0) {
  dfargo_ctrl *c = a.ctrl;
  if (!startup && !c->active) return;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int nr = a.nr, ns = a.ns;
  const double timestep = startup ? timestep0 : c->dt;
  const bool store01 = a.d_feedback, store2 = startup || !c->go_next || (a.d_feedback && a.energy);
  const DustSet P = a.pset[c->pset];
  unsigned long long ts_bits = ~0ull;
  bool outside = false;
  if (k < a.d_np) {
    double r = P.r[k], th = P.th[k];
    const double vrd = P.vr[k], vtd = P.vth[k];
    if (!startup && d_in_grid(a, r)) {
      const double rnew = r + vrd * 0.5 * (2. * timestep);
      th += vtd * r * 0.25 * (2. * timestep) * (1.0 / (r * r) + 1.0 / (rnew * rnew));
      th = d_wrap(a, th);
      th = d_wrap(a, th);
      r = rnew;
      P.r[k] = r;
    }
    // RotateDsys (src/Dsys.c:1153-1169) by the frame's new rate (in the
    // fixed frame a wrap only); the stencils below use the azimuth before it
    if (!startup) P.th[k] = d_wrap(a, th - c->omega_frame * timestep);
    const double frame = startup ? c->omega_frame : c->omega_prev;
    int ip, jp;
    if (!d_in_grid(a, r) || !d_cell(a, r, th, ip, jp)) {
      a.p_cell[k] = -1;
      outside = true;
    } else {
      const int cell = ip * ns + jp;
      a.p_cell[k] = cell;
      a.p_slot[k] = atomicAdd(&a.cell_count[cell], 1);
      const double rp = r, tp = th;
      const double az_jp = a.Azimuth[jp], rmed_ip = a.Rmed[ip];
      double wr0[3], wr[3], wt1[3], wt[3];
      int col1[3], col[3];
      const int i0 = rad_weights<S, 0>(a, ip, rp, rmed_ip, wr0, store01, k);
      const int ic = rad_weights<S, 2>(a, ip, rp, rmed_ip, wr, store01 || store2, k);
      const int jc = azi_weights<S, 2>(a, jp, tp, az_jp, wt, col, store01 || store2, k);
      const int j1 = azi_weights<S, 1>(a, jp, tp, az_jp, wt1, col1, store01, k);
      const int base = (i0 - ip + 1) | (jc - jp + 1) << 2 | (ic - ip + 1) << 4 | (j1 - jp + 1) << 6 |
                       (ic - ip + 1) << 8 | (jc - jp + 1) << 10;
      // vr stencil: gas vr, pressure gradient, indirect and SG accelerations
      double vrg = 0.0, radgradp = 0.0, radind = 0.0, radsg = 0.0;
      stencil_gather<T, S, 0>(a, wr0, wt, col, i0, a.vr, a.radgradp, a.radindacc, a.radsgacc, false,
                              a.indirect_term, a.sg, vrg, radgradp, radind, radsg);
      // vtheta stencil
      double vtg = 0.0, azigradp = 0.0, aziind = 0.0, azisg = 0.0;
      stencil_gather<T, S, 1>(a, wr, wt1, col1, ic, a.vt, a.azigradp, a.aziindacc, a.azisgacc, false,
                              a.indirect_term, a.sg, vtg, azigradp, aziind, azisg, frame);
      // cell-centred stencil: density and the sound speed the sub-step
      // started with
      double densg = 0.0, csg = 0.0, unused0 = 0.0, unused1 = 0.0;
      stencil_gather<T, S, 2>(a, wr, wt, col, ic, a.rho,
                              a.energy ? ((startup ? a.cs : a.cs_old)) : (const void *)a.cs_iso, a.rho, a.rho,
                              !a.energy, false, false, densg, csg, unused0, unused1);
      a.p_base[k] = base;
      // Stokes number (Paardekooper 2007, src/Dsys.c:733-790)
      double vrp = vrd, vtp = vtd;
      const double densg_cgs = 0.1 * densg * a.d_unit_mass * a.d_len_m2;
      const double lambda = 3.34e-8 * (1.0 / densg_cgs) * d_aspect(a, rp) * rp;
      const double Kn = 0.5 * lambda / P.size[k];
      const double Mach = sqrt((vrp - vrg) * (vrp - vrg) + (vtp - vtg) * (vtp - vtg)) / csg;
      const double f_D = sqrt(1.0 + 9.0 * DF_PI * Mach * Mach / 128.0);
      const double Re = 3.0 * sqrt(DF_PI / 8.0) * Mach / Kn;
      double k_D = 0.0;
      if (Re <= 500.0)
        k_D = 1.0 + 0.15 * pow(Re, 0.687);
      else {
        if ((Re > 500.0) && (Re <= 1500.0)) k_D = 3.96e-6 * pow(Re, 2.4);
        if (Re > 1500.0) k_D = 0.11 * Re;
      }
      const double kn1 = 3.0 * Kn + 1.0;
      const double Cdrag = (kn1 * kn1) * (1.0 / (9.0 * Kn * Kn * f_D + 3.0 * Kn * k_D));
      const double St = 0.5 * DF_PI * Cdrag * P.size[k] * a.d_rho_code / densg;
      const double r15 = rp * sqrt(rp);
      const double Ts = St * r15;
      ts_bits = (unsigned long long)__double_as_longlong(Ts);
      P.stokes[k] = St;
      // drag acceleration (src/Dsys.c:800-830)
      if ((Ts < timestep) && a.d_sfta) {
        vrp = vrg + Ts * radgradp / densg;
        vtp = vtg + Ts * azigradp / densg;
      }
      a.p_raddrag[k] = -(vrp - vrg) / Ts;
      a.p_azidrag[k] = -(vtp - vtg) / Ts;
      a.p_ts[k] = Ts;
      a.p_dv2[k] = (vrp - vrg) * (vrp - vrg) + (vtp - vtg) * (vtp - vtg);
      if (!startup) {
        // UpdateDustVelocities (src/DustUpdate.c:290-424) from the velocity
        // the particle had before the drag estimate; its stopping time is
        // Ts (same St, same radius)
        const double rd = r, td = th, stoptime = Ts;
        int local_feel_disk = a.d_feel_disk;
        if ((rd < a.rmin) || (rd > a.rmax)) local_feel_disk = 0;
        if ((stoptime < timestep) && a.d_sfta) {
          const double vth_new = vtg + stoptime * azigradp / densg;
          P.vr[k] = vrg + stoptime * radgradp / densg;
          P.vth[k] = vth_new;
          P.l[k] = rd * vth_new;
        } else {
          double FgravR = -(1.0 / (rd * rd)), FgravTh = 0.;
          if ((fabs(FgravR + vtd * vtd / rd) < 1e-15) && (!a.d_feel_planets) && (!a.d_feel_disk) &&
              (!a.d_feel_sg))
            FgravR = -vtd * vtd / rd;
          if (a.d_feel_planets) {
            for (int q = 0; q < c->nb; q++) {
              const double rpl = c->dust_pl_r[q], tpl = c->dust_pl_t[q], mp = c->dust_pl_m[q];
              const double eps = c->dust_pl_eps[q];
              double sn, cn;
              sincos(td - tpl, &sn, &cn);
              const double dd = sqrt(rd * rd + rpl * rpl - 2.0 * rd * rpl * cn + eps * eps);
              const double id3 = 1.0 / (dd * dd * dd);
              FgravR += mp * (rpl * cn - rd) * id3;
              FgravTh += -mp * rpl * sn * id3;
            }
          }
          if (a.indirect_term) {
            FgravR += radind;
            FgravTh += aziind;
          }
          if (a.sg && a.d_feel_sg) {
            FgravR += radsg;
            FgravTh += azisg;
          }
          const double den = 1.0 + local_feel_disk * timestep / stoptime;
          const double numTh = (vtd - vtg) + timestep * (FgravTh - vrd * vtd / rd);
          const double vth_new = vtg + numTh / den;
          P.vth[k] = vth_new;
          const double numR = (vrd - vrg) + timestep * (FgravR + (vth_new * vth_new) / rd);
          P.vr[k] = vrg + numR / den;
        }
      }
    }
  }
  // the particles outside the grid take slots of their own list, one
  // atomic per wavefront
  {
    const unsigned long long m = __ballot(outside);
    const int lane = threadIdx.x & 63;
    if (outside) {
      const int leader = __ffsll((long long)m) - 1;
      int base0 = 0;
      if (lane == leader) base0 = atomicAdd(&c->out_count, __popcll(m));
      base0 = __shfl(base0, leader, 64);
      a.p_slot[k] = base0 + __popcll(m & ((1ull << lane) - 1ull));
    }
  }
  // minimum stopping time of the block (positive doubles order like their
  // bit patterns), one entry per block: the control kernel of the next
  // sub-step takes the minimum over the blocks (no same-address atomics)
  __shared__ unsigned long long wmin[4];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = (unsigned long long)__shfl_xor((long)ts_bits, off, 64);
    ts_bits = (o < ts_bits) ? o : ts_bits;
  }
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = ts_bits;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long m = wmin[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = (wmin[w] < m) ? wmin[w] : m;
    a.p_tsmin[blockIdx.x] = m;
  }
}

// bucket counts zeroed (start-up; in the sub-steps the CFL kernel does it,
// and the control kernel zeroes the count of particles outside the grid)
__global__ void __launch_bounds__(256) k_dust_zero(KArgs a) {
  const long n = (long)a.nr * a.ns;
  for (long l = blockIdx.x * (long)blockDim.x + threadIdx.x; l < n; l += (long)gridDim.x * blockDim.x)
    a.cell_count[l] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) a.ctrl->out_count = 0;
}

// exclusive scan of x over the block (1024 threads max): wavefront
// shuffles, then the wavefront totals; returns the exclusive prefix and
// the block total
__device__ __forceinline__ int block_exclusive_scan(int x, int *wsum, int &total) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, nw = (blockDim.x + 63) >> 6;
  int v = x;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(v, off, 64);
    if (lane >= off) v += y;
  }
  if (lane == 63 || t == (int)blockDim.x - 1) wsum[w] = v;
  __syncthreads();
  if (w == 0) {
    int s = (lane < nw) ? wsum[lane] : 0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(s, off, 64);
      if (lane >= off) s += y;
    }
    if (lane < nw) wsum[lane] = s;
  }
  __syncthreads();
  total = wsum[nw - 1];
  const int excl = v - x + (w > 0 ? wsum[w - 1] : 0);
  __syncthreads();
  return excl;
}

// Bucket starts, one block per ring: the exclusive scan of the ring's
// counts (ring-local starts) and the ring total
__global__ void __launch_bounds__(1024) k_dust_ring_scan(KArgs a, int force) {
  __shared__ int wsum[16];
  const dfargo_ctrl *c = a.ctrl;
  if (!force && !c->active) return;
  const int i = blockIdx.x, ns = a.ns, t = threadIdx.x, nt = blockDim.x;
  const int per = (ns + nt - 1) / nt, j0 = t * per, j1 = min(j0 + per, ns);
  const long base = (long)i * ns;
  int s = 0;
  for (int j = j0; j < j1; j++) s += a.cell_count[base + j];
  int total;
  int excl = block_exclusive_scan(s, wsum, total);
  for (int j = j0; j < j1; j++) {
    a.cell_local[base + j] = excl;
    excl += a.cell_count[base + j];
  }
  if (t == 0) a.ring_tot[i] = total;
}

// ring offsets: exclusive scan of the ring totals, one block; ring_off[nr]
// is the number of particles inside the grid
__global__ void __launch_bounds__(1024) k_dust_ring_offsets(KArgs a, int force) {
  __shared__ int wsum[16];
  const dfargo_ctrl *c = a.ctrl;
  if (!force && !c->active) return;
  const int nr = a.nr, t = threadIdx.x, nt = blockDim.x;
  int carry = 0;
  for (int b = 0; b < nr; b += nt) {
    const int v = (b + t < nr) ? a.ring_tot[b + t] : 0;
    int tot;
    const int ex = block_exclusive_scan(v, wsum, tot);
    if (b + t < nr) a.ring_off[b + t] = carry + ex;
    carry += tot;
  }
  if (t == 0) a.ring_off[nr] = carry;
}

// particles into their cell's bucket, at the slot their count gave them
// (id and position)
__global__ void __launch_bounds__(256) k_dust_scatter(KArgs a, int force) {
  const dfargo_ctrl *c = a.ctrl;
  if (!force && !c->active) return;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= a.d_np) return;
  const int cell = a.p_cell[k];
  if (cell < 0) return; // outside the grid: k_dust_rank places it
  const unsigned long long id = (unsigned long long)(unsigned)a.pset[c->pset].id[k];
  a.p_sorted[a.ring_off[cell / a.ns] + a.cell_local[cell] + a.p_slot[k]] = (id << 32) | (unsigned)k;
}

// Each particle's rank in its bucket by particle index, one particle per
// thread: the smaller entries of the bucket counted.  The entry goes to its
// place with what the deposit needs of it, (first nodes << 32 | position), and
// in a sub-step the particle to the same place of the other set (the particles
// outside the grid after those inside).  The threads of a bucket read the same
// entries, so a crowded cell costs its particles a pass over it side by side;
// sorting each bucket by one thread took 19 us for a smooth disc of 10^6
// particles and 194 us once the grains had gathered at the gap's edges.
__global__ void __launch_bounds__(256) k_dust_rank(KArgs a, int force) {
  const dfargo_ctrl *c = a.ctrl;
  if (!force && !c->active) return;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= a.d_np) return;
  const int cell = a.p_cell[k];
  const DustSet A = a.pset[c->pset], B = a.pset[c->pset ^ 1];
  const int id = A.id[k];
  int dest;
  if (cell < 0) {
    dest = a.ring_off[a.nr] + a.p_slot[k];
  } else {
    const unsigned long long mine = ((unsigned long long)(unsigned)id << 32) | (unsigned)k;
    const int start = a.ring_off[cell / a.ns] + a.cell_local[cell], n = a.cell_count[cell];
    const unsigned long long *b = a.p_sorted + start;
    int rank = 0;
    if (n > 1) {
      int x = 0;
      for (; x + 4 <= n; x += 4) rank += (b[x] < mine) + (b[x + 1] < mine) + (b[x + 2] < mine) + (b[x + 3] < mine);
      for (; x < n; x++) rank += b[x] < mine;
    }
    dest = start + rank;
    a.p_entry[dest] = ((unsigned long long)(unsigned)a.p_base[k] << 32) | (unsigned)k;
  }
  if (force) return;
  B.r[dest] = A.r[k];
  B.th[dest] = A.th[k];
  B.vr[dest] = A.vr[k];
  B.vth[dest] = A.vth[k];
  B.l[dest] = A.l[k];
  B.size[dest] = A.size[k];
  B.stokes[dest] = A.stokes[k];
  B.id[dest] = id;
}

// The deposit: every cell collects its share of the particles whose stencils
// reach it.  A wavefront holds 64 columns, DEP_OWN of them its own, and walks
// outwards through a strip of S rings (and one ring more on each side).  A lane
// passes over its cell's bucket once, in the order of the ids, and adds each
// particle to the sums of the cells around (ring offsets R0.., column offsets
// C0.. of each stencil, in registers); the sums of neighbouring columns then
// move between lanes, those of neighbouring rings wait in registers until the
// next ring has added its part.  A bucket of more than DEP_MANY particles is
// dealt to the lanes of the wavefront and their sums added in a fixed tree, or
// the most crowded cell would set the pace of its wavefront.  The order of a
// cell's sum (rings outwards, within a ring by column offset, within a bucket by
// id or by the tree) depends on the counts alone, so a replay or another strip
// length gives the same bits; against the reference's particle-index order only
// the rounding differs.  Bound by the chain of loads entry -> weights, drag in
// each bucket.  As one thread a cell that visited the 12 buckets in reach, each
// particle's entry and weights were read up to twelve times (1024 x 3072, 10^6
// grains gathered at the gap's edges: 430 us, 301 us with the crowded cells
// dealt to wavefronts, 126 us now).
// The dust density is a diagnostic: computed at start-up and on the last
// sub-step of a call.
#define DEP_HALO 2
#define DEP_OWN (64 - 2 * DEP_HALO)
#define DEP_MANY 24
__device__ __forceinline__ double dust_wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
// the cells a particle in cell (ip, jp) can reach through stencil KIND: rings
// ip + R0 .. ip + R0 + RN - 1, columns jp + C0 .. jp + C0 + CN - 1; its first
// node is at one of RN - NI + 1 rings and CN - NJ + 1 columns (stencil_base)
template <int S, int KIND> struct Reach {
  static constexpr int NI = nodes_r(S, KIND), NJ = nodes_t(S, KIND);
  static constexpr int R0 = S == DFARGO_INTERP_NGP ? 0 : (S == DFARGO_INTERP_CIC && KIND == 0 ? 0 : -1);
  static constexpr int RN = S == DFARGO_INTERP_CIC && KIND != 0 ? NI + 1 : NI;
  static constexpr int C0 = S == DFARGO_INTERP_NGP ? 0 : (S == DFARGO_INTERP_CIC && KIND == 1 ? 0 : -1);
  static constexpr int CN = (S == DFARGO_INTERP_CIC && KIND != 1) || (S == DFARGO_INTERP_TSC && KIND == 1) ? NJ + 1 : NJ;
};
template <int S, int KIND> struct ReachSum {
  double v[Reach<S, KIND>::RN][Reach<S, KIND>::CN];
};
template <int S, int KIND> __device__ __forceinline__ void reach_clear(ReachSum<S, KIND> &s) {
#pragma unroll
  for (auto &row : s.v)
#pragma unroll
    for (double &x : row) x = 0.0;
}
// particle k with first nodes `code` added to the sums: weight x, times y and
// divided by z where they are given
template <int S, int KIND, bool Y, bool Z>
__device__ __forceinline__ void reach_add(const KArgs &a, int k, int code, double y, double z,
                                          ReachSum<S, KIND> &s) {
  using R = Reach<S, KIND>;
  const long np = a.d_np;
  const bool up = ((code >> (4 * KIND)) & 3) - 1 != R::R0, right = ((code >> (4 * KIND + 2)) & 3) - 1 != R::C0;
  double wr[R::NI], wt[R::NJ];
#pragma unroll
  for (int p = 0; p < R::NI; p++) wr[p] = a.p_w[(3 * w_rad_set(KIND) + p) * np + k];
#pragma unroll
  for (int q = 0; q < R::NJ; q++) wt[q] = a.p_w[(3 * w_azi_set(KIND) + q) * np + k];
#pragma unroll
  for (int p = 0; p < R::RN; p++)
#pragma unroll
    for (int q = 0; q < R::CN; q++) {
      // node (p, q) of the stencil if its first node is the lowest of its
      // range, (p - 1, q - 1) if it is the one after it
      const double r0 = p < R::NI ? wr[p] : 0.0, r1 = p > 0 ? wr[p - 1] : 0.0;
      const double t0 = q < R::NJ ? wt[q] : 0.0, t1 = q > 0 ? wt[q - 1] : 0.0;
      const double a_r = R::RN > R::NI && up ? r1 : r0, a_t = R::CN > R::NJ && right ? t1 : t0;
      double x = a_r * a_t;
      if (Y) x *= y;
      if (Z) x /= z;
      // a node that the particle does not reach takes nothing of it, were its
      // drag infinite
      const bool in_r = R::RN == R::NI || (up ? p > 0 : p < R::NI), in_t = R::CN == R::NJ || (right ? q > 0 : q < R::NJ);
      s.v[p][q] += in_r && in_t ? x : 0.0;
    }
}
// sum over the wavefront into lane L
template <int S, int KIND>
__device__ __forceinline__ void reach_gather(ReachSum<S, KIND> &x, bool mine, ReachSum<S, KIND> &s) {
#pragma unroll
  for (int p = 0; p < Reach<S, KIND>::RN; p++)
#pragma unroll
    for (int q = 0; q < Reach<S, KIND>::CN; q++) {
      const double t = dust_wave_sum(x.v[p][q]);
      s.v[p][q] = mine ? t : s.v[p][q];
    }
}
// the sums of this ring's buckets to the columns they belong to (neighbouring
// lanes), and to the sums of the rings below, at and above this one
template <int S, int KIND>
__device__ __forceinline__ void reach_spread(const ReachSum<S, KIND> &s, double &below, double &here, double &above) {
  using R = Reach<S, KIND>;
  const int lane = threadIdx.x;
#pragma unroll
  for (int p = 0; p < R::RN; p++) {
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < R::CN; q++) t += R::C0 + q == 0 ? s.v[p][q] : __shfl(s.v[p][q], (lane - (R::C0 + q)) & 63, 64);
    (R::R0 + p < 0 ? below : (R::R0 + p == 0 ? here : above)) += t;
  }
}
template <typename T, int S, bool E> __global__ void __launch_bounds__(64) k_dust_deposit(KArgs a, int force, int strip) {
  const dfargo_ctrl *c = a.ctrl;
  if (!force && !c->active) return;
  if (!dust_deposit_needed(a, c, force)) return;
  const int nr = a.nr, ns = a.ns, lane = threadIdx.x;
  const int j = (int)blockIdx.x * DEP_OWN + lane - DEP_HALO, i0 = blockIdx.y * strip, i1 = min(i0 + strip, nr);
  const bool own = lane >= DEP_HALO && lane < DEP_HALO + DEP_OWN && j < ns;
  const bool source = j < ns + DEP_HALO; // further right a bucket serves no cell
  int cj = j < 0 ? j + ns : j;
  cj = source ? (cj >= ns ? cj - ns : cj) : 0; // ns >= 4 > DEP_HALO
  const bool want_fb = a.d_feedback, want_e = E && a.d_feedback, want_dens = force || !c->go_next;
  const double mp = force ? c->particles_mass : c->dust_mp;
  // sums of the rings i - 1, i and i + 1
  double fr0 = 0.0, fr1 = 0.0, ft0 = 0.0, ft1 = 0.0, dd0 = 0.0, dd1 = 0.0, fe0 = 0.0, fe1 = 0.0;
  int local = 0, count = 0;
  if (i0 > 0) {
    local = a.cell_local[(long)(i0 - 1) * ns + cj];
    count = a.cell_count[(long)(i0 - 1) * ns + cj];
  }
  for (int i = i0 - 1; i <= i1; i++) {
    const int n = i >= 0 && i < nr && source ? count : 0, e0 = (i >= 0 && i < nr ? a.ring_off[i] : 0) + local;
    if (i + 1 < nr && i < i1) {
      local = a.cell_local[(long)(i + 1) * ns + cj];
      count = a.cell_count[(long)(i + 1) * ns + cj];
    }
    double fr2 = 0.0, ft2 = 0.0, dd2 = 0.0, fe2 = 0.0;
    if (__ballot(n > 0)) {
      const unsigned long long crowded = __ballot(n > DEP_MANY);
      const int few = n > DEP_MANY ? 0 : n;
      if (want_fb) {
        ReachSum<S, 0> sr;
        ReachSum<S, 1> st;
        reach_clear(sr);
        reach_clear(st);
        for (int e = e0; e < e0 + few; e++) {
          const unsigned long long entry = a.p_entry[e];
          const int k = (int)(unsigned)(entry & 0xffffffffull), code = (int)(entry >> 32);
          reach_add<S, 0, true, false>(a, k, code, a.p_raddrag[k], 1.0, sr);
          reach_add<S, 1, true, false>(a, k, code, a.p_azidrag[k], 1.0, st);
        }
        for (unsigned long long m = crowded; m; m &= m - 1ull) {
          const int L = __ffsll((long long)m) - 1, b0 = __shfl(e0, L, 64), bn = __shfl(n, L, 64);
          ReachSum<S, 0> xr;
          ReachSum<S, 1> xt;
          reach_clear(xr);
          reach_clear(xt);
          for (int e = lane; e < bn; e += 64) {
            const unsigned long long entry = a.p_entry[b0 + e];
            const int k = (int)(unsigned)(entry & 0xffffffffull), code = (int)(entry >> 32);
            reach_add<S, 0, true, false>(a, k, code, a.p_raddrag[k], 1.0, xr);
            reach_add<S, 1, true, false>(a, k, code, a.p_azidrag[k], 1.0, xt);
          }
          reach_gather(xr, lane == L, sr);
          reach_gather(xt, lane == L, st);
        }
        reach_spread(sr, fr0, fr1, fr2);
        reach_spread(st, ft0, ft1, ft2);
      }
      if (want_dens || want_e) {
        ReachSum<S, 2> sd, se;
        reach_clear(sd);
        reach_clear(se);
        for (int e = e0; e < e0 + few; e++) {
          const unsigned long long entry = a.p_entry[e];
          const int k = (int)(unsigned)(entry & 0xffffffffull), code = (int)(entry >> 32);
          reach_add<S, 2, false, false>(a, k, code, 1.0, 1.0, sd);
          if (want_e) reach_add<S, 2, true, true>(a, k, code, a.p_dv2[k], a.p_ts[k], se);
        }
        for (unsigned long long m = crowded; m; m &= m - 1ull) {
          const int L = __ffsll((long long)m) - 1, b0 = __shfl(e0, L, 64), bn = __shfl(n, L, 64);
          ReachSum<S, 2> xd, xe;
          reach_clear(xd);
          reach_clear(xe);
          for (int e = lane; e < bn; e += 64) {
            const unsigned long long entry = a.p_entry[b0 + e];
            const int k = (int)(unsigned)(entry & 0xffffffffull), code = (int)(entry >> 32);
            reach_add<S, 2, false, false>(a, k, code, 1.0, 1.0, xd);
            if (want_e) reach_add<S, 2, true, true>(a, k, code, a.p_dv2[k], a.p_ts[k], xe);
          }
          reach_gather(xd, lane == L, sd);
          if (want_e) reach_gather(xe, lane == L, se);
        }
        reach_spread(sd, dd0, dd1, dd2);
        if (want_e) reach_spread(se, fe0, fe1, fe2);
      }
    }
    // ring i - 1 is complete
    if (i > i0 && own) {
      const long l = (long)(i - 1) * ns + j;
      const double surf = a.Surf[i - 1];
      if (want_fb) {
        const double mg = ldd<T>(a.rho, l) * surf;
        ((T *)a.radfbacc)[l] = (T)(fr0 != 0.0 ? -(fr0 * mp / mg) : 0.0);
        ((T *)a.azifbacc)[l] = (T)(ft0 != 0.0 ? -(ft0 * mp / mg) : 0.0);
      }
      if (want_e) ((T *)a.fbedot)[l] = (T)(mp / surf * fe0);
      if (want_dens) ((T *)a.dustdens)[l] = (T)(dd0 * mp / surf);
    }
    fr0 = fr1, fr1 = fr2, ft0 = ft1, ft1 = ft2;
    dd0 = dd1, dd1 = dd2, fe0 = fe1, fe1 = fe2;
  }
}

// The gas vtheta after the start-up interpolation in a rotating frame:
// vt + Rmed OmegaFrame and back (src/Dsys.c:316,1082), one cell per thread
template <typename T> __global__ void __launch_bounds__(256) k_dust_frame_trip(KArgs a) {
  const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= a.ns) return;
  const long l = (long)i * a.ns + j;
  const double rw = a.Rmed[i] * a.ctrl->omega_frame;
  ((T *)a.vt)[l] = (T)((ldd<T>(a.vt, l) + rw) - rw);
}

}  // namespace

template <typename T, int S> static void dust_launch_s(int id, const KArgs &a, hipStream_t s, int force,
                                                       double timestep) {
  const int np = a.d_np, pb = (np + 255) / 256;
  // the deposit's strips: four rings pass over fewer rings twice than two do,
  // while they still give four wavefronts a SIMD; longer ones leave the chip to
  // the strips of the crowded rings (1024 x 3072, 10^6 grains gathered at the
  // gap's edges: 133 us with strips of 2, 131 of 4, 150 of 8, 203 of 16)
  const int segs = (a.ns + DEP_OWN - 1) / DEP_OWN;
  const int strip = (long)a.nr * segs / 4 < 16L * a.num_cu ? 2 : 4;
  switch (id) {
    case KID_DUST_MOVE:
      if (np > 0) hipLaunchKernelGGL((k_dust_move<T, S>), dim3(pb), dim3(256), 0, s, a, force, timestep);
      break;
    case KID_DUST_SCAN:
      // the bucket counts are zeroed by the CFL kernel of the sub-step (and
      // by the start-up before its move); the ring scan turns them into starts
      hipLaunchKernelGGL(k_dust_ring_scan, dim3(a.nr), dim3(a.ns < 1024 ? ((a.ns + 63) / 64) * 64 : 1024), 0, s,
                         a, force);
      hipLaunchKernelGGL(k_dust_ring_offsets, dim3(1), dim3(1024), 0, s, a, force);
      break;
    case KID_DUST_SCATTER:
      if (np > 0) hipLaunchKernelGGL(k_dust_scatter, dim3(pb), dim3(256), 0, s, a, force);
      break;
    case KID_DUST_RANK:
      if (np > 0) hipLaunchKernelGGL(k_dust_rank, dim3(pb), dim3(256), 0, s, a, force);
      break;
    case KID_DUST_DEPOSIT:
      if (a.energy)
        hipLaunchKernelGGL((k_dust_deposit<T, S, true>), dim3(segs, (a.nr + strip - 1) / strip), dim3(64), 0, s, a,
                           force, strip);
      else
        hipLaunchKernelGGL((k_dust_deposit<T, S, false>), dim3(segs, (a.nr + strip - 1) / strip), dim3(64), 0, s, a,
                           force, strip);
      break;
  }
}

template <typename T> static void dust_launch(int id, const KArgs &a, hipStream_t s, int force, double timestep) {
  switch (a.d_interp) {
    case DFARGO_INTERP_NGP: dust_launch_s<T, DFARGO_INTERP_NGP>(id, a, s, force, timestep); break;
    case DFARGO_INTERP_CIC: dust_launch_s<T, DFARGO_INTERP_CIC>(id, a, s, force, timestep); break;
    default: dust_launch_s<T, DFARGO_INTERP_TSC>(id, a, s, force, timestep); break;
  }
}

template <typename T> void launch_dust_kernel(int id, const KArgs &a, hipStream_t s) { dust_launch<T>(id, a, s, 0, 0.0); }

template <typename T> void launch_dust_startup(const KArgs &a, double timestep, double omega_frame, hipStream_t s) {
  hipLaunchKernelGGL(k_dust_zero, dim3(1024), dim3(256), 0, s, a);
  for (int id : {KID_DUST_MOVE, KID_DUST_SCAN, KID_DUST_SCATTER, KID_DUST_RANK, KID_DUST_DEPOSIT})
    dust_launch<T>(id, a, s, 1, timestep);
  if (omega_frame != 0.0 && a.d_np > 0) {
    const int bx = a.ns < 256 ? a.ns : 256;
    hipLaunchKernelGGL(k_dust_frame_trip<T>, dim3((a.ns + bx - 1) / bx, a.nr), dim3(bx), 0, s, a);
  }
}

template void launch_dust_kernel<double>(int, const KArgs &, hipStream_t);
template void launch_dust_kernel<float>(int, const KArgs &, hipStream_t);
template void launch_dust_startup<double>(const KArgs &, double, double, hipStream_t);
template void launch_dust_startup<float>(const KArgs &, double, double, hipStream_t);
