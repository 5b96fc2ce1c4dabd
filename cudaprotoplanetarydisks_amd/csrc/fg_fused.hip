// Fused substep path: the arithmetic of the per-routine kernels in
// fg_steps.hip (same expressions, same rounding), regrouped so that one
// substep makes five passes over HBM instead of ~100:
//
//   k_src   a wave per column strip and ring band, marching over the rings
//           with its windows in registers: CorrectVtheta, evanescent
//           damping, pressure, potential, Substep1, viscous stress, viscous
//           update, artificial viscosity, velocity update, second damping
//           pass
//           state A -> state B
//   k_trad  column-marching radial van Leer sweep of the five transported
//           quantities (each slope and flux evaluated once), plus one wave
//           per ring for VMed (sequential ring sum)
//           state B -> R (Sigma, RadMomP/M, ThetaMomP/M)
//   k_tazw  one wave per contiguous chunk of a ring: FARGO residual and
//           integer shift, both azimuthal sweeps, the shift, vtheta
//           recovery; R -> X (Sigma, vtheta, RadMomP, RadMomM)
//   k_fin   one ring per workgroup: vrad recovery, third damping pass,
//           temperature, and the next substep's CFL ring minimum
//           X -> state A
//   force   DeviceReduce-order disk force on the star (partials as in
//           fg_reduce.hip) and the CFL count in one final kernel
//           (k_results)
//
// Adiabatic decks add Substep3 (k_src3) between k_src and k_trad and carry
// the energy through the sweeps and k_fin; self-gravitating decks run the
// SG field (fg_sg_fused) first and add its kick in k_src.
//
// Kernel times in the comments are means per launch of a rocprofv3 kernel trace,
// before and after on one card; "by events": HIP events around the launch
// (fg_profile), which add 1 to 5 us.
//
// Supported decks: evanescent boundaries, per-substep CFL; isothermal or
// adiabatic, with or without self-gravity (FP32 bulk mode: isothermal
// without self-gravity).  Everything else uses the per-routine path.
#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "fg_cell.h"
#include "fg_internal.h"
#include "fg_reduce.h"




struct fused_bufs {
  double *Bd, *Bvr, *Bvt;                // after k_src
  double *Rd, *Rrmp, *Rrmm, *Rtmp, *Rtmm;  // after k_trad
  double *Xd, *Xvt, *Xrmp, *Xrmm;        // after k_taz
  double *P;                             // pressure (temperature output only)
  // adiabatic decks: EnergyInt after k_src, energy after k_trad and k_taz;
  // self-gravity: the kick of VradInt / VthetaInt (NULL when not allocated)
  double *Beint, *Re, *Xe, *kick_r, *kick_t;
  // FP32 bulk mode: B, R and X stored in FP32 in the same arrays
  float *fBd() const { return (float *)Bd; }
  float *fBvr() const { return (float *)Bvr; }
  float *fBvt() const { return (float *)Bvt; }
  float *fR(int q) const { return (float *)(q == 0 ? Rrmp : q == 1 ? Rrmm : q == 2 ? Rtmp : q == 3 ? Rtmm : Rd); }
  float *fXd() const { return (float *)Xd; }
  float *fXvt() const { return (float *)Xvt; }
  float *fXrmp() const { return (float *)Xrmp; }
  float *fXrmm() const { return (float *)Xrmm; }
};

struct src_args {
  const double *dens, *vr, *vt;
  double *odens, *ovr, *ovt, *opress;
  const double *nu;   // viscosity of this substep (viscous stress, second damping pass)
  const double *nu1;  // viscosity as the first damping pass sees it (an adiabatic
                      // run refreshes it after that pass on a DT's first substep)
  // adiabatic: energy in, EnergyInt out (SourceEuler.cu:281, Kernels.cu:474-477)
  const double *energy;
  double *oeint;
  double gamma;
  // self-gravity: the kick of Update_sgvelocityKernel per cell (Kernels.cu:915-932,
  // formed by k_sg_acc_fused), and the ring means of the radial SG acceleration
  // that the first (sg1: previous evaluation) and second (sg2: this substep's)
  // damping passes take for vtheta0
  const double *kick_r, *kick_t;
  const double *sg1, *sg2;
  fg_dev_tables t;
  fg_planets_arg P;
  double dt, omega_frame, domega;
  int nr, ns, indirect, evanescent;
  int plain;  // planet_potential_plain applies
  int nstrips, width, band;  // strips of `width` columns, bands of `band` rings
};

// a planet's contribution to the potential at (x, y), and then, behind the
// first planet's, the star's (FillForcesArraysKernel, Kernels.cu:1234-1252)
__device__ __forceinline__ double planet_potential(double x, double y, double xp, double yp, double m, double smooth,
                                                   double invd3, int indirect) {
  const double distance = (x - xp) * (x - xp) + (y - yp) * (y - yp);
  const double distancesmooth = sqrt(distance + smooth);
  double pv = -1.0 * m / distancesmooth;
  if (indirect) pv += 1.0 * m * invd3 * (x * xp + y * yp);
  return pv;
}
// The same where the host found every operand far from the ends of the
// exponent range (plain_potential): neither the square root nor the quotient
// needs its operands scaled, and the root's own iteration (Goldschmidt's, with
// Markstein's corrections) leaves half the reciprocal that the quotient takes,
// after one Newton step.  Both results are the correctly rounded ones: 16
// instructions instead of 29.
__device__ __forceinline__ double planet_potential_plain(double x, double y, double xp, double yp, double m,
                                                         double smooth, double invd3, int indirect) {
  const double d = (x - xp) * (x - xp) + (y - yp) * (y - yp) + smooth;
  const double y0 = __builtin_amdgcn_rsq(d);
  double r = d * y0, h = 0.5 * y0;  // towards sqrt(d) and 1 / (2 sqrt(d))
  const double t = fma(-h, r, 0.5);
  r = fma(r, t, r);
  h = fma(h, t, h);
  r = fma(fma(-r, r, d), h, r);
  r = fma(fma(-r, r, d), h, r);
  double i = h + h;
  i = fma(i, fma(-r, i, 1.0), i);
  double pv = recip64(r, i).div(-1.0 * m);
  if (indirect) pv += 1.0 * m * invd3 * (x * xp + y * yp);
  return pv;
}
// InvDistance = 1.0 / Rm (the ring table holds the same correctly rounded
// quotient), (ix, iy) the indirect term of the star
__device__ __forceinline__ double star_potential(double x, double y, double InvDistance, double ix, double iy) {
  double pv = -1.0 * 1.0 * InvDistance;
  pv -= ix * x + iy * y;
  return pv;
}

// evanescent damping constants of ring i for a step (Kernels.cu:978-1004);
// with self-gravity vtheta0 takes the ring mean of the radial SG
// acceleration (sgacc, NULL without self-gravity)
__device__ __forceinline__ void ev_consts(const fg_dev_tables &t, const double *nu, int i, double step,
                                          double omega_frame, double &lambda, double &vrad0, double &vtheta0,
                                          const double *sgacc = nullptr) {
  const double Rm = t.Rmed[i];
  lambda = t.ev_coef[i] * step / t.ev_period[i];
  vtheta0 = sgacc ? sqrt(t.ev_vtheta_arg[i] - Rm * sgacc[i]) : sqrt(t.ev_vtheta_arg[i]);
  vtheta0 -= Rm * omega_frame;
  vrad0 = -3.0 * nu[i] / Rm * t.vrad0_slope;
}

// x of lane l-1 (lane 0 reads 0): DPP wave_shr:1 on each dword
__device__ __forceinline__ double lane_prev(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x138, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// x of lane l+1 (lane 63 reads 0): DPP wave_shl:1 on each dword
__device__ __forceinline__ double lane_next(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// p as the global pointer it is: read from a struct in memory it would be a
// generic one, and its accesses flat ones, which wait for LDS and memory alike
template <class T>
__device__ __forceinline__ T *global(T *p) {
  return (T *)(__attribute__((address_space(1))) T *)(unsigned long)p;
}

// Workgroups are dispatched round-robin over the 8 XCDs.  The block of a list
// of n that this workgroup of a grid of 8 ceil(n / 8) takes, each XCD a
// contiguous run, so that neighbouring blocks, which read each other's halos,
// share an L2; -1: none.
#define FG_NXCD 8
__device__ __forceinline__ int xcd_block(int n) {
  const int b = (int)(blockIdx.x % FG_NXCD) * ((int)gridDim.x / FG_NXCD) + (int)(blockIdx.x / FG_NXCD);
  return b < n ? b : -1;
}
static inline int xcd_grid(int n) { return (n + FG_NXCD - 1) / FG_NXCD * FG_NXCD; }

// k_src's strips: one wave marches over the rings of a band, a lane per
// column.  SRC_HL / SRC_HR columns at the ends of the wave are halo (a
// result depends on the inputs up to three columns to the left and two to
// the right), and so are the SRC_HT rings above and SRC_HB below the band.
#define SRC_HL 3
#define SRC_HR 2
#define SRC_HT 3
#define SRC_HB 2
#define SRC_W (64 - SRC_HL - SRC_HR)  // most columns a strip outputs
#define SRC_ROWS 32
#define SRC_MAX_BAND (SRC_ROWS - SRC_HT - SRC_HB)
// damping constants of a ring: 1 + lambda and its reciprocal refinement,
// lambda times what Sigma, the energy, vrad and vtheta relax to (the last
// two in the first pass, then in the second)
enum { EV_D, EV_R, EV_S, EV_E, EV_VR1, EV_VT1, EV_VR2, EV_VT2, EV_N };

// (q + lambda q0) / (1 + lambda), Kernels.cu:1006-1012
__device__ __forceinline__ double ev_damp(double q, const double *ev, int which) {
  return recip64(ev[EV_D], ev[EV_R]).div(q + ev[which]);
}

// element at byte offset `off` of a row: the scalar row address plus a 32-bit
// lane offset is the memory instructions' own form, no vector arithmetic
template <class T>
__device__ __forceinline__ T &at(T *row, unsigned off) {
  return *(T *)((char *)row + off);
}
template <class T>
__device__ __forceinline__ T at(const T *row, unsigned off) {
  return *(const T *)((const char *)row + off);
}

// MODE bit 1: adiabatic (energy damped, P = (gamma - 1) e, EnergyInt out);
// bit 2: self-gravity kick after Substep1
//
// One step of the march takes in ring m and completes ring m - 2; what the
// stages need of earlier rings stays in registers (slot ring mod 3, so a
// step is instantiated per m mod 3 and nothing is shifted), the neighbours
// in azimuth come from the neighbouring lanes by DPP.  So there is no LDS
// tile, no barrier, no index
// arithmetic per cell, and a band of H rings by 59 columns evaluates
// (H + 5) / H x 64 / 59 cells per cell, where the 16 x 64 LDS tile with its
// halo of four evaluated 1.55.
// Bound: HBM on large grids (2048 x 4096: 442 MB by the counters, of which
// 403 are the fields read and written once, in 119 us, was 222 us; 1024 x 3072:
// 61 us, was 91, and 50 us by events with the band that suits it, src_band), the
// waves' own issue on small ones (a dependent FP64 operation every nine cycles;
// 512 x 1536: 23 us, was 30; 128 x 384: 9 us, was 13).  Three waves per SIMD
// (168 VGPRs) and two rings in flight without energy and self-gravity; with
// them two waves and one ring (177 to 191 VGPRs), since the third wave would
// spill (512 x 1536 with both 26 us, was 35; by events 29, and 37 with three).
template <int MODE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(MODE ? 2 : 3))) void k_src(src_args a) {
  constexpr int AHEAD = MODE ? 1 : 2;  // rings whose loads are in flight
  constexpr bool ADI = MODE & 1, SGK = MODE & 2;
  __shared__ double tab[SRC_ROWS][RG_N], evc[SRC_ROWS][EV_N];
  const int nr = a.nr, ns = a.ns, lane = threadIdx.x;
  const int block = xcd_block(a.nstrips * ((nr + a.band) / a.band));
  if (block < 0) return;
  const int strip = block % a.nstrips, i0 = block / a.nstrips * a.band;
  const int i1 = min(i0 + a.band, nr + 1);  // rings i0 .. i1 - 1 (the ghost ring with the last band)
  const fg_dev_tables &t = a.t;
  const double dt = a.dt, OF = a.omega_frame;
  const int g = strip * a.width - SRC_HL + lane;  // this lane's column, unwrapped
  const int j = (g % ns + ns) % ns;
  unsigned jb = 8u * j;  // in bytes
  const bool mine = lane >= SRC_HL && lane < SRC_HL + a.width && g < ns;
  const double cosp = t.cos_pot[j], sinp = t.sin_pot[j];
  // ring m's inputs are loaded AHEAD steps ahead (rings clamped into the
  // grid), slot ring mod 3 as below
  double n_s[3], n_vr[3], n_vt[3], n_e[3], n_kr[3], n_kt[3];
  auto fetch = [&](int m, auto phase) __attribute__((always_inline)) {
    constexpr int X = decltype(phase)::value % 3;
    const long l = (long)min(max(m, 0), nr) * ns;
    n_s[X] = at(a.dens + l, jb);
    n_vr[X] = at(a.vr + l, jb);
    n_vt[X] = at(a.vt + l, jb);
    if constexpr (ADI) n_e[X] = at(a.energy + l, jb);
    if constexpr (SGK) {
      n_kr[X] = at(a.kick_r + l, jb);
      n_kt[X] = at(a.kick_t + l, jb);
    }
  };
#define LVL(n) std::integral_constant<int, n>()
  fetch(i0 - SRC_HT, LVL(0));
  if (AHEAD > 1) fetch(i0 - SRC_HT + 1, LVL(1));
  // the tables of the rings the band reads and their damping constants
  // (Kernels.cu:978-1004), a ring per lane, into LDS, from where each step
  // takes them with a uniform address: held in scalar registers they would
  // need three times as many as there are, read through the scalar cache
  // every use is a round trip (1.26 us a step for a lone wave)
  bool damped = false;
  if (lane < i1 - i0 + SRC_HT + SRC_HB) {
    const int i = i0 - SRC_HT + lane, ic = min(max(i, 0), nr - 1);
    double r[RG_NU];
#pragma unroll
    for (int x = 0; x < RG_NU; x++) r[x] = t.rings[(long)ic * RG_NU + x];
    const double v = a.nu[ic];
    damped = a.evanescent && i == ic && t.ev_zone[ic];
#pragma unroll
    for (int x = 0; x < RG_NU; x++) tab[lane][x] = r[x];
    tab[lane][RG_NU] = v;
    if (damped) {
      double lambda, vr0, vt0, *ev = evc[lane];
      ev_consts(t, a.nu1, i, dt, OF, lambda, vr0, vt0, a.sg1);
      const recip64 d(1.0 + lambda);
      ev[EV_D] = d.d;
      ev[EV_R] = d.r;
      ev[EV_S] = lambda * t.SigmaMed[i];
      ev[EV_E] = ADI ? lambda * t.EnergyMed[i] : 0.0;
      ev[EV_VR1] = lambda * vr0;
      ev[EV_VT1] = lambda * vt0;
      ev_consts(t, a.nu, i, dt, OF, lambda, vr0, vt0, a.sg2);
      ev[EV_VR2] = lambda * vr0;
      ev[EV_VT2] = lambda * vt0;
    }
  }
  const unsigned zones = (unsigned)__ballot(damped);  // bit r: ring i0 - SRC_HT + r is damped
  __syncthreads();
  // the first planet and the indirect term in registers, further planets where
  // the launch put them (indexed by a loop, a by-value copy would live in
  // scratch)
  const auto &more = ((__attribute__((address_space(4))) const src_args *)__builtin_amdgcn_kernarg_segment_ptr())->P;
  double px = a.P.x[0], py = a.P.y[0], pm = a.P.m[0], ps = a.P.smooth[0], pi3 = a.P.invd3[0], ix = a.P.ix, iy = a.P.iy;
  asm volatile("" : "+s"(px), "+s"(py), "+s"(pm), "+s"(ps), "+s"(pi3), "+s"(ix), "+s"(iy));
  const double invdphi = t.invdphi, onethird = 1.0 / 3.0;
  // windows, ring x in slot x mod 3: Sigma, its left neighbour, pressure,
  // potential, vtheta and its right neighbour; VradInt / VthetaInt after
  // Substep1 and VradInt after the viscous update; stresses; radial
  // artificial pressure; the halved sums Sigma_i + Sigma_i-1 and
  // Sigma_j + Sigma_j-1 with their reciprocal refinements, which divide in
  // S1, S3 and S5 (x * 2 / d is x / (d / 2), both scalings exact)
  double S[3] = {}, Sl[3] = {}, P[3] = {}, F[3] = {}, T[3] = {}, Tn[3] = {}, EN[3] = {};
  double A1[3] = {}, B1[3] = {}, A3[3] = {}, RR[3] = {}, PP[3] = {}, RP[3] = {}, QR[3] = {};
  double hr[3] = {}, hrr[3] = {}, ha[3] = {}, har[3] = {};
  // LEVEL: how many of the stages ring m's step evaluates (the first steps
  // of a band only fill the windows); IN: rings m - 3 .. m + 1 lie strictly
  // inside the disk, which drops the edge cases
  auto step = [&](int m, auto level, auto phase, auto inner) __attribute__((always_inline)) {
    constexpr int LV = decltype(level)::value, C = decltype(phase)::value, M1 = (C + 2) % 3, M2 = (C + 1) % 3;
    constexpr bool IN = decltype(inner)::value;
    double s = n_s[C], vr = n_vr[C], vt = n_vt[C], e = ADI ? n_e[C] : 0.0;
    const double kr = SGK ? n_kr[C] : 0.0, kt = SGK ? n_kt[C] : 0.0;
    fetch(m + AHEAD, LVL(C + AHEAD));
    // (keeps the lane offset apart from the row address: added up before the
    // loop they would be a vector pointer per field)
    asm volatile("" : "+v"(jb));
    const int row = m - i0 + SRC_HT;  // rings m, k, o in the tables
    const double *Rm = tab[row], *Rk = tab[max(row - 1, 0)], *Ro = tab[max(row - 2, 0)];
    const int k = m - 1, o = m - 2;
    // ---- S0: CorrectVtheta, damping #1, pressure, potential of ring m ----
    double p = 0.0, phi = 0.0;
    if (IN || (m >= 0 && m < nr)) {
      vt = vt - a.domega * Rm[RG_MED];
      if (zones >> row & 1) {
        const double *ev = evc[row];
        vr = ev_damp(vr, ev, EV_VR1);
        vt = ev_damp(vt, ev, EV_VT1);
        s = ev_damp(s, ev, EV_S);
        if (ADI) e = ev_damp(e, ev, EV_E);
      }
      if (ADI) {
        p = (a.gamma - 1.0) * e;  // Kernels.cu:196
      } else {
        const double cs = Rm[RG_CS];
        p = s * cs * cs;
      }
      const double x = Rm[RG_MED] * cosp, y = Rm[RG_MED] * sinp;
      if (a.P.nb > 0) {
        phi = 0.0 + (a.plain ? planet_potential_plain(x, y, px, py, pm, ps, pi3, a.indirect)
                             : planet_potential(x, y, px, py, pm, ps, pi3, a.indirect));
        phi += star_potential(x, y, Rm[RG_IMED], ix, iy);
      }
      for (int q = 1; q < a.P.nb; q++)
        phi += planet_potential(x, y, more.x[q], more.y[q], more.m[q], more.smooth[q], more.invd3[q], a.indirect);
      if (a.opress && mine && m >= i0 && m < i1) at(a.opress + (long)m * ns, jb) = p;  // for the temperature output
    } else if (m != nr) {
      s = vr = vt = 0.0;
    }
    S[C] = s;
    P[C] = p;
    F[C] = phi;
    T[C] = vt;
    Tn[C] = lane_next(vt);
    Sl[C] = lane_prev(s);
    if (ADI) EN[C] = e;
    // ---- S1: Substep1 (Kernels.cu:13-53) of ring m ----
    if constexpr (LV >= 1) {
      double vri = 0.0, vti = 0.0;
      hr[C] = hrr[C] = ha[C] = har[C] = 0.0;
      if (IN || (m >= 0 && m < nr)) {
        if (IN || m > 0) {
          const recip64 hd(0.5 * (s + S[M1]));
          hr[C] = hd.d;
          hrr[C] = hd.r;
          const double idm = Rm[RG_IDMED];
          const double gradp = hd.div(p - P[M1]) * idm;
          const double gradphi = (phi - F[M1]) * idm;
          double vt2 = T[C] + Tn[C] + T[M1] + Tn[M1];
          vt2 = vt2 / 4.0 + OF * Rm[RG_INF];
          vt2 = vt2 * vt2;
          const double vr_src = -gradp - gradphi;
          const double vradint2 = vr_src + vt2 * Rm[RG_IINF];
          vri = vr + dt * vradint2;
        }
        const double invdxtheta = Rm[RG_IDXT];
        const recip64 hd(0.5 * (s + Sl[C]));
        ha[C] = hd.d;
        har[C] = hd.r;
        const double gradp = hd.div(p - lane_prev(p)) * invdxtheta;
        const double gradphi = (phi - lane_prev(phi)) * invdxtheta;
        double v = vt - dt * (gradp + gradphi);
        v += dt * Rm[RG_SUPP];
        vti = v;
        if constexpr (SGK) {  // self-gravity kick (0 on ring 0 of VradInt)
          vri = vri + kr;
          vti = vti + kt;
        }
      }
      A1[C] = vri;  // VradInt (0 on rings 0 and NRAD, as never written)
      B1[C] = vti;  // VthetaInt
    }
    // ---- S2: viscous stress (Kernels.cu:733-771) of ring k ----
    if constexpr (LV >= 2) {
      if (IN || (k >= 0 && k < nr)) {
        const double invRm = Rk[RG_IMED], idsup = Rk[RG_IDSUP], Rinf = Rk[RG_INF], v = Rk[RG_NU];
        const double bn = lane_next(B1[M1]), b = B1[M1], vrl = A1[M1], vrn = A1[C];
        const double drr = (vrn - vrl) * idsup;
        const double dpp = (bn - b) * invdphi * invRm + 0.5 * (vrn + vrl) * invRm;
        double dv = (vrn * Rk[RG_SUP] - vrl * Rinf) * idsup * invRm;
        dv += (bn - b) * invdphi * invRm;
        RR[M1] = 2.0 * S[M1] * v * (drr - onethird * dv);
        PP[M1] = 2.0 * S[M1] * v * (dpp - onethird * dv);
        if (LV >= 3 && (IN || k > 0)) {
          const double drp = 0.5 * (Rinf * (b * invRm - B1[M2] * Ro[RG_IMED]) * Rk[RG_IDMED] +
                                    (vrl - lane_prev(vrl)) * invdphi * Rk[RG_IINF]);
          RP[M1] = 2.0 * 0.25 * (S[M1] + S[M2] + Sl[M1] + Sl[M2]) * v * drp;
        }
      }
    }
    // ---- S3: viscous velocity update (Kernels.cu:118-150): VradInt of ring k ----
    if constexpr (LV >= 3) {
      A3[M1] = A1[M1];
      if (IN || (k >= 1 && k < nr))
        A3[M1] += recip64(hr[M1], hrr[M1])
                      .div(dt * Rk[RG_IINF] *
                           ((Rk[RG_MED] * RR[M1] - Ro[RG_MED] * RR[M2]) * Rk[RG_IDMED] +
                            (lane_next(RP[M1]) - RP[M1]) * invdphi - 0.5 * (PP[M1] + PP[M2])));
    }
    // ---- S4: radial artificial pressure (Kernels.cu:409-434) of ring o ----
    const double dvr = A3[M1] - A3[M2];
    if constexpr (LV >= 4) QR[M2] = (IN || (o >= 0 && o < nr)) ? art_visc_q(S[M2], dvr) : 0.0;
    // ---- ring o: the rest of S3 and S4, S5 ("kernel", Kernels.cu:438-479), damping #2, store ----
    if constexpr (LV >= 5) {
      const long l = (long)o * ns;
      if (!IN && o == nr) {  // ghost ring: VradNew/VthetaNew are never written (0)
        if (mine) {
          at(a.odens + l, jb) = S[M2];
          at(a.ovr + l, jb) = 0.0;
          at(a.ovt + l, jb) = 0.0;
        }
        return;
      }
      const recip64 dr_(hr[M2], hrr[M2]), da_(ha[M2], har[M2]);
      double b = B1[M2];
      if (IN || (o >= 1 && o < nr - 1))
        b += da_.div(dt * Ro[RG_IMED] *
                     ((Ro[RG_SUP] * RP[M1] - Ro[RG_INF] * RP[M2]) * Ro[RG_IDSUP] +
                      (PP[M2] - lane_prev(PP[M2])) * invdphi + 0.5 * (RP[M2] + RP[M1])));
      const double dvt = lane_next(b) - b;
      const double qt = art_visc_q(S[M2], dvt);
      double vrnew = 0.0;
      if (IN || o > 0) {
        const double densint = QR[M2] - QR[C];  // (slot C: ring o - 1, not yet overwritten)
        vrnew = A3[M2] - dr_.div(dt) * densint * Ro[RG_IDMED];
      }
      const double invdxtheta = Ro[RG_IDXT];
      const double tempint = qt - lane_prev(qt);
      double vtnew = b - da_.div(dt) * tempint * invdxtheta;
      double s2 = S[M2];
      double eint = 0.0;
      if constexpr (ADI)
        // EnergyInt ("kernel", Kernels.cu:474-477) from the energy after the
        // first damping pass; the second pass damps Energy, which Substep3
        // then overwrites, so it is not formed
        eint = EN[M2] - dt * QR[M2] * dvr * Ro[RG_IDSUP] - dt * qt * dvt * invdxtheta;
      if (zones >> (row - 2) & 1) {
        const double *ev = evc[row - 2];
        vrnew = ev_damp(vrnew, ev, EV_VR2);
        vtnew = ev_damp(vtnew, ev, EV_VT2);
        s2 = ev_damp(s2, ev, EV_S);
      }
      if (mine) {
        at(a.odens + l, jb) = s2;
        at(a.ovr + l, jb) = vrnew;
        at(a.ovt + l, jb) = vtnew;
        if constexpr (ADI) at(a.oeint + l, jb) = eint;
      }
    }
  };
  auto march = [&](auto inner) __attribute__((always_inline)) {
    // rings i0 - 3 .. i0 + 1 fill the windows; with ring i0 + 2 in slot 2,
    // ring i0 - 3 + x is in slot x mod 3
    const int m0 = i0 - SRC_HT;
    step(m0, LVL(0), LVL(0), inner);
    step(m0 + 1, LVL(1), LVL(1), inner);
    step(m0 + 2, LVL(2), LVL(2), inner);
    step(m0 + 3, LVL(3), LVL(0), inner);
    step(m0 + 4, LVL(4), LVL(1), inner);
    int m = m0 + 5;
    for (; m + 2 <= i1 + 1; m += 3) {
      step(m, LVL(5), LVL(2), inner);
      step(m + 1, LVL(5), LVL(0), inner);
      step(m + 2, LVL(5), LVL(1), inner);
    }
    if (m <= i1 + 1) step(m, LVL(5), LVL(2), inner);
    if (m + 1 <= i1 + 1) step(m + 1, LVL(5), LVL(0), inner);
  };
#undef LVL
  if (i0 - SRC_HT >= 1 && i1 + SRC_HB <= nr)
    march(std::true_type());
  else
    march(std::false_type());
}

// ----------------------------------------------------------- k_src3 ----
// Substep3 of an adiabatic deck (SourceEuler.cu:287-291): the viscous
// terms of the velocities after the second damping pass (ViscousTermsKernel,
// Kernels.cu:733-771), Qplus (Substep3Kernel, Kernels.cu:56-77; ring 0 by
// the power-law extrapolation from rings 1 and 2, Kernels.cu:88-95) and
// the implicit energy update with optional relaxation cooling
// (Substep3Kernel2, Kernels.cu:97-113).  One thread per cell; the
// neighbours are read through the caches.
struct src3_args {
  const double *dens, *vr, *vt, *eint;
  double *energy;
  const double *nu;
  fg_dev_tables t;
  double dt, gamma, lr01, lr12;
  int nr, ns, cooling;
};

// divV of cell (i, j) and, for i >= 1, its Qplus
__device__ __forceinline__ void src3_cell(const src3_args &a, int i, int j, double &qplus, double &divv) {
  const fg_dev_tables &t = a.t;
  const int ns = a.ns;
  const long l = (long)i * ns + j;
  const long JP = (long)i * ns + (j + 1 == ns ? 0 : j + 1), JM = (long)i * ns + (j == 0 ? ns - 1 : j - 1);
  const double invdphi = t.invdphi;
  const double onethird = 1.0 / 3.0;
  const double vrl = a.vr[l], vrn = a.vr[l + ns], vtl = a.vt[l], vtp = a.vt[JP];
  const double drr = (vrn - vrl) * t.invdiffRsup[i];
  const double dpp = (vtp - vtl) * invdphi * t.invRmed[i] + 0.5 * (vrn + vrl) * t.invRmed[i];
  double dv = (vrn * t.Rsup[i] - vrl * t.Rinf[i]) * t.invdiffRsup[i] * t.invRmed[i];
  dv += (vtp - vtl) * invdphi * t.invRmed[i];
  divv = dv;
  qplus = 0.0;
  if (i == 0) return;
  const double d = a.dens[l], nu = a.nu[i];
  if (nu == 0.0) return;
  const double TRR = 2.0 * d * nu * (drr - onethird * dv);
  const double TPP = 2.0 * d * nu * (dpp - onethird * dv);
  const double drp = 0.5 * (t.Rinf[i] * (vtl * t.invRmed[i] - a.vt[l - ns] * t.invRmed[i - 1]) * t.invdiffRmed[i] +
                            (vrl - a.vr[JM]) * invdphi * t.invRinf[i]);
  const double TRP = 2.0 * 0.25 * (d + a.dens[l - ns] + a.dens[JM] + a.dens[JM - ns]) * nu * drp;
  double q = 0.5 / nu / d * (TRR * TRR + TRP * TRP + TPP * TPP);
  q += (2.0 / 9.0) * nu * d * dv * dv;
  qplus = q;
}

__global__ __launch_bounds__(256) void k_src3(src3_args a) {
  const int j = blockIdx.x * 64 + (threadIdx.x & 63);
  const int i = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= a.nr || j >= a.ns) return;
  const fg_dev_tables &t = a.t;
  const long l = (long)i * a.ns + j;
  double qplus, divv;
  src3_cell(a, i, j, qplus, divv);
  if (i == 0) {
    if (a.nu[a.nr - 1] != 0.0) {
      double q1, q2, unused;
      src3_cell(a, 1, j, q1, unused);
      src3_cell(a, 2, j, q2, unused);
      qplus = q1 * exp(log(q1 / q2) * a.lr01 / a.lr12);
    } else {
      qplus = 0.0;
    }
  }
  double num, den;
  if (!a.cooling) {
    num = a.dt * qplus + a.eint[l];
    den = 1.0 + (a.gamma - 1.0) * a.dt * divv;
  } else {
    const double d = a.dens[l];
    num = t.EnergyMed[i] * a.dt * d / t.SigmaMed[i] + t.CoolingTimeMed[i] * a.eint[l] +
          a.dt * t.CoolingTimeMed[i] * (qplus - t.QplusMed[i] * d / t.SigmaMed[i]);
    den = a.dt + t.CoolingTimeMed[i] + (a.gamma - 1.0) * a.dt * t.CoolingTimeMed[i] * divv;
  }
  a.energy[l] = num / den;
}

// ----------------------------------------------------------- k_trad ----
// Radial sweep (OneWindRad, TransportEuler.cu:60-79) marching over rings
// of a band; one thread owns one sector column.  For each ring m the
// momenta (LRMomentaKernel), Work = Q / (Sigma + 1e-20), the slope and
// the face value at face m-1 are formed once and kept in registers; the
// face flux F(k) = dt*dtheta*Rinf[k]*Q*(k)*Sigma*(k)*vrad(k) serves both
// neighbouring rings (Rsup[k-1] == Rinf[k]).
// FP32 bulk mode storage.  The fields passed between the fused kernels
// (after k_src, k_trad and k_taz) are stored in FP32 as offsets from FP64
// backgrounds that writer and reader form alike: Sigma from sbar (ring
// means of the state the substep starts from), vtheta from vref (the ring
// means of vtheta at that state, Vmoy), the angular momenta from the
// cell's own stored Sigma times (vref + R Omega) R (fp32_bg_angmom; the
// writer takes Sigma as rounded for the reader); vrad and the radial
// momenta are stored as they are.  The offsets are small against the
// fields (a few 1e-3 of vtheta, the non-axisymmetric part of Sigma), so
// their FP32 rounding stays far below the FP32 arithmetic's own error; the
// state between substeps stays FP64.
// Near the planets, where circumplanetary material stays for many orbits
// and the rounding of the stored Sigma would add up there, the rings
// [lob0, lob1) store Sigma as a float pair: the high part where every ring
// stores its float (index l < S of an array of S doubles) and the rounding
// residual at S + l, in the array's otherwise unused upper half; a reader
// adds the residual only on those rings.  (Pairs for the velocities and
// momenta as well change nothing measurable.)  The upper-half slots of the
// ghost ring NRAD are never written and stay zero: loads that must be
// issued on every iteration take them for rings outside the band.
__device__ __forceinline__ bool in_lob(int i, int b0, int b1) { return i >= b0 && i < b1; }
__device__ __forceinline__ double rec32(double bg, float hi, float lo) { return bg + ((double)hi + (double)lo); }
__device__ __forceinline__ double fp32_bg_angmom(double sbar, double vref, double R, double omega) {
  return sbar * (vref + R * omega) * R;
}

#define TRAD_TPB 64
#define NQ 5  // RadMomP, RadMomM, ThetaMomP, ThetaMomM, Sigma
#define NQ_MAX 6  // adiabatic: RadMomP, RadMomM, ThetaMomP, ThetaMomM, Energy, Sigma

struct trad_args {
  const double *dens, *vr, *vt;
  const double *energy;  // adiabatic decks (NQT = 6)
  double *out[NQ_MAX];
  // FP32 bulk mode: the same fields stored in FP32 (fp32_store_bg)
  const float *fdens, *fvr, *fvt;
  float *fout[NQ];
  const double *sbar, *vref;  // per-ring backgrounds of Sigma and vtheta
  double *vmed;  // ring means of vtheta for the azimuthal pass
  double *lost;  // ROUTINE: change of ring 0's Sigma per sector (open inner edge), else NULL
  fg_dev_tables t;
  double dt, omega_frame;
  int nr, ns, nstrips;
  int band;        // rings per column strip
  int lob0, lob1;  // FP32 storage: rings stored as float pairs
};

// ComputeAverageThetaVelocitiesKernel (Kernels.cu:1070-1081) for one ring
// by one wave: the lanes stage the ring through LDS 512 sectors at a time
// (the next 512 loaded into registers meanwhile) and lane 0 adds them in j
// order with its LDS reads issued ahead of the dependent adds.  One wave:
// the barrier only orders the LDS accesses, and lane 0 has finished a
// round's sum before the next round's stores in program order.  (The sum by the
// whole wave's lanes, as ring_seq_sum, was no faster here: 512 x 1536 28.8
// against 25.7 us by events for the kernel, 1024 x 3072 the same, 2048 x 4096 131 and
// 137.)
#define RMW_CH 8  // sectors per lane per round
__device__ void ring_mean_wave(const double *v, int ns, double *out) {
  __shared__ double buf[64 * RMW_CH];
  const int lane = threadIdx.x;
  const int nch = (ns + 64 * RMW_CH - 1) / (64 * RMW_CH);
  double nx[RMW_CH];
#pragma unroll
  for (int u = 0; u < RMW_CH; u++) nx[u] = (lane + 64 * u < ns) ? v[lane + 64 * u] : 0.0;
  double sum = 0.0;
  for (int c = 0; c < nch; c++) {
#pragma unroll
    for (int u = 0; u < RMW_CH; u++) buf[lane + 64 * u] = nx[u];
    const int e0 = (c + 1) * 64 * RMW_CH + lane;
#pragma unroll
    for (int u = 0; u < RMW_CH; u++) nx[u] = (e0 + 64 * u < ns) ? v[e0 + 64 * u] : 0.0;
    __syncthreads();
    if (lane == 0) sum = seq_sum_lds(buf, min(64 * RMW_CH, ns - c * 64 * RMW_CH), sum);
    __syncthreads();
  }
  if (lane == 0) *out = sum / (double)ns;
}

// Ring tables of the rings a column strip marches over, one ring per lane
// (lane r holds ring r0 + r, clamped into the nr + 1 entries), read back
// with v_readlane.  Reading the tables from memory inside the ring loop
// would make each iteration wait for that load and, as a wave's vector
// memory operations complete in order, for the next ring's field loads
// issued before it, leaving nothing in flight across the arithmetic.
struct ring_lanes {
  int r0;
  double Rmed, idm, Rinf, isurf;
  __device__ __forceinline__ void load(const fg_dev_tables &t, int base, int nr) {
    r0 = base;
    const int r = min(max(base + (int)threadIdx.x, 0), nr);
    Rmed = t.Rmed[r];
    idm = t.invdiffRmed[r];
    Rinf = t.Rinf[r];
    isurf = t.invSurf[r];
    // consume the loads here, so that no wait for them lands in the loop
    asm volatile("" ::"v"(Rmed), "v"(idm), "v"(Rinf), "v"(isurf));
  }
  // ring m - 2 .. m + 61 can be read: reload when ring m would leave that
  __device__ __forceinline__ int at(const fg_dev_tables &t, int m, int nr) {
    if (m - r0 >= 64) load(t, m - 2, nr);
    return m - r0;
  }
};

// The FP32 storage backgrounds of the rings a column strip marches over,
// one ring per lane like ring_lanes (same first ring r0, reloaded with it)
struct bg_lanes {
  int r0;
  double sb, vb;
  __device__ __forceinline__ void load(const double *sbar, const double *vref, int base, int nr) {
    r0 = base;
    const int r = min(max(base + (int)threadIdx.x, 0), nr);
    sb = sbar[r];
    vb = vref[r];
    asm volatile("" ::"v"(sb), "v"(vb));
  }
};

// FP32 mode's VMed (ComputeAverageThetaVelocitiesKernel, Kernels.cu:
// 1070-1081) of one ring by one wave: vtheta (background + stored offset)
// summed per lane over sectors lane, lane + 64, ... (eight loads in flight),
// then a shuffle tree.  The FP32 mode does not replay the reference's
// one-thread order; the sum is no less accurate.
__device__ void ring_mean_wave32(const float *v, double vb, int ns, double *out) {
  const int lane = threadIdx.x;
  double sum = 0.0;
  for (int j0 = lane; j0 < ns; j0 += 64 * 8) {
    float x[8];
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = (j0 + 64 * u < ns) ? v[j0 + 64 * u] : 0.0f;
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (j0 + 64 * u < ns) sum += vb + (double)x[u];
  }
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
  if (lane == 0) *out = sum / (double)ns;
}

// NQT transported quantities: 5, or 6 with the energy of an adiabatic deck
// (TransportEuler.cu:60-79 sweeps it between the momenta and Sigma).
// ROUTINE: the sweep of fg_transport (the mass lost through an open edge);
// OWN: tables whose rings' outer faces are not the next rings' inner faces, so
// that a ring's outer flux takes its own Rsup (Kernels.cu:1039)
template <int NQT, bool ROUTINE = false, bool OWN = false>
__global__ __launch_bounds__(TRAD_TPB) void k_trad(trad_args a) {
  constexpr bool EN = NQT == 6;
  const int nr = a.nr, ns = a.ns;
  // blocks [0, NRAD): one ring mean each, issued first so that these
  // latency-bound sums overlap the sweep blocks
  if ((int)blockIdx.x < nr) {
    ring_mean_wave(a.vt + (long)blockIdx.x * ns, ns, a.vmed + blockIdx.x);
    return;
  }
  const int bid = blockIdx.x - nr;
  // lanes past the last sector march on column ns - 1 (every lane holds
  // its ring table entry) and store the same values as the lane that owns
  // that column
  const int j = min((bid % a.nstrips) * TRAD_TPB + (int)threadIdx.x, ns - 1);
  const int jp = (j + 1) % ns;
  const int b0 = (bid / a.nstrips) * a.band;
  const int b1 = min(b0 + a.band, nr);
  const fg_dev_tables &t = a.t;
  const double dt = a.dt, OF = a.omega_frame;
  const double cflux = dt * t.dtheta;
  // windows over the last three rings: ring x (its Q, W, Sigma, vrad and
  // slope) and face x (its flux) live in slot x % 3, so a step writes its
  // new ring over the one three back and nothing is shifted; the step for
  // ring m is instantiated per m % 3 to keep the slots static
  double Q[NQT][3] = {}, W[NQT][3] = {}, dq[NQT][3] = {}, F[NQT][3] = {};
  double sg[3] = {}, dqs[3] = {}, vr[3] = {};
  const int m0 = max(b0 - 2, 0);
  ring_lanes rt;
  rt.load(t, m0 - 2, nr);
  // ring m's inputs are loaded one iteration ahead (ring min(m + 1, nr - 1):
  // the loads are unconditional, so that every iteration of a loop issues
  // the same memory operations and the waits for them can count past the
  // stores); vrad of ring m + 1 is carried over as the next ring's own
  double n_s, n_v0, n_v1, n_vtp, n_vt, n_e = 0.0;
  {
    const long l = (long)m0 * ns + j;
    n_s = a.dens[l];
    n_v0 = a.vr[l];
    n_v1 = a.vr[l + ns];
    n_vtp = a.vt[(long)m0 * ns + jp];
    n_vt = a.vt[l];
    if constexpr (EN) n_e = a.energy[l];
    asm volatile("" ::"v"(n_s), "v"(n_v0), "v"(n_v1), "v"(n_vtp), "v"(n_vt), "v"(n_e));
  }
  // inner: the caller guarantees 2 <= m < nr (ring m inside the disk, slope
  // and face of ring m - 1 interior), which drops the edge cases
  auto ring = [&](int m, auto store, auto phase, auto inner) {
    constexpr int C = decltype(phase)::value, B1 = (C + 2) % 3, B2 = (C + 1) % 3;  // rings m, m-1, m-2
    constexpr bool IN = decltype(inner)::value;
    const int r = rt.at(t, m, nr);
    const double c_s = n_s, c_v0 = n_v0, c_v1 = n_v1, c_vtp = n_vtp, c_vt = n_vt, c_e = n_e;
    {
      const long l = (long)min(m + 1, nr - 1) * ns;
      n_s = a.dens[l + j];
      n_v0 = c_v1;
      n_v1 = a.vr[l + ns + j];
      n_vtp = a.vt[l + jp];
      n_vt = a.vt[l + j];
      if constexpr (EN) n_e = a.energy[l + j];
    }
    // ring tables: Rmed[m], Rmed[m-1], Rmed[m-2] at lanes r, r-1, r-2
    const double Rm = lane_get(rt.Rmed, r);
    if (IN || m < nr) {
      const double s = c_s;
      const double v0 = c_v0, v1 = c_v1;
      Q[0][C] = s * v1;
      Q[1][C] = s * v0;
      Q[2][C] = s * (c_vtp + Rm * OF) * Rm;
      Q[3][C] = s * (c_vt + Rm * OF) * Rm;
      if constexpr (EN) Q[4][C] = c_e;
      Q[NQT - 1][C] = s;
      sg[C] = s;
      vr[C] = v0;
      const recip64 rs(s + 1e-20);  // Work = Q / (Sigma + 1e-20), one denominator
      for (int q = 0; q < NQT; q++) W[q][C] = rs.div(Q[q][C]);
    } else {
      for (int q = 0; q < NQT; q++) Q[q][C] = W[q][C] = 0.0;
      sg[C] = 0.0;
      vr[C] = 0.0;  // vrad of the ghost ring
    }
    // slope of ring k = m-1 (zero on rings 0 and NRAD-1)
    const int k = m - 1;
    if (!decltype(store)::value && k < 0) return;  // storing steps have k >= 1
    const bool flat = !IN && (k == 0 || k >= nr - 1);
    const double idm0 = lane_get(rt.idm, r - 1), idm1 = lane_get(rt.idm, r);
    for (int q = 0; q < NQT; q++) dq[q][B1] = flat ? 0.0 : vl_rad_slope(W[q][B2], W[q][B1], W[q][C], idm0, idm1);
    dqs[B1] = flat ? 0.0 : vl_rad_slope(sg[B2], sg[B1], sg[C], idm0, idm1);
    // face k: upwind values (StarRadKernel2); faces 0 and NRAD are zero
    double DS = 0.0;
    double QS[NQT];
    if (IN || (k > 0 && k < nr)) {
      const double vk = vr[B1];
      const double Rkm = lane_get(rt.Rmed, r - 2), Rk = lane_get(rt.Rmed, r - 1);
      DS = vl_rad_star(vk, dt, sg[B2], sg[B1], dqs[B2], dqs[B1], Rkm, Rk, Rm, k);
      for (int q = 0; q < NQT; q++)
        QS[q] = vl_rad_star(vk, dt, W[q][B2], W[q][B1], dq[q][B2], dq[q][B1], Rkm, Rk, Rm, k);
    } else {
      for (int q = 0; q < NQT; q++) QS[q] = 0.0;
    }
    const double vface = (IN || k < nr) ? vr[B1] : 0.0;
    const double Rinf = lane_get(rt.Rinf, r - 1);
    for (int q = 0; q < NQT; q++) F[q][B1] = cflux * Rinf * QS[q] * DS * vface;
    double outer = 0.0;  // radius of ring k - 1's own outer face
    if constexpr (OWN) outer = t.Rsup[max(k - 1, 0)];
    // ring k-1 is complete: Q += (F(k-1) - F(k)) / Surf
    if (decltype(store)::value) {
      const int o = k - 1;
      const long lo = (long)o * ns + j;
      const double isurf = lane_get(rt.isurf, r - 2);
      for (int q = 0; q < NQT; q++) {
        double varq = F[q][B2];
        varq -= OWN ? cflux * outer * QS[q] * DS * vface : F[q][B1];
        a.out[q][lo] = Q[q][B2] + varq * isurf;
        if (ROUTINE && q == NQT - 1 && o == 0 && a.lost) a.lost[j] = varq;
      }
    }
  };
  // a single step in the rotating layout (newest ring in slot 2): shift
  // every window by one, then the step of phase 2.  Three consecutive
  // steps of phases 0, 1, 2 leave the windows in that same layout.
  auto shift = [&]() {
    for (int q = 0; q < NQT; q++) {
      Q[q][0] = Q[q][1];
      Q[q][1] = Q[q][2];
      W[q][0] = W[q][1];
      W[q][1] = W[q][2];
      dq[q][0] = dq[q][1];
      F[q][0] = F[q][1];
    }
    sg[0] = sg[1];
    sg[1] = sg[2];
    vr[0] = vr[1];
    vr[1] = vr[2];
    dqs[0] = dqs[1];
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  using P2 = std::integral_constant<int, 2>;
  // rings m0 .. b0 + 1 fill the window; from m = b0 + 2 on ring m - 2 of
  // the band is complete after every step
  using T = std::true_type;
  using F0 = std::false_type;
  int m = m0;
  for (; m < b0 + 2; m++) {
    shift();
    ring(m, F0(), P2(), F0());
  }
  // the storing loop starts with nothing in flight from the filling one;
  // its steps have m >= b0 + 2 >= 2, so those below nr are inner
  asm volatile("" ::"v"(n_s), "v"(n_v1), "v"(n_vtp), "v"(n_vt), "v"(n_e));
  const int mi = min(b1 + 1, nr - 1);
  for (; m + 2 <= mi; m += 3) {
    ring(m, T(), P0(), T());
    ring(m + 1, T(), P1(), T());
    ring(m + 2, T(), P2(), T());
  }
  asm volatile("" ::"v"(n_s), "v"(n_v1), "v"(n_vtp), "v"(n_vt), "v"(n_e));
  for (; m <= b1 + 1; m++) {
    shift();
    ring(m, T(), P2(), F0());
  }
}

// ------------------------------------------------------------ k_taz ----
// OneWindTheta (TransportEuler.cu:177-194) + the vtheta half of
// ComputeVelocities (Kernels.cu:1206-1207) as wave chunks (k_tazw below),
// FP64 and FP32 bulk mode.  VMed comes from the ring-mean waves of k_trad.

struct taz_args {
  const double *vt;     // vtheta after k_src
  const double *vmed;   // its ring means
  const double *q[NQ_MAX];  // quantities after the radial sweep (Sigma last)
  double *xd, *xvt, *xrmp, *xrmm, *xe;
  // FULL: the angular momenta, Sigma between the two sweeps (DENSINT) and the
  // residual velocity as well
  double *xtmp, *xtmm, *xdint, *xres;
  // FP32 bulk mode: the same fields stored in FP32 (fp32_store_bg)
  const float *fvt, *fq[NQ];
  float *fxd, *fxvt, *fxrmp, *fxrmm;
  const double *sbar, *vref;
  int *nshift;
  fg_dev_tables t;
  double dt, omega_frame;
  int nr, ns, fast;
  int lob0, lob1;  // FP32 storage: rings stored as float pairs
};


// ------------------------------------------------------- k_taz, waves ----
// No workgroup barrier: one 64-lane wave owns a
// contiguous chunk of 64*CL cells of a ring, CL consecutive cells per lane
// in registers.  A cell's neighbours are in the lane's own registers, or for
// a lane's first and last cells in the adjacent lane, fetched by DPP wave
// shifts.  The chunk carries TAZW_HL halo cells on the left and TAZW_HR on
// the right: each sweep's result at a cell depends on the cells up to two
// away, the vtheta recovery on the cell to the left, and the two lanes at
// the chunk's ends see zeros from the shifts, so the outermost 4 (right)
// and 5 (left) results of a chunk are discarded.  Chunks of one ring
// overlap by those halos; each cell is output by exactly one chunk.
#define TAZW_HL 5
#define TAZW_HR 4
// Cells per lane: two on grids below 2^20 cells and in batches, where more and
// shorter chunks fill the chip (k_tazw, us by events with two and three: 128 x 384
// 9.0 and 10.4, 512 x 1536 27.8 and 29.3; FP32 128 x 384 7.9 and 9.1, 512 x 1536 18.3
// and 19.0; 8 batched disks 177 and 180 per substep), three beyond, where the halo's
// bytes count (FP32 1024 x 3072 41.8 and 41.0, FP64 the same within 1 %).  Three
// FP64 cells take 142 or 164 VGPRs and leave three waves per SIMD, four or five
// cells two; three FP32 cells are held to 96 VGPRs, five waves.
#define TAZW_P(CL) (64 * (CL) - TAZW_HL - TAZW_HR)  // cells that a chunk outputs
static int tazw_cells(const fg_ctx *c) { return (long)c->nr * c->ns < (1L << 20) ? 2 : 3; }

__device__ __forceinline__ float lane_prev(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}

__device__ __forceinline__ float lane_next(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));
}

// QuantitiesAdvection (TransportEuler.cu:229-245) on a lane's CL cells with
// velocity V (one value per cell, or the ring's uniform residual when
// UNIFORM); the reference's operations in its order
template <int CL, bool UNIFORM, int NQT>
__device__ __forceinline__ void wave_sweep(double (&q)[NQT][CL], const double (&Vc)[CL], double Vu,
                                           const fg_dev_tables &t, int i, double dt) {
  const double invdxtheta = t.invdxtheta[i], dxtheta = t.dxtheta[i];
  const double dxrad = (t.Rsup[i] - t.Rinf[i]) * dt;
  const double invsurf = t.invSurf[i];
#define V(c) (UNIFORM ? Vu : Vc[c])
  double dens[CL], DS[CL];
  // DensStar from Sigma (ComputeStarTheta(Dens), TransportEuler.cu:232)
#pragma unroll
  for (int c = 0; c < CL; c++) dens[c] = q[NQT - 1][c];
  {
    const double Wm = lane_prev(dens[CL - 1]), Wp = lane_next(dens[0]);
    double D[CL];
#pragma unroll
    for (int c = 0; c < CL; c++)
      D[c] = vl_theta_slope(c ? dens[c - 1] : Wm, dens[c], c < CL - 1 ? dens[c + 1] : Wp, invdxtheta);
    const double Dm = lane_prev(D[CL - 1]);
#pragma unroll
    for (int c = 0; c < CL; c++)
      DS[c] = vl_theta_star(V(c), dt, c ? dens[c - 1] : Wm, dens[c], c ? D[c - 1] : Dm, D[c], dxtheta);
  }
  // VanLeerTheta of each quantity, Sigma last (TransportEuler.cu:234-243);
  // the Work divisions of a cell share its denominator Sigma + 1e-20
  double rd[CL];
#pragma unroll
  for (int c = 0; c < CL; c++) rd[c] = recip64(dens[c] + 1e-20).r;
#pragma unroll
  for (int qq = 0; qq < NQT; qq++) {
    // one quantity at a time: keeps the live registers to this quantity's
    // stencil (the scheduler would otherwise interleave all five)
    __builtin_amdgcn_sched_barrier(0);
    double W[CL], D[CL], F[CL];
#pragma unroll
    for (int c = 0; c < CL; c++) W[c] = recip64(dens[c] + 1e-20, rd[c]).div(q[qq][c]);
    const double Wm = lane_prev(W[CL - 1]), Wp = lane_next(W[0]);
#pragma unroll
    for (int c = 0; c < CL; c++)
      D[c] = vl_theta_slope(c ? W[c - 1] : Wm, W[c], c < CL - 1 ? W[c + 1] : Wp, invdxtheta);
    const double Dm = lane_prev(D[CL - 1]);
#pragma unroll
    for (int c = 0; c < CL; c++) {
      const double QS = vl_theta_star(V(c), dt, c ? W[c - 1] : Wm, W[c], c ? D[c - 1] : Dm, D[c], dxtheta);
      F[c] = dxrad * QS * DS[c] * V(c);
    }
    const double Fp = lane_next(F[0]);
#pragma unroll
    for (int c = 0; c < CL; c++) {
      double varq = F[c];
      varq -= (c < CL - 1 ? F[c + 1] : Fp);
      q[qq][c] += varq * invsurf;
    }
  }
#undef V
}

// The FP32 bulk-mode sweep on a lane's CL cells: W, slopes, upwind values
// and fluxes in FP32 with hardware reciprocals, each increment added to the
// FP64 quantity
template <int CL, bool UNIFORM>
__device__ __forceinline__ void wave_sweep32(double (&q)[NQ][CL], const float (&Vc)[CL], float Vu,
                                             const fg_dev_tables &t, int i, float dt) {
  const float invdxtheta = (float)t.invdxtheta[i], dxtheta = (float)t.dxtheta[i];
  const float dxrad = (float)((t.Rsup[i] - t.Rinf[i]) * (double)dt);
  const float invsurf = (float)t.invSurf[i];
#define V(c) (UNIFORM ? Vu : Vc[c])
  float rs[CL], DS[CL];
  {
    float d[CL], D[CL];
#pragma unroll
    for (int c = 0; c < CL; c++) {
      d[c] = (float)q[NQ - 1][c];
      rs[c] = rcp_f(d[c] + 1e-20f);
    }
    const float Wm = lane_prev(d[CL - 1]), Wp = lane_next(d[0]);
#pragma unroll
    for (int c = 0; c < CL; c++)
      D[c] = vl_theta_slope_f(c ? d[c - 1] : Wm, d[c], c < CL - 1 ? d[c + 1] : Wp, invdxtheta);
    const float Dm = lane_prev(D[CL - 1]);
#pragma unroll
    for (int c = 0; c < CL; c++)
      DS[c] = vl_theta_star_f(V(c), dt, c ? d[c - 1] : Wm, d[c], c ? D[c - 1] : Dm, D[c], dxtheta) * V(c) * dxrad;
  }
#pragma unroll
  for (int qq = 0; qq < NQ; qq++) {
    __builtin_amdgcn_sched_barrier(0);
    float W[CL], D[CL], F[CL];
#pragma unroll
    for (int c = 0; c < CL; c++) W[c] = (float)q[qq][c] * rs[c];
    const float Wm = lane_prev(W[CL - 1]), Wp = lane_next(W[0]);
#pragma unroll
    for (int c = 0; c < CL; c++)
      D[c] = vl_theta_slope_f(c ? W[c - 1] : Wm, W[c], c < CL - 1 ? W[c + 1] : Wp, invdxtheta);
    const float Dm = lane_prev(D[CL - 1]);
#pragma unroll
    for (int c = 0; c < CL; c++)
      F[c] = vl_theta_star_f(V(c), dt, c ? W[c - 1] : Wm, W[c], c ? D[c - 1] : Dm, D[c], dxtheta) * DS[c];
    const float Fp = lane_next(F[0]);
#pragma unroll
    for (int c = 0; c < CL; c++) q[qq][c] += (double)((F[c] - (c < CL - 1 ? F[c + 1] : Fp)) * invsurf);
  }
#undef V
}

// chunk `chunk` of ring i, one wave; F32 selects the FP32 bulk-mode sweeps;
// NQT = 6 adds the energy of an adiabatic deck (FP64 only)
// LDS of one chunk: the load stage, then the output stages (row 0 reused)
template <int CL, int NQT>
struct tazw_lds {
  double ostage[NQT == 6 ? 5 : 4][64 * CL];
};
// PAIRS: a ring of the FP32 mode stored as float pairs (its own instance,
// so that the other rings run without the residuals' loads and branches)
// FULL: the fields that fg_transport leaves besides (FP64)
template <int CL, bool F32, int NQT = 5, bool PAIRS = false, bool FULL = false>
__device__ __forceinline__ void tazw_body(const taz_args &a, int i, int chunk, tazw_lds<CL, NQT> &lds) {
  constexpr int N = 64 * CL, P = N - TAZW_HL - TAZW_HR;
  static_assert(NQT == 5 || !F32, "the FP32 sweeps carry five quantities");
  static_assert(F32 || !PAIRS, "float pairs are an FP32 storage form");
  auto &ostage = lds.ostage;
  double *stage = ostage[0];
  const int ns = a.ns, l = threadIdx.x;
  const int g0 = chunk * P - TAZW_HL;  // unwrapped index of the chunk's first cell
  const fg_dev_tables &t = a.t;
  const long base = (long)i * ns;
  // loads: coalesced global reads into the chunk's LDS stage, then CL
  // consecutive cells per lane (a one-wave workgroup: the barriers only
  // order the LDS accesses of the wave)
  double q[NQT][CL];
  using vel_t = typename std::conditional<F32, float, double>::type;
  vel_t vres[CL];
  const double VMed = a.vmed[i];
  double vt0[CL];
  // ring index of this lane's staged cell m: one modulo, then steps of 64
  int jl[CL];
  {
    int j = ((g0 + l) % ns + ns) % ns;
#pragma unroll
    for (int m = 0; m < CL; m++) {
      jl[m] = j;
      j += 64;
      while (j >= ns) j -= ns;
    }
  }
  // every field's loads are issued before the first is staged, so the six
  // fields cost one memory latency, not six.  FP32 mode: the fields are
  // FP32 offsets from the ring's backgrounds (fp32_store_bg)
  double raw[NQT + 1][CL];
  double sb = 0.0, vb = 0.0, lb = 0.0;
  constexpr bool lob = PAIRS;  // FP32 storage: this ring is stored as float pairs
  const long S = (long)(a.nr + 1) * ns;
  if constexpr (F32) {
    float fr[NQT + 1][CL], fsl[CL];
#pragma unroll
    for (int qq = 0; qq <= NQT; qq++) {
      const float *src = qq < NQT ? a.fq[qq] : a.fvt;
#pragma unroll
      for (int m = 0; m < CL; m++) fr[qq][m] = src[base + jl[m]];
    }
#pragma unroll
    for (int m = 0; m < CL; m++) fsl[m] = lob ? a.fq[4][S + base + jl[m]] : 0.f;
    sb = a.sbar[i];
    vb = a.vref[i];
    const double Rm = t.Rmed[i];
#pragma unroll
    for (int m = 0; m < CL; m++) {
      const double s = rec32(sb, fr[4][m], fsl[m]);
      lb = fp32_bg_angmom(s, vb, Rm, a.omega_frame);  // the cell's angular momentum background
      raw[0][m] = (double)fr[0][m];
      raw[1][m] = (double)fr[1][m];
      raw[2][m] = lb + (double)fr[2][m];
      raw[3][m] = lb + (double)fr[3][m];
      raw[4][m] = s;
      raw[5][m] = vb + (double)fr[5][m];
    }
  } else {
#pragma unroll
    for (int qq = 0; qq <= NQT; qq++) {
      const double *src = qq < NQT ? a.q[qq] : a.vt;
#pragma unroll
      for (int m = 0; m < CL; m++) raw[qq][m] = src[base + jl[m]];
    }
  }
#pragma unroll
  for (int qq = 0; qq <= NQT; qq++) {
#pragma unroll
    for (int m = 0; m < CL; m++) stage[l + 64 * m] = raw[qq][m];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CL; c++) {
      const double v = stage[l * CL + c];
      if (qq < NQT)
        q[qq][c] = v;
      else
        vt0[c] = v - VMed;  // ComputeResidualsKernel
    }
    __syncthreads();
  }
  // ComputeConstantResidualKernel (Kernels.cu:1094-1126)
  const double invdt = 1.0 / a.dt;
  const double dpinvns = 2.0 * FG_PI / (double)ns;
  const double Ntilde = VMed * t.invRmed[i] * a.dt * (double)ns / 2.0 / FG_PI;
  const double Nround = floor(Ntilde + 0.5);
  const int nsh = (int)(long)Nround;
  double vuni = (Ntilde - Nround) * t.Rmed[i] * invdt * dpinvns;
#pragma unroll
  for (int c = 0; c < CL; c++) vres[c] = (vel_t)(a.fast ? vt0[c] : vt0[c] + vuni);
  if (!a.fast) vuni = 0.0;
  if (chunk == 0 && l == 0) a.nshift[i] = nsh;
  if constexpr (F32 && NQT == 5) {
    wave_sweep32<CL, false>(q, vres, 0.0f, t, i, (float)a.dt);
    wave_sweep32<CL, true>(q, vres, (float)vuni, t, i, (float)a.dt);
  } else {
    wave_sweep<CL, false, NQT>(q, vres, 0.0, t, i, a.dt);
    if constexpr (FULL) {  // neither is shifted
#pragma unroll
      for (int c = 0; c < CL; c++) {
        ostage[0][l * CL + c] = q[NQT - 1][c];
        ostage[1][l * CL + c] = vres[c];
      }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < CL; m++) {
        const int k = l + 64 * m, g = g0 + k;
        if (k >= TAZW_HL && k < TAZW_HL + P && g < ns) {
          a.xdint[base + g] = ostage[0][k];
          a.xres[base + g] = ostage[1][k];
        }
      }
      __syncthreads();
    }
    wave_sweep<CL, true, NQT>(q, vres, vuni, t, i, a.dt);
  }
  // vtheta from the angular momenta (Kernels.cu:1206-1207): cells j - 1
  // and j of the unshifted ring
  const double Rm = t.Rmed[i];
  const recip64 rRm(Rm);
  double vt[CL];
  {
    const double Wm = lane_prev(q[2][CL - 1]), Sm = lane_prev(q[NQT - 1][CL - 1]);
#pragma unroll
    for (int c = 0; c < CL; c++) {
      const double s = q[NQT - 1][c];
      vt[c] = rRm.div(((c ? q[2][c - 1] : Wm) + q[3][c]) / (s + (c ? q[NQT - 1][c - 1] : Sm) + 1e-15)) -
              Rm * a.omega_frame;
    }
  }
  // stores with AdvectSHIFT (Kernels.cu:1173-1190) folded in: cell j goes
  // to j + Nshift (mod NSEC); the chunk outputs its cells [HL, HL + P)
  // that lie in [0, NSEC)
  int sh = nsh % ns;
  if (sh < 0) sh += ns;
  // all four outputs staged at once, then their coalesced stores back to
  // back (one LDS round trip instead of four)
#pragma unroll
  for (int c = 0; c < CL; c++) {
    ostage[0][l * CL + c] = q[NQT - 1][c];
    ostage[1][l * CL + c] = vt[c];
    ostage[2][l * CL + c] = q[0][c];
    ostage[3][l * CL + c] = q[1][c];
    if constexpr (NQT == 6) ostage[4][l * CL + c] = q[4][c];
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < CL; m++) {
    const int k = l + 64 * m;
    const int g = g0 + k;
    if (k >= TAZW_HL && k < TAZW_HL + P && g < ns) {
      int jo = g + sh;
      if (jo >= ns) jo -= ns;
      const long lo = base + jo;
      if constexpr (F32) {
        const double xd = ostage[0][k] - sb;
        const float hd = (float)xd;
        a.fxd[lo] = hd;
        a.fxvt[lo] = (float)(ostage[1][k] - vb);
        a.fxrmp[lo] = (float)ostage[2][k];
        a.fxrmm[lo] = (float)ostage[3][k];
        if constexpr (lob) a.fxd[S + lo] = (float)(xd - (double)hd);
      } else {
        a.xd[lo] = ostage[0][k];
        a.xvt[lo] = ostage[1][k];
        a.xrmp[lo] = ostage[2][k];
        a.xrmm[lo] = ostage[3][k];
        if constexpr (NQT == 6) a.xe[lo] = ostage[4][k];
      }
    }
  }
  if constexpr (FULL) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CL; c++) {
      ostage[0][l * CL + c] = q[2][c];
      ostage[1][l * CL + c] = q[3][c];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < CL; m++) {
      const int k = l + 64 * m, g = g0 + k;
      if (k >= TAZW_HL && k < TAZW_HL + P && g < ns) {
        int jo = g + sh;
        if (jo >= ns) jo -= ns;
        a.xtmp[base + jo] = ostage[0][k];
        a.xtmm[base + jo] = ostage[1][k];
      }
    }
  }
}

// blockIdx.x = chunk, blockIdx.y = ring
template <int CL, int NQT>
__global__ __launch_bounds__(64) void k_tazw(taz_args a) {
  __shared__ tazw_lds<CL, NQT> sh;
  tazw_body<CL, false, NQT>(a, blockIdx.y, blockIdx.x, sh);
}

// the azimuthal sweeps of fg_transport
template <int CL, int NQT>
__global__ __launch_bounds__(64) void k_tazw_full(taz_args a) {
  __shared__ tazw_lds<CL, NQT> sh;
  tazw_body<CL, false, NQT, false, true>(a, blockIdx.y, blockIdx.x, sh);
}

// the FP32 bulk mode's single-disk sweep
template <int CL>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(CL == 2 ? 7 : 5))) void k_tazw32(taz_args a) {
  __shared__ tazw_lds<CL, 5> sh;
  if (in_lob(blockIdx.y, a.lob0, a.lob1))
    tazw_body<CL, true, 5, true>(a, blockIdx.y, blockIdx.x, sh);
  else
    tazw_body<CL, true, 5, false>(a, blockIdx.y, blockIdx.x, sh);
}

// ------------------------------------------------------------ k_fin ----
// vrad recovery (Kernels.cu:1200-1205), the third damping pass, the
// temperature and, for the next substep, ConditionCFLKernel1D/2D1/2D2 of
// this ring (vrad of ring i+1 is recomputed here, it is needed by
// Kernels.cu:1302).
struct fin_args {
  const double *xd, *xvt, *xrmp, *xrmm, *press;
  double *dens, *vr, *vt, *temp;
  // adiabatic decks: the transported energy in, Energy out; the sound speed
  // field of the CFL pass (the one of the DT's start, SourceEuler.cu:208),
  // recomputed from the final state when this substep closes the DT
  const double *xe;
  double *energy, *cs;
  double gamma;
  int adiabatic, cs_refresh;
  const double *sgacc;  // self-gravity: ring means of g_r for vtheta0 (else NULL)
  // FP32 bulk mode: the fields of k_taz stored in FP32 (fp32_store_bg) with
  // the backgrounds sbar (Sigma) and vmoy (vtheta, read before this pass
  // overwrites it), and the next substep's Sigma background
  const float *fxd, *fxvt, *fxrmp, *fxrmm;
  const double *sbar;
  double *sbar_next;
  double *vmoy, *newdt;
  double *fpart;  // FP32 mode: per-ring compensated star-force partials (4 per ring), else NULL
  int *crash;     // set to 1 when a stored density is negative or not finite
  const double *nu;
  fg_dev_tables t;
  double dt, omega_frame;
  int nr, ns, evanescent, fast;
  int lob0, lob1;  // FP32 storage: rings stored as float pairs
};


// Neumaier-compensated sums (value s, correction c) of the FP32 mode's
// star force: per thread in cell order, then a fixed shuffle tree per
// wave and the waves in order
__device__ __forceinline__ void kadd(double &s, double &c, double x) {
  const double t = s + x;
  c += (fabs(s) >= fabs(x)) ? ((s - t) + x) : ((x - t) + s);
  s = t;
}
__device__ __forceinline__ void kmerge(double &s, double &c, double s2, double c2) {
  kadd(s, c, s2);
  c += c2;
}
__device__ __forceinline__ void kwave(double &s, double &c) {
  for (int off = 32; off > 0; off >>= 1) {
    const double s2 = __shfl_down(s, off), c2 = __shfl_down(c, off);
    kmerge(s, c, s2, c2);
  }
}

// disk force on the star from the per-ring partials, in a fixed order: each
// thread merges a contiguous run of rings, then a shuffle tree per wave,
// then the waves in order.  Called by every thread of a 256-thread block.
__device__ __forceinline__ void force_rings_final(const double *fpart, int nr, double *out2) {
  __shared__ double ws[4][4];
  const int tid = threadIdx.x, per = (nr + 255) / 256;
  double sx = 0.0, cx = 0.0, sy = 0.0, cy = 0.0;
  for (int q = 0; q < per; q++) {
    const int i = tid * per + q;
    if (i < nr) {
      kmerge(sx, cx, fpart[4 * i], fpart[4 * i + 1]);
      kmerge(sy, cy, fpart[4 * i + 2], fpart[4 * i + 3]);
    }
  }
  kwave(sx, cx);
  kwave(sy, cy);
  if ((tid & 63) == 0) {
    ws[tid >> 6][0] = sx;
    ws[tid >> 6][1] = cx;
    ws[tid >> 6][2] = sy;
    ws[tid >> 6][3] = cy;
  }
  __syncthreads();
  if (tid == 0) {
    double a = ws[0][0], b = ws[0][1], c = ws[0][2], d = ws[0][3];
    for (int w = 1; w < 4; w++) {
      kmerge(a, b, ws[w][0], ws[w][1]);
      kmerge(c, d, ws[w][2], ws[w][3]);
    }
    out2[0] = a + b;
    out2[1] = c + d;
  }
}

// FP32 mode: the star force from the per-ring partials, then the CFL count
// (ConditionCFLKernel2D2 + 2D3, Kernels.cu:1331-1359) in the same launch.
// Up to 1024 rings a thread's force partials (rings tid * per + q, merged
// in q order as force_rings_final does) are loaded together with its CFL
// inputs, so the block waits for memory once.
// The launch's sequence number goes last into slot FG_FUSED_SEQ_SLOT of the
// result block out (behind a system-scope fence: every result above is
// visible to the host first; thread 0 and the lanes that wrote them are in
// wave 0).
__device__ __forceinline__ void seq_store(double *slot, double seq) {
  if (threadIdx.x == 0) {
    __threadfence_system();
    *slot = seq;
  }
}

__device__ __forceinline__ void force_rings_cfl(const double *fpart, int nr, double *out2, double *cfl, double *dt1d,
                                                const double *vmoy, const double *newdt, const double *invRmed,
                                                double coef, double DeltaT) {
  if (nr > 4 * 256) {
    force_rings_final(fpart, nr, out2);
    __syncthreads();
    cfl_final(cfl, dt1d, vmoy, newdt, invRmed, coef, DeltaT, nr);
    return;
  }
  __shared__ double ws[4][4];
  const int tid = threadIdx.x, per = (nr + 255) / 256;
  double fp[4][4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int i = tid * per + q;
#pragma unroll
    for (int c = 0; c < 4; c++) fp[q][c] = (q < per && i < nr) ? fpart[4 * i + c] : 0.0;
  }
  const double best = cfl_ring_min(dt1d, vmoy, newdt, invRmed, coef, nr, tid, 256);
  double sx = 0.0, cx = 0.0, sy = 0.0, cy = 0.0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if (q < per && tid * per + q < nr) {
      kmerge(sx, cx, fp[q][0], fp[q][1]);
      kmerge(sy, cy, fp[q][2], fp[q][3]);
    }
  }
  kwave(sx, cx);
  kwave(sy, cy);
  if ((tid & 63) == 0) {
    ws[tid >> 6][0] = sx;
    ws[tid >> 6][1] = cx;
    ws[tid >> 6][2] = sy;
    ws[tid >> 6][3] = cy;
  }
  const double m = block_min256(best);  // (its barrier also orders ws)
  if (tid == 0) {
    double a = ws[0][0], b = ws[0][1], c = ws[0][2], d = ws[0][3];
    for (int w = 1; w < 4; w++) {
      kmerge(a, b, ws[w][0], ws[w][1]);
      kmerge(c, d, ws[w][2], ws[w][3]);
    }
    out2[0] = a + b;
    out2[1] = c + d;
  }
  cfl_count_store(cfl, m, DeltaT);
}

// minimum over the workgroup's 256 threads into *out (thread 0): within
// each wave by shuffles, then the four wave minima (a minimum does not
// depend on the order of its comparisons)
__device__ __forceinline__ void ring_min_store(double best, double *red, double *out) {
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_down(best, off, 64);
    if (o < best) best = o;
  }
  const int tid = threadIdx.x;
  if ((tid & 63) == 0) red[tid >> 6] = best;
  __syncthreads();
  if (tid == 0) {
    double m = red[0];
    for (int w = 1; w < 4; w++)
      if (red[w] < m) m = red[w];
    *out = m;
  }
}

// One ring by 256 threads, thread t its cells t, t + 256, ...; ring: NSEC doubles
// of LDS.  First the final vtheta of every cell goes to LDS and its ring mean
// is formed (FP64: ring_seq_sum; the FP32 mode, which does not
// replay the reference's summation order, from the threads' own sums), then one
// pass over the cells does the rest: ComputeVelocities (Kernels.cu:1200-1205)
// with the energy, sound speed and temperature of an adiabatic deck, and the
// cell's CFL time step (Kernels.cu:1284-1329).  Every cell issues the same memory
// operations, its loads one cell ahead, so that the waits for them count past
// the stores: threads without a cell left repeat the last one's.
// The ring minimum of dt = 0.5 / sqrt(S) over the cells is taken as one
// quotient at the largest S: rounded sqrt and rounded division are both
// monotone, so 0.5 / sqrt(max S) is the smallest rounded dt bit for bit
// (a NaN S is skipped by both comparisons; the 1e30 start caps both).
// ADI: adiabatic deck; S32: FP32 bulk mode (FP32 storage of k_taz's fields);
// PAIRS: ring i - 1, i or i + 1 stored as float pairs (its own instance, so that
// the other rings run without the residuals' loads).
// Bound: HBM on large grids (2048 x 4096: 478 MB by the counters, 470 of them
// compulsory, in 117 us), latency on small
// ones.  Was one lane's sum of the ring beside a pass that kept its terms in
// registers (and two passes over rings beyond 3072 cells): 1024 x 3072 61 -> 52
// us, 2048 x 4096 198 -> 117, 512 x 1536 22 -> 17 (adiabatic 24 -> 23); FP32
// 1024 x 3072 44 -> 36, 128 x 384 9.2 -> 8.1; FP64 at 128 x 384, where the pass was
// one cell or two a thread, 7.2 -> 8.2.
// Keeping that pass's terms unrolled over 12 or 16 cells was slower than the loop,
// 512 threads a ring too (two rounds of workgroups).
template <bool ADI, bool S32, bool PAIRS>
__device__ __forceinline__ void fin_ring(const fin_args &a, int i, double *ring) {
  using real = typename std::conditional<S32, float, double>::type;
  struct cell {
    real rpm, rm, dm, d, rp, rn, dn;  // momenta and Sigma of rings i - 1, i and i + 1
    float ym, y, yn;                  // PAIRS: Sigma's residuals
    double e, c, cosj, sinj;          // energy, sound speed; S32: the cell's direction
  };
  __shared__ double red[4];
  const int ns = a.ns, nr = a.nr, tid = threadIdx.x;
  const fg_dev_tables &t = a.t;
  const long row = (long)i * ns, rowm = (long)max(i - 1, 0) * ns, rown = row + ns, S2 = (long)(nr + 1) * ns;
  double lam_i = 0, vr0_i = 0, vt0_i = 0, lam_n = 0, vr0_n = 0, vt0_n = 0;
  const bool damp_i = a.evanescent && t.ev_zone[i];
  const bool damp_n = a.evanescent && (i + 1 < nr) && t.ev_zone[i + 1];
  if (damp_i) ev_consts(t, a.nu, i, a.dt, a.omega_frame, lam_i, vr0_i, vt0_i, a.sgacc);
  if (damp_n) ev_consts(t, a.nu, i + 1, a.dt, a.omega_frame, lam_n, vr0_n, vt0_n, a.sgacc);
  const bool radial = i > 0, radial_n = i + 1 < nr;  // vrad is 0 on ring 0 and the ghost ring
  const bool cfl = i > 0;                            // ring 0 has no CFL term (Kernels.cu:1286)
  // FP32 storage: backgrounds of rings i-1, i, i+1 and of vtheta on ring i
  const double sb_m = S32 && radial ? a.sbar[i - 1] : 0.0, sb_i = S32 ? a.sbar[i] : 0.0;
  const double sb_n = S32 && radial_n ? a.sbar[i + 1] : 0.0, vb_i = S32 ? a.vmoy[i] : 0.0;
  const bool lob_m = PAIRS && in_lob(i - 1, a.lob0, a.lob1), lob_i = PAIRS && in_lob(i, a.lob0, a.lob1);
  const bool lob_n = PAIRS && in_lob(i + 1, a.lob0, a.lob1);
  auto fetch = [&](int jc, cell &x) __attribute__((always_inline)) {
    unsigned o = min(jc, ns - 1) * (unsigned)sizeof(real);
    asm volatile("" : "+v"(o));  // (the rows' addresses stay scalar)
    if constexpr (S32) {
      x.rpm = at(a.fxrmp + rowm, o);
      x.rm = at(a.fxrmm + row, o);
      x.dm = at(a.fxd + rowm, o);
      x.d = at(a.fxd + row, o);
      x.rp = at(a.fxrmp + row, o);
      x.rn = at(a.fxrmm + rown, o);
      x.dn = at(a.fxd + rown, o);
      x.cosj = at(t.cos_cell, 2 * o);
      x.sinj = at(t.sin_cell, 2 * o);
      x.ym = x.y = x.yn = 0.f;
      if constexpr (PAIRS) {
        x.ym = at(a.fxd + S2 + rowm, o);
        x.y = at(a.fxd + S2 + row, o);
        x.yn = at(a.fxd + S2 + rown, o);
      }
    } else {
      x.rpm = at(a.xrmp + rowm, o);
      x.rm = at(a.xrmm + row, o);
      x.dm = at(a.xd + rowm, o);
      x.d = at(a.xd + row, o);
      x.rp = at(a.xrmp + row, o);
      x.rn = at(a.xrmm + rown, o);
      x.dn = at(a.xd + rown, o);
      if constexpr (ADI) {
        x.e = at(a.xe + row, o);
        x.c = at((const double *)a.cs + row, o);
      }
    }
  };
  double vsum = 0.0;
  for (int j0 = tid; j0 < ns; j0 += 256 * 4) {
    real v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = min(j0 + 256 * u, ns - 1);
      if constexpr (S32)
        v[u] = a.fxvt[row + j];
      else
        v[u] = a.xvt[row + j];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = j0 + 256 * u;
      double vt = S32 ? vb_i + (double)v[u] : v[u];
      if (damp_i) vt = damp_toward(vt, lam_i, vt0_i);
      if (j < ns) {
        ring[j] = vt;
        if (S32) vsum += vt;
      }
    }
  }
  cell c0, c1;
  fetch(tid, c0);
  __shared__ double fw[S32 ? 4 : 1][5];
  double vm;
  if constexpr (S32) {  // per wave by a shuffle tree, the waves in order
    for (int off = 32; off > 0; off >>= 1) vsum += __shfl_down(vsum, off);
    if ((tid & 63) == 0) red[tid >> 6] = vsum;
    __syncthreads();
    vm = (((red[0] + red[1]) + red[2]) + red[3]) / (double)ns;
  } else {
    __syncthreads();
    vm = ring_seq_sum(ring, ns) / (double)ns;
  }
  if (tid == 0) a.vmoy[i] = vm;
  const double Rm = t.Rmed[i], surf = t.Surf[i];
  // star at the origin (x = y = 0, no smoothing): the cell's distance is
  // Rmed, so 1/d^3 is one value per ring (FP32 mode only; the FP64 path
  // sums the reference's per-cell expression in DeviceReduce order)
  const double inv3 = 1.0 / (Rm * Rm) / Rm;
  double fsx = 0.0, fcx = 0.0, fsy = 0.0, fcy = 0.0, ssum = 0.0;
  const double dxrad = t.Rsup[i] - t.Rinf[i], dxtheta = t.dxtheta_cfl[i];
  const double mindx = (dxtheta < dxrad) ? dxtheta : dxrad;
  const double invdt1r = t.cs_iso[i] / mindx;
  const recip64 rdr(dxrad), rdt(dxtheta);
  const double sigma0 = t.SigmaMed[i], energy0 = ADI ? t.EnergyMed[i] : 0.0;
  bool bad = false;  // a density below 0, infinite or NaN
  double smax = -1.0;
  auto pass = [&](int jc, const cell &x) __attribute__((always_inline)) {
    const bool mine = jc < ns;
    const int j = min(jc, ns - 1);
    unsigned o = 8u * j;
    asm volatile("" : "+v"(o));
    double ld = x.d, ldm = x.dm, ldn = x.dn;
    if constexpr (S32) {
      ld = rec32(sb_i, x.d, lob_i ? x.y : 0.f);
      ldm = rec32(sb_m, x.dm, lob_m ? x.ym : 0.f);
      ldn = rec32(sb_n, x.dn, lob_n ? x.yn : 0.f);
    }
    double vr = radial ? ((double)x.rpm + (double)x.rm) / (ld + ldm + 1e-20) : 0.0;
    const double vt = ring[j];
    double s = ld;
    if (damp_i) {
      vr = damp_toward(vr, lam_i, vr0_i);
      s = damp_toward(s, lam_i, sigma0);
    }
    at(a.dens + row, o) = s;
    bad |= !(s >= 0.0 && s < HUGE_VAL);
    at(a.vr + row, o) = vr;
    at(a.vt + row, o) = vt;
    if constexpr (S32) {
      if (mine) {
        ssum += s;
        const double cm = surf * s;
        kadd(fsx, fcx, cm * (Rm * x.cosj) * inv3);
        kadd(fsy, fcy, cm * (Rm * x.sinj) * inv3);
      }
    }
    double csv = x.c;
    if (ADI) {
      double e = x.e;
      if (damp_i) e = damp_toward(e, lam_i, energy0);
      at(a.energy + row, o) = e;
      bad |= !(e >= 0.0 && e < HUGE_VAL);
      if (a.temp) at(a.temp + row, o) = (a.gamma - 1.0) * e / s;  // Kernels.cu:211
      if (a.cs_refresh) {
        csv = sqrt(a.gamma * (a.gamma - 1.0) * e / s);  // Kernels.cu:181
        at(a.cs + row, o) = csv;
      }
    } else if (a.temp) {
      at(a.temp + row, o) = at(a.press + row, o) / s;
    }
    if (cfl) {
      double vrn = radial_n ? ((double)x.rp + (double)x.rn) / (ldn + ld + 1e-20) : 0.0;
      if (damp_n) vrn = damp_toward(vrn, lam_n, vr0_n);
      const double invdt1 = ADI ? csv / mindx : invdt1r;
      const double invdt2 = rdr.div(fabs(vr));
      double dvr = vrn - vr;
      const double vres = a.fast ? vt - vm : vt;
      const double invdt3 = rdt.div(fabs(vres));
      double dvt = ring[j + 1 == ns ? 0 : j + 1] - vt;
      dvr = (dvr >= 0.0) ? 1e-10 : -dvr;
      dvt = (dvt >= 0.0) ? 1e-10 : -dvt;
      const double xx = rdr.div(dvr), y = rdt.div(dvt);
      double invdt4 = (y > xx) ? y : xx;
      invdt4 *= 4.0 * 1.41 * 1.41;
      const double sq = invdt1 * invdt1 + invdt2 * invdt2 + invdt3 * invdt3 + invdt4 * invdt4;
      if (sq > smax) smax = sq;
    }
  };
  for (int j = tid; j - tid < ns; j += 512) {
    fetch(j + 256, c1);
    pass(j, c0);
    if (j - tid + 256 >= ns) break;
    fetch(j + 512, c0);
    pass(j + 256, c1);
  }
  if (bad) *a.crash = 1;
  if (i == nr - 1) {  // ghost ring after transport: all zero
    for (int j = tid; j < ns; j += 256) {
      a.dens[rown + j] = a.vr[rown + j] = a.vt[rown + j] = 0.0;
      if (ADI) a.energy[rown + j] = 0.0;
    }
  }
  if constexpr (S32) {
    // the gravity of the ring's cells on the star (Kernels.cu:703-727 at x = y =
    // 0: the star sits at the origin with no smoothing, so 1/d^3 is one value
    // per ring) and the ring's Sigma sum (the next substep's background),
    // reduced as above; the force as one compensated partial per ring
    kwave(fsx, fcx);
    kwave(fsy, fcy);
    for (int off = 32; off > 0; off >>= 1) ssum += __shfl_down(ssum, off);
    if ((tid & 63) == 0) {
      double *w = fw[tid >> 6];
      w[0] = fsx;
      w[1] = fcx;
      w[2] = fsy;
      w[3] = fcy;
      w[4] = ssum;
    }
    __syncthreads();
    if (tid == 0) {
      double sx = fw[0][0], cx = fw[0][1], sy = fw[0][2], cy = fw[0][3];
      for (int w = 1; w < 4; w++) {
        kmerge(sx, cx, fw[w][0], fw[w][1]);
        kmerge(sy, cy, fw[w][2], fw[w][3]);
      }
      a.fpart[4 * i] = sx;
      a.fpart[4 * i + 1] = cx;
      a.fpart[4 * i + 2] = sy;
      a.fpart[4 * i + 3] = cy;
      a.sbar_next[i] = (((fw[0][4] + fw[1][4]) + fw[2][4]) + fw[3][4]) / (double)ns;
    }
  }
  if (!cfl) return;
  double best = 1e30;
  if (smax >= 0.0) {
    const double dtc = 0.5 / sqrt(smax);
    if (dtc < best) best = dtc;
  }
  ring_min_store(best, red, a.newdt + i);
}

// Workgroups are dispatched round-robin over the 8 XCDs.  Each XCD gets a
// contiguous band of rings, so neighbouring rings, which read each other's
// momenta and densities, are processed side by side under one L2.
template <bool ADI, bool S32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_fin(fin_args a) {
  extern __shared__ double lds_fin[];
  const int i = xcd_block(a.nr);
  if (i < 0) return;
  if (S32 && in_lob(i, a.lob0 - 1, a.lob1 + 1))
    fin_ring<ADI, S32, true>(a, i, lds_fin);
  else
    fin_ring<ADI, S32, false>(a, i, lds_fin);
}

// ================================================== FP32 bulk mode ====
// Same passes as above with the arithmetic in single precision.  The state
// (Sigma, vrad, vtheta) and the transported quantities between passes stay
// FP64; every FP32 result enters them as an increment added in FP64, so an
// update smaller than one FP32 ulp of the field is not lost and the fields
// do not random-walk by an ulp per substep.  Quantities whose FP32 rounding
// would cancel catastrophically are kept in FP64:
//   - star gravity against the centrifugal term in the radial momentum
//     equation (both ~1/r^2, their sum ~h^2/r^2): formed in FP64 per cell
//     from per-ring values and the cell's vtheta offset;
//   - vtheta is staged in LDS as the offset from a per-ring reference
//     (the ring mean of the previous substep), a few 1e-3 of |vtheta|;
//   - cell-planet separations are differenced in FP64;
//   - the FARGO ring mean, Ntilde/Nshift and the uniform residual, the CFL
//     count and the disk force are the FP64 code of the exact path.
struct src32_args {
  const double *dens, *vr, *vt;
  const double *vref;  // per-ring reference vtheta
  const double *sbar;  // per-ring background of Sigma
  float *odens, *ovr, *ovt;  // FP32 storage (fp32_store_bg)
  double *opress;
  const double *nu;
  fg_dev_tables t;
  fg_planets_arg P;
  double dt, omega_frame, domega;
  int nr, ns, indirect, evanescent;
  int lob0, lob1;            // FP32 storage: rings stored as float pairs
  int nstrips, width, band;  // strips of `width` columns, bands of `band` rings
};

// a planet's part of the potential at (x, y) (the star's -1/r is applied per
// ring); Kernels.cu:1234-1252 with the separation in FP64
__device__ __forceinline__ float planet_potential_f(double x, double y, double xp, double yp, double m, double smooth,
                                                    double invd3, int indirect) {
  const float dx = (float)(x - xp), dy = (float)(y - yp);
  const float mf = (float)m;
  float pv = -mf * __builtin_amdgcn_rsqf(dx * dx + dy * dy + (float)smooth);
  if (indirect) pv += mf * (float)invd3 * (float)(x * xp + y * yp);
  return pv;
}

// k_src's march in the FP32 bulk mode: the same strips, halos, stages and
// windows (there), in single precision, with the ring's FP64 state of
// step m kept until ring m is complete; block `block` of the disk's strips
// and bands.  Per-ring values: in FP64 S3_*, rounded to FP32 S3F_*; VB the
// ring part of the azimuthal velocity at the ring's inner face, STAR the
// star's gravity there, DREF the reference part of the shear.
// Bound: VALU issue (~300 instructions a cell) and latency on small grids; as
// 16 x 64 LDS tiles it evaluated 1.55 cells per cell and 590 instructions.
// 1024 x 3072: 66 -> 42 us; 64 disks of 128 to 384 rings: 214 -> 108 us.
#define SRC32_WAVES 4  // per SIMD
enum { S3_MED, S3_CS, S3_VB, S3_IINF, S3_STAR, S3_VREF, S3_SBAR, S3_N };
enum { S3F_IDMED, S3F_IDXT, S3F_SUPP, S3F_IMED, S3F_IDSUP, S3F_SUP, S3F_INF, S3F_NU, S3F_IINF, S3F_MED, S3F_DREF, S3F_N = 12 };
struct src32_lds {
  double tab[SRC_ROWS][S3_N], evc[SRC_ROWS][EV_N];
  float ftab[SRC_ROWS][S3F_N];
};

// PL: where the planets behind the first one are read (indexed by a loop, a
// by-value copy would live in scratch)
template <class PL>
__device__ __forceinline__ void src32_march(const src32_args &a, const PL &more, int block, src32_lds &lds) {
  constexpr int AHEAD = 2;  // rings whose loads are in flight
  auto &tab = lds.tab;
  auto &evc = lds.evc;
  auto &ftab = lds.ftab;
  const int nr = a.nr, ns = a.ns, lane = threadIdx.x, band = a.band, nstrips = a.nstrips, width = a.width;
  const int strip = block % nstrips, i0 = block / nstrips * band;
  const int i1 = min(i0 + band, nr + 1);
  const fg_dev_tables &t = a.t;
  const double *dens = global(a.dens), *vrad = global(a.vr), *vtheta = global(a.vt);
  float *odens = global(a.odens), *ovr = global(a.ovr), *ovt = global(a.ovt);
  double *opress = global(a.opress);
  const double dt = a.dt, OF = a.omega_frame, domega = a.domega;
  const float dtf = (float)dt;
  const int lob0 = a.lob0, lob1 = a.lob1, indirect = a.indirect, nb = a.P.nb;
  const int g = strip * width - SRC_HL + lane;
  const int j = (g % ns + ns) % ns;
  unsigned jb = 8u * j, jf = 4u * j;
  const bool mine = lane >= SRC_HL && lane < SRC_HL + width && g < ns;
  const double cosp = global(t.cos_pot)[j], sinp = global(t.sin_pot)[j];
  double n_s[3], n_vr[3], n_vt[3];
  auto fetch = [&](int m, auto phase) __attribute__((always_inline)) {
    constexpr int X = decltype(phase)::value % 3;
    const long l = (long)min(max(m, 0), nr) * ns;
    n_s[X] = at(dens + l, jb);
    n_vr[X] = at(vrad + l, jb);
    n_vt[X] = at(vtheta + l, jb);
  };
#define LVL(n) std::integral_constant<int, n>()
  fetch(i0 - SRC_HT, LVL(0));
  if (AHEAD > 1) fetch(i0 - SRC_HT + 1, LVL(1));
  bool damped = false;
  if (lane < i1 - i0 + SRC_HT + SRC_HB) {
    const int i = i0 - SRC_HT + lane, ic = min(max(i, 0), nr - 1), il = max(ic - 1, 0);
    const double *rings = global(t.rings), *vrefs = global(a.vref);
    double r[RG_NU];
#pragma unroll
    for (int x = 0; x < RG_NU; x++) r[x] = rings[(long)ic * RG_NU + x];
    const double v = global(a.nu)[ic], imed_l = rings[(long)il * RG_NU + RG_IMED];
    // the reference velocity and Sigma's background are 0 outside the disk
    const double vref = i == ic ? vrefs[ic] : 0.0, vref_l = vrefs[il];
    const double sbar = i == ic ? global(a.sbar)[ic] : 0.0;
    damped = a.evanescent && i == ic && global(t.ev_zone)[ic];
    tab[lane][S3_MED] = r[RG_MED];
    tab[lane][S3_CS] = r[RG_CS];
    tab[lane][S3_VB] = 0.5 * (vref + vref_l) + OF * r[RG_INF];
    tab[lane][S3_IINF] = r[RG_IINF];
    tab[lane][S3_STAR] = (imed_l - r[RG_IMED]) * r[RG_IDMED];
    tab[lane][S3_VREF] = vref;
    tab[lane][S3_SBAR] = sbar;
    ftab[lane][S3F_IDMED] = (float)r[RG_IDMED];
    ftab[lane][S3F_IDXT] = (float)r[RG_IDXT];
    ftab[lane][S3F_SUPP] = (float)r[RG_SUPP];
    ftab[lane][S3F_IMED] = (float)r[RG_IMED];
    ftab[lane][S3F_IDSUP] = (float)r[RG_IDSUP];
    ftab[lane][S3F_SUP] = (float)r[RG_SUP];
    ftab[lane][S3F_INF] = (float)r[RG_INF];
    ftab[lane][S3F_NU] = (float)v;
    ftab[lane][S3F_IINF] = (float)r[RG_IINF];
    ftab[lane][S3F_MED] = (float)r[RG_MED];
    ftab[lane][S3F_DREF] = (float)(vref * r[RG_IMED] - vref_l * imed_l);
    if (damped) {
      // (Kernels.cu:978-1004; one viscosity: the two passes damp alike)
      const double Rm = r[RG_MED], lambda = global(t.ev_coef)[ic] * dt / global(t.ev_period)[ic];
      const double vt0 = sqrt(global(t.ev_vtheta_arg)[ic]) - Rm * OF, vr0 = -3.0 * v / Rm * t.vrad0_slope;
      const recip64 d(1.0 + lambda);
      double *ev = evc[lane];
      ev[EV_D] = d.d;
      ev[EV_R] = d.r;
      ev[EV_S] = lambda * global(t.SigmaMed)[ic];
      ev[EV_VR1] = lambda * vr0;
      ev[EV_VT1] = lambda * vt0;
    }
  }
  const unsigned zones = (unsigned)__ballot(damped);  // bit r: ring i0 - SRC_HT + r is damped
  __syncthreads();
  double px = a.P.x[0], py = a.P.y[0], pm = a.P.m[0], ps = a.P.smooth[0], pi3 = a.P.invd3[0], ix = a.P.ix, iy = a.P.iy;
  asm volatile("" : "+s"(px), "+s"(py), "+s"(pm), "+s"(ps), "+s"(pi3), "+s"(ix), "+s"(iy));
  const bool star = nb > 0;  // the star's -1/r enters with the first planet
  const float invdphi = (float)t.invdphi, onethird = 1.0f / 3.0f;
  // windows as in k_src (T: vtheta - vref); IR, IT: the velocity increments;
  // Ds, Dvr, Dvt: the state in FP64 after the first damping pass
  double Ds[3] = {}, Dvr[3] = {}, Dvt[3] = {};
  float S[3] = {}, Sl[3] = {}, P[3] = {}, F[3] = {}, T[3] = {}, Tn[3] = {};
  float A1[3] = {}, B1[3] = {}, A3[3] = {}, RR[3] = {}, PP[3] = {}, RP[3] = {}, QR[3] = {}, IR[3] = {}, IT[3] = {};
  float hr[3] = {}, ha[3] = {};  // reciprocals of Sigma_i + Sigma_i-1, Sigma_j + Sigma_j-1
  auto step = [&](int m, auto level, auto phase, auto inner) __attribute__((always_inline)) {
    constexpr int LV = decltype(level)::value, C = decltype(phase)::value, M1 = (C + 2) % 3, M2 = (C + 1) % 3;
    constexpr bool IN = decltype(inner)::value;
    double s = n_s[C], vr = n_vr[C], vt = n_vt[C];
    fetch(m + AHEAD, LVL(C + AHEAD));
    asm volatile("" : "+v"(jb), "+v"(jf));
    const int row = m - i0 + SRC_HT;  // rings m, k, o in the tables
    const double *Dm = tab[row], *Do = tab[max(row - 2, 0)];
    const float *Rm = ftab[row], *Rk = ftab[max(row - 1, 0)], *Ro = ftab[max(row - 2, 0)];
    const int k = m - 1, o = m - 2;
    // ---- S0: CorrectVtheta, damping #1 (FP64), pressure, potential of ring m ----
    float fs = 0.f, fvr = 0.f, fvt = 0.f, p = 0.f, phi = 0.f;
    if (IN || (m >= 0 && m < nr)) {
      vt = vt - domega * Dm[S3_MED];
      if (zones >> row & 1) {
        const double *ev = evc[row];
        vr = ev_damp(vr, ev, EV_VR1);
        vt = ev_damp(vt, ev, EV_VT1);
        s = ev_damp(s, ev, EV_S);
      }
      const double cs = Dm[S3_CS], pd = s * cs * cs;
      p = (float)pd;
      if (opress && mine && m >= i0 && m < i1) at(opress + (long)m * ns, jb) = pd;  // for the temperature output
      const double x = Dm[S3_MED] * cosp, y = Dm[S3_MED] * sinp;
      if (nb > 0) {
        phi = 0.0f + planet_potential_f(x, y, px, py, pm, ps, pi3, indirect);
        phi -= (float)(ix * x + iy * y);
      }
      for (int q = 1; q < nb; q++)
        phi += planet_potential_f(x, y, more.x[q], more.y[q], more.m[q], more.smooth[q], more.invd3[q], indirect);
      fs = (float)s;
      fvr = (float)vr;
      fvt = (float)(vt - Dm[S3_VREF]);
    } else if (m == nr) {
      fs = (float)s;
      fvr = (float)vr;
      fvt = (float)vt;
    }
    Ds[C] = s;
    Dvr[C] = vr;
    Dvt[C] = vt;
    S[C] = fs;
    P[C] = p;
    F[C] = phi;
    T[C] = fvt;
    Tn[C] = lane_next(fvt);
    Sl[C] = lane_prev(fs);
    // ---- S1: Substep1 (Kernels.cu:13-53) of ring m ----
    if constexpr (LV >= 1) {
      float vri = 0.f, vti = 0.f, dvr = 0.f, dvt = 0.f;
      if (IN || (m >= 0 && m < nr)) {
        if (IN || m > 0) {
          const float idr = Rm[S3F_IDMED];
          hr[C] = rcp_f(fs + S[M1]);
          const float gradp = (p - P[M1]) * 2.0f * hr[C] * idr;
          const float gradphi = (phi - F[M1]) * idr;
          // centrifugal minus star gravity in FP64: vbar = ring part + offset
          double vbar = Dm[S3_VB];
          vbar += (double)((T[C] + Tn[C] + T[M1] + Tn[M1]) * 0.25f);
          double bal = vbar * vbar * Dm[S3_IINF];
          if (star) bal -= Dm[S3_STAR];
          dvr = dtf * (-gradp - gradphi + (float)bal);
          vri = fvr + dvr;
        }
        const float invdxtheta = Rm[S3F_IDXT];
        ha[C] = rcp_f(fs + Sl[C]);
        const float gradp = (p - lane_prev(p)) * 2.0f * ha[C] * invdxtheta;
        const float gradphi = (phi - lane_prev(phi)) * invdxtheta;
        dvt = dtf * (Rm[S3F_SUPP] - (gradp + gradphi));
        vti = fvt + dvt;
      }
      A1[C] = vri;
      B1[C] = vti;
      IR[C] = dvr;
      IT[C] = dvt;
    }
    // ---- S2: viscous stress (Kernels.cu:733-771) of ring k ----
    if constexpr (LV >= 2) {
      if (IN || (k >= 0 && k < nr)) {
        const float iRm = Rk[S3F_IMED], idRs = Rk[S3F_IDSUP], v = Rk[S3F_NU];
        const float vr0 = A1[M1], vr1 = A1[C], b = B1[M1];
        const float dv_t = lane_next(b) - b;
        const float drr = (vr1 - vr0) * idRs;
        const float dpp = dv_t * invdphi * iRm + 0.5f * (vr1 + vr0) * iRm;
        float dv = (vr1 * Rk[S3F_SUP] - vr0 * Rk[S3F_INF]) * idRs * iRm;
        dv += dv_t * invdphi * iRm;
        const float nu2s = 2.0f * S[M1] * v;
        RR[M1] = nu2s * (drr - onethird * dv);
        PP[M1] = nu2s * (dpp - onethird * dv);
        if (LV >= 3 && (IN || k > 0)) {
          // d(vtheta/r)/dr with the reference part of vtheta differenced in FP64
          const float dom = Rk[S3F_DREF] + (b * iRm - B1[M2] * Ro[S3F_IMED]);
          const float drp = 0.5f * (Rk[S3F_INF] * dom * Rk[S3F_IDMED] +
                                    (vr0 - lane_prev(vr0)) * invdphi * Rk[S3F_IINF]);
          RP[M1] = 0.5f * (S[M1] + S[M2] + Sl[M1] + Sl[M2]) * v * drp;
        }
      }
    }
    // ---- S3: viscous velocity update (Kernels.cu:118-150): VradInt of ring k ----
    if constexpr (LV >= 3) {
      A3[M1] = A1[M1];
      if (IN || (k >= 1 && k < nr)) {
        const float d = dtf * Rk[S3F_IINF] *
                        ((Rk[S3F_MED] * RR[M1] - Ro[S3F_MED] * RR[M2]) * Rk[S3F_IDMED] +
                         (lane_next(RP[M1]) - RP[M1]) * invdphi - 0.5f * (PP[M1] + PP[M2])) *
                        rcp_f(0.5f * (S[M1] + S[M2]));
        A3[M1] += d;
        IR[M1] += d;
      }
    }
    // ---- S4: radial artificial pressure (Kernels.cu:409-434) of ring o ----
    if constexpr (LV >= 4) QR[M2] = (IN || (o >= 0 && o < nr)) ? art_visc_q_f(S[M2], A3[M1] - A3[M2]) : 0.f;
    // ---- ring o: the rest of S3 and S4, S5 ("kernel", Kernels.cu:438-479), damping #2, store ----
    if constexpr (LV >= 5) {
      const long l = (long)o * ns;
      if (!IN && o == nr) {  // ghost ring (never read)
        if (mine) {
          at(odens + l, jf) = 0.0f;
          at(ovr + l, jf) = 0.0f;
          at(ovt + l, jf) = 0.0f;
        }
        return;
      }
      float b = B1[M2], it = IT[M2];
      if (IN || (o >= 1 && o < nr - 1)) {
        const float d = dtf * Ro[S3F_IMED] *
                        ((Ro[S3F_SUP] * RP[M1] - Ro[S3F_INF] * RP[M2]) * Ro[S3F_IDSUP] +
                         (PP[M2] - lane_prev(PP[M2])) * invdphi + 0.5f * (RP[M2] + RP[M1])) *
                        rcp_f(0.5f * (S[M2] + Sl[M2]));
        b += d;
        it += d;
      }
      const float qt = art_visc_q_f(S[M2], lane_next(b) - b);
      double s2 = Ds[M2], vrnew = 0.0;
      if (IN || o > 0) {
        const float dq = (QR[M2] - QR[C]) * 2.0f * hr[M2] * Ro[S3F_IDMED];  // (slot C: ring o - 1)
        vrnew = Dvr[M2] + (double)(IR[M2] - dtf * dq);
      }
      const float dq = (qt - lane_prev(qt)) * 2.0f * ha[M2] * Ro[S3F_IDXT];
      double vtnew = Dvt[M2] + (double)(it - dtf * dq);
      if (zones >> (row - 2) & 1) {
        const double *ev = evc[row - 2];
        vrnew = ev_damp(vrnew, ev, EV_VR1);
        vtnew = ev_damp(vtnew, ev, EV_VT1);
        s2 = ev_damp(s2, ev, EV_S);
      }
      if (mine) {
        const double xs = s2 - Do[S3_SBAR];
        const float hs = (float)xs;
        at(odens + l, jf) = hs;
        at(ovr + l, jf) = (float)vrnew;
        at(ovt + l, jf) = (float)(vtnew - Do[S3_VREF]);
        if (in_lob(o, lob0, lob1))  // Sigma as a float pair near the planets
          at(odens + (long)(nr + 1) * ns + l, jf) = (float)(xs - (double)hs);
      }
    }
  };
  auto march = [&](auto inner) __attribute__((always_inline)) {
    const int m0 = i0 - SRC_HT;  // (as k_src)
    step(m0, LVL(0), LVL(0), inner);
    step(m0 + 1, LVL(1), LVL(1), inner);
    step(m0 + 2, LVL(2), LVL(2), inner);
    step(m0 + 3, LVL(3), LVL(0), inner);
    step(m0 + 4, LVL(4), LVL(1), inner);
    int m = m0 + 5;
    for (; m + 2 <= i1 + 1; m += 3) {
      step(m, LVL(5), LVL(2), inner);
      step(m + 1, LVL(5), LVL(0), inner);
      step(m + 2, LVL(5), LVL(1), inner);
    }
    if (m <= i1 + 1) step(m, LVL(5), LVL(2), inner);
    if (m + 1 <= i1 + 1) step(m + 1, LVL(5), LVL(0), inner);
  };
#undef LVL
  if (i0 - SRC_HT >= 1 && i1 + SRC_HB <= nr)
    march(std::true_type());
  else
    march(std::false_type());
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(SRC32_WAVES))) void k_src32(src32_args a) {
  __shared__ src32_lds lds;
  const int block = xcd_block(a.nstrips * ((a.nr + a.band) / a.band));
  if (block < 0) return;
  const auto &more = ((__attribute__((address_space(4))) const src32_args *)__builtin_amdgcn_kernarg_segment_ptr())->P;
  src32_march(a, more, block, lds);
}

// Radial sweep in FP32 (k_trad above): Q of each ring is formed in FP64,
// its Work value, slopes, face values and fluxes in FP32; the flux
// divergence is added to the FP64 Q.
// block index blk < NRAD: ring mean of that ring; otherwise one column
// strip of one band of a.band rings
__device__ __forceinline__ void trad32_block(const trad_args &a, int blk) {
  const int nr = a.nr, ns = a.ns;
  if (blk < nr) {
    ring_mean_wave32(a.fvt + (long)blk * ns, a.vref[blk], ns, a.vmed + blk);
    return;
  }
  const int bid = blk - nr;
  // lanes past the last sector: as in k_trad
  const int j = min((bid % a.nstrips) * TRAD_TPB + (int)threadIdx.x, ns - 1);
  const int jp = (j + 1) % ns;
  const int b0 = (bid / a.nstrips) * a.band;
  const int b1 = min(b0 + a.band, nr);
  const fg_dev_tables &t = a.t;
  const double dt = a.dt, OF = a.omega_frame;
  const float dtf = (float)dt;
  const float cflux = (float)(dt * t.dtheta);
  double Q[NQ][3] = {};
  float W[NQ][3] = {}, dq[NQ][2] = {}, F[NQ][2] = {};
  float sg[3] = {}, dqs[2] = {}, vr[3] = {};
  const int m0 = max(b0 - 2, 0);
  ring_lanes rt;
  rt.load(t, m0 - 2, nr);
  bg_lanes bg;
  bg.load(a.sbar, a.vref, rt.r0, nr);
  // Every iteration issues the same memory operations, so that the
  // compiler's wait counts are exact: ring m + 2's inputs are loaded two
  // iterations ahead (the Sigma residual too, from the ghost ring's zero
  // slots outside the float-pair band), and ring m - 2's outputs are
  // stored (the iterations before the strip's first stored ring, and the
  // residuals outside the band, write the never-read ghost-ring slots of
  // the output arrays).  A sweep has one wave per column strip and fewer
  // strips than SIMDs, so only its own prefetch hides memory latency; the
  // three register sets P0..P2 take turns (ring m in one, ring m + 2
  // loaded into the one ring m - 1 left) in a loop unrolled by three, so
  // no register has to be renamed while its load is in flight (each set
  // loads its own ring's vrad as v0, a cache hit: the previous ring loaded
  // it as its v1).
  const long S = (long)(nr + 1) * ns, ghost = (long)nr * ns;
  auto lo_at = [&](int ring, long l) { return in_lob(ring, a.lob0, a.lob1) ? S + l : S + ghost + (l - (long)ring * ns); };
  struct pset {
    float s, v0, v1, vtp, vt, sl;
  };
  auto load = [&](pset &p, int mr) {
    const int mp = min(mr, nr - 1);
    const long l = (long)mp * ns;
    p.s = a.fdens[l + j];
    p.v0 = a.fvr[l + j];
    p.v1 = a.fvr[l + ns + j];
    p.vtp = a.fvt[l + jp];
    p.vt = a.fvt[l + j];
    p.sl = a.fdens[lo_at(mp, l + j)];
  };
  pset P0, P1, P2;
  load(P0, m0);
  load(P1, m0 + 1);
  asm volatile("" ::"v"(P0.s), "v"(P0.v0), "v"(P0.v1), "v"(P0.vtp), "v"(P0.vt), "v"(P0.sl));
  asm volatile("" ::"v"(P1.s), "v"(P1.v0), "v"(P1.v1), "v"(P1.vtp), "v"(P1.vt), "v"(P1.sl));
  auto ring = [&](int m, pset &cur, pset &next2) {
    const int r = rt.at(t, m, nr);
    if (bg.r0 != rt.r0) bg.load(a.sbar, a.vref, rt.r0, nr);
    const float c_s = cur.s, c_v0 = cur.v0, c_v1 = cur.v1, c_vtp = cur.vtp, c_vt = cur.vt;
    const float c_sl = cur.sl;  // 0 outside the band
    load(next2, m + 2);
    for (int q = 0; q < NQ; q++) {
      Q[q][0] = Q[q][1];
      Q[q][1] = Q[q][2];
      W[q][0] = W[q][1];
      W[q][1] = W[q][2];
    }
    sg[0] = sg[1];
    sg[1] = sg[2];
    vr[0] = vr[1];
    vr[1] = vr[2];
    const double Rm = lane_get(rt.Rmed, r);
    if (m < nr) {
      const double vb = lane_get(bg.vb, r);
      const double s = rec32(lane_get(bg.sb, r), c_s, c_sl);
      const double v0 = (double)c_v0, v1 = (double)c_v1;
      Q[0][2] = s * v1;
      Q[1][2] = s * v0;
      Q[2][2] = s * ((vb + (double)c_vtp) + Rm * OF) * Rm;
      Q[3][2] = s * ((vb + (double)c_vt) + Rm * OF) * Rm;
      Q[4][2] = s;
      const float fs = (float)s;
      const float rs = rcp_f(fs + 1e-20f);
      for (int q = 0; q < NQ; q++) W[q][2] = (float)Q[q][2] * rs;
      sg[2] = fs;
      vr[2] = c_v0;
    } else {
      for (int q = 0; q < NQ; q++) {
        Q[q][2] = 0.0;
        W[q][2] = 0.0f;
      }
      sg[2] = 0.0f;
      vr[2] = 0.0f;
    }
    // (k = -1, the first step of the first strip: its slopes and fluxes are
    // of zero quantities and feed no stored ring)
    const int k = m - 1;
    const bool flat = (k == 0 || k >= nr - 1);
    const float idm0 = flat ? 0.f : (float)lane_get(rt.idm, r - 1), idm1 = flat ? 0.f : (float)lane_get(rt.idm, r);
    for (int q = 0; q < NQ; q++) {
      dq[q][0] = dq[q][1];
      dq[q][1] = flat ? 0.0f : vl_rad_slope_f(W[q][0], W[q][1], W[q][2], idm0, idm1);
    }
    dqs[0] = dqs[1];
    dqs[1] = flat ? 0.0f : vl_rad_slope_f(sg[0], sg[1], sg[2], idm0, idm1);
    float DS = 0.0f, QS[NQ];
    if (k > 0 && k < nr) {
      const float vk = vr[1];
      const double Rk = lane_get(rt.Rmed, r - 1);
      const float dm = (float)(Rk - lane_get(rt.Rmed, r - 2)), dp = (float)(Rm - Rk);
      DS = vl_rad_star_f(vk, dtf, sg[0], sg[1], dqs[0], dqs[1], dm, dp);
      for (int q = 0; q < NQ; q++) QS[q] = vl_rad_star_f(vk, dtf, W[q][0], W[q][1], dq[q][0], dq[q][1], dm, dp);
    } else {
      for (int q = 0; q < NQ; q++) QS[q] = 0.0f;
    }
    const float vface = (k < nr) ? vr[1] : 0.0f;
    const float cf = cflux * (float)lane_get(rt.Rinf, r - 1) * DS * vface;
    for (int q = 0; q < NQ; q++) {
      F[q][0] = F[q][1];
      F[q][1] = cf * QS[q];
    }
    {
      // ring o = k - 1 is complete: stored as FP32 offsets from its
      // backgrounds if the strip stores it (o in [b0, b1)), else into the
      // ghost ring's slots, which nothing reads
      const int o = k - 1;
      const long lo_ = (o >= b0 ? (long)o * ns : ghost) + j;
      const float isurf = (float)lane_get(rt.isurf, r - 2);
      const double sb = lane_get(bg.sb, r - 2);
      double val[NQ];
      for (int q = 0; q < NQ; q++) val[q] = Q[q][0] + (double)((F[q][0] - F[q][1]) * isurf);
      // Sigma as the reader will reconstruct it, the angular momenta's background
      const double xs = val[4] - sb;
      const float fs = (float)xs, fsl = (float)(xs - (double)fs);
      const bool pair = in_lob(o, a.lob0, a.lob1);
      const float fsr = pair ? fsl : 0.f;
      const double lb = fp32_bg_angmom(rec32(sb, fs, fsr), lane_get(bg.vb, r - 2), lane_get(rt.Rmed, r - 2), OF);
      a.fout[0][lo_] = (float)val[0];
      a.fout[1][lo_] = (float)val[1];
      a.fout[2][lo_] = (float)(val[2] - lb);
      a.fout[3][lo_] = (float)(val[3] - lb);
      a.fout[4][lo_] = fs;
      // the residual of a float-pair ring (k_taz reads it inside the band only)
      a.fout[4][S + (pair && o >= b0 ? lo_ : ghost + j)] = fsl;
    }
  };
  int m = m0;
  const int end = b1 + 2;  // steps m0 .. b1 + 1 store rings b0 .. b1 - 1
  for (; m + 2 < end; m += 3) {
    ring(m, P0, P2);
    ring(m + 1, P1, P0);
    ring(m + 2, P2, P1);
  }
  if (m < end) ring(m++, P0, P2);
  if (m < end) ring(m++, P1, P0);
}

__global__ __launch_bounds__(TRAD_TPB) void k_trad32(trad_args a) { trad32_block(a, blockIdx.x); }

// ----------------------------------------------------- entry points ----
#define PROF_KERNELS 6

static void prof_mark(fg_ctx *c) {
  if (c->prof_on && c->prof_nev < 16) (void)hipEventRecord(c->prof_ev[c->prof_nev++], c->stream);
}

// fold a completed substep's events into the totals (stream is idle)
static void prof_fold(fg_ctx *c) {
  if (!c->prof_on || !c->prof_pending) return;
  for (int k = 0; k + 1 < c->prof_nev && k < PROF_KERNELS; k++) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, c->prof_ev[k], c->prof_ev[k + 1]) == hipSuccess) {
      c->prof_ms[k] += ms;
      c->prof_calls[k]++;
    }
  }
  c->prof_pending = 0;
  c->prof_nev = 0;
}

extern "C" fg_status fg_profile(fg_ctx *c, int enable) {
  if (!c) return FG_E_INVALID;
  FG_HIP(hipStreamSynchronize(c->stream));
  if (enable && !c->prof_ev[0])
    for (int k = 0; k < 16; k++) FG_HIP(hipEventCreate(&c->prof_ev[k]));
  for (int k = 0; k < 16; k++) {
    c->prof_ms[k] = 0.0;
    c->prof_calls[k] = 0;
  }
  c->prof_nev = 0;
  c->prof_pending = 0;
  c->prof_on = enable;
  return FG_OK;
}

extern "C" int fg_profile_read(fg_ctx *c, double *ms, long *calls, int max) {
  if (!c) return 0;
  (void)hipStreamSynchronize(c->stream);
  prof_fold(c);
  int n = max < PROF_KERNELS ? max : PROF_KERNELS;
  for (int k = 0; k < n; k++) {
    if (ms) ms[k] = c->prof_ms[k];
    if (calls) calls[k] = c->prof_calls[k];
  }
  return n;
}
// The fused path's buffers are published together, only once every
// allocation succeeded (a failed attempt frees what it got and a later call
// starts again).
// arrays in the fused pool: B (3), R (5), X (4), pressure, spare; adiabatic
// or self-gravity decks add EnergyInt, two energies and the two kicks
static int fused_pool_arrays(const fg_ctx *c) { return (c->p.adiabatic || c->p.self_gravity) ? 19 : 14; }

static fg_status fused_alloc(fg_ctx *c) {
  if (c->fu_ring) return FG_OK;
  const size_t S = (size_t)c->S;
  // per-ring star-force partials (4 per ring) and the two Sigma backgrounds
  // of the FP32 storage
  const size_t fpart_bytes = 6 * (size_t)(c->nr + 1) * sizeof(double);
  const size_t pool_bytes = (size_t)fused_pool_arrays(c) * S * sizeof(double);
  double *pool = nullptr, *fpart = nullptr, *h = nullptr, *d = nullptr;
  hipError_t e = hipMalloc((void **)&pool, pool_bytes);
  if (e == hipSuccess) e = hipMemset(pool, 0, pool_bytes);
  if (e == hipSuccess) e = hipMalloc((void **)&fpart, fpart_bytes);
  if (e == hipSuccess) e = hipMemset(fpart, 0, fpart_bytes);
  if (e == hipSuccess)
    e = hipHostMalloc((void **)&h, FG_FUSED_SLOTS * sizeof(double), hipHostMallocCoherent | hipHostMallocMapped);
  if (e == hipSuccess) {
    memset(h, 0, FG_FUSED_SLOTS * sizeof(double));
    e = hipHostGetDevicePointer((void **)&d, h, 0);
  }
  if (e != hipSuccess) {
    if (pool) (void)hipFree(pool);
    if (fpart) (void)hipFree(fpart);
    if (h) (void)hipHostFree(h);
    fg_set_error("fused path buffers: %s", hipGetErrorString(e));
    return e == hipErrorOutOfMemory ? FG_E_NOMEM : FG_E_HIP;
  }
  c->fu_fpart = fpart;
  c->fu_sbar[0] = fpart + 4 * (size_t)(c->nr + 1);
  c->fu_sbar[1] = c->fu_sbar[0] + (c->nr + 1);
  c->fu_sbar_cur = 0;
  c->h_fused = h;
  c->d_fused = d;
  c->fu_ring = pool;
  return FG_OK;
}

static fused_bufs bufs_of(fg_ctx *c) {
  const size_t S = (size_t)c->S;
  double *p = c->fu_ring;
  fused_bufs b;
  b.Bd = p + 0 * S;
  b.Bvr = p + 1 * S;
  b.Bvt = p + 2 * S;
  b.Rd = p + 3 * S;
  b.Rrmp = p + 4 * S;
  b.Rrmm = p + 5 * S;
  b.Rtmp = p + 6 * S;
  b.Rtmm = p + 7 * S;
  b.Xd = p + 8 * S;
  b.Xvt = p + 9 * S;
  b.Xrmp = p + 10 * S;
  b.Xrmm = p + 11 * S;
  b.P = p + 12 * S;
  const bool more = fused_pool_arrays(c) > 14;
  b.Beint = more ? p + 14 * S : nullptr;
  b.Re = more ? p + 15 * S : nullptr;
  b.Xe = more ? p + 16 * S : nullptr;
  b.kick_r = more ? p + 17 * S : nullptr;
  b.kick_t = more ? p + 18 * S : nullptr;
  return b;
}

static fg_status fused_supported(fg_ctx *c) {
  const fg_params &p = c->p;
  if (p.open_inner || p.non_reflecting || !p.evanescent) {
    fg_set_error("fused path: deck needs the per-routine path (open or non-reflecting edges)");
    return FG_E_UNSUPPORTED;
  }
  if ((p.adiabatic || p.self_gravity) && p.precision == FG_PREC_FP32) {
    fg_set_error("fused path: the FP32 bulk mode takes locally isothermal decks without self-gravity");
    return FG_E_UNSUPPORTED;
  }
  if (p.adiabatic && c->nr < 3) {
    fg_set_error("fused path: an adiabatic deck needs NRAD >= 3");
    return FG_E_UNSUPPORTED;
  }
  if (c->ns > 4096) {
    fg_set_error("fused path: NSEC %d > 4096", c->ns);
    return FG_E_UNSUPPORTED;
  }
  return FG_OK;
}

// DeviceReduce of the disk force on several points at once (dreduce_block):
// blockIdx.y takes point y, whose block sums go to its part of `partial`.  The
// star, if it is among them, is point 0.
struct forces_args {
  force_src src;  // (position and smoothing of the star)
  long n;
  int B, star;
  double *partial;
  fg_force_list list;
};
__global__ __launch_bounds__(RED_TPB) void k_forces_partial(forces_args a) {
  force_src src = a.src;
  const int q = (int)blockIdx.y - a.star;
  if (q >= 0) {  // (read where the launch put them: indexed, a by-value copy would live in scratch)
    const auto &list = ((__attribute__((address_space(4))) const forces_args *)__builtin_amdgcn_kernarg_segment_ptr())->list;
    src.x = list.x[q];
    src.y = list.y[q];
    src.rs = list.rs[q];
  }
  dreduce_block<force_src, RED_CH>(src, a.n, a.B, blockIdx.x, a.partial + 2l * FG_RED_BLOCKS * blockIdx.y);
}

// Their final sums, the host loop of DeviceReduce (dreduce_final: lanes 0 and 1
// add the B block sums of x and y in order, then +0.0 for the inner sum,
// SideEuler.cu:144), one workgroup a point, and beside the star's, in waves 1-3
// of workgroup 0, the CFL count of the same state (DT1D of every ring,
// Kernels.cu:1331-1337, and the minimum with the ring minima,
// Kernels.cu:1337-1359; a minimum does not depend on the order its candidates
// are compared in); then the result block's sequence slots.  RINGS: the star's
// force from k_fin's ring partials (FP32 mode).
// Bound: latency, the chain of B = 1024 additions and the write to host memory:
// 11 us however many planets there are, where two planets' own pairs of
// launches took 36 (301 x 998 with two planets: 135 us per substep before it, 104
// with it).
struct results_args {
  const double *partial;
  int B, star;
  double *out;     // result block
  double *cfl;     // CFL count, as a double or an int (neither: not wanted)
  int *icfl;
  double *dt1d;
  const double *vmoy, *newdt, *invRmed, *fpart;
  double coef, DeltaT;
  int nr;
  double seq;      // > 0: into the sequence slots
  fg_force_list list;
};
template <bool RINGS>
__global__ __launch_bounds__(256) void k_results(results_args a) {
  __shared__ double p[2 * FG_RED_BLOCKS];
  __shared__ double wmin[4];
  const int tid = threadIdx.x, q = (int)blockIdx.x - 1, B = a.B;
  if (RINGS && q < 0) {
    force_rings_cfl(a.fpart, a.nr, a.out, a.cfl, a.dt1d, a.vmoy, a.newdt, a.invRmed, a.coef, a.DeltaT);
    seq_store(a.out + FG_FUSED_SEQ_SLOT, a.seq);
    return;
  }
  const double *partial = a.partial + 2l * FG_RED_BLOCKS * (q + a.star);
  for (int k = tid; k < 2 * B; k += 256) p[k] = partial[k];
  __syncthreads();
  int slot = 0;
  if (q >= 0)
    slot = ((__attribute__((address_space(4))) const results_args *)__builtin_amdgcn_kernarg_segment_ptr())->list.slot[q];
  if (tid < 2) {
    double s = seq_sum_lds(p + tid * B, B);
    a.out[slot + tid] = 0.0 + s;
  } else if (tid >= 64 && q < 0 && (a.cfl || a.icfl)) {
    double best = cfl_ring_min(a.dt1d, a.vmoy, a.newdt, a.invRmed, a.coef, a.nr, tid - 64, 192);
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_down(best, off, 64);
      if (o < best) best = o;
    }
    if ((tid & 63) == 0) wmin[tid >> 6] = best;
  }
  __syncthreads();
  if (tid == 0 && q < 0 && (a.cfl || a.icfl)) {
    double newdt_ = wmin[1];
    if (wmin[2] < newdt_) newdt_ = wmin[2];
    if (wmin[3] < newdt_) newdt_ = wmin[3];
    if (a.DeltaT < newdt_) newdt_ = a.DeltaT;
    const int count = (int)(ceil(a.DeltaT / newdt_));
    if (a.cfl)
      a.cfl[0] = (double)count;
    else
      a.icfl[0] = count;
  }
  if (a.seq > 0.0) seq_store(a.out + (q < 0 ? FG_FUSED_SEQ_SLOT : FG_FUSED_PFSEQ_SLOT + q), a.seq);
}

// the block sums of the star, unless its ring partials serve, and of the points
// of c->pf, which are no longer pending then
static fg_status forces_partial(fg_ctx *c, bool star, results_args &r) {
  const long n = (long)c->nr * c->ns;
  const int B = red_blocks(n), points = (star ? 1 : 0) + c->pf.n;
  r.partial = c->red_partial;
  r.B = B;
  r.star = star;
  r.list = c->pf;
  r.dt1d = c->DT1D;
  r.vmoy = c->Vmoy;
  r.newdt = c->newDT;
  r.invRmed = c->t.invRmed;
  r.fpart = c->fu_fpart;
  r.coef = c->t.dt1d_coef;
  r.nr = c->nr;
  if (points > 0) {
    forces_args a;
    a.src = force_src{c->f[FG_DENS], c->t.Surf, c->t.Rmed, c->t.cos_cell, c->t.sin_cell, 0.0, 0.0, 0.0, c->ns};
    a.n = n;
    a.B = B;
    a.star = star;
    a.partial = c->red_partial;
    a.list = c->pf;
    hipLaunchKernelGGL(k_forces_partial, dim3(B, points), dim3(RED_TPB), 0, c->stream, a);
    FG_LAUNCH_CHECK();
  }
  c->pf.n = 0;
  return FG_OK;
}

static void set_forces(fg_force_list &f, int n, const int *k, const double *x, const double *y, const double *rs,
                       int slot0) {
  f.n = n;
  for (int q = 0; q < n; q++) {
    f.x[q] = x[q];
    f.y[q] = y[q];
    f.rs[q] = rs[q];
    f.slot[q] = slot0 + 2 * k[q];
  }
}

void fg_fused_planet_forces(fg_ctx *c, int n, const int *k, const double *x, const double *y, const double *rs) {
  set_forces(c->pf, n, k, x, y, rs, FG_FUSED_PF_SLOT);
}

fg_status fg_routine_results(fg_ctx *c, bool cfl, double DeltaT, int n, const int *k, const double *x, const double *y,
                             const double *rs) {
  if (cfl)
    if (fg_status s = fg_cfl_ring_launch(c)) return s;
  set_forces(c->pf, n, k, x, y, rs, FG_OUT_PF);
  results_args r;
  if (fg_status s = forces_partial(c, true, r)) return s;
  r.out = c->red_out;
  r.cfl = nullptr;
  r.icfl = cfl ? c->cfl_out : nullptr;
  r.DeltaT = DeltaT;
  r.seq = 0.0;
  hipLaunchKernelGGL(k_results<false>, dim3(1 + n), dim3(256), 0, c->stream, r);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

// results of the reductions for the next substep: CFL count and the disk
// force on the star and on the planets of c->pf.
// ring_partials: the star force comes from k_fin's per-ring compensated
// partials (FP32 mode) instead of the DeviceReduce-order sum
static fg_status fused_reductions(fg_ctx *c, double DeltaT, bool ring_partials = false) {
  results_args r;
  const int n = c->pf.n;
  if (fg_status s = forces_partial(c, !ring_partials, r)) return s;
  prof_mark(c);
  r.out = c->d_fused;
  r.cfl = c->d_fused + FG_FUSED_CFL_SLOT;
  r.icfl = nullptr;
  r.DeltaT = DeltaT;
  r.seq = (double)++c->fu_seq;
  c->fu_waits = n;
  hipLaunchKernelGGL(ring_partials ? k_results<true> : k_results<false>, dim3(1 + n), dim3(256), 0, c->stream, r);
  FG_LAUNCH_CHECK();
  prof_mark(c);
  return FG_OK;
}

// CFL ring pass over the current state (first substep, or after the
// per-routine path touched the state)
__global__ void k_cfl_ring(double *vmoy, double *newdt, const double *vr, const double *vt, const double *cs,
                           const double *dens, const double *energy, int *crash, fg_dev_tables t, int nr, int ns,
                           int fast);

// ring means of a field (any summation order: the FP32 storage's Sigma
// background of the first substep after a state was set)
__global__ __launch_bounds__(256) void k_ring_bg(double *out, const double *f, int ns) {
  __shared__ double w[4];
  const int i = blockIdx.x;
  double s = 0.0;
  for (int j = threadIdx.x; j < ns; j += 256) s += f[(long)i * ns + j];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[i] = (w[0] + w[1] + w[2] + w[3]) / (double)ns;
}

extern "C" fg_status fg_fused_prepare(fg_ctx *c, double DeltaT) {
  if (!c) return FG_E_INVALID;
  if (fg_status s = fused_supported(c)) return s;
  if (fg_status s = fused_alloc(c)) return s;
  if (c->p.precision == FG_PREC_FP32) {
    hipLaunchKernelGGL(k_ring_bg, dim3(c->nr), dim3(256), 0, c->stream, c->fu_sbar[c->fu_sbar_cur],
                       (const double *)c->f[FG_DENS], c->ns);
    FG_LAUNCH_CHECK();
  }
  size_t shm = (size_t)(c->ns + 256) * sizeof(double);
  hipLaunchKernelGGL(k_cfl_ring, dim3(c->nr), dim3(256), shm, c->stream, c->Vmoy, c->newDT, c->f[FG_VRAD],
                     c->f[FG_VTHETA], c->f[FG_SOUNDSPEED], c->f[FG_DENS],
                     c->p.adiabatic ? (const double *)c->f[FG_ENERGY] : (const double *)nullptr,
                     (int *)(c->d_fused + FG_FUSED_CRASH_SLOT), c->t, c->nr, c->ns, c->p.fast_transport);
  FG_LAUNCH_CHECK();
  return fused_reductions(c, DeltaT);
}

// Results of the last fused reductions, checked: FG_E_CRASH when a pass
// flagged a negative or non-finite density, or when the CFL count or the
// force shows a time step that went to 0, infinity or NaN (the flag is
// cleared once reported; the next pass over a bad state sets it again).
fg_status fg_fused_check(fg_ctx *c, double cfl, const double *force2) {
  volatile int *flag = (volatile int *)(c->h_fused + FG_FUSED_CRASH_SLOT);
  if (*flag) {
    *flag = 0;
    fg_set_error("crash: negative or non-finite density or energy");
    return FG_E_CRASH;
  }
  return fg_check_substep_results(cfl, force2);
}

void fg_fused_planet_force(const fg_ctx *c, int k, double out2[2]) {
  out2[0] = c->h_fused[FG_FUSED_PF_SLOT + 2 * k];
  out2[1] = c->h_fused[FG_FUSED_PF_SLOT + 2 * k + 1];
}

extern "C" fg_status fg_fused_results(fg_ctx *c, int *ncfl, double *force2, double *lost) {
  if (!c) return FG_E_INVALID;
  if (!c->h_fused) {
    fg_set_error("fg_fused_results: no fused reductions were launched (fg_fused_prepare or fg_step_fused first)");
    return FG_E_INVALID;
  }
  if (c->fu_waits >= 0 && !c->prof_on) {
    // only the final kernel is awaited: watch the slots its workgroups write
    // last (quicker than the stream's completion signal), asking the stream
    // every 1024 polls so that a failed launch still ends the wait
    const double want = (double)c->fu_seq;
    for (int q = -1; q < c->fu_waits; q++) {
      volatile double *slot = c->h_fused + (q < 0 ? FG_FUSED_SEQ_SLOT : FG_FUSED_PFSEQ_SLOT + q);
      for (unsigned n = 1; *slot != want; n++) {
        if ((n & 1023) == 0) {
          const hipError_t e = hipStreamQuery(c->stream);
          if (e == hipErrorNotReady) continue;
          FG_HIP(e);
          if (*slot != want) {
            fg_set_error("fg_fused_results: the final reduction finished without reporting");
            return FG_E_HIP;
          }
          break;
        }
      }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
  } else {
    FG_HIP(hipStreamSynchronize(c->stream));
    prof_fold(c);
  }
  const double cfl = c->h_fused[FG_FUSED_CFL_SLOT];
  const double f[2] = {c->h_fused[0], c->h_fused[1]};
  if (fg_status s = fg_fused_check(c, cfl, f)) return s;
  if (ncfl) *ncfl = (int)cfl;
  if (force2) {
    force2[0] = f[0];
    force2[1] = f[1];
  }
  if (lost) *lost = 0.0;  // evanescent edges: no outflow is recorded
  return FG_OK;
}

// FP32 bulk mode: the rings stored as float pairs, [*b0, *b1): those whose
// centre lies within fp32_pair_hill Hill radii (radially, 1 by default;
// fg_set_fp32_pairs) of a planet, where the circumplanetary material stays
// and the storage rounding would add up (empty without planets or at 0)
static void fp32_pair_rings(const fg_ctx *c, const fg_planet_pot *pl, int nb, int *b0, int *b1) {
  int lo = c->nr, hi = 0;
  for (int k = 0; c->fp32_pair_hill > 0.0 && k < nb; k++) {
    const double rp = sqrt(pl[k].x * pl[k].x + pl[k].y * pl[k].y);
    if (!(pl[k].mass > 0.0) || !(rp > 0.0)) continue;
    const double w = c->fp32_pair_hill * rp * cbrt(pl[k].mass / 3.0);
    for (int i = 0; i < c->nr; i++) {
      const double r = c->h_Rmed[i];
      if (r >= rp - w && r <= rp + w) {
        lo = std::min(lo, i);
        hi = std::max(hi, i + 1);
      }
    }
  }
  if (lo >= hi) lo = hi = 0;
  *b0 = lo;
  *b1 = hi;
}

// whether every squared distance plus smoothing, its root and the planets'
// quotients by it lie well inside the exponent range (planet_potential_plain)
static int plain_potential(const fg_ctx *c, const fg_planet_pot *pl, int nb) {
  const double lo = 1e-100, hi = 1e100;
  bool ok = c->h_Rmed[0] > -hi && c->h_Rmed[c->nr - 1] < hi;
  for (int k = 0; k < nb; k++) {
    const double m = fabs(pl[k].mass);
    ok = ok && fabs(pl[k].x) < hi && fabs(pl[k].y) < hi && pl[k].smooth > lo && pl[k].smooth < hi &&
         (m == 0.0 || (m > lo && m < hi));
  }
  return ok ? 1 : 0;
}

// Rings per band of a kernel whose waves march over `rows` rings in column
// strips: the band with the least estimated time, up to `most`.  A wave
// spends about one time unit (1 us) on a step when it has its SIMD to itself
// and shares the SIMD's issue at `share` units per step and wave, and a band of
// H rings costs H + 3 steps (the first ones are partial); up to `resident` waves
// per SIMD are there at once, so the fullest SIMD counts, beyond that the total
// does.  A batch's disks share the SIMDs.
// disks: rows, strips of each of n
static int march_band(const int2 *disks, int n, int most, int resident = 3, double share = 0.7) {
  const int simds = 1024;
  double best = 0.0;
  int band = 1;
  for (int h = 1; h <= most; h++) {
    long waves = 0;
    for (int k = 0; k < n; k++) waves += (long)disks[k].y * ((disks[k].x + h - 1) / h);
    const double each = (double)waves / simds;
    const double cost = (h + 3) * std::max(1.0, share * (each > resident ? each : ceil(each)));
    if (h == 1 || cost < best) {
      best = cost;
      band = h;
    }
  }
  return band;
}
// Measured for k_src (us by events, FP64 isothermal; *: what the estimate picks):
// 128x384 1* ring 13.4, 2 rings 13.9, 8 rings 18.6; 512x1536 4 rings 27.8, 6 rings
// 25.3, 7* rings 27.1, 9 rings 26.4, 20 rings 35; 2048x4096 8 rings 127, 18 rings 112,
// 27* rings 113; 1024x3072 8 rings 57, 18-20 rings 50-52, 24 rings 55, 27* rings 62.
// There the estimate is off: 27 rings make two full rounds of waves, which it
// takes for quicker than three of 18 to 20 rings; the substep pays 4 % (261 us, 250
// with 20 rings).  Elsewhere it is within 8 % of the best band tried.
static int src_band(int nr, int nstrips) {
  const int2 disk = make_int2(nr + 1, nstrips);
  return march_band(&disk, 1, SRC_MAX_BAND);
}
// Measured for k_src32, four waves per SIMD at 1.4 us a step (us by events):
// 128x384 1* ring 12.7, 8 rings 19, 16 rings 29; 256x768 2* rings 14.8, 8
// rings 20; 512x1536 6 rings 21.9, 13 rings 27.6 (7* picked); 1024x3072 10 rings 42,
// 18* rings 43, 20 rings 40, 27 rings 51.  fg_set_tiles fixes the band instead.
static int src32_band(const int2 *disks, int n) { return march_band(disks, n, SRC_MAX_BAND, SRC32_WAVES, 0.44); }
// Measured for k_trad (us by events): 128x384 2-3 rings 11.9, 16 rings 21.5; 301x998
// (with energy) 3-6 rings 18, 16 rings 25; 512x1536 8 rings 23, 16 rings 26;
// from 1024x3072 on, where HBM bounds it, 10 to 16 rings are within 3 % and
// 20 to 32 cost 5 %; k_trad32 256x768 3-4 rings 14, 16 rings 23.5.  fg_set_tiles
// fixes the band instead.
static int trad_band(const fg_ctx *c, int nstrips) {
  const int2 disk = make_int2(c->nr, nstrips);
  return c->tile_trad_band ? c->tile_trad_band : march_band(&disk, 1, 16);
}

extern "C" fg_status fg_step_fused(fg_ctx *c, double dt, double omega_frame, double domega,
                                   const fg_planet_pot *planets, int nb, double ix, double iy,
                                   double DeltaT_next, int flags) {
  if (!c) return FG_E_INVALID;
  if (fg_status s = fused_supported(c)) return s;
  if (fg_status s = fused_alloc(c)) return s;
  if (nb < 0 || nb > FG_MAX_PLANETS || (nb > 0 && !planets)) {
    fg_set_error("fg_step_fused: planet count %d", nb);
    return FG_E_INVALID;
  }
  const int want_temperature = flags & FG_STEP_TEMPERATURE;
  const int nr = c->nr, ns = c->ns;
  const bool adi = c->p.adiabatic, sg = c->p.self_gravity;
  fused_bufs b = bufs_of(c);
  // this substep's viscosity: refreshed at the close of the last DT, it
  // replaces nu after the first damping pass
  const double *nu = c->nu_pending ? c->nu_next : c->nu;
  if (sg)
    if (fg_status s = fg_sg_fused(c, dt, b.kick_r, b.kick_t)) return s;
  // k_src
  src_args sa;
  sa.dens = c->f[FG_DENS];
  sa.vr = c->f[FG_VRAD];
  sa.vt = c->f[FG_VTHETA];
  sa.odens = b.Bd;
  sa.ovr = b.Bvr;
  sa.ovt = b.Bvt;
  sa.opress = (want_temperature && !adi) ? b.P : nullptr;
  sa.nu = nu;
  sa.nu1 = c->nu;
  sa.energy = adi ? c->f[FG_ENERGY] : nullptr;
  sa.oeint = b.Beint;
  sa.gamma = c->p.adiabatic_index;
  sa.kick_r = b.kick_r;
  sa.kick_t = b.kick_t;
  sa.sg1 = sg ? c->sgacc_prev : nullptr;
  sa.sg2 = sg ? c->sgacc_mean : nullptr;
  sa.t = c->t;
  sa.P.nb = nb;
  for (int k = 0; k < nb; k++) {
    sa.P.x[k] = planets[k].x;
    sa.P.y[k] = planets[k].y;
    sa.P.m[k] = planets[k].mass;
    sa.P.smooth[k] = planets[k].smooth;
    sa.P.invd3[k] = planets[k].inv_d3;
  }
  sa.plain = plain_potential(c, planets, nb);
  sa.P.ix = ix;
  sa.P.iy = iy;
  sa.dt = dt;
  sa.omega_frame = omega_frame;
  sa.domega = domega;
  sa.nr = nr;
  sa.ns = ns;
  sa.indirect = c->p.indirect_term;
  sa.evanescent = c->p.evanescent;
  if (c->prof_on) {
    (void)hipStreamSynchronize(c->stream);
    prof_fold(c);
    c->prof_nev = 0;
    c->prof_pending = 1;
  }
  const bool fp32 = c->p.precision == FG_PREC_FP32;
  int lob0 = 0, lob1 = 0;
  if (fp32) fp32_pair_rings(c, planets, nb, &lob0, &lob1);
  prof_mark(c);
  if (fp32) {
    src32_args s3;
    s3.lob0 = lob0;
    s3.lob1 = lob1;
    s3.dens = sa.dens;
    s3.vr = sa.vr;
    s3.vt = sa.vt;
    s3.vref = c->Vmoy;  // ring means of vtheta from the previous substep
    s3.sbar = c->fu_sbar[c->fu_sbar_cur];
    s3.odens = b.fBd();
    s3.ovr = b.fBvr();
    s3.ovt = b.fBvt();
    s3.opress = sa.opress;
    s3.nu = sa.nu;
    s3.t = sa.t;
    s3.P = sa.P;
    s3.dt = dt;
    s3.omega_frame = omega_frame;
    s3.domega = domega;
    s3.nr = nr;
    s3.ns = ns;
    s3.indirect = sa.indirect;
    s3.evanescent = sa.evanescent;
    s3.nstrips = (ns + SRC_W - 1) / SRC_W;
    s3.width = (ns + s3.nstrips - 1) / s3.nstrips;
    const int2 disk = make_int2(nr + 1, s3.nstrips);
    s3.band = c->tile_src_th ? std::min(c->tile_src_th, SRC_MAX_BAND) : src32_band(&disk, 1);
    hipLaunchKernelGGL(k_src32, dim3(xcd_grid(s3.nstrips * ((nr + s3.band) / s3.band))), dim3(64), 0, c->stream, s3);
  } else {
    sa.nstrips = (ns + SRC_W - 1) / SRC_W;
    sa.width = (ns + sa.nstrips - 1) / sa.nstrips;
    sa.band = src_band(nr, sa.nstrips);
    const dim3 gs(xcd_grid(sa.nstrips * ((nr + sa.band) / sa.band)));
    const int mode = (adi ? 1 : 0) | (sg ? 2 : 0);
    if (mode == 0)
      hipLaunchKernelGGL(k_src<0>, gs, dim3(64), 0, c->stream, sa);
    else if (mode == 1)
      hipLaunchKernelGGL(k_src<1>, gs, dim3(64), 0, c->stream, sa);
    else if (mode == 2)
      hipLaunchKernelGGL(k_src<2>, gs, dim3(64), 0, c->stream, sa);
    else
      hipLaunchKernelGGL(k_src<3>, gs, dim3(64), 0, c->stream, sa);
  }
  FG_LAUNCH_CHECK();
  if (adi) {  // Substep3 (counted with k_src by fg_profile)
    src3_args s3;
    s3.dens = b.Bd;
    s3.vr = b.Bvr;
    s3.vt = b.Bvt;
    s3.eint = b.Beint;
    s3.energy = c->f[FG_ENERGY];
    s3.nu = nu;
    s3.t = c->t;
    s3.dt = dt;
    s3.gamma = c->p.adiabatic_index;
    s3.lr01 = c->lr01;
    s3.lr12 = c->lr12;
    s3.nr = nr;
    s3.ns = ns;
    s3.cooling = c->p.cooling;
    hipLaunchKernelGGL(k_src3, dim3((ns + 63) / 64, (nr + 3) / 4), dim3(256), 0, c->stream, s3);
    FG_LAUNCH_CHECK();
  }
  // k_trad
  trad_args ta;
  ta.dens = b.Bd;
  ta.vr = b.Bvr;
  ta.vt = b.Bvt;
  ta.energy = adi ? c->f[FG_ENERGY] : nullptr;
  ta.out[0] = b.Rrmp;
  ta.out[1] = b.Rrmm;
  ta.out[2] = b.Rtmp;
  ta.out[3] = b.Rtmm;
  ta.out[4] = adi ? b.Re : b.Rd;
  ta.out[5] = b.Rd;
  ta.fdens = b.fBd();
  ta.fvr = b.fBvr();
  ta.fvt = b.fBvt();
  for (int q = 0; q < NQ; q++) ta.fout[q] = b.fR(q);
  ta.sbar = c->fu_sbar[c->fu_sbar_cur];
  ta.vref = c->Vmoy;
  ta.t = c->t;
  ta.dt = dt;
  ta.omega_frame = omega_frame;
  ta.nr = nr;
  ta.ns = ns;
  ta.vmed = c->VMed;
  ta.nstrips = (ns + TRAD_TPB - 1) / TRAD_TPB;
  ta.band = trad_band(c, ta.nstrips);
  ta.lob0 = lob0;
  ta.lob1 = lob1;
  prof_mark(c);
  const dim3 gtrad(nr + ta.nstrips * ((nr + ta.band - 1) / ta.band));
  if (fp32)
    hipLaunchKernelGGL(k_trad32, gtrad, dim3(TRAD_TPB), 0, c->stream, ta);
  else if (adi)
    hipLaunchKernelGGL(k_trad<6>, gtrad, dim3(TRAD_TPB), 0, c->stream, ta);
  else
    hipLaunchKernelGGL(k_trad<5>, gtrad, dim3(TRAD_TPB), 0, c->stream, ta);
  FG_LAUNCH_CHECK();
  // k_taz
  taz_args za;
  za.vt = b.Bvt;
  za.vmed = c->VMed;
  za.q[0] = b.Rrmp;
  za.q[1] = b.Rrmm;
  za.q[2] = b.Rtmp;
  za.q[3] = b.Rtmm;
  za.q[4] = adi ? b.Re : b.Rd;
  za.q[5] = b.Rd;
  za.xd = b.Xd;
  za.xvt = b.Xvt;
  za.xrmp = b.Xrmp;
  za.xrmm = b.Xrmm;
  za.xe = b.Xe;
  za.fvt = b.fBvt();
  for (int q = 0; q < NQ; q++) za.fq[q] = b.fR(q);
  za.fxd = b.fXd();
  za.fxvt = b.fXvt();
  za.fxrmp = b.fXrmp();
  za.fxrmm = b.fXrmm();
  za.sbar = c->fu_sbar[c->fu_sbar_cur];
  za.vref = c->Vmoy;
  za.nshift = c->Nshift;
  za.t = c->t;
  za.dt = dt;
  za.omega_frame = omega_frame;
  za.nr = nr;
  za.ns = ns;
  za.fast = c->p.fast_transport;
  za.lob0 = lob0;
  za.lob1 = lob1;
  prof_mark(c);
  {
    const int cl = tazw_cells(c);
    const dim3 gw((ns + TAZW_P(cl) - 1) / TAZW_P(cl), nr);
    auto taz = fp32 ? (cl == 2 ? k_tazw32<2> : k_tazw32<3>)
               : adi ? (cl == 2 ? k_tazw<2, 6> : k_tazw<3, 6>)
                     : (cl == 2 ? k_tazw<2, 5> : k_tazw<3, 5>);
    hipLaunchKernelGGL(taz, gw, dim3(64), 0, c->stream, za);
  }
  FG_LAUNCH_CHECK();
  // k_fin
  fin_args fa;
  fa.xd = b.Xd;
  fa.xvt = b.Xvt;
  fa.xrmp = b.Xrmp;
  fa.xrmm = b.Xrmm;
  fa.press = b.P;
  fa.dens = c->f[FG_DENS];
  fa.vr = c->f[FG_VRAD];
  fa.vt = c->f[FG_VTHETA];
  fa.temp = want_temperature ? c->f[FG_TEMPERATURE] : nullptr;
  fa.vmoy = c->Vmoy;
  fa.newdt = c->newDT;
  fa.nu = c->nu;
  fa.t = c->t;
  fa.dt = dt;
  fa.omega_frame = omega_frame;
  fa.nr = nr;
  fa.ns = ns;
  fa.evanescent = c->p.evanescent;
  fa.fast = c->p.fast_transport;
  fa.fpart = fp32 ? c->fu_fpart : nullptr;
  fa.crash = (int *)(c->d_fused + FG_FUSED_CRASH_SLOT);
  fa.nu = nu;
  fa.xe = b.Xe;
  fa.energy = adi ? c->f[FG_ENERGY] : nullptr;
  fa.cs = c->f[FG_SOUNDSPEED];
  fa.gamma = c->p.adiabatic_index;
  fa.adiabatic = adi ? 1 : 0;
  fa.cs_refresh = (adi && (flags & FG_STEP_CLOSES_DT)) ? 1 : 0;
  fa.sgacc = sg ? c->sgacc_mean : nullptr;
  fa.fxd = b.fXd();
  fa.fxvt = b.fXvt();
  fa.fxrmp = b.fXrmp();
  fa.fxrmm = b.fXrmm();
  fa.sbar = c->fu_sbar[c->fu_sbar_cur];
  fa.sbar_next = c->fu_sbar[c->fu_sbar_cur ^ 1];
  fa.lob0 = lob0;
  fa.lob1 = lob1;
  prof_mark(c);
  auto fin = adi ? k_fin<true, false> : fp32 ? k_fin<false, true> : k_fin<false, false>;
  hipLaunchKernelGGL(fin, dim3(xcd_grid(nr)), dim3(256), (size_t)ns * sizeof(double), c->stream, fa);
  FG_LAUNCH_CHECK();
  if (fp32) c->fu_sbar_cur ^= 1;  // k_fin wrote the next substep's Sigma background
  prof_mark(c);
  if (c->nu_pending) {  // the refreshed viscosity is now the current one
    std::swap(c->nu, c->nu_next);
    c->nu_pending = 0;
  }
  if (fg_status s = fused_reductions(c, DeltaT_next, fp32)) return s;
  if (fa.cs_refresh && c->p.viscosity_alpha) {
    // the next DT's alpha viscosity from the ring means of the new sound
    // speed (FViscosity via Make1Dprofile, as fg_ring_mean_cs computes it);
    // the next substep's first damping pass still uses this one
    if (fg_status s = fg_viscosity_into(c, c->nu_next)) return s;
    c->nu_pending = 1;
  }
  return FG_OK;
}

// ------------------------------------------- per-routine transport ----
// Transport (TransportEuler.cu:30) with the fused path's sweeps: two
// launches instead of one per quantity and step (86 with the copies), and the
// fields that the routines leave (k_cells forms the velocities).  9 + 7 us at
// 128 x 384, 18 + 17 us at 384 x 1152; bound as the fused path's sweeps are.  A
// 128 x 384 substep with an open edge went from 393 to 121 us with it, one wait for
// all of a substep's reductions, and results that the kernels write to host memory.
fg_status fg_transport_sweeps(fg_ctx *c, double dt, double omega_frame) {
  const int nr = c->nr, ns = c->ns;
  const bool adi = c->p.adiabatic;
  trad_args ta{};
  ta.dens = c->f[FG_DENS];
  ta.vr = c->f[FG_VRAD];
  ta.vt = c->f[FG_VTHETA];
  ta.energy = adi ? c->f[FG_ENERGY] : nullptr;
  for (int q = 0; q < 6; q++) ta.out[q] = c->sw[q];
  ta.vmed = c->VMed;
  ta.lost = c->p.open_inner ? c->LostByDisk : nullptr;
  ta.t = c->t;
  ta.dt = dt;
  ta.omega_frame = omega_frame;
  ta.nr = nr;
  ta.ns = ns;
  ta.nstrips = (ns + TRAD_TPB - 1) / TRAD_TPB;
  ta.band = trad_band(c, ta.nstrips);
  const dim3 gt(nr + ta.nstrips * ((nr + ta.band - 1) / ta.band));
  auto trad = adi ? (c->shared_faces ? k_trad<6, true, false> : k_trad<6, true, true>)
                  : (c->shared_faces ? k_trad<5, true, false> : k_trad<5, true, true>);
  hipLaunchKernelGGL(trad, gt, dim3(TRAD_TPB), 0, c->stream, ta);
  FG_LAUNCH_CHECK();
  taz_args za{};
  za.vt = c->f[FG_VTHETA];
  za.vmed = c->VMed;
  for (int q = 0; q < 6; q++) za.q[q] = c->sw[q];
  za.xd = c->f[FG_DENS];
  za.xvt = c->sw[6];
  za.xrmp = c->f[FG_RADMOMP];
  za.xrmm = c->f[FG_RADMOMM];
  za.xtmp = c->f[FG_THETAMOMP];
  za.xtmm = c->f[FG_THETAMOMM];
  za.xe = c->f[FG_ENERGY];
  za.xdint = c->f[FG_DENSINT];
  za.xres = c->f[FG_VTHETARES];
  za.nshift = c->Nshift;
  za.t = c->t;
  za.dt = dt;
  za.omega_frame = omega_frame;
  za.nr = nr;
  za.ns = ns;
  za.fast = c->p.fast_transport;
  const int cl = tazw_cells(c);
  const dim3 gz((ns + TAZW_P(cl) - 1) / TAZW_P(cl), nr);
  auto taz = adi ? (cl == 2 ? k_tazw_full<2, 6> : k_tazw_full<3, 6>) : (cl == 2 ? k_tazw_full<2, 5> : k_tazw_full<3, 5>);
  hipLaunchKernelGGL(taz, gz, dim3(64), 0, c->stream, za);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

// ================================================== batched ensemble ====
// Many independent disks (uneven grids, FP32 bulk mode) advanced one
// substep together: each fused phase is ONE launch over a work list of
// (disk, tile) items whose workgroups stride through the list, so small
// and large disks share the machine.  Per substep the host writes every
// disk's arguments (dt, planets, frame, active flag) into one pinned
// block; a hipGraph captured once copies it to the device, runs the
// phases and the reductions, and copies back each disk's CFL count and
// star force.  The per-disk arithmetic is the single-disk FP32 code, so
// a disk gives the same bits batched or alone.

struct batch_disk {
  src32_args src;
  trad_args trad;
  taz_args taz;
  fin_args fin;
  double *DT1D, *Vmoy, *newDT;
  const double *invRmed;
  double coef, DeltaT;  // CFL coefficient and the next substep's DeltaT
  int nr, active;
};

struct batch_result {
  double fx, fy;
  int cfl, pad;
};

// Each phase launch covers its whole work list, one workgroup per item.
// Measured on 64 disks: 1.83 ms per batch substep with 4096 looping workgroups
// per phase, 1.61 ms with one item per workgroup.

// work items are the same for the whole workgroup: keep them (and every
// address derived from them) in scalar registers
__device__ __forceinline__ int2 uniform2(int2 w) {
  return make_int2(__builtin_amdgcn_readfirstlane(w.x), __builtin_amdgcn_readfirstlane(w.y));
}

// a phase's arguments with their pointers as global ones
__device__ __forceinline__ fg_dev_tables global_tables(const fg_dev_tables &t) {
  fg_dev_tables g = t;
  for (double **p : {&g.Radii, &g.Rinf, &g.Rsup, &g.Rmed, &g.Surf, &g.invRinf, &g.invSurf, &g.invRmed, &g.invdiffRsup,
                     &g.invdiffRmed, &g.SigmaMed, &g.cs_iso, &g.dxtheta, &g.invdxtheta, &g.dxtheta_cfl, &g.ev_coef,
                     &g.ev_period, &g.ev_vtheta_arg, &g.cos_cell, &g.sin_cell})
    *p = global(*p);
  g.ev_zone = global(g.ev_zone);
  return g;
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(SRC32_WAVES))) void k_batch_src(
    const batch_disk *__restrict__ D, const int2 *__restrict__ items, int n) {
  __shared__ src32_lds lds;
  const int it = xcd_block(n);
  if (it < 0) return;
  const int2 w = uniform2(items[it]);
  if (D[w.x].active) src32_march(D[w.x].src, D[w.x].src.P, w.y, lds);
}

__global__ __launch_bounds__(TRAD_TPB) void k_batch_trad(const batch_disk *__restrict__ D, const int2 *__restrict__ items, int n) {
  if ((int)blockIdx.x >= n) return;
  const int2 w = uniform2(items[blockIdx.x]);
  if (!D[w.x].active) return;
  trad_args a = D[w.x].trad;
  a.t = global_tables(a.t);
  a.fdens = global(a.fdens);
  a.fvr = global(a.fvr);
  a.fvt = global(a.fvt);
  for (int q = 0; q < NQ; q++) a.fout[q] = global(a.fout[q]);
  a.sbar = global(a.sbar);
  a.vref = global(a.vref);
  a.vmed = global(a.vmed);
  trad32_block(a, w.y);
}

// one chunk of one ring per item: y = ring * chunks + chunk
__global__ __launch_bounds__(64) void k_batch_taz(const batch_disk *__restrict__ D, const int2 *__restrict__ items, int n) {
  __shared__ tazw_lds<2, 5> sh;
  if ((int)blockIdx.x >= n) return;
  const int2 w = uniform2(items[blockIdx.x]);
  if (!D[w.x].active) return;
  taz_args a = D[w.x].taz;
  a.t = global_tables(a.t);
  a.vmed = global(a.vmed);
  a.fvt = global(a.fvt);
  for (int q = 0; q < NQ; q++) a.fq[q] = global(a.fq[q]);
  a.fxd = global(a.fxd);
  a.fxvt = global(a.fxvt);
  a.fxrmp = global(a.fxrmp);
  a.fxrmm = global(a.fxrmm);
  a.sbar = global(a.sbar);
  a.vref = global(a.vref);
  a.nshift = global(a.nshift);
  const int nch = (a.ns + TAZW_P(2) - 1) / TAZW_P(2);
  const int i = w.y / nch;
  if (in_lob(i, a.lob0, a.lob1))
    tazw_body<2, true, 5, true>(a, i, w.y % nch, sh);
  else
    tazw_body<2, true, 5, false>(a, i, w.y % nch, sh);
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_batch_fin(
    const batch_disk *__restrict__ D, const int2 *__restrict__ items, int n) {
  extern __shared__ double lds_bfin[];
  if ((int)blockIdx.x >= n) return;
  const int2 w = uniform2(items[blockIdx.x]);
  if (!D[w.x].active) return;
  fin_args a = D[w.x].fin;
  a.t = global_tables(a.t);
  a.dens = global(a.dens);
  a.vr = global(a.vr);
  a.vt = global(a.vt);
  a.fxd = global(a.fxd);
  a.fxvt = global(a.fxvt);
  a.fxrmp = global(a.fxrmp);
  a.fxrmm = global(a.fxrmm);
  a.sbar = global(a.sbar);
  a.sbar_next = global(a.sbar_next);
  a.vmoy = global(a.vmoy);
  a.newdt = global(a.newdt);
  a.fpart = global(a.fpart);
  a.crash = global(a.crash);
  a.nu = global(a.nu);
  a.temp = nullptr;
  a.sgacc = nullptr;
  if (in_lob(w.y, a.lob0 - 1, a.lob1 + 1))
    fin_ring<false, true, true>(a, w.y, lds_bfin);
  else
    fin_ring<false, true, false>(a, w.y, lds_bfin);
}

// per disk: the force's final sum and the CFL count of the next substep
__global__ __launch_bounds__(256) void k_batch_close(const batch_disk *__restrict__ D, batch_result *__restrict__ res, int ndisk) {
  __shared__ double out[2];
  for (int k = blockIdx.x; k < ndisk; k += gridDim.x) {
    const batch_disk &d = D[k];
    if (d.active) {
      force_rings_final(d.fin.fpart, d.nr, out);
      __syncthreads();
      cfl_final(&res[k].cfl, d.DT1D, d.Vmoy, d.newDT, d.invRmed, d.coef, d.DeltaT, d.nr);
      if (threadIdx.x == 0) {
        res[k].fx = out[0];
        res[k].fy = out[1];
      }
    }
    __syncthreads();
  }
}

struct fg_batch_dev {
  int n;
  std::vector<fg_ctx *> ctx;
  hipStream_t stream;
  batch_disk *h_disk, *d_disk;  // pinned host block and its device copy
  batch_result *h_res, *d_res;
  int2 *it_src, *it_trad, *it_taz, *it_fin;
  int n_src, n_trad, n_taz, n_fin;
  int src_band, trad_band;  // of the disks without fixed ones
  int max_ns;
  hipGraph_t graph;
  hipGraphExec_t exec;
  int ready;  // items built and graph instantiated
};

static void batch_free(fg_batch_dev *b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  void *dev[] = {b->d_disk, b->d_res, b->it_src, b->it_trad, b->it_taz, b->it_fin};
  for (void *q : dev)
    if (q) (void)hipFree(q);
  if (b->h_disk) (void)hipHostFree(b->h_disk);
  if (b->h_res) (void)hipHostFree(b->h_res);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
}

void fg_batch_dev_destroy(fg_batch_dev *b) {
  if (!b) return;
  (void)hipStreamSynchronize(b->stream);
  batch_free(b);
}

fg_status fg_batch_dev_create(fg_ctx *const *ctx, int n, fg_batch_dev **out) {
  *out = nullptr;
  if (n <= 0) {
    fg_set_error("batch: no disks");
    return FG_E_INVALID;
  }
  for (int k = 0; k < n; k++) {
    if (!ctx[k] || ctx[k]->p.precision != FG_PREC_FP32) {
      fg_set_error("batch: disk %d is not an FP32 bulk-mode context", k);
      return FG_E_INVALID;
    }
    if (fg_status s = fused_supported(ctx[k])) return s;
    if (fg_status s = fused_alloc(ctx[k])) return s;
    if (ctx[k]->device != ctx[0]->device) {
      fg_set_error("batch: all disks must live on one device");
      return FG_E_INVALID;
    }
  }
  fg_batch_dev *b = new fg_batch_dev();
  b->n = n;
  b->ctx.assign(ctx, ctx + n);
  std::vector<int2> src, trad;
  for (int k = 0; k < n; k++) {
    src.push_back(make_int2(ctx[k]->nr + 1, (ctx[k]->ns + SRC_W - 1) / SRC_W));
    trad.push_back(make_int2(ctx[k]->nr, (ctx[k]->ns + TRAD_TPB - 1) / TRAD_TPB));
  }
  b->src_band = src32_band(src.data(), n);
  b->trad_band = march_band(trad.data(), n, 16);
  hipError_t e = hipStreamCreate(&b->stream);
  if (e == hipSuccess) e = hipHostMalloc((void **)&b->h_disk, n * sizeof(batch_disk), hipHostMallocDefault);
  if (e == hipSuccess) e = hipHostMalloc((void **)&b->h_res, n * sizeof(batch_result), hipHostMallocDefault);
  if (e == hipSuccess) e = hipMalloc((void **)&b->d_disk, n * sizeof(batch_disk));
  if (e == hipSuccess) e = hipMalloc((void **)&b->d_res, n * sizeof(batch_result));
  if (e != hipSuccess) {
    fg_set_error("batch: %s", hipGetErrorString(e));
    batch_free(b);
    return FG_E_HIP;
  }
  std::memset((void *)b->h_disk, 0, n * sizeof(batch_disk));
  std::memset((void *)b->h_res, 0, n * sizeof(batch_result));
  *out = b;
  return FG_OK;
}

template <class T>
static fg_status upload_items(const std::vector<T> &v, T **dev) {
  FG_HIP(hipMalloc((void **)dev, (v.empty() ? 1 : v.size()) * sizeof(T)));
  if (!v.empty()) FG_HIP(hipMemcpy(*dev, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return FG_OK;
}

// rings per band of a batched disk's source march and radial sweep: those that
// suit all the disks together (8 disks of 128 to 384 rings: 8 rings of the radial
// sweep 130 us per substep, 16 rings 135; 64 disks 625 and 617)
static int batch_src_band(const fg_batch_dev *b, const fg_ctx *c) {
  return c->tile_src_th ? std::min(c->tile_src_th, SRC_MAX_BAND) : b->src_band;
}
static int batch_trad_band(const fg_batch_dev *b, const fg_ctx *c) {
  return c->tile_trad_band ? c->tile_trad_band : b->trad_band;
}

// work lists (largest disks first) and the captured graph of one substep
static fg_status batch_build(fg_batch_dev *b) {
  std::vector<int> order(b->n);
  for (int k = 0; k < b->n; k++) order[k] = k;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return b->ctx[x]->S > b->ctx[y]->S; });
  std::vector<int2> src, trad, taz, fin;
  b->max_ns = 1;
  for (int k : order) {
    const fg_ctx *c = b->ctx[k];
    const int nr = c->nr, ns = c->ns, band = batch_trad_band(b, c), sband = batch_src_band(b, c);
    b->max_ns = std::max(b->max_ns, ns);
    const int nsrc = (ns + SRC_W - 1) / SRC_W * ((nr + sband) / sband);
    for (int q = 0; q < nsrc; q++) src.push_back(make_int2(k, q));
    const int nstrips = (ns + TRAD_TPB - 1) / TRAD_TPB;
    const int nblk = nr + nstrips * ((nr + band - 1) / band);
    for (int q = 0; q < nblk; q++) trad.push_back(make_int2(k, q));
    const int nch = (ns + TAZW_P(2) - 1) / TAZW_P(2);
    for (int i = 0; i < nr; i++) {
      for (int ch = 0; ch < nch; ch++) taz.push_back(make_int2(k, i * nch + ch));
      fin.push_back(make_int2(k, i));
    }
  }
  b->n_src = (int)src.size();
  b->n_trad = (int)trad.size();
  b->n_taz = (int)taz.size();
  b->n_fin = (int)fin.size();
  if (fg_status s = upload_items(src, &b->it_src)) return s;
  if (fg_status s = upload_items(trad, &b->it_trad)) return s;
  if (fg_status s = upload_items(taz, &b->it_taz)) return s;
  if (fg_status s = upload_items(fin, &b->it_fin)) return s;
  // capture: arguments in, five phases, two reductions, results out
  hipStream_t st = b->stream;
  FG_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  (void)hipMemcpyAsync(b->d_disk, b->h_disk, b->n * sizeof(batch_disk), hipMemcpyHostToDevice, st);
  hipLaunchKernelGGL(k_batch_src, dim3(xcd_grid(b->n_src)), dim3(64), 0, st, b->d_disk, b->it_src, b->n_src);
  hipLaunchKernelGGL(k_batch_trad, dim3(b->n_trad), dim3(TRAD_TPB), 0, st, b->d_disk, b->it_trad, b->n_trad);
  hipLaunchKernelGGL(k_batch_taz, dim3(b->n_taz), dim3(64), 0, st, b->d_disk, b->it_taz, b->n_taz);
  hipLaunchKernelGGL(k_batch_fin, dim3(b->n_fin), dim3(256), (size_t)b->max_ns * sizeof(double), st, b->d_disk, b->it_fin,
                     b->n_fin);
  hipLaunchKernelGGL(k_batch_close, dim3(b->n), dim3(256), 0, st, b->d_disk, b->d_res, b->n);
  (void)hipMemcpyAsync(b->h_res, b->d_res, b->n * sizeof(batch_result), hipMemcpyDeviceToHost, st);
  hipError_t ce = hipStreamEndCapture(st, &b->graph);
  if (ce != hipSuccess) {
    fg_set_error("batch graph capture: %s", hipGetErrorString(ce));
    return FG_E_HIP;
  }
  FG_HIP(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
  b->ready = 1;
  return FG_OK;
}

// arguments of disk k for its next substep (FP32 fused kernels); active=0
// leaves the disk untouched this substep
fg_status fg_batch_dev_set(fg_batch_dev *b, int k, int active, double dt, double omega_frame, double domega,
                           const fg_planet_pot *planets, int nb, double ix, double iy, double DeltaT_next) {
  if (!b || k < 0 || k >= b->n) return FG_E_INVALID;
  batch_disk &d = b->h_disk[k];
  d.active = active;
  if (!active) return FG_OK;
  if (nb < 0 || nb > FG_MAX_PLANETS || (nb > 0 && !planets)) {
    fg_set_error("batch: planet count %d", nb);
    return FG_E_INVALID;
  }
  fg_ctx *c = b->ctx[k];
  const int nr = c->nr, ns = c->ns;
  fused_bufs fb = bufs_of(c);
  int lob0 = 0, lob1 = 0;
  fp32_pair_rings(c, planets, nb, &lob0, &lob1);
  src32_args &s = d.src;
  s.lob0 = lob0;
  s.lob1 = lob1;
  s.dens = c->f[FG_DENS];
  s.vr = c->f[FG_VRAD];
  s.vt = c->f[FG_VTHETA];
  // FP32 storage backgrounds: this substep reads fu_sbar[cur], its k_fin
  // writes the other one for the next
  const double *sbar = c->fu_sbar[c->fu_sbar_cur];
  double *sbar_next = c->fu_sbar[c->fu_sbar_cur ^ 1];
  c->fu_sbar_cur ^= 1;
  s.vref = c->Vmoy;
  s.sbar = sbar;
  s.odens = fb.fBd();
  s.ovr = fb.fBvr();
  s.ovt = fb.fBvt();
  s.opress = nullptr;
  s.nu = c->nu;
  s.t = c->t;
  s.P.nb = nb;
  for (int q = 0; q < nb; q++) {
    s.P.x[q] = planets[q].x;
    s.P.y[q] = planets[q].y;
    s.P.m[q] = planets[q].mass;
    s.P.smooth[q] = planets[q].smooth;
    s.P.invd3[q] = planets[q].inv_d3;
  }
  s.P.ix = ix;
  s.P.iy = iy;
  s.dt = dt;
  s.omega_frame = omega_frame;
  s.domega = domega;
  s.nr = nr;
  s.ns = ns;
  s.indirect = c->p.indirect_term;
  s.evanescent = c->p.evanescent;
  s.nstrips = (ns + SRC_W - 1) / SRC_W;
  s.width = (ns + s.nstrips - 1) / s.nstrips;
  s.band = batch_src_band(b, c);
  trad_args &ta = d.trad;
  ta.dens = fb.Bd;
  ta.vr = fb.Bvr;
  ta.vt = fb.Bvt;
  ta.out[0] = fb.Rrmp;
  ta.out[1] = fb.Rrmm;
  ta.out[2] = fb.Rtmp;
  ta.out[3] = fb.Rtmm;
  ta.out[4] = fb.Rd;
  ta.fdens = fb.fBd();
  ta.fvr = fb.fBvr();
  ta.fvt = fb.fBvt();
  for (int q = 0; q < NQ; q++) ta.fout[q] = fb.fR(q);
  ta.sbar = sbar;
  ta.vref = c->Vmoy;
  ta.vmed = c->VMed;
  ta.t = c->t;
  ta.dt = dt;
  ta.omega_frame = omega_frame;
  ta.nr = nr;
  ta.ns = ns;
  ta.nstrips = (ns + TRAD_TPB - 1) / TRAD_TPB;
  ta.band = batch_trad_band(b, c);
  ta.lob0 = lob0;
  ta.lob1 = lob1;
  taz_args &za = d.taz;
  za.vt = fb.Bvt;
  za.vmed = c->VMed;
  za.q[0] = fb.Rrmp;
  za.q[1] = fb.Rrmm;
  za.q[2] = fb.Rtmp;
  za.q[3] = fb.Rtmm;
  za.q[4] = fb.Rd;
  za.xd = fb.Xd;
  za.xvt = fb.Xvt;
  za.xrmp = fb.Xrmp;
  za.xrmm = fb.Xrmm;
  za.fvt = fb.fBvt();
  for (int q = 0; q < NQ; q++) za.fq[q] = fb.fR(q);
  za.fxd = fb.fXd();
  za.fxvt = fb.fXvt();
  za.fxrmp = fb.fXrmp();
  za.fxrmm = fb.fXrmm();
  za.sbar = sbar;
  za.vref = c->Vmoy;
  za.nshift = c->Nshift;
  za.t = c->t;
  za.dt = dt;
  za.omega_frame = omega_frame;
  za.nr = nr;
  za.ns = ns;
  za.fast = c->p.fast_transport;
  za.lob0 = lob0;
  za.lob1 = lob1;
  fin_args &fa = d.fin;
  fa.xd = fb.Xd;
  fa.xvt = fb.Xvt;
  fa.xrmp = fb.Xrmp;
  fa.xrmm = fb.Xrmm;
  fa.press = fb.P;
  fa.dens = c->f[FG_DENS];
  fa.vr = c->f[FG_VRAD];
  fa.vt = c->f[FG_VTHETA];
  fa.temp = nullptr;
  fa.vmoy = c->Vmoy;
  fa.newdt = c->newDT;
  fa.nu = c->nu;
  fa.t = c->t;
  fa.dt = dt;
  fa.omega_frame = omega_frame;
  fa.nr = nr;
  fa.ns = ns;
  fa.evanescent = c->p.evanescent;
  fa.fast = c->p.fast_transport;
  fa.fpart = c->fu_fpart;
  fa.crash = (int *)(c->d_fused + FG_FUSED_CRASH_SLOT);
  fa.xe = nullptr;
  fa.energy = fa.cs = nullptr;
  fa.gamma = 0.0;
  fa.adiabatic = fa.cs_refresh = 0;
  fa.sgacc = nullptr;
  fa.fxd = fb.fXd();
  fa.fxvt = fb.fXvt();
  fa.fxrmp = fb.fXrmp();
  fa.fxrmm = fb.fXrmm();
  fa.sbar = sbar;
  fa.sbar_next = sbar_next;
  fa.lob0 = lob0;
  fa.lob1 = lob1;
  d.DT1D = c->DT1D;
  d.Vmoy = c->Vmoy;
  d.newDT = c->newDT;
  d.invRmed = c->t.invRmed;
  d.coef = c->t.dt1d_coef;
  d.DeltaT = DeltaT_next;
  d.nr = nr;
  return FG_OK;
}

// run one substep of every active disk (asynchronous)
fg_status fg_batch_dev_launch(fg_batch_dev *b) {
  if (!b->ready)
    if (fg_status s = batch_build(b)) return s;
  FG_HIP(hipGraphLaunch(b->exec, b->stream));
  return FG_OK;
}

// wait for the last launch; results of disk k
fg_status fg_batch_dev_wait(fg_batch_dev *b) {
  FG_HIP(hipStreamSynchronize(b->stream));
  return FG_OK;
}

void fg_batch_dev_result(const fg_batch_dev *b, int k, int *cfl, double *force2) {
  *cfl = b->h_res[k].cfl;
  force2[0] = b->h_res[k].fx;
  force2[1] = b->h_res[k].fy;
}

// after a tile-shape change the work lists and the graph are rebuilt
void fg_batch_dev_invalidate(fg_batch_dev *b) {
  if (!b || !b->ready) return;
  (void)hipStreamSynchronize(b->stream);
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
  for (void **q : {(void **)&b->it_src, (void **)&b->it_trad, (void **)&b->it_taz, (void **)&b->it_fin}) {
    if (*q) (void)hipFree(*q);
    *q = nullptr;
  }
  b->ready = 0;
}

extern "C" fg_status fg_set_fp32_pairs(fg_ctx *c, double hill_radii) {
  if (!c) return FG_E_INVALID;
  if (!(hill_radii >= 0.0 && hill_radii <= 100.0)) {
    fg_set_error("fg_set_fp32_pairs: %g Hill radii (0..100)", hill_radii);
    return FG_E_INVALID;
  }
  c->fp32_pair_hill = hill_radii;
  return FG_OK;
}

extern "C" fg_status fg_set_tiles(fg_ctx *c, int src_rows, int trad_band) {
  if (!c) return FG_E_INVALID;
  if ((src_rows != 8 && src_rows != 16 && src_rows != 32) || trad_band < 1 || trad_band > 4096) {
    fg_set_error("fg_set_tiles: rows %d (8, 16 or 32), band %d (1..4096)", src_rows, trad_band);
    return FG_E_INVALID;
  }
  c->tile_src_th = src_rows;
  c->tile_trad_band = trad_band;
  return FG_OK;
}

// ------------------------------------------------- shared-divisor check ----
// bitwise comparison of recip64(d).div(n) with the division n / d
__global__ void k_check_recip64(const double *num, const double *den, long n, unsigned long long *bad) {
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double q = num[t] / den[t];
  const double s = recip64(den[t]).div(num[t]);
  if (__double_as_longlong(q) != __double_as_longlong(s)) atomicAdd(bad, 1ull);
}

extern "C" fg_status fg_check_shared_division(const double *num, const double *den, long n, long *mismatches) {
  if (!num || !den || !mismatches || n < 0) return FG_E_INVALID;
  *mismatches = 0;
  if (n == 0) return FG_OK;
  double *dn = nullptr, *dd = nullptr;
  unsigned long long *dbad = nullptr, hbad = 0;
  hipError_t e = hipMalloc((void **)&dn, n * sizeof(double));
  if (e == hipSuccess) e = hipMalloc((void **)&dd, n * sizeof(double));
  if (e == hipSuccess) e = hipMalloc((void **)&dbad, sizeof(unsigned long long));
  if (e == hipSuccess) e = hipMemcpy(dn, num, n * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dd, den, n * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dbad, &hbad, sizeof(hbad), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_check_recip64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, dn, dd, n, dbad);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(&hbad, dbad, sizeof(hbad), hipMemcpyDeviceToHost);
  if (dn) (void)hipFree(dn);
  if (dd) (void)hipFree(dd);
  if (dbad) (void)hipFree(dbad);
  if (e != hipSuccess) {
    fg_set_error("fg_check_shared_division: %s", hipGetErrorString(e));
    return FG_E_HIP;
  }
  *mismatches = (long)hbad;
  return FG_OK;
}
