// Per-routine path: one HIP kernel (or a few) per reference routine, in
// the reference's order.  This is the drop-in granularity of the C-ABI
// (fg_pressure, fg_substep1, ...); the fused path in fg_fused.hip computes
// the same values with fewer passes.
//
// Launch shape: 1D, 256 threads, one thread per cell l = i*ns + j (row-
// major, sectors contiguous, so a wavefront reads 64 consecutive doubles).
#include "fg_cell.h"
#include "fg_internal.h"
#include "fg_reduce.h"

#define TPB 256

#define CELLS(i0, i1)                                                  \
  long l = (long)blockIdx.x * blockDim.x + threadIdx.x + (long)(i0)*ns; \
  if (l >= (long)(i1)*ns) return;                                      \
  const int i = (int)(l / ns);                                         \
  const int j = (int)(l - (long)i * ns);                               \
  (void)j;

#define JP ((long)i * ns + ((j + 1) % ns))
#define JM ((long)i * ns + ((j - 1 + ns) % ns))

#define LAUNCH(kern, i0, i1, ...)                                                              \
  do {                                                                                         \
    long n_ = (long)((i1) - (i0)) * c->ns;                                                     \
    if (n_ > 0) hipLaunchKernelGGL(kern, dim3(fg_blocks(n_, TPB)), dim3(TPB), 0, c->stream, __VA_ARGS__); \
    FG_LAUNCH_CHECK();                                                                         \
  } while (0)

static inline double *F(fg_ctx *c, int k) { return c->f[k]; }

// ---------------------------------------------------------------- EOS --
// Kernels.cu:167-184
__global__ void k_sound_speed(double *cs, const double *dens, const double *energy, const double *cs_iso, int nr,
                              int ns, int adiabatic, double gamma) {
  CELLS(0, nr)
  if (!adiabatic)
    cs[l] = cs_iso[i];
  else
    cs[l] = sqrt(gamma * (gamma - 1.0) * energy[l] / dens[l]);
}

// Make1DprofileKernel, Kernels.cu:610-623: one ring per block, the ring is
// staged in LDS and summed sequentially by one lane (the reference's j
// order) so the mean is bit-identical.
__global__ void k_ring_mean(double *out, const double *field, int nr, int ns) {
  (void)nr;  // one block per ring: the grid holds the ring count
  extern __shared__ double ring[];
  const int i = blockIdx.x;
  for (int j = threadIdx.x; j < ns; j += blockDim.x) ring[j] = field[(long)i * ns + j];
  __syncthreads();
  const double m = ring_seq_sum(ring, ns) / (double)ns;
  if (threadIdx.x == 0) out[i] = m;
}

// FViscosity (Viscosity.cu:33-50) from the ring mean of c_s
__global__ void k_viscosity(double *nu, const double *cs_mean, const double *pow15, const int *cav_on,
                            const double *cav, int nr, int alpha, double alphavisc, double visc) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nr) return;
  double v = visc;
  if (alpha) v = alphavisc * cs_mean[i] * cs_mean[i] * pow15[i];
  if (cav_on[i]) v *= cav[i];
  nu[i] = v;
}

// ------------------------------------------------- cell by cell --
// The routines that take each cell by itself, those of `flags` in this order:
// a public routine launches its own, a substep of the simulation the ones that
// follow each other, since at 128x384 each takes about 2 us and the next launch
// as much again (a substep with an open edge: 20 launches 116 us, 13 launches
// 100 us; 384x1152 with non-reflecting edges, from 20 launches to 14, 6 % less).
enum {
  CELL_POTENTIAL = 1,    // FillForcesArraysKernel, Kernels.cu:1226-1253
  CELL_CLOSE = 2,        // end of the transport, below
  CELL_CORRECT = 4,      // CorrectVthetaKernel, Kernels.cu:1256-1263
  CELL_OPEN = 8,         // OpenBoundaryKernel, Kernels.cu:482-495
  CELL_EVANESCENT = 16,  // EvanescentBoundaryKernel, Kernels.cu:967-1015
  CELL_PRESSURE = 32,    // Kernels.cu:187-200
  CELL_TEMPERATURE = 64  // Kernels.cu:203-213 (MU/R = 1)
};
struct cells_args {
  double *vr, *vt, *dens, *energy, *press, *temp, *pot, *densint, *mom[4];
  const double *xvt, *cs, *nu, *sgacc;
  fg_dev_tables t;
  fg_planets_arg P;
  double domega, dt, omega_frame, sigma0, gamma;
  int flags, nr, ns, adiabatic, sg, indirect;
};
__global__ __launch_bounds__(TPB) void k_cells(cells_args a) {
  const int nr = a.nr, ns = a.ns, flags = a.flags;
  CELLS(0, nr + 1)
  const fg_dev_tables &t = a.t;
  if (i == nr) {
    // what the reference's whole-array copies leave in the ghost ring: the
    // shifted fields 0, DENSINT the density's ghost values
    if (flags & CELL_CLOSE) {
      a.densint[l] = a.dens[l];
      a.dens[l] = 0.0;
      for (int q = 0; q < 4; q++) a.mom[q][l] = 0.0;
      if (a.adiabatic) a.energy[l] = 0.0;
    }
    return;
  }
  const double Rm = t.Rmed[i];
  if (flags & CELL_POTENTIAL) {
    // all planets in one pass (the additions keep the reference's order:
    // planet k, then the star after planet 0)
    const auto &P = ((__attribute__((address_space(4))) const cells_args *)__builtin_amdgcn_kernarg_segment_ptr())->P;
    const double InvDistance = 1.0 / Rm;
    const double x = Rm * t.cos_pot[j];
    const double y = Rm * t.sin_pot[j];
    double acc = 0.0;
    for (int k = 0; k < P.nb; k++) {
      const double xp = P.x[k], yp = P.y[k], m = P.m[k];
      const double distance = (x - xp) * (x - xp) + (y - yp) * (y - yp);
      const double distancesmooth = sqrt(distance + P.smooth[k]);
      double pv = -1.0 * m / distancesmooth;
      if (a.indirect) pv += 1.0 * m * P.invd3[k] * (x * xp + y * yp);
      acc += pv;
      if (k == 0) {
        pv = -1.0 * 1.0 * InvDistance;
        pv -= P.ix * x + P.iy * y;
        acc += pv;
      }
    }
    a.pot[l] = acc;
  }
  // vrad of ring i >= 1 after the transport (Kernels.cu:1193-1210; vtheta
  // comes from the azimuthal sweep)
  auto closed_vr = [&](long m) { return (a.mom[0][m - ns] + a.mom[1][m]) / (a.dens[m] + a.dens[m - ns] + 1e-20); };
  if (flags & CELL_CLOSE) {
    if (!(flags & CELL_OPEN) || i != 1) a.vr[l] = i > 0 ? closed_vr(l) : 0.0;
    a.vt[l] = a.xvt[l];
  }
  if (flags & CELL_CORRECT) a.vt[l] = a.vt[l] - a.domega * Rm;
  if (flags & CELL_OPEN) {  // (rings 1 and 2 keep their density, ring 2 its vrad)
    if (i == 0) {
      a.dens[l] = a.dens[l + ns];
      a.energy[l] = a.energy[l + ns];
    } else if (i == 1) {
      const double next = flags & CELL_CLOSE ? closed_vr(l + ns) : a.vr[l + ns];
      a.vr[l] = (next > 0.0 || a.dens[l] < a.sigma0) ? 0.0 : next;
    }
  }
  if ((flags & CELL_EVANESCENT) && t.ev_zone[i]) {
    // per-ring constants from host tables; lambda, vtheta0 and vrad0
    // evaluated as in the kernel
    const double lambda = t.ev_coef[i] * a.dt / t.ev_period[i];
    double vtheta0 = a.sg ? sqrt(t.ev_vtheta_arg[i] - Rm * a.sgacc[i]) : sqrt(t.ev_vtheta_arg[i]);
    vtheta0 -= Rm * a.omega_frame;
    const double vrad0 = -3.0 * a.nu[i] / Rm * t.vrad0_slope;
    a.vr[l] = damp_toward(a.vr[l], lambda, vrad0);
    a.vt[l] = damp_toward(a.vt[l], lambda, vtheta0);
    a.dens[l] = damp_toward(a.dens[l], lambda, t.SigmaMed[i]);
    if (a.adiabatic) a.energy[l] = damp_toward(a.energy[l], lambda, t.EnergyMed[i]);
  }
  if (flags & CELL_PRESSURE)
    a.press[l] = a.adiabatic ? (a.gamma - 1.0) * a.energy[l] : a.dens[l] * a.cs[l] * a.cs[l];
  if (flags & CELL_TEMPERATURE)
    a.temp[l] = a.adiabatic ? (a.gamma - 1.0) * a.energy[l] / a.dens[l] : a.press[l] / a.dens[l];
}

// --------------------------------------------------------- Substep 1 --
// Substep1Kernel, Kernels.cu:13-53
__global__ void k_substep1(double *vradint, double *vthetaint, const double *P, const double *dens,
                           const double *phi, const double *vr, const double *vt, fg_dev_tables t, double dt,
                           double omega_frame, int nr, int ns) {
  CELLS(0, nr)
  if (i > 0) {
    double gradp = (P[l] - P[l - ns]) * 2.0 / (dens[l] + dens[l - ns]) * t.invdiffRmed[i];
    double gradphi = (phi[l] - phi[l - ns]) * t.invdiffRmed[i];
    double vt2 = vt[l] + vt[JP] + vt[l - ns] + vt[JP - ns];
    vt2 = vt2 / 4.0 + omega_frame * t.Rinf[i];
    vt2 = vt2 * vt2;
    double vr_src = -gradp - gradphi;
    double vradint2 = vr_src + vt2 * t.invRinf[i];
    vradint[l] = vr[l] + dt * vradint2;
  }
  const double invdxtheta = t.invdxtheta[i];
  double gradp = (P[l] - P[JM]) * 2.0 / (dens[l] + dens[JM]) * invdxtheta;
  double gradphi = (phi[l] - phi[JM]) * invdxtheta;
  double v = vt[l] - dt * (gradp + gradphi);
  v += dt * t.supp_torque[i];
  vthetaint[l] = v;
}

// ViscousTermsKernel, Kernels.cu:733-771
__global__ void k_viscous_terms(const double *Vr, const double *Vt, const double *dens, const double *nu,
                                double *divV, double *TRR, double *TPP, double *TRP, fg_dev_tables t, int nr, int ns) {
  CELLS(0, nr)
  const double invdphi = t.invdphi;
  const double onethird = 1.0 / 3.0;
  double drr = (Vr[l + ns] - Vr[l]) * t.invdiffRsup[i];
  double dpp = (Vt[JP] - Vt[l]) * invdphi * t.invRmed[i] + 0.5 * (Vr[l + ns] + Vr[l]) * t.invRmed[i];
  double dv = (Vr[l + ns] * t.Rsup[i] - Vr[l] * t.Rinf[i]) * t.invdiffRsup[i] * t.invRmed[i];
  dv += (Vt[JP] - Vt[l]) * invdphi * t.invRmed[i];
  divV[l] = dv;
  TRR[l] = 2.0 * dens[l] * nu[i] * (drr - onethird * dv);
  TPP[l] = 2.0 * dens[l] * nu[i] * (dpp - onethird * dv);
  if (i > 0) {
    double drp = 0.5 * (t.Rinf[i] * (Vt[l] * t.invRmed[i] - Vt[l - ns] * t.invRmed[i - 1]) * t.invdiffRmed[i] +
                        (Vr[l] - Vr[JM]) * invdphi * t.invRinf[i]);
    TRP[l] = 2.0 * 0.25 * (dens[l] + dens[l - ns] + dens[JM] + dens[JM - ns]) * nu[i] * drp;
  }
}

// UpdateVelocitiesKernel, Kernels.cu:118-150
// and then, unless the edges damp (kepler), ApplySubKeplerianBoundaryKernel
// (Kernels.cu:1416-1430; the sqrt arguments come from the host; with
// self-gravity the ring mean of g_r enters)
__global__ void k_update_velocities(double *vti, double *vri, const double *dens, const double *TRR,
                                    const double *TPP, const double *TRP, fg_dev_tables t, double DeltaT, int nr,
                                    int ns, int kepler, const double *sgacc, double arg_in, double arg_out,
                                    double omega_frame, int sg) {
  CELLS(0, nr)
  const double invdphi = t.invdphi;
  if (kepler && (i == 0 || i == nr - 1)) {
    const double arg = i == 0 ? arg_in : arg_out;
    const double v = sg ? sqrt(arg - t.Rmed[i] * sgacc[i]) : sqrt(arg);
    vti[l] = v - t.Rmed[i] * omega_frame;
  } else if (i > 0 && i < nr - 1) {
    vti[l] += DeltaT * t.invRmed[i] *
              ((t.Rsup[i] * TRP[l + ns] - t.Rinf[i] * TRP[l]) * t.invdiffRsup[i] + (TPP[l] - TPP[JM]) * invdphi +
               0.5 * (TRP[l] + TRP[l + ns])) /
              (0.5 * (dens[l] + dens[JM]));
  }
  if (i == 0) return;
  vri[l] += DeltaT * t.invRinf[i] *
            ((t.Rmed[i] * TRR[l] - t.Rmed[i - 1] * TRR[l - ns]) * t.invdiffRmed[i] + (TRP[JP] - TRP[l]) * invdphi -
             0.5 * (TPP[l] + TPP[l - ns])) /
            (0.5 * (dens[l] + dens[l - ns]));
}

// --------------------------------------------------------- Substep 2 --
// Substep 2: the artificial pressure (Kernels.cu:409-434) into qr and qt, and
// "kernel", Kernels.cu:438-479, which takes the neighbours' formed again, with
// ActualiseGasVrad/Vtheta (SourceEuler.cu:492-503): the new velocities, rows 0
// and NRAD as they were in the New fields, also into Vrad / Vtheta
__global__ void k_substep2(double *vr, double *vt, double *vrnew, double *vtnew, double *eint, double *qr, double *qt,
                           const double *dens, const double *vri, const double *vti, const double *energy,
                           fg_dev_tables t, double dt, int nr, int ns, int adiabatic) {
  CELLS(0, nr + 1)
  if (i == nr) {
    vr[l] = vrnew[l];
    vt[l] = vtnew[l];
    return;
  }
  const double dvr = vri[l + ns] - vri[l], dvt = vti[JP] - vti[l];
  const double q = art_visc_q(dens[l], dvr), w = art_visc_q(dens[l], dvt);
  qr[l] = q;
  qt[l] = w;
  double v = vrnew[l];
  if (i > 0) {
    double d = dens[l] + dens[l - ns];
    double densint = q - art_visc_q(dens[l - ns], vri[l] - vri[l - ns]);
    v = vri[l] - dt * 2.0 / d * densint * t.invdiffRmed[i];
    vrnew[l] = v;
  }
  vr[l] = v;
  const double invdxtheta = t.invdxtheta[i];
  double dens2 = dens[l] + dens[JM];
  double tempint = w - art_visc_q(dens[JM], vti[l] - vti[JM]);
  const double u = vti[l] - dt * 2.0 / dens2 * tempint * invdxtheta;
  vtnew[l] = u;
  vt[l] = u;
  if (adiabatic)
    eint[l] = energy[l] - dt * q * dvr * t.invdiffRsup[i] - dt * w * dvt * invdxtheta;
}

// --------------------------------------------------------- Substep 3 --
// Substep3Kernel, Kernels.cu:56-77
__global__ void k_substep3a(double *qplus, const double *dens, const double *nu, const double *TRR,
                            const double *TRP, const double *TPP, const double *divV, int nr, int ns) {
  CELLS(1, nr)
  if (nu[i] != 0.0) {
    double q = 0.5 / nu[i] / dens[l] * (TRR[l] * TRR[l] + TRP[l] * TRP[l] + TPP[l] * TPP[l]);
    q += (2.0 / 9.0) * nu[i] * dens[l] * divV[l] * divV[l];
    qplus[l] = q;
  } else
    qplus[l] = 0.0;
}

// Substep3Kernel2, Kernels.cu:80-115.  lr01 = log(Rmed0/Rmed1),
// lr12 = log(Rmed1/Rmed2) are host constants; the data-dependent log/exp
// of the power-law extrapolation run on the device.
// with ActualiseGasEnergy (SourceEuler.cu:362): also into Energy, the ghost row as
// it was in EnergyNew
__global__ void k_substep3b(double *energy, double *enew, double *qplus, const double *dens, const double *eint,
                            const double *divV, const double *nu, fg_dev_tables t, double dt, double gamma, double lr01, double lr12,
                            int nr, int ns, int cooling) {
  CELLS(0, nr + 1)
  if (i == nr) {
    energy[l] = enew[l];
    return;
  }
  if (i == 0) {
    if (nu[nr - 1] != 0.0)
      qplus[l] = qplus[l + ns] * exp(log(qplus[l + ns] / qplus[l + 2 * ns]) * lr01 / lr12);
    else
      qplus[l] = 0.0;
  }
  double num, den;
  if (!cooling) {
    num = dt * qplus[l] + eint[l];
    den = 1.0 + (gamma - 1.0) * dt * divV[l];
  } else {
    num = t.EnergyMed[i] * dt * dens[l] / t.SigmaMed[i] + t.CoolingTimeMed[i] * eint[l] +
          dt * t.CoolingTimeMed[i] * (qplus[l] - t.QplusMed[i] * dens[l] / t.SigmaMed[i]);
    den = dt + t.CoolingTimeMed[i] + (gamma - 1.0) * dt * t.CoolingTimeMed[i] * divV[l];
  }
  const double e = num / den;
  enew[l] = e;
  energy[l] = e;
}

// ------------------------------------------------------------------ CFL --
// ConditionCFLKernel1D + 2D1 + 2D2 (Kernels.cu:1267-1335) for one ring
// per block: sequential ring mean of vtheta (bit-identical), per-cell
// time step, ring minimum (min is order independent).  The same pass sets
// *crash = 1 when a density (or, when energy is not NULL, an energy) of the
// ring is negative or not finite: the check of DetectCrash/CrashKernel
// (SourceEuler.cu:453-465, Kernels.cu:953-964, whose call the reference
// leaves commented out at SourceEuler.cu:266-273), NaN included.
__global__ void k_cfl_ring(double *vmoy, double *newdt, const double *vr, const double *vt, const double *cs,
                           const double *dens, const double *energy, int *crash, fg_dev_tables t, int nr, int ns,
                           int fast) {
  (void)nr;  // one block per ring: the grid holds the ring count
  extern __shared__ double sh[];
  double *ring = sh;               // ns
  double *red = sh + ns;           // blockDim
  const int i = blockIdx.x;
  bool bad = false;
  for (int j = threadIdx.x; j < ns; j += blockDim.x) {
    const long l = (long)i * ns + j;
    ring[j] = vt[l];
    const double d = dens[l];
    bad |= !(d >= 0.0 && d < HUGE_VAL);
    if (energy) {
      const double e = energy[l];
      bad |= !(e >= 0.0 && e < HUGE_VAL);
    }
  }
  if (bad) *crash = 1;
  __syncthreads();
  const double vm = ring_seq_sum(ring, ns) / (double)ns;
  if (threadIdx.x == 0) vmoy[i] = vm;
  if (i == 0) return;
  const double dxrad = t.Rsup[i] - t.Rinf[i];
  const double dxtheta = t.dxtheta_cfl[i];
  const double mindx = (dxtheta < dxrad) ? dxtheta : dxrad;  // min2
  double best = 1e30;
  for (int j = threadIdx.x; j < ns; j += blockDim.x) {
    long l = (long)i * ns + j;
    double vres = fast ? (ring[j] - vm) : ring[j];
    double invdt1 = cs[l] / mindx;
    double invdt2 = fabs(vr[l]) / dxrad;
    double invdt3 = fabs(vres) / dxtheta;
    double dvr = vr[l + ns] - vr[l];
    double dvt = ring[(j + 1) % ns] - ring[j];
    dvr = (dvr >= 0.0) ? 1e-10 : -dvr;
    dvt = (dvt >= 0.0) ? 1e-10 : -dvt;
    double a = dvr / dxrad, b = dvt / dxtheta;
    double invdt4 = (b > a) ? b : a;  // max2
    invdt4 *= 4.0 * 1.41 * 1.41;
    double dtc = 0.5 / sqrt(invdt1 * invdt1 + invdt2 * invdt2 + invdt3 * invdt3 + invdt4 * invdt4);
    if (dtc < best) best = dtc;
  }
  red[threadIdx.x] = best;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s && red[threadIdx.x + s] < red[threadIdx.x]) red[threadIdx.x] = red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) newdt[i] = red[0];
}

// ConditionCFLKernel2D2 (DT1D) + 2D3, Kernels.cu:1331-1359
__global__ void k_cfl_final(int *cfl, double *dt1d, const double *vmoy, const double *newdt,
                            const double *invRmed, double coef, double DeltaT, int nr) {
  cfl_final(cfl, dt1d, vmoy, newdt, invRmed, coef, DeltaT, nr);
}

// ----------------------------------------------------- entry points --
void fg_ask_ring_lds() {
  for (const void *k : {(const void *)k_ring_mean, (const void *)k_cfl_ring})
    (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, FG_RING_LDS);
}

static fg_status check(fg_ctx *c) {
  if (!c) {
    fg_set_error("NULL context");
    return FG_E_INVALID;
  }
  return FG_OK;
}

extern "C" fg_status fg_sound_speed(fg_ctx *c) {
  if (fg_status s = check(c)) return s;
  const int nr = c->nr, ns = c->ns;
  LAUNCH(k_sound_speed, 0, nr, F(c, FG_SOUNDSPEED), F(c, FG_DENS), F(c, FG_ENERGY), c->t.cs_iso, nr, ns,
         c->p.adiabatic, c->p.adiabatic_index);
  return FG_OK;
}

static fg_status pack_planets(fg_planets_arg *P, const fg_planet_pot *pl, int nb, double ix, double iy) {
  if (nb < 0 || nb > FG_MAX_PLANETS || (nb > 0 && !pl)) {
    fg_set_error("planet count %d outside 0..%d", nb, FG_MAX_PLANETS);
    return FG_E_INVALID;
  }
  P->nb = nb;
  for (int k = 0; k < nb; k++) {
    P->x[k] = pl[k].x;
    P->y[k] = pl[k].y;
    P->m[k] = pl[k].mass;
    P->smooth[k] = pl[k].smooth;
    P->invd3[k] = pl[k].inv_d3;
  }
  P->ix = ix;
  P->iy = iy;
  return FG_OK;
}

// k_cells with the context's fields; the caller adds what its flags read besides
static cells_args cells(fg_ctx *c, int flags) {
  cells_args a{};
  a.vr = F(c, FG_VRAD);
  a.vt = F(c, FG_VTHETA);
  a.dens = F(c, FG_DENS);
  a.energy = F(c, FG_ENERGY);
  a.press = F(c, FG_PRESSURE);
  a.temp = F(c, FG_TEMPERATURE);
  a.pot = F(c, FG_POTENTIAL);
  a.densint = F(c, FG_DENSINT);
  a.mom[0] = F(c, FG_RADMOMP);
  a.mom[1] = F(c, FG_RADMOMM);
  a.mom[2] = F(c, FG_THETAMOMP);
  a.mom[3] = F(c, FG_THETAMOMM);
  a.xvt = c->sw[6];
  a.cs = F(c, FG_SOUNDSPEED);
  a.nu = c->nu;
  a.sgacc = c->sgacc_mean;
  a.t = c->t;
  a.sigma0 = c->h_SigmaMed[0];
  a.gamma = c->p.adiabatic_index;
  a.flags = flags;
  a.nr = c->nr;
  a.ns = c->ns;
  a.adiabatic = c->p.adiabatic;
  a.sg = c->p.self_gravity;
  a.indirect = c->p.indirect_term;
  return a;
}
static fg_status launch_cells(fg_ctx *c, const cells_args &a) {
  LAUNCH(k_cells, 0, c->nr + 1, a);
  return FG_OK;
}

extern "C" fg_status fg_pressure(fg_ctx *c) {
  if (fg_status s = check(c)) return s;
  return launch_cells(c, cells(c, CELL_PRESSURE));
}

extern "C" fg_status fg_temperature(fg_ctx *c) {
  if (fg_status s = check(c)) return s;
  return launch_cells(c, cells(c, CELL_TEMPERATURE));
}

static fg_status refresh_viscosity(fg_ctx *c, double *nu_out) {
  hipLaunchKernelGGL(k_viscosity, dim3(fg_blocks(c->nr, 256)), dim3(256), 0, c->stream, nu_out, c->cs_mean,
                     c->t.visc_pow15, c->t.visc_cav_on, c->t.visc_cav, c->nr, c->p.viscosity_alpha,
                     c->p.alphaviscosity, c->t.visc_value);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

extern "C" fg_status fg_ring_mean_cs(fg_ctx *c) {
  if (fg_status s = check(c)) return s;
  c->nu_pending = 0;  // nu is current: a fused refresh held back is void
  hipLaunchKernelGGL(k_ring_mean, dim3(c->nr), dim3(256), c->ns * sizeof(double), c->stream, c->cs_mean,
                     F(c, FG_SOUNDSPEED), c->nr, c->ns);
  FG_LAUNCH_CHECK();
  return refresh_viscosity(c, c->nu);
}

// the alpha viscosity of the current sound speed field into nu_out (the
// fused path's refresh at the close of a DT), leaving nu as it is
fg_status fg_viscosity_into(fg_ctx *c, double *nu_out) {
  hipLaunchKernelGGL(k_ring_mean, dim3(c->nr), dim3(256), c->ns * sizeof(double), c->stream, c->cs_mean,
                     F(c, FG_SOUNDSPEED), c->nr, c->ns);
  FG_LAUNCH_CHECK();
  return refresh_viscosity(c, nu_out);
}

fg_status fg_cfl_ring_launch(fg_ctx *c) {
  const int nr = c->nr, ns = c->ns;
  size_t shm = (size_t)(ns + 256) * sizeof(double);
  hipLaunchKernelGGL(k_cfl_ring, dim3(nr), dim3(256), shm, c->stream, c->Vmoy, c->newDT, F(c, FG_VRAD),
                     F(c, FG_VTHETA), F(c, FG_SOUNDSPEED), F(c, FG_DENS),
                     c->p.adiabatic ? (const double *)F(c, FG_ENERGY) : (const double *)nullptr, c->cfl_out + 1, c->t,
                     nr, ns, c->p.fast_transport);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

fg_status fg_cfl_result(fg_ctx *c, int *ncfl) {
  volatile int *h = c->h_cfl;
  if (h[1]) {  // reported once; the next pass over a bad state flags it again
    h[1] = 0;
    fg_set_error("crash: negative or non-finite density or energy");
    return FG_E_CRASH;
  }
  if (fg_status s = fg_check_substep_results((double)h[0], nullptr)) return s;
  *ncfl = h[0];
  return FG_OK;
}

extern "C" fg_status fg_cfl(fg_ctx *c, double DeltaT, int *ncfl) {
  if (fg_status s = check(c)) return s;
  if (!ncfl) return FG_E_INVALID;
  if (fg_status s = fg_cfl_ring_launch(c)) return s;
  hipLaunchKernelGGL(k_cfl_final, dim3(1), dim3(256), 0, c->stream, c->cfl_out, c->DT1D, c->Vmoy, c->newDT,
                     c->t.invRmed, c->t.dt1d_coef, DeltaT, c->nr);
  FG_LAUNCH_CHECK();
  FG_HIP(hipStreamSynchronize(c->stream));
  return fg_cfl_result(c, ncfl);
}

extern "C" fg_status fg_potential(fg_ctx *c, const fg_planet_pot *planets, int nb, double ix, double iy) {
  if (fg_status s = check(c)) return s;
  cells_args a = cells(c, CELL_POTENTIAL);
  if (fg_status s = pack_planets(&a.P, planets, nb, ix, iy)) return s;
  return launch_cells(c, a);
}

extern "C" fg_status fg_correct_vtheta(fg_ctx *c, double domega) {
  if (fg_status s = check(c)) return s;
  cells_args a = cells(c, CELL_CORRECT);
  a.domega = domega;
  return launch_cells(c, a);
}

// the edges' routines behind the cells' (before) and before them (after: the
// pressure or temperature), in as few launches as their order allows: an open or
// an evanescent edge goes with the cells, the non-reflecting ones, which take ring
// means, behind them, and form the edge rings' pressure or temperature anew.  With
// several kinds of edges at once each has its own launch, and so has the end of the
// transport, which reads the neighbours' densities, before the damping
static fg_status with_boundary(fg_ctx *c, cells_args a, int after, double dt, double omega_frame) {
  const fg_params &p = c->p;
  a.dt = dt;
  a.omega_frame = omega_frame;
  const bool one = (p.open_inner != 0) + (p.non_reflecting != 0) + (p.evanescent != 0) <= 1 &&
                   !(p.evanescent && a.flags & CELL_CLOSE);
  if (one) {
    a.flags |= after | (p.open_inner ? CELL_OPEN : 0) | (p.evanescent ? CELL_EVANESCENT : 0);
    if (a.flags)
      if (fg_status s = launch_cells(c, a)) return s;
    if (!p.non_reflecting) return FG_OK;
    if (p.adiabatic)
      if (fg_status s = fg_sound_speed(c)) return s;
    return fg_nonreflecting_internal(c, after & CELL_PRESSURE ? F(c, FG_PRESSURE) : nullptr,
                                     after & CELL_TEMPERATURE ? F(c, FG_TEMPERATURE) : nullptr);
  }
  auto cells_of = [&](int flags) {
    a.flags = flags;
    return flags ? launch_cells(c, a) : FG_OK;
  };
  if (fg_status s = cells_of(a.flags)) return s;
  if (fg_status s = cells_of(p.open_inner ? CELL_OPEN : 0)) return s;
  if (p.non_reflecting) {
    if (p.adiabatic)
      if (fg_status s = fg_sound_speed(c)) return s;
    if (fg_status s = fg_nonreflecting_internal(c, nullptr, nullptr)) return s;
  }
  return cells_of((p.evanescent ? CELL_EVANESCENT : 0) | after);
}

extern "C" fg_status fg_boundary(fg_ctx *c, double dt, double omega_frame) {
  if (fg_status s = check(c)) return s;
  return with_boundary(c, cells(c, 0), 0, dt, omega_frame);
}

// fg_potential, fg_correct_vtheta (if corotating), fg_boundary and fg_pressure
fg_status fg_routine_begin(fg_ctx *c, const fg_planet_pot *planets, int nb, double ix, double iy, bool corotating,
                           double domega, double dt, double omega_frame) {
  cells_args a = cells(c, CELL_POTENTIAL | (corotating ? CELL_CORRECT : 0));
  a.domega = domega;
  if (fg_status s = pack_planets(&a.P, planets, nb, ix, iy)) return s;
  return with_boundary(c, a, CELL_PRESSURE, dt, omega_frame);
}

// Viscous stress of (vr, vt) into the TAU fields (Viscosity.cu:52-67).
// With alpha viscosity the ring mean of c_s is refreshed first.
static fg_status viscous_terms(fg_ctx *c, const double *vr, const double *vt) {
  const int nr = c->nr, ns = c->ns;
  if (c->p.viscosity_alpha)
    if (fg_status s = fg_ring_mean_cs(c)) return s;
  LAUNCH(k_viscous_terms, 0, nr, vr, vt, F(c, FG_DENS), c->nu, F(c, FG_DIVV), F(c, FG_TAURR),
         F(c, FG_TAUPP), F(c, FG_TAURP), c->t, nr, ns);
  return FG_OK;
}

fg_status fg_selfgravity_kick(fg_ctx *c, double dt);

extern "C" fg_status fg_substep1(fg_ctx *c, double dt, double omega_frame) {
  if (fg_status s = check(c)) return s;
  const int nr = c->nr, ns = c->ns;
  LAUNCH(k_substep1, 0, nr, F(c, FG_VRADINT), F(c, FG_VTHETAINT), F(c, FG_PRESSURE), F(c, FG_DENS),
         F(c, FG_POTENTIAL), F(c, FG_VRAD), F(c, FG_VTHETA), c->t, dt, omega_frame, nr, ns);
  if (c->p.self_gravity)
    if (fg_status s = fg_selfgravity_kick(c, dt)) return s;
  if (fg_status s = viscous_terms(c, F(c, FG_VRADINT), F(c, FG_VTHETAINT))) return s;
  // SideEuler.cu:194-206: the sqrt arguments are the evanescent vtheta0
  // arguments of the edge rings (same expression)
  LAUNCH(k_update_velocities, 0, nr, F(c, FG_VTHETAINT), F(c, FG_VRADINT), F(c, FG_DENS), F(c, FG_TAURR),
         F(c, FG_TAUPP), F(c, FG_TAURP), c->t, dt, nr, ns, !c->p.evanescent, c->sgacc_mean, c->h_vtheta_arg[0],
         c->h_vtheta_arg[nr - 1], omega_frame, c->p.self_gravity);
  return FG_OK;
}

extern "C" fg_status fg_substep2(fg_ctx *c, double dt) {
  if (fg_status s = check(c)) return s;
  const int nr = c->nr, ns = c->ns;
  LAUNCH(k_substep2, 0, nr + 1, F(c, FG_VRAD), F(c, FG_VTHETA), F(c, FG_VRADNEW), F(c, FG_VTHETANEW),
         F(c, FG_ENERGYINT), F(c, FG_DENSINT), F(c, FG_TEMPERINT), F(c, FG_DENS), F(c, FG_VRADINT),
         F(c, FG_VTHETAINT), F(c, FG_ENERGY), c->t, dt, nr, ns, c->p.adiabatic);
  return FG_OK;
}

extern "C" fg_status fg_substep3(fg_ctx *c, double dt) {
  if (fg_status s = check(c)) return s;
  if (!c->p.adiabatic) return FG_OK;
  const int nr = c->nr, ns = c->ns;
  if (fg_status s = viscous_terms(c, F(c, FG_VRAD), F(c, FG_VTHETA))) return s;
  LAUNCH(k_substep3a, 1, nr, F(c, FG_QPLUS), F(c, FG_DENS), c->nu, F(c, FG_TAURR), F(c, FG_TAURP), F(c, FG_TAUPP),
         F(c, FG_DIVV), nr, ns);
  const double lr01 = c->lr01, lr12 = c->lr12;
  LAUNCH(k_substep3b, 0, nr + 1, F(c, FG_ENERGY), F(c, FG_ENERGYNEW), F(c, FG_QPLUS), F(c, FG_DENS),
         F(c, FG_ENERGYINT), F(c, FG_DIVV), c->nu, c->t, dt, c->p.adiabatic_index, lr01, lr12, nr, ns, c->p.cooling);
  return FG_OK;
}

fg_status fg_ring_sum_async(fg_ctx *c, const double *ring, double *out_dev);

// the mass that left through an open inner edge (TransportEuler.cu:77); the
// other edges' faces carry no flux
static fg_status sum_lost_mass(fg_ctx *c) {
  return c->p.open_inner ? fg_ring_sum_async(c, c->LostByDisk, c->red_out + 2) : FG_OK;
}

// fg_transport, fg_boundary and fg_temperature
fg_status fg_routine_end(fg_ctx *c, double dt, double omega_frame) {
  if (fg_status s = fg_transport_sweeps(c, dt, omega_frame)) return s;
  if (fg_status s = with_boundary(c, cells(c, CELL_CLOSE), CELL_TEMPERATURE, dt, omega_frame)) return s;
  return sum_lost_mass(c);
}

extern "C" fg_status fg_transport(fg_ctx *c, double dt, double omega_frame, double *lost_mass) {
  if (fg_status s = check(c)) return s;
  if (fg_status s = fg_transport_sweeps(c, dt, omega_frame)) return s;
  if (fg_status s = launch_cells(c, cells(c, CELL_CLOSE))) return s;
  if (fg_status s = sum_lost_mass(c)) return s;
  if (lost_mass) {
    if (c->p.open_inner) FG_HIP(hipStreamSynchronize(c->stream));
    *lost_mass = c->p.open_inner ? c->h_out[2] : 0.0;
  }
  return FG_OK;
}
