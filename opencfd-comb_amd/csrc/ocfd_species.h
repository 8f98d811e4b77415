// ocfd_species.h -- kernels of the multi-species flow path (N_SPEC > 1):
// mixture thermodynamics (perfect or NASA-fit real gas), transport
// coefficients (Sutherland/Pr/Sc or Chemkin fits with Wilke mixing), species
// convection and diffusion, the species RK3 update, primitive recovery with
// Rescaling_di, face re-synthesis and the jet boundary condition.
//
// Same conventions as ocfd_device.h: FP64, no FMA contraction, the
// reference's operation order.  Included once, by ocfd_flow.hip.
#pragma once
#include <type_traits>

#include "ocfd_device.h"
#include "ocfd_exp.h"

#define GAS_NT_MAX 4
#define GAS_R0 8.314       // CHEM_modules.f90:20
#define GAS_ATM 1.013e5    // CHEM_modules.f90:22

// Species data of the flow path (read_Spec, CHEM_thermdyn.f90:16-51; the
// transport fits of TRANSPORT_modules.f90:80-253).
struct FlowGas {
  int ns, n_tct, real_gas, flag_vis, flag_cond, flag_diff;
  double tct[GAS_NT_MAX], tct_max;
  double Mi[OCFD_NS_MAX], rMi[OCFD_NS_MAX], Ri[OCFD_NS_MAX];  // rMi = 1 / Mi
  double coef[OCFD_NS_MAX][GAS_NT_MAX][7], ect[OCFD_NS_MAX][GAS_NT_MAX];
  // (A-1) R, B R, C R, D R, E R, Ect R of each range, and 2.5 R: the products
  // that the mixture's sums of energy start with; cpa = A R, of Cp
  double ev[GAS_NT_MAX][6][OCFD_NS_MAX], rcv[OCFD_NS_MAX], cpa[GAS_NT_MAX][OCFD_NS_MAX];
  double exp2t[CH_EXPN][2];  // chem_exp's table
  double mu_an[OCFD_NS_MAX][4], k_an[OCFD_NS_MAX][4], D_an[OCFD_NS_MAX][OCFD_NS_MAX][4];
  // Wilke factors that depend only on the molar masses, evaluated on the
  // host: wq = (M_j/M_k)^(1/4) and wrec = 1/sqrt(8 (1 + M_k/M_j))
  double wq[OCFD_NS_MAX][OCFD_NS_MAX], wrec[OCFD_NS_MAX][OCFD_NS_MAX];
};
__constant__ FlowGas fg;

// The bank by a pointer that the compiler cannot see through, taken afresh by
// every function below: in a loop the hundreds of constants of an inlined
// gas_T would be hoisted out and spilled (5,400 register moves in k_bc).
typedef const __attribute__((address_space(4))) FlowGas* Gas;
__device__ __forceinline__ Gas gas_bank() {
  Gas g = (Gas)&fg;
  asm volatile("" : "+s"(g));
  return g;
}

// a / b to the last bit, given r = 1 / b correctly rounded: the quotient's
// remainder corrects it (Markstein).  3 instructions against a division's 11.
__device__ __forceinline__ double quot(double a, double b, double r) {
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
__device__ __forceinline__ double gp3(double x) { double x2 = x * x; return x2 * x; }
__device__ __forceinline__ double gp4(double x) { double x2 = x * x; return x2 * x2; }
__device__ __forceinline__ double gp5(double x) { double x2 = x * x; return (x2 * x2) * x; }

__device__ __forceinline__ int gas_range(Gas g, double T) {
  int jc = 0;
  for (int j = 0; j < g->n_tct - 1; j++)
    if (T > g->tct[j]) jc = j + 1;
  return jc;
}

// The species loops below run to the fixed bound, fully unrolled: with all
// species present (FULL) without a test, so that the scalar loads of the bank
// and the loads of the partial densities are all in flight together; with
// fewer, a uniform branch each.  As loops of ns passes each pass waited for
// its own loads: k_bc of a 48x36x36 jet 33 us against 24, k_comput_T_P 13
// against 7.
template <class F>
__device__ __forceinline__ void each_species(F f) {
  if (fg.ns == OCFD_NS_MAX) {
#pragma unroll
    for (int k = 0; k < OCFD_NS_MAX; k++) f(k);
  } else {
#pragma unroll
    for (int k = 0; k < OCFD_NS_MAX; k++)
      if (k < fg.ns) f(k);
  }
}

// sum over the species of the energy polynomial's coefficients in range j (a
// uniform index); CP: of Cp's, whose first is A R and which has no sixth
template <bool CP>
__device__ __forceinline__ void gas_sums(Gas g, const double* di, int j, double* s) {
  constexpr int N = CP ? 5 : 6;
#pragma unroll
  for (int a = 0; a < N; a++) s[a] = 0.0;
  each_species([&](int k) {
    s[0] = s[0] + (CP ? g->cpa[j][k] : g->ev[j][0][k]) * di[k];
#pragma unroll
    for (int a = 1; a < N; a++) s[a] = s[a] + g->ev[j][a][k] * di[k];
  });
}

// ... in range jc of each lane: the lanes of one range at a time, so that the
// coefficients stay scalar loads
template <bool CP>
__device__ __forceinline__ void gas_sums_lane(Gas g, const double* di, int jc, double* s) {
#pragma unroll
  for (int a = 0; a < (CP ? 5 : 6); a++) s[a] = 0.0;
  for (int j = 0; j < g->n_tct; j++)
    if (jc == j) gas_sums<CP>(g, di, j, s);
}

// comput_E_pgas (CHEM_thermdyn.f90:114-122) / comput_E_rgas (:203-231)
__device__ __forceinline__ double gas_E(const double* di, double T) {
  const Gas g = gas_bank();
  if (!g->real_gas) {
    double E = 0.0;
    each_species([&](int k) { E = E + g->rcv[k] * di[k] * T; });
    return E;
  }
  double s[6];
  gas_sums_lane<false>(g, di, gas_range(g, T), s);
  const double A1 = s[0], B1 = s[1], C1 = s[2], D1 = s[3], E1 = s[4], Ect = s[5];
  if (T <= g->tct_max) return A1 * T + B1 * (T * T) / 2.0 + quot(C1 * gp3(T), 3.0, 1.0 / 3.0) + D1 * gp4(T) / 4.0 + quot(E1 * gp5(T), 5.0, 0.2) + Ect;
  const double tm = g->tct_max;
  const double Cv2 = A1 + B1 * tm + C1 * (tm * tm) + D1 * gp3(tm) + E1 * gp4(tm);
  return A1 * tm + B1 * (tm * tm) / 2.0 + quot(C1 * gp3(tm), 3.0, 1.0 / 3.0) + D1 * gp4(tm) / 4.0 + quot(E1 * gp5(tm), 5.0, 0.2) + Ect +
         Cv2 * (T - tm);
}

// comput_T_pgas (CHEM_thermdyn.f90:157-168) / comput_T_rgas (:326-382)
__device__ __forceinline__ double gas_T(const double* di, double E) {
  const Gas g = gas_bank();
  if (!g->real_gas) {
    double rCv = 0.0;
    each_species([&](int k) { rCv = rCv + g->rcv[k] * di[k]; });
    return E / rCv;
  }
  double s[GAS_NT_MAX][6];
#pragma unroll
  for (int j = 0; j < GAS_NT_MAX; j++) {
#pragma unroll
    for (int a = 0; a < 6; a++) s[j][a] = 0.0;
    if (j < g->n_tct) gas_sums<false>(g, di, j, s[j]);
  }
  double T1 = E / s[0][0], T2 = T1;
  for (int ks = 0; ks <= 30; ks++) {
    const int jc = gas_range(g, T1);
    double a = s[0][0], b = s[0][1], c = s[0][2], d = s[0][3], e = s[0][4], ect = s[0][5];
#pragma unroll
    for (int j = 1; j < GAS_NT_MAX; j++)
      if (jc == j) { a = s[j][0]; b = s[j][1]; c = s[j][2]; d = s[j][3]; e = s[j][4]; ect = s[j][5]; }
    double Et1, Ex;
    if (T1 <= g->tct_max) {
      Et1 = a * T1 + b * (T1 * T1) / 2.0 + quot(c * gp3(T1), 3.0, 1.0 / 3.0) + d * gp4(T1) / 4.0 + quot(e * gp5(T1), 5.0, 0.2) + ect;
      Ex = a + b * T1 + c * (T1 * T1) + d * gp3(T1) + e * gp4(T1);
    } else {
      const double tm = g->tct_max;
      Ex = a + b * tm + c * (tm * tm) + d * gp3(tm) + e * gp4(tm);
      Et1 = a * tm + b * (tm * tm) / 2.0 + quot(c * gp3(tm), 3.0, 1.0 / 3.0) + d * gp4(tm) / 4.0 + quot(e * gp5(tm), 5.0, 0.2) + ect +
            Ex * (T1 - tm);
    }
    T2 = T1 - (Et1 - E) / Ex;
    const double error = fabs(T2 - T1);
    T1 = T2;
    if (error < 1.0e-3) break;
  }
  return T2;
}

// comput_P, CHEM_thermdyn.f90:385-395
__device__ __forceinline__ double gas_P(const double* di, double T) {
  const Gas g = gas_bank();
  double p = 0.0;
  each_species([&](int k) { p = p + g->Ri[k] * di[k] * T; });
  return p;
}

// comput_d, CHEM_thermdyn.f90:399-409 (ai = mass fractions)
__device__ __forceinline__ double gas_d(const double* ai, double T, double p) {
  const Gas g = gas_bank();
  double R1 = 0.0;
  each_species([&](int k) { R1 = R1 + g->Ri[k] * ai[k]; });
  return p / (T * R1);
}

// comput_Cp_pgas (CHEM_thermdyn.f90:125-136) / comput_Cp_rgas (:234-266)
__device__ __forceinline__ double gas_Cp(double d, const double* di, double T) {
  const Gas g = gas_bank();
  if (!g->real_gas) {
    double Cp = 0.0;
    each_species([&](int k) { Cp = Cp + 3.5 * g->Ri[k] * di[k]; });
    return Cp / d;
  }
  double s[5];
  gas_sums_lane<true>(g, di, gas_range(g, T), s);
  const double t = T <= g->tct_max ? T : g->tct_max;
  return (s[0] + s[1] * t + s[2] * (t * t) + s[3] * gp3(t) + s[4] * gp4(t)) / d;
}

// comput_hi_pgas (CHEM_thermdyn.f90:176-182) / comput_hi_rgas (:271-293)
__device__ double gas_hi(int k, double T) {
  const Gas g = gas_bank();
  if (!g->real_gas) return 3.5 * g->Ri[k] * T;
  const int jc = gas_range(g, T);
  double c0 = 0.0, c1 = 0.0, c2 = 0.0, c3 = 0.0, c4 = 0.0, ect = 0.0;
  for (int j = 0; j < g->n_tct; j++)  // the lanes of one range at a time: scalar loads
    if (jc == j) {
      c0 = g->coef[k][j][0];
      c1 = g->coef[k][j][1];
      c2 = g->coef[k][j][2];
      c3 = g->coef[k][j][3];
      c4 = g->coef[k][j][4];
      ect = g->ect[k][j];
    }
  if (T <= g->tct_max)
    return (c0 * T + c1 * (T * T) / 2.0 + quot(c2 * gp3(T), 3.0, 1.0 / 3.0) + c3 * gp4(T) / 4.0 + quot(c4 * gp5(T), 5.0, 0.2) + ect) * g->Ri[k];
  const double tm = g->tct_max;
  const double Cp_max = c0 + c1 * tm + c2 * (tm * tm) + c3 * gp3(tm) + c4 * gp4(tm);
  return (c0 * tm + c1 * (tm * tm) / 2.0 + quot(c2 * gp3(tm), 3.0, 1.0 / 3.0) + c3 * gp4(tm) / 4.0 + quot(c4 * gp5(tm), 5.0, 0.2) + ect +
          Cp_max * (T - tm)) * g->Ri[k];
}

// exponent of the Chemkin fit exp(a1 + a2 lnT + a3 lnT^2 + a4 lnT^3),
// TRANSPORT_modules.f90:276-277
__device__ __forceinline__ double chemkin_fit(const double* a, double lT) {
  return __builtin_fma(__builtin_fma(__builtin_fma(a[3], lT, a[2]), lT, a[1]), lT, a[0]);
}

__device__ __forceinline__ void cell_ijk(const DevState& S, long c, int& i, int& j, int& k) {
  i = (int)(c % S.nx) + 1;
  j = (int)((c / S.nx) % S.ny) + 1;
  k = (int)(c / ((long)S.nx * S.ny)) + 1;
}

// ===========================================================================
// comput_Amu_Amk_AMD (Comput_flow_variables.f90:69-98) for N_SPEC > 1:
// comput_vis_coeff (TRANSPORT_modules.f90:259-306), comput_Cp,
// comput_thermal_conductivity (:312-372), comput_diffusion_coeff (:378-424).
// ===========================================================================
// conc: also c_m = di_m / d for the species diffusion (du_scaler_viscous),
// whose di and d are at hand here.
// Bound by its arithmetic: 9 + 9 + 36 exponentials a cell.  The fits are
// Horner FMAs and chem_exp; a fit that the mixture rules divide by is the
// exponential of the negative exponent, and the square roots of the
// viscosities and their inverses come from the half exponent.  Largest
// (mean) relative error of the H2 mixture's fits against 80-bit arithmetic,
// 250 to 3500 K: viscosity 2.7e-15 (5.3e-16), conductivity 5.6e-15 (7.8e-16),
// 1/D 5.2e-15 (9.2e-16); with powers, exp and divisions 5.6e-15 (8.6e-16),
// 1.7e-14 (1.6e-15), 9.6e-15 (1.3e-15).  us before / now: 48x36x36 40 / 21,
// 160x112x64 210 (and 57 for the concentrations) / 112.  first: the launch
// opens a step and resets the negative-Et counters.
template <bool FULL>
__global__ __launch_bounds__(256, 4) void k_transport_ms(DevState S, int first, int conc) {
  __shared__ double2 tab[CH_EXPN];
  if (threadIdx.x < CH_EXPN) tab[threadIdx.x] = make_double2(fg.exp2t[threadIdx.x][0], fg.exp2t[threadIdx.x][1]);
  __syncthreads();
  const long c = cell_index();
  if (first && blockIdx.x == 0 && threadIdx.x == 0) negt_reset(S, 1);
  if (c >= S.ni) return;
  int i, j, k;
  cell_ijk(S, c, i, j, k);
  const long q = hq(S, i, j, k);
  const int ns = FULL ? OCFD_NS_MAX : fg.ns;
  // species loops run to the fixed bound with guards, fully unrolled, so the
  // per-species arrays stay in registers
  double di0[OCFD_NS_MAX], Xi[OCFD_NS_MAX];
#pragma unroll
  for (int m = 0; m < OCFD_NS_MAX; m++) di0[m] = m < ns ? S.di[q + (long)m * S.nh] : 0.0;
  const double T = S.T[q];
  if (conc) {
    const double d = S.d[q], rd = 1.0 / d;
#pragma unroll
    for (int m = 0; m < OCFD_NS_MAX; m++)
      if (m < ns) S.cs[c + (long)m * S.ni] = quot(di0[m], d, rd);
  }
  double X0 = 0.0;
#pragma unroll
  for (int m = 0; m < OCFD_NS_MAX; m++) {
    Xi[m] = m < ns ? quot(di0[m], fg.Mi[m], fg.rMi[m]) : 0.0;
    if (m < ns) X0 = X0 + Xi[m];
  }
  const double rX0 = 1.0 / X0;
#pragma unroll
  for (int m = 0; m < OCFD_NS_MAX; m++)
    if (m < ns) Xi[m] = quot(Xi[m], X0, rX0);
  const double lT = log(T);
  double amu;
  if (fg.flag_vis == 0) {
    const double TA = 288.15, TC = 110.4;
    const double tr = T / TA;
    amu = S.amu0 * sqrt(gp3(tr)) * (TA + TC) / (TC + T);
  } else {
    // Wilke's Phi_kj = (1 + sqrt(mu_k/mu_j) (M_j/M_k)^(1/4))^2 / sqrt(8 (1 +
    // M_k/M_j)) (comput_vis_coeff, TRANSPORT_modules.f90:296-305) with
    // sqrt(mu_k/mu_j) = sqrt(mu_k) / sqrt(mu_j), up to the fits' common
    // factor 0.1
    double smu[OCFD_NS_MAX], rmu[OCFD_NS_MAX];
#pragma unroll
    for (int m = 0; m < OCFD_NS_MAX; m++) {
      const double e = 0.5 * chemkin_fit(fg.mu_an[m], lT);
      smu[m] = m < ns ? chem_exp(tab, e) : 1.0;
      rmu[m] = m < ns ? chem_exp(tab, -e) : 1.0;
    }
    double mu = 0.0;
#pragma unroll
    for (int kk = 0; kk < OCFD_NS_MAX; kk++) {
      if (kk < ns) {
        double Pk0 = 0.0;
#pragma unroll
        for (int jj = 0; jj < OCFD_NS_MAX; jj++) {
          if (jj < ns) {
            const double a = __builtin_fma(smu[kk] * rmu[jj], fg.wq[kk][jj], 1.0);
            Pk0 = __builtin_fma(Xi[jj] * (a * a), fg.wrec[kk][jj], Pk0);
          }
        }
        mu = mu + Xi[kk] * (smu[kk] * smu[kk]) / Pk0;
      }
    }
    amu = mu * 0.1;
  }
  double amk;
  if (fg.flag_cond == 0) {
    amk = amu * gas_Cp(S.d[q], di0, T) / S.pr;
  } else {
    double Amk1 = 0.0, Amk2 = 0.0;
#pragma unroll
    for (int m = 0; m < OCFD_NS_MAX; m++)
      if (m < ns) {
        const double e = chemkin_fit(fg.k_an[m], lT);
        Amk1 = __builtin_fma(Xi[m], chem_exp(tab, e), Amk1);
        Amk2 = __builtin_fma(Xi[m], chem_exp(tab, -e), Amk2);
      }
    amk = 0.5 * (Amk1 + 1.0 / Amk2) * 1.0e-5;
  }
  S.Amu[c] = amu;
  S.Amk[c] = amk;
  if (fg.flag_diff == 0) {
    double d0 = 0.0;
#pragma unroll
    for (int m = 0; m < OCFD_NS_MAX; m++)
      if (m < ns) d0 = d0 + Xi[m] * fg.Mi[m];
#pragma unroll
    for (int m = 0; m < OCFD_NS_MAX; m++)
      if (m < ns)
        S.AmD[c + (long)m * S.ni] = amu * (1.0 - Xi[m] * fg.Mi[m] / d0) / ((1.0 - Xi[m]) * S.sc * S.d[q] + 1.0e-20);
  } else {
    // binary coefficients D(k,j) = D(j,k) from the fit of the pair k < j (the
    // reference fills the lower triangle from the upper one), each evaluated
    // once.  Visiting the pairs (a, b), a < b, with a outer and b inner adds
    // the terms of every ds_k in increasing j, the reference's order.
    const double pq = GAS_ATM / S.p[q];
    double ds[OCFD_NS_MAX];
#pragma unroll
    for (int m = 0; m < OCFD_NS_MAX; m++) ds[m] = 0.0;
#pragma unroll
    for (int a = 0; a < OCFD_NS_MAX; a++)
#pragma unroll
      for (int b = a + 1; b < OCFD_NS_MAX; b++)
        if (b < ns) {
          const double rD = chem_exp(tab, -chemkin_fit(fg.D_an[a][b], lT));
          ds[a] = __builtin_fma(Xi[b], rD, ds[a]);
          ds[b] = __builtin_fma(Xi[a], rD, ds[b]);
        }
#pragma unroll
    for (int kk = 0; kk < OCFD_NS_MAX; kk++) {
      if (kk < ns)
        S.AmD[c + (long)kk * S.ni] = (1.0 - Xi[kk]) / __builtin_fma(ds[kk], 1.0e4, 1.0e-20) * pq;
    }
  }
}

// ===========================================================================
// du_scaler_invis (OCFD_scaler_inviscous.f90:1-84) for all species at once:
// scalar Steger-Warming split F+- = (vs +- |vs|)/2 * di_m with vs = A1 u +
// A2 v + A3 w, the flow's reconstructions and closures, the same hybrid masks.
// Each species only reads its own di, so doing them together equals the
// reference's one-species-at-a-time order.
// ===========================================================================
// A tile's points, NP (TS + 8), and its interfaces, NP (TS + 1), fit the 256
// threads: a thread owns one point and one interface for the whole species
// loop, and what belongs to them (addresses, split velocities, kinds, old
// interface values) stays in registers.  The sweeps are bound by their vector
// instructions (vector units 0.7 to 0.9 busy); with tiles of 64 and 32 cells
// the loops over points and interfaces took their indexes apart again for
// every species, more than half of the instructions.  160x112x64, nine
// species, us x / y / z: 228 / 202 / 162, now 170 / 151 / 134.
template <int DIR> struct SpTile;
template <> struct SpTile<0> { static constexpr int NP = 4, TS = 56; };
template <> struct SpTile<1> { static constexpr int NP = 8, TS = 24; };
template <> struct SpTile<2> { static constexpr int NP = 8, TS = 24; };

// Reconstruction where the wavefront's lanes mostly agree: ku is their common
// kind (a scalar branch) or -1.
__device__ __forceinline__ double recon_wave(int ku, int kind, const double* w, const double* ud7l) {
  switch (ku) {
    case K_UD7L: return recon(K_UD7L, w, ud7l);
    case K_WENO7: return recon_weno7(w);
    case K_WENO5: return recon_weno5(w, 1);
    case K_OMP6: return recon_omp6(w);
  }
  return recon(kind, w, ud7l);
}
__device__ __forceinline__ int common_kind(int kind, bool on) {
  const unsigned long long m = __ballot(on);
  const int k0 = __builtin_amdgcn_readlane(kind, m ? __builtin_ctzll(m) : 0);
  return wave_all(!on || kind == k0) ? k0 : -1;
}

// gridDim.z blocks share the species of a tile, ng each: see species_groups.
template <int DIR>
__global__ __launch_bounds__(256) void k_species_sweep(DevState S, int ma, int me, int ng) {
  const int m0 = ma + (int)blockIdx.z * ng, m1 = min(me, m0 + ng);
  constexpr int NP = SpTile<DIR>::NP, TS = SpTile<DIR>::TS;
  constexpr int NPT = TS + 8, NIF = TS + 1;
  constexpr int LPS = DIR == 0 ? 1 : NP;  // LDS distance of neighbours along the pencil
  static_assert(NP * NPT <= 256 && NP * NIF <= 256, "one point and one interface a thread");
  // one species at a time: split fluxes of the points, values at the interfaces
  __shared__ double sF[2][NP * NPT];
  __shared__ double sH[2][NP * NIF];
  __shared__ PencilBase<DIR, NP> PB;
  const int n = S.n[DIR];
  const long nb = (long)gridDim.x * gridDim.y;
  const long lb = xcd_block((long)blockIdx.y * gridDim.x + blockIdx.x, nb);
  const int bx = (int)(lb % gridDim.x);
  const long by = lb / gridDim.x;
  const int c0 = bx * TS + 1;
  const int ncell = min(TS, n - c0 + 1);
  const long npen = DIR == 0 ? (long)S.ny * S.nz : DIR == 1 ? (long)S.nx * S.nz : (long)S.nx * S.ny;
  const long pen0 = by * NP;
  const int tid = threadIdx.x;
  pencil_bases<DIR, NP>(S, pen0, npen, PB);
  __syncthreads();
  // the thread's point
  const int ppl = DIR == 0 ? tid / NPT : tid % NP, psl = DIR == 0 ? tid % NPT : tid / NP;
  const bool pon = tid < NP * NPT && pen0 + ppl < npen && psl <= ncell + 7;
  double vp = 0.0, vm = 0.0;
  const double* Dp = S.di;
  if (pon) {
    const double* M1 = DIR == 0 ? S.Akx1 : DIR == 1 ? S.Aix1 : S.Asx1;
    const double* M2 = DIR == 0 ? S.Aky1 : DIR == 1 ? S.Aiy1 : S.Asy1;
    const double* M3 = DIR == 0 ? S.Akz1 : DIR == 1 ? S.Aiz1 : S.Asz1;
    const long q = PB.hq1[ppl] + (long)(wrap(c0 - 4 + psl, n, S.per[DIR]) - 1) * S.sh[DIR];
    const double vs = M1[q] * S.u[q] + M2[q] * S.v[q] + M3[q] * S.w[q];
    vp = 0.5 * (vs + fabs(vs));
    vm = 0.5 * (vs - fabs(vs));
    Dp = S.di + q + (long)m0 * S.nh;
  }
  // the thread's interface, and the cell above it
  const int pl = DIR == 0 ? tid / NIF : tid % NP, l = DIR == 0 ? tid % NIF : tid / NP;
  const bool on = tid < NP * NIF && pen0 + pl < npen && l <= ncell;
  const bool out = on && l < ncell;
  int kp = 0, km = 0;
  double* U = S.dus;
  double aj = 0.0;
  if (on) {
    const int s_if = c0 - 1 + l;
    const int mask = S.scheme == OCFD_SCHEME_HYBRID
                         ? (int)S.mask[DIR][PB.mb[pl] + (long)s_if * mask_stride<DIR>(S)] : 0;
    kp = recon_kind(S, DIR, s_if, 0, mask);
    km = recon_kind(S, DIR, s_if, 1, mask);
    if (out) {
      U = S.dus + PB.iq1[pl] + (long)(c0 + l - 1) * S.si[DIR] + (long)m0 * S.ni;
      if (DIR == 2) aj = S.Ajac[PB.hq1[pl] + (long)(c0 + l - 1) * S.sh[DIR]];
    }
  }
  const int kup = common_kind(kp, on), kum = common_kind(km, on);
  const double h1 = S.h_1[DIR];
  const double* Fp = &sF[0][DIR == 0 ? pl * NPT + l : l * NP + pl];
  const double* Fm = Fp + NP * NPT;
  double* Hp = &sH[0][tid];
  for (int m = m0; m < m1; m++, Dp += S.nh, U += S.ni) {
    double old = 0.0;
    if (DIR != 0 && out) old = *U;  // in flight until the end of the pass
    if (pon) {
      const double fs = *Dp;
      sF[0][tid] = vp * fs;
      sF[1][tid] = vm * fs;
    }
    __syncthreads();  // sF complete; the previous species' outputs have read sH
    double hp0 = 0.0, hm0 = 0.0;
    if (on) {
      double w[8];
#pragma unroll
      for (int qq = 0; qq < 8; qq++) w[qq] = Fp[qq * LPS];
      hp0 = recon_wave(kup, kp, w, S.ud7l);
#pragma unroll
      for (int qq = 0; qq < 8; qq++) w[qq] = Fm[(7 - qq) * LPS];
      hm0 = recon_wave(kum, km, w, S.ud7l);
      Hp[0] = hp0;
      Hp[NP * NIF] = hm0;
    }
    __syncthreads();  // sH complete; sF may be overwritten
    if (out) {
      const double hp1 = Hp[LPS], hm1 = Hp[NP * NIF + LPS];
      const double val = (hp1 - hp0 + hm1 - hm0) * h1;
      if (DIR == 0) *U = val;
      else if (DIR == 1) *U = old + val;
      else *U = -(old + val) * aj;
    }
  }
}

// ===========================================================================
// du_scaler_viscous (OCFD_scaler_viscous.f90:4-79), part 1 for all species:
// grad(c_m) with c_m = di_m/d, the flux rho D_m grad(c_m) in the three
// computational directions, and Qp = sum_m rho D_m h_m grad(c_m) in species
// order (zeroed at the first species).  c_m is formed once per cell by
// k_species_conc (the reference's Ev1 = fs/d, :25-31).
// ===========================================================================
__global__ __launch_bounds__(256) void k_species_conc(DevState S, int m0, int m1) {
  const long c = cell_index();
  if (c >= S.ni) return;
  int i, j, k;
  cell_ijk(S, c, i, j, k);
  const long q = hq(S, i, j, k);
  const double d = S.d[q];
  for (int m = m0; m < m1; m++) S.cs[c + (long)m * S.ni] = S.di[q + (long)m * S.nh] / d;
}

// IX, IY, IZ: the stencils of the cell are central there (no wrap, no
// closure), so each species' derivatives are straight-line code whose loads
// issue together.  Species m0, m0 + step, .. < m1; out takes each one's share
// of Qp.
template <int CD, bool IX, bool IY, bool IZ, class Out>
__device__ __forceinline__ void species_visc_prep_cell(const DevState& S, long c, long q, int i, int j, int k, int m0,
                                                       int m1, int step, Out out) {
  const double T0 = S.T[q], d0 = S.d[q];
  const double Akx = S.Akx[q], Aky = S.Aky[q], Akz = S.Akz[q];
  const double Aix = S.Aix[q], Aiy = S.Aiy[q], Aiz = S.Aiz[q];
  const double Asx = S.Asx[q], Asy = S.Asy[q], Asz = S.Asz[q];
  const double Akx1 = S.Akx1[q], Aky1 = S.Aky1[q], Akz1 = S.Akz1[q];
  const double Aix1 = S.Aix1[q], Aiy1 = S.Aiy1[q], Aiz1 = S.Aiz1[q];
  const double Asx1 = S.Asx1[q], Asy1 = S.Asy1[q], Asz1 = S.Asz1[q];
  const long ni = S.ni;
  for (int m = m0; m < m1; m += step) {
    const double* C = S.cs + (long)m * ni + c;
    auto dc = [&](auto central, int dir, int s) {
      const long st = S.si[dir];
      if constexpr (decltype(central)::value) {
        return deriv1<CD, true>(S, dir, s, [&](int o) { return C[o * st]; });
      } else {
        return deriv1<CD>(S, dir, s, [&](int o) {
          const int t = wrap(s + o, S.n[dir], S.per[dir]);
          return C[(t - s) * st];
        });
      }
    };
    const double uk = dc(std::bool_constant<IX>{}, 0, i), ui = dc(std::bool_constant<IY>{}, 1, j),
                 us = dc(std::bool_constant<IZ>{}, 2, k);
    const double dD = d0 * S.AmD[c + (long)m * ni];
    const double hi = gas_hi(m, T0);
    const double cix = uk * Akx + ui * Aix + us * Asx;
    const double ciy = uk * Aky + ui * Aiy + us * Asy;
    const double ciz = uk * Akz + ui * Aiz + us * Asz;
    const double E1 = dD * cix, E2 = dD * ciy, E3 = dD * ciz;
    out(m, E1 * hi, E2 * hi, E3 * hi);
    S.Evs[c + (long)(3 * m) * ni] = E1 * Akx1 + E2 * Aky1 + E3 * Akz1;
    S.Evs[c + (long)(3 * m + 1) * ni] = E1 * Aix1 + E2 * Aiy1 + E3 * Aiz1;
    S.Evs[c + (long)(3 * m + 2) * ni] = E1 * Asx1 + E2 * Asy1 + E3 * Asz1;
  }
}

template <int CD, class Out>
__device__ __forceinline__ void species_visc_prep_at(const DevState& S, long c, int m0, int m1, int step, Out out) {
  constexpr int R = CD == 1 ? 4 : 3;
  int i, j, k;
  cell_ijk(S, c, i, j, k);
  const long q = hq(S, i, j, k);
  // central forms per direction: a wavefront at the xi faces keeps the
  // central eta and zeta forms
  const bool ix = wave_all(central_cell(i, S.nx, R));
  const bool iyz = wave_all(central_cell(j, S.ny, R) && central_cell(k, S.nz, R));
  if (ix && iyz) species_visc_prep_cell<CD, true, true, true>(kernarg_again(S), c, q, i, j, k, m0, m1, step, out);
  else if (iyz) species_visc_prep_cell<CD, false, true, true>(kernarg_again(S), c, q, i, j, k, m0, m1, step, out);
  else species_visc_prep_cell<CD, false, false, false>(kernarg_again(S), c, q, i, j, k, m0, m1, step, out);
}

// Species m0 .. m1-1, one thread per cell.  Qp starts from zero at the first
// species (m0 = 0) and from its stored value otherwise, so species taken one
// at a time add up in the same order as all at once.
template <int CD>
__global__ __launch_bounds__(256) void k_species_visc_prep(DevState S, int m0, int m1) {
  const long c = cell_index();
  if (c >= S.ni) return;
  double Q[3] = {0.0, 0.0, 0.0};
  if (m0 > 0) {
#pragma unroll
    for (int a = 0; a < 3; a++) Q[a] = S.Qp[c + a * S.ni];
  }
  species_visc_prep_at<CD>(S, c, m0, m1, 1, [&](int, double x, double y, double z) {
    Q[0] = Q[0] + x;
    Q[1] = Q[1] + y;
    Q[2] = Q[2] + z;
  });
#pragma unroll
  for (int a = 0; a < 3; a++) S.Qp[c + a * S.ni] = Q[a];
}

// ... all species of 64 cells by three wavefronts, every third species each:
// for grids that would leave most wavefront slots empty (species_groups;
// 48x36x36: 36 us with one thread a cell, 25 so).  The shares of Qp meet in
// LDS and are added in the species' order, one component a wavefront.
template <int CD>
__global__ __launch_bounds__(192) void k_species_visc_prep3(DevState S) {
  __shared__ double sQ[OCFD_NS_MAX][3][64];
  const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  const long c = xcd_block(blockIdx.x, gridDim.x) * 64 + lane;
  const bool in = c < S.ni;
  if (in)
    species_visc_prep_at<CD>(S, c, w, S.ns, 3, [&](int m, double x, double y, double z) {
      sQ[m][0][lane] = x;
      sQ[m][1][lane] = y;
      sQ[m][2][lane] = z;
    });
  __syncthreads();
  if (!in) return;
  double Q = 0.0;
  for (int m = 0; m < S.ns; m++) Q = Q + sQ[m][w][lane];
  S.Qp[c + w * S.ni] = Q;
}

// Species update: Dus += div(diffusive flux) Ajac (OCFD_scaler_viscous.f90:67-77)
// and Scalar_time_adv_RK3 (OCFD_Time_Adv.f90:134-166) for every species;
// krk = 0 stores the complete right-hand side in dus instead.
template <int CD, bool IX, bool IY, bool IZ>
__device__ __forceinline__ void species_rk_cell(const DevState& S, long c, long q, int i, int j, int k, int krk,
                                                double dt, int visc, int save, int m0, int m1) {
  const long ni = S.ni;
  const double ajac = S.Ajac[q];
  auto dv = [&](auto central, const double* F, int dir, int s) {
    const double* Fc = F + c;
    const long st = S.si[dir];
    if constexpr (decltype(central)::value) {
      return deriv1<CD, true>(S, dir, s, [&](int o) { return Fc[o * st]; });
    } else {
      return deriv1<CD>(S, dir, s, [&](int o) {
        const int t = wrap(s + o, S.n[dir], S.per[dir]);
        return Fc[(t - s) * st];
      });
    }
  };
  const double ra = krk == 2 ? 3.0 / 4.0 : 1.0 / 3.0;
  const double rb = krk == 2 ? 1.0 / 4.0 : 2.0 / 3.0;
  for (int m = m0; m < m1; m++) {
    const long qm = q + (long)m * S.nh, cm = c + (long)m * ni;
    // the stage's old values, read with the stencil loads
    const double dn = save ? S.di[qm] : krk >= 1 ? S.din[cm] : 0.0;
    if (save) S.din[cm] = dn;
    const double dold = krk >= 2 ? S.di[qm] : 0.0;
    double val = S.dus[cm];
    if (visc) {
      const double uk = dv(std::bool_constant<IX>{}, S.Evs + (long)(3 * m) * ni, 0, i);
      const double ui = dv(std::bool_constant<IY>{}, S.Evs + (long)(3 * m + 1) * ni, 1, j);
      const double us = dv(std::bool_constant<IZ>{}, S.Evs + (long)(3 * m + 2) * ni, 2, k);
      val = val + (uk + ui + us) * ajac;
    }
    if (krk == 0) {  // right-hand side only
      S.dus[cm] = val;
      continue;
    }
    if (krk == 1) S.di[qm] = dn + dt * val;
    else S.di[qm] = ra * dn + rb * (dold + dt * val);
  }
}

// save: the stage opens a step, which starts from din = di, kept here from the
// di that the update reads.  gridDim.y blocks share the species, ng each.
template <int CD>
__global__ __launch_bounds__(256) void k_species_rk(DevState S, int krk, double dt, int visc, int save, int ma, int me,
                                                    int ng) {
  constexpr int R = CD == 1 ? 4 : 3;
  const int m0 = ma + (int)blockIdx.y * ng, m1 = min(me, m0 + ng);
  const long c = cell_index();
  if (c >= S.ni) return;
  int i, j, k;
  cell_ijk(S, c, i, j, k);
  const long q = hq(S, i, j, k);
  const bool ix = wave_all(central_cell(i, S.nx, R));
  const bool iyz = wave_all(central_cell(j, S.ny, R) && central_cell(k, S.nz, R));
  if (ix && iyz) species_rk_cell<CD, true, true, true>(kernarg_again(S), c, q, i, j, k, krk, dt, visc, save, m0, m1);
  else if (iyz) species_rk_cell<CD, false, true, true>(kernarg_again(S), c, q, i, j, k, krk, dt, visc, save, m0, m1);
  else species_rk_cell<CD, false, false, false>(kernarg_again(S), c, q, i, j, k, krk, dt, visc, save, m0, m1);
}

// The two kernels above for large grids, all species: a workgroup takes 32 x
// 8 cells of a plane and fetches a species' values once, its own by every
// thread and the R cells around the tile by most; the xi and eta taps come
// from LDS.  With every tap a load of its own the kernels were bound by the
// address and data path of the vector cache (19 loads a species and cell, and
// each wavefront load of 512 bytes off a line's start takes twice the cycles).
// The next species' values are in flight while this one's are used; two
// buffers, so one barrier a species.  Tiles in the order of bricks
// (brick_cell), so that the planes of the zeta taps are in the L2 together.
// 160x112x64, nine species, us before / now: viscous preparation 303 / 197,
// update 240 / 145 (of which the order of the tiles is about a tenth).
constexpr int ST_X = 32, ST_Y = 8;
template <int R>
struct SpeciesTile {
  static constexpr int LX = ST_X + 2 * R, LY = ST_Y + 2 * R, NH = 2 * R * (ST_X + ST_Y), NT = (NH + 255) / 256;
  int i, j, k;
  bool act;            // a cell of the grid
  long own;            // source of the thread's position (periodic images included), -1: none
  long src[NT];        // ... of its positions around the tile: eta below ST_X * 2 R, then xi
  int pos[NT];         // their places in an LY x LX array
  __device__ __forceinline__ void init(const DevState& S) {
    const int nti = (S.nx + ST_X - 1) / ST_X, ntj = (S.ny + ST_Y - 1) / ST_Y;
    const int lb = (int)xcd_block((long)blockIdx.x, (long)gridDim.x);
    const int zg = lb / (nti * ntj * BRICK_Z), r = lb - zg * (nti * ntj * BRICK_Z);
    const int zc = min(BRICK_Z, S.nz - zg * BRICK_Z);
    const int tj = r / (nti * zc), r2 = r - tj * (nti * zc), kk = r2 / nti;
    k = zg * BRICK_Z + kk + 1;
    const int i0 = (r2 - kk * nti) * ST_X + 1, j0 = tj * ST_Y + 1;
    auto source = [&](int a, int b) {
      const int ii = wrap(a, S.nx, S.per[0]), jj = wrap(b, S.ny, S.per[1]);
      return ii >= 1 && ii <= S.nx && jj >= 1 && jj <= S.ny ? iq(S, ii, jj, k) : -1L;
    };
    const int lx = (int)threadIdx.x % ST_X, ly = (int)threadIdx.x / ST_X;
    i = i0 + lx;
    j = j0 + ly;
    act = i <= S.nx && j <= S.ny;
    own = source(i, j);
#pragma unroll
    for (int a = 0; a < NT; a++) {
      const int e = (int)threadIdx.x + 256 * a;
      int x, y;
      if (e < 2 * R * ST_X) {
        const int h = e / ST_X;
        x = e % ST_X;
        y = h < R ? h - R : ST_Y + h - R;
      } else {
        const int f = e - 2 * R * ST_X, h = f % (2 * R);
        y = f / (2 * R);
        x = h < R ? h - R : ST_X + h - R;
      }
      src[a] = e < NH ? source(i0 + x, j0 + y) : -1L;
      pos[a] = (y + R) * LX + x + R;
    }
  }
  __device__ __forceinline__ static bool eta_item(int a) { return (int)threadIdx.x + 256 * a < 2 * R * ST_X; }
  __device__ __forceinline__ static int place() {
    return ((int)threadIdx.x / ST_X + R) * LX + (int)threadIdx.x % ST_X + R;
  }
};
inline dim3 species_tiles(const DevState& S) {
  return dim3((unsigned)((long)((S.nx + ST_X - 1) / ST_X) * ((S.ny + ST_Y - 1) / ST_Y) * S.nz));
}

// the zeta taps -R .. R of the field at C, ahead of their use (central cells)
template <int CD, int R>
__device__ __forceinline__ void zeta_taps(const double* C, long st, double* z) {
#pragma unroll
  for (int o = -R; o <= R; o++)
    if (o != 0) z[o + R] = C[o * st];
}

template <int CD>
__global__ __launch_bounds__(256) void k_species_visc_tile(DevState S) {
  constexpr int R = CD == 1 ? 4 : 3;
  typedef SpeciesTile<R> Tile;
  __shared__ double sC[2][Tile::LY * Tile::LX];
  Tile t;
  t.init(S);
  const int i = t.i, j = t.j, k = t.k, at = Tile::place();
  // lanes beyond the grid compute on the plane's first cell and write nothing
  const long ni = S.ni, c = t.act ? t.own : iq(S, 1, 1, k), q = t.act ? hq(S, i, j, k) : hq(S, 1, 1, k);
  const bool ix = wave_all(!t.act || S.per[0] || central_cell(i, S.nx, R));
  const bool iy = wave_all(!t.act || S.per[1] || central_cell(j, S.ny, R));
  const bool iz = central_cell(k, S.nz, R);
  const double T0 = S.T[q], d0 = S.d[q];
  const double Akx = S.Akx[q], Aky = S.Aky[q], Akz = S.Akz[q];
  const double Aix = S.Aix[q], Aiy = S.Aiy[q], Aiz = S.Aiz[q];
  const double Asx = S.Asx[q], Asy = S.Asy[q], Asz = S.Asz[q];
  const double Akx1 = S.Akx1[q], Aky1 = S.Aky1[q], Akz1 = S.Akz1[q];
  const double Aix1 = S.Aix1[q], Aiy1 = S.Aiy1[q], Aiz1 = S.Aiz1[q];
  const double Asx1 = S.Asx1[q], Asy1 = S.Asy1[q], Asz1 = S.Asz1[q];
  double own = 0.0, halo[Tile::NT];
  auto fetch = [&](int m) {
    const double* F = S.cs + (long)m * ni;
    own = t.own >= 0 ? F[t.own] : 0.0;
#pragma unroll
    for (int a = 0; a < Tile::NT; a++) halo[a] = t.src[a] >= 0 ? F[t.src[a]] : 0.0;
  };
  fetch(0);
  double Qx = 0.0, Qy = 0.0, Qz = 0.0;
  for (int m = 0; m < S.ns; m++) {
    double* B = sC[m & 1];
    B[at] = own;
#pragma unroll
    for (int a = 0; a < Tile::NT; a++)
      if ((int)threadIdx.x + 256 * a < Tile::NH) B[t.pos[a]] = halo[a];
    if (m + 1 < S.ns) fetch(m + 1);
    const double* C = S.cs + (long)m * ni + c;
    double z[2 * R + 1];
    if (iz) zeta_taps<CD, R>(C, S.si[2], z);
    const double AmD = S.AmD[c + (long)m * ni];
    __syncthreads();
    auto tx = [&](int o) { return B[at + o]; };
    auto ty = [&](int o) { return B[at + o * Tile::LX]; };
    const double uk = ix ? deriv1<CD, true>(S, 0, i, tx) : deriv1<CD>(S, 0, i, tx);
    const double ui = iy ? deriv1<CD, true>(S, 1, j, ty) : deriv1<CD>(S, 1, j, ty);
    const double us = iz ? deriv1<CD, true>(S, 2, k, [&](int o) { return z[o + R]; })
                         : deriv1<CD>(S, 2, k, [&](int o) {
                             const int s = wrap(k + o, S.nz, S.per[2]);
                             return C[(s - k) * S.si[2]];
                           });
    const double dD = d0 * AmD;
    const double hi = gas_hi(m, T0);
    const double cix = uk * Akx + ui * Aix + us * Asx;
    const double ciy = uk * Aky + ui * Aiy + us * Asy;
    const double ciz = uk * Akz + ui * Aiz + us * Asz;
    const double E1 = dD * cix, E2 = dD * ciy, E3 = dD * ciz;
    Qx = Qx + E1 * hi;
    Qy = Qy + E2 * hi;
    Qz = Qz + E3 * hi;
    if (t.act) {
      S.Evs[c + (long)(3 * m) * ni] = E1 * Akx1 + E2 * Aky1 + E3 * Akz1;
      S.Evs[c + (long)(3 * m + 1) * ni] = E1 * Aix1 + E2 * Aiy1 + E3 * Aiz1;
      S.Evs[c + (long)(3 * m + 2) * ni] = E1 * Asx1 + E2 * Asy1 + E3 * Asz1;
    }
  }
  if (!t.act) return;
  S.Qp[c] = Qx;
  S.Qp[c + ni] = Qy;
  S.Qp[c + 2 * ni] = Qz;
}

template <int CD>
__global__ __launch_bounds__(256) void k_species_rk_tile(DevState S, int krk, double dt, int save) {
  constexpr int R = CD == 1 ? 4 : 3;
  typedef SpeciesTile<R> Tile;
  __shared__ double sE[2][2][Tile::LY * Tile::LX];  // the xi and the eta flux
  Tile t;
  t.init(S);
  const int i = t.i, j = t.j, k = t.k, at = Tile::place();
  // lanes beyond the grid compute on the plane's first cell and write nothing
  const long ni = S.ni, c = t.act ? t.own : iq(S, 1, 1, k), q = t.act ? hq(S, i, j, k) : hq(S, 1, 1, k);
  const bool ix = wave_all(!t.act || S.per[0] || central_cell(i, S.nx, R));
  const bool iy = wave_all(!t.act || S.per[1] || central_cell(j, S.ny, R));
  const bool iz = central_cell(k, S.nz, R);
  const double ajac = S.Ajac[q];
  const double ra = krk == 2 ? 3.0 / 4.0 : 1.0 / 3.0;
  const double rb = krk == 2 ? 1.0 / 4.0 : 2.0 / 3.0;
  double ox = 0.0, oy = 0.0, halo[Tile::NT];
  auto fetch = [&](int m) {
    const double* X = S.Evs + (long)(3 * m) * ni;
    const double* Y = X + ni;
    ox = t.own >= 0 ? X[t.own] : 0.0;
    oy = t.own >= 0 ? Y[t.own] : 0.0;
#pragma unroll
    for (int a = 0; a < Tile::NT; a++) halo[a] = t.src[a] >= 0 ? (Tile::eta_item(a) ? Y : X)[t.src[a]] : 0.0;
  };
  fetch(0);
  for (int m = 0; m < S.ns; m++) {
    double(*B)[Tile::LY * Tile::LX] = sE[m & 1];
    B[0][at] = ox;
    B[1][at] = oy;
#pragma unroll
    for (int a = 0; a < Tile::NT; a++)
      if ((int)threadIdx.x + 256 * a < Tile::NH) B[Tile::eta_item(a)][t.pos[a]] = halo[a];
    if (m + 1 < S.ns) fetch(m + 1);
    const long qm = q + (long)m * S.nh, cm = c + (long)m * ni;
    const double* Z = S.Evs + (long)(3 * m + 2) * ni + c;
    double z[2 * R + 1];
    if (iz) zeta_taps<CD, R>(Z, S.si[2], z);
    // the stage's old values
    const double dn = save ? S.di[qm] : krk >= 1 ? S.din[cm] : 0.0;
    const double dold = krk >= 2 ? S.di[qm] : 0.0;
    double val = S.dus[cm];
    __syncthreads();
    auto tx = [&](int o) { return B[0][at + o]; };
    auto ty = [&](int o) { return B[1][at + o * Tile::LX]; };
    const double uk = ix ? deriv1<CD, true>(S, 0, i, tx) : deriv1<CD>(S, 0, i, tx);
    const double ui = iy ? deriv1<CD, true>(S, 1, j, ty) : deriv1<CD>(S, 1, j, ty);
    const double us = iz ? deriv1<CD, true>(S, 2, k, [&](int o) { return z[o + R]; })
                         : deriv1<CD>(S, 2, k, [&](int o) {
                             const int s = wrap(k + o, S.nz, S.per[2]);
                             return Z[(s - k) * S.si[2]];
                           });
    val = val + (uk + ui + us) * ajac;
    if (t.act) {
      if (save) S.din[cm] = dn;
      if (krk == 0) S.dus[cm] = val;  // right-hand side only
      else if (krk == 1) S.di[qm] = dn + dt * val;
      else S.di[qm] = ra * dn + rb * (dold + dt * val);
    }
  }
}

// Rescaling_di (Comput_flow_variables.f90:101-121) and comput_T_P (:32-46)
// of one cell, given the new density and internal energy.
__device__ __forceinline__ void ms_prims(const DevState& S, long q, double dd, double Et, double& T, double& p) {
  double di[OCFD_NS_MAX];
  double d0 = 0.0;
  each_species([&](int m) {
    double x = S.di[q + (long)m * S.nh];
    if (x < 0.0) x = 0.0;
    di[m] = x;
    d0 = d0 + x;
  });
  const double tmp = dd / d0;
  each_species([&](int m) {
    di[m] = di[m] * tmp;
    S.di[q + (long)m * S.nh] = di[m];
  });
  T = gas_T(di, Et);
  p = gas_P(di, T);
}

// comput_T_P over the interior (after the chemistry substeps, OCFD_NS_Solver.f90:34)
__global__ __launch_bounds__(256) void k_comput_T_P(DevState S) {
  const long c = cell_index();
  if (c >= S.ni) return;
  int i, j, k;
  cell_ijk(S, c, i, j, k);
  const long q = hq(S, i, j, k);
  double di[OCFD_NS_MAX];
  each_species([&](int m) { di[m] = S.di[q + (long)m * S.nh]; });
  const double T = gas_T(di, S.Et[q]);
  S.T[q] = T;
  S.p[q] = gas_P(di, T);
}

// Face re-synthesis (OCFD_BC.f90:33-56) for N_SPEC > 1
__device__ __forceinline__ void face_update_ms(const DevState& S, long q, long c) {
  double di[OCFD_NS_MAX];
  double d0 = 0.0;
  each_species([&](int m) {
    di[m] = S.di[q + (long)m * S.nh];
    d0 = d0 + di[m];
  });
  const double dtmp = S.d[q] / d0;
  each_species([&](int m) {
    di[m] = di[m] * dtmp;
    S.di[q + (long)m * S.nh] = di[m];
  });
  const double T = S.T[q];
  const double Et = gas_E(di, T);
  const double p = gas_P(di, T);
  S.Et[q] = Et;
  S.p[q] = p;
  const double dd = S.d[q], uu = S.u[q], vv = S.v[q], ww = S.w[q];
  S.f[c] = dd;
  S.f[c + S.ni] = dd * uu;
  S.f[c + 2 * S.ni] = dd * vv;
  S.f[c + 3 * S.ni] = dd * ww;
  S.f[c + 4 * S.ni] = Et + dd * (uu * uu + vv * vv + ww * ww) * 0.5;
}

// ocfd_bc_jet inflow (OCFD_BC_jet.f90:22-73): Dirichlet data, or (BC_Para(1)=1)
// the pressure of i=2 where the inflow is subsonic
__device__ __forceinline__ void jet_inlet(const DevState& S, int j, int k) {
  const long q = hq(S, 1, j, k), pl = (long)S.ny * S.nz, r = (j - 1) + (long)S.ny * (k - 1);
  const double* in = S.jet_in;
  if (S.jet_iflag == 0) {
    S.d[q] = in[r]; S.u[q] = in[r + pl]; S.v[q] = in[r + 2 * pl]; S.w[q] = in[r + 3 * pl]; S.T[q] = in[r + 4 * pl];
    each_species([&](int m) { S.di[q + (long)m * S.nh] = in[r + (5L + m) * pl]; });
    return;
  }
  S.u[q] = in[r + pl]; S.v[q] = in[r + 2 * pl]; S.w[q] = in[r + 3 * pl]; S.T[q] = in[r + 4 * pl];
  const double d1 = in[r];
  double di1[OCFD_NS_MAX], ai1[OCFD_NS_MAX];
  double d0 = 0.0;
  each_species([&](int m) {
    di1[m] = in[r + (5L + m) * pl];
    d0 = d0 + di1[m];
  });
  each_species([&](int m) { ai1[m] = di1[m] / d0; });
  const double T1 = S.T[q];
  const double p1 = gas_P(di1, T1);
  const double Et1 = gas_E(di1, T1);
  const double gamma = p1 / Et1 + 1.0;  // comput_soundspeed, CHEM_thermdyn.f90:412-418
  const double c1 = sqrt(gamma * p1 / d1);
  if (S.u[q] < c1) {
    S.p[q] = S.p[hq(S, 2, j, k)];
    const double d1new = gas_d(ai1, T1, S.p[q]);
    S.d[q] = d1new;
    each_species([&](int m) { S.di[q + (long)m * S.nh] = d1new * ai1[m]; });
  } else {
    S.d[q] = d1;
    each_species([&](int m) { S.di[q + (long)m * S.nh] = di1[m]; });
  }
}

// ocfd_bc_jet outflow (OCFD_BC_jet.f90:76-93): zeroth-order extrapolation
__device__ __forceinline__ void jet_outlet(const DevState& S, int j, int k) {
  const long q = hq(S, S.nx, j, k), qa = hq(S, S.nx - 1, j, k);
  S.d[q] = S.d[qa]; S.u[q] = S.u[qa]; S.v[q] = S.v[qa]; S.w[q] = S.w[qa];
  S.T[q] = S.T[qa]; S.p[q] = S.p[qa]; S.Et[q] = S.Et[qa];
  each_species([&](int m) { S.di[q + (long)m * S.nh] = S.di[qa + (long)m * S.nh]; });
}

// Chemistry coupling (Chemical_time_advance, OCFD_Time_Adv.f90:169-196):
// interior di, Et -> batch [ns][interior], E, dt ...
__global__ __launch_bounds__(256) void k_chem_pack(DevState S, double* rho, double* E, double* dtb, double dt2) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= S.ni) return;
  int i, j, k;
  cell_ijk(S, c, i, j, k);
  const long q = hq(S, i, j, k);
  for (int m = 0; m < S.ns; m++) rho[(long)m * S.ni + c] = S.di[q + (long)m * S.nh];
  E[c] = S.Et[q];
  dtb[c] = dt2;
}

// ... and back: di = batch, f5 += Et1 - Et0, Et = Et1
__global__ __launch_bounds__(256) void k_chem_unpack(DevState S, const double* rho, const double* E) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= S.ni) return;
  int i, j, k;
  cell_ijk(S, c, i, j, k);
  const long q = hq(S, i, j, k);
  for (int m = 0; m < S.ns; m++) S.di[q + (long)m * S.nh] = rho[(long)m * S.ni + c];
  const double Et1 = E[c], Et0 = S.Et[q];
  S.f[c + 4 * S.ni] = S.f[c + 4 * S.ni] + (Et1 - Et0);
  S.Et[q] = Et1;
}
