// ocfd_chem_core.h -- the chemistry's device arithmetic: mechanism bank,
// temperature, rates, Jacobian, the implicit solve and one step or attempt of
// each integrator (chemical_timeAdv, CHEM_reactions.f90:374-602).  Included
// once, by ocfd_chem.hip; the per-lane kernels and the one-cell-per-wavefront
// kernel share these functions, so their results agree bit for bit.
//
// What bounds an attempt is its own instruction stream: a stiff cell's
// attempts follow one another (up to about 190 on a jet-flame batch), and one
// wave per SIMD has nothing else to issue.  So the mechanism is laid out for
// few instructions (on MI355X, 9 species / 19 reactions: ChemH2 about 4,100
// issued per attempt, 10 us alone on a SIMD and 15 us for two waves, ChemAny
// 9,100, 29 and 38 us; with the reference's expressions as they stand about
// 40,000 and 82 us):
//   - one exponential per Arrhenius set (chem_arr) instead of pow and exp;
//   - every constant division, the molar-mass ratios and the NASA/R products
//     folded into the bank on the host;
//   - stoichiometry as doubles in scalar registers: a reaction adds nu_i * x
//     to every row in straight-line FMAs, and only the columns of its own
//     species are visited (a bit mask), instead of a scalar branch per entry;
//   - concentrations in LDS, one column per lane, so that a reaction takes
//     its species by a uniform index;
//   - one reciprocal per pivot column, row exchanges only where a lane of
//     the wavefront needs one.
// FMAs are explicit (-ffp-contract=off); sums keep the reference's order of
// species and reactions.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "ocfd_exp.h"

#define CH_NS 9
#define CH_NR_MAX 32
#define CH_NT_MAX 4
#define CH_R0 8.314
#define CH_ATM 1.013e5

// One reaction (read_Reac, CHEM_reactions.f90:15-71).
struct ChemRx {
  double nu[CH_NS];                // vr - vf
  double vf[CH_NS], vr[CH_NS];
  double eff[CH_NS];               // third-body efficiencies
  double a0, b0, e0, a1, b1, e1;   // Arrhenius sets
  double lfc, ac, an;              // Troe: log10 Fc and the two constants formed from it
  double r[5];                     // ReReac 1: A_r, b_r, E_r; ReReac 2: A1r..A5r
  // the species of the forward / reverse mass-action products, one byte
  // each in ascending order, as often as their order (slot CH_NS holds 1 and
  // fills the first CH_SLOTS); count -1: an order that does not fit (ipow)
  unsigned long long sf, sr;
  int nsf, nsr;
  int af_type, tb, sgm, part;      // part: bit j set when species j takes part
};
constexpr int CH_SLOTS = 3;

struct ChemMech {
  int ns, nr, n_tct, rereac;
  double tct[CH_NT_MAX], tct_max;
  double mi[CH_NS], ri[CH_NS];
  double ci6[CH_NS];               // 1e-6 / mi: partial density -> mol/cm3
  double rf[CH_NS];                // ri * coef[.][0][5] (update_Et)
  double rcv[CH_NS];               // 2.5 ri
  double ev[CH_NT_MAX][6][CH_NS];  // (A-1) R, B R, C R, D R, E R, Ect R of each range
  double gb[CH_NS][CH_NT_MAX][7];  // A, B/2, C/6, D/12, E/20, F, G (comput_gibbs)
  double coef[CH_NS][CH_NT_MAX][7];
  double exp2t[64][2];             // 2^(j/64) and its rounding, for chem_exp
  ChemRx rx[CH_NR_MAX];
};

__constant__ ChemMech cm;

// The mechanism as seen by the device functions: a pointer into the constant
// bank (address space 4, so loads through it are scalar loads).  The kernels
// pass it through an empty asm statement at the top of every substep; the
// compiler then cannot hoist the hundreds of constant loads of the rate and
// thermo code out of the substep loop into registers, which otherwise
// exhausts the register file and spills.
#define CH_CONST __attribute__((address_space(4)))
typedef const CH_CONST ChemMech* Mech;
__device__ __forceinline__ Mech mech_opaque(Mech m) {
  asm volatile("" : "+s"(m));
  return m;
}

__device__ __forceinline__ double q2(double x) { return x * x; }
__device__ __forceinline__ double q3(double x) { double x2 = x * x; return x2 * x; }
__device__ __forceinline__ double q4(double x) { double x2 = x * x; return x2 * x2; }
__device__ __forceinline__ double q5(double x) { double x2 = x * x; return (x2 * x2) * x; }
__device__ __forceinline__ double fm(double a, double b, double c) { return __builtin_fma(a, b, c); }
// a / b given r = 1 / b: the quotient's remainder corrects it to the last bit
__device__ __forceinline__ double div_r(double a, double b, double r) {
  const double q = a * r;
  return fm(fm(-b, q, a), r, q);
}

// Fortran x**n for an integer n (repeated squaring; negative n -> 1/x**|n|)
__device__ __forceinline__ double ipow(double x, int n) {
  if (n == 0) return 1.0;
  int m = n < 0 ? -n : n;
  double r = 1.0, b = x;
  bool first = true;
  while (m) {
    if (m & 1) { r = first ? b : r * b; first = false; }
    m >>= 1;
    if (m) b = b * b;
  }
  return n < 0 ? 1.0 / r : r;
}

// ---------------------------------------------------------------------------
// Stoichiometry known when the kernels are compiled.  The kernels take it as
// a template argument: ChemAny reads the bank (any mechanism with Gibbs reverse
// rates), ChemRev is ChemAny for the other reverse rates, ChemH2 is the
// structure of the shipped 9-species / 19-reaction H2-O2 mechanism -- which
// species take part in which reaction, its third bodies and falloffs, and
// which Arrhenius exponents are zero, two temperature ranges.  The numbers (A, b, E, efficiencies,
// thermodynamics) stay in the bank either way; ocfd_chem_set_mechanism
// compares the structure it is given with ChemH2 and picks the kernels.  With
// it known, a reaction is straight-line code over its own species only, the
// scheduler overlaps neighbouring reactions and the species that never react
// drop out of the linear system.  ChemH2 against ChemAny, ms: 300,007 cells,
// five point-implicit steps 0.23 / 0.53; adaptive batches of 50,021 cells
// 1.71 / 2.42 and 2,097,152 cells 4.06 / 8.01; 1000 cells, five Euler steps
// 0.037 / 0.096.  Both give the same bits (what is left out adds zeros).
// ---------------------------------------------------------------------------
struct ChemAny {
  static constexpr bool FIXED = false, ANYT = false;
  static constexpr int NR = 0, NA = CH_NS, NT = 0;
};
// ReReac 1 and 2 give numbers at temperatures that are no ordinary ones (chem_arr);
// kernels of their own, since the loop for them costs the others up to 5%
struct ChemRev : ChemAny {
  static constexpr bool ANYT = true;
};
struct ChemH2 {
  static constexpr bool FIXED = true, ANYT = false;
  static constexpr int NR = 19, NA = 8, NT = 2;  // reactions; species 0 .. NA-1 react (N2 does not); T ranges
  // af_type, third body, bits: 1 b0, 2 e0, 4 b1, 8 e1 not zero
  static constexpr int af[NR] = {0, 0, 0, 0, 0, 0, 0, 0, 1, 0, 0, 0, 0, 2, 1, 0, 0, 0, 2};
  static constexpr int tb[NR] = {0, 0, 0, 0, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0, 1, 0, 0, 0, 0};
  static constexpr int ar[NR] = {3, 3, 3, 3, 3, 1, 1, 1, 7, 2, 2, 0, 2, 10, 10, 2, 2, 3, 8};
  // order of each species O, O2, H2, H2O, OH, H, HO2, H2O2, N2
  static constexpr int vf[NR][CH_NS] = {
      {0, 1, 0, 0, 0, 1, 0, 0, 0}, {1, 0, 1, 0, 0, 0, 0, 0, 0}, {0, 0, 1, 0, 1, 0, 0, 0, 0}, {1, 0, 0, 1, 0, 0, 0, 0, 0},
      {0, 0, 1, 0, 0, 0, 0, 0, 0}, {2, 0, 0, 0, 0, 0, 0, 0, 0}, {1, 0, 0, 0, 0, 1, 0, 0, 0}, {0, 0, 0, 0, 1, 1, 0, 0, 0},
      {0, 1, 0, 0, 0, 1, 0, 0, 0}, {0, 0, 0, 0, 0, 1, 1, 0, 0}, {0, 0, 0, 0, 0, 1, 1, 0, 0}, {1, 0, 0, 0, 0, 0, 1, 0, 0},
      {0, 0, 0, 0, 1, 0, 1, 0, 0}, {0, 0, 0, 0, 0, 0, 2, 0, 0}, {0, 0, 0, 0, 0, 0, 0, 1, 0}, {0, 0, 0, 0, 0, 1, 0, 1, 0},
      {0, 0, 0, 0, 0, 1, 0, 1, 0}, {1, 0, 0, 0, 0, 0, 0, 1, 0}, {0, 0, 0, 0, 1, 0, 0, 1, 0}};
  static constexpr int vr[NR][CH_NS] = {
      {1, 0, 0, 0, 1, 0, 0, 0, 0}, {0, 0, 0, 0, 1, 1, 0, 0, 0}, {0, 0, 0, 1, 0, 1, 0, 0, 0}, {0, 0, 0, 0, 2, 0, 0, 0, 0},
      {0, 0, 0, 0, 0, 2, 0, 0, 0}, {0, 1, 0, 0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 1, 0, 0, 0, 0}, {0, 0, 0, 1, 0, 0, 0, 0, 0},
      {0, 0, 0, 0, 0, 0, 1, 0, 0}, {0, 1, 1, 0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 2, 0, 0, 0, 0}, {0, 1, 0, 0, 1, 0, 0, 0, 0},
      {0, 1, 0, 1, 0, 0, 0, 0, 0}, {0, 1, 0, 0, 0, 0, 0, 1, 0}, {0, 0, 0, 0, 2, 0, 0, 0, 0}, {0, 0, 0, 1, 1, 0, 0, 0, 0},
      {0, 0, 1, 0, 0, 0, 1, 0, 0}, {0, 0, 0, 0, 1, 0, 1, 0, 0}, {0, 0, 0, 1, 0, 0, 1, 0, 0}};
  static constexpr int sgm(int k) {
    int s = 0;
    for (int i = 0; i < CH_NS; i++) s += vr[k][i] - vf[k][i];
    return s;
  }
};

// comput_T_rgas, CHEM_thermdyn.f90:326-382 (Newton, 1e-3 K, <= 31 iterations),
// the polynomials in Horner form
template <class ST = ChemAny>
__device__ __forceinline__ double chem_T(Mech m, const double* di, double E) {
  constexpr int NT = ST::NT ? ST::NT : CH_NT_MAX;  // a fixed count needs no test per range
  double s[NT][6];
#pragma unroll
  for (int j = 0; j < NT; j++) {
#pragma unroll
    for (int a = 0; a < 6; a++) s[j][a] = 0.0;
    if (ST::NT || j < m->n_tct) {
#pragma unroll
      for (int k = 0; k < CH_NS; k++)
#pragma unroll
        for (int a = 0; a < 6; a++) s[j][a] = fm(m->ev[j][a][k], di[k], s[j][a]);
    }
  }
  const double tm = m->tct_max;
  double T1 = E / s[0][0], T2 = T1;
  for (int ks = 0; ks <= 30; ks++) {
    double a = s[0][0], b = s[0][1], c = s[0][2], d = s[0][3], e = s[0][4], ect = s[0][5];
#pragma unroll
    for (int j = 1; j < NT; j++)
      if (ST::NT || j < m->n_tct) {
        const bool up = T1 > m->tct[j - 1];
        a = up ? s[j][0] : a;
        b = up ? s[j][1] : b;
        c = up ? s[j][2] : c;
        d = up ? s[j][3] : d;
        e = up ? s[j][4] : e;
        ect = up ? s[j][5] : ect;
      }
    // above tct_max the heat capacity stays what it is there
    const double t = T1 <= tm ? T1 : tm;
    const double Ex = fm(fm(fm(fm(e, t, d), t, c), t, b), t, a);
    double Et1 = fm(fm(fm(fm(fm(e * 0.2, t, d * 0.25), t, c * (1.0 / 3.0)), t, b * 0.5), t, a), t, ect);
    Et1 = fm(Ex, T1 - t, Et1);
    T2 = T1 - (Et1 - E) / Ex;
    const double error = fabs(T2 - T1);
    T1 = T2;
    if (error < 1.0e-3) break;
  }
  return T2;
}

// What every reaction takes from the temperature: 1/T and ln T with their
// residuals (so that E/T and b ln T carry no rounding of their own into the
// exponent), and (R/atm in cm3) T, the unit of the equilibrium constants.
struct ChemTp {
  double T, iT, iTl, L, Ll, rs, irs;
  const double2* tab;  // chem_exp's table
};
__device__ __forceinline__ ChemTp chem_tp(const double2* tab, double T) {
  ChemTp t;
  t.tab = tab;
  t.T = T;
  t.iT = 1.0 / T;
  t.iTl = fm(-T, t.iT, 1.0) * t.iT;
  t.L = log(T);
  t.Ll = fm(T, chem_exp(tab, -t.L), -1.0);
  t.rs = CH_R0 / CH_ATM * 1.0e6 * T;
  t.irs = 1.0 / t.rs;
  return t;
}

// a T^b exp(-e/T) as one exponential of b ln T - e/T, whose rounding (the
// two products' and the difference's) goes into a last correction, so that
// the result is as near as the exponential itself; with pow and exp apart, e/T
// (up to 60) is rounded before it is raised.  Mean relative error of the
// mechanism's sets on 250-3500 K against 80-bit arithmetic 9.6e-17 (pow and
// exp 3.0e-16), largest 7.9e-16 (1.4e-14).  HB / HE: b / e is not zero; leaving
// out the part that is zero gives the same bits.
template <bool HB, bool HE>
__device__ __forceinline__ double chem_arr_s(double a, double b, double e, const ChemTp& t) {
  if constexpr (!HB && !HE) return a;
  double s, lo;
  const double eh = e * t.iT, el = fm(e, t.iTl, fm(e, t.iT, -eh));
  const double ph = b * t.L, pl = fm(b, t.Ll, fm(b, t.L, -ph));
  if constexpr (!HB) {
    s = -eh;
    lo = -el;
  } else if constexpr (!HE) {
    s = ph;
    lo = pl;
  } else {
    s = ph - eh;
    const double u = s - ph;
    lo = ((ph - (s - u)) - (eh + u)) + (pl - el);
  }
  const double k = chem_exp_times(t.tab, a, s);
  return fm(k, lo, k);
}
// Whether ln T, 1/T and the exponent are ordinary numbers.  They are not for a
// cell without energy (T = 0), of negative energy or NaN: there the expression
// itself decides, since T^b exists for whole b and exp(-e/T) is 0 where e/T is
// infinite.  (The ln T of Gibbs reverse rates makes every rate NaN there, so
// ReReac = 0 needs no test.)
__device__ __forceinline__ bool chem_T_ordinary(double T) { return T >= 1.0e-12 && T <= 1.0e300; }
__device__ __noinline__ double chem_arr_expr(double a, double b, double e, double T) {
  return a * pow(T, b) * exp(-e / T);
}
// ANYT: the temperature may not be an ordinary number
template <bool ANYT>
__device__ __forceinline__ double chem_arr(double a, double b, double e, const ChemTp& t) {
  if constexpr (ANYT)
    if (!chem_T_ordinary(t.T)) return chem_arr_expr(a, b, e, t.T);
  if (b == 0.0 && e == 0.0) return a;
  return chem_arr_s<true, true>(a, b, e, t);
}
// Troe falloff of the two sets' rates (:160-172)
template <class RX>
__device__ __forceinline__ double chem_troe(RX R, double k1, double k2, double ctrb, const ChemTp& t) {
  const double Prs = k1 / k2 * ctrb;
  const double x = log10(Prs) + R->ac;
  const double F = chem_exp(t.tab, R->lfc / (1.0 + q2(x / (R->an - 0.14 * x))) * 2.302585092994045684);
  return k2 * Prs / (1.0 + Prs) * F;
}

// comput_gibbs (CHEM_thermdyn.f90:296-319) over T: G / (R T) of one species
template <class P>
__device__ __forceinline__ double chem_gibbs_range(P c, const ChemTp& t, double oneL) {
  const double p = fm(t.T, fm(t.T, fm(t.T, c[4], c[3]), c[2]), c[1]);
  return fm(-t.T, p, fm(c[5], t.iT, fm(c[0], oneL, -c[6])));
}
template <class ST, class P>
__device__ __forceinline__ double chem_gibbs(Mech m, P gb, const ChemTp& t) {
  constexpr int NT = ST::NT ? ST::NT : CH_NT_MAX;
  const double oneL = 1.0 - t.L;
  double g = chem_gibbs_range(gb[0], t, oneL);
#pragma unroll
  for (int j = 1; j < NT; j++)
    if (ST::NT || j < m->n_tct) {
      const double v = chem_gibbs_range(gb[j], t, oneL);
      g = t.T > m->tct[j - 1] ? v : g;
    }
  return g;
}
// the same above tct_max, where the heat capacity stays what it is there
__device__ __noinline__ double chem_gibbs_high(Mech m, int i, double T) {
  int jc = 0;
  for (int j = 1; j < m->n_tct; j++)
    if (T > m->tct[j - 1]) jc = j;
  const auto c = m->coef[i][jc];
  const double tm = m->tct_max;
  const double Cp_max = c[0] + c[1] * tm + c[2] * q2(tm) + c[3] * q3(tm) + c[4] * q4(tm);
  const double h_max = c[0] * tm + c[1] * q2(tm) / 2.0 + c[2] * q3(tm) / 3.0 + c[3] * q4(tm) / 4.0 + c[4] * q5(tm) / 5.0 + c[5];
  const double S_max = c[0] * log(tm) + c[1] * tm + c[2] * q2(tm) / 2.0 + c[3] * q3(tm) / 3.0 + c[4] * q4(tm) / 4.0 + c[6];
  return (h_max + Cp_max * (T - tm) - T * (S_max + Cp_max * log(T / tm))) / T;
}

// Rates of progress of one reaction: Reaction_rate_coef
// (CHEM_reactions.f90:130-197) and the mass-action products of
// Reaction_rate_and_Matrix (:246-250).  g(i) = G_i / (R T), c(s) =
// concentration of species s, c(CH_NS) = 1.
template <bool ANYT = false, class RX, class G, class C>
__device__ __forceinline__ void chem_reaction(RX R, int rereac, const ChemTp& t, G g, C c, double& wf1, double& wr1) {
  double ctrb = 0.0;
  if (R->tb == 1) {
#pragma unroll
    for (int i = 0; i < CH_NS; i++) ctrb = fm(c(i), R->eff[i], ctrb);
  }
  const double k1 = chem_arr<ANYT>(R->a0, R->b0, R->e0, t);
  double wf, wr;
  if (R->af_type == 0) {
    wf = k1;
  } else {
    const double k2 = chem_arr<ANYT>(R->a1, R->b1, R->e1, t);
    if (R->af_type == 2) wf = k1 + k2;
    else wf = chem_troe(R, k1, k2, ctrb, t);
  }
  if (rereac == 0) {
    // 1 / Kc (comput_KjX, :76-103)
    double dg = 0.0;
#pragma unroll
    for (int i = 0; i < CH_NS; i++) dg = fm(g(i), R->nu[i], dg);
    wr = chem_exp_times(t.tab, wf, dg);  // dg passes 709 for a dissociation at 73 K, wf is as small
    const int sgm = R->sgm;
    if (sgm > 0) wr = wr * ipow(t.rs, sgm);
    else if (sgm < 0) wr = wr * ipow(t.irs, -sgm);
  } else if (rereac == 1) {
    wr = chem_arr<ANYT>(R->r[0], R->r[1], R->r[2], t);  // Arrhenius reverse rate (:180-181)
  } else {
    // ParkCurveFit (:113-118) with the 1e-30 floor (:182-186)
    const double z = 10000.0 / t.T;
    double kp = exp(R->r[0] + R->r[1] * z + R->r[2] * q2(z) + R->r[3] * q3(z) + R->r[4] * q4(z));
    if (kp < 1.0e-30) kp = 1.0e-30;
    wr = wf / kp;
  }
  if (R->tb == 1 && R->af_type != 1) {
    wf = wf * ctrb;
    wr = wr * ctrb;
  }
  const int nf = R->nsf, nr = R->nsr;
  if (nf >= 0 && nr >= 0) {
    const unsigned long long sf = R->sf, sr = R->sr;
#pragma unroll
    for (int a = 0; a < CH_SLOTS; a++) {
      wf = wf * c((int)(sf >> (8 * a)) & 0xff);
      wr = wr * c((int)(sr >> (8 * a)) & 0xff);
    }
    for (int a = CH_SLOTS; a < nf; a++) wf = wf * c((int)(sf >> (8 * a)) & 0xff);
    for (int a = CH_SLOTS; a < nr; a++) wr = wr * c((int)(sr >> (8 * a)) & 0xff);
  } else {
#pragma unroll 1
    for (int i = 0; i < CH_NS; i++) {
      if (R->vf[i] != 0.0) wf = wf * ipow(c(i), (int)R->vf[i]);
      if (R->vr[i] != 0.0) wr = wr * ipow(c(i), (int)R->vr[i]);
    }
  }
  wf1 = wf;
  wr1 = wr;
}

// d(rate of progress)/d(c_j) over the molar mass of j (CHEM_reactions.f90:262-268);
// rc_j = 1 / ((c_j + 1e-20) M_j)
__device__ __forceinline__ double chem_dA(double vf, double vr, double wf1, double wr1, double rc) {
  return fm(vf, wf1, -(vr * wr1)) * rc;
}

template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// chem_reaction of reaction K of ChemH2: the same operations, those with a
// zero order or a zero exponent left out (ReReac = 0)
template <class ST, int K, class G, class C>
__device__ __forceinline__ void chem_reaction_s(const CH_CONST ChemRx* R, const ChemTp& t, G g, C c, double& wf1,
                                                double& wr1) {
  double ctrb = 0.0;
  if constexpr (ST::tb[K] == 1) {
#pragma unroll
    for (int i = 0; i < CH_NS; i++) ctrb = fm(c(i), R->eff[i], ctrb);
  }
  const double k1 = chem_arr_s<(ST::ar[K] & 1) != 0, (ST::ar[K] & 2) != 0>(R->a0, R->b0, R->e0, t);
  double wf = k1;
  if constexpr (ST::af[K] != 0) {
    const double k2 = chem_arr_s<(ST::ar[K] & 4) != 0, (ST::ar[K] & 8) != 0>(R->a1, R->b1, R->e1, t);
    if constexpr (ST::af[K] == 2) wf = k1 + k2;
    else wf = chem_troe(R, k1, k2, ctrb, t);
  }
  double dg = 0.0;
  static_for<CH_NS>([&](auto I) {
    constexpr int i = decltype(I)::value, nu = ST::vr[K][i] - ST::vf[K][i];
    if constexpr (nu != 0) dg = fm(g(i), (double)nu, dg);
  });
  double wr = chem_exp_times(t.tab, wf, dg);
  constexpr int sgm = ST::sgm(K);
  if constexpr (sgm > 0) wr = wr * ipow(t.rs, sgm);
  else if constexpr (sgm < 0) wr = wr * ipow(t.irs, -sgm);
  if constexpr (ST::tb[K] == 1 && ST::af[K] != 1) {
    wf = wf * ctrb;
    wr = wr * ctrb;
  }
  static_for<CH_NS>([&](auto I) {
    constexpr int i = decltype(I)::value;
    for (int q = 0; q < ST::vf[K][i]; q++) wf = wf * c(i);
    for (int q = 0; q < ST::vr[K][i]; q++) wr = wr * c(i);
  });
  wf1 = wf;
  wr1 = wr;
}

// A lane's columns in LDS, species-major, one column per thread of the
// workgroup: concentrations (the last row holds 1), Gibbs functions, the
// Jacobian's 1 / ((c + 1e-20) M) and the cell's partial densities.  A
// reaction reads them by a uniform index, and the registers that they would
// take are what lets two waves of the implicit kernels share a SIMD.  Without
// JAC the rows rc are not there, and three waves of the Euler kernel fit the
// LDS (explicit batches of 300,007 cells, five steps, with the rows / without,
// us: Euler 151 / 136, RK2 539 / 519, RK3 394 / 394).
template <int NT, bool JAC>
struct LaneLds {
  static constexpr int N = NT;
  double c[CH_NS + 1][NT], g[CH_NS][NT];
  double rc[JAC ? CH_NS : 1][NT];
  double2 tab[CH_EXPN];
};
// fills a workgroup's table and constant row (NT = 64: one wavefront, whose
// LDS operations complete in order, so no barrier)
template <class LDS>
__device__ __forceinline__ void lane_lds_init(LDS& L) {
  static_assert(LDS::N == CH_EXPN, "one table entry per thread");
  L.tab[threadIdx.x] = make_double2(cm.exp2t[threadIdx.x][0], cm.exp2t[threadIdx.x][1]);
  L.c[CH_NS][threadIdx.x] = 1.0;
  __syncthreads();
}

// Reaction_rate_coef + Reaction_rate_and_Matrix (:230-272) of the cell of
// this lane, whose concentrations are in its column of L: ri in mol/cm3/s and
// (JAC) A[i][j] = d ri / d cj / M_j.  k is uniform across the wavefront.
template <bool JAC, class ST, class LDS>
__device__ __forceinline__ void lane_rates(Mech m, LDS& L, double T, const double* ci, double* ri,
                                           double (*A)[CH_NS]) {
  const int tid = (int)threadIdx.x;
  const ChemTp t = chem_tp(L.tab, T);
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    L.c[i][tid] = ci[i];
    if constexpr (JAC) L.rc[i][tid] = 1.0 / ((ci[i] + 1.0e-20) * m->mi[i]);
    ri[i] = 0.0;
    if (JAC) {
#pragma unroll
      for (int j = 0; j < CH_NS; j++) A[i][j] = 0.0;
    }
  }
  const int rereac = m->rereac, nr = m->nr;
  if (rereac == 0) {
#pragma unroll
    for (int i = 0; i < CH_NS; i++) L.g[i][tid] = chem_gibbs<ST>(m, m->gb[i], t);
    if (T > m->tct_max) {
#pragma unroll 1
      for (int i = 0; i < CH_NS; i++) L.g[i][tid] = chem_gibbs_high(m, i, T);
    }
  }
  auto conc = [&](int s) { return L.c[s][tid]; };
  auto gibbs = [&](int i) { return L.g[i][tid]; };
  if constexpr (ST::FIXED) {
    static_for<ST::NR>([&](auto K) {
      constexpr int k = decltype(K)::value;
      double wf1, wr1;
      chem_reaction_s<ST, k>(&m->rx[k], t, gibbs, conc, wf1, wr1);
      const double w = wf1 - wr1;
      static_for<CH_NS>([&](auto J) {
        constexpr int j = decltype(J)::value, nuj = ST::vr[k][j] - ST::vf[k][j];
        if constexpr (nuj != 0) ri[j] = fm(w, (double)nuj, ri[j]);
        if constexpr (JAC && (ST::vf[k][j] != 0 || ST::vr[k][j] != 0)) {
          const double dA = chem_dA(ST::vf[k][j], ST::vr[k][j], wf1, wr1, L.rc[j][tid]);
          static_for<CH_NS>([&](auto I) {
            constexpr int i = decltype(I)::value, nu = ST::vr[k][i] - ST::vf[k][i];
            if constexpr (nu != 0) A[i][j] = fm(dA, (double)nu, A[i][j]);
          });
        }
      });
    });
    return;
  }
  auto reactions = [&](auto anyt) {
#pragma unroll 1
    for (int k = 0; k < nr; k++) {
      const CH_CONST ChemRx* R = &m->rx[k];
      double wf1, wr1;
      chem_reaction<decltype(anyt)::value>(R, rereac, t, gibbs, conc, wf1, wr1);
      const double w = wf1 - wr1;
#pragma unroll
      for (int i = 0; i < CH_NS; i++) ri[i] = fm(w, R->nu[i], ri[i]);
      if constexpr (JAC) {
        const int part = R->part;
#pragma unroll
        for (int j = 0; j < CH_NS; j++)
          if ((part >> j) & 1) {
            const double dA = chem_dA(R->vf[j], R->vr[j], wf1, wr1, L.rc[j][tid]);
#pragma unroll
            for (int i = 0; i < CH_NS; i++) A[i][j] = fm(dA, R->nu[i], A[i][j]);
          }
      }
    }
  };
  if constexpr (ST::ANYT) {
    if (__any(!chem_T_ordinary(T))) {
      reactions(std::true_type{});
      return;
    }
  }
  reactions(std::false_type{});
}

// Gauss elimination with partial pivoting (CHEM_reactions.f90:523-567),
// fully unrolled so the system of the N species that react stays in registers; row exchanges are
// selects, entered only where a lane of the wavefront exchanges rows.
template <int N>
__device__ __forceinline__ void chem_gauss(double (*a)[CH_NS], double* b, double* x) {
  double rk[N];
#pragma unroll
  for (int k = 0; k < N - 1; k++) {
    double fmax = fabs(a[k][k]);
    int kk = k;
#pragma unroll
    for (int i = k + 1; i < N; i++)
      if (fabs(a[i][k]) > fmax) { fmax = fabs(a[i][k]); kk = i; }
    if (__any(kk != k)) {
#pragma unroll
      for (int i = k + 1; i < N; i++) {
        const bool sw = (i == kk);
#pragma unroll
        for (int j = k; j < N; j++) {
          const double t = a[k][j];
          a[k][j] = sw ? a[i][j] : a[k][j];
          a[i][j] = sw ? t : a[i][j];
        }
        const double t = b[k];
        b[k] = sw ? b[i] : b[k];
        b[i] = sw ? t : b[i];
      }
    }
    rk[k] = 1.0 / a[k][k];
#pragma unroll
    for (int i = k + 1; i < N; i++) {
      const double f = -div_r(a[i][k], a[k][k], rk[k]);
#pragma unroll
      for (int j = k + 1; j < N; j++) a[i][j] = fm(f, a[k][j], a[i][j]);
      b[i] = fm(f, b[k], b[i]);
    }
  }
  rk[N - 1] = 1.0 / a[N - 1][N - 1];
#pragma unroll
  for (int i = N - 1; i >= 0; i--) {
    double xi = b[i];
#pragma unroll
    for (int j = i + 1; j < N; j++) xi = fm(-a[i][j], x[j], xi);
    x[i] = div_r(xi, a[i][i], rk[i]);
  }
}

// update_Et, CHEM_thermdyn.f90:184-196
__device__ __forceinline__ void chem_update_et(Mech m, const double* di, const double* dinew, double& E) {
#pragma unroll
  for (int i = 0; i < CH_NS; i++) E = fm(-(dinew[i] - di[i]), m->rf[i], E);
}

// The linear system of chemical_Euler_implicit (CHEM_reactions.f90:491-505)
// with step h, solved in place: Ar (rows d ri / d cj / M_j) becomes I - Ar M_i h
// and is eliminated; dd = the increment of the partial densities.
template <class ST>
__device__ __forceinline__ void chem_implicit_solve(Mech m, const double* ri, double (*Ar)[CH_NS], double h, double* dd) {
  double rhs[CH_NS];
#pragma unroll
  for (int i = 0; i < ST::NA; i++) {
    const double hm = m->mi[i] * h;
#pragma unroll
    for (int j = 0; j < ST::NA; j++) Ar[i][j] = fm(-Ar[i][j], hm, i == j ? 1.0 : 0.0);
    rhs[i] = ri[i] * hm * 1.0e6;
  }
  chem_gauss<ST::NA>(Ar, rhs, dd);
#pragma unroll
  for (int i = ST::NA; i < CH_NS; i++) dd[i] = 0.0 * dd[0];  // zero, or NaN with the rest
}

__device__ __forceinline__ void chem_apply(Mech m, double* di, double& E, const double* dd) {
  double dinew[CH_NS];
#pragma unroll
  for (int i = 0; i < CH_NS; i++) dinew[i] = di[i] + dd[i];
  chem_update_et(m, di, dinew, E);
#pragma unroll
  for (int i = 0; i < CH_NS; i++) di[i] = dinew[i];
}

// chemical_Euler_implicit, CHEM_reactions.f90:473-516
template <class ST, class LDS>
__device__ __forceinline__ void chem_step_implicit(Mech m, LDS& L, double* di, double& E, double dt) {
  double ci[CH_NS], ri[CH_NS], Ar[CH_NS][CH_NS];
  const double T = chem_T<ST>(m, di, E);
#pragma unroll
  for (int i = 0; i < CH_NS; i++) ci[i] = di[i] * m->ci6[i];
  lane_rates<true, ST>(m, L, T, ci, ri, Ar);
  double dd[CH_NS];
  chem_implicit_solve<ST>(m, ri, Ar, dt, dd);
  chem_apply(m, di, E, dd);
}

template <class ST, class LDS>
__device__ __forceinline__ void chem_explicit_rates(Mech m, LDS& L, const double* di_c, double T, double* ri) {
  double ci[CH_NS];
#pragma unroll
  for (int i = 0; i < CH_NS; i++) ci[i] = di_c[i] * m->ci6[i];
  lane_rates<false, ST>(m, L, T, ci, ri, nullptr);
}

// chemical_Euler (:395-425), chemical_RK2 (:429-469), chemical_RK3 (:572-602)
template <int MODE, class ST, class LDS>
__device__ __forceinline__ void chem_step(Mech m, LDS& L, double* di, double& E, double dt) {
  if (MODE == -1) {
    chem_step_implicit<ST>(m, L, di, E, dt);
  } else if (MODE == 1) {
    double ri[CH_NS], dinew[CH_NS];
    const double T = chem_T<ST>(m, di, E);
    chem_explicit_rates<ST>(m, L, di, T, ri);
#pragma unroll
    for (int i = 0; i < CH_NS; i++) dinew[i] = di[i] + ri[i] * m->mi[i] * 1.0e6 * dt;
    chem_update_et(m, di, dinew, E);
#pragma unroll
    for (int i = 0; i < CH_NS; i++) di[i] = dinew[i];
  } else if (MODE == 2) {
    // one rate evaluation in a loop of two: the code is there once
    double din[CH_NS], E0 = E;
#pragma unroll
    for (int i = 0; i < CH_NS; i++) din[i] = di[i];
    for (int krk = 0; krk < 2; krk++) {
      double ri[CH_NS], dinew[CH_NS];
      // the reference evaluates the second stage's T from the old densities
      const double T = chem_T<ST>(m, din, E0);
      chem_explicit_rates<ST>(m, L, di, T, ri);
#pragma unroll
      for (int i = 0; i < CH_NS; i++) {
        const double w = ri[i] * m->mi[i] * 1.0e6 * dt;
        dinew[i] = krk == 0 ? di[i] + w : 0.5 * din[i] + 0.5 * di[i] + 0.5 * w;
      }
      chem_update_et(m, di, dinew, E0);
#pragma unroll
      for (int i = 0; i < CH_NS; i++) di[i] = dinew[i];
    }
    E = E0;
  } else {
    const double Ra[3] = {0.0, 3.0 / 4.0, 1.0 / 3.0}, Rb[3] = {1.0, 1.0 / 4.0, 2.0 / 3.0};
    double din[CH_NS], ri[CH_NS], dinew[CH_NS];
#pragma unroll
    for (int i = 0; i < CH_NS; i++) din[i] = di[i];
    for (int krk = 0; krk < 3; krk++) {
      const double T = chem_T<ST>(m, di, E);
      chem_explicit_rates<ST>(m, L, di, T, ri);
#pragma unroll
      for (int i = 0; i < CH_NS; i++) dinew[i] = Ra[krk] * din[i] + Rb[krk] * (di[i] + ri[i] * m->mi[i] * 1.0e6 * dt);
      chem_update_et(m, di, dinew, E);
#pragma unroll
      for (int i = 0; i < CH_NS; i++) di[i] = dinew[i];
    }
  }
}

// Adaptive point-implicit substepping (no reference counterpart).  One
// attempt: T, rates and Jacobian at the current state (negative partial
// densities enter the rates as zero: the reference's regularised Jacobian
// d(ri)/d(cj) ~ 1/(cj + 1e-20) makes cj = -1e-20 mol/cm3 a fixed point of the
// point-implicit update of a consumed species, where it divides by zero);
// proposed step
//   h = min(dt - t, h_cap, min_k s_k/|w_k|, s_T/|q|)
// with s_k = rtol_y (max(rho_k,0) + y_floor rho), s_T = rtol_t T rcv,
// rcv = sum_k 2.5 R_k rho_k, w_k = ri_k M_k 1e6 and q = sum_k w_k R_k F_k;
// the linear solve gives dd, accepted when |dd_k| <= 2 s_k for all k and
// |sum_k dd_k R_k F_k| <= 2 s_T.  Accepted: the update is applied and
// h_cap = 2h.  Rejected: the state is unchanged and h_cap = h/2.  Returns
// whether the attempt was accepted; h_taken is the step on acceptance.
struct ChemCtl {
  double rtol_y, y_floor, rtol_t;
  int max_sub;
};

// Step length and tolerances from the rates (both kernels).  The minimum is
// carried as a numerator and a denominator (num / den < s / |w| where num |w| >
// s den), so that the winner alone is divided.
__device__ __forceinline__ double chem_limit(Mech m, const double* di, const double* ri, double rho, double T, double h0,
                                             const ChemCtl& ctl, double* sk, double& sT) {
  double num = h0, den = 1.0;
  double q = 0.0, rcv = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    const double w = ri[i] * m->mi[i] * 1.0e6;
    sk[i] = ctl.rtol_y * fm(ctl.y_floor, rho, di[i] > 0.0 ? di[i] : 0.0);
    const bool cut = fabs(w) * num > sk[i] * den;
    num = cut ? sk[i] : num;
    den = cut ? fabs(w) : den;
    q = fm(w, m->rf[i], q);
    rcv = fm(m->rcv[i], di[i], rcv);
  }
  sT = ctl.rtol_t * T * rcv;
  const bool cut = fabs(q) * num > sT * den;
  num = cut ? sT : num;
  den = cut ? fabs(q) : den;
  return num / den;
}
__device__ __forceinline__ bool chem_accept(Mech m, const double* dd, const double* sk, double sT) {
  bool ok = true;
  double de = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    ok = ok && fabs(dd[i]) <= 2.0 * sk[i];
    de = fm(dd[i], m->rf[i], de);
  }
  return ok && fabs(de) <= 2.0 * sT;
}

template <class ST, class LDS>
__device__ __forceinline__ bool chem_adaptive_attempt(Mech m, LDS& L, double* di, double& E, double dt, double t,
                                                      double& h_cap, const ChemCtl& ctl, double& h_taken) {
  double ci[CH_NS], ri[CH_NS], Ar[CH_NS][CH_NS], sk[CH_NS], dd[CH_NS];
  const double T = chem_T<ST>(m, di, E);
  double rho = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    ci[i] = (di[i] > 0.0 ? di[i] : 0.0) * m->ci6[i];
    rho = rho + di[i];
  }
  lane_rates<true, ST>(m, L, T, ci, ri, Ar);
  double h = dt - t;
  if (h_cap < h) h = h_cap;
  double sT;
  h = chem_limit(m, di, ri, rho, T, h, ctl, sk, sT);
  chem_implicit_solve<ST>(m, ri, Ar, h, dd);
  if (!chem_accept(m, dd, sk, sT)) {
    h_cap = 0.5 * h;
    return false;
  }
  chem_apply(m, di, E, dd);
  h_cap = 2.0 * h;
  h_taken = h;
  return true;
}

// ---------------------------------------------------------------------------
// One cell per wavefront.  Every lane holds the same copy of the cell's state;
// lane i < CH_NS forms a species' Gibbs function, lane k a reaction's rates,
// and lane j < CH_NS the Jacobian's column j in registers (lane CH_NS the
// right-hand side), so that a pivot search stays inside one lane and a row
// operation is one FMA with the factor broadcast from the pivot's lane.
// Every value is formed by the operations of the per-lane integrator in their
// order, so the results are bit-identical to it.  What counts is latency: an
// attempt is one dependent chain, 7 us against the per-lane one's 14.
// ---------------------------------------------------------------------------
struct CoopLds {
  ChemRx rx[CH_NR_MAX];
  double gb[CH_NS][CH_NT_MAX][7];
  double c[CH_NS + 1], mi[CH_NS];
};
__device__ __forceinline__ void coop_lds_init(Mech m, CoopLds& L, int lane) {
  const int words = m->nr * (int)(sizeof(ChemRx) / sizeof(double));
  const CH_CONST double* src = (const CH_CONST double*)m->rx;
  for (int e = lane; e < words; e += 64) ((double*)L.rx)[e] = src[e];
  const CH_CONST double* gb = (const CH_CONST double*)m->gb;
  for (int e = lane; e < CH_NS * CH_NT_MAX * 7; e += 64) ((double*)L.gb)[e] = gb[e];
  if (lane < CH_NS) L.mi[lane] = m->mi[lane];
  if (lane == CH_NS) L.c[CH_NS] = 1.0;
  __syncthreads();
}

__device__ __forceinline__ double bcast(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <class ST>
__device__ __forceinline__ bool coop_attempt(Mech m, CoopLds& L, const double2* tab, int lane, double* di, double& E,
                                             double dt, double t, double& h_cap, const ChemCtl& ctl, double& h_taken) {
  constexpr int N = ST::NA;
  double ci[CH_NS], ri[CH_NS], sk[CH_NS], dd[CH_NS];
  const double T = chem_T<ST>(m, di, E);
  double rho = 0.0, cl = 0.0;
#pragma unroll
  for (int i = 0; i < CH_NS; i++) {
    ci[i] = (di[i] > 0.0 ? di[i] : 0.0) * m->ci6[i];
    rho = rho + di[i];
    cl = lane == i ? ci[i] : cl;
  }
  const ChemTp tp = chem_tp(tab, T);
  const int rereac = m->rereac, nr = m->nr, li = lane < CH_NS ? lane : 0;
  __syncthreads();  // one wavefront: orders the LDS accesses only
  if (lane < CH_NS) L.c[lane] = cl;
  const double rc = 1.0 / ((cl + 1.0e-20) * L.mi[li]);
  double gl = rereac == 0 ? chem_gibbs<ST>(m, L.gb[li], tp) : 0.0;
  if (T > m->tct_max) gl = chem_gibbs_high(m, li, T);
  double gi[CH_NS];
#pragma unroll
  for (int i = 0; i < CH_NS; i++) gi[i] = bcast(gl, i);
  __syncthreads();
  double wf1 = 0.0, wr1 = 0.0;
  auto reaction = [&](auto anyt) {
    chem_reaction<decltype(anyt)::value>((const ChemRx*)&L.rx[lane], rereac, tp, [&](int i) { return gi[i]; },
                                         [&](int s) { return L.c[s]; }, wf1, wr1);
  };
  if (lane < nr) {
    if (ST::ANYT && !chem_T_ordinary(T)) reaction(std::bool_constant<ST::ANYT>{});
    else reaction(std::false_type{});
  }
  double a[CH_NS];
#pragma unroll
  for (int i = 0; i < CH_NS; i++) a[i] = ri[i] = 0.0;
  auto add = [&](int k, auto nu) {
    const double wf = bcast(wf1, k), wr = bcast(wr1, k), w = wf - wr;
    const double vf = L.rx[k].vf[li], vr = L.rx[k].vr[li];
    const double dA = vf != 0.0 || vr != 0.0 ? chem_dA(vf, vr, wf, wr, rc) : 0.0;
    nu([&](int i, double v) {
      ri[i] = fm(w, v, ri[i]);
      a[i] = fm(dA, v, a[i]);
    });
  };
  if constexpr (ST::FIXED) {
    static_for<ST::NR>([&](auto K) {
      constexpr int k = decltype(K)::value;
      add(k, [&](auto row) {
        static_for<CH_NS>([&](auto I) {
          constexpr int i = decltype(I)::value, nu = ST::vr[k][i] - ST::vf[k][i];
          if constexpr (nu != 0) row(i, (double)nu);
        });
      });
    });
  } else {
#pragma unroll 1
    for (int k = 0; k < nr; k++)
      add(k, [&](auto row) {
#pragma unroll
        for (int i = 0; i < CH_NS; i++) row(i, m->rx[k].nu[i]);
      });
  }
  double h = dt - t;
  if (h_cap < h) h = h_cap;
  double sT;
  h = chem_limit(m, di, ri, rho, T, h, ctl, sk, sT);
#pragma unroll
  for (int i = 0; i < N; i++) {
    const double hm = m->mi[i] * h;
    a[i] = lane == CH_NS ? ri[i] * hm * 1.0e6 : fm(-a[i], hm, i == lane ? 1.0 : 0.0);
  }
  // Gauss elimination with partial pivoting (CHEM_reactions.f90:523-567)
  double rk[N];
#pragma unroll
  for (int k = 0; k < N - 1; k++) {
    double fmax = fabs(a[k]);
    int kl = k;
#pragma unroll
    for (int i = k + 1; i < N; i++)
      if (fabs(a[i]) > fmax) { fmax = fabs(a[i]); kl = i; }
    const int kk = __builtin_amdgcn_readlane(kl, k);
    if (kk != k) {
#pragma unroll
      for (int i = k + 1; i < N; i++)
        if (i == kk) {
          const double s = a[k];
          a[k] = a[i];
          a[i] = s;
        }
    }
    const double r = 1.0 / a[k];
    rk[k] = bcast(r, k);
#pragma unroll
    for (int i = k + 1; i < N; i++) {
      const double f = -div_r(a[i], a[k], r);
      a[i] = fm(bcast(f, k), a[k], a[i]);
    }
  }
  rk[N - 1] = bcast(1.0 / a[N - 1], N - 1);
#pragma unroll
  for (int i = N - 1; i >= 0; i--) {
    double xi = bcast(a[i], CH_NS);
#pragma unroll
    for (int j = i + 1; j < N; j++) xi = fm(-bcast(a[i], j), dd[j], xi);
    dd[i] = div_r(xi, bcast(a[i], i), rk[i]);
  }
#pragma unroll
  for (int i = N; i < CH_NS; i++) dd[i] = 0.0 * dd[0];
  if (!__builtin_amdgcn_readfirstlane(chem_accept(m, dd, sk, sT) ? 1 : 0)) {
    h_cap = 0.5 * h;
    return false;
  }
  chem_apply(m, di, E, dd);
  h_cap = 2.0 * h;
  h_taken = h;
  return true;
}
