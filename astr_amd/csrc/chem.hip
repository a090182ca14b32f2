// chem.hip -- per-cell chemical source terms on gfx950 and their C ABI.
//
// Replaces the reference's per-cell Cantera calls on the hot path:
//   chemrate(den,tmp,spc,wi)   src/thermchem.F90:1553-1575  (setState_TRY +
//                              getNetProductionRates, wi = wdot*W)
//   cpeval(tmp,spc,cp=)        src/thermchem.F90:1342-1428  (cp_mass)
//   enthpy(tmp,hi)             src/thermchem.F90:1498-1541  (h_k = H/RT *
//                              (8314.2/W_k) * T)
// for a CTML mechanism (Cantera's XML format, e.g.
// chemMech/Jachimowski88_H2-9-19.xml): ideal gas, NASA 7-coefficient
// thermodynamics, elementary and three-body mass-action reactions with
// Arrhenius rate constants, reverse rates from the equilibrium constant.
// One thread evaluates one cell; all arithmetic is FP64.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/astr_hip.h"
#include "rate_exp.hpp"

namespace {

thread_local std::string g_cerr;
int cfail(const std::string& m) {
  g_cerr = m;
  return -1;
}

#define CHIP_OK(x)                                                               \
  do {                                                                           \
    hipError_t e_ = (x);                                                         \
    if (e_ != hipSuccess) return cfail(std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int NSMAX = 16;
constexpr int NRMAX = 48;
constexpr int NTERM = 3;  // species per side of a reaction

// gas constant (J/kmol/K) of Cantera 2.5 (CODATA 2018 Avogadro x Boltzmann),
// used inside Cantera's thermodynamics and kinetics
constexpr double kRgas = 8314.46261815324;
// the reference's own constant in enthpy/rgcmix (thermchem.F90:26,490,1513)
constexpr double kRref = 8314.2;

struct Mech {
  int ns, nr;
  double W[NSMAX];         // molecular weights, kg/kmol
  double tmid[NSMAX];
  double lo[NSMAX][7], hi[NSMAX][7];
  double lnA[NRMAX], b[NRMAX], EaR[NRMAX];
  int rev[NRMAX], tb[NRMAX];
  double eff[NRMAX][NSMAX];  // third-body efficiencies
  int nre[NRMAX], rsp[NRMAX][NTERM];
  double rnu[NRMAX][NTERM];
  int npr[NRMAX], psp[NRMAX][NTERM];
  double pnu[NRMAX][NTERM];
  double dnu[NRMAX];       // sum of product minus reactant coefficients
  double p0;               // standard-state pressure of the thermo data, Pa
  // the same data in the form the cell kernels read it, laid out once by
  // prepare_cells: every access is uniform over a wavefront, so a record comes
  // in with a few scalar loads, and no division is left to the cells
  double iW[NSMAX], rW[NSMAX];  // 1/W, kRref/W
  struct Range {           // one NASA range: cp/R, h/RT and g/RT as polynomials
    double a0, a1, a2, a3, a4;
    double h1, h2, h3, h4;  // a1/2, a2/3, a3/4, a4/5
    double g1, g2, g3, g4;  // -a1/2, -a2/6, -a3/12, -a4/20
    double a5, a6;
  } th[NSMAX][2];
  struct Rx {
    double lnA, b, EaR;
    unsigned sp;           // unit terms: 3 reactants, 3 products, 4 bits each
    unsigned fl;           // bits 0-1 / 2-3: unit terms per side, 4: reversible, 5: three-body,
                           // 6: a product of unit terms on both sides
    double nu[NSMAX];      // product minus reactant coefficients
    double eff[NSMAX];
  } rx[NRMAX];
  double lnp0R;            // ln(p0 / kRgas)
  int unit;                // every order is a whole number and a side has at most NTERM of them
};

// ---------------------------------------------------------------------------
// device evaluation
// ---------------------------------------------------------------------------
// Reaction orders other than 1 and 2 go through pow, kept out of line: the
// inlined pow's temporaries set the register peak of every kernel that
// evaluates rates, although orders 1 and 2 never reach it.
__device__ __attribute__((noinline)) double conc_pow_general(double c, double nu) {
  return pow(c, nu);
}

__device__ __forceinline__ double conc_pow(double c, double nu) {
  return nu == 1.0 ? c : (nu == 2.0 ? c * c : conc_pow_general(c, nu));
}

// Thermodynamics and kinetics of one state: molar concentrations from rho and
// Y; per species cp/R (cpr), h/RT (hrt); net molar production rates w
// (kmol/m^3/s).  GasKinetics: kf = A T^b exp(-E/RT), kr = kf / Kc with
// Kc = exp(-dG/RT) (p0/RT)^dnu, three-body [M] = sum eff_k C_k.
__device__ __forceinline__ void kinetics(const Mech* __restrict__ M, double T, double rho,
                                         const double* y, double* w, double* cpr, double* hrt) {
  const int ns = M->ns, nr = M->nr;
  double c[NSMAX], g[NSMAX];
  const double logT = log(T), invT = 1.0 / T;
  const double T2 = T * T, T3 = T2 * T, T4 = T3 * T;
  for (int k = 0; k < ns; k++) {
    c[k] = rho * y[k] / M->W[k];
    const double* a = T <= M->tmid[k] ? M->lo[k] : M->hi[k];
    // NASA 7-coefficient polynomials
    cpr[k] = a[0] + a[1] * T + a[2] * T2 + a[3] * T3 + a[4] * T4;
    hrt[k] = a[0] + a[1] * T / 2.0 + a[2] * T2 / 3.0 + a[3] * T3 / 4.0 + a[4] * T4 / 5.0 +
             a[5] * invT;
    const double sr = a[0] * logT + a[1] * T + a[2] * T2 / 2.0 + a[3] * T3 / 3.0 +
                      a[4] * T4 / 4.0 + a[6];
    g[k] = hrt[k] - sr;
    w[k] = 0.0;
  }
  const double lc0 = log(M->p0 / (kRgas * T));  // ln of the standard concentration
  for (int r = 0; r < nr; r++) {
    const double kf = exp(M->lnA[r] + M->b[r] * logT - M->EaR[r] * invT);
    double fwd = kf;
    double dg = 0.0;
    for (int j = 0; j < M->nre[r]; j++) {
      fwd *= conc_pow(c[M->rsp[r][j]], M->rnu[r][j]);
      dg -= M->rnu[r][j] * g[M->rsp[r][j]];
    }
    double rv = 0.0;
    if (M->rev[r]) {
      double pp = 1.0;
      for (int j = 0; j < M->npr[r]; j++) {
        pp *= conc_pow(c[M->psp[r][j]], M->pnu[r][j]);
        dg += M->pnu[r][j] * g[M->psp[r][j]];
      }
      const double kr = exp(M->lnA[r] + M->b[r] * logT - M->EaR[r] * invT + dg - M->dnu[r] * lc0);
      rv = kr * pp;
    }
    double q = fwd - rv;
    if (M->tb[r]) {
      double cm = 0.0;
      for (int k = 0; k < ns; k++) cm += M->eff[r][k] * c[k];
      q *= cm;
    }
    for (int j = 0; j < M->nre[r]; j++) w[M->rsp[r][j]] -= M->rnu[r][j] * q;
    for (int j = 0; j < M->npr[r]; j++) w[M->psp[r][j]] += M->pnu[r][j] * q;
  }
}

// An array in registers read at an index that is uniform over the wavefront.
// Kept as two vectors of 32-bit halves: a register tuple exists for every
// count of 9..12 32-bit elements, while an array of 9 doubles is rounded up to
// a tuple of 16 (32 registers for 18).
// N < NSMAX: one more element, 1, where unit()'s unused indices point.
template <int N>
struct RegArray {
  static constexpr bool PAD = N < NSMAX;
  typedef unsigned V __attribute__((ext_vector_type(N + PAD)));
  V lo, hi;
  __device__ __forceinline__ RegArray() {
    if constexpr (PAD) set(N, 1.0);
  }
  __device__ __forceinline__ void set(int k, double x) {
    lo[k] = (unsigned)__double2loint(x);
    hi[k] = (unsigned)__double2hiint(x);
  }
  __device__ __forceinline__ double get(int k) const { return __hiloint2double((int)hi[k], (int)lo[k]); }
  // the product of up to three elements: 4-bit indices in sp, their count in
  // the low bits of fl; with the pad, three without a branch
  __device__ __forceinline__ double unit(unsigned sp, unsigned fl) const {
    double p = get(sp & 15);
    if (PAD || (fl & 3) > 1) p *= get(sp >> 4 & 15);
    if (PAD || (fl & 3) > 2) p *= get(sp >> 8 & 15);
    return p;
  }
};

// e^x for the rate constants (rate_exp.hpp) in about 20 instructions where exp
// takes 33: exp's constants sit in vector registers that its multiply-adds
// overwrite, so each is copied first; here they are scalar operands (ExpK, made
// once per thread in scalar registers), and the checks for overflow and
// underflow are one comparison, with exp's own result for the lanes outside
// +-700.
struct ExpK : astr::RateExpConstants {
  __device__ __forceinline__ ExpK() {
    asm volatile("" : "+s"(l2e), "+s"(rnd), "+s"(hi), "+s"(lo), "+s"(c3), "+s"(c4), "+s"(c5));
    asm volatile("" : "+s"(c6), "+s"(c7), "+s"(c8), "+s"(c9), "+s"(c10), "+s"(c11), "+s"(c12));
  }
};
// several at once, with one branch after their chains of multiply-adds
template <int N>
__device__ __forceinline__ void rate_exps(const double (&x)[N], const ExpK& K, double (&e)[N]) {
  bool in = true;
#pragma unroll
  for (int j = 0; j < N; j++) {
    e[j] = rate_exp_in(x[j], K);
    in = in && fabs(x[j]) < 700.0;
  }
  if (__any(!in)) {
#pragma unroll
    for (int j = 0; j < N; j++) e[j] = fabs(x[j]) < 700.0 ? e[j] : exp(x[j]);
  }
}

// cp/R, h/RT and g/RT - ln(p0/RT) of species k, from both NASA ranges
// (uniform coefficients, one scalar operand per multiply-add) and the cell's
// range picked.  With ln(p0/RT) in g, ln kr = ln kf + sum nu_k g_k: the
// equilibrium constant's (p0/RT)^dnu needs no term of its own.
struct Thermo {
  double cp, h, g;
};
__device__ __forceinline__ Thermo species(const Mech* __restrict__ M, int k, double T, double invT,
                                          double omlogT, double lc0) {
  Thermo t[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const Mech::Range& R = M->th[k][q];
    const double b = R.a5 * invT;
    t[q].cp = R.a0 + T * (R.a1 + T * (R.a2 + T * (R.a3 + T * R.a4)));
    t[q].h = R.a0 + T * (R.h1 + T * (R.h2 + T * (R.h3 + T * R.h4))) + b;
    t[q].g = R.a0 * omlogT + T * (R.g1 + T * (R.g2 + T * (R.g3 + T * R.g4))) + b - R.a6 - lc0;
  }
  const bool low = T <= M->tmid[k];
  return {low ? t[0].cp : t[1].cp, low ? t[0].h : t[1].h, low ? t[0].g : t[1].g};
}

// The net molar production rates w (kmol/m^3/s) of one cell from its
// concentrations c and its g (as species() returns it).  What a reaction adds
// to dg and takes from q goes over all species with its row of coefficients:
// nine multiply-adds with a scalar operand each, against three to six indexed
// register accesses of about eight instructions.  A reaction whose rate is
// not finite must leave the species alone that take no part in it: it makes
// every w of that sum NaN, w[0] too, and the sums are then formed again with
// the zeros of the rows skipped (CAREFUL).  c, g and the coefficients past ns
// are zero.  UNIT: every mass-action product is one of at most NTERM
// concentrations; otherwise the reactions that have other orders go through
// conc_pow, whose call to pow sets the register peak of the whole kernel
// (2^20 cells of 9 species 114 us with it, 88 us without).
template <int NSA, bool UNIT, bool CAREFUL>
__device__ __forceinline__ void reaction_sums(const Mech* __restrict__ M, int ns, double logT, double invT,
                                              const RegArray<NSA>& c, const double (&g)[NSA], double (&w)[NSA]) {
  const int nr = M->nr;
  const ExpK K;
#pragma unroll
  for (int k = 0; k < NSA; k++) w[k] = 0.0;
#pragma unroll 1
  for (int r = 0; r < nr; r++) {
    const Mech::Rx& R = M->rx[r];
    double nu[NSA];  // read with the record's head, ahead of the exponentials
#pragma unroll
    for (int k = 0; k < NSA; k++) nu[k] = R.nu[k];
    const unsigned fl = R.fl;
    const double lkf = R.lnA + R.b * logT - R.EaR * invT;
    double fw = 1.0, q;
    if (UNIT || (fl & 64)) {
      fw = c.unit(R.sp, fl);
    } else {
      for (int j = 0; j < M->nre[r]; j++) fw *= conc_pow(c.get(M->rsp[r][j]), M->rnu[r][j]);
    }
    if (fl & 16) {
      double dg = 0.0, bw = 1.0, k[2];
#pragma unroll
      for (int k = 0; k < NSA; k++) dg += nu[k] * g[k];
      if (UNIT || (fl & 64)) {
        bw = c.unit(R.sp >> 12, fl >> 2);
      } else {
        for (int j = 0; j < M->npr[r]; j++) bw *= conc_pow(c.get(M->psp[r][j]), M->pnu[r][j]);
      }
      rate_exps({lkf, lkf + dg}, K, k);  // kr = kf / Kc
      q = k[0] * fw - k[1] * bw;
    } else {
      double k[1];
      rate_exps({lkf}, K, k);
      q = k[0] * fw;
    }
    if (fl & 32) {
      double cm = 0.0;
#pragma unroll
      for (int k = 0; k < NSA; k++) cm += R.eff[k] * c.get(k);
      q *= cm;
    }
#pragma unroll
    for (int k = 0; k < NSA; k++)
      if (!CAREFUL || nu[k] != 0.0) w[k] += nu[k] * q;
  }
}

template <int NSA, bool UNIT>
__device__ __forceinline__ void cell_rates(const Mech* __restrict__ M, int ns, double logT, double invT,
                                           const RegArray<NSA>& c, const double (&g)[NSA], double (&w)[NSA]) {
  reaction_sums<NSA, UNIT, false>(M, ns, logT, invT, c, g, w);
  if (__any(!(fabs(w[0]) <= 1.7976931348623157e308)))
    reaction_sums<NSA, UNIT, true>(M, ns, logT, invT, c, g, w);
}

// cells per workgroup: one wavefront, so that few cells spread over many
// compute units (1000 cells 14 us, 16 with four wavefronts; 2^20 alike)
constexpr int kCellBlock = 64;

// NSA: the per-cell arrays' size.  NSA = NSMAX serves any mechanism (up to
// M->ns); an instance with NSA = the mechanism's species count has every loop
// over the species unrolled.  Bound by FP64 arithmetic: about 2500 vector
// instructions a cell with 9 species and 19 reactions (two exponentials per
// reaction are 760 of them), 64 us of issue for 2^20 cells against 38 us for
// the cells' 176 bytes.  124 registers leave four wavefronts per SIMD to cover
// the scalar loads of the reaction records (96 spill: 220 us; three: 93 us).
// 2^20 cells 190 -> 88 us, 1000 cells 29 -> 12 us against divisions in the
// thermodynamics, indexed sums and the library's exponential; 8 species in
// the NSMAX instance 253 -> 129 us, with general orders 264 -> 168 us.
template <int NSA, bool UNIT>
__global__ __launch_bounds__(kCellBlock, NSA == NSMAX ? 2 : UNIT ? 4 : 3) void k_chem(const Mech* __restrict__ M, long long n,
                                              const double* __restrict__ Tin,
                                              const double* __restrict__ RPin, int input_is_p,
                                              const double* __restrict__ Y, double* __restrict__ wdot,
                                              double* __restrict__ hmix, double* __restrict__ cpmix,
                                              double* __restrict__ hk) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int ns = NSA == NSMAX ? M->ns : NSA;
  const double T = Tin[i];
  double y[NSA], g[NSA], w[NSA];
  RegArray<NSA> c;
  double winv = 0.0;
#pragma unroll
  for (int k = 0; k < NSA; k++) {
    y[k] = NSA != NSMAX || k < ns ? Y[k * n + i] * M->iW[k] : 0.0;
    winv += y[k];
  }
  const double rho = input_is_p ? RPin[i] / (kRgas * T * winv) : RPin[i];
  const double logT = log(T), invT = 1.0 / T;
  const double lc0 = M->lnp0R - logT;  // ln of the standard concentration
  double cp = 0.0, h = 0.0;
#pragma unroll
  for (int k = 0; k < NSA; k++) {
    c.set(k, NSA != NSMAX || k < ns ? rho * y[k] : 0.0);
    g[k] = 0.0;
    if (NSA == NSMAX && k >= ns) continue;
    const Thermo t = species(M, k, T, invT, 1.0 - logT, lc0);
    g[k] = t.g;
    cp += y[k] * t.cp;
    h += y[k] * t.h;
    // evaluated here: sunk to their uses, all species' polynomials would wait
    // there with all their coefficients in (spilled) scalar registers
    asm volatile("" : "+v"(g[k]), "+v"(cp), "+v"(h));
    if (hk) hk[k * n + i] = t.h * M->rW[k] * T;
  }
  cell_rates<NSA, UNIT>(M, ns, logT, invT, c, g, w);
#pragma unroll
  for (int k = 0; k < NSA; k++)
    if (NSA != NSMAX || k < ns) wdot[k * n + i] = w[k] * M->W[k];
  if (hmix) hmix[i] = h * kRref * T;
  if (cpmix) cpmix[i] = cp * kRgas;
}

// srccomb (solver.F90:500-537): at every computed point (i, j, k) of
// 0:im x 0:jm x 0:km, chemrate of (rho, tmp, spc) (wirate = wdot_k W_k,
// thermchem.F90:1553-1575) times jacob added to qrhs(i,j,k,6:5+ns).  rho,
// tmp, jacob: (-hm:im+hm, -hm:jm+hm, -hm:km+hm), spc: the same with a last
// species index, qrhs: (0:im, 0:jm, 0:km, 1:numq), all column-major as the
// reference allocates them (commarray.F90).
template <int NSA, bool UNIT>
__global__ __launch_bounds__(kCellBlock, NSA == NSMAX ? 2 : UNIT ? 4 : 3) void k_srccomb(const Mech* __restrict__ M, int im, int jm, int km,
                                                 int hm, const double* __restrict__ rho,
                                                 const double* __restrict__ tmp,
                                                 const double* __restrict__ spc,
                                                 const double* __restrict__ jacob,
                                                 double* __restrict__ qrhs) {
  const long long nx = im + 1, ny = jm + 1, ncell = nx * ny * (km + 1);
  const long long cell = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (cell >= ncell) return;
  const int ns = NSA == NSMAX ? M->ns : NSA;
  const long long i = cell % nx, j = (cell / nx) % ny, k = cell / (nx * ny);
  const long long sx = im + 1 + 2 * hm, sy = jm + 1 + 2 * hm, sz = km + 1 + 2 * hm;
  const long long hp = ((k + hm) * sy + (j + hm)) * sx + (i + hm);
  const long long hs = sx * sy * sz;
  const double T = tmp[hp], r = rho[hp];
  const double logT = log(T), invT = 1.0 / T;
  double g[NSA], w[NSA];
  RegArray<NSA> c;
#pragma unroll
  for (int s = 0; s < NSA; s++) {
    c.set(s, 0.0);
    g[s] = 0.0;
    if (NSA == NSMAX && s >= ns) continue;
    c.set(s, r * (spc[s * hs + hp] * M->iW[s]));
    g[s] = species(M, s, T, invT, 1.0 - logT, M->lnp0R - logT).g;
    asm volatile("" : "+v"(g[s]));  // as in k_chem
  }
  cell_rates<NSA, UNIT>(M, ns, logT, invT, c, g, w);
  const double jac = jacob[hp];
#pragma unroll
  for (int s = 0; s < NSA; s++) {
    if (NSA == NSMAX && s >= ns) continue;
    double* q = qrhs + (5 + s) * ncell + cell;
    *q = *q + (w[s] * M->W[s]) * jac;
  }
}

// ---------------------------------------------------------------------------
// temperature_calc (thermchem.F90:1775-1786): T from the mass-specific
// internal energy e at fixed density and composition (Cantera setState_UV;
// for an ideal gas e does not depend on density).  Newton on
//   e(T) = sum_k Y_k (h_k(T) - R T / W_k),  de/dT = cv = cp - R sum Y_k/W_k
// with the NASA-7 polynomials and Cantera's R, from the guess in T.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void e_cv_of(const Mech* __restrict__ M, const double* y, double T,
                                        double& e, double& cv) {
  const int ns = M->ns;
  const double T2 = T * T, T3 = T2 * T, T4 = T3 * T;
  double h = 0.0, cp = 0.0, winv = 0.0;
  for (int k = 0; k < ns; k++) {
    const double* a = T <= M->tmid[k] ? M->lo[k] : M->hi[k];
    const double cpr = a[0] + a[1] * T + a[2] * T2 + a[3] * T3 + a[4] * T4;
    const double hrt = a[0] + a[1] * T / 2.0 + a[2] * T2 / 3.0 + a[3] * T3 / 4.0 + a[4] * T4 / 5.0 +
                       a[5] / T;
    const double yw = y[k] / M->W[k];
    h += yw * hrt * T;
    cp += yw * cpr;
    winv += yw;
  }
  e = kRgas * (h - winv * T);
  cv = kRgas * (cp - winv);
}

__global__ __launch_bounds__(256) void k_temperature(const Mech* __restrict__ M, long long n,
                                                     const double* __restrict__ Y,
                                                     const double* __restrict__ E,
                                                     double* __restrict__ T, int* __restrict__ iters) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double y[NSMAX];
  for (int k = 0; k < M->ns; k++) y[k] = Y[k * n + i];
  const double et = E[i];
  double t = T[i];
  int it = 0;
  for (; it < 50; it++) {
    double e, cv;
    e_cv_of(M, y, t, e, cv);
    const double dt = (et - e) / cv;
    t += dt;
    if (fabs(dt) <= 1e-13 * fabs(t)) break;
  }
  T[i] = t;
  if (iters) iters[i] = it + 1;
}

// ---------------------------------------------------------------------------
// 0-D constant-pressure adiabatic reactor (no reference counterpart: the
// reference's 0dreactor is constant-volume).  State y = (T, Y_1..Y_ns):
//   dY_k/dt = wdot_k W_k / rho,  dT/dt = -sum_k h_k dY_k/dt / cp,
// rho = p / (R T sum Y_k/W_k), h_k = (h/RT)_k R T / W_k, cp = R sum Y_k cpr_k/W_k,
// so the mixture enthalpy is conserved.  Integrated by RODAS4, the stiffly
// accurate, L-stable Rosenbrock method of order 4 with an embedded order-3
// solution (Hairer and Wanner, Solving Ordinary Differential Equations II,
// 2nd ed. 1996, Sect. VI.4), in the transformed form of their RODAS code:
// with A = I - gamma h J (J by forward differences, column by column),
//   U_i = gamma h A^-1 ( f(y + sum_{j<i} a_ij U_j) + sum_{j<i} (c_ij/h) U_j ),
// stage 6's argument Y_6 = Y_5 + U_5, y_new = Y_6 + U_6, error estimate U_6;
// step control h_new = h min(6, max(0.2, 0.9 err^(-1/4))) on a scaled
// max-norm.
// ---------------------------------------------------------------------------
constexpr double kRoGamma = 0.25;
// a_ij of stages 2..5 (row i-2 holds a_i1..a_i(i-1)) and c_ij of stages 2..6
constexpr double kRoA[4][4] = {
    {1.544, 0.0, 0.0, 0.0},
    {0.9466785280815826, 0.2557011698983284, 0.0, 0.0},
    {3.314825187068521, 2.896124015972201, 0.9986419139977817, 0.0},
    {1.221224509226641, 6.019134481288629, 12.53708332932087, -0.6878860361058950}};
constexpr double kRoC[5][5] = {
    {-5.6688, 0.0, 0.0, 0.0, 0.0},
    {-2.430093356833875, -0.2063599157091915, 0.0, 0.0, 0.0},
    {-0.1073529058151375, -9.594562251023355, -20.47028614809616, 0.0, 0.0},
    {7.496443313967647, -10.24680431464352, -33.99990352819905, 11.70890893206160, 0.0},
    {8.083246795921522, -7.981132988064893, -31.52159432874371, 16.31930543123136, -6.058818238834054}};

// the step-size factor after a step of scaled error err
__device__ __forceinline__ double ro_factor(double err, bool accepted) {
  if (accepted) return fmin(6.0, fmax(0.2, 0.9 / sqrt(sqrt(fmax(err, 1e-16)))));
  return err < 1e300 ? fmax(0.2, fmin(0.9, 0.9 / sqrt(sqrt(err)))) : 0.2;
}

constexpr int NYMAX = NSMAX + 1;

__device__ void reactor_rhs(const Mech* __restrict__ M, double p, const double* yv, double* f) {
  const int ns = M->ns;
  const double T = yv[0];
  const double* Y = yv + 1;
  double w[NSMAX], cpr[NSMAX], hrt[NSMAX];
  double winv = 0.0;
  for (int k = 0; k < ns; k++) winv += Y[k] / M->W[k];
  const double rho = p / (kRgas * T * winv);
  kinetics(M, T, rho, Y, w, cpr, hrt);
  double cp = 0.0, dh = 0.0;
  for (int k = 0; k < ns; k++) {
    cp += Y[k] * cpr[k] / M->W[k];
    const double dY = w[k] * M->W[k] / rho;
    f[1 + k] = dY;
    dh += hrt[k] * T / M->W[k] * dY;  // (h_k / R) dY_k/dt
  }
  f[0] = -dh / cp;                    // R cancels between h_k and cp
}

// LU with partial pivoting of the n x n matrix a (row-major, stride NYMAX)
__device__ bool lu_factor(double* a, int* piv, int n) {
  for (int k = 0; k < n; k++) {
    int pk = k;
    double m = fabs(a[k * NYMAX + k]);
    for (int i = k + 1; i < n; i++) {
      const double v = fabs(a[i * NYMAX + k]);
      if (v > m) { m = v; pk = i; }
    }
    piv[k] = pk;
    if (!(m > 0.0)) return false;
    if (pk != k)
      for (int j = 0; j < n; j++) {
        const double t = a[k * NYMAX + j];
        a[k * NYMAX + j] = a[pk * NYMAX + j];
        a[pk * NYMAX + j] = t;
      }
    const double inv = 1.0 / a[k * NYMAX + k];
    for (int i = k + 1; i < n; i++) {
      const double l = a[i * NYMAX + k] * inv;
      a[i * NYMAX + k] = l;
      for (int j = k + 1; j < n; j++) a[i * NYMAX + j] -= l * a[k * NYMAX + j];
    }
  }
  return true;
}

// The factorization swaps whole rows (its stored multipliers included), so
// the solve applies every interchange to b first, then the unit lower and the
// upper triangular solves (as LAPACK's getrs does).
__device__ void lu_solve(const double* a, const int* piv, int n, double* b) {
  for (int k = 0; k < n; k++) {
    if (piv[k] != k) {
      const double t = b[k];
      b[k] = b[piv[k]];
      b[piv[k]] = t;
    }
  }
  for (int k = 0; k < n; k++)
    for (int i = k + 1; i < n; i++) b[i] -= a[i * NYMAX + k] * b[k];
  for (int k = n - 1; k >= 0; k--) {
    double s = b[k];
    for (int j = k + 1; j < n; j++) s -= a[k * NYMAX + j] * b[j];
    b[k] = s / a[k * NYMAX + k];
  }
}

struct ReactorPool {
  double* y;     // NYMAX x cap: T then Y_k
  double* t;     // time reached
  double* h;     // next step size
  double* tend;
  double* p;
  int* status;   // 0 free, 1 running, 2 done, 3 failed
  int* nstep;    // accepted steps
  int* nrej;     // rejected steps
  int cap;
};

enum { RX_FREE = 0, RX_RUN = 1, RX_DONE = 2, RX_FAIL = 3 };

// Advance every running reactor by up to max_tries step attempts (or to its
// end time).  A reactor's steps depend only on its own state, so splitting a
// run into launches, or sharing a launch with other reactors, does not change
// its result.
__global__ __launch_bounds__(64) void k_reactor(const Mech* __restrict__ M, ReactorPool P,
                                                int max_tries, double rtol, double atol) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.cap || P.status[i] != RX_RUN) return;
  const int n = M->ns + 1;
  const double gam = kRoGamma;
  double y[NYMAX], f0[NYMAX], f1[NYMAX], yt[NYMAX], y5[NYMAX], U[6][NYMAX];
  double a[NYMAX * NYMAX];
  int piv[NYMAX];
  for (int k = 0; k < n; k++) y[k] = P.y[(size_t)k * P.cap + i];
  double t = P.t[i], h = P.h[i];
  const double tend = P.tend[i], p = P.p[i];
  int nstep = P.nstep[i], nrej = P.nrej[i], st = RX_RUN;
  for (int it = 0; it < max_tries; it++) {
    if (t >= tend) { st = RX_DONE; break; }
    if (h > tend - t) h = tend - t;
    if (!(h > 1e-18)) { st = RX_FAIL; break; }
    reactor_rhs(M, p, y, f0);
    // forward-difference Jacobian, column by column
    for (int j = 0; j < n; j++) {
      for (int k = 0; k < n; k++) yt[k] = y[k];
      // floor 1e-6 for mass fractions: a smaller step on a trace species
      // leaves the difference quotient to rounding
      const double d = 1.4901161193847656e-08 * fmax(fabs(y[j]), j == 0 ? 1.0 : 1e-6);
      yt[j] = y[j] + d;
      reactor_rhs(M, p, yt, f1);
      for (int k = 0; k < n; k++) a[k * NYMAX + j] = -gam * h * (f1[k] - f0[k]) / d;
    }
    for (int k = 0; k < n; k++) a[k * NYMAX + k] += 1.0;
    bool ok = lu_factor(a, piv, n);
    double err = 2.0;
    if (ok) {
      const double gh = gam * h;
      for (int k = 0; k < n; k++) U[0][k] = f0[k];
      lu_solve(a, piv, n, U[0]);
      for (int k = 0; k < n; k++) U[0][k] = gh * U[0][k];
      for (int s = 1; s < 6; s++) {
        for (int k = 0; k < n; k++) {
          double v = y[k];
          if (s < 5) {
            for (int j = 0; j < s; j++) v += kRoA[s - 1][j] * U[j][k];
            if (s == 4) y5[k] = v;
          } else {
            v = y5[k] + U[4][k];
          }
          yt[k] = v;
        }
        reactor_rhs(M, p, yt, f1);
        for (int k = 0; k < n; k++) {
          double c = 0.0;
          for (int j = 0; j < s; j++) c += (kRoC[s - 1][j] / h) * U[j][k];
          U[s][k] = f1[k] + c;
        }
        lu_solve(a, piv, n, U[s]);
        for (int k = 0; k < n; k++) U[s][k] = gh * U[s][k];
      }
      err = 0.0;
      for (int k = 0; k < n; k++) {
        const double yn = yt[k] + U[5][k];
        const double sc = (k == 0 ? 1e-6 : atol) + rtol * fmax(fabs(y[k]), fabs(yn));
        const double e = fabs(U[5][k]) / sc;
        if (!(e <= err)) err = e;  // a NaN makes err NaN and rejects the step
        yt[k] = yn;
      }
    }
    if (err <= 1.0) {
      t += h;
      for (int k = 0; k < n; k++) y[k] = yt[k];
      nstep++;
      h *= ro_factor(err, true);
    } else {
      nrej++;
      h *= ro_factor(err, false);
    }
    if (t >= tend) { st = RX_DONE; break; }
  }
  for (int k = 0; k < n; k++) P.y[(size_t)k * P.cap + i] = y[k];
  P.t[i] = t;
  P.h[i] = h;
  P.nstep[i] = nstep;
  P.nrej[i] = nrej;
  P.status[i] = st;
}

// ---------------------------------------------------------------------------
// The same reactor for a mechanism of exactly NS species, with every species
// loop unrolled so the per-reactor state stays in registers (the generic
// kernel's arrays, indexed at run time, live in scratch memory).  Species
// picked by a reaction (uniform indices) are read and updated through select
// chains; the Rosenbrock matrix of each thread sits in LDS, element (i,j) of
// thread t at [(i*N + j)*64 + t].  Same method, same arithmetic order as
// k_reactor.
// ---------------------------------------------------------------------------
template <int NS>
__device__ __forceinline__ double pick(const double (&v)[NS], int idx) {
  double r = v[0];
#pragma unroll
  for (int k = 1; k < NS; k++) r = idx == k ? v[k] : r;
  return r;
}

template <int NS>
__device__ __forceinline__ void add_at(double (&v)[NS], int idx, double x) {
#pragma unroll
  for (int k = 0; k < NS; k++)
    if (idx == k) v[k] += x;
}

// Lanes of a reactor team (one DPP row); the team kernel is further down.
constexpr int kTeam = 16;

// Inlined at every call, so that the caller's state arrays stay in registers
// (a call would take them by address, in scratch memory).
template <int NS>
__device__ __forceinline__ void reactor_rhs_n(const Mech* __restrict__ M, double p, const double (&yv)[NS + 1],
                                              double (&f)[NS + 1]) {
  const double T = yv[0];
  double c[NS], g[NS], w[NS], cpr[NS], hrt[NS];
  double winv = 0.0;
#pragma unroll
  for (int k = 0; k < NS; k++) winv += yv[1 + k] / M->W[k];
  const double rho = p / (kRgas * T * winv);
  const double logT = log(T), invT = 1.0 / T;
  const double T2 = T * T, T3 = T2 * T, T4 = T3 * T;
#pragma unroll
  for (int k = 0; k < NS; k++) {
    c[k] = rho * yv[1 + k] / M->W[k];
    const double* a = T <= M->tmid[k] ? M->lo[k] : M->hi[k];
    cpr[k] = a[0] + a[1] * T + a[2] * T2 + a[3] * T3 + a[4] * T4;
    hrt[k] = a[0] + a[1] * T / 2.0 + a[2] * T2 / 3.0 + a[3] * T3 / 4.0 + a[4] * T4 / 5.0 +
             a[5] * invT;
    const double sr = a[0] * logT + a[1] * T + a[2] * T2 / 2.0 + a[3] * T3 / 3.0 +
                      a[4] * T4 / 4.0 + a[6];
    g[k] = hrt[k] - sr;
    w[k] = 0.0;
  }
  const double lc0 = log(M->p0 / (kRgas * T));
  for (int r = 0; r < M->nr; r++) {
    const double kf = exp(M->lnA[r] + M->b[r] * logT - M->EaR[r] * invT);
    double fwd = kf;
    double dg = 0.0;
    for (int j = 0; j < M->nre[r]; j++) {
      const int sp = M->rsp[r][j];
      fwd *= conc_pow(pick<NS>(c, sp), M->rnu[r][j]);
      dg -= M->rnu[r][j] * pick<NS>(g, sp);
    }
    double rv = 0.0;
    if (M->rev[r]) {
      double pp = 1.0;
      for (int j = 0; j < M->npr[r]; j++) {
        const int sp = M->psp[r][j];
        pp *= conc_pow(pick<NS>(c, sp), M->pnu[r][j]);
        dg += M->pnu[r][j] * pick<NS>(g, sp);
      }
      const double kr = exp(M->lnA[r] + M->b[r] * logT - M->EaR[r] * invT + dg - M->dnu[r] * lc0);
      rv = kr * pp;
    }
    double q = fwd - rv;
    if (M->tb[r]) {
      double cm = 0.0;
#pragma unroll
      for (int k = 0; k < NS; k++) cm += M->eff[r][k] * c[k];
      q *= cm;
    }
    for (int j = 0; j < M->nre[r]; j++) add_at<NS>(w, M->rsp[r][j], -M->rnu[r][j] * q);
    for (int j = 0; j < M->npr[r]; j++) add_at<NS>(w, M->psp[r][j], M->pnu[r][j] * q);
  }
  double cp = 0.0, dh = 0.0;
#pragma unroll
  for (int k = 0; k < NS; k++) {
    cp += yv[1 + k] * cpr[k] / M->W[k];
    const double dY = w[k] * M->W[k] / rho;
    f[1 + k] = dY;
    dh += hrt[k] * T / M->W[k] * dY;
  }
  f[0] = -dh / cp;
}

// c^(nu-1) nu: the derivative of c^nu
__device__ __forceinline__ double conc_pow_d(double c, double nu) {
  return nu == 1.0 ? 1.0 : (nu == 2.0 ? 2.0 * c : nu * conc_pow_general(c, nu - 1.0));
}

// Column j (0: T, 1 + m: Y_m) of the reactor's Jacobian J = d f / d(T, Y),
// analytic, by the chain rule through the concentrations c_k = rho Y_k / W_k:
//   dc_k/dY_m = rho/W_m delta_km - c_k / (W_m sum_i Y_i/W_i),  dc_k/dT = -c_k/T,
// so per reaction, with s_r = sum_i c_i dq_r/dc_i (mass action is
// homogeneous: s_r = o_f fwd - o_r rev, times [M] and plus [M] (fwd - rev)
// for a three-body reaction, o = the sum of the orders),
//   dq_r/dY_m = dq_r/dc_m rho/W_m - s_r / (W_m sum Y/W),
//   dq_r/dT   = [M] (fwd dln kf/dT - rev dln kr/dT) - s_r / T,
//   dln kf/dT = b/T + E/(R T^2),  dln kr/dT = dln kf/dT - dH_r/(R T^2) + dnu_r/T;
// then f_Y = w W / rho and f_T = -sum_k h_k f_Yk / cp give the column.  f0 is
// f(y).  The one-thread kernel's form, a column at a time; the team forms its
// columns from the reactions' derivatives (Team::matrix).
template <int NS>
__device__ __forceinline__ void reactor_jac_col(const Mech* __restrict__ M, double p, const double (&yv)[NS + 1],
                                                const double (&f0)[NS + 1], int j, double (&col)[NS + 1]) {
#pragma clang fp contract(off)
  const double T = yv[0];
  double c[NS], g[NS], cpr[NS], hrt[NS], dw[NS];
  double winv = 0.0;
#pragma unroll
  for (int k = 0; k < NS; k++) winv += yv[1 + k] / M->W[k];
  const double rho = p / (kRgas * T * winv);
  const double logT = log(T), invT = 1.0 / T;
  const double T2 = T * T, T3 = T2 * T, T4 = T3 * T;
  double dcpm = 0.0;
#pragma unroll
  for (int k = 0; k < NS; k++) {
    c[k] = rho * yv[1 + k] / M->W[k];
    const double* a = T <= M->tmid[k] ? M->lo[k] : M->hi[k];
    cpr[k] = a[0] + a[1] * T + a[2] * T2 + a[3] * T3 + a[4] * T4;
    hrt[k] = a[0] + a[1] * T / 2.0 + a[2] * T2 / 3.0 + a[3] * T3 / 4.0 + a[4] * T4 / 5.0 + a[5] * invT;
    const double sr = a[0] * logT + a[1] * T + a[2] * T2 / 2.0 + a[3] * T3 / 3.0 + a[4] * T4 / 4.0 + a[6];
    g[k] = hrt[k] - sr;
    dw[k] = 0.0;
    if (j == 0) dcpm += yv[1 + k] * (a[1] + 2.0 * a[2] * T + 3.0 * a[3] * T2 + 4.0 * a[4] * T3) / M->W[k];
  }
  const int m = j - 1;
  const double cm_ = m >= 0 ? pick<NS>(c, m) : 0.0;
  const double Wm = m >= 0 ? M->W[m] : 1.0;
  const double lc0 = log(M->p0 / (kRgas * T));
  for (int r = 0; r < M->nr; r++) {
    const double kf = exp(M->lnA[r] + M->b[r] * logT - M->EaR[r] * invT);
    double fwd = kf, ofw = 0.0, dfw = 0.0, dg = 0.0, dh = 0.0;
    for (int q = 0; q < M->nre[r]; q++) {
      const int sp = M->rsp[r][q];
      const double nu = M->rnu[r][q];
      fwd *= conc_pow(pick<NS>(c, sp), nu);
      ofw += nu;
      dg -= nu * pick<NS>(g, sp);
      dh -= nu * pick<NS>(hrt, sp);
      if (sp == m) {
        double d = kf * conc_pow_d(cm_, nu);
        for (int q2 = 0; q2 < M->nre[r]; q2++)
          if (q2 != q) d *= conc_pow(pick<NS>(c, M->rsp[r][q2]), M->rnu[r][q2]);
        dfw += d;
      }
    }
    double rv = 0.0, orv = 0.0, drv = 0.0, dlkr = 0.0;
    const double dlkf = M->b[r] * invT + M->EaR[r] * invT * invT;
    if (M->rev[r]) {
      for (int q = 0; q < M->npr[r]; q++) {
        const int sp = M->psp[r][q];
        dg += M->pnu[r][q] * pick<NS>(g, sp);
        dh += M->pnu[r][q] * pick<NS>(hrt, sp);
      }
      const double kr = exp(M->lnA[r] + M->b[r] * logT - M->EaR[r] * invT + dg - M->dnu[r] * lc0);
      rv = kr;
      for (int q = 0; q < M->npr[r]; q++) {
        const int sp = M->psp[r][q];
        const double nu = M->pnu[r][q];
        rv *= conc_pow(pick<NS>(c, sp), nu);
        orv += nu;
        if (sp == m) {
          double d = kr * conc_pow_d(cm_, nu);
          for (int q2 = 0; q2 < M->npr[r]; q2++)
            if (q2 != q) d *= conc_pow(pick<NS>(c, M->psp[r][q2]), M->pnu[r][q2]);
          drv += d;
        }
      }
      dlkr = dlkf - dh * invT + M->dnu[r] * invT;
    }
    double s, dq;
    if (M->tb[r]) {
      double cmb = 0.0;
#pragma unroll
      for (int k = 0; k < NS; k++) cmb += M->eff[r][k] * c[k];
      s = cmb * ((ofw + 1.0) * fwd - (orv + 1.0) * rv);
      dq = m >= 0 ? cmb * (dfw - drv) + (fwd - rv) * M->eff[r][m] : cmb * (fwd * dlkf - rv * dlkr);
    } else {
      s = ofw * fwd - orv * rv;
      dq = m >= 0 ? dfw - drv : fwd * dlkf - rv * dlkr;
    }
    const double dqy = m >= 0 ? dq * rho / Wm - s / (Wm * winv) : dq - s * invT;
    for (int q = 0; q < M->nre[r]; q++) add_at<NS>(dw, M->rsp[r][q], -M->rnu[r][q] * dqy);
    for (int q = 0; q < M->npr[r]; q++) add_at<NS>(dw, M->psp[r][q], M->pnu[r][q] * dqy);
  }
  double cp = 0.0, dH = 0.0;
#pragma unroll
  for (int k = 0; k < NS; k++) {
    const double fY = f0[1 + k];
    const double v = M->W[k] / rho * dw[k] + (m >= 0 ? fY / (Wm * winv) : fY * invT);
    col[1 + k] = v;
    cp += yv[1 + k] * cpr[k] / M->W[k];
    dH += hrt[k] * T / M->W[k] * v;
    if (j == 0) dH += cpr[k] / M->W[k] * fY;
  }
  const double dcp = m >= 0 ? pick<NS>(cpr, m) / Wm : dcpm;
  col[0] = -(dH + f0[0] * dcp) / cp;
}

// solve with LU factors in LDS, element (r,c) of this thread's matrix at
// a[(r*N + c)*64]: the matrices of a wavefront's reactors are interleaved.
// The factorization swaps whole rows (its stored multipliers included), so
// every interchange is applied to b before the unit lower triangular solve.
template <int N>
__device__ __forceinline__ void lu_solve_n(const double* a, const int (&piv)[N], double (&b)[N]) {
#pragma unroll
  for (int k = 0; k < N; k++) {
    // the row swap of step k
    const double bk = b[k];
    double bp = bk;
#pragma unroll
    for (int r = k + 1; r < N; r++) bp = piv[k] == r ? b[r] : bp;
#pragma unroll
    for (int r = k + 1; r < N; r++)
      if (piv[k] == r) b[r] = bk;
    b[k] = bp;
  }
#pragma unroll
  for (int k = 0; k < N; k++) {
#pragma unroll
    for (int r = k + 1; r < N; r++) b[r] -= a[(r * N + k) * 64] * b[k];
  }
#pragma unroll
  for (int k = N - 1; k >= 0; k--) {
    double sum = b[k];
#pragma unroll
    for (int c = k + 1; c < N; c++) sum -= a[(k * N + c) * 64] * b[c];
    b[k] = sum / a[(k * N + k) * 64];
  }
}

// RODAS4's six stages from the factored A = I - gamma h J (in LDS)
// and f0 = f(y): the new state into ynew, the scaled error as the result
template <int NS>
__device__ __forceinline__ double ro_stages(const Mech* __restrict__ M, double p, double h, const double* a,
                                            const int (&piv)[NS + 1], const double (&y)[NS + 1],
                                            const double (&f0)[NS + 1], double (&ynew)[NS + 1], double rtol,
                                            double atol) {
  constexpr int N = NS + 1;
  double U[6][N], yt[N], y5[N], f1[N];
  const double gh = kRoGamma * h;
#pragma unroll
  for (int k = 0; k < N; k++) U[0][k] = f0[k];
  lu_solve_n<N>(a, piv, U[0]);
#pragma unroll
  for (int k = 0; k < N; k++) U[0][k] = gh * U[0][k];
#pragma unroll
  for (int s = 1; s < 6; s++) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      double v = y[k];
      if (s < 5) {
#pragma unroll
        for (int j = 0; j < s; j++) v += kRoA[s - 1][j] * U[j][k];
        if (s == 4) y5[k] = v;
      } else {
        v = y5[k] + U[4][k];
      }
      yt[k] = v;
    }
    reactor_rhs_n<NS>(M, p, yt, f1);
#pragma unroll
    for (int k = 0; k < N; k++) {
      double c = 0.0;
#pragma unroll
      for (int j = 0; j < s; j++) c += (kRoC[s - 1][j] / h) * U[j][k];
      U[s][k] = f1[k] + c;
    }
    lu_solve_n<N>(a, piv, U[s]);
#pragma unroll
    for (int k = 0; k < N; k++) U[s][k] = gh * U[s][k];
  }
  double err = 0.0;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const double yn = yt[k] + U[5][k];
    const double sc = (k == 0 ? 1e-6 : atol) + rtol * fmax(fabs(y[k]), fabs(yn));
    const double e = fabs(U[5][k]) / sc;
    if (!(e <= err)) err = e;  // a NaN makes err NaN and rejects the step
    ynew[k] = yn;
  }
  return err;
}

template <int NS>
__global__ __launch_bounds__(64) void k_reactor_n(const Mech* __restrict__ M, ReactorPool P,
                                                  int max_tries, double rtol, double atol) {
  constexpr int N = NS + 1;
  __shared__ double sA[N * N * 64];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.cap || P.status[i] != RX_RUN) return;
  double* a = sA + threadIdx.x;
#define AIJ(r, c) a[((r) * N + (c)) * 64]
  const double gam = kRoGamma;
  double y[N], f0[N], f1[N], yt[N];
  int piv[N];
#pragma unroll
  for (int k = 0; k < N; k++) y[k] = P.y[(size_t)k * P.cap + i];
  double t = P.t[i], h = P.h[i];
  const double tend = P.tend[i], p = P.p[i];
  int nstep = P.nstep[i], nrej = P.nrej[i], st = RX_RUN;
  for (int it = 0; it < max_tries; it++) {
    if (t >= tend) { st = RX_DONE; break; }
    if (h > tend - t) h = tend - t;
    if (!(h > 1e-18)) { st = RX_FAIL; break; }
    reactor_rhs_n<NS>(M, p, y, f0);
    // the analytic Jacobian, column by column: A = I - gamma h J
#pragma unroll 1
    for (int j = 0; j < N; j++) {
      reactor_jac_col<NS>(M, p, y, f0, j, f1);
#pragma unroll
      for (int k = 0; k < N; k++) AIJ(k, j) = -gam * h * f1[k];
    }
#pragma unroll
    for (int k = 0; k < N; k++) AIJ(k, k) += 1.0;
    // LU with partial pivoting (rows swapped in LDS)
    bool ok = true;
#pragma unroll
    for (int k = 0; k < N; k++) {
      int pk = k;
      double m = fabs(AIJ(k, k));
#pragma unroll
      for (int r = k + 1; r < N; r++) {
        const double v = fabs(AIJ(r, k));
        if (v > m) { m = v; pk = r; }
      }
      piv[k] = pk;
      ok = ok && (m > 0.0);
      if (pk != k) {
        for (int c = 0; c < N; c++) {
          const double tmp = AIJ(k, c);
          AIJ(k, c) = AIJ(pk, c);
          AIJ(pk, c) = tmp;
        }
      }
      const double inv = 1.0 / AIJ(k, k);
#pragma unroll
      for (int r = k + 1; r < N; r++) {
        const double l = AIJ(r, k) * inv;
        AIJ(r, k) = l;
#pragma unroll
        for (int c = k + 1; c < N; c++) AIJ(r, c) -= l * AIJ(k, c);
      }
    }
    double err = 2.0;
    if (ok) err = ro_stages<NS>(M, p, h, a, piv, y, f0, yt, rtol, atol);
    if (err <= 1.0) {
      t += h;
#pragma unroll
      for (int k = 0; k < N; k++) y[k] = yt[k];
      nstep++;
      h *= ro_factor(err, true);
    } else {
      nrej++;
      h *= ro_factor(err, false);
    }
    if (t >= tend) { st = RX_DONE; break; }
  }
#undef AIJ
#pragma unroll
  for (int k = 0; k < N; k++) P.y[(size_t)k * P.cap + i] = y[k];
  P.t[i] = t;
  P.h[i] = h;
  P.nstep[i] = nstep;
  P.nrej[i] = nrej;
  P.status[i] = st;
}


// The right-hand side and the analytic Jacobian of the one-thread integrator
// (before the -gamma h scaling) at n states, one thread per state: y, f
// row-major N per state, jac N x N per state (row k, column j)
template <int NS>
__global__ __launch_bounds__(64) void k_reactor_eval(const Mech* __restrict__ M, int n, const double* p,
                                                     const double* y, double* f, double* jac) {
  constexpr int N = NS + 1;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double yv[N], f0[N], yt[N], f1[N];
#pragma unroll
  for (int k = 0; k < N; k++) yv[k] = y[(size_t)i * N + k];
  reactor_rhs_n<NS>(M, p[i], yv, f0);
#pragma unroll
  for (int k = 0; k < N; k++) f[(size_t)i * N + k] = f0[k];
  if (!jac) return;
#pragma unroll 1
  for (int j = 0; j < N; j++) {
    reactor_jac_col<NS>(M, p[i], yv, f0, j, f1);
#pragma unroll
    for (int k = 0; k < N; k++) jac[((size_t)i * N + k) * N + j] = f1[k];
  }
  (void)yt;
}

// ---------------------------------------------------------------------------
// The same reactor integrated by a team of 16 lanes (one DPP row), four
// reactors per wavefront, for latency.  A few dozen reactors leave almost the
// whole chip idle, and what an ignition takes is the length of one reactor's
// chain of operations; so every vector of the method is spread over the lanes
// and nothing is computed twice:
//   lane l < N holds component l of the state and of every stage vector (0 the
//     temperature, 1 + k species k, whose thermodynamics it evaluates);
//   lane r evaluates reactions r, r + 16, r + 32, its records in registers;
//   lane j < N forms column j of the analytic Jacobian from the reactions'
//     derivatives, and after a transposition holds row j of I - gamma h J for
//     the elimination and the triangular solves.
// Sums over species and the solves' broadcasts go through DPP row operations;
// concentrations, reaction rates and the reactions' derivative rows go through
// the team's LDS, where each lane reads the species of its own reactions.
// A step attempt (six right-hand sides, a Jacobian, a factorisation, six
// solves) takes 18 us, against 167 us with the whole right-hand side's species
// part, the stage sums and the triangular solves repeated by every lane
// (20 attempts: 40 reactors 4.0 -> 0.36 ms, 1024 3.4 -> 0.32, 16384 14.6 ->
// 1.4; the one-thread kernel 13 ms at each).
// A team's lanes hold identical scalars (t, h, err), so its control flow is
// uniform; teams of one wavefront may diverge, which is why the kernel uses
// no workgroup barrier.  A team is part of one wavefront, whose LDS accesses
// complete in order, so a wave barrier (for the compiler) orders one lane's
// write before another lane's read.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void team_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int CTRL>
__device__ __forceinline__ double row_dpp(double v) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false));
}
// lane L's v on every lane of the team
template <int L>
__device__ __forceinline__ double row_lane(double v) {
  return row_dpp<0x150 + L>(v);  // row_newbcast
}
// The sum over the team, the same bits on every lane: after each rotation two
// lanes that differ by it hold the same pair of addends.
__device__ __forceinline__ double row_sum(double v) {
  v += row_dpp<0x128>(v);  // row_ror
  v += row_dpp<0x124>(v);
  v += row_dpp<0x122>(v);
  v += row_dpp<0x121>(v);
  return v;
}
// the largest bit pattern over the team
__device__ __forceinline__ unsigned long long row_max(unsigned long long u) {
  auto step = [&](double r) {
    const unsigned long long o = (unsigned long long)__double_as_longlong(r);
    u = o > u ? o : u;
  };
  step(row_dpp<0x128>(__longlong_as_double((long long)u)));
  step(row_dpp<0x124>(__longlong_as_double((long long)u)));
  step(row_dpp<0x122>(__longlong_as_double((long long)u)));
  step(row_dpp<0x121>(__longlong_as_double((long long)u)));
  return u;
}
// F(integral_constant<0>) ... F(integral_constant<N - 1>)
template <int N, class F, int K = 0>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (K < N) {
    f(std::integral_constant<int, K>{});
    static_for<N, F, K + 1>(static_cast<F&&>(f));
  }
}

// RODAS4's coefficients by the stage vector that they multiply: stage s > j
// takes kTeamA[j][s - 1 - j] U_j into its argument and kTeamC[j][s - 1 - j] / h
// U_j into its right-hand side.  Stage 5's argument is stage 4's plus U_4.
struct TeamCoef {
  double a[5][5] = {}, c[5][5] = {};
  constexpr TeamCoef() {
    for (int j = 0; j < 5; j++)
      for (int s = j + 1; s < 6; s++) {
        a[j][s - 1 - j] = s < 5 ? kRoA[s - 1][j] : j < 4 ? kRoA[3][j] : 1.0;
        c[j][s - 1 - j] = kRoC[s - 1][j];
      }
  }
};
__constant__ const TeamCoef kTeamCoef;

template <int NS, bool UNIT>
struct Team {
  static constexpr int N = NS + 1;
  static constexpr int RS = N + 2;  // row of the reactions' derivatives: N columns and where pads go
  struct Lds {
    double c[NS + 1], g[NS + 1], h[NS + 1];  // with a pad: 1, 0, 0
    double q[NRMAX];                         // zero past the last reaction
    double d[NRMAX][RS];
    double a[N][N];
  };
  // one reaction, with one side's terms at a time
  struct Rx {
    double lnA, b, EaR, of, ob, eff[NS];
    unsigned sp, fl;
  };
  struct Side {
    double prod, g, h, td[3];  // td: the product's derivative by each term's concentration
    int ix[3];
  };

  const Mech* __restrict__ M;
  Lds& S;
  const int lane, nr;
  const double p, ip;
  double W, iW, tmid, lo[15], hi[15];  // this lane's species (lanes without one: W = 0, iW = 0)
  Rx rx[2];                            // reactions lane and lane + 16
  double nu[32];                       // this species' coefficients in reactions 0..31
  const ExpK K;
  // of the last rhs()
  double T, invT, rho, winv, yw, cpr, hrt, cp;

  __device__ __forceinline__ static Rx record(const Mech* __restrict__ M, int r, int nr) {
    Rx x;
    const Mech::Rx& R = M->rx[r < nr ? r : 0];
    const bool tb = R.fl & 32;
    x.lnA = R.lnA, x.b = R.b, x.EaR = R.EaR, x.sp = R.sp, x.fl = r < nr ? R.fl : 0;
    x.of = x.ob = 0.0;
    for (int j = 0; j < M->nre[r < nr ? r : 0]; j++) x.of += M->rnu[r < nr ? r : 0][j];
    for (int j = 0; j < M->npr[r < nr ? r : 0]; j++) x.ob += M->pnu[r < nr ? r : 0][j];
#pragma unroll
    for (int k = 0; k < NS; k++) x.eff[k] = tb ? R.eff[k] : 0.0;
    return x;
  }

  __device__ __forceinline__ Team(const Mech* __restrict__ M_, Lds& S_, int lane_, double p_)
      : M(M_), S(S_), lane(lane_), nr(M_->nr), p(p_), ip(1.0 / p_) {
    const bool has = lane >= 1 && lane <= NS;
    const int k = has ? lane - 1 : 0;
    W = has ? M->W[k] : 0.0;
    iW = has ? M->iW[k] : 0.0;
    tmid = M->tmid[k];
    const double* c0 = &M->th[k][0].a0;
    const double* c1 = &M->th[k][1].a0;
#pragma unroll
    for (int j = 0; j < 15; j++) lo[j] = c0[j], hi[j] = c1[j];
    rx[0] = record(M, lane, nr);
    rx[1] = record(M, lane + kTeam, nr);
#pragma unroll
    for (int r = 0; r < 32; r++) nu[r] = has && r < nr ? M->rx[r].nu[k] : 0.0;
    if (lane == 0) S.c[NS] = 1.0, S.g[NS] = 0.0, S.h[NS] = 0.0;
    for (int r = lane; r < NRMAX; r += kTeam) S.q[r] = 0.0;
    team_sync();
  }

  // one side of a reaction from the concentrations in LDS
  template <bool DER>
  __device__ __forceinline__ Side side(const Rx& x, int r, bool products) const {
    Side s;
    if (UNIT || (x.fl & 64)) {
      const unsigned sp = products ? x.sp >> 12 : x.sp;
#pragma unroll
      for (int j = 0; j < 3; j++) s.ix[j] = sp >> (4 * j) & 15;
      const double c0 = S.c[s.ix[0]], c1 = S.c[s.ix[1]], c2 = S.c[s.ix[2]];
      s.g = S.g[s.ix[0]] + S.g[s.ix[1]] + S.g[s.ix[2]];
      s.prod = c0 * c1 * c2;
      if (DER) {
        s.h = S.h[s.ix[0]] + S.h[s.ix[1]] + S.h[s.ix[2]];
        s.td[0] = c1 * c2, s.td[1] = c0 * c2, s.td[2] = c0 * c1;
      }
      return s;
    }
    s.prod = 1.0, s.g = s.h = 0.0;
    double c[3], v[3], w[3];
    const int n = products ? M->npr[r] : M->nre[r];
#pragma unroll
    for (int j = 0; j < 3; j++) {
      s.ix[j] = j < n ? (products ? M->psp[r][j] : M->rsp[r][j]) : NS;
      v[j] = j < n ? (products ? M->pnu[r][j] : M->rnu[r][j]) : 0.0;
      c[j] = S.c[s.ix[j]];
      w[j] = j < n ? conc_pow(c[j], v[j]) : 1.0;
      s.prod *= w[j];
      s.g += v[j] * S.g[s.ix[j]];
      s.h += v[j] * S.h[s.ix[j]];
    }
    if (DER) {
#pragma unroll
      for (int j = 0; j < 3; j++)
        s.td[j] = j < n ? conc_pow_d(c[j], v[j]) * w[(j + 1) % 3] * w[(j + 2) % 3] : 0.0;
    }
    return s;
  }

  // The rates of NR reactions a lane, the first being r, into S.q, without a
  // branch (UNIT) so that their chains overlap; past the last reaction a lane
  // evaluates reaction 0 and stores zero.  DER: their rows of derivatives, into
  // S.d: column 0 dq/dT at fixed Y, column 1 + m dq/dY_m divided by rho/W_m.
  template <bool DER, int NR>
  __device__ __forceinline__ void reactions(const Rx* x, int r, double logT) const {
    Side f[NR], b[NR];
    double ex[2 * NR], k[2 * NR], cm[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) {
      const int ri = r + kTeam * i < nr ? r + kTeam * i : 0;
      f[i] = side<DER>(x[i], ri, false);
      b[i] = side<DER>(x[i], ri, true);
      ex[2 * i] = x[i].lnA + x[i].b * logT - x[i].EaR * invT;
      ex[2 * i + 1] = x[i].fl & 16 ? ex[2 * i] + (b[i].g - f[i].g) : 0.0;
      cm[i] = 0.0;
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const double c = S.c[s];
#pragma unroll
      for (int i = 0; i < NR; i++) cm[i] += x[i].eff[s] * c;
    }
    rate_exps(ex, K, k);
#pragma unroll
    for (int i = 0; i < NR; i++) {
      const bool rev = x[i].fl & 16, tb = x[i].fl & 32;
      const double kf = k[2 * i], kr = rev ? k[2 * i + 1] : 0.0;
      if (!tb) cm[i] = 1.0;
      const double fw = kf * f[i].prod, bw = rev ? kr * b[i].prod : 0.0, net = fw - bw;
      S.q[r + kTeam * i] = r + kTeam * i < nr ? cm[i] * net : 0.0;
      if constexpr (DER) {
        const double dlf = x[i].b * invT + x[i].EaR * invT * invT;
        const double dlr = dlf - (b[i].h - f[i].h) * invT + (x[i].ob - x[i].of) * invT;
        const double one = tb ? 1.0 : 0.0;
        const double s = cm[i] * ((x[i].of + one) * fw - (x[i].ob + one) * bw);
        const double base = s / (rho * winv);
        double* d = S.d[r + kTeam * i];
        d[0] = cm[i] * (fw * dlf - bw * dlr) - s * invT;
#pragma unroll
        for (int m = 0; m < NS; m++) d[1 + m] = net * x[i].eff[m] - base;
        const double cf = cm[i] * kf, cb = rev ? -cm[i] * kr : 0.0;
#pragma unroll
        for (int j = 0; j < 3; j++) add(&d[1 + f[i].ix[j]], cf * f[i].td[j]);
#pragma unroll
        for (int j = 0; j < 3; j++) add(&d[1 + b[i].ix[j]], rev ? cb * b[i].td[j] : 0.0);
      }
    }
  }
  // an addition that nothing waits for; one lane's own row, in its order
  __device__ __forceinline__ static void add(double* a, double v) {
    __builtin_amdgcn_ds_atomic_fadd_f64((__attribute__((address_space(3))) double*)a, v);
  }

  // this lane's component of f(y); y = 0 on the lanes past the last one
  template <bool DER>
  __device__ __forceinline__ double rhs(double y) {
    T = row_lane<0>(y);
    invT = 1.0 / T;
    const double logT = log(T), omlogT = 1.0 - logT, lc0 = M->lnp0R - logT;
    yw = y * iW;
    winv = row_sum(yw);
    const double rtw = kRgas * T * winv;
    rho = p / rtw;
    const bool low = T <= tmid;
    const auto poly = [&](const double (&r)[15], double& cpo, double& ho, double& go) {
      const double b = r[13] * invT;
      cpo = r[0] + T * (r[1] + T * (r[2] + T * (r[3] + T * r[4])));
      ho = r[0] + T * (r[5] + T * (r[6] + T * (r[7] + T * r[8]))) + b;
      go = r[0] * omlogT + T * (r[9] + T * (r[10] + T * (r[11] + T * r[12]))) + b - r[14] - lc0;
    };
    double c0, h0, g0, c1, h1, g1;
    poly(lo, c0, h0, g0);
    poly(hi, c1, h1, g1);
    cpr = low ? c0 : c1;
    hrt = low ? h0 : h1;
    if (lane >= 1 && lane <= NS) {
      S.c[lane - 1] = rho * yw;
      S.g[lane - 1] = low ? g0 : g1;
      if (DER) S.h[lane - 1] = hrt;
    }
    team_sync();
    if (nr > kTeam) reactions<DER, 2>(rx, lane, logT);
    else reactions<DER, 1>(rx, lane, logT);
    if (nr > 2 * kTeam) {
      const Rx x = record(M, lane + 2 * kTeam, nr);
      reactions<DER, 1>(&x, lane + 2 * kTeam, logT);
    }
    team_sync();
    double w[4] = {0.0, 0.0, 0.0, 0.0};
    const auto sum8 = [&](auto first) {
#pragma unroll
      for (int r = decltype(first)::value; r < decltype(first)::value + 8; r++) w[r & 3] += nu[r] * S.q[r];
    };
    sum8(std::integral_constant<int, 0>{});
    sum8(std::integral_constant<int, 8>{});
    if (nr > 16) sum8(std::integral_constant<int, 16>{});
    if (nr > 24) sum8(std::integral_constant<int, 24>{});
    if (nr > 32 && lane >= 1 && lane <= NS)
      for (int r = 32; r < nr; r++) w[r & 3] += M->rx[r].nu[lane - 1] * S.q[r];
    const double dY = ((w[0] + w[1]) + (w[2] + w[3])) * W * (rtw * ip);
    cp = row_sum(yw * cpr);
    const double dh = row_sum(hrt * T * iW * dY);
    return lane == 0 ? -dh / cp : dY;
  }

  // Row `lane` of A = I - gh J at the last rhs<true>(), f its result there.
  // Column j by lane j: with dw_k = sum_r nu_rk dq_r/dY_j,
  //   dY_k' = W_k/rho dw_k + f_k / (W_j sum Y/W)  (dT column: + f_k / T),
  //   dT'   = -(sum_k h_k dY_k' + f_T dcp) / cp.
  __device__ __forceinline__ void matrix(double f, double gh, double (&row)[N]) {
    double dw[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) dw[k] = 0.0;
    const int j = lane < N ? lane : 0;
#pragma unroll 2
    for (int r = 0; r < nr; r++) {
      const double q = S.d[r][j];
#pragma unroll
      for (int k = 0; k < NS; k++) dw[k] += M->rx[r].nu[k] * q;
    }
    const bool low = T <= tmid;
    const auto dpoly = [&](const double (&r)[15]) {
      return r[1] + T * (2.0 * r[2] + T * (3.0 * r[3] + T * (4.0 * r[4])));
    };
    const double dcpT = row_sum(yw * (low ? dpoly(lo) : dpoly(hi)));
    const double dcp = lane == 0 ? dcpT : cpr * iW;
    const double irho = kRgas * T * winv * ip;
    const double sc = lane == 0 ? irho : iW;       // rho/W_j of the derivatives' scaling, times 1/rho
    const double fs = lane == 0 ? invT : iW / winv;
    const double hk = hrt * T * iW, ck = cpr * iW;
    double dH = 0.0;
    static_for<NS>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const double fk = row_lane<1 + k>(f);
      const double v = row_lane<1 + k>(W) * sc * dw[k] + fk * fs;
      dw[k] = v;
      dH += row_lane<1 + k>(hk) * v;
      const double cT = row_lane<1 + k>(ck) * fk;
      dH += lane == 0 ? cT : 0.0;
    });
    const double top = -(dH + row_lane<0>(f) * dcp) / cp;
    if (lane < N) {
      S.a[0][lane] = (lane == 0 ? 1.0 : 0.0) - gh * top;
#pragma unroll
      for (int k = 0; k < NS; k++) S.a[1 + k][lane] = (lane == 1 + k ? 1.0 : 0.0) - gh * dw[k];
    }
    team_sync();
#pragma unroll
    for (int k = 0; k < N; k++) row[k] = S.a[j][k];
    team_sync();
  }

  // LU of the matrix whose row `lane` is a: pivots by the largest element (its
  // low four bits give way to the lane, so that one maximum finds both), rows
  // left where they are until the end, when lane i takes row src, position i.
  // lw: the multipliers left of the diagonal, up: the row right of it divided
  // by the diagonal element, dinv its reciprocal; zeros elsewhere.
  __device__ __forceinline__ bool factor(double (&a)[N], double (&lw)[N], double (&up)[N], double& dinv,
                                         int& src) {
    bool used = lane >= N, ok = true;
    double inv_own = 0.0;
    src = lane;
    static_for<N>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const unsigned long long mag = (unsigned long long)__double_as_longlong(fabs(a[k]));
      const unsigned long long best = row_max(used ? 0ull : (mag & ~15ull) | (unsigned)(15 - lane));
      const double inv = 1.0 / a[k];
      const int pk = 15 - (int)(best & 15);
      if (lane == k) src = pk;
      double piv[N];
#pragma unroll
      for (int c = k; c < N; c++) piv[c] = __shfl(a[c], pk, kTeam);
      ok = ok && fabs(piv[k]) > 0.0;
      const double pinv = __shfl(inv, pk, kTeam);
      if (lane == pk) {
        used = true;
        inv_own = inv;
      }
      const double l = used ? 0.0 : a[k] * pinv;
      if (!used) a[k] = l;
#pragma unroll
      for (int c = k + 1; c < N; c++) a[c] -= l * piv[c];
    });
    dinv = __shfl(inv_own, src, kTeam);
#pragma unroll
    for (int k = 0; k < N; k++) {
      const double v = __shfl(a[k], src, kTeam);
      lw[k] = k < lane && lane < N ? v : 0.0;
      up[k] = k > lane ? v * dinv : 0.0;
    }
    return ok;
  }

  // this lane's component of the solution for the right-hand side b
  __device__ __forceinline__ double solve(const double (&lw)[N], const double (&up)[N], double dinv, int src,
                                          double b) const {
    b = __shfl(b, src, kTeam);
    static_for<N - 1>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      b -= lw[k] * row_lane<k>(b);
    });
    b *= dinv;
    static_for<N - 1>([&](auto kc) {
      constexpr int k = N - 1 - decltype(kc)::value;
      b -= up[k] * row_lane<k>(b);
    });
    return b;
  }
};

template <int NS, bool UNIT>
__global__ __launch_bounds__(64) void k_reactor_team(const Mech* __restrict__ M, ReactorPool P,
                                                     int max_tries, double rtol, double atol) {
  using TeamN = Team<NS, UNIT>;
  constexpr int N = NS + 1;
  constexpr int TPB = 64 / kTeam;
  static_assert(N <= kTeam && NRMAX <= 3 * kTeam, "a lane per component, three reactions per lane");
  __shared__ typename TeamN::Lds lds[TPB];
  const int team = threadIdx.x / kTeam, lane = threadIdx.x % kTeam;
  const int i = blockIdx.x * TPB + team;
  if (i >= P.cap || P.status[i] != RX_RUN) return;  // the whole team leaves
  TeamN R(M, lds[team], lane, P.p[i]);
  double y = lane < N ? P.y[(size_t)lane * P.cap + i] : 0.0;
  double t = P.t[i], h = P.h[i];
  const double tend = P.tend[i];
  int nstep = P.nstep[i], nrej = P.nrej[i], st = RX_RUN;
  for (int it = 0; it < max_tries; it++) {
    if (t >= tend) { st = RX_DONE; break; }
    if (h > tend - t) h = tend - t;
    if (!(h > 1e-18)) { st = RX_FAIL; break; }
    const double gh = kRoGamma * h, ih = 1.0 / h;
    double f = R.template rhs<true>(y);
    double a[N], lw[N], up[N], dinv;
    int src;
    R.matrix(f, gh, a);
    const bool ok = R.factor(a, lw, up, dinv, src);
    double err = 2.0, yn = y;
    if (ok) {
      // the arguments and the U sums of the stages still to come, [0] the next
      double ya[5], cs[5];
#pragma unroll
      for (int s = 0; s < 5; s++) ya[s] = y, cs[s] = 0.0;
      double u = gh * R.solve(lw, up, dinv, src, f);
#pragma unroll 1
      for (int j = 0; j < 5; j++) {
#pragma unroll
        for (int s = 0; s < 5; s++) {
          ya[s] += kTeamCoef.a[j][s] * u;
          cs[s] += (kTeamCoef.c[j][s] * ih) * u;
        }
        yn = ya[0];
        f = R.template rhs<false>(yn);
        u = gh * R.solve(lw, up, dinv, src, f + cs[0]);
#pragma unroll
        for (int s = 0; s < 4; s++) ya[s] = ya[s + 1], cs[s] = cs[s + 1];
      }
      yn += u;
      const double sc = (lane == 0 ? 1e-6 : atol) + rtol * fmax(fabs(y), fabs(yn));
      // the largest of the lanes' errors; a NaN's bits are above all others,
      // it makes err NaN and rejects the step
      const double e = lane < N ? fabs(fabs(u) / sc) : 0.0;
      err = __longlong_as_double((long long)row_max((unsigned long long)__double_as_longlong(e)));
    }
    if (err <= 1.0) {
      t += h;
      y = yn;
      nstep++;
      h *= ro_factor(err, true);
    } else {
      nrej++;
      h *= ro_factor(err, false);
    }
    if (t >= tend) { st = RX_DONE; break; }
  }
  if (lane < N) P.y[(size_t)lane * P.cap + i] = y;
  if (lane == 0) {
    P.t[i] = t;
    P.h[i] = h;
    P.nstep[i] = nstep;
    P.nrej[i] = nrej;
    P.status[i] = st;
  }
}

// What the team integrator is made of, at n states laid out as in
// k_reactor_eval: the right-hand side, the Jacobian and the solution of
// (I - gh J) x = f by its factorisation and solve.  The Jacobian comes out of
// matrix(), which forms I - g J, with a power of two as -g that is large
// against any 1/J, so that taking I off costs no digits of J's entries.
template <int NS, bool UNIT>
__global__ __launch_bounds__(64) void k_reactor_team_eval(const Mech* __restrict__ M, int n, const double* p,
                                                          const double* y, double gh, double* f, double* jac,
                                                          double* sol) {
  using TeamN = Team<NS, UNIT>;
  constexpr int N = NS + 1;
  constexpr double kScale = 0x1p60;
  __shared__ typename TeamN::Lds lds[64 / kTeam];
  const int team = threadIdx.x / kTeam, lane = threadIdx.x % kTeam;
  const int i = blockIdx.x * (64 / kTeam) + team;
  if (i >= n) return;  // the whole team leaves
  TeamN R(M, lds[team], lane, p[i]);
  const double fl = R.template rhs<true>(lane < N ? y[(size_t)i * N + lane] : 0.0);
  if (lane < N) f[(size_t)i * N + lane] = fl;
  double row[N];
  if (jac) {
    R.matrix(fl, -kScale, row);
    if (lane < N)
#pragma unroll
      for (int j = 0; j < N; j++) jac[((size_t)i * N + lane) * N + j] = (row[j] - (lane == j ? 1.0 : 0.0)) / kScale;
  }
  if (sol) {
    double lw[N], up[N], dinv;
    int src;
    R.matrix(fl, gh, row);
    const bool ok = R.factor(row, lw, up, dinv, src);
    const double x = R.solve(lw, up, dinv, src, fl);
    if (lane < N) sol[(size_t)i * N + lane] = ok ? x : __longlong_as_double(0x7ff8000000000000ll);
  }
}

// A slot's state in and out: one launch each (set: 17 copies of 4 or 8 bytes
// before, get: 13).  A reactor set, read and released takes 47 us, 290 with
// the copies.
struct SlotState {
  double y[NYMAX], h, tend, p;
};
__global__ __launch_bounds__(64) void k_reactor_set(ReactorPool P, int slot, int n, SlotState s) {
  const int k = threadIdx.x;
#pragma unroll
  for (int j = 0; j < NYMAX; j++)
    if (k == j && j < n) P.y[(size_t)j * P.cap + slot] = s.y[j];
  if (k == 0) {
    P.t[slot] = 0.0;
    P.h[slot] = s.h;
    P.tend[slot] = s.tend;
    P.p[slot] = s.p;
    P.nstep[slot] = 0;
    P.nrej[slot] = 0;
    P.status[slot] = RX_RUN;
  }
}

// out: y, then at NYMAX t and the two step counts
__global__ __launch_bounds__(64) void k_reactor_get(ReactorPool P, int slot, int n, double* __restrict__ out) {
  const int k = threadIdx.x;
  if (k < n) out[k] = P.y[(size_t)k * P.cap + slot];
  if (k == NYMAX) out[k] = P.t[slot];
  if (k == NYMAX + 1) out[k] = (double)P.nstep[slot];
  if (k == NYMAX + 2) out[k] = (double)P.nrej[slot];
}

__global__ void k_reactor_mark(ReactorPool P, int slot, int status) { P.status[slot] = status; }

// ---------------------------------------------------------------------------
// CTML reading (the subset the reference's mechanisms use)
// ---------------------------------------------------------------------------
std::string trim(const std::string& s) {
  size_t a = s.find_first_not_of(" \t\r\n"), b = s.find_last_not_of(" \t\r\n");
  return a == std::string::npos ? std::string() : s.substr(a, b - a + 1);
}

// text between <tag ...> and </tag> starting at pos; attributes in attr
bool element(const std::string& x, const std::string& tag, size_t& pos, std::string& attr,
             std::string& body) {
  for (;;) {
    size_t a = x.find("<" + tag, pos);
    if (a == std::string::npos) return false;
    const char nc = x[a + 1 + tag.size()];
    if (nc != ' ' && nc != '>' && nc != '\t' && nc != '\n' && nc != '/') {
      pos = a + 1;
      continue;
    }
    size_t e = x.find('>', a);
    if (e == std::string::npos) return false;
    attr = x.substr(a + 1 + tag.size(), e - a - 1 - tag.size());
    if (x[e - 1] == '/') {
      body.clear();
      pos = e + 1;
      return true;
    }
    size_t c = x.find("</" + tag + ">", e);
    if (c == std::string::npos) return false;
    body = x.substr(e + 1, c - e - 1);
    pos = c + tag.size() + 3;
    return true;
  }
}

std::string attr_of(const std::string& attrs, const std::string& key) {
  size_t p = attrs.find(key + "=\"");
  if (p == std::string::npos) return "";
  p += key.size() + 2;
  size_t e = attrs.find('"', p);
  return attrs.substr(p, e - p);
}

// "A:1.0 B:2" -> pairs
std::vector<std::pair<std::string, double>> pairs_of(const std::string& s) {
  std::vector<std::pair<std::string, double>> out;
  std::istringstream is(s);
  std::string tok;
  while (is >> tok) {
    size_t c = tok.find(':');
    if (c == std::string::npos) continue;
    out.push_back({tok.substr(0, c), std::stod(tok.substr(c + 1))});
  }
  return out;
}

std::vector<double> floats_of(const std::string& s) {
  std::vector<double> v;
  std::string t = s;
  for (char& ch : t)
    if (ch == ',') ch = ' ';
  std::istringstream is(t);
  double d;
  while (is >> d) v.push_back(d);
  return v;
}

// atomic weights (kg/kmol) of the elements the reference's mechanisms use
double atomic_weight(const std::string& e) {
  static const std::map<std::string, double> w = {
      {"H", 1.008}, {"O", 15.999}, {"N", 14.007}, {"C", 12.011}, {"AR", 39.95}, {"Ar", 39.95},
      {"HE", 4.002602}, {"He", 4.002602}};
  auto it = w.find(e);
  return it == w.end() ? -1.0 : it->second;
}

// factor turning an activation energy in the given units into E/R (K)
bool ea_factor(const std::string& units, double& f) {
  if (units == "cal/mol") f = 4184.0 / kRgas;
  else if (units == "kcal/mol") f = 4184000.0 / kRgas;
  else if (units == "J/mol") f = 1000.0 / kRgas;
  else if (units == "kJ/mol") f = 1.0e6 / kRgas;
  else if (units == "J/kmol") f = 1.0 / kRgas;
  else if (units == "K") f = 1.0;
  else return false;
  return true;
}

// the cell kernels' form of the mechanism (Mech::th, rx)
void prepare_cells(Mech& m) {
  m.lnp0R = std::log(m.p0 / kRgas);
  for (int k = 0; k < m.ns; k++) {
    m.iW[k] = 1.0 / m.W[k];
    m.rW[k] = kRref / m.W[k];
    for (int q = 0; q < 2; q++) {
      const double* a = q == 0 ? m.lo[k] : m.hi[k];
      m.th[k][q] = {a[0], a[1], a[2], a[3], a[4], a[1] / 2.0, a[2] / 3.0, a[3] / 4.0, a[4] / 5.0,
                    -a[1] / 2.0, -a[2] / 6.0, -a[3] / 12.0, -a[4] / 20.0, a[5], a[6]};
    }
  }
  m.unit = 1;
  for (int r = 0; r < m.nr; r++) {
    Mech::Rx& R = m.rx[r];
    R.lnA = m.lnA[r];
    R.b = m.b[r];
    R.EaR = m.EaR[r];
    R.sp = 0;
    R.fl = (m.rev[r] ? 16u : 0u) | (m.tb[r] ? 32u : 0u) | 64u;
    for (int k = 0; k < m.ns; k++) {
      R.nu[k] = 0.0;
      R.eff[k] = m.eff[r][k];
    }
    for (int side = 0; side < 2; side++) {
      const int n = side ? m.npr[r] : m.nre[r];
      const int* sp = side ? m.psp[r] : m.rsp[r];
      const double* nu = side ? m.pnu[r] : m.rnu[r];
      int terms = 0;
      for (int j = 0; j < n; j++) {
        R.nu[sp[j]] += side ? nu[j] : -nu[j];
        const int whole = nu[j] == 1.0 ? 1 : nu[j] == 2.0 ? 2 : nu[j] == 3.0 ? 3 : NTERM + 1;
        for (int i = 0; i < whole && terms <= NTERM; i++, terms++)
          if (terms < NTERM) R.sp |= (unsigned)sp[j] << (12 * side + 4 * terms);
      }
      if (terms < 1 || terms > NTERM) {
        R.fl &= ~64u;
        m.unit = 0;
      }
      for (int i = terms; i < NTERM; i++)  // RegArray's pad
        if (m.ns < NSMAX) R.sp |= (unsigned)m.ns << (12 * side + 4 * i);
      R.fl |= (unsigned)(terms & 3) << (2 * side);
    }
  }
}

int parse_ctml(const std::string& path, const std::string& phase_id, Mech& m,
               std::vector<std::string>& names) {
  std::ifstream f(path);
  if (!f) return cfail("cannot open mechanism file " + path);
  std::stringstream ss;
  ss << f.rdbuf();
  const std::string x = ss.str();
  std::memset(&m, 0, sizeof(m));
  // phase: species order
  size_t pos = 0;
  std::string attr, body;
  bool found = false;
  while (element(x, "phase", pos, attr, body)) {
    if (attr_of(attr, "id") == phase_id) { found = true; break; }
  }
  if (!found) return cfail("phase '" + phase_id + "' not found in " + path);
  {
    size_t p2 = 0;
    std::string a2, b2;
    if (!element(body, "speciesArray", p2, a2, b2)) return cfail("phase without speciesArray");
    std::istringstream is(b2);
    std::string nm;
    while (is >> nm) names.push_back(nm);
    p2 = 0;
    if (element(body, "kinetics", p2, a2, b2) && attr_of(a2, "model") != "GasKinetics")
      return cfail("unsupported kinetics model " + attr_of(a2, "model"));
  }
  m.ns = (int)names.size();
  if (m.ns < 1 || m.ns > NSMAX) return cfail("species count out of range");
  std::map<std::string, int> idx;
  for (int k = 0; k < m.ns; k++) idx[names[k]] = k;
  // species data
  int nfound = 0;
  pos = 0;
  m.p0 = -1.0;
  while (element(x, "species", pos, attr, body)) {
    auto it = idx.find(attr_of(attr, "name"));
    if (it == idx.end()) continue;
    const int k = it->second;
    size_t p2 = 0;
    std::string a2, b2;
    if (!element(body, "atomArray", p2, a2, b2)) return cfail("species without atomArray");
    double W = 0.0;
    for (auto& pr : pairs_of(b2)) {
      const double aw = atomic_weight(pr.first);
      if (aw < 0) return cfail("unknown element " + pr.first);
      W += pr.second * aw;
    }
    m.W[k] = W;
    p2 = 0;
    int nr = 0;
    while (element(body, "NASA", p2, a2, b2)) {
      size_t p3 = 0;
      std::string a3, b3;
      if (!element(b2, "floatArray", p3, a3, b3)) return cfail("NASA block without coeffs");
      auto v = floats_of(b3);
      if (v.size() != 7) return cfail("NASA block needs 7 coefficients");
      const double tmin = std::stod(attr_of(a2, "Tmin")), tmax = std::stod(attr_of(a2, "Tmax"));
      const std::string sp0 = attr_of(a2, "P0");
      if (!sp0.empty()) m.p0 = std::stod(sp0);
      double* dst = nr == 0 ? m.lo[k] : m.hi[k];
      for (int j = 0; j < 7; j++) dst[j] = v[j];
      if (nr == 0) m.tmid[k] = tmax;
      else if (tmin < m.tmid[k]) {  // listed high range first: swap
        double tmp[7];
        std::memcpy(tmp, m.lo[k], sizeof(tmp));
        std::memcpy(m.lo[k], m.hi[k], sizeof(tmp));
        std::memcpy(m.hi[k], tmp, sizeof(tmp));
        m.tmid[k] = tmax;
      }
      nr++;
    }
    if (nr != 2) return cfail("species " + names[k] + " needs two NASA ranges");
    nfound++;
  }
  if (nfound != m.ns) return cfail("species data missing for some phase species");
  if (m.p0 <= 0) m.p0 = 101325.0;
  // reactions
  pos = 0;
  int r = 0;
  while (element(x, "reaction", pos, attr, body)) {
    if (r >= NRMAX) return cfail("too many reactions");
    const std::string type = attr_of(attr, "type");
    if (!type.empty() && type != "threeBody") return cfail("unsupported reaction type " + type);
    m.tb[r] = type == "threeBody";
    m.rev[r] = attr_of(attr, "reversible") != "no";
    size_t p2 = 0;
    std::string a2, b2;
    if (!element(body, "Arrhenius", p2, a2, b2)) return cfail("reaction without Arrhenius");
    {
      size_t p3 = 0;
      std::string a3, b3;
      if (!element(b2, "A", p3, a3, b3)) return cfail("Arrhenius without A");
      const double A = std::stod(trim(b3));
      p3 = 0;
      if (!element(b2, "b", p3, a3, b3)) return cfail("Arrhenius without b");
      m.b[r] = std::stod(trim(b3));
      p3 = 0;
      if (!element(b2, "E", p3, a3, b3)) return cfail("Arrhenius without E");
      std::string u = attr_of(a3, "units");
      if (u.empty()) u = "cal/mol";
      double fac = 0.0;
      if (!ea_factor(u, fac)) return cfail("unsupported energy units " + u);
      m.EaR[r] = std::stod(trim(b3)) * fac;
      if (A <= 0) return cfail("non-positive pre-exponential factor");
      m.lnA[r] = std::log(A);
    }
    for (int k = 0; k < m.ns; k++) m.eff[r][k] = 1.0;
    p2 = 0;
    if (element(body, "efficiencies", p2, a2, b2)) {
      const std::string d = attr_of(a2, "default");
      const double def = d.empty() ? 1.0 : std::stod(d);
      for (int k = 0; k < m.ns; k++) m.eff[r][k] = def;
      for (auto& pr : pairs_of(b2)) {
        auto it = idx.find(pr.first);
        if (it != idx.end()) m.eff[r][it->second] = pr.second;
      }
    }
    double sr = 0.0, sp = 0.0;
    p2 = 0;
    if (!element(body, "reactants", p2, a2, b2)) return cfail("reaction without reactants");
    for (auto& pr : pairs_of(b2)) {
      auto it = idx.find(pr.first);
      if (it == idx.end() || m.nre[r] >= NTERM) return cfail("bad reactant " + pr.first);
      m.rsp[r][m.nre[r]] = it->second;
      m.rnu[r][m.nre[r]++] = pr.second;
      sr += pr.second;
    }
    p2 = 0;
    if (!element(body, "products", p2, a2, b2)) return cfail("reaction without products");
    for (auto& pr : pairs_of(b2)) {
      auto it = idx.find(pr.first);
      if (it == idx.end() || m.npr[r] >= NTERM) return cfail("bad product " + pr.first);
      m.psp[r][m.npr[r]] = it->second;
      m.pnu[r][m.npr[r]++] = pr.second;
      sp += pr.second;
    }
    m.dnu[r] = sp - sr;
    r++;
  }
  m.nr = r;
  prepare_cells(m);
  return 0;
}

}  // namespace

struct astr_chem {
  Mech host;
  Mech* dev = nullptr;
  std::vector<std::string> names;
  int device = 0;
};

struct astr_reactor_pool {
  astr_chem* chem = nullptr;
  ReactorPool P{};
  void* base = nullptr;
  double rtol = 1e-6, atol = 1e-12;
  hipStream_t stream = nullptr;
  int lanes = 1;  // lanes per reactor: 1, or kTeam for the team kernel
  double* pin = nullptr;  // pinned host memory that k_reactor_get writes, one call at a time
  std::mutex pin_mutex;
};

extern "C" {

const char* astr_hip_chem_last_error(void) { return g_cerr.c_str(); }

int astr_hip_chem_create(const char* ctml_path, const char* phase_id, astr_chem** out) {
  if (!ctml_path || !out) return cfail("null argument");
  *out = nullptr;
  astr_chem* c = new astr_chem();
  if (parse_ctml(ctml_path, phase_id ? phase_id : "gas", c->host, c->names)) {
    delete c;
    return -1;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
    delete c;
    return cfail("no HIP device");
  }
  (void)hipGetDevice(&c->device);
  if (hipMalloc(&c->dev, sizeof(Mech)) != hipSuccess) {
    delete c;
    return cfail("hipMalloc of mechanism failed");
  }
  if (hipMemcpy(c->dev, &c->host, sizeof(Mech), hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(c->dev);
    delete c;
    return cfail("copy of mechanism failed");
  }
  *out = c;
  return 0;
}

int astr_hip_chem_destroy(astr_chem* c) {
  if (!c) return 0;
  (void)hipSetDevice(c->device);
  (void)hipFree(c->dev);
  delete c;
  return 0;
}

int astr_hip_chem_info(astr_chem* c, int* nsp, int* nrx, double* mw, char* names, int name_len) {
  if (!c) return cfail("null mechanism");
  if (nsp) *nsp = c->host.ns;
  if (nrx) *nrx = c->host.nr;
  for (int k = 0; k < c->host.ns; k++) {
    if (mw) mw[k] = c->host.W[k];
    if (names && name_len > 0) {
      std::strncpy(names + (size_t)k * name_len, c->names[k].c_str(), name_len - 1);
      names[(size_t)k * name_len + name_len - 1] = 0;
    }
  }
  return 0;
}

int astr_hip_chem_rates_device(astr_chem* c, long long n, const double* T, const double* rho_or_p,
                               int input_is_p, const double* Y, double* wdot, double* h_mix,
                               double* cp_mix, double* h_k, void* stream) {
  if (!c) return cfail("null mechanism");
  if (n < 0) return cfail("negative cell count");
  if (n == 0) return 0;
  if (!T || !rho_or_p || !Y || !wdot) return cfail("null buffer");
  CHIP_OK(hipSetDevice(c->device));
  const int bs = kCellBlock;
  const dim3 grid((unsigned)((n + bs - 1) / bs));
  const bool nine = c->host.ns == 9, unit = c->host.unit != 0;
  auto kern = nine ? (unit ? k_chem<9, true> : k_chem<9, false>)
                   : (unit ? k_chem<NSMAX, true> : k_chem<NSMAX, false>);
  hipLaunchKernelGGL(kern, grid, dim3(bs), 0, (hipStream_t)stream, c->dev, n, T, rho_or_p, input_is_p,
                     Y, wdot, h_mix, cp_mix, h_k);
  CHIP_OK(hipGetLastError());
  return 0;
}

int astr_hip_chem_rates(astr_chem* c, long long n, const double* T, const double* rho_or_p,
                        int input_is_p, const double* Y, double* wdot, double* h_mix,
                        double* cp_mix, double* h_k) {
  if (!c) return cfail("null mechanism");
  if (n < 0) return cfail("negative cell count");
  if (n == 0) return 0;
  if (!T || !rho_or_p || !Y || !wdot) return cfail("null buffer");
  CHIP_OK(hipSetDevice(c->device));
  const int ns = c->host.ns;
  const size_t b1 = (size_t)n * sizeof(double);
  double* d = nullptr;
  const size_t nbuf = 2 + 2 * (size_t)ns + 2 + (h_k ? ns : 0);
  CHIP_OK(hipMalloc(&d, nbuf * b1));
  double* dT = d;
  double* dR = dT + n;
  double* dY = dR + n;
  double* dW = dY + (size_t)ns * n;
  double* dH = dW + (size_t)ns * n;
  double* dC = dH + n;
  double* dK = h_k ? dC + n : nullptr;
  int rc = 0;
  if (hipMemcpy(dT, T, b1, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dR, rho_or_p, b1, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dY, Y, b1 * ns, hipMemcpyHostToDevice) != hipSuccess) {
    rc = cfail("copy to device failed");
  }
  if (!rc) rc = astr_hip_chem_rates_device(c, n, dT, dR, input_is_p, dY, dW, dH, dC, dK, nullptr);
  if (!rc && hipDeviceSynchronize() != hipSuccess) rc = cfail("chemistry kernel failed");
  if (!rc) {
    if (hipMemcpy(wdot, dW, b1 * ns, hipMemcpyDeviceToHost) != hipSuccess ||
        (h_mix && hipMemcpy(h_mix, dH, b1, hipMemcpyDeviceToHost) != hipSuccess) ||
        (cp_mix && hipMemcpy(cp_mix, dC, b1, hipMemcpyDeviceToHost) != hipSuccess) ||
        (h_k && hipMemcpy(h_k, dK, b1 * ns, hipMemcpyDeviceToHost) != hipSuccess))
      rc = cfail("copy from device failed");
  }
  (void)hipFree(d);
  return rc;
}

static int srccomb_check(astr_chem* c, int im, int jm, int km, int hm, int numq, const void* rho,
                         const void* tmp, const void* spc, const void* jacob, const void* qrhs) {
  if (!c) return cfail("srccomb: null mechanism");
  if (im < 0 || jm < 0 || km < 0 || hm < 0) return cfail("srccomb: negative extent or halo");
  if (numq != 5 + c->host.ns)
    return cfail("srccomb: numq must be 5 + the species count (qrhs(6:numq) takes the rates)");
  if (!rho || !tmp || !spc || !jacob || !qrhs) return cfail("srccomb: null buffer");
  return 0;
}

int astr_hip_srccomb_device(astr_chem* c, int im, int jm, int km, int hm, int numq, const double* rho,
                            const double* tmp, const double* spc, const double* jacob, double* qrhs,
                            void* stream) {
  if (int rc = srccomb_check(c, im, jm, km, hm, numq, rho, tmp, spc, jacob, qrhs)) return rc;
  CHIP_OK(hipSetDevice(c->device));
  const long long ncell = (long long)(im + 1) * (jm + 1) * (km + 1);
  const int bs = kCellBlock;
  const dim3 grid((unsigned)((ncell + bs - 1) / bs));
  const bool nine = c->host.ns == 9, unit = c->host.unit != 0;
  auto kern = nine ? (unit ? k_srccomb<9, true> : k_srccomb<9, false>)
                   : (unit ? k_srccomb<NSMAX, true> : k_srccomb<NSMAX, false>);
  hipLaunchKernelGGL(kern, grid, dim3(bs), 0, (hipStream_t)stream, c->dev, im, jm, km, hm, rho, tmp, spc,
                     jacob, qrhs);
  CHIP_OK(hipGetLastError());
  return 0;
}

int astr_hip_srccomb(astr_chem* c, int im, int jm, int km, int hm, int numq, const double* rho,
                     const double* tmp, const double* spc, const double* jacob, double* qrhs) {
  if (int rc = srccomb_check(c, im, jm, km, hm, numq, rho, tmp, spc, jacob, qrhs)) return rc;
  CHIP_OK(hipSetDevice(c->device));
  const size_t nh = (size_t)(im + 1 + 2 * hm) * (jm + 1 + 2 * hm) * (km + 1 + 2 * hm);
  const size_t nq = (size_t)(im + 1) * (jm + 1) * (km + 1) * numq;
  const size_t ns = c->host.ns;
  double* d = nullptr;
  CHIP_OK(hipMalloc(&d, ((3 + ns) * nh + nq) * sizeof(double)));
  double *dr = d, *dt = dr + nh, *dj = dt + nh, *ds = dj + nh, *dq = ds + ns * nh;
  const size_t b = nh * sizeof(double);
  int rc = 0;
  if (hipMemcpy(dr, rho, b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dt, tmp, b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dj, jacob, b, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(ds, spc, b * ns, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dq, qrhs, nq * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
    rc = cfail("srccomb: copy to device failed");
  if (!rc) rc = astr_hip_srccomb_device(c, im, jm, km, hm, numq, dr, dt, ds, dj, dq, nullptr);
  if (!rc && hipDeviceSynchronize() != hipSuccess) rc = cfail("srccomb: kernel failed");
  if (!rc && hipMemcpy(qrhs, dq, nq * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
    rc = cfail("srccomb: copy from device failed");
  (void)hipFree(d);
  return rc;
}

int astr_hip_reactor_rhs(astr_chem* chem, int n, const double* p, const double* y, double* f, double* jac) {
  if (!chem || !p || !y || !f || n < 1) return cfail("reactor_rhs: null argument or no states");
  if (chem->host.ns != 9) return cfail("reactor_rhs: 9-species mechanisms only (the unrolled kernel)");
  CHIP_OK(hipSetDevice(chem->device));
  constexpr int N = 10;
  double* d = nullptr;
  const size_t ny = (size_t)n * N, nj = jac ? (size_t)n * N * N : 0;
  CHIP_OK(hipMalloc(&d, (n + 2 * ny + nj) * sizeof(double)));
  double *dp = d, *dy = d + n, *df = dy + ny, *dj = jac ? df + ny : nullptr;
  int rc = 0;
  if (hipMemcpy(dp, p, n * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dy, y, ny * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
    rc = cfail("reactor_rhs: copy in failed");
  } else {
    hipLaunchKernelGGL(k_reactor_eval<9>, dim3((n + 63) / 64), dim3(64), 0, nullptr, chem->dev, n, dp, dy, df, dj);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(f, df, ny * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess ||
        (jac && hipMemcpy(jac, dj, nj * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess))
      rc = cfail("reactor_rhs: kernel or copy out failed");
  }
  (void)hipFree(d);
  return rc;
}

int astr_hip_reactor_team_eval(astr_chem* chem, int n, const double* p, const double* y, double gh, double* f,
                               double* jac, double* sol) {
  if (!chem || !p || !y || !f || n < 1) return cfail("reactor_team_eval: null argument or no states");
  if (chem->host.ns != 9) return cfail("reactor_team_eval: 9-species mechanisms only (the team kernel)");
  CHIP_OK(hipSetDevice(chem->device));
  constexpr int N = 10;
  double* d = nullptr;
  const size_t ny = (size_t)n * N, nj = ny * N;
  CHIP_OK(hipMalloc(&d, (n + 3 * ny + nj) * sizeof(double)));
  double *dp = d, *dy = d + n, *df = dy + ny, *ds = df + ny, *dj = ds + ny;
  int rc = 0;
  if (hipMemcpy(dp, p, n * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dy, y, ny * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
    rc = cfail("reactor_team_eval: copy in failed");
  } else {
    constexpr int per = 64 / kTeam;
    hipLaunchKernelGGL((chem->host.unit ? k_reactor_team_eval<9, true> : k_reactor_team_eval<9, false>),
                       dim3((n + per - 1) / per), dim3(64), 0, nullptr, chem->dev, n, dp, dy, gh, df,
                       jac ? dj : nullptr, sol ? ds : nullptr);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(f, df, ny * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess ||
        (sol && hipMemcpy(sol, ds, ny * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess) ||
        (jac && hipMemcpy(jac, dj, nj * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess))
      rc = cfail("reactor_team_eval: kernel or copy out failed");
  }
  (void)hipFree(d);
  return rc;
}

int astr_hip_reactor_method(double* coef, int n) {
  if (!coef || n < 26) return cfail("reactor_method needs 26 values");
  int k = 0;
  coef[k++] = kRoGamma;
  for (int i = 0; i < 4; i++)
    for (int j = 0; j <= i; j++) coef[k++] = kRoA[i][j];
  for (int i = 0; i < 5; i++)
    for (int j = 0; j <= i; j++) coef[k++] = kRoC[i][j];
  return 0;
}

int astr_hip_reactor_create(astr_chem* chem, int capacity, double rtol, double atol,
                            astr_reactor_pool** out) {
  if (!chem || !out || capacity < 1) return cfail("bad argument to astr_hip_reactor_create");
  if (!(rtol > 0.0) || !(atol > 0.0)) return cfail("tolerances must be positive");
  *out = nullptr;
  CHIP_OK(hipSetDevice(chem->device));
  astr_reactor_pool* r = new astr_reactor_pool();
  r->chem = chem;
  r->rtol = rtol;
  r->atol = atol;
  const size_t cap = (size_t)capacity;
  const size_t bytes = (NYMAX + 4) * cap * sizeof(double) + 4 * cap * sizeof(int);
  if (hipMalloc(&r->base, bytes) != hipSuccess) { delete r; return cfail("hipMalloc of reactor pool failed"); }
  double* d = (double*)r->base;
  r->P.y = d;
  r->P.t = d + NYMAX * cap;
  r->P.h = r->P.t + cap;
  r->P.tend = r->P.h + cap;
  r->P.p = r->P.tend + cap;
  int* iv = (int*)(r->P.p + cap);
  r->P.status = iv;
  r->P.nstep = iv + cap;
  r->P.nrej = iv + 2 * cap;
  r->P.cap = capacity;
  r->lanes = chem->host.ns == 9 ? kTeam : 1;
  if (hipHostMalloc(&r->pin, (NYMAX + 3) * sizeof(double), hipHostMallocDefault) != hipSuccess ||
      hipMemset(r->base, 0, bytes) != hipSuccess ||
      hipStreamCreateWithFlags(&r->stream, hipStreamNonBlocking) != hipSuccess) {
    (void)hipFree(r->base);
    if (r->pin) (void)hipHostFree(r->pin);
    delete r;
    return cfail("reactor pool set-up failed");
  }
  *out = r;
  return 0;
}

int astr_hip_reactor_destroy(astr_reactor_pool* r) {
  if (!r) return 0;
  (void)hipSetDevice(r->chem->device);
  (void)hipStreamSynchronize(r->stream);
  (void)hipFree(r->base);
  (void)hipHostFree(r->pin);
  (void)hipStreamDestroy(r->stream);
  delete r;
  return 0;
}

int astr_hip_reactor_set(astr_reactor_pool* r, int slot, double T0, double p, const double* Y0,
                         double t_end, double h0) {
  if (!r || !Y0) return cfail("null argument");
  if (slot < 0 || slot >= r->P.cap) return cfail("reactor slot out of range");
  if (!(T0 > 0.0) || !(p > 0.0) || !(t_end >= 0.0) || !(h0 > 0.0)) return cfail("bad reactor state");
  CHIP_OK(hipSetDevice(r->chem->device));
  const int ns = r->chem->host.ns;
  SlotState st{};
  st.y[0] = T0;
  for (int k = 0; k < ns; k++) st.y[1 + k] = Y0[k];
  st.h = h0;
  st.tend = t_end;
  st.p = p;
  hipLaunchKernelGGL(k_reactor_set, dim3(1), dim3(64), 0, r->stream, r->P, slot, ns + 1, st);
  CHIP_OK(hipGetLastError());
  CHIP_OK(hipStreamSynchronize(r->stream));
  return 0;
}

int astr_hip_reactor_advance(astr_reactor_pool* r, int max_tries) {
  if (!r) return cfail("null pool");
  if (max_tries < 1) return cfail("max_tries must be positive");
  CHIP_OK(hipSetDevice(r->chem->device));
  const int bs = 64;
  const dim3 grid((r->P.cap + bs - 1) / bs);
  if (r->lanes == kTeam)
    hipLaunchKernelGGL((r->chem->host.unit ? k_reactor_team<9, true> : k_reactor_team<9, false>),
                       dim3((r->P.cap + bs / kTeam - 1) / (bs / kTeam)), dim3(bs), 0, r->stream, r->chem->dev, r->P,
                       max_tries, r->rtol, r->atol);
  else if (r->chem->host.ns == 9)
    hipLaunchKernelGGL(k_reactor_n<9>, grid, dim3(bs), 0, r->stream, r->chem->dev, r->P, max_tries,
                       r->rtol, r->atol);
  else
    hipLaunchKernelGGL(k_reactor, grid, dim3(bs), 0, r->stream, r->chem->dev, r->P, max_tries,
                       r->rtol, r->atol);
  CHIP_OK(hipGetLastError());
  return 0;
}

int astr_hip_reactor_set_lanes(astr_reactor_pool* r, int lanes) {
  if (!r) return cfail("null pool");
  if (lanes == kTeam && r->chem->host.ns != 9)
    return cfail("the team kernel is built for mechanisms of 9 species");
  if (lanes != 1 && lanes != kTeam) return cfail("lanes per reactor must be 1 or 16");
  CHIP_OK(hipStreamSynchronize(r->stream));
  r->lanes = lanes;
  return 0;
}

int astr_hip_reactor_get_lanes(astr_reactor_pool* r, int* lanes) {
  if (!r || !lanes) return cfail("null argument");
  *lanes = r->lanes;
  return 0;
}

int astr_hip_reactor_query(astr_reactor_pool* r, int* idle) {
  if (!r || !idle) return cfail("null argument");
  CHIP_OK(hipSetDevice(r->chem->device));
  const hipError_t e = hipStreamQuery(r->stream);
  if (e == hipErrorNotReady) {
    *idle = 0;
    return 0;
  }
  CHIP_OK(e);
  *idle = 1;
  return 0;
}

int astr_hip_reactor_sync(astr_reactor_pool* r) {
  if (!r) return cfail("null pool");
  CHIP_OK(hipStreamSynchronize(r->stream));
  return 0;
}

int astr_hip_reactor_status(astr_reactor_pool* r, int* status) {
  if (!r || !status) return cfail("null argument");
  CHIP_OK(hipSetDevice(r->chem->device));
  CHIP_OK(hipMemcpyAsync(status, r->P.status, r->P.cap * sizeof(int), hipMemcpyDeviceToHost, r->stream));
  CHIP_OK(hipStreamSynchronize(r->stream));
  return 0;
}

int astr_hip_reactor_get(astr_reactor_pool* r, int slot, double* t, double* yv, int* nstep, int* nrej) {
  if (!r) return cfail("null pool");
  if (slot < 0 || slot >= r->P.cap) return cfail("reactor slot out of range");
  CHIP_OK(hipSetDevice(r->chem->device));
  const int n = r->chem->host.ns + 1;
  std::lock_guard<std::mutex> lock(r->pin_mutex);
  hipLaunchKernelGGL(k_reactor_get, dim3(1), dim3(64), 0, r->stream, r->P, slot, n, r->pin);
  CHIP_OK(hipGetLastError());
  CHIP_OK(hipStreamSynchronize(r->stream));
  if (yv) std::memcpy(yv, r->pin, n * sizeof(double));
  if (t) *t = r->pin[NYMAX];
  if (nstep) *nstep = (int)r->pin[NYMAX + 1];
  if (nrej) *nrej = (int)r->pin[NYMAX + 2];
  return 0;
}

int astr_hip_reactor_release(astr_reactor_pool* r, int slot) {
  if (!r) return cfail("null pool");
  if (slot < 0 || slot >= r->P.cap) return cfail("reactor slot out of range");
  CHIP_OK(hipSetDevice(r->chem->device));
  hipLaunchKernelGGL(k_reactor_mark, dim3(1), dim3(1), 0, r->stream, r->P, slot, (int)RX_FREE);
  CHIP_OK(hipGetLastError());
  CHIP_OK(hipStreamSynchronize(r->stream));
  return 0;
}

int astr_hip_chem_temperature_device(astr_chem* c, long long n, const double* Y, const double* e,
                                     double* T, void* stream) {
  if (!c) return cfail("null mechanism");
  if (n < 0) return cfail("negative cell count");
  if (n == 0) return 0;
  if (!Y || !e || !T) return cfail("null buffer");
  CHIP_OK(hipSetDevice(c->device));
  const int bs = 256;
  hipLaunchKernelGGL(k_temperature, dim3((unsigned)((n + bs - 1) / bs)), dim3(bs), 0,
                     (hipStream_t)stream, c->dev, n, Y, e, T, nullptr);
  CHIP_OK(hipGetLastError());
  return 0;
}

int astr_hip_chem_temperature(astr_chem* c, long long n, const double* Y, const double* e, double* T) {
  if (!c) return cfail("null mechanism");
  if (n < 0) return cfail("negative cell count");
  if (n == 0) return 0;
  if (!Y || !e || !T) return cfail("null buffer");
  CHIP_OK(hipSetDevice(c->device));
  const int ns = c->host.ns;
  const size_t b1 = (size_t)n * sizeof(double);
  double* d = nullptr;
  CHIP_OK(hipMalloc(&d, (2 + (size_t)ns) * b1));
  double* dY = d;
  double* dE = dY + (size_t)ns * n;
  double* dT = dE + n;
  int rc = 0;
  if (hipMemcpy(dY, Y, b1 * ns, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dE, e, b1, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dT, T, b1, hipMemcpyHostToDevice) != hipSuccess)
    rc = cfail("copy to device failed");
  if (!rc) rc = astr_hip_chem_temperature_device(c, n, dY, dE, dT, nullptr);
  if (!rc && hipDeviceSynchronize() != hipSuccess) rc = cfail("temperature kernel failed");
  if (!rc && hipMemcpy(T, dT, b1, hipMemcpyDeviceToHost) != hipSuccess) rc = cfail("copy from device failed");
  (void)hipFree(d);
  return rc;
}

}  // extern "C"
