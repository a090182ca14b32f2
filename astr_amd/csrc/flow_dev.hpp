// flow_dev.hpp -- device side of the per-stage line passes of flow.hip: the
// case description FlowArgs, the pointwise thermodynamics and fluxes, and the
// pass kernel k_pass templated on launch shape, pass program and register
// budget.  passes.hip instantiates it once per launch shape.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "lines.hpp"

namespace astr {

// ---------------------------------------------------------------------------
// device-side description of one case
// ---------------------------------------------------------------------------
struct FlowArgs {
  int n[3];             // im, jm, km
  int ndir;             // 3, or 2 when km==0
  int pitch;            // doubles between rows (j)
  long long plane;      // doubles between planes (k)
  long long fs;         // doubles between fields
  double inv_d[3];      // 1/dx, 1/dy, 1/dz
  double const2, const5, const6;
  double reynolds, prandtl, suth, suth1;
  double rk_a, rk_b, rk_c, dt;
  int trash;            // a point index inside every field's padding
  double alfa, bhalo;   // filter alpha and halo-row beta (LHS of the filter rows)
  int stage;            // 0,1,2
  int dostats;          // stage-1 KE/enstrophy partial sums (1) or none (0)
  // q holds the current state.  No RK stage updates it in place or copies it:
  // the arrays change roles (rk3_run).  The first stage leaves q as the saved
  // state and writes the new one to qsave; the second writes it over qrhs,
  // whose values it is the last to read; the third, with the second's q as
  // its qrhs, writes it over the saved state, so a step starts and ends in
  // one array.
  double* q;            // 5 fields
  double* qsave;        // 5 fields
  double* qrhs;         // 5 fields
  double* dv;           // 12 fields: dvel(m,d) at m+3d, dtmp(d) at 9+d
  double* sg;           // 9 fields: sigma 11,12,13,22,23,33, qflux 1,2,3
  double* p;            // the pressure of q (miniapp; written by the stage's
                        // first gradient pass, read by the passes that follow)
  double* stats;        // 2 doubles per tile
  const double* dac[3]; // derivative LU tables [ac1|ac2|ac3] per direction
  const double* fac[3]; // filter LU tables
  FilterCoef fc;
  // Main-path semantics (src/mainloop.F90:396-482; passes instantiated with
  // MAIN = true).  The metrics of a uniform Cartesian grid: inv_d[d] holds
  // dxi(d,d) and jac the Jacobian; dxi(d,n) = 0 for d != n.
  int main_sem;         // 1: main path, 0: miniapp
  double jac;
  double* pr;           // 6 fields: the primitives rho, u, v, w, p, T as the
                        // last updatefvar / qswap left them
  const double* hx;     // halo sources of the x-lines on j or k boundary planes
  const double* hy;     // halo sources of the y-lines on k boundary planes
  long long hxs, hys;   // field strides of hx, hy
  // Main path, physical boundaries and non-uniform grids: the boundary bits
  // of each direction (bit 0: physical boundary at 0, bit 1: at n; 0 for a
  // periodic direction) and, for a grid that is not uniform, the metrics per
  // point as 10 fields: J, then dxi(d,n) at 1 + d + 3n (nullptr: the uniform
  // grid's jac and inv_d above, dxi(d,n) = 0 for d != n)
  int bnd[3];
  const double* met;
  // main path: the convective term is the upwind-biased one (upwind.hip),
  // which the flux passes then leave out
  int uwd;
  // main path: the RK pass also applies the next stage's filterq sweep along
  // its direction to the new q, after updatefvar took the primitives
  int rk_filter;
  // the stress pass computes the x gradients itself (its lines are x-lines),
  // no x gradient pass before it; store_gx: it also stores them (read through
  // StageArgs: a batch copies these arguments whatever call set them last)
  int gradx, store_gx;
};

// Halo sources kept by qswap for the lines whose halo the reference fills
// before a later direction averages the source points (qswap's i step copies
// the x-halo of the lines on the j and k boundary planes before the j and k
// steps average those planes; its j step copies the y-halo of the lines on
// the k boundary planes before the k step).  Ten rows per line: rows 1..5 and
// n-5..n-1 of the line, whose copies are the halo rows n+1..n+5 and -5..-1.
constexpr int kHaloSrcRows = 10;
__host__ __device__ inline long long hx_lines(const int n[3], int ndir) {
  return 2ll * (n[2] + 1) + (ndir == 3 ? 2ll * (n[1] + 1) : 0);
}
__host__ __device__ inline long long hy_lines(const int n[3], int ndir) {
  return ndir == 3 ? 2ll * (n[0] + 1) : 0;
}
// index of the halo source (line, hrow) of an x-line (j,k) or y-line (i,k)
// in hx / hy, or -1 when the line takes its halo from the current q
__host__ __device__ inline int halo_src_index(const int n[3], int ndir, int dir, int i, int j, int k,
                                              int hrow) {
  if (dir == 0) {
    if (j == 0 || j == n[1]) return ((j == 0 ? 0 : 1) * (n[2] + 1) + k) * kHaloSrcRows + hrow;
    if (ndir == 3 && (k == 0 || k == n[2]))
      return (2 * (n[2] + 1) + (k == 0 ? 0 : 1) * (n[1] + 1) + j) * kHaloSrcRows + hrow;
  } else if (dir == 1 && ndir == 3) {
    if (k == 0 || k == n[2]) return ((k == 0 ? 0 : 1) * (n[0] + 1) + i) * kHaloSrcRows + hrow;
  }
  return -1;
}

// Pass programs.  Per stage: the gradients of u, v, w and T along y and z
// (GC_MID, GC_LAST), then per direction the derivative of the whole flux,
// viscous minus convective (V_MID along x and y, V_LAST_RHS or V_LAST_RK along
// the last direction).  Taking the two fluxes' difference before the line
// solve leaves 5 solves per direction where separate derivatives take 9, and
// qrhs is accumulated once per direction.
//   V_MID along x (kernels V_FIRST and V_FIRST_G) also forms the stress and
//   heat flux, and the statistics, from the gradients; V_FIRST_G computes the
//   x gradients itself, on the lines it holds anyway, which saves a pass that
//   would read q and store four fields for this one to read back;
//   GC_FIRST is the x gradients on their own, stored, where something else
//   reads them: the shock sensor, per-point metrics (whose gradients
//   accumulate over the directions), physical ends;
//   FGC_FIRST is GC_FIRST preceded by the previous stage's filter sweep along
//   the same lines (x): it filters the q it loads, writes it back and goes on
//   with the filtered values (the sweeps along different indices commute, so
//   the x sweep may come last).
// Ids 7 and 8 were the halves of a split last gradient pass; they stay
// reserved so that the ids of the launch selection keep their meaning.
enum Prog { GC_FIRST = 0, GC_MID, GC_LAST, V_MID, V_LAST_RHS, V_LAST_RK, F_ONLY, RESERVED_7, RESERVED_8,
            FGC_FIRST, V_FIRST, V_FIRST_G };
constexpr int kNumProgs = 10;  // V_FIRST, V_FIRST_G: V_MID's kernels along x, no ids of their own

// ntiles of direction dir for lines-per-tile TL
__host__ __device__ inline int tiles_of(const int n[3], int dir, int TL) {
  const int ni = (n[0] + TL) / TL;  // ceil((im+1)/TL)
  if (dir == 0) return ((n[1] + 1) * (n[2] + 1) + TL - 1) / TL;
  if (dir == 1) return ni * (n[2] + 1);
  return ni * (n[1] + 1);
}

// Blocks are handed to the 8 XCDs round robin; give each XCD a contiguous
// range of tiles so tiles sharing cache lines share an L2.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
  const int x = b & 7, s = b >> 3, q = nb >> 3, r = nb & 7;
  return x * q + (x < r ? x : r) + s;
}

template <class C>
struct Slots {
  unsigned g[C::NPT];  // byte offset inside a field; the trash point for lines
                       // past the end of the lattice (partial last tile)
  int s[C::NPT];  // index of the point in a line buffer (l*LT + r)
  int h[C::NPT];  // line-buffer index of the slot's periodic halo copy
  int ex[C::NPT]; // main path: index of the halo copy's value in hx / hy
                  // (halo_src_index), or -1: the copy takes the point's q
  int interior;   // bit t: i,j,k >= 1 (stats domain)
};

// FP64 load / store at a byte offset from a field's base pointer.  The base is
// the same for every lane and the offset a 32-bit per-lane value, so the
// access uses the scalar-base + vector-offset address mode and one offset
// register per point serves every field.
// The base passes through readfirstlane so the compiler keeps it a scalar
// value and does not fold the field index into the per-lane address.
template <class T>
__device__ __forceinline__ T* uniform_ptr(T* p) {
  const unsigned long long v = reinterpret_cast<unsigned long long>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return reinterpret_cast<T*>(((unsigned long long)hi << 32) | lo);
}
// a value that is the same on every lane, kept in scalar registers
__device__ __forceinline__ double uniform(double x) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                          __builtin_amdgcn_readfirstlane(__double2loint(x)));
}
// The accesses are made through global (address space 1) pointers so the
// compiler emits global, not flat, instructions.
typedef __attribute__((address_space(1))) const char gchar_c;
typedef __attribute__((address_space(1))) char gchar;
__device__ __forceinline__ double ldg(const double* base, unsigned off) {
  gchar_c* b = (gchar_c*)uniform_ptr(base);
  return *(__attribute__((address_space(1))) const double*)(b + off);
}
__device__ __forceinline__ void stg(double* base, unsigned off, double v) {
  gchar* b = (gchar*)uniform_ptr(base);
  *(__attribute__((address_space(1))) double*)(b + off) = v;
}

// LDS of a pass: the output lines X (TL x LT), then the input lines T
// (TL x LT), then a write-only dummy cell.  A slot holding no point (past the
// tile) or no halo copy points s/h at index TL*LT: its T writes land in the
// dummy cell (T + kLineOff + TL*LT) and its X reads return T's zero padding
// (X + TL*LT = row -8 of T's first line), so no slot needs a guard.
// After them sit the filter's halo-row coefficients (3 rows x 11), staged
// once per tile so that no filter solve waits on a global load.
// The table also holds the rows of a physical boundary (boundary_row in
// lines.hpp): coefh (33), coefb (21), coef6i (4), coef8i (5).
constexpr int kHaloCoefs = kBndCoefs;
constexpr int kHaloSlot = 64;
template <class C>
constexpr int lds_line_doubles() {
  return (2 * C::TL * C::LT > 2 * C::NT ? 2 * C::TL * C::LT : 2 * C::NT) + kLineOff + 8;
}
// After the halo slot: the LU factors ac2, ac1 of every chunk row of the
// pass's line systems, staged once per tile.  Each solve reads its chunk's
// factors back just before it runs instead of holding them in registers for
// the whole pass; the registers freed raise the waves per SIMD of the last
// gradient pass, the viscous passes and the filter pass.
template <class C>
constexpr int lds_coef_offset() {
  return lds_line_doubles<C>() + kHaloSlot;
}
// Regions of 2 P R doubles a pass stages: two (the derivative's and the
// filter's) in the RK pass and the filtering first gradient pass, one in the
// others.
constexpr int coef_regions(int prog) { return prog == V_LAST_RK || prog == FGC_FIRST ? 2 : 1; }
// Main path, gradient passes: the primitives u, v, w, T of the halo copies
// (kHaloSrcRows per line), evaluated once by the slots that own them.
constexpr int halo_prims(int prog, int TL, bool main_sem) {
  return main_sem && (prog <= GC_LAST || prog == V_FIRST_G) ? 4 * kHaloSrcRows * TL : 0;
}
template <class C>
constexpr int lds_doubles(int prog, bool main_sem = false) {
  return lds_coef_offset<C>() + coef_regions(prog) * 2 * C::P * C::R + halo_prims(prog, C::TL, main_sem);
}

// Stage the chunk factors of a line of M rows into coefficient region `region`
// (2 P R doubles each, after the halo slot): c2 (ac2, 1 at row 0) at [u],
// c1 (ac1, 0 at row M-1) at [P*R + u], 0 past the rows.
template <class C>
__device__ __forceinline__ double* stage_chunk_coefs(const double* __restrict__ ac, int M, double* smem,
                                                     int region) {
  double* cs = smem + lds_coef_offset<C>() + region * 2 * C::P * C::R;
  for (int u = threadIdx.x; u < C::P * C::R; u += C::NT) {
    const bool ok = u < M;
    const int uu = ok ? u : 0;
    double a1 = ac[uu], a2 = ac[M + uu];
    if (u == 0) a2 = 1.0;
    if (u == M - 1) a1 = 0.0;
    cs[u] = ok ? a2 : 0.0;
    cs[C::P * C::R + u] = ok ? a1 : 0.0;
  }
  return cs;
}

template <class C>
__device__ __forceinline__ void lds_chunk_coef(ChunkCoef<C::R, false>& CD, const double* cs, int u0) {
#pragma unroll
  for (int k = 0; k < C::R; k++) {
    CD.c2[k] = cs[u0 + k];
    CD.c1[k] = cs[C::P * C::R + u0 + k];
  }
}

// the filter's: also its last-row exception (load_chunk_coef in lines.hpp)
template <class C>
__device__ __forceinline__ void lds_chunk_coef_f(ChunkCoef<C::R, true>& CF, const double* cs, int u0,
                                                 int M, double c3last) {
#pragma unroll
  for (int k = 0; k < C::R; k++) {
    CF.c2[k] = cs[u0 + k];
    CF.c1[k] = cs[C::P * C::R + u0 + k];
  }
  const int kl = M - 1 - u0;
  CF.klast = kl >= 0 && kl < C::R ? kl : -1;
  CF.c3last = c3last;
}

// A line solve of a pass: the periodic form, or (main path, general-grid
// kernels only) the closed form of a direction with physical ends
template <class C, bool FILT, bool GEN>
__device__ __forceinline__ void solve_pass_line(const double* Tl, double* Xl, int n, int p,
                                                const ChunkCoef<C::R, FILT>& CC, const FilterCoef& fc,
                                                int bnd) {
  if constexpr (GEN) {
    if (bnd) {
      solve_line<C::P, C::R, FILT, true>(Tl, Xl, n, p, CC, fc, bnd);
      return;
    }
  }
  solve_line<C::P, C::R, FILT>(Tl, Xl, n, p, CC, fc);
}

// Copy the filter's halo-row coefficients into the tile's LDS; the barrier
// before the first filter solve publishes them.  Every read of the previous
// tile's copy ended before that tile's last barrier.
template <class C>
__device__ __forceinline__ FilterCoef stage_halo_coefs(const FilterCoef& fc, double* smem) {
  double* ch = smem + lds_line_doubles<C>();
  if (threadIdx.x < kHaloCoefs) ch[threadIdx.x] = fc.ch[threadIdx.x];
  FilterCoef f = fc;
  f.ch = ch;
  return f;
}

// Map the tile's points onto slots.  dir 0: lines are (j,k), rows i; dir 1:
// lines (i,k) rows j; dir 2: lines (i,j) rows k.
template <class C, bool MAIN = false>
__device__ __forceinline__ void make_slots(Slots<C>& S, const FlowArgs& a, int dir, int tile) {
  const int n = a.n[dir];
  const int np = C::TL * (n + 1);
  const int ni = (a.n[0] + C::TL) / C::TL;
  const int dummy = C::TL * C::LT;
  S.interior = 0;
#pragma unroll
  for (int t = 0; t < C::NPT; t++) {
    const int e = threadIdx.x + t * C::NT;
    S.g[t] = (unsigned)a.trash * 8u;
    S.s[t] = dummy;
    S.h[t] = dummy;
    if (MAIN) S.ex[t] = -1;
    if (e < np) {
      int l, r, i, j, k;
      bool ok;
      if (dir == 0) {
        l = e / (n + 1);
        r = e - l * (n + 1);
        const int L = tile * C::TL + l;
        j = L % (a.n[1] + 1);
        k = L / (a.n[1] + 1);
        i = r;
        ok = L < (a.n[1] + 1) * (a.n[2] + 1);
      } else {
        l = e & (C::TL - 1);
        r = e / C::TL;
        const int it = tile % ni, o = tile / ni;
        i = it * C::TL + l;
        ok = i <= a.n[0];
        if (dir == 1) { j = r; k = o; } else { j = o; k = r; }
      }
      S.s[t] = l * C::LT + r;
      // rows n-5..n-1 are copied to the halo rows -5..-1, rows 1..5 to
      // n+1..n+5 (disjoint for n >= 11)
      if (r >= n - 5 && r <= n - 1) S.h[t] = S.s[t] - n;
      if (r >= 1 && r <= 5) S.h[t] = S.s[t] + n;
      if (MAIN && ok && S.h[t] != dummy)
        S.ex[t] = halo_src_index(a.n, a.ndir, dir, i, j, k, r <= 5 ? r - 1 : r - (n - 5) + 5);
      if (ok) {
        S.g[t] = (unsigned)((long long)k * a.plane + (long long)j * a.pitch + i) * 8u;
        const bool in = i >= 1 && j >= 1 && (a.ndir == 2 || k >= 1);
        if (in) S.interior |= 1 << t;
      }
    }
  }
}

// byte offset of row 0 of a tile's first line
template <class C>
__device__ __forceinline__ unsigned tile_first(const FlowArgs& a, int dir, int tile) {
  if (dir == 0) {
    const int L = tile * C::TL, rows = a.n[1] + 1;
    return (unsigned)((long long)(L / rows) * a.plane + (long long)(L % rows) * a.pitch) * 8u;
  }
  const int ni = (a.n[0] + C::TL) / C::TL;
  return (unsigned)((long long)(tile / ni) * (dir == 1 ? a.plane : a.pitch) + tile % ni * C::TL) * 8u;
}

// store slot t's value into its input line with the periodic halo copies
// q(-h)=q(n-h), q(n+h)=q(h) (tgvsolver.F90:371-440)
template <class C>
__device__ __forceinline__ void put(double* T, const Slots<C>& S, int t, double v) {
  T[kLineOff + S.s[t]] = v;
  T[kLineOff + S.h[t]] = v;
}

// zero the padding rows -8..-6 and n+6..P*R+2 of every input line (never
// written by put; read by the chunks at the ends of a line)
template <class C>
__device__ __forceinline__ void zero_pad(double* T, int n) {
  const int npad = 3 + (C::P * C::R + 2 - (n + 6) + 1);
  for (int e = threadIdx.x; e < C::TL * npad; e += C::NT) {
    const int l = e / npad, k = e - l * npad;
    const int row = k < 3 ? k - 8 : n + 6 + (k - 3);
    T[l * C::LT + kLineOff + row] = 0.0;
  }
}

// q2fvar + thermal_scar (tgvsolver.F90:73-121).  Pointwise thermodynamics is
// evaluated without FMA contraction and in the reference's operation order:
// p ~ 1/(gamma Ma^2) is large against its gradient, so one rounding step in p
// becomes a visible error in grad p.
__device__ __forceinline__ double pressure_of(const FlowArgs& a, double q1, double q2, double q3,
                                              double q4, double q5) {
#pragma clang fp contract(off)
  const double u = q2 / q1, v = q3 / q1, w = q4 / q1;
  return (q5 - 0.5 * q1 * (u * u + v * v + w * w)) / a.const6;
}

struct Prim {
  double r, u, v, w, p, t;
};

__device__ __forceinline__ Prim prim_of(const FlowArgs& a, double q1, double q2, double q3,
                                        double q4, double q5) {
#pragma clang fp contract(off)
  Prim P;
  P.r = q1;
  P.u = q2 / q1;
  P.v = q3 / q1;
  P.w = q4 / q1;
  P.p = (q5 - 0.5 * q1 * (P.u * P.u + P.v * P.v + P.w * P.w)) / a.const6;
  P.t = P.p / q1 * a.const2;
  return P;
}

// The viscous flux v minus the convective flux of component m along dir
// (tgvsolver.F90:559-564, 586-591, 613-618) from q_m, the velocity along dir
// and p.  v is 1e-3 of the convective flux: subtracted from the product in one
// fused operation, the difference rounds once at that flux's size, as the flux
// alone does; formed from the rounded product it rounds twice there (at 28 x 27
// x 24, Mach 1, the energy right-hand side's error is 1.12 times that of the
// convective part alone with two roundings, 1.01 with one).  The momentum along
// dir carries p, from which f0, a pressure of the state, goes off first.  Where p
// is large against the momentum flux (f0 above kLargeP; q_m u is of order one
// in these units) it keeps the reference's q_m u + p, whose rounding at p's size
// is the largest of either, and f0 goes off that exactly.  Otherwise f0 goes off
// p, exactly within a factor of two of it, and nothing rounds at p's size: the
// momentum's error on an isentropic vortex at Mach 0.5 is then below that of the
// parts differentiated apart, 1.026 times it with the first form.
enum FluxKind { FLUX_PLAIN, FLUX_ALONG, FLUX_ALONG_LARGE_P, FLUX_ENERGY };
constexpr double kLargeP = 4.0;
template <int KIND>
__device__ __forceinline__ double flux_diff(double qm, double uu, double p, double f0, double v) {
#pragma clang fp contract(off)
  if (KIND == FLUX_ALONG_LARGE_P) return v - (qm * uu + p - f0);
  if (KIND == FLUX_ALONG) return fma(-qm, uu, v) - (p - f0);
  return fma(-(KIND == FLUX_ENERGY ? qm + p : qm), uu, v);
}

// Sutherland (tgvsolver.F90:123-140)
__device__ __forceinline__ double miucal(const FlowArgs& a, double t) {
#pragma clang fp contract(off)
  return t * sqrt(t) * a.suth1 / (t + a.suth);
}

// what changes from stage to stage (the same for every case of a batch)
struct StageArgs {
  int stage;            // 0,1,2
  int dostats;          // stage-1 KE/enstrophy partial sums (1) or none (0)
  double rk_a, rk_b, rk_c;
  int alt;              // batches: stages whose change of array roles applies (0, 1, 2)
  int store_gx;         // the stress pass also stores the x gradients it computes (batches: never)
};

// the arrays in their roles after `alt` stages of a step
struct Arrays {
  double *q, *qsave, *qrhs;
};
__device__ __forceinline__ Arrays arrays_of(const FlowArgs& a, int alt) {
  if (alt == 0) return Arrays{a.q, a.qsave, a.qrhs};
  if (alt == 1) return Arrays{a.qsave, a.q, a.qrhs};
  return Arrays{a.qrhs, a.q, a.qsave};
}

__device__ __forceinline__ StageArgs stage_of(const FlowArgs& a) {
  return StageArgs{a.stage, a.dostats, a.rk_a, a.rk_b, a.rk_c, 0, a.store_gx};
}

// q <- a*qsave + b*q + c*qrhs*dt in the reference's order (tgvsolver.F90:1055-1057)
__device__ __forceinline__ double rk_update(const StageArgs& sa, double dt, double qs, double qo,
                                            double qr) {
#pragma clang fp contract(off)
  return sa.rk_a * qs + sa.rk_b * qo + sa.rk_c * qr * dt;
}

// stress, heat flux (tgvsolver.F90:663-691); g[m][d] = d u_m / d x_d
__device__ __forceinline__ void visc_flux(const FlowArgs& a, const double g[3][3],
                                          const double gt[3], const Prim& P, double out[9]) {
#pragma clang fp contract(off)
  const double s11 = g[0][0];
  const double s12 = 0.5 * (g[0][1] + g[1][0]);
  const double s13 = 0.5 * (g[0][2] + g[2][0]);
  const double s22 = g[1][1];
  const double s23 = 0.5 * (g[1][2] + g[2][1]);
  const double s33 = g[2][2];
  const double skk = (1.0 / 3.0) * (s11 + s22 + s33);
  const double miu = miucal(a, P.t) / a.reynolds;
  const double miu2 = 2.0 * miu;
  const double hcc = (miu / a.prandtl) / a.const5;
  out[0] = miu2 * (s11 - skk);
  out[1] = miu2 * s12;
  out[2] = miu2 * s13;
  out[3] = miu2 * (s22 - skk);
  out[4] = miu2 * s23;
  out[5] = miu2 * (s33 - skk);
  out[6] = hcc * gt[0] + out[0] * P.u + out[1] * P.v + out[2] * P.w;
  out[7] = hcc * gt[1] + out[1] * P.u + out[3] * P.v + out[4] * P.w;
  out[8] = hcc * gt[2] + out[2] * P.u + out[4] * P.v + out[5] * P.w;
}

// Main path (convrsdcal6, src/solver.F90:2196-2207): flux component m along
// dir, J (q_m U + dxi(dir,m) p) with the contravariant velocity
// U = sum_n dxi(dir,n) u_n, for the metrics of a uniform Cartesian grid
// (dxi(dir,n) = 0 for n != dir, so those products add exact zeros); v minus it
// as in flux_diff
template <int KIND>
__device__ __forceinline__ double flux_diff_main(double jac, double dx, double qm, double ud, double p, double f0,
                                                 double v) {
#pragma clang fp contract(off)
  const double uu = dx * ud;
  if (KIND == FLUX_ALONG_LARGE_P) return v - (jac * (qm * uu + dx * p) - jac * (dx * f0));
  if (KIND == FLUX_ALONG) return fma(-jac, qm * uu + dx * (p - f0), v);
  return fma(-(jac * (KIND == FLUX_ENERGY ? qm + p : qm)), uu, v);
}

// Main path: the Jacobian J and dxi(dir,dir) of a point on a uniform grid
struct Met {
  double j, d;
};
__device__ __forceinline__ Met met_of(const FlowArgs& a, int dir) { return Met{a.jac, a.inv_d[dir]}; }

// Main path on a grid that is not uniform: J and the row dxi(dir, 0..2) of a point
struct MetRow {
  double j, r[3];
};
__device__ __forceinline__ MetRow met_row(const FlowArgs& a, int dir, unsigned g) {
  MetRow M;
  M.j = ldg(a.met, g);
#pragma unroll
  for (int nn = 0; nn < 3; nn++) M.r[nn] = ldg(a.met + (1 + dir + 3 * nn) * a.fs, g);
  return M;
}
// the Jacobian of a point, either grid (GEN: a general-grid kernel, which
// alone reads per-point metrics)
template <bool GEN>
__device__ __forceinline__ double jac_of(const FlowArgs& a, unsigned g) {
  return GEN && a.met ? ldg(a.met, g) : a.jac;
}

// convrsdcal6 (src/solver.F90:2196-2207) with the full metric row:
// U = dxi(d,1) u + dxi(d,2) v + dxi(d,3) w, F_m = J (q_m U + dxi(d,m) p); v
// minus it, rounded once as in flux_diff (jm, rm: J and dxi(d,m))
__device__ __forceinline__ double contravariant(const MetRow& M, double u, double v, double w) {
#pragma clang fp contract(off)
  return M.r[0] * u + M.r[1] * v + M.r[2] * w;
}
__device__ __forceinline__ double flux_diff_full(double jm, double rm, int m, double qm, double uu, double p,
                                                 double v) {
#pragma clang fp contract(off)
  if (m == 0 || m == 4) return fma(-(jm * (m == 4 ? qm + p : qm)), uu, v);
  return fma(-jm, qm * uu + rm * p, v);
}

// diffrsdcal6 (src/solver.F90:2623-2635) with the full metric row: column
// c of direction dir, (s_c1 dxi(d,1) + s_c2 dxi(d,2) + s_c3 dxi(d,3)) J with
// s_c = the stress row c (c < 3) or the heat flux (c = 3)
__device__ __forceinline__ double visc_col_row(const MetRow& M, double s0, double s1, double s2) {
#pragma clang fp contract(off)
  return (s0 * M.r[0] + s1 * M.r[1] + s2 * M.r[2]) * M.j;
}
__device__ __forceinline__ int visc_term(int c, int i) {
  const int k[4][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}, {6, 7, 8}};
  return k[c][i];
}
__device__ __forceinline__ double visc_col_full(const FlowArgs& a, int dir, int c, unsigned g) {
  return visc_col_row(met_row(a, dir, g), ldg(a.sg + visc_term(c, 0) * a.fs, g),
                      ldg(a.sg + visc_term(c, 1) * a.fs, g), ldg(a.sg + visc_term(c, 2) * a.fs, g));
}

// Main path: component m of q of the halo copy of slot t.  qswap fills the
// halo of a line from the filtered q; the lines on boundary planes that a
// later qswap step averages take the values kept before that step (hx / hy),
// the others the current q of the source point, which the slot owns.
template <class C>
__device__ __forceinline__ double halo_q(const FlowArgs& a, const double* q, const Slots<C>& S, int t, int dir,
                                         int m) {
  if (S.ex[t] >= 0) return (dir == 0 ? a.hx + m * a.hxs : a.hy + m * a.hys)[S.ex[t]];
  return ldg(q + m * a.fs, S.g[t]);
}

// main path RK3 update (src/mainloop.F90:441-449):
// q <- (a qsave + b q J + c qrhs dt) / J, in the reference's order
__device__ __forceinline__ double rk_update_main(const StageArgs& sa, double dt, double jac, double qs,
                                                 double qo, double qr) {
#pragma clang fp contract(off)
  return (sa.rk_a * qs + sa.rk_b * qo * jac + sa.rk_c * qr * dt) / jac;
}

// ---------------------------------------------------------------------------
// the pass kernel
// ---------------------------------------------------------------------------
// stress and heat flux of a point from its gradients (diffusion,
// tgvsolver.F90:659-694) and its terms of the statistics (stacal, :893-942);
// gx: the x gradients of u, v, w, T where the pass has them, nullptr: stored
__device__ __forceinline__ void stress_point(const FlowArgs& a, unsigned o, const Prim& P, const double* gx,
                                             double f[9], bool stats, double& sk, double& se) {
#pragma clang fp contract(off)
  double g[3][3], gt[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const bool own = d == 0 && gx;
#pragma unroll
    for (int m = 0; m < 3; m++)
      g[m][d] = own ? gx[m] : (d < a.ndir ? ldg(a.dv + (m + 3 * d) * a.fs, o) : 0.0);
    gt[d] = own ? gx[3] : (d < a.ndir ? ldg(a.dv + (9 + d) * a.fs, o) : 0.0);
  }
  visc_flux(a, g, gt, P, f);
  if (stats) {
    sk += P.r * (P.u * P.u + P.v * P.v + P.w * P.w);
    const double o1 = g[2][1] - g[1][2];
    const double o2 = g[0][2] - g[2][0];
    const double o3 = g[1][0] - g[0][1];
    se += P.r * (o1 * o1 + o2 * o2 + o3 * o3);
  }
}

// MINB: workgroups per CU the register allocation is held to (each
// workgroup puts one wave on each SIMD, so MINB waves per SIMD)
// One tile of one pass.  `a` describes the case, `sa` the stage.
// MAIN: the main path's semantics (src/mainloop.F90:396-482): the gradients
// and fluxes take the stored primitives (pr) as the last updatefvar left them
// and their halo copies from the filtered q (qswap), the fluxes carry the
// metrics J and dxi (convrsdcal6, diffrsdcal6), and the RK pass is followed by
// updatefvar (k_fvar) instead of ending with this stage's filter.
// Each pass reads its chunk factors back from LDS before each solve instead
// of holding them in registers, and issues a solve's accumulation loads and
// the next solve's inputs before it, so that their latency overlaps it.
// A: the arrays of the current state, the saved one and qrhs (FlowArgs::q).
// ONE: the workgroup takes one component (`field`) of the pass, five or four
// workgroups share a tile.  The components' solves are independent, and
// where a pass has few tiles their serial chain in one workgroup is its time.
template <class C, int PROG, bool MAIN = false, bool GEN = false, bool ONE = false>
__device__ __forceinline__ void pass_body(const FlowArgs& a, const StageArgs& sa, const Arrays& A, int dir_, int tile,
                                          double* smem, int field = 0) {
  const int dir = PROG == FGC_FIRST || PROG == V_FIRST || PROG == V_FIRST_G ? 0 : dir_;
  double* const qc = A.q;
  double* const qo = A.qsave;
  double* const qrhs = A.qrhs;
  constexpr int NPT = C::NPT;
  constexpr int kDummy = C::TL * C::LT;
  const int n = a.n[dir];
  double* X = smem;                 // output lines, TL x LT (rows at offset 0)
  double* T = smem + C::TL * C::LT; // input lines, TL x LT
  Slots<C> S;
  make_slots<C, MAIN>(S, a, dir, tile);
  zero_pad<C>(T, n);
  const int ln = threadIdx.x / C::P, p = threadIdx.x % C::P;
  double* Tl = T + ln * C::LT;
  double* Xl = X + ln * C::LT;
  const double idn = a.inv_d[dir];
  const long long fs = a.fs;

  // derivative of the staged lines, between the barriers that publish the
  // staging and the results
  const double* cs = nullptr;
  auto derive = [&]() __attribute__((always_inline)) {
    __syncthreads();
    {
      ChunkCoef<C::R, false> CD;
      lds_chunk_coef<C>(CD, cs, p * C::R);
      solve_pass_line<C, false, GEN>(Tl, Xl, n, p, CD, a.fc, a.bnd[dir]);
    }
    __syncthreads();
  };
  const double* csf = nullptr;
  double c3l = 0.0;
  FilterCoef fl;
  auto filter_setup = [&](int region) __attribute__((always_inline)) {
    csf = stage_chunk_coefs<C>(a.fac[dir], n + 7, smem, region);
    c3l = a.fac[dir][2 * (n + 7) + (n + 7) - 1];
    fl = stage_halo_coefs<C>(a.fc, smem);
  };
  auto filter = [&]() __attribute__((always_inline)) {
    __syncthreads();
    {
      ChunkCoef<C::R, true> CF;
      lds_chunk_coef_f<C>(CF, csf, p * C::R, n + 7, c3l);
      solve_pass_line<C, true, GEN>(Tl, Xl, n, p, CF, fl, a.bnd[dir]);
    }
    __syncthreads();
  };

  // Gradients of u, v, w, T along dir (gradcal, tgvsolver.F90:450-537;
  // src/comsolver.F90:280-321).  Miniapp: of q; the stage's first gradient
  // pass forms the pressure and leaves it for the others.  Main path: of the
  // stored primitives, with the halo copies from the primitives of the halo's
  // q (qswap's q2fvar).
  constexpr bool GRAD = PROG == GC_FIRST || PROG == FGC_FIRST || PROG == GC_MID || PROG == V_FIRST_G;
  double pv[4][GRAD ? NPT : 1];
  double* hal = smem + lds_doubles<C>(PROG);
  auto hslot = [&](int t) {  // the slot's halo primitives, written and read by its own thread
    const int l = S.s[t] / C::LT, r = S.s[t] - l * C::LT;
    return hal + 4 * (l * kHaloSrcRows + (r <= 5 ? r - 1 : r - (n - 5) + 5));
  };
  auto load_prims = [&]() __attribute__((always_inline)) {
    if constexpr (MAIN) {
#pragma unroll
      for (int t = 0; t < NPT; t++)
#pragma unroll
        for (int c = 0; c < 4; c++) pv[c][t] = ldg(a.pr + (c < 3 ? 1 + c : 5) * fs, S.g[t]);
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        if (S.h[t] != kDummy) {
          double qh[5];
#pragma unroll
          for (int m = 0; m < 5; m++) qh[m] = halo_q<C>(a, qc, S, t, dir, m);
          const Prim P = prim_of(a, qh[0], qh[1], qh[2], qh[3], qh[4]);
          double* h = hslot(t);
          h[0] = P.u; h[1] = P.v; h[2] = P.w; h[3] = P.t;
        }
      }
    } else {
      constexpr bool PRES = PROG == GC_FIRST || PROG == FGC_FIRST;
      double qv[5][NPT];
#pragma unroll
      for (int t = 0; t < NPT; t++)
#pragma unroll
        for (int m = 0; m < 5; m++) qv[m][t] = ldg(!PRES && m == 4 ? a.p : qc + m * fs, S.g[t]);
      if constexpr (PROG == FGC_FIRST) {
        // the previous stage's filter sweep along these lines (filterq,
        // tgvsolver.F90:805-825), as the filter pass does it, on the loaded
        // q; the filtered q is stored and the gradients take it
        filter_setup(1);
#pragma unroll
        for (int m = 0; m < 5; m++) {
#pragma unroll
          for (int t = 0; t < NPT; t++) put<C>(T, S, t, qv[m][t]);
          filter();
#pragma unroll
          for (int t = 0; t < NPT; t++) {
            qv[m][t] = X[S.s[t]];
            stg(qc + m * fs, S.g[t], qv[m][t]);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        double pr = qv[4][t];
        if constexpr (PRES) {
          pr = pressure_of(a, qv[0][t], qv[1][t], qv[2][t], qv[3][t], qv[4][t]);
          stg(a.p, S.g[t], pr);
        }
#pragma unroll
        for (int c = 0; c < 3; c++) pv[c][t] = qv[c + 1][t] / qv[0][t];
        pv[3][t] = pr / qv[0][t] * a.const2;
      }
    }
  };
  // derivative of component c (u, v, w, T), left in X
  auto gradient = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NPT; t++) {
      if constexpr (MAIN) {
        T[kLineOff + S.s[t]] = pv[c][t];
        if (S.h[t] != kDummy) T[kLineOff + S.h[t]] = hslot(t)[c];
      } else {
        put<C>(T, S, t, pv[c][t]);
      }
    }
    derive();
  };

  // one component's primitive alone, in pv[0]
  auto load_one = [&](int c) __attribute__((always_inline)) {
    if constexpr (MAIN) {
#pragma unroll
      for (int t = 0; t < NPT; t++) pv[0][t] = ldg(a.pr + (c < 3 ? 1 + c : 5) * fs, S.g[t]);
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        if (S.h[t] != kDummy) {
          const double r = halo_q<C>(a, qc, S, t, dir, 0);
          if (c < 3) {
            hslot(t)[0] = halo_q<C>(a, qc, S, t, dir, c + 1) / r;
          } else {
            double qh[5];
#pragma unroll
            for (int m = 1; m < 5; m++) qh[m] = halo_q<C>(a, qc, S, t, dir, m);
            hslot(t)[0] = prim_of(a, r, qh[1], qh[2], qh[3], qh[4]).t;
          }
        }
      }
    } else {
      constexpr bool PRES = PROG == GC_FIRST;
      double r[NPT];
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        r[t] = ldg(qc, S.g[t]);
        pv[0][t] = ldg(c < 3 ? qc + (c + 1) * fs : (PRES ? qc + 4 * fs : a.p), S.g[t]);
      }
      if (c < 3) {
#pragma unroll
        for (int t = 0; t < NPT; t++) pv[0][t] = pv[0][t] / r[t];
      } else {
#pragma unroll
        for (int t = 0; t < NPT; t++) {
          if constexpr (PRES) {
            pv[0][t] = pressure_of(a, r[t], ldg(qc + fs, S.g[t]), ldg(qc + 2 * fs, S.g[t]), ldg(qc + 3 * fs, S.g[t]),
                                   pv[0][t]);
            stg(a.p, S.g[t], pv[0][t]);
          }
          pv[0][t] = pv[0][t] / r[t] * a.const2;
        }
      }
    }
  };

  if constexpr (GRAD && PROG != V_FIRST_G) {
    cs = stage_chunk_coefs<C>(a.dac[dir], n + 3, smem, 0);
    if constexpr (ONE) load_one(field);
    else load_prims();
#pragma unroll
    for (int cc = 0; cc < (ONE ? 1 : 4); cc++) {
      const int c = ONE ? field : cc;
      gradient(cc);
      const int fld = c < 3 ? c + 3 * dir : 9 + dir;
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        const unsigned o = S.g[t];
        const double x = X[S.s[t]];
        if (GEN && a.met) {
          // gradcal's accumulation dvel(m,n) += D_d(u_m) dxi(d,n) over
          // every n (src/comsolver.F90:300-321)
#pragma unroll
          for (int nn = 0; nn < 3; nn++) {
#pragma clang fp contract(off)
            if (nn >= a.ndir) continue;
            const int f2 = c < 3 ? c + 3 * nn : 9 + nn;
            const double v = x * ldg(a.met + (1 + dir + 3 * nn) * fs, o);
            if (PROG == GC_FIRST) stg(a.dv + f2 * fs, o, v);
            else stg(a.dv + f2 * fs, o, ldg(a.dv + f2 * fs, o) + v);
          }
        } else {
          // dvel(m,n) = D_d(u_m) dxi(d,n): dxi(d,d) of the uniform grid
          stg(a.dv + fld * fs, o, x * (MAIN ? met_of(a, dir).d : idn));
        }
      }
    }
  } else if constexpr (PROG == V_FIRST || PROG == V_FIRST_G || PROG == V_MID || PROG == V_LAST_RK) {
    // The derivative along dir of the viscous (diffusion, tgvsolver.F90:
    // 700-787) minus the convective flux (convection, :539-633), the sign
    // qrhs has after rhscal, accumulated over the directions.  Viscous columns
    // per direction: x (s11,s12,s13,q1), y (s12,s22,s23,q2), z (s13,s23,s33,q3);
    // density has none.
    constexpr bool FIRST = PROG == V_FIRST || PROG == V_FIRST_G;
    constexpr bool RK = PROG == V_LAST_RK;
    // the main path's upwind-biased convection left its part in qrhs
    const bool uwd = MAIN && a.uwd;
    cs = stage_chunk_coefs<C>(a.dac[dir], n + 3, smem, 0);
    double sx[4][FIRST ? NPT : 1];
    if constexpr (FIRST) {
      // Stress and heat flux of every point from the gradients, here
      // because x-lines leave a lane only NPT points to hold; columns s11 and
      // q1, which no other direction reads, stay in registers.  And the
      // stage-1 KE / enstrophy partial sums.
      double gx[4][PROG == V_FIRST_G ? NPT : 1];
      if constexpr (PROG == V_FIRST_G) {
        load_prims();
#pragma unroll
        for (int c = 0; c < 4; c++) {
          gradient(c);
#pragma unroll
          for (int t = 0; t < NPT; t++) {
            gx[c][t] = X[S.s[t]] * (MAIN ? met_of(a, dir).d : idn);
            if (sa.store_gx) stg(a.dv + (c < 3 ? c : 9) * fs, S.g[t], gx[c][t]);
          }
        }
      }
      double sk = 0.0, se = 0.0;
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        const unsigned o = S.g[t];
        Prim P;
        P.p = 0.0;
        if constexpr (PROG == V_FIRST_G) {
          P.r = sa.dostats ? ldg(MAIN ? a.pr : qc, o) : 0.0;
          P.u = pv[0][t]; P.v = pv[1][t]; P.w = pv[2][t]; P.t = pv[3][t];
        } else if constexpr (MAIN) {
          // diffrsdcal6 (src/solver.F90:2433-2545) and the statistics
          // (statistic.F90:871-992) take the stored rho, vel, tmp
          P.r = sa.dostats ? ldg(a.pr, o) : 0.0;
          P.u = ldg(a.pr + fs, o);
          P.v = ldg(a.pr + 2 * fs, o);
          P.w = ldg(a.pr + 3 * fs, o);
          P.t = ldg(a.pr + 5 * fs, o);
        } else {
          P.r = ldg(qc, o);
          P.u = ldg(qc + fs, o) / P.r;
          P.v = ldg(qc + 2 * fs, o) / P.r;
          P.w = ldg(qc + 3 * fs, o) / P.r;
          P.t = ldg(a.p, o) / P.r * a.const2;
        }
        double f[9], gp[4];
#pragma unroll
        for (int c = 0; c < 4; c++) gp[c] = PROG == V_FIRST_G ? gx[c][PROG == V_FIRST_G ? t : 0] : 0.0;
        stress_point(a, o, P, PROG == V_FIRST_G ? gp : nullptr, f, sa.dostats && ((S.interior >> t) & 1), sk, se);
        const bool all = GEN && a.met;
#pragma unroll
        for (int m = 0; m < 9; m++)
          if (all || (m != 0 && m != 6)) stg(a.sg + m * fs, o, f[m]);
        if (all) {
          const MetRow M = met_row(a, dir, o);
#pragma unroll
          for (int c = 0; c < 4; c++)
            sx[c][t] = visc_col_row(M, f[c == 3 ? 6 : c], f[c == 0 ? 1 : (c == 1 ? 3 : (c == 2 ? 4 : 7))],
                                    f[c == 0 ? 2 : (c == 1 ? 4 : (c == 2 ? 5 : 8))]);
        } else {
#pragma unroll
          for (int c = 0; c < 4; c++) sx[c][t] = f[c == 3 ? 6 : c];
        }
      }
      if (sa.dostats) {
        // deterministic block reduction into this tile's slot
        __syncthreads();
        X[threadIdx.x] = sk;
        X[C::NT + threadIdx.x] = se;
        __syncthreads();
        for (int h = C::NT / 2; h > 0; h >>= 1) {
          if ((int)threadIdx.x < h) {
            X[threadIdx.x] += X[threadIdx.x + h];
            X[C::NT + threadIdx.x] += X[C::NT + threadIdx.x + h];
          }
          __syncthreads();
        }
        if (threadIdx.x == 0) {
          a.stats[2 * tile] = X[0];
          a.stats[2 * tile + 1] = X[C::NT];
        }
        __syncthreads();
      }
    }
    const bool metg = GEN && a.met;
    // velocity along dir (general grids: contravariant) and pressure of the
    // points; hu, hp those of the halo copies where they differ (main path)
    double ud[NPT], pp[NPT], hu[NPT], hp[NPT];
    if (!uwd) {
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        const unsigned o = S.g[t];
        if constexpr (MAIN) {
          // convrsdcal6 takes the stored vel and prs (src/solver.F90:2196-2207)
          if (!ONE || field == 4 || field == dir + 1 || (metg && field > 0)) pp[t] = ldg(a.pr + 4 * fs, o);
          if (metg)
            ud[t] = contravariant(met_row(a, dir, o), ldg(a.pr + fs, o), ldg(a.pr + 2 * fs, o), ldg(a.pr + 3 * fs, o));
          else ud[t] = PROG == V_FIRST_G ? pv[0][t] : ldg(a.pr + (1 + dir) * fs, o);
        } else {
          if (!ONE || field == 4 || field == dir + 1) pp[t] = ldg(a.p, o);
          ud[t] = PROG == V_FIRST_G ? pv[0][t] : ldg(qc + (1 + dir) * fs, o) / ldg(qc, o);
        }
      }
      if constexpr (MAIN) {
#pragma unroll
        for (int t = 0; t < NPT; t++) {
          if (S.h[t] != kDummy) {
            double qh[5];
#pragma unroll
            for (int m = 0; m < 5; m++) qh[m] = halo_q<C>(a, qc, S, t, dir, m);
            hp[t] = pressure_of(a, qh[0], qh[1], qh[2], qh[3], qh[4]);
            // a periodic halo copy carries the source point's metrics, which are this point's
            if (metg) hu[t] = contravariant(met_row(a, dir, S.g[t]), qh[1] / qh[0], qh[2] / qh[0], qh[3] / qh[0]);
            else hu[t] = (dir == 0 ? qh[1] : (dir == 1 ? qh[2] : qh[3])) / qh[0];
          }
        }
      }
    }
    // inputs of the next solve: q_m and the viscous column (general grids
    // form their column when it is staged)
    double qn[NPT], vn[NPT];
    auto load_inputs = [&](int m) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        if (!uwd || RK) qn[t] = ldg(qc + m * fs, S.g[t]);
        if (!FIRST && m > 0 && !metg) {
          const int col = m == 4 ? 6 + dir : (dir == 1 ? (m == 1 ? 1 : (m == 2 ? 3 : 4)) : (m == 1 ? 2 : (m == 2 ? 4 : 5)));
          vn[t] = ldg(a.sg + col * fs, S.g[t]);
        }
      }
    };
    // Stage component m's flux difference with its halo copies (without the
    // convective flux where that is upwind-biased).  The momentum flux along dir
    // carries p ~ 1/(gamma Ma^2), large against everything the derivative keeps
    // of it; f0, the pressure of the tile's first point, drops out of the
    // derivative and goes off it first.  (The reference pressure in its place
    // would round a state of another pressure level at its own size; so would
    // f0 a point of its lines whose p is less than half of it.)  Per-point
    // metrics have no such constant; the fused operation alone keeps their
    // difference to one rounding at the flux's size.
    double f0 = 0.0;
    if (!uwd && !metg && (!ONE || field == dir + 1)) {
      f0 = ldg(MAIN ? a.pr + 4 * fs : a.p, tile_first<C>(a, dir, tile));
      f0 = uniform(__builtin_isfinite(f0) ? f0 : 0.0);
    }
    auto stage_kind = [&](auto kind, int m) __attribute__((always_inline)) {
      constexpr int KIND = decltype(kind)::value;
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        const unsigned o = S.g[t];
        double v = 0.0;
        if (m > 0) {
          if constexpr (FIRST) v = sx[m - 1][t];
          else v = metg ? visc_col_full(a, dir, m - 1, o) : vn[t];
          if (MAIN && !metg) {
            // (sigma . dxi(dir,:)) J (diffrsdcal6, src/solver.F90:2623-2635)
            const Met M = met_of(a, dir);
            v = v * M.d * M.j;
          }
        }
        if constexpr (!MAIN) {
          put<C>(T, S, t, flux_diff<KIND>(qn[t], ud[t], pp[t], f0, v));
        } else {
          if (uwd) {
            put<C>(T, S, t, v);
            continue;
          }
          if (metg) {
            const double jm = ldg(a.met, o), rm = m > 0 && m < 4 ? ldg(a.met + (1 + dir + 3 * (m - 1)) * fs, o) : 0.0;
            T[kLineOff + S.s[t]] = flux_diff_full(jm, rm, m, qn[t], ud[t], pp[t], v);
            if (S.h[t] != kDummy) {
              const double qh = S.ex[t] >= 0 ? halo_q<C>(a, qc, S, t, dir, m) : qn[t];
              T[kLineOff + S.h[t]] = flux_diff_full(jm, rm, m, qh, hu[t], hp[t], v);
            }
          } else {
            const Met M = met_of(a, dir);
            T[kLineOff + S.s[t]] = flux_diff_main<KIND>(M.j, M.d, qn[t], ud[t], pp[t], f0, v);
            if (S.h[t] != kDummy) {
              const double qh = S.ex[t] >= 0 ? halo_q<C>(a, qc, S, t, dir, m) : qn[t];
              T[kLineOff + S.h[t]] = flux_diff_main<KIND>(M.j, M.d, qh, hu[t], hp[t], f0, v);
            }
          }
        }
      }
    };
    auto stage_flux = [&](int m) __attribute__((always_inline)) {
      if (m == 4) stage_kind(std::integral_constant<int, FLUX_ENERGY>{}, m);
      else if (m == dir + 1 && f0 > kLargeP) stage_kind(std::integral_constant<int, FLUX_ALONG_LARGE_P>{}, m);
      else if (m == dir + 1) stage_kind(std::integral_constant<int, FLUX_ALONG>{}, m);
      else stage_kind(std::integral_constant<int, FLUX_PLAIN>{}, m);
    };
    // its derivative at slot t (the main path's fluxes carry the metrics: no
    // 1/dx after the solve)
    auto dflux = [&](int t) __attribute__((always_inline)) {
      const double x = X[S.s[t]];
      return MAIN ? x : x * idn;
    };
    if constexpr (!RK) {
      const int m0 = uwd ? 1 : 0;
      if (ONE && field < m0) return;  // without convection density has no flux
      load_inputs(ONE ? field : m0);
#pragma unroll
      for (int mm = 0; mm < (ONE ? 1 : 5); mm++) {
        const int m = ONE ? field : mm;
        if (m < m0) continue;
        stage_flux(m);
        double* dst = qrhs + m * fs;
        double qr[NPT];
        if (!FIRST || uwd) {
#pragma unroll
          for (int t = 0; t < NPT; t++) qr[t] = ldg(dst, S.g[t]);
        }
        if (!ONE && m < 4) load_inputs(m + 1);
        derive();
#pragma unroll
        for (int t = 0; t < NPT; t++) stg(dst, S.g[t], FIRST && !uwd ? dflux(t) : qr[t] + dflux(t));
      }
    } else {
      // each variable's RK3 stage update (tgvsolver.F90:1043-1059;
      // src/mainloop.F90:430-482) and, in the miniapp, its filter along dir
      // follow its flux derivative at once
      // the state the step began with (qsave of the reference) is q itself
      // in the first stage
      double* const qnew = sa.stage == 1 ? qrhs : qo;
      double qr[NPT], qs[NPT];
      auto load_rk = [&](int m) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NPT; t++) {
          qr[t] = ldg(qrhs + m * fs, S.g[t]);
          qs[t] = sa.stage == 0 ? 0.0 : ldg(qo + m * fs, S.g[t]);
        }
      };
      const int m = field;
      const bool solve = m > 0 || !uwd;  // without convection density has no flux
      load_inputs(m);
      load_rk(m);
      if (solve) {
        stage_flux(m);
        derive();
      }
      double qw[NPT];
#pragma unroll
      for (int t = 0; t < NPT; t++) {
        const double v = solve ? qr[t] + dflux(t) : qr[t];
        const double s0 = sa.stage == 0 ? qn[t] : qs[t];
        const double jb = MAIN ? jac_of<GEN>(a, S.g[t]) : 1.0;
        qw[t] = MAIN ? rk_update_main(sa, a.dt, jb, s0 * jb, qn[t], v)  // qsave = q J (mainloop.F90:423-427)
                     : rk_update(sa, a.dt, s0, qn[t], v);
      }
      if (MAIN && !a.rk_filter) {
#pragma unroll
        for (int t = 0; t < NPT; t++) stg(qnew + m * fs, S.g[t], qw[t]);
        return;
      }
      if constexpr (MAIN) {
        // updatefvar needs all five components of the unfiltered state:
        // they go to the first fields of the gradients, which the flux
        // passes no longer read, for k_fvar
#pragma unroll
        for (int t = 0; t < NPT; t++) stg(a.dv + m * fs, S.g[t], qw[t]);
      }
      // the filter sweep along dir: the miniapp's of this stage, the main
      // path's of the next (comsolver.F90:514-632)
      filter_setup(1);
#pragma unroll
      for (int t = 0; t < NPT; t++) put<C>(T, S, t, qw[t]);
      filter();
#pragma unroll
      for (int t = 0; t < NPT; t++) stg(qnew + m * fs, S.g[t], X[S.s[t]]);
    }
  } else {  // F_ONLY: filter of q along dir, in place (filterq, tgvsolver.F90:791-883)
    filter_setup(0);
#pragma unroll
    for (int mm = 0; mm < (ONE ? 1 : 5); mm++) {
      const int m = ONE ? field : mm;
#pragma unroll
      for (int t = 0; t < NPT; t++)
        put<C>(T, S, t, ldg(qc + m * fs, S.g[t]));
      filter();
      double* dst = qc + m * fs;
#pragma unroll
      for (int t = 0; t < NPT; t++)
        stg(dst, S.g[t], X[S.s[t]]);
    }
  }
}

// one pass of one case: block b handles tile xcd_tile(b)
// GEN (main path only): the general-grid form, for a direction with
// physical ends or a grid with per-point metrics; the periodic, uniform-grid
// kernels leave that code out (it would multiply their code size several
// times over, past what the instruction cache holds)
template <class C, int PROG, int MINB, bool MAIN = false, bool GEN = false>
__global__ __launch_bounds__(C::NT, MINB) void k_pass(FlowArgs a, int dir) {
  extern __shared__ double smem[];
  pass_body<C, PROG, MAIN, GEN>(a, stage_of(a), arrays_of(a, 0), dir, xcd_tile(blockIdx.x, gridDim.x), smem);
}

// Components a pass runs as separate workgroups, 0: it cannot (the stress
// pass's fluxes share the stress).
constexpr int pass_fields(int prog) {
  if (prog == GC_FIRST || prog == GC_MID || prog == GC_LAST) return 4;
  if (prog == V_MID || prog == V_LAST_RHS || prog == F_ONLY || prog == V_LAST_RK) return 5;
  return 0;
}
// Whether a pass of nt tiles runs one component per workgroup.  With few
// tiles its time is one workgroup's chain of solves, which this divides by
// the components; with many it only repeats each tile's set-up (the slots'
// index arithmetic, the coefficients) and the loads components share.
// Measured, us per launch, whole tile -> components: filter sweep 33^3 (69
// tiles) 17 -> 9, 65^3 (265) 20 -> 15.6, 97^3 (1177) 34 -> 38; flux derivative
// 11.7 -> 8.4, 16.1 -> 15.5, 33 -> 39; gradients 10.3 -> 7.6, 13.5 -> 12.2,
// 23.8 -> 25.7, and where they form the pressure too 10.3 -> 9.2, 13.8 -> 16.5.
// The RK pass solves twice per component and gains at every size (miniapp
// 33^3 23.5 -> 12, 129^3 132 -> 129; 257^3 1113 in a step), so it has that
// form only.  The general-grid kernels follow the same limits: with them, and
// one solve of each flux difference instead of one per part, a step of a
// wall-bounded stretched grid takes at 32^3 985 -> 485 us, 96x80x64 2002 ->
// 1403, 128^3 6321 -> 4935.
constexpr bool pass_one(int prog, bool pres, int nt) {
  if (pass_fields(prog) == 0) return false;
  if (prog == V_LAST_RK) return true;
  if (prog == F_ONLY) return nt <= 512;
  if (prog <= GC_LAST) return nt <= (pres ? 128 : 384);
  return nt <= 320;
}

// one component of one pass per workgroup: the tile's components are
// neighbouring blocks of one XCD, so what they share is read once into its L2
template <class C, int PROG, int MINB, bool MAIN = false, bool GEN = false>
__global__ __launch_bounds__(C::NT, MINB) void k_pass_one(FlowArgs a, int dir) {
  extern __shared__ double smem[];
  constexpr int NF = pass_fields(PROG);
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  pass_body<C, PROG, MAIN, GEN, true>(a, stage_of(a), arrays_of(a, 0), dir, b / NF, smem, b % NF);
}

// updatefvar (fludyna.F90:191-242), after the main path's RK pass and on its
// own: rho, u, v, w, p, T at every computed point of the state q.  Bound by
// bytes (11 fields), the threads go through the rows as they lie in memory: a
// workgroup of one row's points each left cache lines half written where rows
// start on half of one (on its own 129^3 32.7 -> 29.6 us, 257^3 301 -> 295).
inline dim3 fvar_grid(const FlowArgs& a) {
  return dim3(((unsigned)a.pitch * (a.n[1] + 1) * (a.n[2] + 1) + 255) / 256);
}
__global__ __launch_bounds__(256) inline void k_fvar(FlowArgs a, const double* q) {
  const unsigned rows = (a.n[1] + 1) * (a.n[2] + 1);
  const unsigned e = blockIdx.x * 256 + threadIdx.x;
  const unsigned row = e / a.pitch, i = e - row * a.pitch;
  if (row >= rows || i > (unsigned)a.n[0]) return;
  const unsigned o = e * 8u;  // rows are contiguous
  const long long fs = a.fs;
  const Prim P = prim_of(a, ldg(q, o), ldg(q + fs, o), ldg(q + 2 * fs, o), ldg(q + 3 * fs, o), ldg(q + 4 * fs, o));
  stg(a.pr, o, P.r);
  stg(a.pr + fs, o, P.u);
  stg(a.pr + 2 * fs, o, P.v);
  stg(a.pr + 3 * fs, o, P.w);
  stg(a.pr + 4 * fs, o, P.p);
  stg(a.pr + 5 * fs, o, P.t);
}

// The tiles of one pass over several cases: case k owns global tiles
// tstart[k]..tstart[k+1]-1.  Device arrays, built by the batch host code.
struct BatchLaunch {
  const FlowArgs* cases;
  const int* tstart;
  int ncases;
  int total;
};

// one pass over a batch of cases, a workgroup per tile (ONE: per component of
// a tile): the blocks of XCD x take the contiguous range [x*total/8,
// (x+1)*total/8) so neighbouring tiles share that XCD's L2.  The grid is the
// tiles, rounded up to 8: as many persistent blocks as the register budget
// names (1 or 2 per CU) left the passes of few registers without the
// wavefronts that fit (a mixed batch of 12 cases of side 32 to 96: 16.6 ->
// 15.3 ms for 5 steps).
template <class C, int PROG, int MINB, bool ONE = false>
__global__ __launch_bounds__(C::NT, MINB) void k_pass_batch(BatchLaunch bl, int dir, StageArgs sa) {
  extern __shared__ double smem[];
  const int x = blockIdx.x & 7;
  constexpr int NF = ONE ? pass_fields(PROG) : 1;
  const long long total = (long long)bl.total * NF;
  const int e = (int)(total * x / 8) + (int)(blockIdx.x >> 3);
  if (e >= (int)(total * (x + 1) / 8)) return;
  const int g = e / NF;
  int kl = 0, kh = bl.ncases;  // tstart[kl] <= g < tstart[kh]
  while (kh - kl > 1) {
    const int mid = (kl + kh) >> 1;
    if (bl.tstart[mid] <= g) kl = mid;
    else kh = mid;
  }
  const FlowArgs& a = bl.cases[kl];
  pass_body<C, PROG, false, false, ONE>(a, sa, arrays_of(a, sa.alt), dir, g - bl.tstart[kl], smem, e % NF);
}

template <class C, int MINB>
hipError_t launch_batch_c(int prog, const BatchLaunch& bl, int dir, const StageArgs& sa, int nblocks,
                          hipStream_t st) {
  const size_t lds = (size_t)lds_doubles<C>(prog) * sizeof(double);
  dim3 g(nblocks), b(C::NT);
#define ASTR_BATCH_PASS(P, O) hipLaunchKernelGGL((k_pass_batch<C, P, MINB, O>), g, b, lds, st, bl, dir, sa)
  const bool one = pass_one(prog, dir == 1, bl.total);
  switch (prog) {
    // the y gradient pass is a stage's first: it forms the pressure
    case GC_MID:
    case GC_LAST:
      if (dir == 1) {
        if (one) ASTR_BATCH_PASS(GC_FIRST, true);
        else ASTR_BATCH_PASS(GC_FIRST, false);
      } else {
        if (one) ASTR_BATCH_PASS(GC_MID, true);
        else ASTR_BATCH_PASS(GC_MID, false);
      }
      break;
    case V_MID:
      if (dir == 0) ASTR_BATCH_PASS(V_FIRST_G, false);
      else if (one) ASTR_BATCH_PASS(V_MID, true);
      else ASTR_BATCH_PASS(V_MID, false);
      break;
    case V_LAST_RK: ASTR_BATCH_PASS(V_LAST_RK, true); break;
    // single-case passes only
    case GC_FIRST:
    case V_LAST_RHS:
    case FGC_FIRST:
    case RESERVED_7:
    case RESERVED_8: return hipErrorInvalidValue;
    default:
      if (one) ASTR_BATCH_PASS(F_ONLY, true);
      else ASTR_BATCH_PASS(F_ONLY, false);
      break;
  }
#undef ASTR_BATCH_PASS
  return hipGetLastError();
}

template <class C, int MINB, bool MAIN, bool GEN>
void launch_pass_m(int prog, const FlowArgs& a, int dir, hipStream_t st) {
  const int nt = tiles_of(a.n, dir, C::TL);
  const size_t lds = (size_t)lds_doubles<C>(prog, MAIN) * sizeof(double);
  dim3 g(nt), b(C::NT);
  const bool pres = !MAIN && (prog == GC_FIRST || (a.gradx && dir == 1));
  if (!(prog == V_MID && dir == 0) && pass_one(prog, pres, nt)) {
    switch (prog) {
      case GC_FIRST:
      case GC_MID:
      case GC_LAST:
        if (pres || prog == GC_FIRST)
          hipLaunchKernelGGL((k_pass_one<C, GC_FIRST, MINB, MAIN, GEN>), dim3(4 * nt), b, lds, st, a, dir);
        else
          hipLaunchKernelGGL((k_pass_one<C, GC_MID, MINB, MAIN, GEN>), dim3(4 * nt), b, lds, st, a, dir);
        return;
      case V_MID:
      case V_LAST_RHS:
        hipLaunchKernelGGL((k_pass_one<C, V_MID, MINB, MAIN, GEN>), dim3(5 * nt), b, lds, st, a, dir);
        return;
      case V_LAST_RK:
        hipLaunchKernelGGL((k_pass_one<C, V_LAST_RK, MINB, MAIN, GEN>), dim3(5 * nt), b, lds, st, a, dir);
        if constexpr (MAIN) {
          const double* q = a.rk_filter ? a.dv : (a.stage == 1 ? a.qrhs : a.qsave);
          hipLaunchKernelGGL(k_fvar, fvar_grid(a), dim3(256), 0, st, a, q);
        }
        return;
      case F_ONLY:
        hipLaunchKernelGGL((k_pass_one<C, F_ONLY, MINB, GEN, GEN>), dim3(5 * nt), b, lds, st, a, dir);
        return;
      default: break;
    }
  }
  switch (prog) {
    case GC_FIRST: hipLaunchKernelGGL((k_pass<C, GC_FIRST, MINB, MAIN, GEN>), g, b, lds, st, a, dir); break;
    case GC_MID:
    case GC_LAST:
      // miniapp, without an x gradient pass: the stage's first, which forms
      // the pressure
      if constexpr (!MAIN) {
        if (a.gradx && dir == 1) {
          hipLaunchKernelGGL((k_pass<C, GC_FIRST, MINB, false, false>), g, b, lds, st, a, dir);
          break;
        }
      }
      hipLaunchKernelGGL((k_pass<C, GC_MID, MINB, MAIN, GEN>), g, b, lds, st, a, dir);
      break;
    case V_MID:
      if (dir == 0) {
        if constexpr (!GEN) {
          if (a.gradx) {
            const size_t ldsg = (size_t)lds_doubles<C>(V_FIRST_G, MAIN) * sizeof(double);
            hipLaunchKernelGGL((k_pass<C, V_FIRST_G, MINB, MAIN, false>), g, b, ldsg, st, a, dir);
            break;
          }
        }
        hipLaunchKernelGGL((k_pass<C, V_FIRST, MINB, MAIN, GEN>), g, b, lds, st, a, dir);
        break;
      }
      [[fallthrough]];
    case V_LAST_RHS: hipLaunchKernelGGL((k_pass<C, V_MID, MINB, MAIN, GEN>), g, b, lds, st, a, dir); break;
    case V_LAST_RK: break;  // pass_one always
    // the filtering first pass exists for the miniapp's stage only (the main
    // path filters at the start of its stage); launch_pass_c refuses it there
    case FGC_FIRST:
      if constexpr (!MAIN) hipLaunchKernelGGL((k_pass<C, FGC_FIRST, MINB, false, false>), g, b, lds, st, a, dir);
      break;
    // the filter pass of the main path also takes physical boundaries
    default: hipLaunchKernelGGL((k_pass<C, F_ONLY, MINB, MAIN, GEN>), g, b, lds, st, a, dir); break;
  }
}

template <class C, int MINB>
hipError_t launch_pass_c(int prog, const FlowArgs& a, int dir, hipStream_t st) {
  if (prog == FGC_FIRST && (a.main_sem || dir != 0)) return hipErrorInvalidValue;
  if (prog == RESERVED_7 || prog == RESERVED_8) return hipErrorInvalidValue;
  if (a.main_sem && (a.met || a.bnd[dir])) launch_pass_m<C, MINB, true, true>(prog, a, dir, st);
  else if (a.main_sem) launch_pass_m<C, MINB, true, false>(prog, a, dir, st);
  else launch_pass_m<C, MINB, false, false>(prog, a, dir, st);
  return hipGetLastError();
}

// launch shapes (threads, lines per tile, chunk length, point slots per thread)
using CfgA = LineCfg<256, 4, 5, 5>;    // P=64, n <= 313
using CfgB = LineCfg<256, 4, 9, 9>;    // P=64, n <= 569
using CfgC = LineCfg<256, 16, 5, 5>;   // P=16, n <= 73
using CfgD = LineCfg<256, 8, 9, 9>;    // P=32, n <= 281
using CfgE = LineCfg<256, 8, 5, 5>;    // P=32, n <= 153
using CfgF = LineCfg<512, 8, 5, 5>;    // P=64, n <= 313: CfgA's lines, 64-byte row segments
using CfgG = LineCfg<128, 4, 9, 9>;    // P=32, n <= 281: CfgD's lines, two workgroups per CU at 1 wave/SIMD
using CfgH = LineCfg<128, 2, 5, 5>;    // P=64, n <= 313: CfgA's lines in half-size workgroups
using CfgI = LineCfg<64, 1, 5, 5>;     // P=64, n <= 313: one line per single-wavefront workgroup
using CfgJ = LineCfg<64, 2, 9, 9>;     // P=32, n <= 281: two lines per single-wavefront workgroup
using CfgK = LineCfg<256, 16, 9, 9>;   // P=16, n <= 137: 128-byte row segments for mid-size lines
using CfgL = LineCfg<512, 8, 9, 9>;    // P=64, n <= 569: CfgB's lines, 64-byte row segments
using CfgM = LineCfg<64, 1, 9, 9>;     // P=64, n <= 569: one long line per single-wavefront workgroup
constexpr int kNumShapes = 13;
constexpr int kMinbVariants = 2;       // MINB = 1, 2

// one per shape, each in its own translation unit (passes.hip)
#define ASTR_DECLARE_SHAPE(K)                                                                 \
  hipError_t launch_pass_s##K(int prog, int minb, const FlowArgs& a, int dir, hipStream_t st); \
  hipError_t launch_batch_s##K(int prog, int minb, const BatchLaunch& bl, int dir,             \
                               const StageArgs& sa, int nblocks, hipStream_t st);
ASTR_DECLARE_SHAPE(0)
ASTR_DECLARE_SHAPE(1)
ASTR_DECLARE_SHAPE(2)
ASTR_DECLARE_SHAPE(3)
ASTR_DECLARE_SHAPE(4)
ASTR_DECLARE_SHAPE(5)
ASTR_DECLARE_SHAPE(6)
ASTR_DECLARE_SHAPE(7)
ASTR_DECLARE_SHAPE(8)
ASTR_DECLARE_SHAPE(9)
ASTR_DECLARE_SHAPE(10)
ASTR_DECLARE_SHAPE(11)
ASTR_DECLARE_SHAPE(12)
#undef ASTR_DECLARE_SHAPE

}  // namespace astr
