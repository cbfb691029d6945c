// The advective face flux on the device: face sides by constant or MUSCL
// reconstruction, then KEEP (kepaec), HLLC or Rusanov.
//
// Every function here is evaluated with one rounding per written operation, in the order the
// reference's templates write it: the face fluxes feed the next stage's EOS, whose ln T
// polynomials turn any last-bit difference into 1e-11 of T, so a contracted multiply-add
// here would show at 1e-10 after a hundred steps.
#pragma once

#include "pga_eos.hpp"

namespace pga {

enum { RECON_CONSTANT = 0, RECON_MUSCL = 1 };
enum { FLUX_KEPAEC = 0, FLUX_HLLC = 1, FLUX_RUSANOV = 2 };

template <int NS>
struct FaceState {
  EosState s;
  double u, v, w;
  double Y[NS > 1 ? NS - 1 : 1];
};

enum { LIM_NONE = 0, LIM_KOREN = 1, LIM_MINMOD = 2, LIM_MC = 3, LIM_SUPERBEE = 4, LIM_VANLEER = 5 };

// half of b phi(a / b), b >= 0, without the ratio (recon/{koren,minmod,mc,superbee,vanleer}.mako). Koren's
// min(min(2a, (2b + a) / 3), 2b) halved is min(min(a, ((2b + a) / 3) / 2), b): halving is exact, and so is
// 2b inside the fused add
template <int LIM>
__device__ __forceinline__ double half_limit(double a, double b) {
#pragma clang fp contract(off)
  if constexpr (LIM == LIM_KOREN) return fmax(0.0, fmin(fmin(a, 0.5 * (fma(2.0, b, a) * (1.0 / 3.0))), b));
  if constexpr (LIM == LIM_MINMOD) return fmax(0.0, 0.5 * fmin(b, a));
  if constexpr (LIM == LIM_MC) return fmax(0.0, fmin(fmin(a, 0.5 * ((b + a) * 0.5)), b));
  if constexpr (LIM == LIM_SUPERBEE) return 0.5 * fmax(0.0, fmax(fmin(2.0 * a, b), fmin(a, 2.0 * b)));
  return 0.5 * ((a + fabs(a)) * b / (b + fabs(a)));
}

// recon/muscl.mako:5-13 for both sides of a face: L = vL + phi(vL - vLL, dp) / 2 and R = vR - phi(vRR - vR,
// dp) / 2, dp = vR - vL, phi the limited slope carried to dp's sign and back. The sign is a factor +-1 whose
// product is exact, so it is folded into the last add. A zero dp gives a zero slope by itself (b = 0), but
// van Leer's, which would divide by b. Evaluated on every lane and selected, so the 26 slopes of a face
// stay one basic block the scheduler can interleave. 21 instructions a pair where the two slopes apart,
// with their scalings and a select each, were 33: 170 of the 1230 a nine-species face takes
template <int LIM>
__device__ __forceinline__ void limited_sides(double vLL, double vL, double vR, double vRR, double &l, double &r) {
#pragma clang fp contract(off)
  const double dp = vR - vL, s = copysign(1.0, dp), b = fabs(dp);
  double hl = half_limit<LIM>(s * (vL - vLL), b), hr = half_limit<LIM>(s * (vRR - vR), b);
  if constexpr (LIM == LIM_VANLEER) {
    hl = dp != 0.0 ? hl : 0.0;
    hr = dp != 0.0 ? hr : 0.0;
  }
  l = fma(s, hl, vL);
  r = fma(-s, hr, vR);
}

// the face's sides from the two cells as they are (recon/constant.mako:3-18); o is the offset of the
// face's right cell R, d the stride along the axis
template <int NS>
__device__ __forceinline__ void constant_sides(const View &Q, const View &st, int64_t o, int64_t d, FaceState<NS> &L,
                                               FaceState<NS> &R) {
#pragma clang fp contract(off)
  const int64_t oL = o - d;
  load_state(st, oL, L.s);
  load_state(st, o, R.s);
  const double rL = Q.at(oL, 0), rR = Q.at(o, 0);
  L.u = Q.at(oL, 1) / rL;
  L.v = Q.at(oL, 2) / rL;
  L.w = Q.at(oL, 3) / rL;
  R.u = Q.at(o, 1) / rR;
  R.v = Q.at(o, 2) / rR;
  R.w = Q.at(o, 3) / rR;
#pragma unroll
  for (int n = 0; n < NS - 1; n++) {
    L.Y[n] = Q.at(oL, 5 + n) / rL;
    R.Y[n] = Q.at(o, 5 + n) / rR;
  }
}

// the primitives MUSCL limits, by number: p, T, the velocity, the carried mass fractions
enum { PRIM_P = 0, PRIM_T = 1, PRIM_U = 2, PRIM_Y = 5 };

// the primitives of a face's four cells LL, L, R, RR (m = 0..3), read from the cell arrays
template <int NS>
struct ArrayStencil {
  const View &Q, &st;
  int64_t o, d;
  double ri[4];
  __device__ __forceinline__ ArrayStencil(const View &Q_, const View &st_, int64_t o_, int64_t d_)
      : Q(Q_), st(st_), o(o_), d(d_) {
#pragma unroll
    for (int m = 0; m < 4; m++) ri[m] = st.at(o + (m - 2) * d, 2);
  }
  __device__ __forceinline__ double operator()(int v, int m) const {
#pragma clang fp contract(off)
    const int64_t om = o + (m - 2) * d;
    if (v < PRIM_U) return st.at(om, v);
    return Q.at(om, v < PRIM_Y ? v - 1 : v) * ri[m];
  }
};

// the face's sides by MUSCL (recon/muscl.mako:15-51): p, T, Y and the velocity limited, each side closed
// by the eos from p, T, Y. Evaluated with one rounding per operation: the sides' p and T feed the EOS's
// ill-conditioned ln T polynomials, where a last-bit change in T moves e by 1e-11 of itself
template <int NS, int EOS, int LIM, class SRC>
__device__ __forceinline__ void muscl_sides(const Gas<NS> &g, const SRC &x, FaceState<NS> &L, FaceState<NS> &R) {
#pragma clang fp contract(off)
  const auto sides = [&](int v, double &l, double &r) {
    limited_sides<LIM>(x(v, 0), x(v, 1), x(v, 2), x(v, 3), l, r);
  };
  // T and its logarithms first: the species' constants, which the branch in elog2 would otherwise keep in
  // scalar registers across it, are not loaded yet
  double pL, pR, TL, TR, uL = 0.0, uR = 0.0;
  sides(PRIM_T, TL, TR);
  if constexpr (EOS == EOS_TPG) elog2(TL, TR, uL, uR);
  sides(PRIM_P, pL, pR);
#pragma unroll
  for (int n = 0; n < NS - 1; n++) sides(PRIM_Y + n, L.Y[n], R.Y[n]);
  MixMom<NS, EOS> mL, mR;
  mixmom2<NS, EOS>(g, [&](int n) { return L.Y[n]; }, [&](int n) { return R.Y[n]; }, mL, mR);
  frompT<NS, EOS>(g, mL, [&](int n) { return L.Y[n]; }, pL, TL, [&]() { return uL; }, L.s);
  sides(PRIM_U, L.u, R.u);
  sides(PRIM_U + 1, L.v, R.v);
  sides(PRIM_U + 2, L.w, R.w);
  frompT<NS, EOS>(g, mR, [&](int n) { return R.Y[n]; }, pR, TR, [&]() { return uR; }, R.s);
}

// function/kepaec.mako:2-20 (Shima et al. 2021): arithmetic means, the harmonic mean of cv T
template <int NS>
__device__ __forceinline__ void kepaec(const FaceState<NS> &L, const FaceState<NS> &R, const double S[3],
                                       double F[NS + 4]) {
#pragma clang fp contract(off)
  const double uf = 0.5 * (R.u + L.u), vf = 0.5 * (R.v + L.v), wf = 0.5 * (R.w + L.w);
  const double U = S[0] * uf + S[1] * vf + S[2] * wf;
  const double pf = 0.5 * (R.s.p + L.s.p);
  const double rho = 0.5 * (R.s.rho + L.s.rho);
  const double C = rho * U;
  F[0] = C;
  F[1] = C * uf + pf * S[0];
  F[2] = C * vf + pf * S[1];
  F[3] = C * wf + pf * S[2];
  const double Kj = C * 0.5 * (R.u * L.u + R.v * L.v + R.w * L.w);
  const double Pj = 0.5 * (L.s.p * (R.u * S[0] + R.v * S[1] + R.w * S[2]) + R.s.p * (L.u * S[0] + L.v * S[1] + L.w * S[2]));
  const double thL = L.s.cp / L.s.gamma * L.s.T, thR = R.s.cp / R.s.gamma * R.s.T;
  const double ef = 2.0 * thL * thR / (thL + thR) + 0.5 * ((L.s.e - thL) + (R.s.e - thR));
  F[4] = ef * C + Kj + Pj;
#pragma unroll
  for (int n = 0; n < NS - 1; n++) F[5 + n] = 0.5 * (R.Y[n] + L.Y[n]) * C;
}

// function/hllc.mako:2-43: Davis wave speeds, the star jump through drho and dU
template <int NS>
__device__ __forceinline__ void hllc(const FaceState<NS> &L, const FaceState<NS> &R, const double S[3],
                                     double F[NS + 4]) {
#pragma clang fp contract(off)
  const double area = sqrt(S[0] * S[0] + S[1] * S[1] + S[2] * S[2]);
  const double nx = S[0] / area, ny = S[1] / area, nz = S[2] / area;
  const double unL = (L.u * S[0] + L.v * S[1] + L.w * S[2]) / area;
  const double unR = (R.u * S[0] + R.v * S[1] + R.w * S[2]) / area;
  const double SL = unL - L.s.c, SR = unR + R.s.c;
  const double Sstar = (R.s.p - L.s.p + L.s.rho * unL * (SL - unL) - R.s.rho * unR * (SR - unR)) /
                       (L.s.rho * (SL - unL) - R.s.rho * (SR - unR));
  const bool left = SL >= 0.0 || Sstar >= 0.0;
  const bool star = !(SL >= 0.0) && (Sstar >= 0.0 || SR >= 0.0);
  // the upwind side's values, selected one by one (a reference to one side would put both in memory)
  const double Xrho = left ? L.s.rho : R.s.rho, Xp = left ? L.s.p : R.s.p, Xe = left ? L.s.e : R.s.e;
  const double Xu = left ? L.u : R.u, Xv = left ? L.v : R.v, Xw = left ? L.w : R.w;
  const double U = left ? unL : unR, SX = left ? SL : SR;
  const double et = Xe + 0.5 * (Xu * Xu + Xv * Xv + Xw * Xw);
  const double mdot = U * Xrho * area;
  F[0] = mdot;
  F[1] = mdot * Xu + Xp * S[0];
  F[2] = mdot * Xv + Xp * S[1];
  F[3] = mdot * Xw + Xp * S[2];
  F[4] = mdot * et + U * Xp * area;
#pragma unroll
  for (int n = 0; n < NS - 1; n++) F[5 + n] = mdot * (left ? L.Y[n] : R.Y[n]);
  if (star) {
    const double rhostar = Xrho * ((SX - U) / (SX - Sstar));
    const double drho = rhostar - Xrho, dU = rhostar * (Sstar - U);
    const double jump = SX * area;
    F[0] += jump * drho;
    F[1] += jump * (drho * Xu + dU * nx);
    F[2] += jump * (drho * Xv + dU * ny);
    F[3] += jump * (drho * Xw + dU * nz);
    F[4] += jump * (drho * et + dU * (Sstar + Xp / (Xrho * (SX - U))));
#pragma unroll
    for (int n = 0; n < NS - 1; n++) F[5 + n] += jump * drho * (left ? L.Y[n] : R.Y[n]);
  }
}

// function/rusanov.mako:2-19: the central flux less the largest Davis wave speed's jump
template <int NS>
__device__ __forceinline__ void rusanov(const FaceState<NS> &L, const FaceState<NS> &R, const double S[3],
                                        double F[NS + 4]) {
#pragma clang fp contract(off)
  const double area = sqrt(S[0] * S[0] + S[1] * S[1] + S[2] * S[2]);
  const double unL = (L.u * S[0] + L.v * S[1] + L.w * S[2]) / area;
  const double unR = (R.u * S[0] + R.v * S[1] + R.w * S[2]) / area;
  const double lam = fmax(fabs(unL) + L.s.c, fabs(unR) + R.s.c) * area;
  const double UL = unL * area, UR = unR * area;
  const double rL = L.s.rho, rR = R.s.rho;
  F[0] = 0.5 * (UR * rR + UL * rL - lam * (rR - rL));
  F[1] = 0.5 * (UR * rR * R.u + R.s.p * S[0] + UL * rL * L.u + L.s.p * S[0] - lam * (rR * R.u - rL * L.u));
  F[2] = 0.5 * (UR * rR * R.v + R.s.p * S[1] + UL * rL * L.v + L.s.p * S[1] - lam * (rR * R.v - rL * L.v));
  F[3] = 0.5 * (UR * rR * R.w + R.s.p * S[2] + UL * rL * L.w + L.s.p * S[2] - lam * (rR * R.w - rL * L.w));
  const double EL = rL * (L.s.e + 0.5 * (L.u * L.u + L.v * L.v + L.w * L.w));
  const double ER = rR * (R.s.e + 0.5 * (R.u * R.u + R.v * R.v + R.w * R.w));
  F[4] = 0.5 * (UR * (ER + R.s.p) + UL * (EL + L.s.p) - lam * (ER - EL));
#pragma unroll
  for (int n = 0; n < NS - 1; n++) {
    const double rhoYL = rL * L.Y[n], rhoYR = rR * R.Y[n];
    F[5 + n] = 0.5 * (rhoYR * UR + rhoYL * UL - lam * (rhoYR - rhoYL));
  }
}

template <int NS, int PRIMARY>
__device__ __forceinline__ void flux_function(const FaceState<NS> &L, const FaceState<NS> &R, const double S[3],
                                              double F[NS + 4]) {
  if constexpr (PRIMARY == FLUX_KEPAEC)
    kepaec<NS>(L, R, S, F);
  else if constexpr (PRIMARY == FLUX_HLLC)
    hllc<NS>(L, R, S, F);
  else
    rusanov<NS>(L, R, S, F);
}

// the face's area vector, read by this face alone
__device__ __forceinline__ void load_area(const View &S, int i, int j, int k, double (&Sv)[3]) {
  uint32_t b = View::bytes(S.off(i, j, k));
#pragma unroll
  for (int d = 0; d < 3; d++) Sv[d] = __builtin_nontemporal_load(&S.run(b, d));
}

// The face's flux stored past the caches: a face value is written once and read back by the stage from HBM
// in any case, and the stencil's Q and state keep L2 (5% on the 128^3 step's faces)
template <int NS>
__device__ __forceinline__ void store_flux(const View &F, int i, int j, int k, const double (&Fv)[NS + 4]) {
  uint32_t b = View::bytes(F.off(i, j, k));
#pragma unroll
  for (int l = 0; l < NS + 4; l++) __builtin_nontemporal_store(Fv[l], &F.run(b, l));
}

// the face (i, j, k) of `axis` (between cells k - 1 and k along it): its sides, its area into Sv and its
// flux into Fv
template <int NS, int EOS, int RECON, int PRIMARY, int LIM>
__device__ __forceinline__ void flux_at(const double *__restrict__ K, int axis, const View &Q, const View &st,
                                        const View &S, int i, int j, int k, double (&Sv)[3], double (&Fv)[NS + 4]) {
  const Gas<NS> g{K};
  const int64_t o = Q.off(i, j, k);
  const int64_t d = axis == 0 ? 1 : axis == 1 ? Q.sj : Q.sk;
  FaceState<NS> L, R;
  // the constant reconstruction's face waits on memory once, its area among the cells' values and cached: a
  // small block's areas stay in L2 from stage to stage
  if constexpr (RECON == RECON_CONSTANT) {
    uint32_t b = View::bytes(S.off(i, j, k));
#pragma unroll
    for (int m = 0; m < 3; m++) Sv[m] = S.run(b, m);
    constant_sides<NS>(Q, st, o, d, L, R);
  } else {
    muscl_sides<NS, EOS, LIM>(g, ArrayStencil<NS>(Q, st, o, d), L, R);
    load_area(S, i, j, k, Sv);
  }
  flux_function<NS, PRIMARY>(L, R, Sv, Fv);
}

// the face's flux into the face array
template <int NS, int EOS, int RECON, int PRIMARY, int LIM>
__device__ __forceinline__ void flux_face(const double *__restrict__ K, int axis, const View &Q, const View &st,
                                          const View &S, const View &F, int i, int j, int k) {
  double Sv[3], Fv[NS + 4];
  flux_at<NS, EOS, RECON, PRIMARY, LIM>(K, axis, Q, st, S, i, j, k, Sv, Fv);
  store_flux<NS>(F, i, j, k, Fv);
}

// ---------------------------------------------------------------------------
// MUSCL faces by tiles: the workgroup's 256 faces read their cells' primitives from LDS, where each cell
// of the tile is put once. A face of its own reads 56 values of the cell arrays for nine species, more than
// registers hold in flight beside the sides and their EOS, so it waited on memory several times over at
// three waves a SIMD. Staged, a thread has the 14 loads of a cell or two in flight at once and waits once,
// the velocities and mass fractions are divided out once a cell and not four times, and the stencils'
// reads are LDS's: the faces of the reacting 128^3 block went from 440 to 409 us a launch, 382 with the
// limiter's and the indexes' shorter forms below, which is 4.2 TB/s of the 4.8 a plain copy reaches here
// (four waves a SIMD in place of three then change nothing). The cubic real gas is bound by its roots and
// logarithms, not by these loads: staged, the faces of the 256 x 128 x 64 layer took 732 us against 686,
// so it reads its stencils from the arrays.
//
// i faces: nf consecutive faces of the box's rows, a row's run of them with its three cells more. j and k
// faces: wi faces along i by 256 / wi along the axis, with three planes of cells more. A cell's values lie
// side by side (an odd number of doubles, so the lanes' slots spread over every bank) and a face's four
// cells are `step` slots apart.
// ---------------------------------------------------------------------------
constexpr int slot_doubles(int ns) { return (ns + 4) | 1; }
template <int NS>
constexpr int SLOT = slot_doubles(NS);
// the LDS a tile may take, whatever the species count: what any launch may ask for without its limit raised
constexpr unsigned FACE_LDS = 65536;

constexpr bool staged(int eos, int recon) { return recon == RECON_MUSCL && eos != EOS_REAL; }

template <int NS>
struct SlotStencil {
  const double *s;  // the face's LL cell
  int step;
  __device__ __forceinline__ double operator()(int v, int m) const { return s[m * step * SLOT<NS> + v]; }
};

// one axis's faces in tiles: nf (i) or the log of wi (j, k)
struct FaceTiles {
  int axis, shape;
  Box3 b;
  FastDiv row, run, plane;  // i: by the row's faces, its cells, the box's rows. j, k: by the tiles along i, along the axis
};

__host__ inline unsigned face_tile_slots(const FaceTiles &t) {
  if (t.axis == 0) return (unsigned)(t.shape + 3 * std::min(t.shape, (t.shape - 2) / t.b.e0 + 2));
  return (1u << t.shape) * ((unsigned)(FLAT >> t.shape) + 3);
}

__host__ inline int64_t face_tile_count(const FaceTiles &t) {
  const Box3 &b = t.b;
  if (t.axis == 0) return ((int64_t)b.e0 * b.e1 * b.e2 + t.shape - 1) / t.shape;
  const int wi = 1 << t.shape, ta = FLAT / wi;
  const int64_t ea = t.axis == 1 ? b.e1 : b.e2, eo = t.axis == 1 ? b.e2 : b.e1;
  return (int64_t)((b.e0 + wi - 1) / wi) * ((ea + ta - 1) / ta) * eo;
}

// The tile shape of a box's faces. i: 256 faces, fewer where short rows would bring more than 352 slots
// (36 KB for nine species, 58 for the most a case may have). j, k: the width whose waves and staged cells cost
// least, a wave of faces taken as eight times its 64 lanes' staging, among those whose slots fit FACE_LDS:
// widths 16, 32 and 64 stage 304, 352 and 448 cells, so from 14 species on (68 KB) 64 is not taken
__host__ inline FaceTiles face_tiles(int axis, const Box3 &b, int ns) {
  FaceTiles t{axis, 256, b, {}, {}, {}};
  if (axis == 0) {
    while (t.shape > 64 && face_tile_slots(t) > 352) t.shape /= 2;
    t.row = fast_div(b.e0), t.run = fast_div(b.e0 + 3), t.plane = fast_div(b.e1);
    return t;
  }
  const int64_t ea = axis == 1 ? b.e1 : b.e2;
  int64_t least = 0;
  for (int s = 4; s <= 6; s++) {
    const int64_t wi = 1 << s, ta = FLAT / wi, nbi = (b.e0 + wi - 1) / wi, full = ea / ta, rem = ea % ta;
    if (wi * (ta + 3) * slot_doubles(ns) * (int64_t)sizeof(double) > FACE_LDS) continue;
    const int64_t waves = nbi * (full * (FLAT / 64) + (rem * wi + 63) / 64);
    const int64_t cost = waves * 64 * 8 + nbi * wi * (ea + 3 * (full + (rem > 0)));
    if (s == 4 || cost < least) least = cost, t.shape = s;
  }
  const unsigned wi = 1u << t.shape, ta = FLAT / wi;
  t.row = fast_div((b.e0 + wi - 1) / wi), t.run = fast_div((unsigned)(ea + ta - 1) / ta);
  return t;
}

// Stages tile t's cells into lds and gives the thread its face: false for a thread with none. Ends in a
// barrier that every thread of the workgroup passes.
template <int NS>
__device__ __forceinline__ bool face_tile(const FaceTiles &ft, unsigned t, const View &Q, const View &st, double *lds,
                                          int &i, int &j, int &k, SlotStencil<NS> &x) {
#pragma clang fp contract(off)
  const Box3 &b = ft.b;
  const unsigned tid = threadIdx.x, e0 = b.e0, e1 = b.e1;
  unsigned nslot, slot;
  bool on;
  // slot q's cell
  unsigned col0 = 0, row0 = 0, len0 = 0, ibeg = 0, abeg = 0;
  int fixed = 0;
  if (ft.axis == 0) {
    const unsigned f0 = t * (unsigned)ft.shape, total = e0 * e1 * (unsigned)b.e2;
    const unsigned n = min((unsigned)ft.shape, total - f0);
    row0 = ft.row(f0), col0 = f0 - row0 * e0;
    len0 = min(e0 - col0, n) + 3;
    nslot = n + 3 * (ft.row(col0 + n - 1) + 1);
    const unsigned c = col0 + tid, seg = ft.row(c), row = row0 + seg, p = ft.plane(row);
    on = tid < n;
    slot = tid + 3 * seg;
    i = b.s0 + (int)(c - seg * e0), j = b.s1 + (int)(row - p * e1), k = b.s2 + (int)p;
    x.step = 1;
  } else {
    const unsigned lw = ft.shape, wi = 1u << lw, ta = FLAT >> lw;
    const unsigned ea = ft.axis == 1 ? e1 : (unsigned)b.e2;
    const unsigned rest = ft.row(t);
    ibeg = (t - rest * ft.row.d) << lw, fixed = (int)ft.run(rest), abeg = (rest - (unsigned)fixed * ft.run.d) * ta;
    const unsigned na = min(ta, ea - abeg), ii = ibeg + (tid & (wi - 1)), aa = tid >> lw;
    on = ii < e0 && aa < na;
    nslot = (na + 3) << lw;
    slot = tid;
    i = b.s0 + (int)ii;
    j = b.s1 + (ft.axis == 1 ? (int)(abeg + aa) : fixed), k = b.s2 + (ft.axis == 1 ? fixed : (int)(abeg + aa));
    x.step = (int)wi;
  }
  const auto cell = [&](unsigned q) -> int64_t {
    if (ft.axis == 0) {
      const bool first = q < len0;
      const unsigned r = first ? 0 : q - len0, seg = ft.run(r);
      const unsigned row = first ? row0 : row0 + 1 + seg, p = ft.plane(row);
      const int ci = first ? (int)(col0 + q) - 2 : (int)(r - seg * (e0 + 3)) - 2;
      return Q.off(b.s0 + ci, b.s1 + (int)(row - p * e1), b.s2 + (int)p);
    }
    // columns past the box repeat its last
    const int ci = b.s0 + (int)min(ibeg + (q & ((1u << ft.shape) - 1)), e0 - 1), ca = (int)(abeg + (q >> ft.shape)) - 2;
    return ft.axis == 1 ? Q.off(ci, b.s1 + ca, b.s2 + fixed) : Q.off(ci, b.s1 + fixed, b.s2 + ca);
  };
  const auto load = [&](unsigned q, double (&r)[NS + 5]) {
    uint32_t o = View::bytes(cell(q));
    r[NS + 4] = st.run(o, 2);
    r[0] = st.run(o, 0), r[1] = st.run(o, 1);
#pragma unroll
    for (int c = 1; c < 4; c++) r[1 + c] = Q.run(o, c);
#pragma unroll
    for (int n = 0; n < NS - 1; n++) r[5 + n] = Q.run(o, 5 + n);
  };
  const auto put = [&](unsigned q, const double (&r)[NS + 5]) {
    double *s = lds + q * SLOT<NS>;
    s[0] = r[0], s[1] = r[1];
#pragma unroll
    for (int v = 2; v < NS + 4; v++) s[v] = r[v] * r[NS + 4];
  };
  for (unsigned q = tid; q < nslot; q += 2 * FLAT) {
    double r0[NS + 5], r1[NS + 5];
    load(q, r0);
    const bool two = q + FLAT < nslot;
    if (two) load(q + FLAT, r1);
    put(q, r0);
    if (two) put(q + FLAT, r1);
  }
  __syncthreads();
  x.s = lds + slot * SLOT<NS>;
  return on;
}

// the area Sv and flux Fv of face (i, j, k) from its staged stencil
template <int NS, int EOS, int PRIMARY, int LIM>
__device__ __forceinline__ void flux_slots(const double *__restrict__ K, const SlotStencil<NS> &x, const View &S, int i,
                                           int j, int k, double (&Sv)[3], double (&Fv)[NS + 4]) {
  load_area(S, i, j, k, Sv);
  FaceState<NS> L, R;
  muscl_sides<NS, EOS, LIM>(Gas<NS>{K}, x, L, R);
  flux_function<NS, PRIMARY>(L, R, Sv, Fv);
}

}  // namespace pga
