// Walls (simulator/euler/bcs.py:15-27, navstokes/bcs.py:27-53): each wall's halo from the interior's
// image across it (the preadvflux hook) and the wall's own flux through its faces (the postflux
// hook), for the six kinds the reference names:
//   slp-adia-wall, slp-isot-wall      the velocity mirrored across the wall (euler/kernels/bcs/
//                                     slp-{adia,isot}-wall.mako); no shear
//   no-slp-adia-wall, no-slp-isot-wall the velocity held at zero, and mov-adia-wall, mov-isot-wall
//   mov-adia-wall, mov-isot-wall      at the wall's own (navstokes/kernels/bcs/{no-slp,mov}-*.mako,
//                                     wall.mako stuckhalo, stuckhaloisot)
// an isothermal wall's halo takes the wall's T (its state by the EOS from p, T_w), and its flux the
// heat flux from T_w and the transport properties at the wall (wall.mako wallcoeffs, isotflux).
//
// A block's walls go in one launch of each kind: they are planes of a few thousand cells, each worth a
// few microseconds of latency and a launch, and none reads what another writes (each writes its own
// halo, or its own faces, from interior cells). Six launches a hook had been 12 of a shock tube's 14
// launches a stage: a step of a 400-cell tube went from 160 to 57 us, of a walled 96 x 64 x 48 box by
// rk34 from 736 to 389 us, of the 256 x 128 x 64 layer with two walls from 3.68 to 3.52 ms. A wall begins on a workgroup's boundary, so a workgroup's wall is a scalar choice;
// within it the lanes run along the wall's first axis other than its own, i for the j and k walls, so
// their loads coalesce (lanes along k on a j wall had touched a line per lane).
#include "pga_internal.hpp"
#include "pga_trans.hpp"

namespace pga {

enum { WALL_SLP_ADIA = 0, WALL_SLP_ISOT = 1, WALL_NOSLP_ADIA = 2, WALL_NOSLP_ISOT = 3, WALL_MOV_ADIA = 4,
       WALL_MOV_ISOT = 5 };
enum { TRANS_NONE = -1 };

__host__ __device__ inline bool wall_isot(int kind) { return kind == WALL_SLP_ISOT || kind == WALL_NOSLP_ISOT || kind == WALL_MOV_ISOT; }
__host__ __device__ inline bool wall_stuck(int kind) { return kind >= WALL_NOSLP_ADIA; }

// one wall: n cells along its axis, n1 x n2 across it (n1 along the lanes), its first workgroup
struct WallTask {
  View S, xf, F;
  int axis, side, kind, n, n1, n2;
  unsigned first;
  double wall[3], Tw;
};

struct WallArgs {
  const double *K;
  View Q, st, tr, xcc;
  int ng, ntask;
  WallTask t[6];
};

// the wall of the thread's workgroup and the thread's number in it
__device__ __forceinline__ const WallTask &wall_of(const WallArgs &a, unsigned &r) {
  int n = 0;
  while (n + 1 < a.ntask && blockIdx.x >= a.t[n + 1].first) n++;
  r = (blockIdx.x - a.t[n].first) * 256 + threadIdx.x;
  return a.t[n];
}

__device__ __forceinline__ void wall_index(const WallArgs &a, const WallTask &t, int plane, int b1, int b2, int &i,
                                           int &j, int &k) {
  i = t.axis == 0 ? plane : a.ng + b1;
  j = t.axis == 1 ? plane : a.ng + (t.axis == 0 ? b1 : b2);
  k = t.axis == 2 ? plane : a.ng + b2;
}

// solution.mako:14-23 fromprims: a cell's Q and state from p, T, the velocity and the carried Y
template <int NS, int EOS, class YF>
__device__ __forceinline__ void fromprims_cell(const Gas<NS> &g, double p, double T, const double (&u)[3], const YF &Y,
                                               const View &Q, const View &st, int64_t o) {
#pragma clang fp contract(off)
  MixMom<NS, EOS> m;
  mixmom<NS, EOS>(g, Y, m);
  EosState s;
  frompT<NS, EOS>(g, m, Y, p, T, s);
  Q.at(o, 0) = s.rho;
  Q.at(o, 1) = s.rho * u[0];
  Q.at(o, 2) = s.rho * u[1];
  Q.at(o, 3) = s.rho * u[2];
  Q.at(o, 4) = s.rho * (s.e + 0.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]));
#pragma unroll
  for (int n = 0; n < NS - 1; n++) Q.at(o, 5 + n) = s.rho * Y(n);
  store_state<EOS>(st, o, s);
}

// The halo cell h planes out from the interior cell h planes in, a thread per halo cell. Each cell's
// reads come before its first store: a store the compiler cannot tell from the next load would make
// every row wait on memory of its own (a 96 x 64 wall took 12.4 us so, and six of them 75)
template <int NS, int EOS>
__global__ __launch_bounds__(256) void k_wall_mirror(WallArgs a) {
#pragma clang fp contract(off)
  constexpr int NE = NS + 4, NST = EOS == EOS_REAL ? 9 : 8;
  unsigned r;
  const WallTask &t = wall_of(a, r);
  const unsigned plane = (unsigned)t.n1 * (unsigned)t.n2, h = r / plane, rest = r - h * plane;
  if (h >= (unsigned)a.ng) return;
  const int b2 = (int)(rest / (unsigned)t.n1), b1 = (int)(rest - (unsigned)b2 * (unsigned)t.n1);
  const Gas<NS> g{a.K};
  int i, j, k;
  wall_index(a, t, t.side ? a.ng + t.n : a.ng, b1, b2, i, j, k);
  const int64_t of = t.S.off(i, j, k);
  // a block thinner than the halo reflects its last cell into every deeper layer
  // (launch/policy.py:168-184, MirrorOffset)
  const int hm = (int)h < t.n ? (int)h : t.n - 1;
  wall_index(a, t, t.side ? a.ng + t.n + (int)h : a.ng - 1 - (int)h, b1, b2, i, j, k);
  const int64_t oh = a.Q.off(i, j, k), sh = a.st.off(i, j, k);
  wall_index(a, t, t.side ? a.ng + t.n - 1 - hm : a.ng + hm, b1, b2, i, j, k);
  const int64_t om = a.Q.off(i, j, k), sm = a.st.off(i, j, k);
  const double Sx = t.S.at(of, 0), Sy = t.S.at(of, 1), Sz = t.S.at(of, 2);
  double q[NE], st[NST];
#pragma unroll
  for (int l = 0; l < NE; l++) q[l] = a.Q.at(om, l);
#pragma unroll
  for (int c = 0; c < NST; c++) st[c] = a.st.at(sm, c);
  const double Sinv = 1.0 / sqrt(Sx * Sx + Sy * Sy + Sz * Sz);
  const double nx = Sx * Sinv, ny = Sy * Sinv, nz = Sz * Sinv;
  if (wall_isot(t.kind)) {
    // an isothermal wall: the image's p and mass fractions at the wall's T, by the EOS
    const double rhoinv = 1.0 / q[0];
    double u[3];
    if (t.kind == WALL_SLP_ISOT) {
      const double uin = q[1] * rhoinv, vin = q[2] * rhoinv, win = q[3] * rhoinv;
      const double un = 2.0 * (uin * nx + vin * ny + win * nz);
      u[0] = uin - un * nx;
      u[1] = vin - un * ny;
      u[2] = win - un * nz;
    } else {
#pragma unroll
      for (int d = 0; d < 3; d++) u[d] = 2.0 * t.wall[d] - q[1 + d] * rhoinv;
    }
    double Y[NS > 1 ? NS - 1 : 1];
#pragma unroll
    for (int n = 0; n < NS - 1; n++) Y[n] = q[5 + n] * rhoinv;
    fromprims_cell<NS, EOS>(g, st[0], t.Tw, u, [&](int n) { return Y[n]; }, a.Q, a.st, oh);
    return;
  }
  if (t.kind == WALL_SLP_ADIA) {
    // the momentum's normal part, taken off twice; the whole state the image's (no EOS runs)
    const double mn = 2.0 * (q[1] * nx + q[2] * ny + q[3] * nz);
    q[1] -= mn * nx;
    q[2] -= mn * ny;
    q[3] -= mn * nz;
  } else {
    // stuckhalo: the velocity reflected about the wall's, the energy carrying the change in the
    // kinetic part, the state the image's
    const double rho = q[0], rhoinv = 1.0 / rho;
    double ke = 0.0, kehalo = 0.0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const double u = q[1 + d] * rhoinv, uh = 2.0 * t.wall[d] - u;
      q[1 + d] = rho * uh;
      ke += u * u;
      kehalo += uh * uh;
    }
    q[4] = q[4] + 0.5 * rho * (kehalo - ke);
  }
#pragma unroll
  for (int l = 0; l < NE; l++) a.Q.at(oh, l) = q[l];
#pragma unroll
  for (int c = 0; c < NST; c++) a.st.at(sh, c) = st[c];
}

// the wall's flux from the cell next to it: p_w = max(p + rho c u_n, 0), u_n toward the wall
// (wall.mako wallpressure); a viscous wall adds the stress of the two-point normal velocity gradient
// relative to the wall (every component where the flow is held, the normal one where it slips), the
// wall's work, and the heat flux from T_w (navstokes wall.mako wallfaceflux)
template <int NS, int EOS, int TRANS>
__global__ __launch_bounds__(256) void k_wall_flux(WallArgs a) {
#pragma clang fp contract(off)
  unsigned r;
  const WallTask &t = wall_of(a, r);
  const int b2 = (int)(r / (unsigned)t.n1), b1 = (int)(r - (unsigned)b2 * (unsigned)t.n1);
  if (b2 >= t.n2) return;
  int f[3], ic[3];
  wall_index(a, t, t.side ? a.ng + t.n : a.ng, b1, b2, f[0], f[1], f[2]);
  wall_index(a, t, t.side ? a.ng + t.n - 1 : a.ng, b1, b2, ic[0], ic[1], ic[2]);
  const double outward = t.side ? 1.0 : -1.0;
  const int64_t of = t.S.off(f[0], f[1], f[2]), oc = a.Q.off(ic[0], ic[1], ic[2]), osc = a.st.off(ic[0], ic[1], ic[2]);
  const double S3[3] = {t.S.at(of, 0), t.S.at(of, 1), t.S.at(of, 2)};
  const double q[4] = {a.Q.at(oc, 0), a.Q.at(oc, 1), a.Q.at(oc, 2), a.Q.at(oc, 3)};
  const double area = sqrt(S3[0] * S3[0] + S3[1] * S3[1] + S3[2] * S3[2]);
  const double un = outward * (q[1] * S3[0] + q[2] * S3[1] + q[3] * S3[2]) / (q[0] * area);
  const double pw = fmax(a.st.at(osc, 0) + q[0] * a.st.at(osc, 7) * un, 0.0);
  double F1 = pw * S3[0], F2 = pw * S3[1], F3 = pw * S3[2], F4 = 0.0;
  if constexpr (TRANS != TRANS_NONE) {
    const bool isot = wall_isot(t.kind);
    const double stuck = wall_stuck(t.kind) ? 1.0 : 0.0;
    double mu, kappa, dT;
    if (isot) {
      // wallcoeffs: the transport properties at the wall, the cell's composition at p and T_w
      const Gas<NS> g{a.K};
      const double rhoinv = 1.0 / q[0];
      double Y[NS], Ylast = 1.0;
#pragma unroll
      for (int n = 0; n < NS - 1; n++) {
        Y[n] = a.Q.at(oc, 5 + n) * rhoinv;
        Ylast -= a.Q.at(oc, 5 + n) * rhoinv;
      }
      Y[NS - 1] = fmax(Ylast, 0.0);
      MixMom<NS, EOS> m;
      mixmom<NS, EOS>(g, [&](int n) { return Y[n]; }, m);
      EosState thermo;
      frompT<NS, EOS>(g, m, [&](int n) { return Y[n]; }, a.st.at(osc, 0), t.Tw, thermo);
      double denom = 0.0;
#pragma unroll
      for (int n = 0; n < NS; n++) denom += Y[n] * g.MWinv(n);
      const double MWmix = 1.0 / denom;
      double X[NS];
#pragma unroll
      for (int n = 0; n < NS; n++) X[n] = Y[n] * g.MWinv(n) * MWmix;
      mu_kappa<NS, TRANS>(g, X, t.Tw, elog(t.Tw), thermo.rho, mu, kappa);
      dT = t.Tw - a.st.at(osc, 1);
    } else {
      const int64_t ot = a.tr.off(ic[0], ic[1], ic[2]);
      mu = a.tr.at(ot, 0);
      kappa = a.tr.at(ot, 1);
      dT = 0.0;
    }
    const int64_t ox = a.xcc.off(ic[0], ic[1], ic[2]), oxf = t.xf.off(f[0], f[1], f[2]);
    const double Sabs = sqrt(S3[0] * S3[0] + S3[1] * S3[1] + S3[2] * S3[2]), Sinv = 1.0 / Sabs;
    const double nv[3] = {S3[0] * Sinv, S3[1] * Sinv, S3[2] * Sinv};
    const double dn = fabs((a.xcc.at(ox, 0) - t.xf.at(oxf, 0)) * nv[0] + (a.xcc.at(ox, 1) - t.xf.at(oxf, 1)) * nv[1] +
                           (a.xcc.at(ox, 2) - t.xf.at(oxf, 2)) * nv[2]);
    const double rhoinv = 1.0 / q[0];
    double dun[3];
    for (int d = 0; d < 3; d++) dun[d] = outward * (t.wall[d] - q[1 + d] * rhoinv) / dn;
    const double div = dun[0] * nv[0] + dun[1] * nv[1] + dun[2] * nv[2];
    for (int d = 0; d < 3; d++) dun[d] = div * nv[d] + stuck * (dun[d] - div * nv[d]);
    double work = 0.0, tS[3];
    for (int d = 0; d < 3; d++) {
      tS[d] = -mu * Sabs * (dun[d] + div * nv[d] / 3.0);
      work += t.wall[d] * tS[d];
    }
    F1 += tS[0];
    F2 += tS[1];
    F3 += tS[2];
    F4 += work - kappa * outward * (dT) / dn * Sabs;
  }
  const int64_t off_ = t.F.off(f[0], f[1], f[2]);
  t.F.at(off_, 0) = 0.0;
  t.F.at(off_, 1) = F1;
  t.F.at(off_, 2) = F2;
  t.F.at(off_, 3) = F3;
  t.F.at(off_, 4) = F4;
  for (int l = 5; l < NS + 4; l++) t.F.at(off_, l) = 0.0;
}

// wall n's task: false (with the error set) for a wall the case does not have
static bool wall_task(const pga_case *c, int axis, int side, const pga_wall *w, const int32_t *ncell, WallTask &t,
                      const char *who) {
  if (axis < 0 || axis > 2 || side < 0 || side > 1) {
    set_error("%s: null case or ncell, an axis other than 0..2, a side other than 0 or 1, or ng < 1", who);
    return false;
  }
  t.axis = axis, t.side = side, t.n = ncell[axis];
  t.n1 = ncell[axis == 0 ? 1 : 0], t.n2 = ncell[axis == 2 ? 1 : 2];
  t.kind = w ? w->kind : WALL_SLP_ADIA;
  t.Tw = w ? w->T : 0.0;
  for (int d = 0; d < 3; d++) t.wall[d] = w && t.kind >= WALL_MOV_ADIA ? w->u[d] : 0.0;
  if (t.kind < WALL_SLP_ADIA || t.kind > WALL_MOV_ISOT) {
    set_error("%s: no wall kind %d (0 slp-adia, 1 slp-isot, 2 no-slp-adia, 3 no-slp-isot, 4 mov-adia, 5 mov-isot)",
              who, t.kind);
    return false;
  }
  if (wall_isot(t.kind) && !(t.Tw > 0.0)) {
    set_error("%s: an isothermal wall at T = %g", who, t.Tw);
    return false;
  }
  if (t.kind >= WALL_NOSLP_ADIA && c->desc.trans < 0) {
    set_error("%s: a wall that holds the flow needs a viscous case (an Euler case has slp-adia and slp-isot walls)", who);
    return false;
  }
  return true;
}

// the arguments common to both hooks; false (with the error set) for what neither takes
static bool wall_args(const pga_case *c, int nwall, const int32_t *axes, const int32_t *sides, const pga_wall *const *w,
                      const int32_t *ncell, int ng, WallArgs &a, const char *who) {
  if (!c || !ncell || ng < 1) {
    set_error("%s: null case or ncell, an axis other than 0..2, a side other than 0 or 1, or ng < 1", who);
    return false;
  }
  if (nwall < 0 || nwall > 6 || (nwall && (!axes || !sides || !w))) {
    set_error("%s: null walls, or other than 0 to 6 of them", who);
    return false;
  }
  for (int d = 0; d < 3; d++)
    if (ncell[d] < 1) {
      set_error("%s: a block of %d x %d x %d cells", who, ncell[0], ncell[1], ncell[2]);
      return false;
    }
  a.K = c->K;
  a.ng = ng, a.ntask = nwall;
  for (int n = 0; n < nwall; n++) {
    for (int m = 0; m < n; m++)
      if (axes[m] == axes[n] && sides[m] == sides[n]) {
        set_error("%s: walls %d and %d are the same face", who, m, n);
        return false;
      }
    if (!wall_task(c, axes[n], sides[n], w[n], ncell, a.t[n], who)) return false;
  }
  return true;
}

// the workgroups of `layers` cells deep walls, each wall on a workgroup's boundary; false when one
// wall's cells pass 32 bits
static bool wall_grid(WallArgs &a, int layers, dim3 &grid, const char *who) {
  int64_t blocks = 0;
  for (int n = 0; n < a.ntask; n++) {
    const int64_t cells = (int64_t)a.t[n].n1 * a.t[n].n2 * layers;
    a.t[n].first = (unsigned)blocks;
    blocks += (cells + 255) / 256;
    if (cells >= FLAT_MAX || blocks > 0x7fffffff) {
      set_error("%s: a wall of %d x %d cells", who, a.t[n].n1, a.t[n].n2);
      return false;
    }
  }
  grid = dim3((unsigned)blocks);
  return true;
}

static int32_t wall_mirrors(const char *who, const pga_case *c, int nwall, const int32_t *axes, const int32_t *sides,
                            const pga_wall *const *w, const int32_t *ncell, int ng, const pga_view &Q,
                            const pga_view &state, const pga_view *S, void *stream) {
  WallArgs a{};
  if (!wall_args(c, nwall, axes, sides, w, ncell, ng, a, who)) return PGA_EINVAL;
  if (!nwall) return PGA_OK;
  for (int n = 0; n < nwall; n++) {
    WallTask &t = a.t[n];
    // the halo slab ng deep and its mirror: the whole padded extent along the axis, the interior across
    pga_box cells{{ng, ng, ng}, {ncell[0], ncell[1], ncell[2]}};
    cells.start[t.axis] = 0;
    cells.extent[t.axis] = ncell[t.axis] + 2 * ng;
    pga_box faces{{ng, ng, ng}, {ncell[0], ncell[1], ncell[2]}};
    faces.start[t.axis] = t.side ? ng + ncell[t.axis] : ng;
    faces.extent[t.axis] = 1;
    PGA_REQUIRE(covers(Q, cells, c->desc.ns + 4) && covers(state, cells, nstate(c->desc)) && covers(S[n], faces, 3),
                "%s: the halo, its mirror or the wall faces reach outside Q, state or S", who);
    t.S = view(S[n]);
  }
  PGA_REQUIRE(Q.sj == state.sj && Q.sk == state.sk, "%s: Q and state must share their layout", who);
  a.Q = view(Q), a.st = view(state);
  dim3 grid;
  if (!wall_grid(a, ng, grid, who)) return PGA_ERANGE;
  const bool done = dispatch_eos(c->desc, [&]<int N, int E>() {
    hipLaunchKernelGGL((k_wall_mirror<N, E>), grid, dim3(256), 0, stream_of(stream), a);
  });
  if (!done) {
    set_error("%s: no kernel for %d species with eos %d", who, c->desc.ns, c->desc.eos);
    return PGA_EUNSUP;
  }
  return launched(who);
}

static int32_t wall_fluxes(const char *who, const pga_case *c, int nwall, const int32_t *axes, const int32_t *sides,
                           const pga_wall *const *w, const int32_t *ncell, int ng, const pga_view &Q,
                           const pga_view &state, const pga_view &trstate, const pga_view &xcc, const pga_view *xf,
                           const pga_view *S, const pga_view *F, void *stream) {
  WallArgs a{};
  if (!wall_args(c, nwall, axes, sides, w, ncell, ng, a, who)) return PGA_EINVAL;
  if (!nwall) return PGA_OK;
  const int ne = c->desc.ns + 4;
  const bool viscous = c->desc.trans >= 0 && trstate.data != nullptr;
  for (int n = 0; n < nwall; n++) {
    WallTask &t = a.t[n];
    pga_box cell{{ng, ng, ng}, {ncell[0], ncell[1], ncell[2]}};
    cell.start[t.axis] = t.side ? ng + ncell[t.axis] - 1 : ng;
    cell.extent[t.axis] = 1;
    pga_box faces = cell;
    faces.start[t.axis] = t.side ? ng + ncell[t.axis] : ng;
    PGA_REQUIRE(covers(Q, cell, ne) && covers(state, cell, nstate(c->desc)) && covers(S[n], faces, 3) &&
                    covers(F[n], faces, ne),
                "%s: the wall's cells or faces reach outside Q, state, S or F", who);
    if (viscous)
      PGA_REQUIRE(covers(trstate, cell, 2 + c->desc.ns) && covers(xcc, cell, 3) && covers(xf[n], faces, 3),
                  "%s: the wall's cells or faces reach outside trstate, xcc or xf", who);
    PGA_REQUIRE(viscous || t.kind <= WALL_SLP_ISOT, "%s: a wall that holds the flow needs trstate", who);
    t.S = view(S[n]), t.F = view(F[n]);
    if (viscous) t.xf = view(xf[n]);
  }
  a.Q = view(Q), a.st = view(state);
  if (viscous) a.tr = view(trstate), a.xcc = view(xcc);
  dim3 grid;
  if (!wall_grid(a, 1, grid, who)) return PGA_ERANGE;
  const int trans = viscous ? c->desc.trans : TRANS_NONE;
  const bool done = dispatch_eos(c->desc, [&]<int N, int E>() {
    if (trans == TRANS_NONE)
      hipLaunchKernelGGL((k_wall_flux<N, E, TRANS_NONE>), grid, dim3(256), 0, stream_of(stream), a);
    else if (trans == TRANS_CONSTANT)
      hipLaunchKernelGGL((k_wall_flux<N, E, TRANS_CONSTANT>), grid, dim3(256), 0, stream_of(stream), a);
    else if (trans == TRANS_KINETIC)
      hipLaunchKernelGGL((k_wall_flux<N, E, TRANS_KINETIC>), grid, dim3(256), 0, stream_of(stream), a);
    else if constexpr (E == EOS_REAL)
      hipLaunchKernelGGL((k_wall_flux<N, E, TRANS_CHUNG>), grid, dim3(256), 0, stream_of(stream), a);
  });
  if (!done) {
    set_error("%s: no kernel for %d species with eos %d", who, c->desc.ns, c->desc.eos);
    return PGA_EUNSUP;
  }
  return launched(who);
}

}  // namespace pga

using namespace pga;

extern "C" int32_t pga_wall_mirror(const pga_case *c, int32_t axis, int32_t side, const pga_wall *w,
                                   const int32_t *ncell, int32_t ng, pga_view Q, pga_view state, pga_view S,
                                   void *stream) {
  return wall_mirrors("pga_wall_mirror", c, 1, &axis, &side, &w, ncell, ng, Q, state, &S, stream);
}

extern "C" int32_t pga_wall_flux(const pga_case *c, int32_t axis, int32_t side, const pga_wall *w,
                                 const int32_t *ncell, int32_t ng, pga_view Q, pga_view state, pga_view trstate,
                                 pga_view xcc, pga_view xf, pga_view S, pga_view F, void *stream) {
  return wall_fluxes("pga_wall_flux", c, 1, &axis, &side, &w, ncell, ng, Q, state, trstate, xcc, &xf, &S, &F, stream);
}

// the walls' pointers of a contiguous array (null: every wall an adiabatic slip wall)
static void wall_pointers(int32_t nwall, const pga_wall *walls, const pga_wall *(&w)[6]) {
  for (int n = 0; n < 6; n++) w[n] = walls && n < nwall ? walls + n : nullptr;
}

extern "C" int32_t pga_wall_mirrors(const pga_case *c, int32_t nwall, const int32_t *axes, const int32_t *sides,
                                    const pga_wall *walls, const int32_t *ncell, int32_t ng, pga_view Q,
                                    pga_view state, const pga_view *S, void *stream) {
  if (nwall > 0 && !S) {
    set_error("pga_wall_mirrors: null S");
    return PGA_EINVAL;
  }
  const pga_wall *w[6];
  wall_pointers(nwall, walls, w);
  return wall_mirrors("pga_wall_mirrors", c, nwall, axes, sides, w, ncell, ng, Q, state, S, stream);
}

extern "C" int32_t pga_wall_fluxes(const pga_case *c, int32_t nwall, const int32_t *axes, const int32_t *sides,
                                   const pga_wall *walls, const int32_t *ncell, int32_t ng, pga_view Q, pga_view state,
                                   pga_view trstate, pga_view xcc, const pga_view *xf, const pga_view *S,
                                   const pga_view *F, void *stream) {
  if (nwall > 0 && (!S || !F || (c && c->desc.trans >= 0 && trstate.data && !xf))) {
    set_error("pga_wall_fluxes: null S, F or (viscous) xf");
    return PGA_EINVAL;
  }
  const pga_wall *w[6];
  wall_pointers(nwall, walls, w);
  return wall_fluxes("pga_wall_fluxes", c, nwall, axes, sides, w, ncell, ng, Q, state, trstate, xcc, xf, S, F, stream);
}
