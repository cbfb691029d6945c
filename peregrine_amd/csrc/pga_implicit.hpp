// Implicit chemistry (device code, shared by pga_implicit.hip and the launches over a table of
// blocks in pga_batch.hip): each cell integrates its own finite-rate chemistry over the step by the
// linearly implicit (Rosenbrock) Euler method in `parts` equal parts, the same 0D system the
// sub-stepped form integrates explicitly (chemint/kernels/substep.mako:5-83: the ns mass fractions
// and T at constant density and internal energy, dT/dt = -sum e_n w_n / (rho cv)), and begins dQ
// with the mean rate over the step.
//
// A part of length h from y0 = (Y_0 .. Y_{ns-1}, T) takes y1 = y0 + h x with (I - h J) x = f(y0):
// backward Euler's first Newton step, first order and stable however stiff the chemistry. J is
// formed in FP64 by forward differences of f (one more evaluation of the rates per unknown); the
// matrix is kept in FP64 and, rounded to FP32, factored in registers. The
// solve is an iterative refinement: x += (LU)^-1 r with the residual r = f - A x taken in FP64
// against the FP64 matrix, until every row's residual is within `tolerance` of that row's scale
// (|f_i| + sum_j |A_ij x_j|, the componentwise backward error), so x is the FP64 solution whatever
// the factors' rounding. The Arrhenius exponentials, the Gibbs polynomials, the residuals and the
// update stay FP64. No pivoting: the matrices are I - h J of a chemical source, whose diagonal grows with
// the destruction rates; the FP64 refinement corrects what the FP32 factors leave.
//
// The batched LU of caller-given systems takes 16 matrices per wave, padded to 12 x 12 (three 4 x 4 blocks a
// side), one lane quad per matrix: lane 4b + q holds column q of each of matrix b's blocks, a block's row i
// in its register i. That is the accumulator layout of v_mfma_f32_4x4x1f32 (16 independent 4 x 4
// products per instruction), so the Schur-complement updates of the blocked right-looking LU,
// A_IJ -= L_IK U_KJ, are four rank-one MFMAs each for all 16 matrices at once; the diagonal blocks'
// factorisation and the two triangular block solves run on the VALU within the quad, with DPP
// broadcasts.
//
// The implicit form's work array holds the FP64 matrices, [group of 16 cells][(ns + 1)^2 entries]
// [16 cells] (a row of the 16 cells' same entry is 128 contiguous bytes, so the lane-per-cell
// kernels move whole segments), then y, f at y's FP32 rounding and f at y, [ns + 1][cells] doubles each, then
// the caches of a mechanism too large for LDS (im_cache_work).
// The FP32 factors never leave the registers of the solve. The batched solve of caller-given systems
// keeps its FP32 factors in a work array the same way, [group][144 entries][16 cells].
#pragma once

#include <type_traits>

#include "generated/mechanisms.hpp"
#include "pga_chem.hpp"
#include "pga_internal.hpp"

namespace pga {

constexpr int IM_G = 16;                   // matrices per MFMA group: a wave's 16 lane quads
constexpr int IM_N = 12;                   // matrices padded to 12 x 12
constexpr int IM_E = IM_N * IM_N;          // entries of a padded matrix
constexpr int IM_GROUP = IM_E * IM_G;      // floats per group
constexpr int IM_FAIL = 1000;              // added to a cell's count for each part that did not converge

typedef float v4f __attribute__((ext_vector_type(4)));

// entry (r, c) of matrix `cell` in the group-major factor array
__device__ __forceinline__ int64_t lu_at(int64_t cell, int r, int c) {
  return (cell >> 4) * IM_GROUP + (int64_t)(r * IM_N + c) * IM_G + (cell & 15);
}

template <int B, int E, class F>
__host__ __device__ __forceinline__ void sfor(F &&f) {
  if constexpr (B < E) {
    f.template operator()<B>();
    sfor<B + 1, E>(f);
  }
}

// lane P's x within each quad, to all four lanes of the quad (DPP quad_perm P, P, P, P)
template <int P>
__device__ __forceinline__ float qb(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), P * 0x55, 0xf, 0xf, false));
}

// The blocked LU of one lane quad's matrix per quad, 16 per wave, in registers: lane q holds column q
// of each 4 x 4 block, block (I, J)'s row i in blk[I][J][i]. Every lane of the wave takes part (the
// MFMAs need every lane).
template <int NB>
__device__ __forceinline__ void lu_factor(v4f (&blk)[NB][NB], int q) {
  sfor<0, NB>([&]<int K>() {
    v4f &D = blk[K][K];
    // the diagonal block: lane q holds its column q; L (unit, strictly below) and U overwrite it
    sfor<0, 4>([&]<int p>() {
      const float rp = 1.0f / qb<p>(D[p]);
      sfor<p + 1, 4>([&]<int i>() {
        const float li = qb<p>(D[i]) * rp;
        D[i] = q > p ? D[i] - li * D[p] : (q == p ? li : D[i]);
      });
    });
    // L_KK[i][p], broadcast to the quad
    float Lkk[4][4];
    sfor<0, 4>([&]<int p>() { sfor<p + 1, 4>([&]<int i>() { Lkk[i][p] = qb<p>(D[i]); }); });
    // U_KJ = L_KK^-1 A_KJ right of the diagonal, column by column in each lane
    sfor<K + 1, NB>([&]<int J>() {
      v4f &X = blk[K][J];
      sfor<0, 3>([&]<int p>() { sfor<p + 1, 4>([&]<int i>() { X[i] = X[i] - Lkk[i][p] * X[p]; }); });
    });
    // L_IK = A_IK U_KK^-1 below it, row by row across the quad; aL[I][p] is the MFMA operand of
    // column p, lane 4b + i holding -L_IK[i][p]
    const float ud = q == 0 ? D[0] : q == 1 ? D[1] : q == 2 ? D[2] : D[3];
    const float rud = 1.0f / ud;
    float aL[NB][4];
    sfor<K + 1, NB>([&]<int I>() {
      v4f &X = blk[I][K];
      sfor<0, 4>([&]<int p>() { aL[I][p] = 0.0f; });
      sfor<0, 4>([&]<int i>() {
        sfor<0, 4>([&]<int p>() {
          const float xp = qb<p>(X[i] * rud);
          X[i] = q > p ? X[i] - xp * D[p] : (q == p ? xp : X[i]);
          aL[I][p] = q == i ? -xp : aL[I][p];
        });
      });
    });
    // the Schur complement on the matrix cores: A_IJ += sum_p (-L_IK[:, p]) U_KJ[p, :]
    sfor<K + 1, NB>([&]<int I>() {
      sfor<K + 1, NB>([&]<int J>() {
        sfor<0, 4>([&]<int p>() {
          blk[I][J] = __builtin_amdgcn_mfma_f32_4x4x1f32(aL[I][p], blk[K][J][p], blk[I][J], 0, 0, 0);
        });
      });
    });
  });
}

// The batched LU of 16 matrices per wave, in place in the group-major array W. A wave exits
// whole; the lanes of a group's missing matrices factor the identity.
template <int NB>
__global__ __launch_bounds__(256) void k_lu(float *__restrict__ W, int64_t ncell) {
  const int64_t grp = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (grp * IM_G >= ncell) return;
  const int lane = threadIdx.x & 63, b = lane >> 2, q = lane & 3;
  const bool real = grp * IM_G + b < ncell;
  float *base = W + grp * IM_GROUP + b;
  v4f blk[NB][NB];
  sfor<0, NB>([&]<int I>() {
    sfor<0, NB>([&]<int J>() {
      sfor<0, 4>([&]<int i>() {
        const int r = 4 * I + i, c = 4 * J + q;
        blk[I][J][i] = real ? base[(r * IM_N + c) * IM_G] : (r == c ? 1.0f : 0.0f);
      });
    });
  });
  lu_factor<NB>(blk, q);
  if (!real) return;
  sfor<0, NB>([&]<int I>() {
    sfor<0, NB>([&]<int J>() {
      sfor<0, 4>([&]<int i>() { base[((4 * I + i) * IM_N + 4 * J + q) * IM_G] = blk[I][J][i]; });
    });
  });
}

// x = (L U)^-1 z in FP32 from the factors of matrix `cell`, in place (L unit lower)
template <int NV>
__device__ __forceinline__ void lu_solve(const float *__restrict__ W, int64_t cell, float (&z)[NV]) {
#pragma unroll
  for (int r = 1; r < NV; r++) {
#pragma unroll
    for (int c = 0; c < r; c++) z[r] -= W[lu_at(cell, r, c)] * z[c];
  }
#pragma unroll
  for (int r = NV - 1; r >= 0; r--) {
#pragma unroll
    for (int c = r + 1; c < NV; c++) z[r] -= W[lu_at(cell, r, c)] * z[c];
    z[r] = z[r] / W[lu_at(cell, r, r)];
  }
}

struct ImArgs {
  const double *K, *C;
  View Q, st, out;
  int begin_dQ, first, last;
  double *A;     // the FP64 matrices, group-major with nv^2 entries
  double *y;     // [ns + 1][ncell] three times: the part's start (then its end), f at its FP32 rounding, f at it
  double *tc;    // [im_cache_work][ncell]: the caches of a mechanism whose workgroups' caches pass LDS
  int64_t ncell;
  int32_t *sweeps;
  const double *dt;
  Box3 b;
  int parts, maxsweeps;
  double tol;
};

// entry (r, c) of FP64 matrix `cell` with nv unknowns
template <int NV>
__device__ __forceinline__ int64_t a64_at(int64_t cell, int r, int c) {
  return (cell >> 4) * (NV * NV * IM_G) + (int64_t)(r * NV + c) * IM_G + (cell & 15);
}

// f(y) of the 0D reactor at constant density: the species' rates over rho and dT/dt at constant
// volume, as the sub-stepped form takes them (substep.mako:14-50: ln T from the rate state, cv and
// each species' internal energy by their ln T polynomials)
template <class M>
__device__ __forceinline__ void rhs0d(const Gas<M::NS> &g, const double *__restrict__ C, double rho, double rhoinv,
                                      const double (&y)[M::NS + 1], double (&f)[M::NS + 1]) {
#pragma clang fp contract(off)
  constexpr int NS = M::NS;
  double Y[NS], rate[NS], D[NS];
#pragma unroll
  for (int n = 0; n < NS; n++) Y[n] = y[n];
  const double T = y[NS];
  typename M::Rates s;
  M::ratestate(g, constants(C), rho, Y, T, s);
  M::template fold<false>(constants(C), s, rate, D);
  double cv = 0.0, dTdt = 0.0;
#pragma unroll
  for (int n = 0; n < NS; n++) {
    const double cpR = cpR_species(g, n, s.logT);
    const double e = e_species(g, n, T, s.logT, s.Tinv);
    cv += (cpR - 1.0) * g.Rsp(n) * Y[n];
    dTdt -= e * rate[n];
  }
  const double cvrhoinv = 1.0 / (cv * rho);
#pragma unroll
  for (int n = 0; n < NS; n++) f[n] = rate[n] * rhoinv;
  f[NS] = dTdt * cvrhoinv;
}

// What f(y) shares over every composition at one T: the rates' T-only values (M::TCache: ln T, 1/T,
// the Gibbs terms and their exponentials, each reaction's cached rate constant, ln k or Troe fit) and
// each species' cv share (cp/R - 1) R_n and internal energy e_n. A forward-difference column of a
// species changes the composition at the same T, so it takes f from this and the composition alone;
// every value is the expression rhs0d evaluates, so the column keeps rhs0d's bits.
template <class M>
struct ImCache {
  typename M::TCache t;
  double ea[M::NS], ee[M::NS];
};

template <class M>
constexpr int im_cache_n = sizeof(ImCache<M>) / sizeof(double);

__device__ __forceinline__ int64_t im_code(const Box3 &b, int i, int j, int k) {
  return (i - b.s0) + (int64_t)b.e0 * ((j - b.s1) + (int64_t)b.e1 * (k - b.s2));
}

// the step of unknown m's forward difference: 2^-14 of T or of a mass fraction, at least 2^-14 * 1e-3
// for a trace species. Far above the square root of the rounding unit on purpose: the rates'
// rounding divided by the step is what the difference adds of its own, and a step of 2^-26 would
// turn a last-bit change of y into a 1e-6 change of a stiff part's result and mass drift through
// the columns' sums; the step's truncation is smooth in y, and the linearly implicit Euler step
// is first order with any fixed matrix. The step taken is the difference the rounding leaves
__device__ __forceinline__ double fd_step(double ym, bool temperature) {
#pragma clang fp contract(off)
  const double scale = temperature ? ym : fmax(fabs(ym), 1e-3);
  return (ym + 6.103515625e-05 * scale) - ym;
}

// x = A^-1 b by iterative refinement on the FP32 factors W (the batched solve of caller-given
// systems), the residual b - A x in FP64 against A (entry (r, c) at A[at(r, c)]); a lane per system;
// stops when every row's residual is within tol of its scale
// |b_r| + sum_c |A_rc x_c|, or after maxsweeps corrections. Returns the corrections taken, or
// maxsweeps + 1 when the last one left a row outside the tolerance
template <int NV, class At>
__device__ __forceinline__ int refine(const float *__restrict__ W, const double *__restrict__ A, At at, int64_t cell,
                                      const double (&bv)[NV], double (&x)[NV], int maxsweeps, double tol) {
#pragma clang fp contract(off)
  double r[NV];
#pragma unroll
  for (int m = 0; m < NV; m++) {
    x[m] = 0.0;
    r[m] = bv[m];
  }
  int s = 0;
  bool done = false;
#pragma unroll 1
  while (s < maxsweeps && !done) {
    const float *Ws = opaque(W);
    const double *As = opaque(A);
    float z[NV];
#pragma unroll
    for (int m = 0; m < NV; m++) z[m] = (float)r[m];
    lu_solve<NV>(Ws, cell, z);
#pragma unroll
    for (int m = 0; m < NV; m++) x[m] += (double)z[m];
    done = true;
#pragma unroll
    for (int m = 0; m < NV; m++) {
      double acc = bv[m], scale = fabs(bv[m]);
#pragma unroll
      for (int c = 0; c < NV; c++) {
        const double ax = As[at(cell, m, c)] * x[c];
        acc = acc - ax;
        scale = scale + fabs(ax);
      }
      r[m] = acc;
      done = done && fabs(acc) <= tol * scale;
    }
    s++;
  }
  return done ? s : maxsweeps + 1;
}

// A = I - h J at the part's start, J by forward differences, in two launches: the species columns, with y
// and f(y^) (y^: y rounded to FP32), and then the T column and f(y), the solve's right-hand side, a whole
// evaluation each. J is taken at y^: a last-bit change of y (the oracle's FP64 solve against the device's
// refined one, a part's start after another part) then leaves the matrix as it was, where the differences'
// own rounding would move it by 1e-12 of itself and a stiff part's result by more; the linearly implicit
// Euler step is first order with the matrix of any nearby state.
//
// The species columns: 64 cells a workgroup, a wave a group of M::COLS species. The waves make the cache of
// y^'s T between them into LDS (a share each, M::tstate_part), then each takes f at y^ and at its group's
// columns from it, evaluating a reaction again only for the columns whose species it reads
// (M::fold_columns; each column's sums its own, in order). A lane a column, with the cache in HBM, read its
// 68 values for every column and was bound by that; three columns a lane reading it from L2 waited on each
// value in turn (280 us against 191 for 64^3 cells), and from LDS, where the cache never leaves the chip, the
// two launches take 97 + 69 us for the 64^3 cells in place of 260, at three waves a SIMD. The 64^3 step went
// from 1.45 to 1.16 ms, that of 16 boxes of 3.0 million cells in all from 16.9 to 13.0 ms.

// A workgroup's caches pass gfx950's 160 KB of LDS from 321 values a cell on, some 280 reactions of nine
// species: such a mechanism's go through the work array, the same code and values.

constexpr int IM_CELLS = 64;  // cells of a workgroup of the species columns
constexpr size_t IM_LDS = 163840;

// the doubles of the work array a cell's cache takes, and the LDS of a workgroup's
template <class M>
constexpr int im_cache_work = sizeof(double) * im_cache_n<M> * IM_CELLS > IM_LDS ? im_cache_n<M> : 0;
template <class M>
constexpr size_t im_cols_lds = im_cache_work<M> ? 0 : sizeof(double) * im_cache_n<M> * IM_CELLS;

// im_cache_work of the library's mechanism of that number
inline int im_cache_work_of(int mechanism) {
  int n = 0;
#define X(NAME, IDX) \
  if (mechanism == IDX) n = im_cache_work<Mech_##NAME>;
  PGA_MECHANISMS(X)
#undef X
  return n;
}

// lets a kernel of the columns be launched with its LDS where that passes the 64 KB any launch may ask for
template <class M>
inline int32_t im_room(const void *kernel, const char *who) {
  if constexpr (im_cols_lds<M> > 65536) {
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)im_cols_lds<M>);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      set_error("%s: %d bytes of LDS a workgroup: %s", who, (int)im_cols_lds<M>, hipGetErrorString(e));
      return PGA_EHIP;
    }
  }
  return PGA_OK;
}

// the y of a cell at the part's start: the first part's from Q and the state, a later one's as the last part
// left it (selected rather than branched, one copy of the code)
template <class M>
__device__ __forceinline__ void im_y0(const ImArgs &a, const View &Q, const View &st, int64_t o, int64_t ost,
                                      double rhoinv, int64_t code, double (&y0)[M::NS + 1]) {
  constexpr int NS = M::NS;
  double Y[NS];
  massfrac<NS>(Q, o, rhoinv, Y);
#pragma unroll
  for (int n = 0; n < NS; n++) y0[n] = a.first ? Y[n] : a.y[n * a.ncell + code];
  y0[NS] = a.first ? st.at(ost, 1) : a.y[NS * a.ncell + code];
}

// a wave's view of the constants and of its lane's place in the cache, as values the compiler cannot match
// with another group's: it would read what the groups share ahead of the branch that tells them apart, and
// hold it in registers
template <bool WORK>
struct ImGroup {
  Constants K, C;
  double *lds;
  unsigned lane;
  __device__ __forceinline__ ImGroup(const ImArgs &a, double *l, int64_t) : K(constants(a.K)), C(constants(a.C)), lds(l) {
    lane = threadIdx.x % IM_CELLS;
    asm volatile("" : "+s"(K), "+s"(C), "+v"(lane));
  }
  // entry e of the lane's cell
  __device__ __forceinline__ double &operator()(int e) const { return lds[e * IM_CELLS + lane]; }
};

// the same of a cache in the work array
template <>
struct ImGroup<true> {
  Constants K, C;
  double *tc;
  int64_t nc;
  __device__ __forceinline__ ImGroup(const ImArgs &a, double *, int64_t code)
      : K(constants(a.K)), C(constants(a.C)), tc(a.tc + code), nc(a.ncell) {
    asm volatile("" : "+s"(K), "+s"(C), "+v"(tc));
  }
  __device__ __forceinline__ double &operator()(int e) const { return tc[e * nc]; }
};

// ends a group's branch: without it the stores that end every branch are made one store where they join,
// with every value waiting in registers
__device__ __forceinline__ void im_branch_end() { asm volatile(""); }

// group G's share of a cell's cache at T
template <class M, int G>
__device__ __forceinline__ void ijac_part(const ImArgs &a, double T, double *lds, int64_t code) {
#pragma clang fp contract(off)
  constexpr int NS = M::NS, NT = sizeof(typename M::TCache) / sizeof(double);
  const ImGroup<(im_cache_work<M> > 0)> X(a, lds, code);
  const Gas<NS> g{X.K};
  const auto put = [&](int e, double v) { X(e) = v; };
  M::template tstate_part<G>(g, X.C, T, put);
  const double logT = tlog(T), Tinv = 1.0 / T;
#pragma unroll
  for (int n = G; n < NS; n += M::GROUPS) {
    const double cpR = cpR_species(g, n, logT);
    put(NT + n, (cpR - 1.0) * g.Rsp(n));
    put(NT + NS + n, e_species(g, n, T, logT, Tinv));
  }
  im_branch_end();
}

// group G's species columns of a cell
template <class M, int G>
__device__ __forceinline__ void ijac_group(const ImArgs &a, double rho, double rhoinv, const double (&Y)[M::NS],
                                           double *lds, int64_t code) {
#pragma clang fp contract(off)
  constexpr int NS = M::NS, NV = NS + 1, NT = sizeof(typename M::TCache) / sizeof(double);
  constexpr int m0 = G * M::COLS, nm = NS - m0 < M::COLS ? NS - m0 : M::COLS;
  const ImGroup<(im_cache_work<M> > 0)> X(a, lds, code);
  double Yp[M::COLS] = {}, hd[M::COLS] = {}, omega[M::COLS + 1][NS];
  const double h = *a.dt / a.parts;
#pragma unroll
  for (int c = 0; c < nm; c++) {
    const double dlt = fd_step(Y[m0 + c], false);
    Yp[c] = Y[m0 + c] + dlt;
    hd[c] = h / dlt;
  }
  M::template fold_columns<G>(X.K, X.C, rho, Y, Yp, X, omega);
  // dT/dt of a composition from its rates, rhs0d's sums
  const auto dTdt = [&](int v) {
    double cv = 0.0, d = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) {
      cv += X(NT + n) * (v && n == m0 + v - 1 ? Yp[v - 1] : Y[n]);
      d -= X(NT + NS + n) * omega[v][n];
    }
    return d * (1.0 / (cv * rho));
  };
  double f0[NV];
#pragma unroll
  for (int r = 0; r < NS; r++) f0[r] = omega[0][r] * rhoinv;
  f0[NS] = dTdt(0);
  if constexpr (G == 0) {
    double *fh = a.y + NV * a.ncell + code;
#pragma unroll
    for (int r = 0; r < NV; r++) fh[r * a.ncell] = f0[r];
  }
#pragma unroll
  for (int c = 0; c < nm; c++) {
    const int m = m0 + c;
#pragma unroll
    for (int r = 0; r < NS; r++)
      a.A[a64_at<NV>(code, r, m)] = (r == m ? 1.0 : 0.0) - (omega[c + 1][r] * rhoinv - f0[r]) * hd[c];
    a.A[a64_at<NV>(code, NS, m)] = 0.0 - (dTdt(c + 1) - f0[NS]) * hd[c];
  }
}

// f<G>() for the wave's group, the last for any other wave; each ends its caller's path, as branches that
// joined again would hold more
template <int GROUPS, class F>
__device__ __forceinline__ void im_group(int wave, F &&f) {
  static_assert(GROUPS >= 1 && GROUPS <= 4);
  if constexpr (GROUPS > 1)
    if (wave == 0) return f.template operator()<0>();
  if constexpr (GROUPS > 2)
    if (wave == 1) return f.template operator()<1>();
  if constexpr (GROUPS > 3)
    if (wave == 2) return f.template operator()<2>();
  if (wave == GROUPS - 1) return f.template operator()<GROUPS - 1>();
}

// a workgroup's species columns: lds im_cols_lds<M> bytes, the lane's cell (i, j, k) at work place code. A lane
// past the cells takes the last one again, the same values to the same places: a branch around the stores
// would cut the columns' one block in two, which the compiler then fills 512 registers between
template <class M>
__device__ __forceinline__ void ijac_columns(const ImArgs &a, const View &Q, const View &st, double *lds, int i, int j,
                                             int k, int64_t code) {
#pragma clang fp contract(off)
  constexpr int NS = M::NS, NV = NS + 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / IM_CELLS);
  const int64_t o = Q.off(i, j, k);
  const double rho = Q.at(o, 0), rhoinv = 1.0 / rho;
  double y0[NV], Y[NS];
  im_y0<M>(a, Q, st, o, st.off(i, j, k), rhoinv, code, y0);
  if (wave == 0 && a.first) {
#pragma unroll
    for (int r = 0; r < NV; r++) a.y[r * a.ncell + code] = y0[r];
  }
  const double T = (double)(float)y0[NS];
  im_group<M::GROUPS>(wave, [&]<int G>() { ijac_part<M, G>(a, T, lds, code); });
  __syncthreads();
#pragma unroll
  for (int n = 0; n < NS; n++) Y[n] = (double)(float)y0[n];
  im_group<M::GROUPS>(wave, [&]<int G>() { ijac_group<M, G>(a, rho, rhoinv, Y, lds, code); });
}

// slice 0: the T column of A by a whole evaluation; slice 1: f(y)
template <class M>
__device__ __forceinline__ void ijac_whole(const ImArgs &a, const View &Q, int i, int j, int k, int64_t code,
                                           int slice) {
#pragma clang fp contract(off)
  constexpr int NS = M::NS, NV = NS + 1;
  const int64_t nc = a.ncell;
  const double rho = Q.at(Q.off(i, j, k), 0), rhoinv = 1.0 / rho;
  const double *y = a.y + code, *fh = a.y + NV * nc + code;
  double yp[NV], f1[NV];
#pragma unroll
  for (int r = 0; r < NV; r++) {
    const double yr = y[r * nc];
    yp[r] = slice == 0 ? (double)(float)yr : yr;
  }
  const double dlt = fd_step(yp[NS], true);
  yp[NS] = slice == 0 ? yp[NS] + dlt : yp[NS];
  rhs0d<M>(Gas<NS>{a.K}, a.C, rho, rhoinv, yp, f1);
  if (slice == 1) {
    double *bv = a.y + 2 * NV * nc + code;
#pragma unroll
    for (int r = 0; r < NV; r++) bv[r * nc] = f1[r];
    return;
  }
  const double hd = *a.dt / a.parts / dlt;
#pragma unroll
  for (int r = 0; r < NV; r++) a.A[a64_at<NV>(code, r, NS)] = (r == NS ? 1.0 : 0.0) - (f1[r] - fh[r * nc]) * hd;
}

// The part's solve and step, a lane per cell: (I - h J) x = f(y) by iterative refinement, then y += h x. The
// lane loads its FP64 matrix once and keeps it, and the FP32 factors of its rounding, in registers, at one
// wave a SIMD; each sweep solves L U z = r in FP32, adds z to x and takes r = f - A x in FP64 with the row
// scales |f_m| + sum_c |A_mc x_c|. A cell stops when every row's residual is within tol of its scale, or
// after maxsweeps. A cell's x depends only on its own matrix and f, whichever cells share its wave.
//
// A quad of lanes per cell, with the matrix cores' rank-one updates between the quads' broadcasts, took 2150
// vector instructions for 16 cells where this takes some 2500 for 64, each triangular solve a chain four lanes
// share: 106 us for 64^3 cells, 60 here, 3.6 TB/s of the matrices' and vectors' bytes (the same factors, sums
// and x to the bit). The 381 registers a lane holds leave one wave a SIMD; read again each sweep instead, the
// matrices would be three passes over HBM.
//
// The sums go column c into the (c mod 4)-th of four partial sums, then ((0) + (1)) + ((2) + (3)).
//
// The last part's end, the mean rate over the step, rho (Y_end - Y_start) / dt, goes from the lane's x into
// out as the sub-stepped form begins dQ (or into the rates): a launch of its own read y and Q again, 11 us
// for 64^3 cells.
template <int NV>
__device__ __forceinline__ void lu_refine_cell(const ImArgs &a, const View &Q, const View &out, int i, int j, int k,
                                               int64_t cell) {
#pragma clang fp contract(off)
  constexpr int NS = NV - 1;
  const int64_t nc = a.ncell;
  const double *A = a.A + a64_at<NV>(cell, 0, 0), *bvp = a.y + 2 * NV * nc + cell;
  double Ad[NV][NV], bv[NV], x[NV], r[NV];
  sfor<0, NV>([&]<int m>() { sfor<0, NV>([&]<int c>() { Ad[m][c] = A[(m * NV + c) * IM_G]; }); });
  sfor<0, NV>([&]<int m>() { bv[m] = bvp[m * nc]; });
  // no pivoting: L unit below the diagonal, U on and above it, in place
  float W[NV][NV], rdiag[NV];
  sfor<0, NV>([&]<int m>() { sfor<0, NV>([&]<int c>() { W[m][c] = (float)Ad[m][c]; }); });
  sfor<0, NV>([&]<int p>() {
    rdiag[p] = 1.0f / W[p][p];
    sfor<p + 1, NV>([&]<int m>() {
      W[m][p] = W[m][p] * rdiag[p];
      sfor<p + 1, NV>([&]<int c>() { W[m][c] = fmaf(-W[m][p], W[p][c], W[m][c]); });
    });
  });
  sfor<0, NV>([&]<int m>() {
    x[m] = 0.0;
    r[m] = bv[m];
  });
  int count = a.maxsweeps + IM_FAIL;
#pragma unroll 1
  for (int s = 1; s <= a.maxsweeps; s++) {
    float z[NV];
    sfor<0, NV>([&]<int m>() {
      z[m] = (float)r[m];
      sfor<0, m>([&]<int c>() { z[m] -= W[m][c] * z[c]; });
    });
    sfor<0, NV>([&]<int n>() {
      constexpr int m = NV - 1 - n;
      sfor<m + 1, NV>([&]<int c>() { z[m] -= W[m][c] * z[c]; });
      z[m] = z[m] * rdiag[m];
    });
    sfor<0, NV>([&]<int m>() { x[m] = x[m] + (double)z[m]; });
    int ok = 1;
    sfor<0, NV>([&]<int m>() {
      double p[4] = {0.0, 0.0, 0.0, 0.0}, sc[4] = {0.0, 0.0, 0.0, 0.0};
      sfor<0, NV>([&]<int c>() {
        const double ax = Ad[m][c] * x[c];
        p[c % 4] = p[c % 4] + ax;
        sc[c % 4] = sc[c % 4] + fabs(ax);
      });
      r[m] = bv[m] - ((p[0] + p[1]) + (p[2] + p[3]));
      const double scale = fabs(bv[m]) + ((sc[0] + sc[1]) + (sc[2] + sc[3]));
      ok = ok & (fabs(r[m]) <= a.tol * scale ? 1 : 0);
    });
    if (ok) {
      count = s;
      break;
    }
  }
  a.sweeps[cell] = a.first ? count : a.sweeps[cell] + count;
  const double h = *a.dt / a.parts;
  sfor<0, NV>([&]<int m>() { x[m] = a.y[m * nc + cell] + h * x[m]; });
  if (!a.last) {
    sfor<0, NV>([&]<int m>() { a.y[m * nc + cell] = x[m]; });
    return;
  }
  const int64_t o = Q.off(i, j, k), oo = out.off(i, j, k);
  const double rho = Q.at(o, 0), rhoinv = 1.0 / rho;
  double Ys[NS];
  massfrac<NS>(Q, o, rhoinv, Ys);
  const double rdt = rho / *a.dt;
  const int row = a.begin_dQ ? 5 : 0;
  if (a.begin_dQ) {
#pragma unroll
    for (int l = 0; l < 5; l++) out.at(oo, l) = 0.0;
  }
#pragma unroll
  for (int n = 0; n < NS - 1; n++) out.at(oo, row + n) = (x[n] - Ys[n]) * rdt;
}

template <class M>
__global__ __launch_bounds__(M::GROUPS *IM_CELLS) void k_icol(ImArgs a) {
  extern __shared__ double lds[];
  const unsigned c = min(xcd_block() * IM_CELLS + threadIdx.x % IM_CELLS, (unsigned)a.ncell - 1);
  int i, j, k;
  cell_at(a.b, c, i, j, k);
  ijac_columns<M>(a, a.Q, a.st, lds, i, j, k, c);
}

// a tile's two slices in workgroups numbered one after another, so one XCD's L2 serves y to both
template <class M>
__global__ __launch_bounds__(FLAT) void k_iwhole(ImArgs a) {
  const unsigned g = xcd_block();
  int i, j, k;
  if (!flat_at(a.b, g / 2, i, j, k)) return;
  ijac_whole<M>(a, a.Q, i, j, k, im_code(a.b, i, j, k), (int)(g % 2));
}

template <int NV>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1))) void k_lusolve(ImArgs a) {
  const unsigned cell = blockIdx.x * 64 + threadIdx.x;
  int i, j, k;
  if (cell < (unsigned)a.ncell && cell_at(a.b, cell, i, j, k)) lu_refine_cell<NV>(a, a.Q, a.out, i, j, k, cell);
}

}  // namespace pga
