// The alpha-damped viscous flux of one face (navstokes/kernels/flux/alpha-damping.mako:3-99), in
// registers: shared by the viscous sweep of one axis (pga_diffflux) and the launch over every face of
// a block (pga_faces), so both give the same bits.
//
// A face reads some 30 + 14 NS doubles of the cell arrays beside the advective flux's, and a few hundred
// operations turn them into its flux: it is bound by how often a wave waits on memory. Left to itself the
// compiler's schedule puts each load just ahead of its use, twenty and more waits a face at the registers
// of one row, so the reads are made in groups that end in a scheduling barrier: the rows of the velocity
// and T, then the species' two at a time (four at a time is no faster). The arrays share their layout, and
// a cell's reads go through View::run: each array's plane is a scalar base, the cell one vector offset. With
// the advective flux as it stands, a Taylor-Green box's faces take 11.6 us a launch at 32^3 and 34.5 at 57^3 so,
// 14.9 and 38.8 with the reads left to the schedule (the faces of an earlier advective flux, whose schedule
// happened to be kinder, took 11.0 and 35.4: at 32^3 the groups only win that back); the step of the 256 x
// 128 x 64 real-gas layer 3.47 ms against 3.59; nine species with MUSCL as long either way (110 us at 80 x 48 x 56).
#pragma once

#include "pga_common.hpp"

namespace pga {

// what a face reads of its two cells ([0] the left) for the rows u, v, w, T, and where it lies
struct DiffRows {
  double tr[2][2], x[2][3], xf[3], g[4][2][3];
  double Dl[2], hl[2];  // the last species' D and h
};

// a face's cells, as byte offsets into a plane of a cell array, and its own
struct DiffAt {
  int64_t oL, oR;
  uint32_t bL, bR, bx;
};

__device__ __forceinline__ DiffAt diff_at(const View &Q, const View &xf, int axis, int i, int j, int k) {
  DiffAt at;
  at.oR = Q.off(i, j, k), at.oL = at.oR - (axis == 0 ? 1 : axis == 1 ? Q.sj : Q.sk);
  at.bL = View::bytes(at.oL), at.bR = View::bytes(at.oR), at.bx = View::bytes(xf.off(i, j, k));
  return at;
}

template <int NS>
__device__ __forceinline__ void diff_load(const View &tr, const View &hsp, const View &gr, const View &xcc,
                                          const View &xf, DiffAt at, DiffRows &r) {
#pragma unroll
  for (int d = 0; d < 3; d++) r.xf[d] = xf.run(at.bx, d);
#pragma unroll
  for (int m = 0; m < 2; m++) {
    uint32_t &b = m ? at.bR : at.bL;
#pragma unroll
    for (int d = 0; d < 3; d++) r.x[m][d] = xcc.run(b, d);
    r.tr[m][0] = tr.run(b, 0), r.tr[m][1] = tr.run(b, 1);
#pragma unroll
    for (int l = 0; l < 4; l++)
#pragma unroll
      for (int d = 0; d < 3; d++) r.g[l][m][d] = gr.run(b, 3 * l + d);
    r.Dl[m] = tr.run(b, NS + 1), r.hl[m] = hsp.run(b, NS - 1);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// navstokes/kernels/flux/alpha-damping.mako:3-99: the alpha-damped viscous flux of the face at `at`, its
// area vector S, added to its flux Fv (every component but the mass), in registers
template <int NS>
__device__ __forceinline__ void diff_face(const View &Q, const View &st, const View &tr, const View &hsp,
                                          const View &gr, const DiffRows &rows, DiffAt at, const double (&S)[3],
                                          double alpha, double (&Fv)[NS + 4]) {
#pragma clang fp contract(off)
  // the species whose reads are in flight at once
  constexpr int G = NS > 3 ? 2 : NS > 1 ? NS - 1 : 1;
  const int64_t oR = at.oR, oL = at.oL;
  const double bulkvisc = 0.0;
  const double Sx = S[0], Sy = S[1], Sz = S[2];
  const double Sabs = sqrt(Sx * Sx + Sy * Sy + Sz * Sz), Sinv = 1.0 / Sabs;
  const double nx = Sx * Sinv, ny = Sy * Sinv, nz = Sz * Sinv;
  const double mu = 0.5 * (rows.tr[1][0] + rows.tr[0][0]);
  const double kappa = 0.5 * (rows.tr[1][1] + rows.tr[0][1]);
  const double lambda = bulkvisc - 2.0 / 3.0 * mu;
  const double rhoinvL = st.at(oL, 2), rhoinvR = st.at(oR, 2);
  const double uL = Q.at(oL, 1) * rhoinvL, vL = Q.at(oL, 2) * rhoinvL, wL = Q.at(oL, 3) * rhoinvL;
  const double uR = Q.at(oR, 1) * rhoinvR, vR = Q.at(oR, 2) * rhoinvR, wR = Q.at(oR, 3) * rhoinvR;
  const double ex = rows.x[1][0] - rows.x[0][0], ey = rows.x[1][1] - rows.x[0][1], ez = rows.x[1][2] - rows.x[0][2];
  const double en0 = ex * nx, en1 = ey * ny, en2 = ez * nz;
  const double dampinv = alpha / sqrt(en0 * en0 + en1 * en1 + en2 * en2);
  const double dampx = dampinv * nx, dampy = dampinv * ny, dampz = dampinv * nz;
  const double xLx = rows.xf[0] - rows.x[0][0], xLy = rows.xf[1] - rows.x[0][1], xLz = rows.xf[2] - rows.x[0][2];
  const double xRx = rows.xf[0] - rows.x[1][0], xRy = rows.xf[1] - rows.x[1][1], xRz = rows.xf[2] - rows.x[1][2];
  const auto facegrad = [&](const double (&g)[2][3], double phiL, double phiR, double &gx, double &gy, double &gz) {
    const double wl = phiL + g[0][0] * xLx + g[0][1] * xLy + g[0][2] * xLz;
    const double wr = phiR + g[1][0] * xRx + g[1][1] * xRy + g[1][2] * xRz;
    const double jump = wr - wl;
    gx = 0.5 * (g[1][0] + g[0][0]) + dampx * jump;
    gy = 0.5 * (g[1][1] + g[0][1]) + dampy * jump;
    gz = 0.5 * (g[1][2] + g[0][2]) + dampz * jump;
  };
  double dudx, dudy, dudz, dvdx, dvdy, dvdz, dwdx, dwdy, dwdz;
  facegrad(rows.g[0], uL, uR, dudx, dudy, dudz);
  facegrad(rows.g[1], vL, vR, dvdx, dvdy, dvdz);
  facegrad(rows.g[2], wL, wR, dwdx, dwdy, dwdz);
  const double div = dudx + dvdy + dwdz;
  const double txx = -2.0 * mu * dudx - lambda * div;
  const double txy = -mu * (dvdx + dudy);
  const double txz = -mu * (dwdx + dudz);
  const double tyy = -2.0 * mu * dvdy - lambda * div;
  const double tyz = -mu * (dwdy + dvdz);
  const double tzz = -2.0 * mu * dwdz - lambda * div;
  Fv[1] += txx * Sx + txy * Sy + txz * Sz;
  Fv[2] += txy * Sx + tyy * Sy + tyz * Sz;
  Fv[3] += txz * Sx + tyz * Sy + tzz * Sz;
  double dTx, dTy, dTz;
  facegrad(rows.g[3], st.at(oL, 1), st.at(oR, 1), dTx, dTy, dTz);
  const double heatflux = -kappa * (dTx * Sx + dTy * Sy + dTz * Sz);
  const double uf = 0.5 * (uR + uL), vf = 0.5 * (vR + vL), wf = 0.5 * (wR + wL);
  double f4 = (uf * txx + vf * txy + wf * txz) * Sx + (uf * txy + vf * tyy + wf * tyz) * Sy +
              (uf * txz + vf * tyz + wf * tzz) * Sz + heatflux;
  double Vc = 0.0, gradYns = 0.0, sumYh = 0.0, Yns = 1.0;
  const double rho = 0.5 * (Q.at(oR, 0) + Q.at(oL, 0));
  double Ym[NS];
#pragma unroll
  for (int n0 = 0; n0 < NS - 1; n0 += G) {
    double y[G][2], D[G][2], h[G][2], g[G][2][3];
#pragma unroll
    for (int m = 0; m < 2; m++) {
      uint32_t &b = m ? at.bR : at.bL;
#pragma unroll
      for (int c = 0; c < G; c++) {
        const int n = n0 + c;
        if (n >= NS - 1) continue;
        y[c][m] = Q.run(b, 5 + n);
        D[c][m] = tr.run(b, 2 + n);
        h[c][m] = hsp.run(b, n);
#pragma unroll
        for (int d = 0; d < 3; d++) g[c][m][d] = gr.run(b, 12 + 3 * n + d);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < G; c++) {
      const int n = n0 + c;
      if (n >= NS - 1) continue;
      const double yL = y[c][0] * rhoinvL, yR = y[c][1] * rhoinvR;
      const double Dk = 0.5 * (D[c][1] + D[c][0]);
      double dYx, dYy, dYz;
      facegrad(g[c], yL, yR, dYx, dYy, dYz);
      const double gradYk = dYx * Sx + dYy * Sy + dYz * Sz;
      gradYns -= gradYk;
      Vc += Dk * gradYk;
      const double Jk = -rho * Dk * gradYk;
      const double hk = 0.5 * (h[c][1] + h[c][0]);
      const double Yk = 0.5 * (yR + yL);
      Yns -= Yk;
      sumYh += Yk * hk;
      Ym[n] = Yk;
      Fv[5 + n] = Fv[5 + n] + Jk;
      f4 += Jk * hk;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const double Dk = 0.5 * (rows.Dl[1] + rows.Dl[0]);
  Vc += Dk * gradYns;
  const double corr = rho * Vc;
#pragma unroll
  for (int n = 0; n < NS - 1; n++) Fv[5 + n] = Fv[5 + n] + Ym[n] * corr;
  f4 += corr * sumYh;
  const double hns = 0.5 * (rows.hl[1] + rows.hl[0]);
  f4 += (-rho * Dk * gradYns + Yns * corr) * hns;
  Fv[4] += f4;
}

}  // namespace pga
