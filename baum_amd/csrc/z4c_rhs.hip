// z4c_rhs.hip -- Z4c right-hand side on gfx950, FP64.
//
// Equations: src/projects/z4/z4_rhs_movpunc_N.m:217-467 (conformal
// connection and Ricci, conformal-factor terms, 1+log / Gamma-driver gauge,
// Kreiss-Oliger dissipation, optional addlinear update with trace removal and
// det normalisation).  Stencils: src/math/MathToC/discretize.m:18-46,97-135
// and src/main/amr/bam_amr_advection.h:28-155.  Box-edge rules (order 2 one
// point from the edge, shifted advection stencils within rstencil points, KO
// only two or more points away): src/main/amr/bam_amr_loops_box.h:186-215.
//
// Layout: SoA, one double array per grid function, ijk = i + m*j + m*n*k
// within a box, boxes concatenated at noffset.
//
// The usual parameters (order 4, lop-sided 1) run in the tile kernel of
// z4c_tile.h, planned and launched here.  Any other choice runs in the per-point
// kernel below, whose derivative provider follows the reference's order
// selection point by point.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "bamhip_internal.h"
#include "z4c_tile.h"

namespace bamhip {

// ---------------------------------------------------------------- providers
// lop-sided advection rows: stencil4[offset] of order 4 and the order-2 rows
// (bam_amr_advection.h:28-36,90-146), row index = offset
__constant__ double kAdvSt4[5][5] = {{25. / 12, -48. / 12, 36. / 12, -16. / 12, 3. / 12},
                                     {3. / 12, 10. / 12, -18. / 12, 6. / 12, -1. / 12},
                                     {-1. / 12, 8. / 12, 0. / 12, -8. / 12, 1. / 12},
                                     {1. / 12, -6. / 12, 18. / 12, -10. / 12, -3. / 12},
                                     {-3. / 12, 16. / 12, -36. / 12, 48. / 12, -25. / 12}};
__constant__ double kAdvSt2[3][3] = {{1.5, -2.0, 0.5}, {0.5, 0.0, -0.5}, {-0.5, 2.0, -1.5}};

// runtime-order provider following the reference per point
struct Edge {
  long q;
  long s[3];
  const Z4cGeo &G;
  int ordc, orda, twoormore;
  int pos[3], pmax[3];
  __device__ Edge(const Z4cGeo &g, long q_, int i, int j, int k, const Z4cK &K) : q(q_), G(g) {
    s[0] = 1;
    s[1] = g.sj;
    s[2] = g.sk;
    pos[0] = i;
    pos[1] = j;
    pos[2] = k;
    pmax[0] = g.m - 1;
    pmax[1] = g.n - 1;
    pmax[2] = g.o - 1;
    const int away1 = (i == 1 || j == 1 || k == 1 || i == pmax[0] - 1 || j == pmax[1] - 1 || k == pmax[2] - 1);
    twoormore = (i >= 2 && j >= 2 && k >= 2 && i <= pmax[0] - 2 && j <= pmax[1] - 2 && k <= pmax[2] - 2);
    ordc = (K.order_centered == 2 || away1) ? 2 : 4;
    orda = (K.order_advection == 2 || away1) ? 2 : 4;
  }
  __device__ double d1(const double *__restrict__ f, int a) const {
    const long t = s[a];
    if (ordc == 2) return (f[q + t] - f[q - t]) * G.i2h[a];
    return ((f[q - 2 * t] - f[q + 2 * t]) + 8.0 * (f[q + t] - f[q - t])) * G.i12h[a];
  }
  __device__ double d2(const double *__restrict__ f, int a) const {
    const long t = s[a];
    if (ordc == 2) return (f[q - t] + f[q + t] - 2.0 * f[q]) * G.ihh[a];
    return (16.0 * (f[q - t] + f[q + t]) - (f[q - 2 * t] + f[q + 2 * t]) - 30.0 * f[q]) * G.i12hh[a];
  }
  __device__ double dd(const double *__restrict__ f, int a, int b) const {
    if (a == b) return d2(f, a);
    const long t = s[a], w = s[b];
    if (ordc == 2) {
      return ((f[q + t + w] - f[q + t - w]) - (f[q - t + w] - f[q - t - w])) * G.i4hh[mixid(a, b)];
    }
    auto row = [&](long o) { return (f[o - 2 * w] - f[o + 2 * w]) + 8.0 * (f[o + w] - f[o - w]); };
    return ((row(q - 2 * t) - row(q + 2 * t)) + 8.0 * (row(q + t) - row(q - t))) * G.i144hh[mixid(a, b)];
  }
  // advection weights over offsets -4..4 (slot 4 = centre), rows of
  // set_advection4 / stencil4 (bam_amr_advection.h:28-155)
  double W[3][9];
  __device__ void set_adv(const double beta[3], const Z4cK &K) {
    for (int a = 0; a < 3; a++) {
      for (int k = 0; k < 9; k++) W[a][k] = 0.0;
      const double wx = beta[a] * G.ih[a];
      const int i = pos[a], imax = pmax[a];
      const int rst = (orda == 2) ? 2 : 4 - K.lopsided;
      int wsign, offset;
      if (wx < 0) {
        wsign = -1;
        offset = (i >= rst) ? 0 : rst - i;
      } else if (wx > 0) {
        wsign = 1;
        offset = (imax - i >= rst) ? 0 : rst - (imax - i);
      } else {
        wsign = 0;
        offset = 0;
      }
      if (wsign == 0) continue;
      if (orda == 2) {
        for (int k = 0; k < 3; k++) W[a][4 + wsign * (k - offset)] += -wsign * wx * kAdvSt2[offset][k];
      } else {
        offset += K.lopsided;
        for (int k = 0; k < 5; k++) W[a][4 + wsign * (k - offset)] += -wsign * wx * kAdvSt4[offset][k];
      }
    }
  }
  __device__ double adv(const double *__restrict__ f) const {
    double acc = 0;
    for (int a = 0; a < 3; a++)
      for (int k = 0; k < 9; k++)
        if (W[a][k] != 0.0) acc += W[a][k] * f[q + (k - 4) * s[a]];
    return acc;
  }
  __device__ bool ko_on(const Z4cK &K) const { return K.order_dissipation == 4 && twoormore; }
  __device__ double ko(const double *__restrict__ f) const {
    double acc = 0;
    for (int a = 0; a < 3; a++) {
      const long t = s[a];
      acc += ((f[q - 2 * t] + f[q + 2 * t]) - 4.0 * (f[q - t] + f[q + t]) + 6.0 * f[q]) * G.ih[a];
    }
    return -acc;
  }
};

// write one point: raw RHS, or upre + c*RHS with trace removal and det
// normalisation (z4_rhs_movpunc_N.m:446-467)
__device__ __forceinline__ void store_point(const Z4cPtrs &P, const Z4cK &K, long q, double *rhs) {
  if (K.rk) {
    // all loads before any store: the lists may alias (the accumulator read
    // and the next state written at the point, for one), and loads written
    // after a store would each wait for it
    double av[25], pv[25];
#pragma unroll
    for (int v = 0; v < 25; v++) av[v] = P.a[v][q];
    if (K.has_v || K.has_cp) {
#pragma unroll
      for (int v = 0; v < 25; v++) pv[v] = P.p[v][q];
    }
#pragma unroll
    for (int v = 0; v < 25; v++) P.c[v][q] = av[v] + K.wc * rhs[v];
    if (K.has_v) {
#pragma unroll
      for (int v = 0; v < 25; v++) P.r[v][q] = pv[v] + K.wv * rhs[v];
    }
    if (K.has_cp) {
#pragma unroll
      for (int v = 0; v < 25; v++) P.cp[v][q] = pv[v];
    }
    return;
  }
  if (K.addlinear) {
#pragma unroll
    for (int v = 0; v < 25; v++) rhs[v] = P.p[v][q] + K.c * rhs[v];
    double ng[6], nA[6];
#pragma unroll
    for (int c = 0; c < 6; c++) {
      ng[c] = rhs[c];
      nA[c] = rhs[7 + c];
    }
    const double a0 = ng[3] * ng[5] - ng[4] * ng[4], a1 = ng[2] * ng[4] - ng[1] * ng[5];
    const double a2 = ng[1] * ng[4] - ng[2] * ng[3], a3 = ng[0] * ng[5] - ng[2] * ng[2];
    const double a4 = ng[1] * ng[2] - ng[0] * ng[4], a5 = ng[0] * ng[3] - ng[1] * ng[1];
    const double detnginv = 1.0 / (ng[0] * a0 + ng[1] * a1 + ng[2] * a2);
    if (K.subtractA) {
      const double trA =
          detnginv * (a0 * nA[0] + a3 * nA[3] + a5 * nA[5] + 2.0 * (a1 * nA[1] + a2 * nA[2] + a4 * nA[4]));
#pragma unroll
      for (int c = 0; c < 6; c++) rhs[7 + c] = nA[c] - (trA / 3.0) * ng[c];
    }
    if (K.normalizedetg) {
      const double aux = pow(detnginv, 1.0 / 3.0);
#pragma unroll
      for (int c = 0; c < 6; c++) rhs[c] = aux * ng[c];
    }
  }
#pragma unroll
  for (int v = 0; v < 25; v++) P.r[v][q] = rhs[v];
}

// ------------------------------------------------------------------ algebra
template <class D>
__device__ __forceinline__ bool z4c_point(D &dv, const Z4cPtrs &P, const Z4cK &K, long q) {
  const double *const *u = P.u;
  // point values (list order of z4.c:234-242)
  double g[6], A[6], Gm[3], beta[3], Bv[3];
#pragma unroll
  for (int c = 0; c < 6; c++) {
    g[c] = u[c][q];
    A[c] = u[7 + c][q];
  }
#pragma unroll
  for (int a = 0; a < 3; a++) {
    Gm[a] = u[14 + a][q];
    beta[a] = u[19 + a][q];
    Bv[a] = u[22 + a][q];
  }
  const double chi = u[6][q], Khat = u[13][q], Theta = u[17][q], alpha = u[18][q];

  // advection terms (lie*, adv*) of all 25 fields, weighted by their
  // coefficients in the right-hand sides
  dv.set_adv(beta, K);
  double rhs[25];
#pragma unroll
  for (int c = 0; c < 6; c++) {
    rhs[c] = dv.adv(u[c]);
    rhs[7 + c] = dv.adv(u[7 + c]);
  }
  rhs[6] = dv.adv(u[6]);
  rhs[13] = dv.adv(u[13]);
  double advG[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    advG[a] = dv.adv(u[14 + a]);
    rhs[19 + a] = K.withShiftadv * dv.adv(u[19 + a]);
    rhs[22 + a] = K.withBadv * dv.adv(u[22 + a]);
  }
  rhs[17] = dv.adv(u[17]);
  rhs[18] = K.oplogwithshift * dv.adv(u[18]);

  BH_PHASE();
  // inverse conformal metric
  double ig[6];
  ig[0] = g[3] * g[5] - g[4] * g[4];
  ig[1] = g[2] * g[4] - g[1] * g[5];
  ig[2] = g[1] * g[4] - g[2] * g[3];
  ig[3] = g[0] * g[5] - g[2] * g[2];
  ig[4] = g[1] * g[2] - g[0] * g[4];
  ig[5] = g[0] * g[3] - g[1] * g[1];
  const double detginv = 1.0 / (g[0] * ig[0] + g[1] * ig[1] + g[2] * ig[2]);
#pragma unroll
  for (int c = 0; c < 6; c++) ig[c] *= detginv;

  BH_PHASE();
  // Christoffels: lower Gd[c][ab] = Gamma_{c ab}, upper Gu[c][ab] = Gamma^c_ab
  double Gd[3][6];
  {
    double dg[3][6];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int ab = 0; ab < 6; ab++) dg[c][ab] = dv.d1(u[ab], c);
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = a; b < 3; b++)
          Gd[c][sy(a, b)] = 0.5 * (dg[a][sy(b, c)] + dg[b][sy(a, c)] - dg[c][sy(a, b)]);
  }
  double Gu[3][6];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int ab = 0; ab < 6; ab++)
      Gu[c][ab] = ig[sy(c, 0)] * Gd[0][ab] + ig[sy(c, 1)] * Gd[1][ab] + ig[sy(c, 2)] * Gd[2][ab];
  double Gfg[3];
#pragma unroll
  for (int a = 0; a < 3; a++)
    Gfg[a] = ig[0] * Gu[a][0] + ig[3] * Gu[a][3] + ig[5] * Gu[a][5] +
             2.0 * (ig[1] * Gu[a][1] + ig[2] * Gu[a][2] + ig[4] * Gu[a][4]);

  BH_PHASE();
  // Ricci of the conformal metric
  double R[6];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = a; b < 3; b++) {
      double s = 0.0;
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int d = 0; d < 3; d++) {
          double t = 0.0;
#pragma unroll
          for (int e = 0; e < 3; e++)
            t += Gu[e][sy(c, a)] * Gd[b][sy(e, d)] + Gu[e][sy(c, b)] * Gd[a][sy(e, d)] +
                 Gu[e][sy(a, d)] * Gd[e][sy(c, b)];
          s += ig[sy(c, d)] * t;
        }
      double t2 = 0.0;
#pragma unroll
      for (int c = 0; c < 3; c++) t2 += Gfg[c] * (Gd[a][sy(b, c)] + Gd[b][sy(a, c)]);
      R[sy(a, b)] = s + 0.5 * t2;
    }
  BH_PHASE();
  // - 1/2 g^cd d_c d_d g_ab, consumed component by component
#pragma unroll
  for (int ab = 0; ab < 6; ab++) {
    const double *f = u[ab];
    const double lap = ig[0] * dv.d2(f, 0) + ig[3] * dv.d2(f, 1) + ig[5] * dv.d2(f, 2) +
                       2.0 * (ig[1] * dv.dd(f, 0, 1) + ig[2] * dv.dd(f, 0, 2) + ig[4] * dv.dd(f, 1, 2));
    R[ab] -= 0.5 * lap;
    BH_PHASE();
  }
  BH_PHASE();
  // + 1/2 (g_ca d_b G^c + g_cb d_a G^c)
  {
    double dG[3][3];  // dG[b][c] = d_b G^c
#pragma unroll
    for (int b = 0; b < 3; b++)
#pragma unroll
      for (int c = 0; c < 3; c++) dG[b][c] = dv.d1(u[14 + c], b);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = a; b < 3; b++) {
        double t = 0.0;
#pragma unroll
        for (int c = 0; c < 3; c++) t += g[sy(c, a)] * dG[b][c] + g[sy(c, b)] * dG[a][c];
        R[sy(a, b)] += 0.5 * t;
      }
  }

  BH_PHASE();
  // conformal factor
  const double chig = (chi < K.chiDivFloor) ? K.chiDivFloor : chi;
  const double oocp = 1.0 / K.chipsipower;
  const double psim4 = exp(-4.0 * oocp * log(chig));
  const double oochig = 1.0 / chig;
  double dchi[3], df[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    dchi[a] = dv.d1(u[6], a);
    df[a] = oocp * dchi[a] * oochig;
  }
  double cddf[6];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = a; b < 3; b++) {
      const int ab = sy(a, b);
      cddf[ab] = oocp * dv.dd(u[6], a, b) * oochig - K.chipsipower * df[a] * df[b] -
                 (Gu[0][ab] * df[0] + Gu[1][ab] * df[1] + Gu[2][ab] * df[2]);
    }
  auto trace = [&](const double *t6) {
    return ig[0] * t6[0] + ig[3] * t6[3] + ig[5] * t6[5] + 2.0 * (ig[1] * t6[1] + ig[2] * t6[2] + ig[4] * t6[4]);
  };
  auto contract = [&](const double *x, const double *y) {
    return ig[0] * x[0] * y[0] + ig[3] * x[1] * y[1] + ig[5] * x[2] * y[2] +
           ig[1] * (x[0] * y[1] + x[1] * y[0]) + ig[2] * (x[0] * y[2] + x[2] * y[0]) +
           ig[4] * (x[1] * y[2] + x[2] * y[1]);
  };
  const double trcddf = trace(cddf);
  const double dfdf = contract(df, df);
  // R + Rphi
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = a; b < 3; b++) {
      const int ab = sy(a, b);
      R[ab] += 4.0 * df[a] * df[b] - 2.0 * cddf[ab] - 2.0 * g[ab] * trcddf - 4.0 * g[ab] * dfdf;
    }

  BH_PHASE();
  // lapse derivatives
  double da[3];
#pragma unroll
  for (int a = 0; a < 3; a++) da[a] = dv.d1(u[18], a);
  const double dfda = contract(df, da);
  double cdda[6];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = a; b < 3; b++) {
      const int ab = sy(a, b);
      cdda[ab] = dv.dd(u[18], a, b) - (Gu[0][ab] * da[0] + Gu[1][ab] * da[1] + Gu[2][ab] * da[2]) -
                 2.0 * (df[a] * da[b] + df[b] * da[a] - g[ab] * dfda);
    }
  const double trcdda = psim4 * trace(cdda);

  BH_PHASE();
  // extrinsic-curvature terms
  double Ainv[6], AA[6];
  {
    double Au[3][3];  // Au[a][b] = g^ac A_cb (mixed)
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++)
        Au[a][b] = ig[sy(a, 0)] * A[sy(0, b)] + ig[sy(a, 1)] * A[sy(1, b)] + ig[sy(a, 2)] * A[sy(2, b)];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = a; b < 3; b++) {
        Ainv[sy(a, b)] = Au[a][0] * ig[sy(0, b)] + Au[a][1] * ig[sy(1, b)] + Au[a][2] * ig[sy(2, b)];
        AA[sy(a, b)] = A[sy(a, 0)] * Au[0][b] + A[sy(a, 1)] * Au[1][b] + A[sy(a, 2)] * Au[2][b];
      }
  }
  const double cAA = trace(AA);
  const double K_ = Khat + 2.0 * Theta;
  double dKT[3];  // 2 dKhat + dTheta
#pragma unroll
  for (int a = 0; a < 3; a++) dKT[a] = 2.0 * dv.d1(u[13], a) + dv.d1(u[17], a);
  double divAinv[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    double s = 0.0;
#pragma unroll
    for (int bc = 0; bc < 6; bc++) s += ((bc == 0 || bc == 3 || bc == 5) ? 1.0 : 2.0) * Gu[a][bc] * Ainv[bc];
    s -= 1.5 * oochig * (Ainv[sy(a, 0)] * dchi[0] + Ainv[sy(a, 1)] * dchi[1] + Ainv[sy(a, 2)] * dchi[2]);
    s -= (1.0 / 3.0) * (ig[sy(a, 0)] * dKT[0] + ig[sy(a, 1)] * dKT[1] + ig[sy(a, 2)] * dKT[2]);
    divAinv[a] = s;
  }
  const double Rhat = psim4 * trace(R);   // R holds R + Rphi
  const double Hhat = Rhat + 2.0 * K_ * K_ / 3.0 - cAA;

  BH_PHASE();
  // shift terms
  double db[3][3];  // db[a][b] = d_a beta^b
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) db[a][b] = dv.d1(u[19 + b], a);
  const double divbeta = db[0][0] + db[1][1] + db[2][2];
  const double tdb = (2.0 / 3.0) * divbeta;
  double pG[3];
  {
    // g^bc d_b d_c beta^a + g^ab (1/3) d_b d_c beta^c
    double ddbc[3][6];
#pragma unroll
    for (int cc = 0; cc < 3; cc++)
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = a; b < 3; b++) ddbc[cc][sy(a, b)] = dv.dd(u[19 + cc], a, b);
    double ootd[3];
#pragma unroll
    for (int a = 0; a < 3; a++) ootd[a] = (1.0 / 3.0) * (ddbc[0][sy(a, 0)] + ddbc[1][sy(a, 1)] + ddbc[2][sy(a, 2)]);
#pragma unroll
    for (int a = 0; a < 3; a++)
      pG[a] = trace(ddbc[a]) + ig[sy(a, 0)] * ootd[0] + ig[sy(a, 1)] * ootd[1] + ig[sy(a, 2)] * ootd[2] -
              (Gfg[0] * db[0][a] + Gfg[1] * db[1][a] + Gfg[2] * db[2][a]) + Gfg[a] * tdb + advG[a];
  }

  BH_PHASE();
  // right-hand sides
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = a; b < 3; b++) {
      const int ab = sy(a, b);
      double lg = -g[ab] * tdb, lA = -A[ab] * tdb;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        lg += db[a][c] * g[sy(b, c)] + db[b][c] * g[sy(a, c)];
        lA += db[a][c] * A[sy(b, c)] + db[b][c] * A[sy(a, c)];
      }
      rhs[ab] += -2.0 * alpha * A[ab] + lg;
      rhs[7 + ab] += psim4 * (-cdda[ab] + alpha * R[ab]) - (1.0 / 3.0) * g[ab] * (-trcdda + alpha * Rhat) +
                     alpha * (K_ * A[ab] - 2.0 * AA[ab]) + lA;
    }
  double rG[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    rG[a] = -2.0 * (Ainv[sy(a, 0)] * da[0] + Ainv[sy(a, 1)] * da[1] + Ainv[sy(a, 2)] * da[2]) +
            2.0 * alpha * divAinv[a] - 2.0 * alpha * K.kappa1 * (Gm[a] - Gfg[a]) + pG[a];
    rhs[14 + a] = rG[a];
  }
  rhs[13] += -trcdda + alpha * (cAA + K_ * K_ / 3.0) + K.kappa1 * (1.0 - K.kappa2) * alpha * Theta;
  rhs[6] += (K.chipsipower / 6.0) * chig * divbeta - (K.chipsipower / 6.0) * chig * alpha * K_;
  rhs[17] = (alpha * (0.5 * Hhat - (2.0 + K.kappa2) * K.kappa1 * Theta) + rhs[17]) * K.zeroThetaRHS;

  BH_PHASE();
  // gauge
  const double falpha =
      K.oploglapse * K.lapseharmonicf + K.oploglapse2 * (8.0 / 3.0) / (3.0 - alpha) + K.harmoniclapse * alpha;
  rhs[18] -= falpha * alpha * Khat;
  if (K.withB != 0.0) {
    const double betaF = K.shiftgammacoeff * pow(alpha, K.shiftalphapower);
#pragma unroll
    for (int a = 0; a < 3; a++) {
      rhs[19 + a] += (K.gamma2factor + K.gamma0factor * betaF) * Bv[a];
      rhs[22 + a] += (K.gamma0factor + K.gamma2factor * betaF) * (rG[a] - K.withGadv * advG[a]) -
                     K.shiftdriver * Bv[a];
    }
  } else {
#pragma unroll
    for (int a = 0; a < 3; a++) {
      rhs[22 + a] = 0.0;
      rhs[19 + a] += Gm[a] - K.shiftdriver * beta[a];
    }
  }

  BH_PHASE();
  // Kreiss-Oliger dissipation
  if (dv.ko_on(K)) {
#pragma unroll
    for (int v = 0; v < 25; v++) rhs[v] += K.dissfactor * dv.ko(u[v]);
  }

  bool finite = true;
#pragma unroll
  for (int v = 0; v < 25; v++) finite = finite && isfinite(rhs[v]);

  store_point(P, K, q, rhs);
  return finite;
}

// ------------------------------------------------------------------ kernels
// all computed points that are not in [blo, bhi] (the bulk region), or all
// computed points when edge_only == 0
__global__ void __launch_bounds__(256) z4c_rhs_edge(Z4cPtrs P, Z4cGeo G, Z4cK K, int blo0, int blo1, int blo2,
                                                   int bhi0, int bhi1, int bhi2, int *flag) {
  const int i = G.lo[0] + blockIdx.x * 64 + threadIdx.x;
  const int j = G.lo[1] + blockIdx.y * 4 + threadIdx.y;
  const int k = G.lo[2] + blockIdx.z;
  if (i > G.hi[0] || j > G.hi[1] || k > G.hi[2]) return;
  if (G.edge_only && i >= blo0 && i <= bhi0 && j >= blo1 && j <= bhi1 && k >= blo2 && k <= bhi2) return;
  const long q = G.noffset + i + G.sj * j + G.sk * k;
  Edge dv(G, q, i, j, k, K);
  if (!z4c_point(dv, P, K, q)) *flag = 1;
}

__global__ void set_int(int *p, int v) { *p = v; }

static Z4cK make_k(const bamhip_z4c_params *p, double c) {
  Z4cK K;
  K.order_centered = p->order_centered;
  K.order_advection = p->order_advection;
  K.lopsided = p->advection_lopsided;
  K.order_dissipation = p->order_dissipation;
  K.dissfactor = p->dissfactor;
  K.kappa1 = p->kappa1;
  K.kappa2 = p->kappa2;
  K.zeroThetaRHS = p->zeroThetaRHS;
  K.subtractA = p->subtractA;
  K.normalizedetg = p->normalizedetg;
  K.oploglapse = p->oploglapse;
  K.oploglapse2 = p->oploglapse2;
  K.oplogwithshift = p->oplogwithshift;
  K.harmoniclapse = p->harmoniclapse;
  K.lapseharmonicf = p->lapseharmonicf;
  K.gamma0factor = p->gamma0factor;
  K.gamma2factor = p->gamma2factor;
  K.withGadv = p->withGadv;
  K.withShiftadv = p->withShiftadv;
  K.withBadv = p->withBadv;
  K.withB = p->withB;
  K.shiftalphapower = p->shiftalphapower;
  K.shiftgammacoeff = p->shiftgammacoeff;
  K.shiftdriver = p->shiftdriver;
  K.chiDivFloor = p->chiDivFloor;
  K.chipsipower = p->chipsipower;
  K.oocp = 1.0 / p->chipsipower;
  K.c = c;
  K.addlinear = (c != 0.0);
  K.rk = 0;
  K.has_v = 0;
  K.has_cp = 0;
  K.wc = K.wv = 0.0;
  return K;
}

static void make_geo(const DevBox &B, Z4cGeo &G) {
  G.m = B.m;
  G.n = B.n;
  G.o = B.o;
  G.noffset = B.noffset;
  G.lo[0] = B.skip[0];
  G.hi[0] = B.m - 1 - B.skip[1];
  G.lo[1] = B.skip[2];
  G.hi[1] = B.n - 1 - B.skip[3];
  G.lo[2] = B.skip[4];
  G.hi[2] = B.o - 1 - B.skip[5];
  G.sj = B.m;
  G.sk = (long)B.m * B.n;
  const double h[3] = {B.dx, B.dy, B.dz};
  for (int a = 0; a < 3; a++) {
    G.h[a] = h[a];
    G.ih[a] = 1.0 / h[a];
    G.i12h[a] = 1.0 / (12.0 * h[a]);
    G.i12hh[a] = 1.0 / (12.0 * h[a] * h[a]);
    G.i2h[a] = 1.0 / (2.0 * h[a]);
    G.ihh[a] = 1.0 / (h[a] * h[a]);
  }
  G.i144hh[0] = 1.0 / (144.0 * h[0] * h[1]);
  G.i144hh[1] = 1.0 / (144.0 * h[0] * h[2]);
  G.i144hh[2] = 1.0 / (144.0 * h[1] * h[2]);
  G.i4hh[0] = 1.0 / (4.0 * h[0] * h[1]);
  G.i4hh[1] = 1.0 / (4.0 * h[0] * h[2]);
  G.i4hh[2] = 1.0 / (4.0 * h[1] * h[2]);
  G.edge_only = 0;
}

// tile regions of one level, by layout
struct LevelTiles {
  std::vector<Z4cGeo> bulk;
  std::vector<Z4cGeo> sx, sy, sz;  // shell as slabs (up to two points thick) normal to x, y, z
};

static void add_region(std::vector<Z4cGeo> &v, const Z4cGeo &G0, const int lo[3], const int hi[3]) {
  if (hi[0] < lo[0] || hi[1] < lo[1] || hi[2] < lo[2]) return;
  Z4cGeo G = G0;
  for (int a = 0; a < 3; a++) {
    G.lo[a] = lo[a];
    G.hi[a] = hi[a];
  }
  v.push_back(G);
}

static int g_xcd_map = 1;  // XCD-aware tile numbering in the tile kernels
int tile_xcd_map() { return g_xcd_map; }

// Split one box into its bulk region (>= 3 points from every edge) and the
// slabs of its edge shell (fast parameters), or launch the generic per-point
// kernel for the other parameter choices.
static int plan_box(const DevBox &B, const Z4cPtrs &P, const Z4cK &K, int *flag, bool fast, LevelTiles &T) {
  Z4cGeo G;
  make_geo(B, G);
  if (G.hi[0] < G.lo[0] || G.hi[1] < G.lo[1] || G.hi[2] < G.lo[2]) return BAMHIP_OK;
  int blo[3], bhi[3];
  const int dims[3] = {B.m, B.n, B.o};
  bool have_bulk = fast;
  for (int a = 0; a < 3; a++) {
    blo[a] = G.lo[a] > 3 ? G.lo[a] : 3;
    bhi[a] = G.hi[a] < dims[a] - 4 ? G.hi[a] : dims[a] - 4;
    if (bhi[a] < blo[a]) have_bulk = false;
  }
  if (have_bulk) add_region(T.bulk, G, blo, bhi);
  const bool need_edge = !have_bulk || blo[0] > G.lo[0] || bhi[0] < G.hi[0] || blo[1] > G.lo[1] ||
                         bhi[1] < G.hi[1] || blo[2] > G.lo[2] || bhi[2] < G.hi[2];
  if (need_edge && fast) {
    // The shell of points closer than 3 to an edge, as disjoint slabs: the
    // layers along x over all y, z; along y over the x interior; along z over
    // the x and y interior.  Layers of axis a: [lo, min(hi, 2)] and
    // [max(dim - 3, end of the first + 1), hi].
    int lay[3][2][2], ilo[3], ihi[3];
    for (int a = 0; a < 3; a++) {
      lay[a][0][0] = G.lo[a];
      lay[a][0][1] = std::min(G.hi[a], 2);
      lay[a][1][0] = std::max(dims[a] - 3, lay[a][0][1] + 1);
      lay[a][1][1] = G.hi[a];
      ilo[a] = std::max(G.lo[a], 3);
      ihi[a] = std::min(G.hi[a], dims[a] - 4);
    }
    for (int s = 0; s < 2; s++) {
      const int xl[3] = {lay[0][s][0], G.lo[1], G.lo[2]}, xh[3] = {lay[0][s][1], G.hi[1], G.hi[2]};
      add_region(T.sx, G, xl, xh);
      const int yl[3] = {ilo[0], lay[1][s][0], G.lo[2]}, yh[3] = {ihi[0], lay[1][s][1], G.hi[2]};
      add_region(T.sy, G, yl, yh);
      const int zl[3] = {ilo[0], ilo[1], lay[2][s][0]}, zh[3] = {ihi[0], ihi[1], lay[2][s][1]};
      add_region(T.sz, G, zl, zh);
    }
  } else if (need_edge) {
    G.edge_only = have_bulk ? 1 : 0;
    dim3 grid((G.hi[0] - G.lo[0] + 64) / 64, (G.hi[1] - G.lo[1] + 4) / 4, G.hi[2] - G.lo[2] + 1);
    {
      TimerScope t("z4_rhs_edge");
      z4c_rhs_edge<<<grid, dim3(64, 4, 1), 0, stream()>>>(P, G, K, blo[0], blo[1], blo[2], bhi[0], bhi[1], bhi[2],
                                                          flag);
    }
    BH_HIP(hipGetLastError());
  }
  return BAMHIP_OK;
}

// ---- autotuner of the tile kernels
// A variant is one staging of the tile kernel: through registers, or by
// LDS-DMA in dwords or in 16-byte units.  Every variant evaluates the same
// per-point arithmetic in the same order, so all give bitwise the same
// right-hand side.  The first time a level's boxes are seen outside graph
// capture, each launch that may run is timed on them with every variant (one
// warm-up launch, then two timed with HIP events): the bulk tiles, the slabs of
// the box-edge shell, and both in one launch.  A level with bulk and shell takes
// one launch unless two, each with its own fastest variant, took less: the
// kernel of all four bodies is larger and spills more than that of the bulk
// alone, but leaves no tail between the two.  (Timed on the two launches only,
// the choice said nothing of the one that ran.)
struct Variant {
  const char *name;
  bool dma;    // LDS-DMA staging: byte offsets within a field must fit 32 bits
  bool pairs;  // 16-byte LDS-DMA units: needs 16-byte aligned element pairs
  LaunchFn fn;
};
constexpr int kMaxVariants = 3;
enum { kBulk, kShell, kBoth, kLaunches };
static const Variant kVariants[kLaunches][kMaxVariants] = {{{"bulk 16x4x4 dma3", true, false, tile_dma},
                                                            {"bulk 16x4x4 reg", false, false, tile_reg},
                                                            {"bulk 16x4x4 dma3 x4", true, true, tile_dma_x4}},
                                                           {{"shell slabs dma3", true, false, tile_dma},
                                                            {"shell slabs reg", false, false, tile_reg},
                                                            {"shell slabs dma3 x4", true, true, tile_dma_x4}},
                                                           {{"one launch dma3", true, false, tile_dma},
                                                            {"one launch reg", false, false, tile_reg},
                                                            {"one launch dma3 x4", true, true, tile_dma_x4}}};
// variant 0 is the default; variant 1 needs no LDS-DMA
// The variant behind each public index: tile shapes, numbers of buffers and
// thread orders that had indices of their own now share their staging's kernel.
static const int kNumIndex[2] = {9, 6};
static const int kVariantOf[2][9] = {{0, 1, 0, 0, 0, 2, 2, 2, 0}, {0, 1, 0, 0, 2, 2}};

struct TuneEntry {
  int choice[kLaunches];               // fastest variant, -1: no such tiles
  double ms[kLaunches][kMaxVariants];  // -1: not admissible
  bool one;                            // bulk and shell in one launch
};
struct TuneState {
  int overlap = 1;  // shell and bulk tiles in one launch
  int mode = 1;  // 0: defaults only; 1: tune each new region set
  int forced[2] = {-1, -1};
  std::map<std::string, TuneEntry> chosen;
};
static TuneState g_tune;

// the regions, and which stagings they admit: that depends on the whole level
// (its size, the boxes' offsets) and not on the regions alone
static std::string region_signature(const RegionLists &R, bool dma_ok, bool pairs_ok) {
  std::string s = dma_ok ? pairs_ok ? "x4" : "x1" : "reg";
  char buf[96];
  for (const auto *v : R.kind) {
    s += '|';
    if (!v) continue;
    for (const Z4cGeo &G : *v) {
      snprintf(buf, sizeof buf, "%d,%d,%d:%d-%d,%d-%d,%d-%d;", G.m, G.n, G.o, G.lo[0], G.hi[0], G.lo[1], G.hi[1],
               G.lo[2], G.hi[2]);
      s += buf;
    }
  }
  return s;
}

// times every admissible variant of one launch over the regions R
static int time_launch(int launch, const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, bool dma_ok,
                       bool pairs_ok, TuneEntry &te) {
  const Variant *V = kVariants[launch];
  hipEvent_t a, b;
  BH_HIP(hipEventCreate(&a));
  BH_HIP(hipEventCreate(&b));
  double best = 1e300;
  int e = BAMHIP_OK;
  for (int v = 0; v < kMaxVariants && e == BAMHIP_OK; v++) {
    if ((V[v].dma && !dma_ok) || (V[v].pairs && !pairs_ok)) continue;
    if ((e = V[v].fn(P, R, K, flag, stream()))) break;
    BH_HIP(hipEventRecord(a, stream()));
    for (int rep = 0; rep < 2 && e == BAMHIP_OK; rep++) e = V[v].fn(P, R, K, flag, stream());
    BH_HIP(hipEventRecord(b, stream()));
    BH_HIP(hipEventSynchronize(b));
    float ms = 0.0f;
    BH_HIP(hipEventElapsedTime(&ms, a, b));
    te.ms[launch][v] = ms / 2.0;
    if (te.ms[launch][v] < best) {
      best = te.ms[launch][v];
      te.choice[launch] = v;
    }
  }
  BH_HIP(hipEventDestroy(a));
  BH_HIP(hipEventDestroy(b));
  return e;
}

// The tuner's choices for a level's regions R (by launch): those kept, or (mode
// 1, outside capture, repeatable launches) those found by timing all variants on
// the library stream; *te stays null otherwise.
static int tuned(const Z4cPtrs &P, const RegionLists R[kLaunches], const bool has[kLaunches], const Z4cK &K, int *flag,
                 bool repeatable, bool dma_ok, bool pairs_ok, const TuneEntry **te) {
  const std::string sig = region_signature(R[kBoth], dma_ok, pairs_ok);
  auto it = g_tune.chosen.find(sig);
  if (it == g_tune.chosen.end()) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    BH_HIP(hipStreamIsCapturing(stream(), &cs));
    if (g_tune.mode == 0 || !repeatable || cs != hipStreamCaptureStatusNone) return BAMHIP_OK;
    TuneEntry n;
    for (int l = 0; l < kLaunches; l++) {
      n.choice[l] = -1;
      for (double &t : n.ms[l]) t = -1.0;
      if (!has[l]) continue;
      if (int e = time_launch(l, P, R[l], K, flag, dma_ok, pairs_ok, n)) return e;
    }
    n.one = has[kBoth] && n.ms[kBoth][n.choice[kBoth]] <=
                              n.ms[kBulk][n.choice[kBulk]] + n.ms[kShell][n.choice[kShell]];
    it = g_tune.chosen.emplace(sig, n).first;
  }
  *te = &it->second;
  return BAMHIP_OK;
}

// The tile and edge kernels of one RHS evaluation (plain, addlinear or fused
// RK4 stage, as K says) over all boxes of a level.  A fused stage rewrites u_c,
// so its kernels cannot be timed on the real lists: the tuner then times the
// plain RHS into scratch (when given) and the stage runs the chosen variant.
static int run_rhs(bamhip_level *lev, const Z4cPtrs &P, const Z4cK &K, bool check_finite, double *const *scratch) {
  int e;
  if (check_finite) set_int<<<1, 1, 0, stream()>>>(lev->d_flag, 0);
  const bool fast = (K.order_centered == 4 && K.order_advection == 4 && K.lopsided == 1 &&
                     (K.order_dissipation == 4 || K.order_dissipation == 0));
  // The tile kernel stores a field's result while later fields' operands are
  // still to be loaded, so an output may alias the operands of its own field
  // only; lists crossed any other way go through the per-point kernel, which
  // loads every operand before its first store.
  bool crossed = false;
  for (int v = 0; v < 25; v++)
    for (int w = 0; w < 25; w++)
      if (v != w)
        for (const double *o : {(const double *)P.r[v], (const double *)P.c[v], (const double *)P.cp[v]})
          crossed = crossed || (o && (o == P.a[w] || ((K.rk || K.addlinear) && o == P.p[w])));
  LevelTiles T;
  for (const DevBox &B : lev->boxes) {
    // a tile's points (at most 8 planes) within a 32-bit byte offset
    const bool near32 = (long)B.m * B.n * 8 * 8 < 0xfffffff0L;
    if ((e = plan_box(B, P, K, lev->d_flag, fast && !crossed && near32, T))) return e;
  }
  // repeated launches (tuning) give the same result unless the kernels write
  // what they read
  bool repeatable = !K.rk;
  for (int v = 0; v < 25 && repeatable; v++)
    for (int w = 0; w < 25; w++)
      if (P.r[v] == P.p[w]) repeatable = false;
  Z4cPtrs PT = P;  // lists the tuner runs on
  Z4cK KT = K;
  if (K.rk && scratch) {
    for (int v = 0; v < 25; v++) {
      PT.r[v] = scratch[v];
      PT.p[v] = P.u[v];
    }
    KT.rk = 0;
    KT.has_v = 0;
    KT.addlinear = 0;
    KT.c = 0.0;
    repeatable = true;
  }
  const bool dma_ok = (long)lev->npoints * 8 < (1L << 32);
  const RegionLists R[kLaunches] = {{{&T.bulk, nullptr, nullptr, nullptr}},
                                    {{nullptr, &T.sx, &T.sy, &T.sz}},
                                    {{&T.bulk, &T.sx, &T.sy, &T.sz}}};
  const bool bulk = !T.bulk.empty(), shell = !T.sx.empty() || !T.sy.empty() || !T.sz.empty();
  const bool has[kLaunches] = {bulk, shell, bulk && shell};
  // 16-byte units hold element pairs (x, x + 1) with x even in every box:
  // even box rows, box offsets and tile rows (first staged x = i0 - 3 even)
  bool pairs_ok = true;
  for (const auto *v : {&T.bulk, &T.sx, &T.sy, &T.sz})
    for (const Z4cGeo &G : *v) pairs_ok = pairs_ok && G.m % 2 == 0 && G.noffset % 2 == 0 && (G.lo[0] - HALO) % 2 == 0;
  const TuneEntry *te = nullptr;
  if (((bulk && g_tune.forced[kBulk] < 0) || (shell && g_tune.forced[kShell] < 0)) &&
      (e = tuned(PT, R, has, KT, lev->d_flag, repeatable, dma_ok, pairs_ok, &te)))
    return e;
  int v[kLaunches] = {-1, -1, -1};
  for (int l : {kBulk, kShell}) {
    if (!has[l]) continue;
    v[l] = g_tune.forced[l];
    if (v[l] < 0) {
      v[l] = te ? te->choice[l] : dma_ok ? 0 : 1;
      continue;
    }
    if (kVariants[l][v[l]].dma && !dma_ok)
      return set_error(BAMHIP_EINVAL, "z4c tile variant '%s' needs a level below 2^29 points", kVariants[l][v[l]].name);
    if (kVariants[l][v[l]].pairs && !pairs_ok)
      return set_error(BAMHIP_EINVAL, "z4c tile variant '%s' needs even box sizes and offsets", kVariants[l][v[l]].name);
  }
  if (has[kBoth] && g_tune.overlap) {
    if (te && g_tune.forced[kBulk] < 0 && g_tune.forced[kShell] < 0)
      v[kBoth] = te->one ? te->choice[kBoth] : -1;
    else if (v[kBulk] == v[kShell])
      v[kBoth] = v[kBulk];
  }
  if (v[kBoth] >= 0) v[kBulk] = v[kShell] = -1;
  for (int l = 0; l < kLaunches; l++) {
    if (v[l] < 0) continue;
    TimerScope t(l == kShell ? "z4_rhs_edge" : "z4_rhs");
    if ((e = kVariants[l][v[l]].fn(P, R[l], K, lev->d_flag, stream()))) return e;
  }
  if (check_finite) {
    int h = 0;
    BH_HIP(hipMemcpyAsync(&h, lev->d_flag, sizeof(int), hipMemcpyDeviceToHost, stream()));
    BH_HIP(hipStreamSynchronize(stream()));
    if (h) return set_error(BAMHIP_ENONFINITE, "bamhip_z4c_rhs: non-finite right-hand side on level %d", lev->l);
  }
  return BAMHIP_OK;
}

int z4c_rhs_impl(bamhip_level *lev, const bamhip_z4c_params *par, const int *unew, const int *upre, double c,
                 const int *ucur, bool check_finite) {
  if (!lev || !par) return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs: NULL argument");
  if (par->order_centered != 2 && par->order_centered != 4)
    return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs: order_centered=%d not implemented (2, 4)", par->order_centered);
  if (par->order_advection != 2 && par->order_advection != 4)
    return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs: order_advection=%d not implemented (2, 4)",
                     par->order_advection);
  if (par->advection_lopsided < 0 || par->advection_lopsided > 2)
    return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs: advection_lopsided=%d", par->advection_lopsided);
  if (par->order_dissipation != 0 && par->order_dissipation != 4)
    return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs: order_dissipation=%d not implemented (0, 4)",
                     par->order_dissipation);
  Z4cPtrs P;
  int e;
  if ((e = gather_ptrs(lev, ucur, 25, const_cast<double **>(P.u), "bamhip_z4c_rhs(ucur)"))) return e;
  if ((e = gather_ptrs(lev, unew, 25, P.r, "bamhip_z4c_rhs(unew)"))) return e;
  if (c != 0.0) {
    if ((e = gather_ptrs(lev, upre, 25, const_cast<double **>(P.p), "bamhip_z4c_rhs(upre)"))) return e;
  } else {
    for (int v = 0; v < 25; v++) P.p[v] = P.u[v];
  }
  for (int v = 0; v < 25; v++) {
    P.c[v] = nullptr;
    P.a[v] = nullptr;
    P.cp[v] = nullptr;
  }
  for (int v = 0; v < 25; v++)
    for (int w = 0; w < 25; w++)
      if (P.r[v] == P.u[w])
        return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs: unew[%d] aliases ucur[%d] (stencils need the old data)", v, w);
  // the stencil reach (3 with lop-sided advection, 4 with one-sided) must stay
  // inside every box
  for (const DevBox &B : lev->boxes)
    for (int f = 0; f < 6; f++)
      if (B.skip[f] < 1) return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs: box face %d has no flagged layer", f);
  const Z4cK K = make_k(par, c);
  return run_rhs(lev, P, K, check_finite, nullptr);
}

static int check_params(const bamhip_z4c_params *par, const char *what) {
  if (par->order_centered != 2 && par->order_centered != 4)
    return set_error(BAMHIP_EINVAL, "%s: order_centered=%d not implemented (2, 4)", what, par->order_centered);
  if (par->order_advection != 2 && par->order_advection != 4)
    return set_error(BAMHIP_EINVAL, "%s: order_advection=%d not implemented (2, 4)", what, par->order_advection);
  if (par->advection_lopsided < 0 || par->advection_lopsided > 2)
    return set_error(BAMHIP_EINVAL, "%s: advection_lopsided=%d", what, par->advection_lopsided);
  if (par->order_dissipation != 0 && par->order_dissipation != 4)
    return set_error(BAMHIP_EINVAL, "%s: order_dissipation=%d not implemented (0, 4)", what, par->order_dissipation);
  return BAMHIP_OK;
}

// One RK4 stage with the update fused into the RHS kernels' store: at every
// computed point accout = acc + wc RHS(src), when vout != NULL vout = base +
// wv RHS(src), and when copy != NULL copy = base.  src is read by the
// stencils, so no output may alias it; acc and base are read at the point
// only, so an output may alias them: of its own field in the tile kernel, which
// reads a field's operands before it stores that field (the accumulator read
// from the list the next state goes to, for one), of any field in the per-point
// kernel, which takes such lists and reads all operands first.  The outputs must
// differ from each other.  scratch (optional): 25 variables the tuner may use as a
// plain RHS output the first time a box set is seen; it must not alias an
// input (src, acc, base).
int z4c_rhs_rk4_impl(bamhip_level *lev, const bamhip_z4c_params *par, const int *src, const int *acc,
                     const int *accout, const int *base, const int *vout, const int *copy, double wc, double wv,
                     const int *scratch) {
  if (!lev || !par || !src || !acc || !accout || !base)
    return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs_rk4_stage: NULL argument");
  int e;
  if ((e = check_params(par, "bamhip_z4c_rhs_rk4_stage"))) return e;
  Z4cPtrs P;
  if ((e = gather_ptrs(lev, src, 25, const_cast<double **>(P.u), "bamhip_z4c_rhs_rk4_stage(src)"))) return e;
  if ((e = gather_ptrs(lev, acc, 25, const_cast<double **>(P.a), "bamhip_z4c_rhs_rk4_stage(acc)"))) return e;
  if ((e = gather_ptrs(lev, accout, 25, P.c, "bamhip_z4c_rhs_rk4_stage(accout)"))) return e;
  if ((e = gather_ptrs(lev, base, 25, const_cast<double **>(P.p), "bamhip_z4c_rhs_rk4_stage(base)"))) return e;
  if (vout) {
    if ((e = gather_ptrs(lev, vout, 25, P.r, "bamhip_z4c_rhs_rk4_stage(vout)"))) return e;
  } else {
    for (int v = 0; v < 25; v++) P.r[v] = nullptr;
  }
  if (copy) {
    if ((e = gather_ptrs(lev, copy, 25, P.cp, "bamhip_z4c_rhs_rk4_stage(copy)"))) return e;
  } else {
    for (int v = 0; v < 25; v++) P.cp[v] = nullptr;
  }
  for (int v = 0; v < 25; v++)
    for (int w = 0; w < 25; w++) {
      const double *outs[3] = {P.c[v], P.r[v], P.cp[v]}, *outw[3] = {P.c[w], P.r[w], P.cp[w]};
      for (int x = 0; x < 3; x++) {
        if (!outs[x]) continue;
        if (outs[x] == P.u[w])
          return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs_rk4_stage: an output list aliases src");
        for (int y = 0; y < 3; y++)
          if (y != x && outs[x] == outw[y])
            return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs_rk4_stage: the output lists alias each other");
      }
    }
  for (const DevBox &B : lev->boxes)
    for (int f = 0; f < 6; f++)
      if (B.skip[f] < 1)
        return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs_rk4_stage: box face %d has no flagged layer", f);
  double *scr[BAMHIP_Z4C_NVARS];
  if (scratch) {
    if ((e = gather_ptrs(lev, scratch, 25, scr, "bamhip_z4c_rhs_rk4_stage(scratch)"))) return e;
    for (int v = 0; v < 25; v++)
      for (int w = 0; w < 25; w++)
        if (scr[v] == P.u[w] || scr[v] == P.a[w] || scr[v] == P.p[w])
          return set_error(BAMHIP_EINVAL, "bamhip_z4c_rhs_rk4_stage: scratch aliases an input list");
  }
  Z4cK K = make_k(par, 0.0);
  K.rk = 1;
  K.has_v = vout ? 1 : 0;
  K.has_cp = copy ? 1 : 0;
  K.wc = wc;
  K.wv = wv;
  return run_rhs(lev, P, K, lev->check_mode != 0, scratch ? scr : nullptr);
}

}  // namespace bamhip

extern "C" int bamhip_z4c_rhs_rk4_stage(bamhip_level *lev, const bamhip_z4c_params *par, const int *src,
                                        const int *acc, const int *accout, const int *base, const int *vout,
                                        const int *copy, double wc, double wv, const int *scratch) {
  return bamhip::z4c_rhs_rk4_impl(lev, par, src, acc, accout, base, vout, copy, wc, wv, scratch);
}

extern "C" int bamhip_z4c_rhs(bamhip_level *lev, const bamhip_z4c_params *par, const int *unew, const int *upre,
                              double c, const int *ucur) {
  return bamhip::z4c_rhs_impl(lev, par, unew, upre, c, ucur, lev ? lev->check_mode != 0 : true);
}

extern "C" int bamhip_z4c_tune_mode(int mode) {
  if (mode != 0 && mode != 1) return bamhip::set_error(BAMHIP_EINVAL, "bamhip_z4c_tune_mode: mode %d (0, 1)", mode);
  const int old = bamhip::g_tune.mode;
  bamhip::g_tune.mode = mode;
  return old;
}

extern "C" int bamhip_z4c_set_overlap(int on) {
  const int old = bamhip::g_tune.overlap;
  bamhip::g_tune.overlap = on != 0;
  return old;
}

extern "C" int bamhip_z4c_set_xcd_map(int on) {
  const int old = bamhip::g_xcd_map;
  bamhip::g_xcd_map = on != 0;
  return old;
}

extern "C" int bamhip_z4c_tune_clear(void) {
  bamhip::g_tune.chosen.clear();
  return BAMHIP_OK;
}

extern "C" int bamhip_z4c_variant_count(int kind) {
  if (kind != 0 && kind != 1) return bamhip::set_error(BAMHIP_EINVAL, "bamhip_z4c_variant_count: kind %d", kind);
  return bamhip::kNumIndex[kind];
}

extern "C" const char *bamhip_z4c_variant_name(int kind, int idx) {
  if (kind != 0 && kind != 1) return nullptr;
  if (idx < 0 || idx >= bamhip::kNumIndex[kind]) return nullptr;
  return bamhip::kVariants[kind][bamhip::kVariantOf[kind][idx]].name;
}

extern "C" int bamhip_z4c_force_variant(int kind, int idx) {
  if (kind != 0 && kind != 1) return bamhip::set_error(BAMHIP_EINVAL, "bamhip_z4c_force_variant: kind %d", kind);
  if (idx < -1 || idx >= bamhip::kNumIndex[kind])
    return bamhip::set_error(BAMHIP_EINVAL, "bamhip_z4c_force_variant: variant %d of %d", idx,
                             bamhip::kNumIndex[kind]);
  bamhip::g_tune.forced[kind] = idx < 0 ? -1 : bamhip::kVariantOf[kind][idx];
  return BAMHIP_OK;
}

extern "C" int bamhip_z4c_tune_report(char *buf, int len) {
  using namespace bamhip;
  std::string s;
  char line[160];
  for (const auto &kv : g_tune.chosen) {
    const TuneEntry &te = kv.second;
    // the launches of a line, the ones that run first
    const std::vector<int> one = {kBoth}, two = {kBulk, kShell};
    for (const auto *ls : te.one ? std::initializer_list<const std::vector<int> *>{&one, &two}
                                 : std::initializer_list<const std::vector<int> *>{&two, &one}) {
      std::string name, times;
      for (int l : *ls) {
        if (te.choice[l] < 0) continue;
        name += (name.empty() ? "" : ", ") + std::string(kVariants[l][te.choice[l]].name);
        for (int v = 0; v < kMaxVariants; v++) {
          snprintf(line, sizeof line, " %s=%.4fms", kVariants[l][v].name, te.ms[l][v]);
          times += line;
        }
      }
      if (name.empty()) continue;
      snprintf(line, sizeof line, " <- %zu regions:", (size_t)std::count(kv.first.begin(), kv.first.end(), ';'));
      s += name + line + times + '\n';
    }
  }
  if (buf && len > 0) {
    const int n = (int)std::min<size_t>(s.size(), (size_t)len - 1);
    memcpy(buf, s.data(), n);
    buf[n] = '\0';
  }
  return (int)s.size() + 1;
}
