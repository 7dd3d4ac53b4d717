// z4c_tile.h -- the tile kernel of the Z4c right-hand side, shared by the
// files that instantiate it (z4c_tile_*.hip) and the host side that plans and
// launches it (z4c_rhs.hip).
#pragma once

#include <algorithm>
#include <type_traits>
#include <utility>
#include <vector>

#include "bamhip_internal.h"

// Contraction of a*b + c into an FMA only within one source expression: the
// fused operations are then fixed by the source, not by per-kernel backend
// choices, so every instantiation of the tile kernel (tile shape, staging,
// register budget) rounds identically and gives bitwise the same RHS.
#pragma clang fp contract(on)

// compile-time loop: f(integral_constant<int, I>) for I = 0..N-1; used for
// loops whose body holds a barrier, which the compiler does not unroll, so
// that per-field arrays keep constant indices and stay in registers
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

namespace bamhip {

// u: the state the stencils read; r: output (the RHS, unew = upre + c RHS, or
// in an RK4 stage the next stage's state); p: upre, or the RK4 step's start
// state in a stage.  In an RK4 stage (read and written at the point only):
// a: the accumulator read, c: the accumulator written (c = a + wc RHS), cp:
// where the start state p is copied to (or unused).
struct Z4cPtrs {
  const double *u[BAMHIP_Z4C_NVARS];
  double *r[BAMHIP_Z4C_NVARS];
  const double *p[BAMHIP_Z4C_NVARS];
  double *c[BAMHIP_Z4C_NVARS];
  const double *a[BAMHIP_Z4C_NVARS];
  double *cp[BAMHIP_Z4C_NVARS];
};

struct Z4cGeo {
  int m, n, o;      // box points
  long noffset;
  int lo[3], hi[3]; // computed index range [lo, hi] per direction
  long sj, sk;      // strides (di = 1)
  double h[3], ih[3];
  double i12h[3], i12hh[3], i144hh[3];  // 4th order: 1/(12h), 1/(12h^2), mixed 1/(144 ha hb) (xy, xz, yz)
  double i2h[3], ihh[3], i4hh[3];       // 2nd order: 1/(2h), 1/h^2, mixed 1/(4 ha hb)
  int edge_only;    // Edge kernel: skip points that the bulk kernel computes
};

struct Z4cK {
  int order_centered, order_advection, lopsided, order_dissipation;
  double dissfactor, kappa1, kappa2, zeroThetaRHS;
  int subtractA, normalizedetg;
  double oploglapse, oploglapse2, oplogwithshift, harmoniclapse, lapseharmonicf;
  double gamma0factor, gamma2factor, withGadv, withShiftadv, withBadv, withB;
  double shiftalphapower, shiftgammacoeff, shiftdriver;
  double chiDivFloor, chipsipower, oocp;  // oocp = 1 / chipsipower
  double c;
  int addlinear;
  // RK4 stage (rk.c:231-252) fused into the store: c = a + wc RHS, when
  // has_v r = p + wv RHS, when has_cp cp = p
  int rk, has_v, has_cp;
  double wc, wv;
};

// scheduling fence: keeps the machine scheduler from hoisting the loads of
// later derivative groups above earlier ones, which would keep hundreds of
// FP64 stencil values live at once and spill
#define BH_PHASE() __builtin_amdgcn_sched_barrier(0)

// index of component (a,b) in xx xy xz yy yz zz storage; closed form (not
// recursive) so that it folds to a constant once the loops are unrolled and
// every tensor array stays in registers
__device__ __forceinline__ constexpr int sy(int a, int b) {
  return (a < b ? a : b) * (5 - (a < b ? a : b)) / 2 + (a < b ? b : a);
}
__device__ __forceinline__ constexpr int mixid(int a, int b) {  // xy=0 xz=1 yz=2
  return (a + b) - 1;
}

// ------------------------------------------------------- tile kernel (LDS)
// Output tile of TX x TY x TZ points per block (256 threads, one point per
// thread).  Each of the 25 grid functions is staged in turn into an LDS tile
// with a halo of 3 points (the reach of the lop-sided advection stencil), so
// every stencil neighbour is an immediate-offset ds_read_b64 from one
// per-thread LDS address.  The algebra is ordered by staged field: each
// field's derivatives, advection and dissipation are consumed as soon as the
// field is in LDS.  The bulk uses 16 x 4 x 4 tiles (long x rows for
// coalesced loads); the box-edge shell, two points thick, uses slabs of
// 2 x 16 x 8, 16 x 2 x 8 and 16 x 8 x 2 on the x, y and z faces.
constexpr int HALO = 3;
constexpr int NTHR = 256;
template <int TX_, int TY_, int TZ_>
struct Lay {
  static constexpr int TX = TX_, TY = TY_, TZ = TZ_;
  static constexpr int SX = TX + 2 * HALO, SY = TY + 2 * HALO, SZ = TZ + 2 * HALO;
  static constexpr int TILE = SX * SY * SZ;
  static constexpr int NLOAD = (TILE + NTHR - 1) / NTHR;
  static_assert(TX * TY * TZ == NTHR, "one point per thread");
  __device__ static void coords(int t, int &x, int &y, int &z) {
    x = t % TX;
    y = (t / TX) % TY;
    z = t / (TX * TY);
  }
};
using LBulk = Lay<16, 4, 4>;
// x faces: rows of 2 points.  (Rows padded from 8 to 10 doubles spread the lanes
// of a read phase over all banks, but take 98 KB of LDS, so one block per CU.)
using LSlabX = Lay<2, 16, 8>;
using LSlabY = Lay<16, 2, 8>;
using LSlabZ = Lay<16, 8, 2>;

// a thread's tile corner in the LDS tile of layout L (its point is at +HALO)
template <class L>
struct TP {
  const double *p;
};

template <int DX, int DY, int DZ, class L>
__device__ __forceinline__ double at(TP<L> T) {
  return T.p[(DX + HALO) + L::SX * ((DY + HALO) + L::SY * (DZ + HALO))];
}
// neighbour at offset o along direction A
template <int A, int O, class L>
__device__ __forceinline__ double ax(TP<L> T) {
  return at<(A == 0 ? O : 0), (A == 1 ? O : 0), (A == 2 ? O : 0)>(T);
}
// The seven points of one axis through the point, the inner ones also as odd
// and even pairs: d_k = f(k) - f(-k), s_k = f(k) + f(-k).
struct Line {
  double d1, d2, s1, s2;
  double p[3], m[3];  // f(k), f(-k)
};
template <int A, class L>
__device__ __forceinline__ Line t_line(TP<L> T) {
  const double m1 = ax<A, -1>(T), p1 = ax<A, 1>(T), m2 = ax<A, -2>(T), p2 = ax<A, 2>(T), m3 = ax<A, -3>(T),
               p3 = ax<A, 3>(T);
  return {p1 - m1, p2 - m2, p1 + m1, p2 + m2, {p1, p2, p3}, {m1, m2, m3}};
}
// Lop-sided advection, dissipation, first and second derivative along one
// axis from the same pairs.  The upwind row of w = beta/h is
//   w > 0: w/12 (-3 f(-1) - 10 f(0) + 18 f(1) - 6 f(2) + f(3)),
//   w < 0: its mirror image.
// The points that both rows use, f(-1) and f(1), enter as parts odd and even in
// the offset; of the outer ones the upwind side is selected, so the downwind
// ones, which the row leaves out, do not enter at all (through odd and even
// parts of their own they would cancel up to rounding only):
//   w/12 (21/2 d1) + |w|/12 (f(3) - 6 f(2) + 15/2 s1 - 10 f(0)), f(k) upwind.
// 13 FP64 operations and a select for advection and dissipation together,
// where the two one-sided rows took 17 and shared nothing with the derivatives.
template <int A>
__device__ __forceinline__ double l_adv(const Line &l, double f0, double w12) {
  const double p = l.p[2] - 6.0 * l.p[1], m = l.m[2] - 6.0 * l.m[1];
  const double up = w12 > 0.0 ? p : m;
  return w12 * (10.5 * l.d1) + fabs(w12) * ((up + 7.5 * l.s1) - 10.0 * f0);
}
template <int A>
__device__ __forceinline__ double l_ko(const Line &l, double f0, const Z4cGeo &G) {
  return ((l.s2 - 4.0 * l.s1) + 6.0 * f0) * G.ih[A];
}
template <int A>
__device__ __forceinline__ double l_d1(const Line &l, const Z4cGeo &G) {
  return (8.0 * l.d1 - l.d2) * G.i12h[A];
}
template <int A>
__device__ __forceinline__ double l_d2(const Line &l, double f0, const Z4cGeo &G) {
  return ((16.0 * l.s1 - l.s2) - 30.0 * f0) * G.i12hh[A];
}
// ---- stencils of the box-edge shell (bam_amr_loops_box.h:186-215,
// bam_amr_advection.h:90-146): a point one away from an edge uses order-2
// centred differences and order-2 advection rows, dissipation needs two or
// more points to every edge, and the advection row is the upwind one where it
// fits between the point and the edge and the centred one elsewhere.  All of
// it as coefficients set once per point and selects, so the shell reads the same
// neighbours at fixed LDS offsets as the bulk and has no branch (one inside a
// stage let the register allocator place copies of live values where only part
// of the wave was enabled).  What an order-2 derivative leaves out is selected
// away, not multiplied by 0: it may hold anything.  The advection takes one
// coefficient per neighbour, 0 for one that its row leaves out; a neighbour
// outside the box is read from a staging slot that holds 0 or box data.
//   order 4 (e = 1) / order 2 (e = 0):
//     first derivative  ((6 + 2 e) d1 - e d2) / (12 h)
//     second            ((12 + 4 e) s1 - e s2 - (24 + 6 e) f) / (12 h^2)
//     mixed             ((36 + 28 e) q11 + e (q22 - 8 (q12 + q21))) / (144 h h')
//     advection, w = beta / h, f(k) counted in the direction of w:
//       upwind   |w|/12 (-3 f(-1) - 10 f(0) + 18 f(1) - 6 f(2) + f(3)),  |w|/2 (-3 f(0) + 4 f(1) - f(2))
//       centred  |w|/12 (8 (f(1) - f(-1)) - (f(2) - f(-2))),             |w|/2 (f(1) - f(-1))
struct Sten {
  bool o4;                        // order 4, and dissipation on
  double c1, p1, p0, k1;          // the coefficients above: 6 + 2e, 12 + 4e, 24 + 6e, 36 + 28e
  double ap[3][3], am[3][3], a0;  // advection: coefficients of f(1..3) and f(-1..-3) per axis, and of f
};

// pos: distances (low, high) of the point to the box's edges per axis
__device__ __forceinline__ void set_sten(Sten &S, const int dl[3], const int dh[3], const double w12[3]) {
  int dmin = 1 << 30;
#pragma unroll
  for (int a = 0; a < 3; a++) dmin = min(dmin, min(dl[a], dh[a]));
  const bool o4 = S.o4 = dmin >= 2;
  S.c1 = o4 ? 8.0 : 6.0;
  S.p1 = o4 ? 16.0 : 12.0;
  S.p0 = o4 ? 30.0 : 24.0;
  S.k1 = o4 ? 64.0 : 36.0;
  S.a0 = 0.0;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const double aw = fabs(w12[a]);
    const bool pos = w12[a] > 0.0, up = (pos ? dh[a] : dl[a]) >= (o4 ? 3 : 2);
    const double f1 = aw * (o4 ? (up ? 18.0 : 8.0) : (up ? 24.0 : 6.0));
    const double f2 = aw * (o4 ? (up ? -6.0 : -1.0) : (up ? -6.0 : 0.0));
    const double f3 = aw * (o4 && up ? 1.0 : 0.0);
    const double b1 = aw * (o4 ? (up ? -3.0 : -8.0) : (up ? 0.0 : -6.0));
    const double b2 = aw * (o4 && !up ? 1.0 : 0.0);
    S.ap[a][0] = pos ? f1 : b1;
    S.ap[a][1] = pos ? f2 : b2;
    S.ap[a][2] = pos ? f3 : 0.0;
    S.am[a][0] = pos ? b1 : f1;
    S.am[a][1] = pos ? b2 : f2;
    S.am[a][2] = pos ? 0.0 : f3;
    S.a0 += aw * (up ? (o4 ? -10.0 : -18.0) : 0.0);
  }
}

// the four corner sums q11, q12 (one along A, two along B), q21, q22 of a
// mixed derivative: f(i,j) - f(-i,j) - f(i,-j) + f(-i,-j)
template <int A, int B, int I, int K, class L>
__device__ __forceinline__ double t_corner(TP<L> T) {
  constexpr int AX = I * (A == 0), AY = I * (A == 1), AZ = I * (A == 2);
  constexpr int BX = K * (B == 0), BY = K * (B == 1), BZ = K * (B == 2);
  return (at<AX + BX, AY + BY, AZ + BZ>(T) - at<-AX + BX, -AY + BY, -AZ + BZ>(T)) -
         (at<AX - BX, AY - BY, AZ - BZ>(T) - at<-AX - BX, -AY - BY, -AZ - BZ>(T));
}
template <bool SH, int A, int B, class L>
__device__ __forceinline__ double t_mixed(TP<L> T, const Z4cGeo &G, const Sten &S) {
  const double q11 = t_corner<A, B, 1, 1>(T), q12 = t_corner<A, B, 1, 2>(T), q21 = t_corner<A, B, 2, 1>(T),
               q22 = t_corner<A, B, 2, 2>(T);
  const double outer = q22 - 8.0 * (q12 + q21);
  if constexpr (SH) return ((S.o4 ? outer : 0.0) + S.k1 * q11) * G.i144hh[A + B - 1];
  return (outer + 64.0 * q11) * G.i144hh[A + B - 1];
}
// advection, dissipation, first and second derivative along one axis
template <bool SH, int A>
__device__ __forceinline__ double s_adv(const Line &l, double f0, double w12, const Sten &S) {
  if constexpr (SH)
    return S.ap[A][0] * l.p[0] + S.ap[A][1] * l.p[1] + S.ap[A][2] * l.p[2] + S.am[A][0] * l.m[0] +
           S.am[A][1] * l.m[1] + S.am[A][2] * l.m[2];
  return l_adv<A>(l, f0, w12);
}
template <bool SH, int A>
__device__ __forceinline__ double s_d1(const Line &l, const Z4cGeo &G, const Sten &S) {
  if constexpr (SH) return (S.c1 * l.d1 - (S.o4 ? l.d2 : 0.0)) * G.i12h[A];
  return l_d1<A>(l, G);
}
template <bool SH, int A>
__device__ __forceinline__ double s_d2(const Line &l, double f0, const Z4cGeo &G, const Sten &S) {
  if constexpr (SH) return ((S.p1 * l.s1 - (S.o4 ? l.s2 : 0.0)) - S.p0 * f0) * G.i12hh[A];
  return l_d2<A>(l, f0, G);
}

// What one staged field contributes at the point: its value f0, advection,
// dissipation sum and, as asked, gradient and second derivatives.
struct Fld {
  double f0, adv, ko;
};
template <bool SH, bool GRAD, bool HESS, class L>
__device__ __forceinline__ Fld field(TP<L> T, const Z4cGeo &G, const double w12[3], const Sten &S, double d[3],
                                     double h6[6]) {
  Fld F;
  F.f0 = ax<0, 0>(T);
  const Line x = t_line<0>(T);
  F.adv = s_adv<SH, 0>(x, F.f0, w12[0], S);
  if constexpr (SH) F.adv = F.adv + S.a0 * F.f0;
  F.ko = l_ko<0>(x, F.f0, G);
  if constexpr (GRAD) d[0] = s_d1<SH, 0>(x, G, S);
  if constexpr (HESS) h6[0] = s_d2<SH, 0>(x, F.f0, G, S);
  BH_PHASE();
  const Line y = t_line<1>(T);
  F.adv += s_adv<SH, 1>(y, F.f0, w12[1], S);
  F.ko += l_ko<1>(y, F.f0, G);
  if constexpr (GRAD) d[1] = s_d1<SH, 1>(y, G, S);
  if constexpr (HESS) h6[3] = s_d2<SH, 1>(y, F.f0, G, S);
  BH_PHASE();
  const Line z = t_line<2>(T);
  F.adv += s_adv<SH, 2>(z, F.f0, w12[2], S);
  F.ko = -(F.ko + l_ko<2>(z, F.f0, G));
  if constexpr (SH) F.ko = S.o4 ? F.ko : 0.0;
  if constexpr (GRAD) d[2] = s_d1<SH, 2>(z, G, S);
  if constexpr (HESS) {
    h6[5] = s_d2<SH, 2>(z, F.f0, G, S);
    BH_PHASE();
    h6[1] = t_mixed<SH, 0, 1>(T, G, S);
    BH_PHASE();
    h6[2] = t_mixed<SH, 0, 2>(T, G, S);
    BH_PHASE();
    h6[4] = t_mixed<SH, 1, 2>(T, G, S);
    BH_PHASE();
  }
  return F;
}

// Staging of one field into the LDS tile, software-pipelined: the global
// loads of the next field are issued into registers (NLOAD per thread, all
// in flight together) before the current field is computed, and written to
// LDS between two barriers at the start of the next stage.
// staging order of the 25 fields: beta^i, gt_ij, Gamma^i, chi, alpha, Khat,
// Theta, At_ij, B^i.  The shift's gradients come first and the curvature is
// complete after the lapse, so that nearly every field's right-hand side is
// final at the field's own stage and is stored there (see z4c_rhs_tile).
constexpr int STAGE_ORDER[25] = {19, 20, 21, 0, 1, 2, 3, 4, 5,  14, 15, 16, 6,
                                            18, 13, 17, 7, 8, 9, 10, 11, 12, 22, 23, 24};
// the field whose store operands stage s loads and whose result is final at
// its end, and the field whose result stage s stores (-1: none).  Gamma^i is
// final after Theta and leaves beside At_xx, At_xy, At_xz.
constexpr int STAGE_LOADS[25] = {19, 20, 21, 0,  1,  2,  3, 4, 5, -1, -1, -1, 6,
                                 18, 13, 17, 7,  8,  9,  10, 11, 12, 22, 23, 24};
constexpr int STAGE_STORES[25] = {-1, 19, 20, 21, 0,  1,  2, 3, 4, 5,  -1, -1, -1,
                                  6,  18, 13, 17, 7,  8,  9, 10, 11, 12, 22, 23};
constexpr int kGammaStage = 16;  // Gamma^c: operands at stage kGammaStage + c, stored one later
// result stores that stage s issues
constexpr int stage_nstores(int s) {
  return s < 0 || s > 24 ? 0 : (STAGE_STORES[s] >= 0 ? 1 : 0) + (s > kGammaStage && s <= kGammaStage + 3 ? 1 : 0);
}
// A wave's memory operations that may still be outstanding when it waits for
// its transfers of stage s's field, with each field's transfers (nper
// operations) issued `lead` stages ahead and `per` stores a result: the later
// fields' transfers and the stores of the stages since.  Loads, and the reloads
// of spilled registers, between them are not counted, which only waits for more.
constexpr int stage_outstanding(int s, int lead, int nper, int per) {
  int n = 0;
  for (int t = s - lead + 1; t < s; t++) n += (t + lead < 25 ? nper : 0) + per * stage_nstores(t);
  return n;
}

template <class L>
struct Stager {
  static constexpr int NLOAD = L::NLOAD;
  int goff[NLOAD];
  unsigned ok;      // bit k: slot k lies inside the tile and the box
  long cbase;       // linear index of the tile corner (i0-3, j0-3, k0-3); may lie before the box
  double pf[NLOAD];
  __device__ Stager(const Z4cGeo &G, int i0, int j0, int k0, int tid) {
    cbase = G.noffset + (i0 - HALO) + G.sj * (j0 - HALO) + G.sk * (k0 - HALO);
    ok = 0;
#pragma unroll
    for (int k = 0; k < NLOAD; k++) {
      const int idx = tid + k * NTHR;
      const int x = idx % L::SX, y = (idx / L::SX) % L::SY, z = idx / (L::SX * L::SY);
      const int gi = i0 - HALO + x, gj = j0 - HALO + y, gk = k0 - HALO + z;
      const bool in = idx < L::TILE && gi >= 0 && gj >= 0 && gk >= 0 && gi < G.m && gj < G.n && gk < G.o;
      goff[k] = in ? (int)(x + G.sj * y + G.sk * z) : 0;
      ok |= in ? (1u << k) : 0u;
    }
  }
  // slots outside the box are staged as 0; a stencil has coefficient 0 there or selects them away
  __device__ __forceinline__ void load(const double *__restrict__ f) {
#pragma unroll
    for (int k = 0; k < NLOAD; k++) pf[k] = (ok >> k & 1u) ? f[cbase + goff[k]] : 0.0;
  }
  __device__ __forceinline__ void commit(double *tile, int tid) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NLOAD; k++)
      if (tid + k * NTHR < L::TILE) tile[tid + k * NTHR] = pf[k];
    __syncthreads();
  }
};

// Staging through the LDS-DMA path: global_load_lds moves each field
// straight from HBM into one of NB LDS buffers (no registers, no ds_write), so
// NB - 1 fields are in flight while one is computed.  A wave's 64 lanes write
// 64 consecutive units of LDS (lane l -> unit l), so the tile is cut into
// chunks of 64 units, NPER per wave.  VEC = 1: a unit is one dword, the low
// (even unit) or high half of a tile element; VEC = 4: a unit is 16 bytes,
// the two tile elements (x, x + 1) with x even, which needs an even row
// length and 16-byte aligned pairs in HBM (checked by the host).  Slots of
// the tile outside the box load the nearest point of the box (a pair stays a
// pair), so that every staged value is box data: the shell's advection reads
// such slots with weight 0.
#define BH_LDS(p) ((__attribute__((address_space(3))) void *)(p))
template <class L, int NB, int VEC>
struct DmaStager {
  static_assert(VEC == 1 || VEC == 4, "dword or 16-byte units");
  static_assert(VEC == 1 || (L::SX % 2 == 0 && L::TX % 2 == 0), "16-byte units need even rows and tile steps");
  static constexpr int NW = NTHR / 64;
  static constexpr int NUNIT = VEC == 1 ? 2 * L::TILE : L::TILE / 2;
  static constexpr int NCH = (NUNIT + 63) / 64;
  static constexpr int NPER = (NCH + NW - 1) / NW;
  static constexpr int CHD = 64 * VEC / 2;      // doubles per chunk
  static constexpr int BUFD = NPER * NW * CHD;  // doubles per buffer, padded to whole chunks
  static_assert(NB >= 2 && NB <= 4 && (NB - 2) * NPER <= 63, "vmcnt range");
  unsigned boff[NPER];  // byte offset of each chunk's unit from the field's base
  int wave;
  __device__ DmaStager(const Z4cGeo &G, int i0, int j0, int k0, int tid) {
    const int lane = tid & 63;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
    for (int c = 0; c < NPER; c++) {
      const int d = (wave * NPER + c) * 64 + lane;
      const int e = VEC == 1 ? d >> 1 : 2 * d;
      const int x = e % L::SX, y = (e / L::SX) % L::SY, z = e / (L::SX * L::SY);
      const int gi = i0 - HALO + x, gj = j0 - HALO + y, gk = k0 - HALO + z;
      const bool in = e < L::TILE;
      // clamped into the box; for 16-byte units gi is even and so is the
      // box's row length, so the clamped pair is (0, 1) or (m - 2, m - 1)
      const int ci = min(max(gi, 0), G.m - (VEC == 1 ? 1 : 2)), cj = min(max(gj, 0), G.n - 1),
                ck = min(max(gk, 0), G.o - 1);
      const long el = in ? G.noffset + ci + G.sj * cj + G.sk * ck : G.noffset;
      boff[c] = (unsigned)(el * 8 + (VEC == 1 && in ? (d & 1) * 4 : 0));
    }
  }
  __device__ __forceinline__ void issue(const double *f, double *buf) const {
#pragma unroll
    for (int c = 0; c < NPER; c++) {
      const void *src = (const void *)((const char *)f + boff[c]);
      if constexpr (VEC == 1)
        __builtin_amdgcn_global_load_lds(src, BH_LDS(buf + (wave * NPER + c) * CHD), 4, 0, 0);
      else
        __builtin_amdgcn_global_load_lds(src, BH_LDS(buf + (wave * NPER + c) * CHD), 16, 0, 0);
    }
  }
};
// s_waitcnt vmcnt(n) lgkmcnt(0) (expcnt not waited), n a small constant
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N >= 0 && N <= 63, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}
// workgroup barrier without a memory fence (a fence would also wait for the
// LDS-DMA loads still in flight); the empty asm statements keep the compiler
// from moving memory accesses across it
__device__ __forceinline__ void bare_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Pin a value in registers at this point of the program: an empty volatile
// asm that reads and writes it.  Placed after each staged field, it keeps the
// compiler from sinking that field's arithmetic past the next stage's
// barrier, which would keep every staged tile's values live to the end of
// the kernel (and spill).
__device__ __forceinline__ void pin(double &x) { asm volatile("" : "+v"(x)); }
template <int N>
__device__ __forceinline__ void pin(double (&a)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++) pin(a[i]);
}

// Regions of one launch: index ranges [lo, hi] of boxes of a level (bulk
// regions, and slabs of the box-edge shell), each with its box geometry, and
// the first block of each region.
// The grid spacing constants are common to the regions of one launch (one
// level), so a region carries only integer geometry.
constexpr int kMaxRegions = 32;
// kind: the tile layout, 0 bulk, 1 to 3 slabs normal to x, y and z
struct RegionGeo {
  long noffset;
  int m, n, o;
  int lo[3], hi[3];
  int kind;
};
struct Spacing {
  double h[3], ih[3], i12h[3], i12hh[3], i144hh[3];
};
struct TileJobs {
  int n;
  int blk0[kMaxRegions + 1];  // first tile of each region; blk0[n] = number of tiles
  int nshell;                 // tiles of the slabs, which come before the bulk's
  int xcd;                    // 1: XCD-aware numbering of the tiles (grid padded)
  RegionGeo reg[kMaxRegions];
  Spacing sp;
};
// The lists' pointers in the order the stages use them, so that a stage's
// scalar loads are one contiguous record: the field whose transfer it starts,
// the operands it loads and the outputs it stores.
struct StagePtrs {
  const double *issue, *a, *p;
  double *c, *r, *cp;
};
struct TilePtrs {
  StagePtrs st[26];       // st[25]: the last result's outputs
  StagePtrs gam[3];       // Gamma^i: operands and outputs
  const double *u[BAMHIP_Z4C_NVARS];  // by field, for the point values
};
struct TileArgs {
  TilePtrs P;
  TileJobs J;
  Z4cK K;
  int *flag;
};
static_assert(sizeof(TileArgs) <= 4096, "arguments of the tile kernel within 4 KiB");

// What a result is stored as: the right-hand side; upre + c RHS with the
// projection; or an RK4 stage's accumulator with (V) the next state and (C)
// the copy of the start state.
template <bool RK_, bool ADD_, bool V_, bool C_>
struct StoreAs {
  static constexpr bool RK = RK_, ADD = ADD_, V = V_, C = C_;
  static constexpr int per = RK_ ? 1 + (V_ ? 1 : 0) + (C_ ? 1 : 0) : 1;  // stores per result
};

// Store at a 32-bit offset from a block-uniform base through a buffer
// descriptor whose range ends at 2^32 - 16: a thread without a point of its own
// takes an offset past it, and its store is dropped.  So no stage has a branch
// on the thread, every wave issues the same memory operations (the waits count
// them), and the kernel body is one basic block.
constexpr unsigned kNoStore = 0xfffffff8u;
__device__ __forceinline__ void store_at(double *base, unsigned off, double x) {
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, x),
                                        __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)0xfffffff0u, 0x00020000),
                                        (int)off, 0, 0);
}

// unew = upre + c RHS at one point, after its raw values have been stored:
// trace removal and det normalisation (z4_rhs_movpunc_N.m:446-467).  The point's
// own thread stored them, so it reads them back in program order.
__device__ __forceinline__ void project_point(const TilePtrs &P, const Z4cK &K, long q) {
  double ng[6], nA[6];
#pragma unroll
  for (int c = 0; c < 6; c++) {
    ng[c] = P.st[4 + c].r[q];   // outputs of gt_ij and At_ij (STAGE_STORES)
    nA[c] = P.st[17 + c].r[q];
  }
  const double a0 = ng[3] * ng[5] - ng[4] * ng[4], a1 = ng[2] * ng[4] - ng[1] * ng[5];
  const double a2 = ng[1] * ng[4] - ng[2] * ng[3], a3 = ng[0] * ng[5] - ng[2] * ng[2];
  const double a4 = ng[1] * ng[2] - ng[0] * ng[4], a5 = ng[0] * ng[3] - ng[1] * ng[1];
  const double detnginv = 1.0 / (ng[0] * a0 + ng[1] * a1 + ng[2] * a2);
  if (K.subtractA) {
    const double trA =
        detnginv * (a0 * nA[0] + a3 * nA[3] + a5 * nA[5] + 2.0 * (a1 * nA[1] + a2 * nA[2] + a4 * nA[4]));
#pragma unroll
    for (int c = 0; c < 6; c++) P.st[17 + c].r[q] = nA[c] - (trA / 3.0) * ng[c];
  }
  if (K.normalizedetg) {
    const double aux = pow(detnginv, 1.0 / 3.0);
#pragma unroll
    for (int c = 0; c < 6; c++) P.st[4 + c].r[q] = aux * ng[c];
  }
}

// SH = false: every point of the regions is >= 3 from each edge (standard
// stencils).  SH = true: the regions are slabs of the box-edge shell; only
// points closer than 3 to an edge are computed, with the per-point rules of
// Sten.
template <class L, int NB, int VEC>
struct StageBuf {  // LDS doubles of the staging buffers
  static constexpr int n = NB * DmaStager<L, NB, VEC>::BUFD;
};
template <class L, int VEC>
struct StageBuf<L, 0, VEC> {
  static constexpr int n = L::TILE;
};

// LDS of a block: the staging buffers, then per thread six values of the
// Gamma^i stages that are needed again at the end.  One array: with two, the
// compiler tells LDS objects apart and waits for every transfer before each
// stage's reads.
template <class L, int NB, int VEC>
constexpr int tile_lds() {
  return StageBuf<L, NB, VEC>::n + 6 * NTHR;
}

// One tile, number b of region r.  NB = 0: one LDS tile, staged through
// registers (Stager); NB >= 2: NB LDS buffers filled by the LDS-DMA path
// (DmaStager).
template <class L, bool SH, class ST, int NB, int VEC>
__device__ __forceinline__ void tile_body(double *tile, int r, int b) {
  // the kernel's arguments, read anew by each layout's body: shared, the
  // compiler loads them all ahead of the branch on the layout and spills
  // hundreds of scalar registers
  auto *ka = (const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(ka));
  const TileArgs &args = *(const TileArgs *)ka;
  const TilePtrs &P = args.P;
  const TileJobs &J = args.J;
  const Z4cK &K = args.K;
  double *const park = tile + StageBuf<L, NB, VEC>::n;
  // copies: indexing the argument array by r through a reference would stage it in scratch
  const RegionGeo Rg = J.reg[r];
  Z4cGeo G;
  G.m = Rg.m;
  G.n = Rg.n;
  G.o = Rg.o;
  G.noffset = Rg.noffset;
  G.sj = Rg.m;
  G.sk = (long)Rg.m * Rg.n;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    G.lo[a] = Rg.lo[a];
    G.hi[a] = Rg.hi[a];
    G.h[a] = J.sp.h[a];
    G.ih[a] = J.sp.ih[a];
    G.i12h[a] = J.sp.i12h[a];
    G.i12hh[a] = J.sp.i12hh[a];
    G.i144hh[a] = J.sp.i144hh[a];
  }
  G.edge_only = 0;
  const int ntx = (G.hi[0] - G.lo[0] + L::TX) / L::TX, nty = (G.hi[1] - G.lo[1] + L::TY) / L::TY;
  const int tid = (int)threadIdx.x;
  int tx, ty, tz;
  L::coords(tid, tx, ty, tz);
  const int i0 = G.lo[0] + (b % ntx) * L::TX, j0 = G.lo[1] + ((b / ntx) % nty) * L::TY,
            k0 = G.lo[2] + (b / (ntx * nty)) * L::TZ;
  const int i = i0 + tx, j = j0 + ty, k = k0 + tz;
  bool active = (i <= G.hi[0] && j <= G.hi[1] && k <= G.hi[2]);
  // positions past hi (padding threads, never stored) are clamped to hi, so
  // that their stencil reach stays within the halo
  const int ci = min(i, G.hi[0]), cj = min(j, G.hi[1]), ck = min(k, G.hi[2]);
  const int dl[3] = {ci, cj, ck}, dh[3] = {G.m - 1 - ci, G.n - 1 - cj, G.o - 1 - ck};
  if constexpr (SH) {
    int dmin = 1 << 30;
#pragma unroll
    for (int a = 0; a < 3; a++) dmin = min(dmin, min(dl[a], dh[a]));
    active = active && dmin <= 2;
  }
  // the point as the block's first point (uniform) and a 32-bit byte offset
  const long qb = G.noffset + i0 + G.sj * j0 + G.sk * k0;
  const unsigned loc = (unsigned)((tx + (int)G.m * ty) * 8) + (unsigned)tz * (unsigned)(G.m * G.n) * 8u;
  const unsigned ldo = active ? loc : 0u, sto = active ? loc : kNoStore;
  auto ld = [&](const double *f) { return *(const double *)((const char *)(f + qb) + ldo); };
  auto sv = [&](double *f, double x) { store_at(f + qb, sto, x); };
  const int toff = tx + L::SX * (ty + L::SY * tz);
  TP<L> T{tile + toff};
  const double *const *u = P.u;

  // the first fields' transfers go out before the point values are loaded,
  // so that a block waits for one round trip to HBM at its start, not two
  using St = typename std::conditional<NB == 0, Stager<L>, DmaStager<L, (NB == 0 ? 2 : NB), VEC>>::type;
  St st(G, i0, j0, k0, tid);
  constexpr int NBUF = NB == 0 ? 1 : NB, LEAD = NB == 0 ? 1 : NB - 1;
  constexpr int BUFD = StageBuf<L, NB, VEC>::n / NBUF;
  if constexpr (NB == 0) {
    st.load(u[STAGE_ORDER[0]]);
  } else {
#pragma unroll
    for (int p = 0; p < NB - 1; p++) st.issue(u[STAGE_ORDER[p]], tile + p * BUFD);
  }

  // Metric, shift and lapse at the point: needed from the first stage on.
  // Every other value is read from its field's staged tile, or loaded a stage
  // before its use.  (A thread without a point of its own loads the block's
  // first point; its results are not stored.)
  const bool withB = K.withB != 0.0;
  double g[6], w12[3];
  double pv[2];  // point values loaded a stage before their use
#pragma unroll
  for (int c = 0; c < 6; c++) g[c] = ld(u[c]);
#pragma unroll
  for (int a = 0; a < 3; a++) w12[a] = ld(u[19 + a]) * G.ih[a] * (1.0 / 12.0);
  const double alpha = ld(u[18]);
  pv[0] = ld(withB ? u[22] : u[14]);
  Sten S{};
  if constexpr (SH) set_sten(S, dl, dh, w12);
  // Memory traffic of a stage, in the order it is issued right after the
  // stage's barrier: the loads of this stage's store operands (an RK4 stage's
  // accumulator and start state, or upre) and of the point values the next
  // stage uses; the transfer of a later field; the stores of the stage before
  // (a field's results leave one stage after they are final).  A wave's memory
  // operations complete in order, so the next stage's wait for its own field
  // then covers the loads, and neither the transfer just begun nor the stores
  // are ever waited for within a stage of being issued.  (With the loads after
  // the transfer, or the stores before it, each stage waited a memory round
  // trip: 3.4 to 4.4 ms on 192^3.)
  struct Out {
    double x, a, p;
  };
  Out E[2] = {}, Q[2] = {};  // by the parity of the stage; Q: a stage's second result
  int bad = 0;               // a right-hand side of this point is not finite
  auto fetch = [&](Out &o, const StagePtrs &sp) {
    if constexpr (ST::RK) o.a = ld(sp.a);
    if constexpr (ST::ADD || ST::V || ST::C) o.p = ld(sp.p);
  };
  auto emit = [&](Out &o, double x) {
    // settled at once: left to the end, the values would stay live (and spill)
    bad |= isfinite(x) ? 0 : 1;
    asm volatile("" : "+v"(bad));
    o.x = x;
    pin(o.x);
  };
  auto flush = [&](const Out &o, const StagePtrs &sp) {
    if constexpr (ST::RK) {
      sv(sp.c, o.a + K.wc * o.x);
      if constexpr (ST::V) sv(sp.r, o.p + K.wv * o.x);
      if constexpr (ST::C) sv(sp.cp, o.p);
    } else if constexpr (ST::ADD) {
      sv(sp.r, o.p + K.c * o.x);
    } else {
      sv(sp.r, o.x);
    }
  };
  // stage s: make its field visible in LDS, load the operands of its result
  // and the next stage's point values (pre), start the transfer of a later
  // field and store the result of the stage before
  auto advance = [&](auto S_, auto pre) {
    constexpr int s = decltype(S_)::value;
    if constexpr (NB == 0) {
      st.commit(tile, tid);
    } else {
      // this wave's loads of the field are done; the barrier makes every
      // wave's done
      constexpr int out = stage_outstanding(s, LEAD, St::NPER, ST::per);
      wait_vm_lgkm0<(out <= 63 ? out : 63)>();
      bare_barrier();
    }
    if constexpr (STAGE_LOADS[s] >= 0) fetch(E[s % 2], P.st[s]);
    if constexpr (s >= kGammaStage && s < kGammaStage + 3) fetch(Q[s % 2], P.gam[s - kGammaStage]);
    pre();
    asm volatile("" ::: "memory");
    if constexpr (s + LEAD < 25) {
      if constexpr (NB == 0)
        st.load(P.st[s].issue);
      else  // the buffer held the field before this one, whose reads every wave completed before the barrier
        st.issue(P.st[s].issue, tile + ((s + LEAD) % NBUF) * BUFD);
    }
    if constexpr (NB != 0) T.p = tile + (s % NBUF) * BUFD + toff;
    asm volatile("" ::: "memory");
    if constexpr (STAGE_STORES[s] >= 0) flush(E[(s + 1) % 2], P.st[s]);
    if constexpr (s > kGammaStage && s <= kGammaStage + 3) flush(Q[(s + 1) % 2], P.gam[s - kGammaStage - 1]);
  };
  auto nothing = [] {};
  // the powers, while few registers are in use: psi^-4 = chi^(-4/chipsipower),
  // chi itself in the usual chi = psi^-4 (and not a number below 0, where the
  // power has no value), and the driver's alpha^p
  double psim4 = ld(u[6]), betaF = 0.0;
  psim4 = (psim4 < K.chiDivFloor) ? K.chiDivFloor : psim4;
  if (K.chipsipower != -4.0) psim4 = exp(-4.0 * K.oocp * log(psim4));
  else psim4 = (psim4 < 0.0) ? __builtin_nan("") : psim4;
  if (withB)
    betaF = K.shiftgammacoeff * (K.shiftalphapower == 0.0   ? 1.0
                                 : K.shiftalphapower == 1.0 ? alpha
                                                            : pow(alpha, K.shiftalphapower));
  // the division also where its coefficient is 0: no value at alpha = 3
  const double fa0 = K.oploglapse * K.lapseharmonicf + K.oploglapse2 * (8.0 / 3.0) / (3.0 - alpha);
  double fa = (fa0 + K.harmoniclapse * alpha) * alpha;
  pin(psim4);
  pin(betaF);
  pin(fa);
  const bool ko = (K.order_dissipation == 4);
  const double eps = ko ? K.dissfactor : 0.0;

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
  auto trace = [&](const double *t6) {
    return ig[0] * t6[0] + ig[3] * t6[3] + ig[5] * t6[5] + 2.0 * (ig[1] * t6[1] + ig[2] * t6[2] + ig[4] * t6[4]);
  };
  auto contract = [&](const double *x, const double *y) {
    return ig[0] * x[0] * y[0] + ig[3] * x[1] * y[1] + ig[5] * x[2] * y[2] + ig[1] * (x[0] * y[1] + x[1] * y[0]) +
           ig[2] * (x[0] * y[2] + x[2] * y[0]) + ig[4] * (x[1] * y[2] + x[2] * y[1]);
  };
  double none3[3], none6[6];

  // ---- shift: d_a beta^b, g^bc d_b d_c beta^a, (1/3) d_a d_c beta^c
  // rG accumulates the right-hand side of Gamma^a
  double db[3][3], rG[3];  // db[a][b] = d_a beta^b
  {
    double ootd[3];
    static_for<3>([&](auto I_) {
      constexpr int c = decltype(I_)::value;
      const double drive = pv[0];
      advance(I_, [&] {
        if constexpr (c < 2) pv[0] = ld(withB ? u[23 + c] : u[15 + c]);
        else pv[0] = ld(u[7]);
      });
      double d[3], h6[6];
      const Fld F = field<SH, true, true>(T, G, w12, S, d, h6);
#pragma unroll
      for (int a = 0; a < 3; a++) {
        db[a][c] = d[a];
        pin(db[a][c]);
      }
      rG[c] = trace(h6);
#pragma unroll
      for (int a = 0; a < 3; a++) ootd[a] = (c == 0 ? 0.0 : ootd[a]) + (1.0 / 3.0) * h6[sy(a, c)];
      pin(rG[c]);
      pin(ootd);
      const double r = K.withShiftadv * F.adv + eps * F.ko;
      emit(E[c % 2], r + (withB ? (K.gamma2factor + K.gamma0factor * betaF) * drive : drive - K.shiftdriver * F.f0));
    });
#pragma unroll
    for (int a = 0; a < 3; a++)
      rG[a] += ig[sy(a, 0)] * ootd[0] + ig[sy(a, 1)] * ootd[1] + ig[sy(a, 2)] * ootd[2];
    pin(rG);
  }
  const double divbeta = db[0][0] + db[1][1] + db[2][2];
  const double tdb = (2.0 / 3.0) * divbeta;

  // ---- conformal metric: first derivatives, Laplacian part of Ricci
  double R[6];  // Ricci accumulators (conformal + phi part)
  double Gu[3][6];
  double lA[6] = {};  // the shift's part of the right-hand side of At_ij, summed component by component
  {
    double dg[3][6], Gfg[3];
    static_for<6>([&](auto I_) {
      constexpr int ab = decltype(I_)::value;
      constexpr int a = ab < 3 ? 0 : (ab < 5 ? 1 : 2), b = ab < 3 ? ab : (ab < 5 ? ab - 2 : 2);
      const double Aab = pv[0];
      advance(std::integral_constant<int, 3 + ab>{}, [&] {
        if constexpr (ab < 5) pv[0] = ld(u[8 + ab]);
      });
      double d[3], h6[6];
      const Fld F = field<SH, true, true>(T, G, w12, S, d, h6);
#pragma unroll
      for (int e = 0; e < 3; e++) {
        dg[e][ab] = d[e];
        pin(dg[e][ab]);
      }
      R[ab] = -0.5 * trace(h6);
      pin(R[ab]);
      double lg = -g[ab] * tdb;
#pragma unroll
      for (int c = 0; c < 3; c++) lg += db[a][c] * g[sy(b, c)] + db[b][c] * g[sy(a, c)];
      emit(E[(3 + ab) % 2], F.adv + eps * F.ko + (lg - 2.0 * alpha * Aab));
      // lA_ij = d_i beta^c A_cj + d_j beta^c A_ci - 2/3 A_ij d_c beta^c: the terms with A_ab
#pragma unroll
      for (int e = 0; e < 3; e++) {
        lA[sy(e, b)] += (e == b ? 2.0 : 1.0) * db[e][a] * Aab;
        if (a != b) lA[sy(e, a)] += (e == a ? 2.0 : 1.0) * db[e][b] * Aab;
      }
      lA[ab] -= tdb * Aab;
      pin(lA);
    });
    // Christoffels
    double Gd[3][6];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = a; b < 3; b++)
          Gd[c][sy(a, b)] = 0.5 * (dg[a][sy(b, c)] + dg[b][sy(a, c)] - dg[c][sy(a, b)]);
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
      for (int ab = 0; ab < 6; ab++)
        Gu[c][ab] = ig[sy(c, 0)] * Gd[0][ab] + ig[sy(c, 1)] * Gd[1][ab] + ig[sy(c, 2)] * Gd[2][ab];
#pragma unroll
    for (int a = 0; a < 3; a++)
      Gfg[a] = ig[0] * Gu[a][0] + ig[3] * Gu[a][3] + ig[5] * Gu[a][5] +
               2.0 * (ig[1] * Gu[a][1] + ig[2] * Gu[a][2] + ig[4] * Gu[a][4]);
#pragma unroll
    for (int a = 0; a < 3; a++)
      rG[a] += Gfg[a] * (tdb + 2.0 * alpha * K.kappa1) -
               (Gfg[0] * db[0][a] + Gfg[1] * db[1][a] + Gfg[2] * db[2][a]);
    pin(rG);
    pin(Gu[0]);
    pin(Gu[1]);
    pin(Gu[2]);
    BH_PHASE();
    // quadratic Christoffel terms of R_ab,
    //   g^cd (Gam^x_ca Gam_bxd + Gam^x_cb Gam_axd + Gam^x_ad Gam_xcb)
    //   + 1/2 Gam^c (Gam_abc + Gam_bac),
    // through X[x][d] = g^dc Gam_exc of one lowered index e at a time: the
    // first two terms take X against Gam^x_da for (a, e) and (e, a), the third
    // X[b][d] against Gam^e_ad.  About 300 FP64 operations, where the double
    // sum over c and d for each of the six components took 600.
#pragma unroll
    for (int e = 0; e < 3; e++) {
      double X[3][3];
#pragma unroll
      for (int x = 0; x < 3; x++)
#pragma unroll
        for (int d = 0; d < 3; d++)
          X[x][d] = ig[sy(d, 0)] * Gd[e][sy(x, 0)] + ig[sy(d, 1)] * Gd[e][sy(x, 1)] + ig[sy(d, 2)] * Gd[e][sy(x, 2)];
#pragma unroll
      for (int a = 0; a < 3; a++) {
        double m = 0.5 * (Gfg[0] * Gd[e][sy(a, 0)] + Gfg[1] * Gd[e][sy(a, 1)] + Gfg[2] * Gd[e][sy(a, 2)]);
#pragma unroll
        for (int x = 0; x < 3; x++)
          m += Gu[x][sy(0, a)] * X[x][0] + Gu[x][sy(1, a)] * X[x][1] + Gu[x][sy(2, a)] * X[x][2];
        R[sy(a, e)] += (a == e ? 2.0 : 1.0) * m;
#pragma unroll
        for (int b = a; b < 3; b++)
          R[sy(a, b)] += Gu[e][sy(a, 0)] * X[b][0] + Gu[e][sy(a, 1)] * X[b][1] + Gu[e][sy(a, 2)] * X[b][2];
      }
      pin(R);
      BH_PHASE();
    }
  }

  // ---- Gamma^i: + 1/2 (g_ca d_b G^c + g_cb d_a G^c) in R_ab
  static_for<3>([&](auto I_) {
    constexpr int c = decltype(I_)::value;
    advance(std::integral_constant<int, 9 + c>{}, [&] {
      if constexpr (c == 2) {
        pv[0] = ld(u[13]);
        pv[1] = ld(u[17]);
      }
    });
    double dG[3];
    const Fld F = field<SH, true, false>(T, G, w12, S, dG, none6);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = a; b < 3; b++) R[sy(a, b)] += 0.5 * (g[sy(c, a)] * dG[b] + g[sy(c, b)] * dG[a]);
    rG[c] += F.adv - 2.0 * alpha * K.kappa1 * F.f0;
    park[c * NTHR + tid] = eps * F.ko;
    park[(3 + c) * NTHR + tid] = K.withGadv * F.adv;
    pin(R);
    pin(rG[c]);
  });

  // ---- conformal factor
  double df[3];
  const double Khat = pv[0], Theta = pv[1];
  {
    advance(std::integral_constant<int, 12>{}, nothing);
    double dchi[3], h6[6];
    const Fld F = field<SH, true, true>(T, G, w12, S, dchi, h6);
    const double chi = F.f0;
    const double chig = (chi < K.chiDivFloor) ? K.chiDivFloor : chi;
    const double oochig = 1.0 / chig;
#pragma unroll
    for (int a = 0; a < 3; a++) df[a] = K.oocp * dchi[a] * oochig;
    double cddf[6];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = a; b < 3; b++) {
        const int ab = sy(a, b);
        cddf[ab] = K.oocp * h6[ab] * oochig - K.chipsipower * df[a] * df[b] -
                   (Gu[0][ab] * df[0] + Gu[1][ab] * df[1] + Gu[2][ab] * df[2]);
      }
    pin(cddf);
    BH_PHASE();
    const double trcddf = trace(cddf);
    const double dfdf = contract(df, df);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = a; b < 3; b++) {
        const int ab = sy(a, b);
        R[ab] += 4.0 * df[a] * df[b] - 2.0 * cddf[ab] - 2.0 * g[ab] * trcddf - 4.0 * g[ab] * dfdf;
      }
    pin(R);
    pin(df);
    emit(E[12 % 2],
         F.adv + eps * F.ko + (K.chipsipower / 6.0) * chig * (divbeta - alpha * (Khat + 2.0 * Theta)));
  }

  // ---- lapse; after this stage sA holds the curvature terms of At_ij
  double sA[6], da[3], trcdda, Rhat;
  {
    advance(std::integral_constant<int, 13>{}, nothing);
    double cdda[6], h6[6];
    const Fld F = field<SH, true, true>(T, G, w12, S, da, h6);
    emit(E[13 % 2], K.oplogwithshift * F.adv + eps * F.ko - fa * Khat);
    const double dfda = contract(df, da);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = a; b < 3; b++) {
        const int ab = sy(a, b);
        cdda[ab] = h6[ab] - (Gu[0][ab] * da[0] + Gu[1][ab] * da[1] + Gu[2][ab] * da[2]) -
                   2.0 * (df[a] * da[b] + df[b] * da[a] - g[ab] * dfda);
      }
    pin(cdda);
    pin(da);
    BH_PHASE();
    trcdda = psim4 * trace(cdda);
    Rhat = psim4 * trace(R);
#pragma unroll
    for (int c = 0; c < 6; c++)
      sA[c] = psim4 * (alpha * R[c] - cdda[c]) - (1.0 / 3.0) * g[c] * (alpha * Rhat - trcdda) + lA[c];
    pin(sA);
    pin(trcdda);
    pin(Rhat);
  }

  // ---- Khat, with the terms in At_ij: sA is then the whole right-hand side
  // of At_ij but for its advection and dissipation
  double Hhat;
  {
    double A[6];
    advance(std::integral_constant<int, 14>{}, [&] {
#pragma unroll
      for (int c = 0; c < 6; c++) A[c] = ld(u[7 + c]);
    });
    double d[3];
    Fld F = field<SH, true, false>(T, G, w12, S, d, none6);
    const double K_ = Khat + 2.0 * Theta;  // Khat alone is the lapse's source: K - 2 Theta would cancel
#pragma unroll
    for (int a = 0; a < 3; a++)
      rG[a] -= (4.0 / 3.0) * alpha * (ig[sy(a, 0)] * d[0] + ig[sy(a, 1)] * d[1] + ig[sy(a, 2)] * d[2]);
    BH_PHASE();
    double Ainv[6], AA[6];
    {
      double Au[3][3];
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
#pragma unroll
    for (int c = 0; c < 6; c++) sA[c] += alpha * (K_ * A[c] - 2.0 * AA[c]);
#pragma unroll
    for (int a = 0; a < 3; a++) {
      double s = 0.0;
#pragma unroll
      for (int bc = 0; bc < 6; bc++) s += ((bc == 0 || bc == 3 || bc == 5) ? 1.0 : 2.0) * Gu[a][bc] * Ainv[bc];
      // 3/2 d chi / chi = 3/2 chipsipower df
      s -= 1.5 * K.chipsipower * (Ainv[sy(a, 0)] * df[0] + Ainv[sy(a, 1)] * df[1] + Ainv[sy(a, 2)] * df[2]);
      rG[a] += 2.0 * alpha * s - 2.0 * (Ainv[sy(a, 0)] * da[0] + Ainv[sy(a, 1)] * da[1] + Ainv[sy(a, 2)] * da[2]);
    }
    Hhat = Rhat + (2.0 / 3.0) * K_ * K_ - cAA;
    emit(E[14 % 2], F.adv + eps * F.ko +
                 (alpha * (cAA + (1.0 / 3.0) * K_ * K_) - trcdda + K.kappa1 * (1.0 - K.kappa2) * alpha * Theta));
    pin(sA);
    pin(rG);
    pin(Hhat);
  }

  // ---- Theta
  {
    double d[3];
    advance(std::integral_constant<int, 15>{}, nothing);
    const Fld F = field<SH, true, false>(T, G, w12, S, d, none6);
#pragma unroll
    for (int a = 0; a < 3; a++)
      rG[a] -= (2.0 / 3.0) * alpha * (ig[sy(a, 0)] * d[0] + ig[sy(a, 1)] * d[1] + ig[sy(a, 2)] * d[2]);
    // the dissipation of Theta is added after the zeroThetaRHS factor
    emit(E[15 % 2], (alpha * (0.5 * Hhat - (2.0 + K.kappa2) * K.kappa1 * Theta) + F.adv) * K.zeroThetaRHS + eps * F.ko);
    pin(rG);
  }

  // ---- trace-free extrinsic curvature; Gamma^i leaves with the first three
  static_for<6>([&](auto I_) {
    constexpr int ab = decltype(I_)::value;
    advance(std::integral_constant<int, 16 + ab>{}, nothing);
    const Fld F = field<SH, false, false>(T, G, w12, S, none3, none6);
    emit(E[(16 + ab) % 2], F.adv + eps * F.ko + sA[ab]);
    if constexpr (ab < 3) emit(Q[(16 + ab) % 2], rG[ab] + park[ab * NTHR + tid]);
  });

  // ---- B: advection and dissipation, and the driver
  static_for<3>([&](auto I_) {
    constexpr int c = decltype(I_)::value;
    advance(std::integral_constant<int, 22 + c>{}, nothing);
    const Fld F = field<SH, false, false>(T, G, w12, S, none3, none6);
    const double drive = K.withBadv * F.adv + ((K.gamma0factor + K.gamma2factor * betaF) *
                                                   (rG[c] - park[(3 + c) * NTHR + tid]) -
                                               K.shiftdriver * F.f0);
    const double r = (withB ? drive : 0.0) + eps * F.ko;
    emit(E[(22 + c) % 2], r);
  });
  flush(E[24 % 2], P.st[25]);
  if (!active) return;
  if (bad) *args.flag = 1;
  if constexpr (ST::ADD) project_point(P, K, qb + loc / 8);
}

// The right-hand side of a level: slab and bulk tiles of all its boxes in one
// launch.  (As one launch for the bulk and one per slab orientation on a second
// stream, the slabs' few blocks, each as long as any other, ran one orientation
// after another and ended the evaluation: 24^3 box 0.11 ms, 64^3 0.16 ms.)
// The slab tiles come first, so that none is left to the end.  Two blocks per
// CU: 80 KB of LDS and 256 registers each.  SLABS = false: bulk regions only, as
// of a periodic box.  All kernels but one spill: by the compiler's report the
// bulk alone 6-12 registers with 16-byte units, 14-21 with dwords and 0-8 through
// registers, the kernel of all four bodies 79-128, 444-495 and 221-260 (8% more
// time on 192^3 when that ran a box without slabs).  The slab bodies hold the
// point's 18 advection coefficients besides, the dword units 20 offsets.  A
// reload ends in a wait for every transfer in flight.
//
// Workgroups are dispatched to the 8 XCDs round-robin (workgroup w to XCD w mod
// 8), each XCD with its own L2.  With xcd set, each XCD takes one contiguous
// range of the slab tiles and one of the bulk tiles, so that neighbouring tiles,
// which stage the same halo points, meet in the same L2.
template <class ST, int NB, int VEC, bool SLABS>
__global__ void __launch_bounds__(NTHR, 2) z4c_rhs_tile(TileArgs args) {
  constexpr int n0 = tile_lds<LBulk, NB, VEC>(), n1 = tile_lds<LSlabX, NB, VEC>(), n2 = tile_lds<LSlabY, NB, VEC>(),
                n3 = tile_lds<LSlabZ, NB, VEC>();
  constexpr int nl = (n0 > n1 ? n0 : n1) > (n2 > n3 ? n2 : n3) ? (n0 > n1 ? n0 : n1) : (n2 > n3 ? n2 : n3);
  static_assert(nl * sizeof(double) <= 80 * 1024, "two blocks per CU");
  __shared__ double tile[nl];
  const TileJobs &J = args.J;
  int t = (int)blockIdx.x;
  if (J.xcd) {
    const int per = (J.nshell + 7) / 8, perb = (J.blk0[J.n] - J.nshell + 7) / 8, x = t % 8, i = t / 8;
    const bool shell = i < per;
    t = shell ? x * per + i : J.nshell + x * perb + (i - per);
    // padding workgroup (whole block, before any barrier)
    if (t >= (shell ? J.nshell : J.blk0[J.n])) return;
  }
  // region of this block (uniform): the regions' tiles are numbered in order
  int r = 0;
  while (r + 1 < J.n && t >= J.blk0[r + 1]) r++;
  const int b = t - J.blk0[r], kind = SLABS ? J.reg[r].kind : 0;
  if (kind == 0) tile_body<LBulk, false, ST, NB, VEC>(tile, r, b);
  else if (kind == 1) tile_body<LSlabX, true, ST, NB, VEC>(tile, r, b);
  else if (kind == 2) tile_body<LSlabY, true, ST, NB, VEC>(tile, r, b);
  else tile_body<LSlabZ, true, ST, NB, VEC>(tile, r, b);
}

// XCD-aware tile numbering on (bamhip_z4c_set_xcd_map)
int tile_xcd_map();

template <class L>
int ntiles(const Z4cGeo &G) {
  return ((G.hi[0] - G.lo[0] + L::TX) / L::TX) * ((G.hi[1] - G.lo[1] + L::TY) / L::TY) *
         ((G.hi[2] - G.lo[2] + L::TZ) / L::TZ);
}

inline bool same_spacing(const Z4cGeo &a, const Z4cGeo &b) {
  return a.h[0] == b.h[0] && a.h[1] == b.h[1] && a.h[2] == b.h[2];
}

// regions of one level by layout: the bulk, and slabs normal to x, y and z
struct RegionLists {
  const std::vector<Z4cGeo> *kind[4];  // null: none of that kind
};
// one launch for all of them, or one per kMaxRegions regions and grid spacing
template <int NB, int VEC>
int launch_tiles(const Z4cPtrs &F, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  struct Reg {
    const Z4cGeo *g;
    int kind;
  };
  std::vector<Reg> regs;
  // grouped so that a launch's slabs come before its bulk regions and a level
  // of few boxes is one launch
  for (int kind : {1, 2, 3, 0})
    if (R.kind[kind])
      for (const Z4cGeo &G : *R.kind[kind]) regs.push_back({&G, kind});
  constexpr int LEAD = NB == 0 ? 1 : NB - 1;
  TilePtrs P{};
  for (int v = 0; v < 25; v++) P.u[v] = F.u[v];
  auto outputs = [&](StagePtrs &S, int v) {
    S.c = F.c[v];
    S.r = F.r[v];
    S.cp = F.cp[v];
  };
  auto operands = [&](StagePtrs &S, int v) {
    S.a = F.a[v];
    S.p = F.p[v];
  };
  for (int s = 0; s < 25; s++) {
    if (s + LEAD < 25) P.st[s].issue = F.u[STAGE_ORDER[s + LEAD]];
    if (STAGE_LOADS[s] >= 0) operands(P.st[s], STAGE_LOADS[s]);
    if (STAGE_STORES[s] >= 0) outputs(P.st[s], STAGE_STORES[s]);
  }
  outputs(P.st[25], STAGE_LOADS[24]);
  for (int c = 0; c < 3; c++) {
    operands(P.gam[c], 14 + c);
    outputs(P.gam[c], 14 + c);
  }
  size_t r0 = 0;
  while (r0 < regs.size()) {
    TileJobs J{};
    const Z4cGeo &G0 = *regs[r0].g;
    for (int a = 0; a < 3; a++) {
      J.sp.h[a] = G0.h[a];
      J.sp.ih[a] = G0.ih[a];
      J.sp.i12h[a] = G0.i12h[a];
      J.sp.i12hh[a] = G0.i12hh[a];
      J.sp.i144hh[a] = G0.i144hh[a];
    }
    int blk = 0;
    J.n = 0;
    while (r0 < regs.size() && J.n < kMaxRegions && same_spacing(*regs[r0].g, G0)) {
      const Z4cGeo &G = *regs[r0].g;
      const int kind = regs[r0++].kind;
      RegionGeo &Rg = J.reg[J.n];
      Rg.kind = kind;
      Rg.m = G.m;
      Rg.n = G.n;
      Rg.o = G.o;
      Rg.noffset = G.noffset;
      for (int a = 0; a < 3; a++) {
        Rg.lo[a] = G.lo[a];
        Rg.hi[a] = G.hi[a];
      }
      J.blk0[J.n++] = blk;
      blk += kind == 0 ? ntiles<LBulk>(G) : kind == 1 ? ntiles<LSlabX>(G) : kind == 2 ? ntiles<LSlabY>(G)
                                                                                        : ntiles<LSlabZ>(G);
      if (kind) J.nshell = blk;
    }
    J.blk0[J.n] = blk;
    if (blk == 0) continue;
    J.xcd = tile_xcd_map();
    const unsigned grid = J.xcd ? (unsigned)(8 * ((J.nshell + 7) / 8 + (blk - J.nshell + 7) / 8)) : (unsigned)blk;
    auto go = [&](auto st_) {
      if (J.nshell)
        z4c_rhs_tile<decltype(st_), NB, VEC, true><<<grid, NTHR, 0, st>>>(TileArgs{P, J, K, flag});
      else
        z4c_rhs_tile<decltype(st_), NB, VEC, false><<<grid, NTHR, 0, st>>>(TileArgs{P, J, K, flag});
    };
    if (!K.rk) {
      if (K.addlinear) go(StoreAs<false, true, false, false>{});
      else go(StoreAs<false, false, false, false>{});
    } else if (K.has_v) {
      if (K.has_cp) go(StoreAs<true, false, true, true>{});
      else go(StoreAs<true, false, true, false>{});
    } else {
      if (K.has_cp) go(StoreAs<true, false, false, true>{});
      else go(StoreAs<true, false, false, false>{});
    }
    BH_HIP(hipGetLastError());
  }
  return BAMHIP_OK;
}

// launchers of the staging variants, one per file (z4c_tile_*.hip)
using LaunchFn = int (*)(const Z4cPtrs &, const RegionLists &, const Z4cK &, int *, hipStream_t);
int tile_dma(const Z4cPtrs &, const RegionLists &, const Z4cK &, int *, hipStream_t);
int tile_reg(const Z4cPtrs &, const RegionLists &, const Z4cK &, int *, hipStream_t);
int tile_dma_x4(const Z4cPtrs &, const RegionLists &, const Z4cK &, int *, hipStream_t);

}  // namespace bamhip
