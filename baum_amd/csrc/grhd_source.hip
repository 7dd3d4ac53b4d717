// grhd_source.hip -- GRHD source terms and matter ADM variables on gfx950.
//
// Reference: grhd_sources (src/projects/grhd/grhd_sources.m:8-190, generated
// as grhd_sources.c), MATTER.sources of matter_rhs (matter.c:438-442), with
// the reference's defaults grhd_source_computation = prim and grhd_cooling =
// 0 (bam_grhd.c:51-52).  At every inner point of every box:
//   - detg <= 0 or alpha <= 0: no source and matter ADM variables 0;
//   - centred first derivatives of alpha, beta^i, g_ij, 2nd order at distance
//     1 from a box face (or with order_centered 2), else 4th order, in the
//     multiplied form of the generated code;
//   - T^00, T^0i, T^ij, T^0_j from the primitives, W capped at grhd_Wlor_max
//     when v^2 >= 1;
//   - s_tau = alpha sqrt(g) (T^00 (beta beta K - beta d alpha)
//     + T^0i (2 beta^j K_ij - d_i alpha) + T^ij K_ij),
//     s_S_c = alpha sqrt(g) (T^00 (beta beta d_c g / 2 - alpha d_c alpha)
//     + T^0i beta^j d_c g_ij + T^0_j d_c beta^j + T^ij d_c g_ij / 2);
//   - matter ADM variables rho, S_i, S_ij, S for the Z4c matter terms;
//   - no momentum source below the atmosphere density, no tau source for a
//     cold EOS, all 16 values 0 when any is not finite;
//   - unew += source (times c when c != 0).
// A block computes a 16x4x4 tile of points.  The stress-energy terms come from
// the values at the point, so they are formed first; then the ten metric fields
// pass through LDS two at a time (the tile plus 2 points on every side, indices
// clamped to the box: only the stencils of inner points read the halo, and they
// stay inside it), and the derivatives of a field go straight into the sums of
// the sources, in the order of the full 3x3 index ranges: what an off-diagonal
// component still has to add is kept until its turn.  FP contraction is off, so
// the results are bitwise those of the C restatement that the tests compare
// with.
// Bound by latency and instructions, not by memory (173 us of traffic on 131^3
// points): 440 us with one field at a time through LDS, all 30 derivatives kept
// (210 registers, two waves per SIMD) and a branch on the order at each; 360 us
// with the running sums (three waves; forced to four they spill: 412 us); 328 us
// with runs of tiles per XCD (335 us without the groups of kYG rows); 318 us with
// the destinations loaded ahead of the stores.
#pragma clang fp contract(off)

#include <cmath>

#include "bamhip_internal.h"

namespace bamhip {
namespace {

constexpr int kSrcBlock = 256;
constexpr int kTX = 16, kTY = 4, kTZ = 4, kHalo = 2;
constexpr int kSX = kTX + 2 * kHalo, kSY = kTY + 2 * kHalo, kSZ = kTZ + 2 * kHalo, kSN = kSX * kSY * kSZ;
constexpr int kPer = (kSN + kSrcBlock - 1) / kSrcBlock;  // staged values per thread and field
constexpr int kYG = 4;                                   // rows of tiles walked through z together
constexpr int kGrp = 2;                                  // fields staged together
static_assert(kPer * kSrcBlock == kSN, "a whole number of staged values per thread");
static_assert(kTX * kTY * kTZ == kSrcBlock, "one point of the tile per thread");

struct SrcArgs {
  int m, n, o, skip[6];
  double oo2h[3];  // 1 / (2 h)
  double rhoatm, wlormax, c;
  int cold, order_centered;
  int distinct;  // no two of rhs and madm are one variable: rhs can be loaded ahead
  const double *met[10], *K[6], *prim[6];
  double *rhs[5], *madm[11];
};

// component (a, b) of a symmetric tensor among xx xy xz yy yz zz, and back
__device__ constexpr int s6(int a, int b) { return a * b == 0 ? a + b : a + b + 1; }
constexpr int kRow[6] = {0, 0, 0, 1, 1, 2}, kCol[6] = {0, 1, 2, 1, 2, 2};

// first derivative, centred, in the form of the generated code
// (grhd_sources.c: oo2dx (-u[-1] + u[1]), 1/6 oo2dx (u[-2] + 8 (-u[-1] + u[1]) - u[2]))
// both orders formed and one chosen: a branch on the point's order would split
// the wavefront at each of the 30 derivatives
__device__ __forceinline__ double d1(const double *u, int q, int s, double oo2h, int ord) {
  const double um2 = u[q - 2 * s], t = -u[q - s] + u[q + s], up2 = u[q + 2 * s];
  const double o2 = oo2h * t, o4 = 0.16666666666666666667 * oo2h * (um2 + 8. * t - up2);
  return ord == 2 ? o2 : o4;
}

// forms a value here: only inner points use the sums, and moved down to there
// the staged values would be held instead (300 registers)
__device__ __forceinline__ void keep(double &x) { asm volatile("" : "+v"(x)); }

__global__ void __launch_bounds__(kSrcBlock) grhd_source_kernel(SrcArgs A) {
  __shared__ double buf[2][kGrp][kSN];
  const int tid = threadIdx.x;
  // the blocks of an XCD (the workgroup number modulo 8) take one run of tiles,
  // so that neighbouring tiles find their halo in its L2
  const unsigned t = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
  const unsigned gx = (A.m + kTX - 1) / kTX, gy = (A.n + kTY - 1) / kTY, gz = (A.o + kTZ - 1) / kTZ;
  if (t >= gx * gy * gz) return;
  const unsigned grp = t / (gx * gz * kYG), w = min(gy - grp * kYG, (unsigned)kYG), u = t - grp * gx * gz * kYG;
  const int i0 = u % gx * kTX, j0 = (grp * kYG + u / gx % w) * kTY, k0 = u / (gx * w) * kTZ;
  const int i = i0 + tid % kTX, j = j0 + (tid / kTX) % kTY, k = k0 + tid / (kTX * kTY);
  const int imax = A.m - 1, jmax = A.n - 1, kmax = A.o - 1;
  const bool inner = i >= A.skip[0] && i <= imax - A.skip[1] && j >= A.skip[2] && j <= jmax - A.skip[3] &&
                     k >= A.skip[4] && k <= kmax - A.skip[5];
  const int ord =
      (A.order_centered == 2 || i == 1 || j == 1 || k == 1 || i == imax - 1 || j == jmax - 1 || k == kmax - 1) ? 2 : 4;
  // position of the point in the staged tile and the staged strides
  const int c = (tid % kTX + kHalo) + kSX * ((tid / kTX) % kTY + kHalo) + kSX * kSY * (tid / (kTX * kTY) + kHalo);
  const int sst[3] = {1, kSX, kSX * kSY};
  long off[kPer];
#pragma unroll
  for (int e = 0; e < kPer; e++) {
    const int idx = tid + e * kSrcBlock;
    const int sx = idx % kSX, sy = (idx / kSX) % kSY, sz = idx / (kSX * kSY);
    const int gi = min(max(i0 - kHalo + sx, 0), A.m - 1), gj = min(max(j0 - kHalo + sy, 0), A.n - 1),
              gk = min(max(k0 - kHalo + sz, 0), A.o - 1);
    off[e] = gi + (long)A.m * gj + (long)A.m * A.n * gk;
  }
  double r[kGrp][kPer];
#pragma unroll
  for (int f = 0; f < kGrp; f++)
#pragma unroll
    for (int e = 0; e < kPer; e++) r[f][e] = A.met[f][off[e]];

  // the terms of the values at the point (threads outside the box: the point of
  // the box next to theirs, unused)
  const long q = min(i, imax) + (long)A.m * min(j, jmax) + (long)A.m * A.n * min(k, kmax);
  const double al = A.met[0][q];
  double be[3], T0i[3], T0j[3], Tij[6], bK[3], bbK = 0., tk = 0., T00, sqrtmdetg;
#pragma unroll
  for (int a = 0; a < 3; a++) be[a] = A.met[1 + a][q];
  const double rho = A.prim[0][q];
  bool ok, bad = false;
  {
    double g[6], K[6], vu[3];
#pragma unroll
    for (int a = 0; a < 6; a++) g[a] = A.met[4 + a][q], K[a] = A.K[a][q];
    const double eps = A.prim[1][q], p = A.prim[5][q];
    vu[0] = A.prim[2][q], vu[1] = A.prim[3][q], vu[2] = A.prim[4][q];
    const double adj[6] = {g[3] * g[5] - g[4] * g[4], g[2] * g[4] - g[1] * g[5], g[1] * g[4] - g[2] * g[3],
                           g[0] * g[5] - g[2] * g[2], g[1] * g[2] - g[0] * g[4], g[0] * g[3] - g[1] * g[1]};
    const double detg = g[0] * adj[0] + g[1] * adj[1] + g[2] * adj[2];
    ok = detg > 0. && al > 0.;
    const double detginv = 1. / detg;
    double gi[6];
#pragma unroll
    for (int a = 0; a < 6; a++) gi[a] = detginv * adj[a];
    const double sqrtdetg = sqrt(detg);
    sqrtmdetg = al * sqrtdetg;
    double vl[3], vsq = 0.;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      vl[a] = 0.;
#pragma unroll
      for (int b = 0; b < 3; b++) vl[a] += g[s6(a, b)] * vu[b];
    }
#pragma unroll
    for (int a = 0; a < 3; a++) vsq += vu[a] * vl[a];
    double W = 1. / sqrt(1. - vsq);
    if (vsq >= 1.) W = A.wlormax;
    const double W2hrho = W * W * (rho + rho * eps + p);
    const double al2 = al * al;
    double vs[3];
#pragma unroll
    for (int a = 0; a < 3; a++) vs[a] = vu[a] - be[a] / al;
    T00 = (W2hrho - p) / al2;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      T0i[a] = W2hrho * vs[a] / al + p * be[a] / al2;
      T0j[a] = W2hrho * vl[a] / al;
    }
#pragma unroll
    for (int f = 0; f < 6; f++) {
      const int a = kRow[f], b = kCol[f];
      Tij[f] = W2hrho * vs[a] * vs[b] + p * (gi[f] - be[a] * be[b] / al2);
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
      bK[a] = 0.;
#pragma unroll
      for (int b = 0; b < 3; b++) {
        bbK += be[a] * be[b] * K[s6(a, b)];
        bK[a] += be[b] * K[s6(a, b)];
        tk += Tij[s6(a, b)] * K[s6(a, b)];
      }
    }
    double ad[11], vv = 0.;
#pragma unroll
    for (int a = 0; a < 3; a++) vv += vl[a] * vu[a];
    ad[0] = W2hrho - p;
#pragma unroll
    for (int a = 0; a < 3; a++) ad[1 + a] = W2hrho * vu[a];
#pragma unroll
    for (int f = 0; f < 6; f++) ad[4 + f] = W2hrho * vl[kRow[f]] * vl[kCol[f]] + g[f] * p;
    ad[10] = W2hrho * vv + 3. * p;
#pragma unroll
    for (int a = 0; a < 11; a++) bad |= !isfinite(ad[a]);
    // stored here, where they need not be kept; taken back below where a source
    // is not finite
    if (inner) {
#pragma unroll
      for (int a = 0; a < 11; a++) A.madm[a][q] = ok && !bad ? ad[a] : 0.;
    }
  }

  double sT = 0., dal[3], bbdg[3], t0dg[3], tdg[3], tdb[3], dk1[3], dk2[3], old[5];
#pragma unroll
  for (int d = 0; d < 3; d++) bbdg[d] = t0dg[d] = tdg[d] = tdb[d] = 0.;
#pragma unroll
  for (int h = 0; h < 10 / kGrp; h++) {
    // buf[h & 1] was last read before the barrier of the previous group
#pragma unroll
    for (int f = 0; f < kGrp; f++)
#pragma unroll
      for (int e = 0; e < kPer; e++) buf[h & 1][f][tid + e * kSrcBlock] = r[f][e];
    if (h + 1 == 10 / kGrp) {  // the destinations, so that they are there at the end
#pragma unroll
      for (int v = 0; v < 5; v++) old[v] = A.rhs[v][q];
    } else {
#pragma unroll
      for (int f = 0; f < kGrp; f++)
#pragma unroll
        for (int e = 0; e < kPer; e++) r[f][e] = A.met[(h + 1) * kGrp + f][off[e]];
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < kGrp; f++) {
      const int v = h * kGrp + f;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        const double x = d1(buf[h & 1][f], c, sst[d], A.oo2h[d], ord);
        const auto add = [&](int a, int b, double y) {  // the (a, b) terms of the sums over d_d g_ab
          bbdg[d] += be[a] * be[b] * y;
          t0dg[d] += T0i[a] * be[b] * y;
          tdg[d] += Tij[s6(a, b)] * y;
        };
        switch (v) {
          case 0: dal[d] = x; break;
          case 1: case 2: case 3: tdb[d] += T0j[v - 1] * x; break;
          case 4: add(0, 0, x); break;
          case 5: add(0, 1, x), dk1[d] = x; break;
          case 6: add(0, 2, x), add(1, 0, dk1[d]), dk2[d] = x; break;
          case 7: add(1, 1, x); break;
          case 8: add(1, 2, x), add(2, 0, dk2[d]), add(2, 1, x); break;
          case 9: add(2, 2, x); break;
        }
      }
      if (v == 0) {
        double bda = 0., t0 = 0.;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          bda += be[a] * dal[a];
          t0 += T0i[a] * (2. * bK[a] - dal[a]);
        }
        sT = sqrtmdetg * (T00 * (bbK - bda) + t0 + tk);
        keep(sT);
      }
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
      if (h == 0) keep(dal[d]);
      if (h < 2) keep(tdb[d]);
      if (h >= 2) keep(bbdg[d]), keep(t0dg[d]), keep(tdg[d]);
    }
  }
  if (!inner) return;
  double sD = 0., sS[3];
#pragma unroll
  for (int d = 0; d < 3; d++)
    sS[d] = sqrtmdetg * (T00 * (0.5 * bbdg[d] - al * dal[d]) + t0dg[d] + tdb[d] + 0.5 * tdg[d]);
  if (rho < A.rhoatm) sS[0] = sS[1] = sS[2] = 0.;
  if (A.cold) sT = 0.;
  const bool sbad = !isfinite(sT) || !isfinite(sS[0]) || !isfinite(sS[1]) || !isfinite(sS[2]);
  if (sbad && ok && !bad) {
#pragma unroll
    for (int a = 0; a < 11; a++) A.madm[a][q] = 0.;
  }
  if (sbad || bad || !ok) sT = sS[0] = sS[1] = sS[2] = 0.;
  const double s5[5] = {sD, sT, sS[0], sS[1], sS[2]};
  if (A.distinct) {
#pragma unroll
    for (int v = 0; v < 5; v++) A.rhs[v][q] = A.c != 0. ? old[v] + A.c * s5[v] : old[v] + s5[v];
  } else {
    for (int v = 0; v < 5; v++) A.rhs[v][q] = A.c != 0. ? A.rhs[v][q] + A.c * s5[v] : A.rhs[v][q] + s5[v];
  }
}

}  // namespace
}  // namespace bamhip

using namespace bamhip;

extern "C" int bamhip_grhd_sources(bamhip_level *lev, const bamhip_hrsc_params *par, double rhoatm, int order_centered,
                                   const int *unew, double c, const int *metric, const int *Kij, const int *prim,
                                   const int *madm) {
  const char *what = "bamhip_grhd_sources";
  if (!lev || !par) return set_error(BAMHIP_EINVAL, "%s: NULL argument", what);
  if (par->eos != 0 && par->eos != 1) return set_error(BAMHIP_EINVAL, "%s: eos=%d (0 ideal, 1 poly)", what, par->eos);
  if (order_centered != 2 && order_centered != 4)
    return set_error(BAMHIP_EINVAL, "%s: order_centered=%d (2 or 4)", what, order_centered);
  double *met[10], *kk[6], *pr[6], *rhs[5], *ad[11];
  int e;
  if ((e = gather_ptrs(lev, metric, 10, met, "bamhip_grhd_sources(metric)"))) return e;
  if ((e = gather_ptrs(lev, Kij, 6, kk, "bamhip_grhd_sources(Kij)"))) return e;
  if ((e = gather_ptrs(lev, prim, 6, pr, "bamhip_grhd_sources(prim)"))) return e;
  if ((e = gather_ptrs(lev, unew, 5, rhs, "bamhip_grhd_sources(unew)"))) return e;
  if ((e = gather_ptrs(lev, madm, 11, ad, "bamhip_grhd_sources(madm)"))) return e;
  for (const DevBox &B : lev->boxes) {
    // the 4th-order stencil of an inner point reaches 2 points: inner points
    // at distance 0 from a face would read outside the box
    for (int f = 0; f < 6; f++)
      if (B.skip[f] < 1) return set_error(BAMHIP_EINVAL, "%s: box face %d has no boundary layer", what, f);
  }
  double *out[16];
  for (int a = 0; a < 16; a++) out[a] = a < 5 ? rhs[a] : ad[a - 5];
  TimerScope ts("matter_rhs_source");
  for (const DevBox &B : lev->boxes) {
    SrcArgs A{};
    A.m = B.m, A.n = B.n, A.o = B.o;
    for (int f = 0; f < 6; f++) A.skip[f] = B.skip[f];
    A.oo2h[0] = 1 / (2 * B.dx), A.oo2h[1] = 1 / (2 * B.dy), A.oo2h[2] = 1 / (2 * B.dz);
    A.rhoatm = rhoatm, A.wlormax = par->wlormax, A.c = c;
    A.cold = par->eos == 1, A.order_centered = order_centered, A.distinct = distinct(out, 16);
    for (int a = 0; a < 10; a++) A.met[a] = met[a] + B.noffset;
    for (int a = 0; a < 6; a++) A.K[a] = kk[a] + B.noffset, A.prim[a] = pr[a] + B.noffset;
    for (int a = 0; a < 5; a++) A.rhs[a] = rhs[a] + B.noffset;
    for (int a = 0; a < 11; a++) A.madm[a] = ad[a] + B.noffset;
    const long tiles = (long)((B.m + kTX - 1) / kTX) * ((B.n + kTY - 1) / kTY) * ((B.o + kTZ - 1) / kTZ);
    grhd_source_kernel<<<(unsigned)((tiles + 7) / 8 * 8), kSrcBlock, 0, stream()>>>(A);
  }
  BH_HIP(hipGetLastError());
  return BAMHIP_OK;
}
