// The element one-body kernel's block (launched from kernels.hip, alone and in
// batches) and the series' convergence test.
#pragma once

#include "devmath.hpp"
#include "kernels.hpp"

namespace td1c {

// ---------------------------------------------------------------------------
// One-body part h01 = (T_l + h1) psi (hprod_tprodp, src/hprod/hprod_tprod.F90:152-235;
// hprod_zprodp, hprod_zprod.F90:108-135; hprod_pzprodp, hprod_pzprod.F90:114-213)
// in element-local form: a block of BS threads owns GE = (BS - 1) / (n + 1)
// consecutive elements of one orbital and walks lc consecutive l values.  Lane
// (element, m) keeps row m of the element's kinetic and d/dr matrices in
// registers.  Plane by plane, psi(l) of the block's points goes through LDS
// and one pass over it gives both T psi(l) and d psi(l)/dr of the lane's row;
// the output of l takes T(l) and the derivatives of l - 1 and l + 1, which
// stay in registers.  (The products of psi(l-1) and psi(l+1) used to be formed
// anew for every l, with three LDS reads per matrix element where one serves
// now.)  Bound by latency at 3 wavefronts per SIMD: the two matrix rows take
// 84 registers.  9 orbitals x 64 l x 2399 points, velocity gauge: 98 us beside
// the mean-field chain of a step and 37 alone, against 134 and 40; the half
// step's right-hand side in length gauge on 799 points 6.6 against 11.9; n =
// 17 against the band kernels that n != 20 had: 9 against 26.  An interior point needs one row product; a
// bridge adds the last row of the element on its left (the lane after the GE
// elements recomputes it for the block's first element).  A block of 64
// threads is a single wavefront and its bridge partials move by lane shuffles
// instead of LDS.  The (BS, lc) pair is a launch shape chosen per problem by
// the autotuner; every shape gives the same bits.  NM = n for n = 20, else an
// upper bound of n (16, 24, 32): the rows are padded with zeros.
// ---------------------------------------------------------------------------
// The convergence test of a clh1itr term (cn_check_body's arithmetic) in a
// block of BS threads: the partial sums added by 256 lanes in cn_check_body's
// order (lane v takes v, v + 256, ...; a butterfly in each wave of 64
// lanes; the four wave sums in order), so that every block size decides
// with the same bits.  Every thread of the block gets the result.
template <int BS>
__device__ __forceinline__ bool cn_series_done(const double* __restrict__ part, int ntot, int nfun, double thresh) {
  constexpr int V = 256;
  static_assert(V % BS == 0 && BS % 64 == 0, "block of whole waves dividing 256");
  __shared__ double sw[V / 64];
  const int t = threadIdx.x;
#pragma unroll
  for (int j = 0; j < V / BS; ++j) {
    const int v = t + j * BS;
    double s = 0.0;
    for (int q = v; q < ntot; q += V) s += part[q];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((v & 63) == 0) sw[v >> 6] = s;
  }
  __syncthreads();
  double tot = 0.0;
#pragma unroll
  for (int w = 0; w < V / 64; ++w) tot += sw[w];
  return sqrt(tot / nfun) < thresh;
}

constexpr int onebody_elements(int BS, int n) { return (BS - 1) / (n + 1); }

template <int NM, int BS, int CN>
__device__ __forceinline__ void onebody_el_body(const double2* __restrict__ orb, double2* __restrict__ h01, const OneBodyElArgs& a, int lc, const Blk bk) {
  if (CN == 2 && a.stop[0]) return;
  if (CN == 2 && a.chk_part) {
    if (cn_series_done<BS>(a.chk_part, a.chk_n, a.chk_nfun, a.chk_thresh)) {
      if (bk.x == 0 && bk.y == 0 && bk.z == 0 && threadIdx.x == 0) *a.chk_flag = 1;
      return;
    }
  }
  const double2 zf = make_double2(a.lf[2], 0.0), ef = make_double2(a.lf[5], 0.0);
  constexpr bool ONE_WAVE = BS == 64;
  constexpr int NPM = NM + 1;
  constexpr int CAP = BS + 2 * NM;   // points of elements e0-1 .. e0+GE-1, then zeros for padded rows
  __shared__ double2 sPsi[2][CAP];
  __shared__ double2 sT[ONE_WAVE ? 1 : BS], sD[ONE_WAVE ? 1 : BS];
  const int N = NM == 20 ? 20 : a.ndvr, NP = N + 1;
  const int GE = onebody_elements(BS, N), TILE = (GE + 1) * N + 1;
  const int f = bk.z;
  const int e0 = bk.x * GE;
  const int l0 = bk.y * lc;
  const int l1 = min(a.L1, l0 + lc);
  const int tid = threadIdx.x;
  // lane -> (element, local row)
  int e, m;
  if (tid < GE * NP) {
    e = e0 + tid / NP;
    m = tid % NP;
  } else if (tid == GE * NP) {
    e = e0 - 1;
    m = N;
  } else {
    e = -1;
    m = 0;
  }
  const bool lane_ok = e >= 0 && e < a.nfe;
  const int ee = lane_ok ? a.emap[e] : 0;  // the element's matrix block
  const int mf = a.mval[CN ? a.fshift + f : f];
  const int am = mf < 0 ? -mf : mf;
  const bool fc = CN ? false : f < a.nfcore;
  const int rows = fc ? a.nradfc : a.nr;
  const int ibase = (e0 - 1) * N - 1;        // global interior index of tile slot 0
  // tile slot of this lane's element point 0
  const int eslot = lane_ok ? (e - (e0 - 1)) * N : 0;
  const bool need_t = CN != 2, need_d = a.igauge == 1 && (CN != 1 || a.isplit == 1);
  const double2* base_f = orb + (size_t)f * a.L1 * a.nr;
  // l = 0 has its own kinetic matrix of the first element: its difference to
  // the other l's, applied to psi(0) (ahead of the loop, whose registers the
  // two matrix rows fill)
  double2 corr = make_double2(0.0, 0.0);
  if (need_t && l0 == 0 && lane_ok && e == 0) {
#pragma unroll 1
    for (int k = 1; k < NP; ++k) {  // (point 0 is r = 0)
      const double dk = a.eK0[(size_t)k * NP + m] - a.eK[(size_t)k * NP + m];
      const double2 x = base_f[k - 1];
      corr.x = fma(dk, x.x, corr.x);
      corr.y = fma(dk, x.y, corr.y);
    }
  }
  double Kr[NPM], Pr[NPM];
#pragma unroll
  for (int k = 0; k < NPM; ++k) {
    const bool ok = lane_ok && k <= N;
    Kr[k] = ok && need_t ? a.eK[((size_t)ee * NP + k) * NP + m] : 0.0;
    Pr[k] = ok && need_d ? a.eP[((size_t)ee * NP + k) * NP + m] : 0.0;
  }
  const int i = e * N + m - 1;               // global interior index of (e, m)
  // owner: interior rows, and row 0 of elements >= 1 (the bridge)
  const bool owner = lane_ok && tid < GE * NP && m < N && i >= 0 && i < a.nr;
  const double xr = owner ? a.xr[i] : 1.0;
  const double* al = a.alph + (size_t)(mf + a.mmax1) * a.L1;
  // the lane holding the left element's last row: the previous lane, or the
  // extra lane for the first element
  const int pl = tid >= NP ? tid - 1 : GE * NP;
  const double2 zero = make_double2(0.0, 0.0);
  if (NM != 20)  // zeros behind the tile
    for (int q = TILE + tid; q < CAP; q += BS) sPsi[0][q] = sPsi[1][q] = zero;
  // plane q is read from global memory one trip ahead, into registers, so
  // that its latency overlaps the previous plane's products
  constexpr int RP = 2;
  double2 nx[RP];
  auto fetch = [&](int q) {
#pragma unroll
    for (int j = 0; j < RP; ++j) {
      const int t = tid + j * BS, gi = ibase + t;
      nx[j] = (t < TILE && q >= 0 && q < a.L1 && gi >= 0 && gi < a.nr) ? base_f[(size_t)q * a.nr + gi] : make_double2(0.0, 0.0);
    }
  };
  // own point, T psi and d psi/dr of planes l-1, l and l+1 (completed rows)
  double2 pd = zero, p0 = zero, pu = zero, Tc = zero, Tn = zero, Dd = zero, Dc = zero, Dn = zero;
  fetch(l0 - 1);
#pragma unroll 1
  for (int q = l0 - 1; q <= l1; ++q) {  // plane q, then the output of l = q - 1
    double2* buf = sPsi[q & 1];
#pragma unroll
    for (int j = 0; j < RP; ++j)
      if (tid + j * BS < TILE) buf[tid + j * BS] = nx[j];
    if (q < l1) fetch(q + 1);
    __syncthreads();
    pd = p0;
    p0 = pu;
    Dd = Dc;
    Dc = Dn;
    Tc = Tn;
    pu = lane_ok ? buf[eslot + m] : make_double2(0.0, 0.0);
    const bool tq = need_t && q >= l0 && q < l1;
    double2 pT = zero, pD = zero;
    const double2* s0 = buf + eslot;
    if (CN == 2 || !tq) {
      if (need_d) {
#pragma unroll
        for (int k = 0; k < NPM; ++k) {
          const double2 x = s0[k];
          pD.x = fma(Pr[k], x.x, pD.x);
          pD.y = fma(Pr[k], x.y, pD.y);
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < NPM; ++k) {
        const double2 x = s0[k];
        pT.x = fma(Kr[k], x.x, pT.x);
        pT.y = fma(Kr[k], x.y, pT.y);
        pD.x = fma(Pr[k], x.x, pD.x);  // (the rows of d/dr are zero where they are not needed)
        pD.y = fma(Pr[k], x.y, pD.y);
      }
      if (q == 0) pT = cadd(pT, corr);
    }
    // the left neighbour's partials (bridge rows)
    double2 lT, lD;
    if (ONE_WAVE) {
      lT = make_double2(__shfl(pT.x, pl, 64), __shfl(pT.y, pl, 64));
      lD = make_double2(__shfl(pD.x, pl, 64), __shfl(pD.y, pl, 64));
    } else {
      sT[tid] = pT;
      sD[tid] = pD;
      __syncthreads();
      lT = sT[pl];
      lD = sD[pl];
    }
    if (m == 0) {  // bridge: add the left element's last row
      pT = cadd(pT, lT);
      pD = cadd(pD, lD);
    }
    Tn = pT;
    Dn = pD;
    const int l = q - 1;
    if (l < l0 || !owner) continue;
    double2 out = zero;
    if (l >= am && i < rows) {
      double2 h = zero;
      // T psi (CN 0, 1, 3; a frozen core with iprojfc = 1 gets only the
      // velocity-gauge E.z term, hprod_htot.F90:100-124), then the dipole
      // coupling of l +- 1 in the chosen gauge: CN 1 with isplit = 1 only
      // (the clh1itr right-hand sides, h1itr_prop.F90:57-70,106-114), CN 2
      // nothing else, CN 3 (T + V) psi (hprod_h1tot, hprod_h1tot.F90:2-53)
      const bool full = CN != 0 || !fc || a.fc_full;
      if (CN != 2 && full) {
        h = Tc;
        cfma(h, p0, a.tzor[(size_t)l * a.nr + i]);
      }
      if (CN == 1 ? a.isplit == 1 : full) {
        if (a.igauge == 0) {
          if (l + 1 < a.L1) cfma(h, pu, cscale(zf, xr * al[l]));
          if (l - 1 >= am) cfma(h, pd, cscale(zf, xr * al[l - 1]));
        } else {
          if (l + 1 < a.L1) {
            cfma(h, Dn, cmul(zf, make_double2(0.0, -al[l])));
            cfma(h, pu, cmul(zf, make_double2(0.0, -(al[l] * (l + 1.0)) / xr)));
          }
          if (l - 1 >= am) {
            cfma(h, Dd, cmul(zf, make_double2(0.0, -al[l - 1])));
            cfma(h, pd, cscale(cmul(zf, make_double2(0.0, -(al[l - 1] * (double)l) / xr)), -1.0));
          }
        }
      }
      if (CN == 0 && fc && a.igauge == 1) {  // E.z on the frozen core in the velocity gauge (hprod_htot.F90:123)
        if (l + 1 < a.L1) cfma(h, pu, cscale(ef, xr * al[l]));
        if (l - 1 >= am) cfma(h, pd, cscale(ef, xr * al[l - 1]));
      }
      if (CN == 0) {
        out = h;
      } else {
        if (CN == 1) out = p0;
        cfma(out, a.cv, h);
      }
    }
    h01[((size_t)f * a.L1 + l) * a.nr + i] = out;
  }
}

}  // namespace td1c
