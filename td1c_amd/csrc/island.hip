// FP64 island of the hprod: CI reduced density matrices, regularised
// inverse of the 1-RDM, MO integrals, energies, the X matrix and the CI
// derivative.  One 256-thread workgroup does it without a host round trip:
// the small matrices live in LDS, loops over matrix entries / determinants
// are spread over the threads.  CI vectors whose work exceeds the LDS budget
// take launches over the chip for their O(n^4 determinants) parts.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace td1c {

namespace {

constexpr int kT = 256;
constexpr int kN2 = kMaxAct * kMaxAct;          // 64
constexpr int kF2 = kMaxFun * kMaxFun;          // 256

__device__ __forceinline__ double2 zmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 zconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 zadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 zsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 zscal(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ __forceinline__ double zabs(double2 a) { return sqrt(a.x * a.x + a.y * a.y); }
__device__ __forceinline__ double2 zero2() { return make_double2(0.0, 0.0); }

// The CI work of the one-block form, in LDS.
struct CiView {
  double2 *C, *D, *S, *T;       // D[n*n][nc] (D_pq = E_pq C), C[nc], S[nc], T[n*n][nc]
  const int *exA, *sgA, *exB, *sgB;
};

// Bytes of dynamic LDS a CI view needs (0: it does not fit).
__host__ __device__ inline size_t ci_lds_bytes(int n, int nstr_a, int nstr_b) {
  const size_t nc = (size_t)nstr_a * nstr_b;
  const size_t z = nc * ((size_t)2 * n * n + 2) * sizeof(double2);
  const size_t t = (size_t)2 * (nstr_a + nstr_b) * n * n * sizeof(int);
  const size_t b = z + t;
  return b <= kIslandLds ? b : 0;
}

// Sets up the view and copies the string tables in (caller syncs).
__device__ CiView ci_view(const IslandArgs& a, unsigned char* dyn) {
  const int n = a.nact, na = a.nstr_a, nb = a.nstr_b;
  const size_t nc = (size_t)na * nb, nt = (size_t)n * n;
  CiView v;
  v.D = reinterpret_cast<double2*>(dyn);
  v.C = v.D + nt * nc;
  v.S = v.C + nc;
  v.T = v.S + nc;
  int* eA = reinterpret_cast<int*>(v.T + nt * nc);
  int* gA = eA + na * nt;
  int* eB = gA + na * nt;
  int* gB = eB + nb * nt;
  for (size_t q = threadIdx.x; q < na * nt; q += kT) {
    eA[q] = a.exA[q];
    gA[q] = a.sgA[q];
  }
  for (size_t q = threadIdx.x; q < nb * nt; q += kT) {
    eB[q] = a.exB[q];
    gB[q] = a.sgB[q];
  }
  v.exA = eA; v.sgA = gA; v.exB = eB; v.sgB = gB;
  return v;
}

// (E_pq x)[f] for determinant f = (ib, it) by gathering from the source
// determinants: E_pq |s> = sg |t> exactly when E_qp |t> = sg |s>, so the
// source string is the E_qp image of the target string, alpha then beta.
__device__ __forceinline__ double2 gather_E(const IslandArgs& a, const CiView& v, int p, int q, const double2* x,
                                            int f) {
  const int ns = a.nstr_a, n = a.nact;
  const int ib = f / ns, it = f % ns;
  double2 t = zero2();
  const int ka = (it * n + q) * n + p;
  const int sa = v.exA[ka];
  if (sa >= 0) t = zadd(t, zscal(x[ib * ns + sa], (double)v.sgA[ka]));
  const int kb = (ib * n + q) * n + p;
  const int sb = v.exB[kb];
  if (sb >= 0) t = zadd(t, zscal(x[sb * ns + it], (double)v.sgB[kb]));
  return t;
}

// Hermitian eigen-decomposition by complex Jacobi rotations (stand-in for
// LAPACK zheev in hprod_invden_inv, src/hprod/hprod_invden.F90:62-107), by the
// whole block (n <= 8).  A round rotates the disjoint pairs of a round-robin
// schedule together: lane (slot, k) of the first 32 owns row or column k of
// pair slot, lanes 32..63 the rows of U.  A serial chain: one lane sweeping
// the pairs one by one took about 200 us for n = 6.  Ends when each squared
// element is below 1e-34 of the product of its two diagonal ones (rounding):
// weakly occupied orbitals make a graded matrix, whose small eigenvalues the
// rotations give to full relative accuracy if they run until then.  (Measured
// against the squared diagonal of all, the inverse lost up to 3e-10 of its norm
// at occupations down to 1e-12, where this loses 4e-15.)
__device__ void herm_eig(int n, double2* A, double* w, double2* U, int* s_more) {
  const int tid = threadIdx.x;
  for (int i = tid; i < n * n; i += kT) U[i] = make_double2(i % n == i / n ? 1.0 : 0.0, 0.0);
  const int N = n + (n & 1);  // players of the schedule; index n of an odd n sits out
  const int slot = (tid >> 3) & 3, k = tid & 7;
  for (int sweep = 0; sweep < 60; ++sweep) {
    __syncthreads();
    if (tid < 64) {
      const int i = tid & 7, j = tid >> 3;
      bool more = false;
      if (i < n && j < n && i != j) {
        const double2 z = A[i + n * j];
        more = !(z.x * z.x + z.y * z.y <= fmax(1e-34 * fabs(A[i + n * i].x * A[j + n * j].x), 1e-300));
      }
      const unsigned long long any = __ballot(more);
      if (tid == 0) *s_more = any != 0;
    }
    __syncthreads();
    if (*s_more == 0) break;
    for (int round = 0; round < N - 1; ++round) {
      // the pair of this slot: the fixed player N-1 meets `round`, the others
      // pair off symmetrically around it
      int p = slot == 0 ? N - 1 : (round + slot) % (N - 1);
      int q = slot == 0 ? round : (round - slot + N - 1) % (N - 1);
      if (p > q) {
        const int t = p;
        p = q;
        q = t;
      }
      const bool on = tid < 64 && slot < N / 2 && q < n && k < n;
      double c = 1.0, s = 0.0;
      double2 ph = make_double2(1.0, 0.0);
      if (on) {
        const double2 apq = A[p + n * q];
        const double mag = zabs(apq), app = A[p + n * p].x, aqq = A[q + n * q].x;
        if (mag > 1e-300) {
          // tan(2 th) = 2 mag / (aqq - app), the smaller root
          const double tau = (aqq - app) / (2.0 * mag);
          const double t = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
          c = 1.0 / sqrt(1.0 + t * t);
          s = t * c;
          ph = zscal(apq, 1.0 / mag);
        }
      }
      const double2 sph = zscal(ph, s), sphc = zscal(zconj(ph), s);
      __syncthreads();
      if (on) {  // columns p, q of A (lanes below 32) and of U
        double2* M = tid < 32 ? A : U;
        const double2 mp = M[k + n * p], mq = M[k + n * q];
        M[k + n * p] = zsub(zscal(mp, c), zmul(sphc, mq));
        M[k + n * q] = zadd(zmul(sph, mp), zscal(mq, c));
      }
      __syncthreads();
      if (on && tid < 32) {  // rows p, q of A
        const double2 apk = A[p + n * k], aqk = A[q + n * k];
        double2 np = zsub(zscal(apk, c), zmul(sph, aqk)), nq = zadd(zmul(sphc, apk), zscal(aqk, c));
        // the rotated pair's element is zero and its diagonal real
        if (k == p) nq = zero2(), np.y = 0.0;
        if (k == q) np = zero2(), nq.y = 0.0;
        A[p + n * k] = np;
        A[q + n * k] = nq;
      }
      __syncthreads();
    }
  }
  for (int i = tid; i < n; i += kT) w[i] = A[i + n * i].x;
  __syncthreads();
}

// entry e = i + n j of the regularised inverse U diag(d/(d^2+thresh)) U^+
// (hprod_invden_inv, src/hprod/hprod_invden.F90:62-107)
__device__ double2 inv_entry(int n, double thresh, const double2* U, const double* w, int e) {
  const int i = e % n, j = e / n;
  double2 t = zero2();
  for (int k = 0; k < n; ++k) {
    const double d = w[k];
    const double invd = thresh > 0.0 ? d / (d * d + thresh) : 1.0 / d;
    t = zadd(t, zscal(zmul(U[i + n * k], zconj(U[j + n * k])), invd));
  }
  return t;
}

}  // namespace

// the RDM entry e of ormas_mkden2 (den2(p,q,r,t) = <E_qp E_tr> - delta_pt
// den1(r,q), from <D_pq|D_tr>) and the mean-field kernel's act2 coefficient:
// den2 where the m values balance and |den2| > 1e-15 (the terms hprod_mfprod2
// keeps), else 0
__device__ __forceinline__ void put_den2(const IslandArgs& a, int e, double2 s, const double2* s_d1) {
  const int n = a.nact;
  const int p = e % n, q = (e / n) % n, r = (e / (n * n)) % n, t = e / (n * n * n);
  if (p == t) s = zsub(s, s_d1[r + n * q]);
  a.den2[e] = s;
  const int* mv = a.mval + a.ncore;
  const bool keep = mv[q] + mv[t] == mv[p] + mv[r] && s.x * s.x + s.y * s.y > 1.0e-30;
  a.mfc[e] = keep ? s : zero2();
}
// den1 entry e and the actx weight of the mean-field kernel (-den1/2 where m
// matches)
__device__ __forceinline__ void put_den1(const IslandArgs& a, int e, double2 s, double2* s_d1) {
  const int n = a.nact;
  s_d1[e] = s;
  a.den1[e] = s;
  const bool mm = a.mval[a.ncore + e % n] == a.mval[a.ncore + e / n];
  a.mfc[(size_t)n * n * n * n + e] = mm ? zscal(s, -0.5) : zero2();
}
// rden = D^-1 and rrden = (2 - D)^-1, regularised, from den1 in LDS
__device__ void put_inverses(const IslandArgs& a, const double2* s_d1) {
  __shared__ double2 s_A[kN2], s_U[kN2];
  __shared__ double s_w[kMaxAct];
  __shared__ int s_more;
  const int n = a.nact;
  for (int e = threadIdx.x; e < n * n; e += kT) s_A[e] = s_d1[e];
  herm_eig(n, s_A, s_w, s_U, &s_more);
  for (int e = threadIdx.x; e < n * n; e += kT) {
    const double2 r = inv_entry(n, a.throcc1, s_U, s_w, e);
    a.rden[e] = r;
    const bool mm = a.mval[a.ncore + e % n] == a.mval[a.ncore + e / n];
    a.mfc[(size_t)n * n * n * n + n * n + e] = mm ? r : zero2();
  }
  if (a.ncore == 0) return;
  if (n * 2 == a.nelact2) {
    for (int e = threadIdx.x; e < n * n; e += kT) a.rrden[e] = zero2();
    return;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n * n; e += kT) {
    const double d = e % n == e / n ? 2.0 : 0.0;
    s_A[e] = make_double2(d - s_d1[e].x, -s_d1[e].y);
  }
  herm_eig(n, s_A, s_w, s_U, &s_more);
  for (int e = threadIdx.x; e < n * n; e += kT) a.rrden[e] = inv_entry(n, a.throcc2, s_U, s_w, e);
}

// Stage A: den1, den2 from the CI vector (ormas_mkden1/2, den1(a,b) = <E_ba>,
// den2(a,b,c,d) = <E_ba E_dc> - delta_ad den1(c,b)), rden, rrden
// (hprod_invden, src/hprod/hprod_invden.F90:2-60).  This one-block form holds
// the CI work in LDS; longer CI vectors take the launches after it.
__global__ void __launch_bounds__(kT) k_island_a(const IslandArgs a) {
  extern __shared__ __align__(16) unsigned char dyn[];
  __shared__ double2 s_d1[kN2];
  const int n = a.nact;
  if (n == 0) return;
  const int nc = a.nstr_a * a.nstr_b;
  const CiView v = ci_view(a, dyn);
  double2* D = v.D;
  double2* C = v.C;
  for (int f = threadIdx.x; f < nc; f += kT) C[f] = a.det_of[f] >= 0 ? a.cic[a.det_of[f]] : zero2();
  __syncthreads();
  for (size_t e = threadIdx.x; e < (size_t)n * n * nc; e += kT) {
    const int pq = (int)(e / nc), f = (int)(e % nc);
    D[e] = gather_E(a, v, pq / n, pq % n, C, f);
  }
  __syncthreads();
  // den1(x,y) = sum conj(C) (E_yx C)
  for (int e = threadIdx.x; e < n * n; e += kT) {
    const int x = e % n, y = e / n;
    const double2* dv = D + (size_t)(y * n + x) * nc;
    double2 s = zero2();
    for (int d = 0; d < nc; ++d) s = zadd(s, zmul(zconj(C[d]), dv[d]));
    put_den1(a, e, s, s_d1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n * n * n * n; e += kT) {
    const int p = e % n, q = (e / n) % n, r = (e / (n * n)) % n, t = e / (n * n * n);
    const double2* u = D + (size_t)(p * n + q) * nc;
    const double2* w = D + (size_t)(t * n + r) * nc;
    double2 s = zero2();
    for (int k = 0; k < nc; ++k) s = zadd(s, zmul(zconj(u[k]), w[k]));
    put_den2(a, e, s, s_d1);
  }
  // D goes to the global work buffer for stage B
  for (size_t q = threadIdx.x; q < (size_t)n * n * nc; q += kT) a.ci_work[q] = D[q];
  put_inverses(a, s_d1);
}

// The same for CI vectors whose work exceeds the LDS budget (5 and more
// active orbitals).  One block did all of it in 1210 us for CAS(8e, 6o), 225
// determinants: n^4 sums of nc terms, a thread each, and the serial
// eigenvectors.  Now D_pq = E_pq C over the chip, the overlaps of these n^2
// vectors and C in tiles of 4 x 4 (a block per tile, each value loaded feeds
// 4 products, the lower triangle by conjugation), and one block that forms
// the RDMs and inverses from them.
__global__ void __launch_bounds__(kT) k_ci_excite(const IslandArgs a) {
  const int n = a.nact, ns = a.nstr_a, nc = ns * a.nstr_b;
  const int e = blockIdx.x * kT + threadIdx.x;
  if (e >= (n * n + 1) * nc) return;
  const int pq = e / nc, f = e - pq * nc;
  auto C = [&](int g) {
    const int d = a.det_of[g];
    return d >= 0 ? a.cic[d] : zero2();
  };
  double2 t = zero2();
  if (pq == n * n) {  // C itself, after the n^2 vectors
    t = C(f);
  } else {
    const int p = pq / n, q = pq - p * n, ib = f / ns, it = f - ib * ns;
    const int ka = (it * n + q) * n + p, kb = (ib * n + q) * n + p;
    const int sa = a.exA[ka], sb = a.exB[kb];
    if (sa >= 0) t = zadd(t, zscal(C(ib * ns + sa), (double)a.sgA[ka]));
    if (sb >= 0) t = zadd(t, zscal(C(sb * ns + it), (double)a.sgB[kb]));
  }
  a.ci_work[e] = t;
}

__global__ void __launch_bounds__(kT) k_ci_overlaps(const IslandArgs a) {
  const int nv = a.nact * a.nact + 1, nc = a.nstr_a * a.nstr_b;
  const int nt = (nv + 3) / 4;
  // tile (ta, tb), ta <= tb, of the upper triangle
  int ta = 0, rest = blockIdx.x;
  while (rest >= nt - ta) rest -= nt - ta, ++ta;
  const int tb = ta + rest;
  const double2* u[4];
  const double2* w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u[i] = a.ci_work + (size_t)min(4 * ta + i, nv - 1) * nc;
    w[i] = a.ci_work + (size_t)min(4 * tb + i, nv - 1) * nc;
  }
  double2 s[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) s[i][j] = zero2();
  for (int k = threadIdx.x; k < nc; k += kT) {
    double2 x[4], y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = zconj(u[i][k]);
      y[i] = w[i][k];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[i][j].x = fma(x[i].x, y[j].x, fma(-x[i].y, y[j].y, s[i][j].x));
        s[i][j].y = fma(x[i].x, y[j].y, fma(x[i].y, y[j].x, s[i][j].y));
      }
  }
  // transposing butterfly: lane t ends with double t % 32 of the tile
  double v[32];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    v[2 * i] = s[i / 4][i % 4].x;
    v[2 * i + 1] = s[i / 4][i % 4].y;
  }
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 16; h > 0; h >>= 1)
#pragma unroll
    for (int j = 0; j < h; ++j) {
      const bool up = (lane & h) != 0;
      const double send = up ? v[j] : v[j + h], keep = up ? v[j + h] : v[j];
      v[j] = keep + __shfl_xor(send, h, 64);
    }
  v[0] += __shfl_xor(v[0], 32, 64);
  __shared__ double red[kT / 64][32];
  if (lane < 32) red[threadIdx.x >> 6][lane] = v[0];
  __syncthreads();
  if (threadIdx.x < 16) {
    const int t = threadIdx.x, i = 4 * ta + t / 4, j = 4 * tb + t % 4;
    if (i < nv && j < nv) {
      double2 z = zero2();
#pragma unroll
      for (int q = 0; q < kT / 64; ++q) z = zadd(z, make_double2(red[q][2 * t], red[q][2 * t + 1]));
      a.ci_gram[(size_t)i * nv + j] = z;
      if (ta != tb) a.ci_gram[(size_t)j * nv + i] = zconj(z);
    }
  }
}

__global__ void __launch_bounds__(kT) k_ci_rdm(const IslandArgs a) {
  __shared__ double2 s_d1[kN2];
  const int n = a.nact, nv = n * n + 1;
  for (int e = threadIdx.x; e < n * n; e += kT)  // <C|D_yx>
    put_den1(a, e, a.ci_gram[(size_t)(n * n) * nv + (e / n) * n + e % n], s_d1);
  __syncthreads();
  for (int e = threadIdx.x; e < n * n * n * n; e += kT) {
    const int p = e % n, q = (e / n) % n, r = (e / (n * n)) % n, t = e / (n * n * n);
    put_den2(a, e, a.ci_gram[(size_t)(p * n + q) * nv + t * n + r], s_d1);
  }
  put_inverses(a, s_d1);
}

// Stage B: int1e, int2e (hprod_mkint1_sph / hprod_mkint2_sph), energies
// (hprod_ene_dcore, hprod_ene_act), X matrix (hprod_htot_mkxmat_fc/cc/ca/aa1,
// src/hprod/hprod_htot_mkxmat.F90) and the CI derivative (ormas_xact2 with one
// ORMAS subspace, src/ormas/ormas_xact2.F90:2-102).
__device__ __forceinline__ void island_b_body(const IslandArgs& a, const Blk bk) {
  extern __shared__ __align__(16) unsigned char dyn[];
  __shared__ double2 s_H[kF2], s_G[kF2], s_V[kF2], s_F[kF2], s_X[kF2], s_FM[kF2];
  __shared__ double2 s_hp[kN2];
  __shared__ double2 s_i1[kN2], s_d1[kN2], s_rr[kN2];
  __shared__ double s_red[kT / 64];
  __shared__ double s_eact;
  __shared__ int s_mval[kMaxFun];
  __shared__ int s_q[4 * kF2];  // the four l-space product maps (partial-sum mode)
  const int nf = a.nfun, nfc = a.nfcore, ncore = a.ncore, na = a.nact;
  const int tid = threadIdx.x;
  // every global input first (the index maps, then what they point at), so
  // the gather costs two memory round trips
  double2* I2 = a.int2e;
  if (a.i2_lds) I2 = reinterpret_cast<double2*>(dyn + a.ci_lds_off);
  for (int e = tid; e < nf; e += kT) s_mval[e] = a.mval[e];
  const int nf2 = nf * nf;
  if (a.lnblk > 0) {
    // the l-space products from their partial sums: the maps first, then
    // four lanes per referenced entry (quads stay together in the loop)
    for (int e = tid; e < nf2; e += kT) {
      s_q[e] = a.mapH[e];
      s_q[nf2 + e] = a.mapG[e];
      s_q[2 * nf2 + e] = a.mapV[e];
      s_q[3 * nf2 + e] = a.mapF[e];
      s_X[e] = zero2();
    }
    __syncthreads();
    for (int slot = tid >> 2; slot < 4 * nf2; slot += kT / 4) {
      const int q = s_q[slot], sub = tid & 3;
      double2 acc = zero2();
      if (q >= 0)
        for (int b = sub; b < a.lnblk; b += 4) acc = zadd(acc, a.lpart[(size_t)q * a.lnblk + b]);
      acc.x += __shfl_xor(acc.x, 1, 64);
      acc.y += __shfl_xor(acc.y, 1, 64);
      acc.x += __shfl_xor(acc.x, 2, 64);
      acc.y += __shfl_xor(acc.y, 2, 64);
      if (sub == 0) {
        const int w = slot / nf2, e = slot - w * nf2;
        double2* dst = w == 0 ? s_H : w == 1 ? s_G : w == 2 ? s_V : s_F;
        dst[e] = acc;
      }
    }
  } else {
    for (int e = tid; e < nf2; e += kT) {
      const int qh = a.mapH[e], qg = a.mapG[e], qv = a.mapV[e], qf = a.mapF[e];
      s_H[e] = qh >= 0 ? a.lprod[qh] : zero2();
      s_G[e] = qg >= 0 ? a.lprod[qg] : zero2();
      s_V[e] = qv >= 0 ? a.lprod[qv] : zero2();
      s_F[e] = qf >= 0 ? a.lprod[qf] : zero2();
      s_X[e] = zero2();
    }
  }
  for (int e = tid; e < na * na; e += kT) {
    s_d1[e] = a.den1[e];
    s_rr[e] = a.rrden[e];
  }
  // int2e(i,j,k,l): i >= j from the products, the rest by conjugate symmetry;
  // kept in LDS (after the CI view) when it fits
  for (int e = tid; e < na * na * na * na; e += kT) {
    const int ia = e % na, ja = (e / na) % na, ka = (e / (na * na)) % na, la = e / (na * na * na);
    int src = e;
    bool cj = false;
    if (ja > ia) {
      src = ja + na * (ia + na * (la + na * ka));
      cj = true;
    }
    const int q = a.map2e[src];
    double2 v = q >= 0 ? a.pprod[q] : zero2();
    if (cj) v = zconj(v);
    I2[e] = v;
    if (a.i2_lds) a.int2e[e] = v;
  }
  // inputs of the CI derivative and of the Runge-Kutta update that do not
  // depend on the Gram products, loaded together with the gather above
  const bool wide = na > 0 && !a.ci_lds;  // the CI derivative follows in launches of its own
  const int nc = na > 0 ? a.nstr_a * a.nstr_b : 0;
  CiView v{};
  if (na > 0 && !wide) {
    v = ci_view(a, dyn);
    for (size_t q = tid; q < (size_t)na * na * nc; q += kT) v.D[q] = a.ci_work[q];
    for (int f = tid; f < nc; f += kT) v.C[f] = a.det_of[f] >= 0 ? a.cic[a.det_of[f]] : zero2();
  }
  const bool rk_pre = !wide && a.kout != nullptr && tid < a.lcic;  // this thread's first CI coefficient
  double2 rk_w0 = zero2(), rk_acc = zero2(), rk_kp[kMaxStages];
  if (rk_pre) {
    if (a.acc != nullptr) rk_acc = a.acc[tid];
    if (a.next != nullptr) {
      rk_w0 = a.w0[tid];
      for (int j = 0; j < a.nprev; ++j) rk_kp[j] = a.kprev[j][tid];
    }
  }
  __syncthreads();
#define H(j, i) s_H[(j) * nf + (i)]
#define G(j, i) s_G[(j) * nf + (i)]
#define V(j, i) s_V[(j) * nf + (i)]
#define F(j, i) s_F[(j) * nf + (i)]
#define HGV(j, i) zadd(V(j, i), zadd(G(j, i), H(j, i)))
  // int1e(j,i) = <j|g + h1 + h0|i> for j <= i, Hermitian fill
  for (int e = tid; e < na * na; e += kT) {
    const int ja = e % na, ia = e / na;
    const int i = ncore + ia, j = ncore + ja;
    double2 v = zero2();
    if (ja <= ia) {
      if (s_mval[i] == s_mval[j]) v = zadd(G(j, i), H(j, i));
    } else if (s_mval[i] == s_mval[j]) {
      v = zconj(zadd(G(i, j), H(i, j)));
    }
    s_i1[e] = v;
    a.int1e[e] = v;
  }
  __syncthreads();
  // energies: ene_act = Re sum int1e(i,j) den1(j,i) + 1/2 Re sum int2e(i,j,k,l) den2(j,i,l,k)
  double part = 0.0;
  for (int e = tid; e < na * na * na * na; e += kT) {
    const int ia = e % na, ja = (e / na) % na, ka = (e / (na * na)) % na, la = e / (na * na * na);
    part += 0.5 * zmul(I2[e], a.den2[ja + na * (ia + na * (la + na * ka))]).x;
  }
  for (int e = tid; e < na * na; e += kT) {
    const int ia = e % na, ja = e / na;
    part += zmul(s_i1[ia + na * ja], s_d1[ja + na * ia]).x;
  }
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
  if ((tid & 63) == 0) s_red[tid >> 6] = part;
  __syncthreads();
  if (tid == 0) {
    double ene_dcore = 0.0;
    for (int i = nfc; i < ncore; ++i) ene_dcore += zadd(G(i, i), zscal(H(i, i), 2.0)).x;
    const double ene_act = na > 0 ? (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]) : 0.0;
    s_eact = ene_act;
    a.ene[1] = ene_dcore;
    a.ene[2] = a.ene[0] + ene_dcore;
    a.ene[3] = ene_act;
    a.ene[4] = a.ene[2] + ene_act;
  }
  const double2 tfac = a.icomp == 0 ? make_double2(a.dtime, 0.0) : make_double2(0.0, a.dtime);
#define XM(j, i) s_X[(i) * nf + (j)]
  // fc-dyn, core-core and active-active blocks (one entry per thread)
  for (int e = tid; e < nf * nf; e += kT) {
    const int j = e % nf, i = e / nf;
    if (s_mval[j] != s_mval[i]) continue;
    if (j < nfc && i >= nfc) XM(j, i) = zmul(zadd(F(j, i), zadd(G(j, i), V(j, i))), tfac);
    else if (j >= nfc && j < ncore && i >= nfc && i < ncore) XM(j, i) = zmul(HGV(j, i), tfac);
    else if (j >= ncore && i >= ncore) XM(j, i) = zmul(HGV(j, i), tfac);
  }
  __syncthreads();
  // core-active blocks (mkxmat_ca / ca0), small: one lane
  if (tid == 0 && na > 0 && ncore > nfc) {
    if (na * 2 == a.nelact2) {
      for (int i = nfc; i < ncore; ++i)
        for (int j = ncore; j < nf; ++j)
          if (s_mval[j] == s_mval[i]) {
            XM(j, i) = zmul(HGV(j, i), tfac);
            XM(i, j) = zmul(HGV(i, j), tfac);
          }
    } else {
      double2* FM = s_FM;
      for (int q = 0; q < nf * nf; ++q) FM[q] = zero2();
      for (int i = nfc; i < ncore; ++i)
        for (int j = ncore; j < nf; ++j)
          if (s_mval[j] == s_mval[i]) {
            FM[i * nf + j] = HGV(j, i);
            FM[j * nf + i] = HGV(i, j);
          }
      for (int i = nfc; i < ncore; ++i)
        for (int j = ncore; j < nf; ++j) {
          XM(j, i) = zmul(FM[i * nf + j], tfac);
          XM(i, j) = zmul(FM[j * nf + i], tfac);
        }
      for (int i = nfc; i < ncore; ++i)
        for (int ja = 0; ja < na; ++ja) {
          int j = ncore + ja;
          double2 fji = zscal(FM[i * nf + j], 2.0);
          double2 t = zero2();
          for (int ka = 0; ka < na; ++ka) t = zadd(t, zmul(s_d1[ja + na * ka], zconj(FM[(ncore + ka) * nf + i])));
          FM[i * nf + j] = zsub(fji, t);
        }
      for (int i = nfc; i < ncore; ++i)
        for (int ja = 0; ja < na; ++ja) {
          int j = ncore + ja;
          double2 t = zero2();
          for (int ka = 0; ka < na; ++ka) t = zadd(t, zmul(s_rr[ja + na * ka], FM[i * nf + ncore + ka]));
          double2 bji = zscal(zmul(tfac, t), -1.0);
          XM(j, i) = zadd(XM(j, i), bji);
          XM(i, j) = zadd(XM(i, j), zscal(zconj(bji), -1.0));
        }
    }
  }
  __syncthreads();
  for (int e = tid; e < nf * nf; e += kT) a.xmat[e] = s_X[e];
#undef XM
#undef H
#undef G
#undef V
#undef F
#undef HGV
  // CI derivative: dC = fac (H_CI - E_act) C, with D_pq = E_pq C from stage A
  if (na > 0) {
    double2* D = v.D;
    double2* C = v.C;
    double2* S = v.S;
    double2* T = v.T;
    // h'_pq = int1e(p,q) - 1/2 sum_r int2e(p,r,r,q)
    for (int e = tid; e < na * na; e += kT) {
      const int p = e % na, q = e / na;
      double2 hpq = s_i1[p + na * q];
      for (int r = 0; r < na; ++r) hpq = zsub(hpq, zscal(I2[p + na * (r + na * (r + na * q))], 0.5));
      s_hp[e] = hpq;
      if (wide) a.ci_hp[e] = hpq;
    }
    if (wide) return;
    __syncthreads();
    // T_pq = 1/2 sum_rs int2e(p,q,r,s) D_rs for every (p, q) at once
    for (size_t e = tid; e < (size_t)na * na * nc; e += kT) {
      const int pq = (int)(e / nc), f = (int)(e % nc);
      const int p = pq / na, q = pq % na;
      double2 t = zero2();
      for (int r = 0; r < na; ++r)
        for (int s2 = 0; s2 < na; ++s2)
          t = zadd(t, zmul(zscal(I2[p + na * (q + na * (r + na * s2))], 0.5), D[(size_t)(r * na + s2) * nc + f]));
      T[e] = t;
    }
    __syncthreads();
    // S = sum_pq h'_pq E_pq C + sum_pq E_pq T_pq, one determinant per thread
    for (int f = tid; f < nc; f += kT) {
      double2 acc = zero2();
      for (int p = 0; p < na; ++p)
        for (int q = 0; q < na; ++q) acc = zadd(acc, zmul(s_hp[p + na * q], D[(size_t)(p * na + q) * nc + f]));
      for (int p = 0; p < na; ++p)
        for (int q = 0; q < na; ++q) acc = zadd(acc, gather_E(a, v, p, q, T + (size_t)(p * na + q) * nc, f));
      S[f] = acc;
    }
    const double2 fac = a.icomp == 1 ? make_double2(0.0, -a.dtime) : make_double2(-a.dtime, 0.0);
    const double eact = s_eact;
    for (int f = tid; f < nc; f += kT) {
      int d = a.det_of[f];
      if (d < 0) continue;
      a.dcic[d] = zmul(zsub(S[f], zscal(C[f], eact)), fac);
    }
  } else {
    for (int d = tid; d < a.lcic; d += kT) a.dcic[d] = zero2();
  }
  if (a.kout != nullptr) {
    __syncthreads();
    for (int d = tid; d < a.lcic; d += kT) {
      const double2 k = a.dcic[d];
      const bool pre = d == tid && rk_pre;  // inputs already in registers
      // w0 may alias acc: both read before acc is written
      const double2 acc0 = a.acc != nullptr ? (pre ? rk_acc : a.acc[d]) : zero2();
      const double2 w0v = a.next != nullptr ? (pre ? rk_w0 : a.w0[d]) : zero2();
      a.kout[d] = k;
      if (a.acc != nullptr) {
        if (a.w0out != nullptr) a.w0out[d] = acc0;
        a.acc[d] = zadd(acc0, zscal(k, a.dtw));
      }
      if (a.next != nullptr) {
        double2 t = w0v;
        for (int j = 0; j < a.nprev; ++j) t = zadd(t, zscal(pre ? rk_kp[j] : a.kprev[j][d], a.cprev[j]));
        a.next[d] = zadd(t, zscal(k, a.cnew));
      }
    }
  }
}

__global__ void __launch_bounds__(kT) k_island_b(const IslandArgs a) {
  island_b_body(a, hw_blk());
}

// The CI derivative of long CI vectors over the chip (330 us in the one
// block for 225 determinants of 6 orbitals, T's n^4 nc products most of it).
// T_pq = 1/2 sum_rs int2e(p,q,r,s) D_rs: a wavefront takes 64 determinants
// and four pq, whose coefficients are wave-uniform scalar loads.
__global__ void __launch_bounds__(kT) k_ci_t(const IslandArgs a) {
  const int n = a.nact, n2 = n * n, nc = a.nstr_a * a.nstr_b;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pq0 = (blockIdx.y * (kT / 64) + wave) * 4;  // p + n q
  const int f = blockIdx.x * 64 + (threadIdx.x & 63);
  if (pq0 >= n2) return;
  const double2* __restrict__ D = a.ci_work;
  const double2* __restrict__ I2 = a.int2e;
  double2 t[4];
  int at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    t[i] = zero2();
    at[i] = min(pq0 + i, n2 - 1);
  }
  const int fc = min(f, nc - 1);
#pragma unroll 6
  for (int rs = 0; rs < n2; ++rs) {  // r n + s
    const int r = rs / n, s = rs - r * n;
    const double2 d = D[(size_t)rs * nc + fc];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double2 c = I2[at[i] + n2 * (r + n * s)];
      t[i].x = fma(c.x, d.x, fma(-c.y, d.y, t[i].x));
      t[i].y = fma(c.x, d.y, fma(c.y, d.x, t[i].y));
    }
  }
  if (f >= nc) return;
  double2* T = a.ci_work + (size_t)(n2 + 2) * nc;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (pq0 + i < n2) {
      const int p = (pq0 + i) % n, q = (pq0 + i) / n;
      T[(size_t)(p * n + q) * nc + f] = zscal(t[i], 0.5);
    }
}

// S = sum_pq h'_pq E_pq C + sum_pq E_pq T_pq, dC = fac (S - E_act C) and the
// Runge-Kutta update: 16 lanes per determinant share the pq
__global__ void __launch_bounds__(kT) k_ci_deriv(const IslandArgs a) {
  const int n = a.nact, n2 = n * n, ns = a.nstr_a, nc = ns * a.nstr_b;
  const int sub = threadIdx.x & 15, f = blockIdx.x * (kT / 16) + (threadIdx.x >> 4);
  const int d = f < nc ? a.det_of[f] : -1;
  const double2* __restrict__ D = a.ci_work;
  const double2* __restrict__ T = a.ci_work + (size_t)(n2 + 2) * nc;
  double2 s = zero2();
  if (d >= 0) {
    const int ib = f / ns, it = f - ib * ns;
#pragma unroll 4
    for (int pq = sub; pq < n2; pq += 16) {
      const int p = pq / n, q = pq - p * n;
      const int ka = (it * n + q) * n + p, kb = (ib * n + q) * n + p;
      const int sa = a.exA[ka], sb = a.exB[kb];
      s = zadd(s, zmul(a.ci_hp[p + n * q], D[(size_t)pq * nc + f]));
      if (sa >= 0) s = zadd(s, zscal(T[(size_t)pq * nc + ib * ns + sa], (double)a.sgA[ka]));
      if (sb >= 0) s = zadd(s, zscal(T[(size_t)pq * nc + sb * ns + it], (double)a.sgB[kb]));
    }
  }
  for (int o = 8; o > 0; o >>= 1) {
    s.x += __shfl_xor(s.x, o, 64);
    s.y += __shfl_xor(s.y, o, 64);
  }
  if (sub != 0 || d < 0) return;
  const double2 fac = a.icomp == 1 ? make_double2(0.0, -a.dtime) : make_double2(-a.dtime, 0.0);
  const double2 k = zmul(zsub(s, zscal(D[(size_t)n2 * nc + f], a.ene[3])), fac);  // C follows the D_pq
  a.dcic[d] = k;
  if (a.kout == nullptr) return;
  // w0 may alias acc: both read before acc is written
  const double2 acc0 = a.acc != nullptr ? a.acc[d] : zero2();
  const double2 w0v = a.next != nullptr ? a.w0[d] : zero2();
  a.kout[d] = k;
  if (a.acc != nullptr) {
    if (a.w0out != nullptr) a.w0out[d] = acc0;
    a.acc[d] = zadd(acc0, zscal(k, a.dtw));
  }
  if (a.next != nullptr) {
    double2 t = w0v;
    for (int j = 0; j < a.nprev; ++j) t = zadd(t, zscal(a.kprev[j][d], a.cprev[j]));
    a.next[d] = zadd(t, zscal(k, a.cnew));
  }
}

void island_lds_plan(IslandArgs& a) {
  a.ci_lds = 0;
  a.i2_lds = 0;
  a.ci_lds_off = 0;
  a.lds_bytes = 0;
  if (a.nact == 0) return;
  const size_t ci = ci_lds_bytes(a.nact, a.nstr_a, a.nstr_b);
  if (ci > 0) {
    a.ci_lds = 1;
    a.ci_lds_off = (ci + 15) / 16 * 16;
  }
  const size_t i2 = (size_t)a.nact * a.nact * a.nact * a.nact * sizeof(double2);
  if (a.ci_lds_off + i2 <= kIslandLds) a.i2_lds = 1;
  a.lds_bytes = a.ci_lds_off + (a.i2_lds ? i2 : 0);
}

void launch_island_a(const IslandArgs& a, hipStream_t s) {
  if (active_recorder()) return record_unsupported("the CI density stage (active orbitals)");
  if (a.ci_lds) {
    hipLaunchKernelGGL(k_island_a, dim3(1), dim3(kT), a.ci_lds_off, s, a);
    return;
  }
  const int nv = a.nact * a.nact + 1, nt = (nv + 3) / 4;
  const size_t nc = (size_t)a.nstr_a * a.nstr_b;
  hipLaunchKernelGGL(k_ci_excite, dim3((unsigned)((nv * nc + kT - 1) / kT)), dim3(kT), 0, s, a);
  hipLaunchKernelGGL(k_ci_overlaps, dim3(nt * (nt + 1) / 2), dim3(kT), 0, s, a);
  hipLaunchKernelGGL(k_ci_rdm, dim3(1), dim3(kT), 0, s, a);
}
void launch_island_b(const IslandArgs& a, hipStream_t s) {
  if (active_recorder()) {
    const int var[4] = {0, 0, 0, 0};
    return record_launch(kRecIslandB, var, dim3(1), kT, a.lds_bytes, a);
  }
  hipLaunchKernelGGL(k_island_b, dim3(1), dim3(kT), a.lds_bytes, s, a);
  if (a.nact > 0 && !a.ci_lds) {
    const int n2 = a.nact * a.nact, nc = a.nstr_a * a.nstr_b;
    hipLaunchKernelGGL(k_ci_t, dim3((nc + 63) / 64, (n2 + 15) / 16), dim3(kT), 0, s, a);
    hipLaunchKernelGGL(k_ci_deriv, dim3((nc + kT / 16 - 1) / (kT / 16)), dim3(kT), 0, s, a);
  }
}

__global__ void __launch_bounds__(kT) k_island_b_batch(const IslandArgs* __restrict__ recs, const BatchMap map) {
  __shared__ __align__(16) unsigned char raw[sizeof(IslandArgs)];
  int have = -1;
  batch_walk(map, NoSkip(), [&](int m, const Blk& bk) {
    const IslandArgs& r = stage_rec(recs, m, raw, have);
    island_b_body(r, bk);
  });
}

bool launch_batch_island(const LaunchRec& p, const void* recs, const BatchMap& map, int grid, size_t lds,
                         hipStream_t s, bool dry) {
  if (p.kind != kRecIslandB || p.block != kT) return false;
  if (!dry)
    hipLaunchKernelGGL(k_island_b_batch, dim3(grid), dim3(kT), lds, s, static_cast<const IslandArgs*>(recs), map);
  return true;
}

}  // namespace td1c
