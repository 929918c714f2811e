// psb_tail.h -- the lowest smoothing level of the multigrid cycle in one
// workgroup.
//
// The level above the coarsest holds a few thousand cells: a launch there is
// all latency (about 4.2 us each in the 256^3 mixed solve, 1.7 us of it the
// graph node), and the K-cycle visits it most often: 13 launches per K-step
// of the 16^3 level, four K-steps per CG iteration.  Here a workgroup of 1024
// threads holds the whole level -- matrix and right-hand side in registers,
// the correction in LDS -- so that sweeps, restriction, prolongation and the
// K-step's dot products follow each other with workgroup barriers.  The one
// part a single CU cannot do is the coarsest level's dense product (2 MB of
// FP64 at 8^3): a launch that ends in it runs a workgroup per 16 rows (one
// per wave), all of them descending redundantly on the same data, workgroup 0
// alone writing what later launches read.  A cycle is then two launches and a
// K-step three:
//   descent                pre-sweeps, restriction, rows of z = G r
//   ascent                 prolongation and post-sweeps
//   ascent + K + descent   first cycle's end, alpha1, residual update, second
//                          cycle's descent
//   ascent + combination   second cycle's end, alpha2, z = a c + alpha2 d
// What bounds it now is instruction issue on one CU: 16 waves on 4 SIMDs take
// 6.7 ns per instruction of the kernel, a sweep 0.6 us.  Hence one cell vector
// per thread at most (kTailVec): levels of two per thread measured no faster
// than their separate launches (FP64 16^3 level: 52 us per K-step against 55;
// two levels of 12x12x48 and 12x12x24 in one launch: 33 us per visit against
// 31).  Measured at 16^3 in FP32 (K-step): 8.4 + 12.9 + 9.8 us where the
// thirteen launches took 55 us with their gaps; 128^3 time step 12.5 -> 10.6 ms,
// 256^3 mixed solve 20.5 -> 18.6 ms (mean of three systems).
// The arithmetic is that of the span kernels (k_jacobi, k_restrict, k_gemv,
// k_kc_*), and the dot products are summed in the order of their blocks and
// of fin_sum: results are bit-identical.
#pragma once

#include "psb_kernels.h"

namespace psb {

constexpr int kTailBlock = 1024;
constexpr int kTailWaves = kTailBlock / 64;
constexpr int kTailVec = kTailBlock;  // cell vectors of the level at most

template <typename T, typename M>
struct TailArgs {
  Grid g, gc;             // the level, the coarsest level
  DMat<M> A;              // the smoother's matrix
  DMat<T> K;              // the level's own
  const uint8_t *af, *afc;
  const T *c;             // diagonal of the first sweep
  int sI, sJ, sK;         // coarsening shifts
  int nu1, nu2;
  T omega, om0, cfac, kscale;  // om0: omega / scale (first sweep)
  int m;                  // coarsest cells
  const double *G;
  // right-hand side; the first sweep (descent) or the pre-smoothed correction
  // (ascent) and the coarsest level's correction.  The output arrays differ
  // from the inputs: all workgroups read, workgroup 0 writes.
  const T *r, *e, *zin;
  T *eout, *zout, *out;   // pre-smoothed correction, coarsest correction, the ascent's result
  T *kc, *kv, *krt;       // K-step: first correction, A of it, updated right-hand side
  double *kst;
};

// a / c by its correctly rounded reciprocal rc, as the division rounds it:
// the product is within two units in the last place, each step's remainder is
// exact, so the first leaves a faithful quotient and the second the rounded one
// (P. Markstein, IBM J. Res. Dev. 34 (1990) 111-119).  That holds while c, rc, the
// quotient and the remainder are normal numbers: numerators below some 1e-31
// (FP32; FP64 1e-291) can round their last bit the other way, an infinite one gives
// NaN where the division gives infinity.  (The preconditioner's values there have
// lost their digits or the solve has ended: solves with the right-hand side scaled
// by 1e-300 to 1e300 are those of the separate kernels, NaN for NaN.)  Five
// instructions where the division takes eleven (FP32) or more; the sweeps divide by
// one diagonal over and over.
__device__ __forceinline__ float div_by(float a, float c, float rc) {
  float q = a * rc;
  q = __builtin_fmaf(__builtin_fmaf(-c, q, a), rc, q);
  return __builtin_fmaf(__builtin_fmaf(-c, q, a), rc, q);
}
__device__ __forceinline__ double div_by(double a, double c, double rc) {
  double q = a * rc;
  q = __builtin_fma(__builtin_fma(-c, q, a), rc, q);
  return __builtin_fma(__builtin_fma(-c, q, a), rc, q);
}

// where a cell vector's neighbours lie in the level's operand: the cell
// itself where there is none (the coupling is 0 there)
struct TailAt {
  int P, w, e, s, n, b, t;
};

// a cell vector's row of the matrix in the working precision, the couplings
// to e, n and t as the neighbours' w, s and b, 0 on the walls
template <typename T, int V>
struct TailRow {
  VecN<T, V> d, w, e, s, n, b;
  T bt;
  template <typename M>
  __device__ __forceinline__ void load(const Grid &g, const DMat<M> &A, int P, int i, int j,
                                       int k) {
    const Coef<M, V, true> C = load_coef<M, V, true>(g, A, P, i, j, k);
    d = cvtv<T, M, V>(C.c);
    w = cvtv<T, M, V>(C.w);
    s = cvtv<T, M, V>(C.s);
    b = cvtv<T, M, V>(C.b);
    e = vsel<T, V>(i < g.nx - 1, cvtv<T, M, V>(C.e));
    n = vsel<T, V>(j < g.ny - 1, cvtv<T, M, V>(C.n));
    bt = k + V < g.nz ? (T)C.bt : T(0);
  }
  // the gather of gather_c for the operand x (also in buf)
  template <bool FLUX>
  __device__ __forceinline__ void gather(const VecN<T, V> &x, const T *buf, const TailAt &at,
                                         Gath<T, V> &G) const {
    const VecN<T, V> xw = ldv<T, V>(buf + at.w), xe = ldv<T, V>(buf + at.e);
    const VecN<T, V> xs = ldv<T, V>(buf + at.s), xn = ldv<T, V>(buf + at.n);
    const T xb0 = buf[at.b], xtV = buf[at.t];
#pragma unroll
    for (int q = 0; q < V; q++) {
      const T xb = q == 0 ? xb0 : x.v[q - 1], xt = q == V - 1 ? xtV : x.v[q + 1];
      const T tq = q == V - 1 ? bt : b.v[q + 1], xq = x.v[q];
      G.cx.v[q] = d.v[q] * xq;
      if constexpr (FLUX) {
        G.s1.v[q] = w.v[q] * (xw.v[q] - xq) + e.v[q] * (xe.v[q] - xq);
        G.s2.v[q] = s.v[q] * (xs.v[q] - xq) + n.v[q] * (xn.v[q] - xq);
        G.s3.v[q] = b.v[q] * (xb - xq) + tq * (xt - xq);
      } else {
        G.s1.v[q] = w.v[q] * xw.v[q] + e.v[q] * xe.v[q];
        G.s2.v[q] = s.v[q] * xs.v[q] + n.v[q] * xn.v[q];
        G.s3.v[q] = b.v[q] * xb + tq * xt;
      }
    }
  }
  // the Jacobi divisor (gather_c's G.c)
  template <bool FLUX>
  __device__ __forceinline__ VecN<T, V> diag() const {
    VecN<T, V> c;
#pragma unroll
    for (int q = 0; q < V; q++) {
      const T tq = q == V - 1 ? bt : b.v[q + 1];
      const T cc = d.v[q] + (((w.v[q] + e.v[q]) + (s.v[q] + n.v[q])) + (b.v[q] + tq));
      c.v[q] = !FLUX ? d.v[q] : cc > T(0) ? cc : T(1);
    }
    return c;
  }
};

// a thread's cell vector: vector tid % 256 of block tid / 256 of the span
// kernels' grid (at most 4 blocks, whose order no remap changes)
template <typename T, int V>
struct TailTile {
  TailRow<T, V> A;
  VecN<T, V> c, rc, R, E;
  TailAt at;
  int i, j, k, nb;
  bool act;

  __device__ __forceinline__ void place(const Grid &g) {
    const int nvec = g.N / V;
    nb = (nvec + kBlock - 1) / kBlock;
    const int per = (nvec + nb - 1) / nb, t = (int)threadIdx.x & (kBlock - 1);
    const int q = ((int)threadIdx.x >> 8) * per + t;
    act = t < per && q < nvec;
    const int P = act ? q * V : 0;
    g.ijk(P, i, j, k);
    at.P = P;
    at.w = i > 0 ? P - g.sI : P;
    at.e = i < g.nx - 1 ? P + g.sI : P;
    at.s = j > 0 ? P - g.nz : P;
    at.n = j < g.ny - 1 ? P + g.nz : P;
    at.b = k > 0 ? P - 1 : P;
    at.t = k + V < g.nz ? P + V : P;
  }
  __device__ __forceinline__ void put(T *buf, const VecN<T, V> &x) const {
    if (act) stv<T, V>(buf + at.P, x);
  }
};

// nu sweeps on the operand in buf (on entry written, not yet waited for); the
// result in tl.E and in buf (waited for)
template <bool FLUX, typename T, int V>
__device__ __forceinline__ void tail_sweeps(TailTile<T, V> &tl, T *buf, T omega, int nu) {
  __syncthreads();
#pragma unroll 1
  for (int s = 0; s < nu; s++) {
    Gath<T, V> G;
    tl.A.template gather<FLUX>(tl.E, buf, tl.at, G);
    const VecN<T, V> t = resid<T, V>(tl.R, G);
#pragma unroll
    for (int u = 0; u < V; u++)
      tl.E.v[u] = tl.E.v[u] + div_by(omega * t.v[u], tl.c.v[u], tl.rc.v[u]);
    __syncthreads();
    tl.put(buf, tl.E);
    __syncthreads();
  }
}

// totals over the level in the order of the span kernels' reductions: wave
// sums, the four waves of a block in turn, then fin_sum's sum over the blocks;
// left in st (not yet waited for)
template <int NR, typename T, int V>
__device__ __forceinline__ void tail_sum(const TailTile<T, V> &tl, const double (&acc)[NR],
                                         double (&tot)[NR], double (*sm)[NR]) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const double w = wave_sum(acc[r]);
    if (lane == 0) sm[wid][r] = w;
  }
  __syncthreads();
  if (wid != 0) return;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    double p = 0.0;
    if (lane < tl.nb)
      for (int q = 0; q < kWaves; q++) p += sm[lane * kWaves + q][r];
    tot[r] = 0.0 + wave_sum(0.0 + p);
  }
}

// UP: ascent from zin; KMID / KEND: the K-step's middle and end; DOWN: descent
// to zout
template <typename T, int V, typename M, bool FLUX, bool UP, bool KMID, bool KEND, bool DOWN>
__global__ __launch_bounds__(kTailBlock) void k_tail(TailArgs<T, M> a) {
  extern __shared__ __align__(16) char tail_lds[];
  T *const buf = reinterpret_cast<T *>(tail_lds), *const zbuf = buf + a.g.N;
  constexpr int NR = KMID ? 2 : 3;
  __shared__ double sm[kTailWaves][NR], ks[2];
  const Grid &g = a.g;
  TailTile<T, V> tl;
  tl.place(g);
  const int P = tl.at.P;
  // everything from memory in one round: the level, the coarsest level's
  // correction, the K-step's data, the first columns of this wave's row of G
  tl.A.load(g, a.A, P, tl.i, tl.j, tl.k);
  tl.R = ldv<T, V>(a.r + P);
  tl.E = ldv<T, V>(a.e + P);
  const uint32_t fw = flag_word<V>(a.af, P, a.c);
  constexpr bool OWNK = std::is_same<T, M>::value;  // the smoother's matrix is the level's own
  TailRow<T, V> Kr;
  VecN<T, V> Kv, Kc;
  double rho1 = 0.0, al1 = 0.0;
  if constexpr (!OWNK && (KMID || KEND)) Kr.load(g, a.K, P, tl.i, tl.j, tl.k);
  if constexpr (KMID) Kc = ldv<T, V>(a.c + P);  // the second first sweep's divisor
  if constexpr (KEND) {
    Kv = ldv<T, V>(a.kv + P);
    Kc = ldv<T, V>(a.kc + P);
    rho1 = a.kst[0];
    al1 = a.kst[1];
  }
  const int lane = (int)threadIdx.x & 63;
  const int row = (int)blockIdx.x * kTailWaves + ((int)threadIdx.x >> 6);
  const double *grow = a.G + (size_t)min(row, a.m - 1) * a.m;
  double g8[8];
  auto load_g = [&]() {
#pragma unroll
    for (int q = 0; q < 8; q++) g8[q] = grow[min(lane + 64 * q, a.m - 1)];
  };
  if constexpr (DOWN && !KMID) load_g();  // (with KMID later: registers)
  if constexpr (UP)
    for (int Q = (int)threadIdx.x; Q < a.m; Q += kTailBlock) zbuf[Q] = a.zin[Q];
  tl.c = tl.A.template diag<FLUX>();
#pragma unroll
  for (int u = 0; u < V; u++) tl.rc.v[u] = T(1) / tl.c.v[u];
  if constexpr (UP) {
    // e + cfac P zH, then the post-sweeps
    __syncthreads();
    const int base = ((tl.i >> a.sI) * a.gc.ny + (tl.j >> a.sJ)) * a.gc.nz;
#pragma unroll
    for (int u = 0; u < V; u++) {
      const T h = zbuf[base + ((tl.k + u) >> a.sK)];
      tl.E.v[u] = flag_on(fw, u) ? tl.E.v[u] + a.cfac * h : tl.E.v[u];
    }
    tl.put(buf, tl.E);
    tail_sweeps<FLUX>(tl, buf, a.omega, a.nu2);
    if constexpr (!KMID && !KEND) tl.put(a.out, tl.E);
  }
  if constexpr (KMID || KEND) {
    // s A c (KMID: v) or s A d (KEND) with the level's own matrix
    Gath<T, V> G;
    if constexpr (OWNK) tl.A.template gather<FLUX>(tl.E, buf, tl.at, G);
    else Kr.template gather<FLUX>(tl.E, buf, tl.at, G);
    VecN<T, V> Av = apply_A<T, V>(G);
    double acc[NR] = {}, tot[NR];
#pragma unroll
    for (int u = 0; u < V; u++) {
      Av.v[u] = a.kscale * Av.v[u];
      const double x = (double)tl.E.v[u];
      if constexpr (KMID) {
        acc[0] += x * (double)Av.v[u];
        acc[1] += x * (double)tl.R.v[u];
      } else {
        acc[0] += x * (double)Kv.v[u];
        acc[1] += x * (double)Av.v[u];
        acc[2] += x * (double)tl.R.v[u];
      }
    }
    if (!tl.act)
      for (double &v : acc) v = 0.0;
    tail_sum<NR>(tl, acc, tot, sm);
    if (threadIdx.x == 0) {
      if constexpr (KMID) {
        ks[0] = tot[0] > 0.0 ? tot[1] / tot[0] : 0.0;
        if (blockIdx.x == 0) {
          a.kst[0] = tot[0];
          a.kst[1] = ks[0];
        }
      } else {
        const double den = rho1 > 0.0 ? tot[1] - tot[0] * tot[0] / rho1 : 0.0;
        const double a2 = den > 0.0 ? tot[2] / den : 0.0;
        ks[0] = al1 - (rho1 > 0.0 ? tot[0] * a2 / rho1 : 0.0);
        ks[1] = a2;
        a.kst[2] = ks[0];
        a.kst[3] = a2;
      }
    }
    __syncthreads();
    if constexpr (KMID) {
      // rt = r - alpha1 v and the second cycle's first sweep
      const T a1 = (T)ks[0];
      if (blockIdx.x == 0) {
        tl.put(a.kc, tl.E);
        tl.put(a.kv, Av);
      }
#pragma unroll
      for (int u = 0; u < V; u++) {
        tl.R.v[u] = tl.R.v[u] - a1 * Av.v[u];
        tl.E.v[u] = a.om0 * tl.R.v[u] / Kc.v[u];
      }
      if (blockIdx.x == 0) tl.put(a.krt, tl.R);
    } else {
      const T ac = (T)ks[0], a2 = (T)ks[1];
      VecN<T, V> O;
#pragma unroll
      for (int u = 0; u < V; u++) O.v[u] = ac * Kc.v[u] + a2 * tl.E.v[u];
      tl.put(a.out, O);
    }
  }
  if constexpr (DOWN) {
    if constexpr (KMID) load_g();
    tl.put(buf, tl.E);
    tail_sweeps<FLUX>(tl, buf, a.omega, a.nu1 - 1);
    if (blockIdx.x == 0) tl.put(a.eout, tl.E);
    // the residual, then its block sums into the coarsest right-hand side
    Gath<T, V> G;
    tl.A.template gather<FLUX>(tl.E, buf, tl.at, G);
    VecN<T, V> t = resid<T, V>(tl.R, G);
#pragma unroll
    for (int u = 0; u < V; u++) t.v[u] = keep_if(flag_on(fw, u), t.v[u]);
    __syncthreads();
    tl.put(buf, t);
    __syncthreads();
    for (int Q = (int)threadIdx.x; Q < a.m; Q += kTailBlock) {
      int I, J, K;
      a.gc.ijk(Q, I, J, K);
      const int F = ((I << a.sI) * g.ny + (J << a.sJ)) * g.nz + (K << a.sK);
      T s = T(0);
      for (int ci = 0; ci <= a.sI; ci++)
        for (int cj = 0; cj <= a.sJ; cj++)
          for (int ck = 0; ck <= a.sK; ck++) s += buf[F + ci * g.sI + cj * g.nz + ck];
      zbuf[Q] = keep_if(flag_on(flag_word<1>(a.afc, Q, a.c), 0), s);
    }
    __syncthreads();
    // this workgroup's rows of z = G r, one per wave (as k_gemv)
    if (row < a.m) {
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (lane + 64 * q < a.m) s += g8[q] * (double)zbuf[lane + 64 * q];
#pragma unroll 8
      for (int c = lane + 512; c < a.m; c += 64) s += grow[c] * (double)zbuf[c];
      s = wave_sum(s);
      if (lane == 0) a.zout[row] = (T)s;
    }
  }
}

}  // namespace psb
