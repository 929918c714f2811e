// psb_two.h -- two stencil stages of a level in one pass over it.
//
// The last pre-sweep and the restriction, and the two post-sweeps, each read
// the level's matrix and right-hand side: as two kernels they stream 37.5 and
// 44.5 bytes a cell (FP16 smoother copy), 107 and 121 (FP64); in one pass 21.5
// and 24.5, 59 and 65.  Here a block marches through the i planes with both
// stages in flight: stage 1 forms plane i of the swept correction while stage 2
// works on plane i - 1 of it.
//   * A thread owns one cell vector of a (j, k) tile.  Two planes of the
//     operand of stage 1 (with a halo row below and above) and of the swept
//     correction are in LDS, and one barrier per plane orders everything.
//   * Stage 1 is needed one cell beyond the tile stage 2 writes: the tile has
//     R + 2 rows of which R are output, a column vector more on each side
//     where the rows are split along k, and a slab of TI planes takes two
//     planes more.  Of a halo vector only the cell next to the tile is used;
//     the others may hold anything.
//   * Matrix, right-hand side and operand of the next plane are loaded a plane
//     ahead; a plane's w couplings are the plane before's e.
// What bounds it: at 256^3 (FP16 copy) the first pair, its operand formed from r
// and c (TwoFirst), takes 385 MB of HBM traffic (1.07 of what it must move) in 99
// us, 3.9 TB/s with the vector units half busy; the post-sweeps 436 MB (1.06) in
// 102 us, 4.3 TB/s.  Measured in traced solves, us, one pass against two kernels:
//   first pair, FP16 copy: 256^3 99 / 78 + 67 (with the first sweep stored, 24 us
//     more in the x/r step: 87), 128^3 19.7 / 11.5 + 9.3, 64^3 8.8, 32^3 8.0 / 4.5 + 5.5
//   first pair, FP64:      256^3 217 / 399, 128^3 30 / 25 + 21, 64^3 9.9, 32^3 7.1 / 3.9 + 4.9
//   post-sweeps, FP16 copy: 256^3 102 / 76 + 81, 128^3 19.0 / 11.5 + 11.7, 64^3 8.6 /
//     4.8 + 4.7, 32^3 8.2 / 4.5 + 4.7
//   post-sweeps, FP64:      256^3 278 / 195 + 214, 128^3 26 / 25 + 21, 64^3 8.9, 32^3
//     6.7 / 4.6 + 4.6
// In untraced solves small levels gain less than these figures say, or lose:
// post_two_pays (psb_api.hip) has what a visit gains there and where the line is.
// The arithmetic is the separate kernels' (gather_c), so that the results are
// bit-identical; only the rho partials are summed over other blocks.
#pragma once

#include "psb_march.h"

namespace psb {

// threads of a block: what the registers allow (two planes of matrix rows
// and the prefetch of a third: about 165)
constexpr int kTwoThreads = 768;

struct TwoShape {
  int RT, KT, KO;  // rows and vectors of a tile (stage 1), its output vectors along k
  int ntj, ntk, TI, nblocks, threads;
  size_t lds;      // elements
};

// Tile and slab for a level: rows whole where four of them fit a block, else
// split along k; of the row counts and slab depths the cheapest by
//   rounds of blocks over the CUs * planes per block * waves on a CU
// (what the redundant rows and planes cost against CUs without a block;
// measured at 256^3, FP32: R = 8 and 32 planes, one block per CU, 90 us, R = 8
// and 16 planes 97, R = 4 and 64 planes 106, R = 10 and 28 planes, 260 blocks,
// 127).  The registers allow 3 waves per SIMD.  nblocks 0: the rows have no
// whole vectors.  The search costs 2 to 30 us of the host, so that it is made
// once per level, and looks at each number of slabs once (at its shallowest
// depth) and at a row count only where it changes the tiles or the waves.
template <typename T>
inline TwoShape two_shape(const Grid &g) {
  constexpr int V = 16 / (int)sizeof(T);
  TwoShape s{};
  if (g.nz % V != 0) return s;
  const int nv = g.nz / V;
  double best = 0.0;
  for (const int KO : {nv, 64, 32, 16}) {
    if (KO > nv || (KO != nv && best > 0.0)) continue;
    const int KT = KO == nv ? nv : KO + 2, ntk = (nv + KO - 1) / KO;
    int waves = 0, ntj = 0;
    for (int R = 2; (R + 2) * KT <= kTwoThreads; R += 2) {
      const size_t lds = (size_t)(2 * (R + 4) + 2 * (R + 2) + R) * KT * V;
      if (lds * sizeof(T) > 150 * 1024) break;
      if (((R + 2) * KT + 63) / 64 == waves && (g.ny + R - 1) / R == ntj) continue;
      waves = ((R + 2) * KT + 63) / 64;
      ntj = (g.ny + R - 1) / R;
      const int per_cu = 12 / waves > 1 ? 12 / waves : 1;
      const long long nt = (long long)ntj * ntk;
      for (int TI = 2, slabs;; TI = ((g.nx + slabs - 2) / (slabs - 1) + 1) & ~1) {
        slabs = (g.nx + TI - 1) / TI;
        const long long nb = nt * slabs, cus = (nb + 255) / 256;
        const long long rounds = (nb + 256 * per_cu - 1) / (256 * per_cu);
        const long long act = cus < per_cu ? cus : per_cu;
        const double cost = (double)rounds * (TI + 2) * (4 + waves * act);
        if (nb < (1 << 30) && !(best > 0.0 && cost >= best)) {
          best = cost;
          s = TwoShape{R + 2, KT, KO, ntj, ntk, TI, (int)nb, waves * 64, lds};
        }
        if (slabs == 1) break;
      }
    }
  }
  return s;
}

// V values at a byte offset from a uniform pointer: the offset of a thread's
// vector in its plane is constant, the plane's base advances in scalar
// registers, and a load takes no vector instruction or register for its
// address.  (The empty asm keeps the base there: the compiler would otherwise
// carry a 64-bit address per array and thread through the loop, and spill.)
template <int BYTES>
struct RawBytes;
template <>
struct RawBytes<16> { using type = uint32_t __attribute__((ext_vector_type(4))); };
template <>
struct RawBytes<8> { using type = uint32_t __attribute__((ext_vector_type(2))); };
template <>
struct RawBytes<4> { using type = uint32_t; };
template <>
struct RawBytes<2> { using type = uint16_t; };
template <>
struct RawBytes<1> { using type = uint8_t; };
#define PSB_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ uint64_t uniform_base(const void *base) {
  const uint64_t b = (uint64_t)base;
  uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
  uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  asm("" : "+s"(lo), "+s"(hi));
  return (uint64_t)hi << 32 | lo;
}
template <typename T, int V>
__device__ __forceinline__ VecN<T, V> ldo(const T *base, uint32_t off) {
  using W = typename RawBytes<(int)sizeof(T) * V>::type;
  const PSB_GLOBAL char *p = (const PSB_GLOBAL char *)uniform_base(base);
  return __builtin_bit_cast(VecN<T, V>, *(const PSB_GLOBAL W *)(p + off));
}
template <typename T, int V>
__device__ __forceinline__ void sto(T *base, uint32_t off, const VecN<T, V> &x) {
  using W = typename RawBytes<(int)sizeof(T) * V>::type;
  PSB_GLOBAL char *p = (PSB_GLOBAL char *)uniform_base(base);
  *(PSB_GLOBAL W *)(p + off) = __builtin_bit_cast(W, x);
}
#undef PSB_GLOBAL
// the active flags of a vector's cells as one word
template <int V>
__device__ __forceinline__ uint32_t ldflags(const uint8_t *base, uint32_t off) {
  const VecN<uint8_t, V> f = ldo<uint8_t, V>(base, off);
  return (uint32_t)__builtin_bit_cast(typename RawBytes<V>::type, f);
}

// a vector's matrix row as loaded: of the couplings, w is the row below's e
template <typename M, int V>
struct TwoRaw {
  VecN<M, V> c, s, b, e, n;
  M bt;
};
// ... and in the working precision, the couplings to e, n and t 0 on the walls
template <typename T, int V>
struct TwoRow {
  VecN<T, V> d, w, e, s, n, b;
  T bt;
  template <typename M>
  __device__ __forceinline__ void take(const TwoRaw<M, V> &C, const VecN<T, V> &below_e,
                                       bool he, bool hn, bool ht) {
    d = cvtv<T, M, V>(C.c);
    w = below_e;
    s = cvtv<T, M, V>(C.s);
    b = cvtv<T, M, V>(C.b);
    e = vsel<T, V>(he, cvtv<T, M, V>(C.e));
    n = vsel<T, V>(hn, cvtv<T, M, V>(C.n));
    bt = ht ? (T)C.bt : T(0);
  }
  // gather_c's terms for the operand x, xw, xe in registers, its plane in LDS
  // at `at` (the neighbours' places relative to it; the cell itself where there
  // is none, its coupling being 0)
  template <bool FLUX>
  __device__ __forceinline__ void gather(const VecN<T, V> &xw, const VecN<T, V> &x,
                                         const VecN<T, V> &xe, const T *at, int os, int on,
                                         int ob, int ot, Gath<T, V> &G) const {
    const VecN<T, V> xs = ldv<T, V>(at + os), xn = ldv<T, V>(at + on);
    const T xb0 = at[ob], xtV = at[ot];
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
  // one damped Jacobi step from the gather: x + omega (r - A x) / c
  template <bool FLUX>
  __device__ __forceinline__ VecN<T, V> sweep(const VecN<T, V> &x, const VecN<T, V> &r,
                                              const Gath<T, V> &G, T omega) const {
    const VecN<T, V> t = resid<T, V>(r, G);
    VecN<T, V> o;
#pragma unroll
    for (int q = 0; q < V; q++) {
      T c = d.v[q];
      if constexpr (FLUX) {
        const T tq = q == V - 1 ? bt : b.v[q + 1];
        const T cc = c + (((w.v[q] + e.v[q]) + (s.v[q] + n.v[q])) + (b.v[q] + tq));
        c = cc > T(0) ? cc : T(1);
      }
      o.v[q] = x.v[q] + omega * t.v[q] / c;
    }
    return o;
  }
};

// a block's tile and slab, a thread's place in it
struct TwoAt {
  int rr, kk, j, k;     // tile row and vector, cell coordinates (clamped into tile and grid)
  int hk, hj, hrow;     // halo vector of the stage 1 operand this thread loads
  int i0, i1;           // the slab's output planes
  bool in, out, halo;   // takes part in stage 1 / stage 2, loads a halo vector
  bool hn, ht;          // has a neighbour at j + 1, at k + V
  int os, on, ob, ot;   // neighbours in an LDS plane
  uint32_t P, HP, Pn, Pt;  // cells in a plane: own and halo vector, j + 1, k + V
};
// thread t of block wi.  A block has whole waves, so that its last threads can
// lie past the tile: they write nothing, and their place is in the tile's last
// row, so that what they read with the others (and use for nothing) is inside
// the block's LDS.  (A branch around that read instead costs the FP64 post-sweeps
// eight more spilled registers: 256^3 solve 29.8 against 29.5 ms.)
template <int V>
__host__ __device__ __forceinline__ TwoAt two_place(const Grid &g, const TwoShape &s, int wi,
                                                    int t) {
  TwoAt a;
  const int per = s.ntj * s.ntk;
  const int slab = wi / per, tile = wi - slab * per;
  const int tj = tile / s.ntk, tk = tile - tj * s.ntk;
  const int nv = g.nz / V;
  const bool split = s.KO < s.KT;
  const int rr = t / s.KT;
  a.rr = rr < s.RT ? rr : s.RT - 1;
  a.kk = t - rr * s.KT;
  const int j0 = tj * (s.RT - 2) - 1, k0 = split ? tk * s.KO - 1 : 0;
  const int j = j0 + rr, kv = k0 + a.kk;
  const bool kin = kv >= 0 && kv < nv;
  a.in = rr < s.RT && j >= 0 && j < g.ny && kin;
  a.out = a.in && a.rr >= 1 && a.rr < s.RT - 1 && (!split || (a.kk >= 1 && a.kk <= s.KO));
  a.j = a.in ? j : 0;
  a.k = a.in ? kv * V : 0;
  // the rows below and above the tile: threads [0, KT) and [KT, 2 KT)
  const int hkk = t < s.KT ? t : t - s.KT;
  const int hj = t < s.KT ? j0 - 1 : j0 + s.RT, hkv = k0 + hkk;
  a.halo = t < 2 * s.KT && hj >= 0 && hj < g.ny && hkv >= 0 && hkv < nv;
  a.hj = a.halo ? hj : 0;
  a.hk = a.halo ? hkv * V : 0;
  a.hrow = (t < s.KT ? 0 : s.RT + 1) * s.KT + hkk;
  a.i0 = slab * s.TI;
  a.i1 = a.i0 + s.TI < g.nx ? a.i0 + s.TI : g.nx;
  a.hn = a.j < g.ny - 1;
  a.ht = a.k + V < g.nz;
  a.os = a.j > 0 ? -s.KT * V : 0;
  a.on = a.hn ? s.KT * V : 0;
  a.ob = a.k > 0 ? -1 : 0;
  a.ot = a.ht ? V : 0;
  a.P = (uint32_t)(a.j * g.nz + a.k);
  a.HP = (uint32_t)(a.hj * g.nz + a.hk);
  a.Pn = a.hn ? a.P + g.nz : a.P;
  a.Pt = a.ht ? a.P + V : a.P;
  return a;
}
template <int V>
__device__ __forceinline__ TwoAt two_at(const Grid &g, const TwoShape &s, int wi) {
  TwoAt a = two_place<V>(g, s, wi, (int)threadIdx.x);
  a.i0 = __builtin_amdgcn_readfirstlane(a.i0);  // (the divisions left them in VGPRs)
  a.i1 = __builtin_amdgcn_readfirstlane(a.i1);
  return a;
}

// stage 1's operand, loaded apart from the arithmetic that forms it (which
// would wait for the loads where it stands): an array, or with the
// prolongation e + cfac * eH[parent] (ProlX; CK the coarsening along k)
template <typename T, int V>
struct TwoArr {
  const T *e;
  int sI;
  struct At {
    uint32_t o;
  };
  using Raw = VecN<T, V>;
  __device__ __forceinline__ At place(int j, int k, int nz) const {
    return At{(uint32_t)(j * nz + k) * (uint32_t)sizeof(T)};
  }
  __device__ __forceinline__ Raw load(int i, const At &a) const {
    return ldo<T, V>(e + (size_t)i * sI, a.o);
  }
  __device__ __forceinline__ VecN<T, V> form(const Raw &x) const { return x; }
};
// the first sweep from zero, omega r / c, formed where it is used: the finest
// level's operand needs neither its writing by the CG step before nor its c there
template <typename T, int V>
struct TwoFirst {
  const T *r, *c;
  T omega;
  int sI;
  struct At {
    uint32_t o;
  };
  struct Raw {
    VecN<T, V> R, C;
  };
  __device__ __forceinline__ At place(int j, int k, int nz) const {
    return At{(uint32_t)(j * nz + k) * (uint32_t)sizeof(T)};
  }
  __device__ __forceinline__ Raw load(int i, const At &a) const {
    return Raw{ldo<T, V>(r + (size_t)i * sI, a.o), ldo<T, V>(c + (size_t)i * sI, a.o)};
  }
  __device__ __forceinline__ VecN<T, V> form(const Raw &x) const {
    VecN<T, V> o;
#pragma unroll
    for (int u = 0; u < V; u++) o.v[u] = omega * x.R.v[u] / x.C.v[u];
    return o;
  }
};
template <typename T, int V, int CK>
struct TwoProl {
  const T *e, *eH;
  const uint8_t *af;
  T cfac;
  int sI, sIH, pI, pJ, nZH;  // plane sizes, coarsening shifts along i and j
  struct At {
    uint32_t o, h, f;
  };
  struct Raw {
    VecN<T, V> E;
    VecN<T, V / CK> H;
    uint32_t f;
  };
  __device__ __forceinline__ At place(int j, int k, int nz) const {
    const uint32_t P = (uint32_t)(j * nz + k);
    return At{P * (uint32_t)sizeof(T), (uint32_t)((j >> pJ) * nZH + k / CK) * (uint32_t)sizeof(T),
              P};
  }
  __device__ __forceinline__ Raw load(int i, const At &a) const {
    Raw x;
    x.E = ldo<T, V>(e + (size_t)i * sI, a.o);
    x.H = ldo<T, V / CK>(eH + (size_t)(i >> pI) * sIH, a.h);
    x.f = af ? ldflags<V>(af + (size_t)i * sI, a.f) : 0xffffffffu;
    return x;
  }
  __device__ __forceinline__ VecN<T, V> form(const Raw &x) const {
    VecN<T, V> o;
#pragma unroll
    for (int u = 0; u < V; u++) {
      const T v = x.E.v[u] + cfac * x.H.v[u / CK];
      o.v[u] = !af || flag_on(x.f, u) ? v : x.E.v[u];
    }
    return o;
  }
};

// the swept correction of plane i in the step after the one that formed it
template <typename T, int V>
__device__ __forceinline__ VecN<T, V> two_swept(const TwoShape &s, const TwoAt &a, const T *lds,
                                                int i) {
  const int pitch = s.KT * V;
  return ldv<T, V>(lds + (2 * (s.RT + 2) + (i & 1) * s.RT + a.rr) * pitch + a.kk * V);
}

// both stages over the block's slab.  base: the operand of stage 1; top(i):
// the first thing in the step whose stage 2 works on plane i (global stores
// belong here; two_swept gives the swept correction there); pre(i): what that stage 2
// reads besides; st2(i, G, R, E, p): stage 2 on an output vector (G its gather
// over the swept correction E, p what pre gave); plane(i): every thread, after
// the step's barrier; lds: the stages' planes.
// Loads and stores share one in-order counter, and a wait for a value waits for
// everything before it: hence per step first the stores, then what this step
// needs, then the next step's loads, all without branches (where a plane is not
// needed its loads repeat the current one), so that nothing in the step waits
// for the prefetch.  Two steps per turn of the loop, so that the matrix rows of
// two planes swap roles without moves.
template <typename T, int V, typename M, bool FLUX, class B, class Top, class Pre, class S2,
          class Plane>
__device__ __forceinline__ void two_march(const Grid &g, const DMat<M> &A, const T *r,
                                          const B &base, T omega, const TwoShape &s,
                                          const TwoAt &a, T *lds, Top top, Pre pre, S2 st2,
                                          Plane plane) {
  const int pitch = s.KT * V, n0 = (s.RT + 2) * pitch, n1 = s.RT * pitch;
  T *const own0 = lds + (a.rr + 1) * pitch + a.kk * V;
  T *const own1 = lds + 2 * n0 + a.rr * pitch + a.kk * V;
  T *const halo0 = lds + a.hrow * V;
  const auto at = base.place(a.j, a.k, g.nz), hat = base.place(a.hj, a.hk, g.nz);
  const uint32_t oT = a.P * (uint32_t)sizeof(T), oM = a.P * (uint32_t)sizeof(M),
                 oN = a.Pn * (uint32_t)sizeof(M), oB = a.Pt * (uint32_t)sizeof(M);
  auto raw = [&](int i) {
    const size_t p = (size_t)i * g.sI;
    TwoRaw<M, V> C;
    C.c = ldo<M, V>(A.c + p, oM);
    C.s = ldo<M, V>(A.s + p, oM);
    C.b = ldo<M, V>(A.b + p, oM);
    C.e = ldo<M, V>(A.w + (i < g.nx - 1 ? p + g.sI : p), oM);
    C.n = ldo<M, V>(A.s + p, oN);
    C.bt = ldo<M, 1>(A.b + p, oB).v[0];
    return C;
  };
  const int ia = max(a.i0 - 1, 0), last = g.nx - 1;
  VecN<T, V> next = base.form(base.load(min(ia + 1, last), at));
  VecN<T, V> R = ldo<T, V>(r + (size_t)ia * g.sI, oT), Rp = R;
  // own column: the operand's planes i - 1 and i and the swept correction's
  // i - 1 and i - 2 are read from LDS in each step rather than kept in registers
  // the loop has none left for.  Plane i + 1 takes the place of i - 1 at a
  // step's end: only its own thread reads that.
  const int ip = (ia & 1) ^ 1;
  if (a.in) {
    stv<T, V>(own0 + ip * n0, base.form(base.load(max(ia - 1, 0), at)));
    stv<T, V>(own0 + (n0 - ip * n0), base.form(base.load(ia, at)));
    stv<T, V>(own1, zerov<T, V>());
    stv<T, V>(own1 + n1, zerov<T, V>());
  }
  if (a.halo) stv<T, V>(halo0 + (n0 - ip * n0), base.form(base.load(ia, hat)));
  TwoRow<T, V> row0, row1;
  row0.take(raw(ia), cvtv<T, M, V>(ldo<M, V>(A.w + (size_t)ia * g.sI, oM)), ia < last, a.hn, a.ht);
  row1 = row0;
  __builtin_amdgcn_s_waitcnt(0);  // nothing of the first loads pending inside the loop
  // the step whose stage 1 works on plane i with row, stage 2 on i - 1 with rowp;
  // rowp becomes plane i + 1's
  auto step = [&](int i, const TwoRow<T, V> &row, TwoRow<T, V> &rowp) {
    const bool sweep = i <= last, stage2 = i > a.i0;
    if (stage2) top(i - 1);
    const auto pv = pre(max(i - 1, 0));
    const int in = min(min(i + 1, a.i1), last);
    const auto nn = base.load(min(min(i + 2, a.i1 + 1), last), at), hn = base.load(in, hat);
    const TwoRaw<M, V> C = raw(in);
    const VecN<T, V> Rn = ldo<T, V>(r + (size_t)in * g.sI, oT);
    // this plane's places in LDS (opaque to the compiler, which would otherwise
    // keep every neighbour's address of both parities in a register and spill:
    // a spill's reload waits for the prefetch)
    int p0 = (i & 1) * n0, p1 = (i & 1) * n1;
    asm volatile("" : "+s"(p0), "+s"(p1));
    __syncthreads();
    if (stage2) plane(i - 1);
    VecN<T, V> x0 = zerov<T, V>();
    const VecN<T, V> x2 = ldv<T, V>(own1 + p1);
    if (sweep && a.in) {
      Gath<T, V> G;
      const VecN<T, V> prev = ldv<T, V>(own0 + (n0 - p0)), cur = ldv<T, V>(own0 + p0);
      row.template gather<FLUX>(prev, cur, next, own0 + p0, a.os, a.on, a.ob, a.ot, G);
      x0 = row.template sweep<FLUX>(cur, R, G, omega);
      stv<T, V>(own1 + p1, x0);
    }
    if (stage2 && a.out) {
      Gath<T, V> G;
      const VecN<T, V> x1 = ldv<T, V>(own1 + (n1 - p1));
      rowp.template gather<FLUX>(x2, x1, x0, own1 + (n1 - p1), a.os, a.on, a.ob, a.ot, G);
      st2(i - 1, G, Rp, rowp, x1, pv);
    }
    if (a.in) stv<T, V>(own0 + (n0 - p0), next);
    if (a.halo) stv<T, V>(halo0 + (n0 - p0), base.form(hn));
    next = base.form(nn);
    Rp = R;
    R = Rn;
    rowp.take(C, row.e, in < last, a.hn, a.ht);
  };
  for (int i = ia;; i += 2) {
    step(i, row0, row1);
    if (i + 1 > a.i1) break;
    step(i + 1, row1, row0);
    if (i + 2 > a.i1) break;
  }
}

// the last pre-sweep eout = e + omega (r - A e) / c and the restriction of
// r - A eout with the coarse level's first sweep (as k_jacobi and k_restrict,
// CI = CJ = 2).  A coarse cell's sum runs in (i, j, k) order: the even row's
// thread adds its own residuals and, a step later, the odd row's from LDS.
// (block wi of s.nblocks)
template <typename T, int V, typename M, bool FLUX, int CK, class B>
__device__ __forceinline__ void pre_restrict_body(int wi, Grid g, DMat<M> A, const T *r, const B &e,
                                                  T *eout, const uint8_t *af, Grid gH, const T *cH,
                                                  const uint8_t *afH, T *rH, T *eH1, T omega,
                                                  T omegaH, TwoShape s) {
  extern __shared__ __align__(16) char two_lds[];
  T *const lds = reinterpret_cast<T *>(two_lds);
  const TwoAt a = two_at<V>(g, s, wi);
  const int pitch = s.KT * V, nt = (s.RT - 2) / 2 * pitch;
  T *const lt = lds + (2 * (s.RT + 2) + 2 * s.RT) * pitch;  // odd rows' residuals, two planes
  const bool odd = (a.rr & 1) == 0;  // output row rr - 1
  const int mine = (a.rr - 1) / 2 * pitch + a.kk * V;
  constexpr int NC = V / CK;
  T sum[NC], done[NC];  // running sums; a finished coarse plane's
  VecN<T, NC> cq{};     // the coarse diagonal
  uint32_t act = 0;     // ... and flags
  int Qd = -1;  // the finished coarse plane
#pragma unroll
  for (int u = 0; u < NC; u++) sum[u] = done[u] = T(0);
  const uint32_t QH = (uint32_t)((a.j >> 1) * gH.nz + a.k / CK);
  // the odd row's residuals of plane p, and after an odd plane the coarse cells
  auto add_odd = [&](int p) {
    const VecN<T, V> t = *reinterpret_cast<const VecN<T, V> *>(lt + (p & 1) * nt + mine);
#pragma unroll
    for (int u = 0; u < NC; u++)
#pragma unroll
      for (int c = 0; c < CK; c++) sum[u] += t.v[u * CK + c];
    if (p & 1) {
#pragma unroll
      for (int u = 0; u < NC; u++) {
        done[u] = sum[u];
        sum[u] = T(0);
      }
    }
  };
  auto store = [&]() {
    if (Qd < 0) return;
    const size_t at = (size_t)Qd * gH.sI;
    Qd = -1;
    if (!a.out || odd) return;
    VecN<T, NC> rq, eq;
#pragma unroll
    for (int u = 0; u < NC; u++) {
      rq.v[u] = !afH || flag_on(act, u) ? done[u] : T(0);
      eq.v[u] = omegaH * rq.v[u] / cq.v[u];
    }
    sto<T, NC>(rH + at, QH * (uint32_t)sizeof(T), rq);
    sto<T, NC>(eH1 + at, QH * (uint32_t)sizeof(T), eq);
  };
  // called in the step whose stage 2 works on the even plane i: coarse plane
  // i / 2 - 1 is finished in it
  auto load_c = [&](int i) {
    const size_t p = (size_t)max(i / 2 - 1, 0) * gH.sI;
    cq = ldo<T, NC>(cH + p, QH * (uint32_t)sizeof(T));
    if (afH) act = ldflags<NC>(afH + p, QH);
  };
  two_march<T, V, M, FLUX>(
      g, A, r, e, omega, s, a, lds,
      [&](int i) {
        if (a.out)
          sto<T, V>(eout + (size_t)i * g.sI, a.P * (uint32_t)sizeof(T),
                    two_swept<T, V>(s, a, lds, i));
        store();
      },
      [&](int i) {
        if (!(i & 1)) load_c(i);
        return af ? ldflags<V>(af + (size_t)i * g.sI, a.P) : 0xffffffffu;
      },
      [&](int i, const Gath<T, V> &G, const VecN<T, V> &R, const TwoRow<T, V> &,
          const VecN<T, V> &, uint32_t fw) {
        VecN<T, V> t = resid<T, V>(R, G);
        if (af) {
#pragma unroll
          for (int u = 0; u < V; u++) t.v[u] = keep_if(flag_on(fw, u), t.v[u]);
        }
        if (odd) {
          stv<T, V>(lt + (i & 1) * nt + mine, t);
        } else {
#pragma unroll
          for (int u = 0; u < NC; u++)
#pragma unroll
            for (int c = 0; c < CK; c++) sum[u] += t.v[u * CK + c];
        }
      },
      [&](int i) {
        if (i <= a.i0) return;
        if ((i - 1) & 1) Qd = (i - 1) >> 1;
        if (a.out && !odd) add_odd(i - 1);
      });
  __syncthreads();
  store();
  if (a.out && !odd) add_odd(a.i1 - 1);
  load_c(a.i1);
  Qd = (a.i1 - 1) >> 1;
  store();
}

// (FIRST: the operand is the first sweep om0 r / c, e is not read)
template <typename T, int V, typename M, bool FLUX, int CK, bool FIRST>
__global__ __launch_bounds__(kTwoThreads) void k_pre_restrict(
    Grid g, DMat<M> A, const T *r, const T *e, const T *c, T om0, T *eout, const uint8_t *af,
    Grid gH, const T *cH, const uint8_t *afH, T *rH, T *eH1, T omega, T omegaH,
    const DevState *st, TwoShape s) {
  if (skip_done(st, g.N)) return;
  if constexpr (FIRST)
    pre_restrict_body<T, V, M, FLUX, CK>(xcd_block(), g, A, r, TwoFirst<T, V>{r, c, om0, g.sI},
                                         eout, af, gH, cH, afH, rH, eH1, omega, omegaH, s);
  else
    pre_restrict_body<T, V, M, FLUX, CK>(xcd_block(), g, A, r, TwoArr<T, V>{e, g.sI}, eout, af,
                                         gH, cH, afH, rH, eH1, omega, omegaH, s);
}

// the two post-sweeps of a level, the prolongation of eH fused into the first
// (as k_jacobi with PROL, then without); RHO: the finest level, whose second
// sweep leaves z times zscale and the rho partials (rho_accq), one set per
// block (zeros past the last)
template <typename T, int V, typename M, bool FLUX, int CK, bool RHO>
__device__ __forceinline__ void post_two_body(int wi, Grid g, DMat<M> A, const T *r,
                                              TwoProl<T, V, CK> pr, T *eout, T omega, T zscale,
                                              const uint8_t *af, const T *qf, Work w,
                                              TwoShape s) {
  if (wi >= s.nblocks) {
    if (RHO && threadIdx.x < kRhoParts)
      w.partial[(size_t)blockIdx.x * kRhoParts + threadIdx.x] = 0.0;
    return;
  }
  extern __shared__ __align__(16) char two_lds[];
  T *const lds = reinterpret_cast<T *>(two_lds);
  const TwoAt a = two_at<V>(g, s, wi);
  const uint32_t oT = a.P * (uint32_t)sizeof(T);
  double acc[kRhoParts] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int count = 0;   // active cells (an integer takes half the registers)
  VecN<T, V> z{};  // a plane's result, stored a step later
  struct Q {
    VecN<T, V> q;
    uint32_t f;
  };
  auto put = [&](int i) {
    if (a.out) sto<T, V>(eout + (size_t)i * g.sI, oT, z);
  };
  two_march<T, V, M, FLUX>(
      g, A, r, pr, omega, s, a, lds, [&](int i) {
        if (i > a.i0) put(i - 1);
      },
      [&](int i) {
        Q o{};
        if constexpr (RHO) {
          o.q = ldo<T, V>((qf ? qf : r) + (size_t)i * g.sI, oT);
          o.f = af ? ldflags<V>(af + (size_t)i * g.sI, a.P) : 0xffffffffu;
        }
        return o;
      },
      [&](int, const Gath<T, V> &G, const VecN<T, V> &R, const TwoRow<T, V> &row,
          const VecN<T, V> &E, const Q &o) {
        z = row.template sweep<FLUX>(E, R, G, omega);
        if constexpr (RHO) {
#pragma unroll
          for (int u = 0; u < V; u++) {
            z.v[u] = zscale * z.v[u];
            const bool on = !af || flag_on(o.f, u);
            rho_accq<T, false>(acc, R.v[u], z.v[u], qf != nullptr, o.q.v[u], on);
            count += on ? 1 : 0;
          }
        }
      },
      [](int) {});
  put(a.i1 - 1);
  if constexpr (RHO) {
    acc[3] = (double)count;
    // one partial per block: wave sums, then the waves in turn
    __shared__ double sm[kTwoThreads / 64][kRhoParts];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
#pragma unroll
    for (int q = 0; q < kRhoParts; q++) {
      const double v = wave_sum(acc[q]);
      if (lane == 0) sm[wid][q] = v;
    }
    __syncthreads();
    if (threadIdx.x < kRhoParts) {
      double t = 0.0;
      for (int q = 0; q < nw; q++) t += sm[q][threadIdx.x];
      w.partial[(size_t)blockIdx.x * kRhoParts + threadIdx.x] = t;
    }
  }
}

template <typename T, int V, typename M, bool FLUX, int CK, bool RHO>
__global__ __launch_bounds__(kTwoThreads) void k_post_two(Grid g, DMat<M> A, const T *r,
                                                          TwoProl<T, V, CK> pr, T *eout, T omega,
                                                          T zscale, const uint8_t *af,
                                                          const T *qf, const DevState *st, Work w,
                                                          TwoShape s) {
  if (skip_done(st, g.N)) return;
  post_two_body<T, V, M, FLUX, CK, RHO>(xcd_block(), g, A, r, pr, eout, omega, zscale, af, qf, w,
                                        s);
}

}  // namespace psb
