// psb_dense.h -- the coarsest level's dense operator on the device:
// G = Pi (A_pinned)^-1 Pi over the active cells (dense_pinv in psb_api.hip says
// what it is and computes it where the band is too wide for this form).
//
// k_band_chol: banded Cholesky in one workgroup, right-looking, the window of
// the bw + 1 rows that a step touches in LDS.  Row i and column j of it sit in
// slots i, j modulo bw + 1, a pair of slots in one place whatever their order
// (the window is symmetric): (bw + 1)(bw + 2) / 2 values.  A step divides the
// column by its pivot and subtracts its products: per entry the same operations
// in the same order as dense_pinv's row-by-row form.
// k_band_inverse: the columns of the inverse, one wave each: two triangular
// solves by columns with the right-hand side in LDS.  Also the columns' sums.
// k_band_rows, k_band_total, k_band_project: the rows' sums, the sum of all
// entries, and G with the means taken off.  Every sum runs in dense_pinv's
// order: G is the same to the last bit.
// What bounds it: the chain of m steps, each a square root, a division, two
// barriers and the products (U per thread of one compute unit).  Measured:
// 8^3 cells (band 64) 0.55 ms for the factor, 0.29 for the inverse and 0.3 for
// the sums, against 2.7 ms on 16 host threads with the copies; 12^3 (144)
// 4.0 + 1.3 + 1.8 against 51.
// The line (kBandMax) is where the window stops fitting the LDS.
#pragma once

#include "psb_kernels.h"

namespace psb {

constexpr int kBandThreads = 1024;
// widest band whose window fits the LDS (154 KB at 195)
constexpr int kBandMax = 195;
constexpr int kBandMaxCells = 4096;  // two dense m x m arrays of 134 MB

struct BandArgs {
  int nx, ny, nz, bw;
  const double *c, *w, *s, *b;
  const uint8_t *act;  // NULL: all active
  double *Lc, *Lr;     // L[k + d][k] and L[i][i - d] at (k or i) * (bw + 1) + d
};

__device__ __forceinline__ int band_at(int a, int b) {
  const int hi = max(a, b), lo = min(a, b);
  return (int)(__umul24(hi, hi + 1) >> 1) + lo;
}

// entry (i, j) of the matrix, j <= i (0 beyond the last row; jj, kk row i's
// place along y and z): loaded without a branch, so that it can be under way
// while another step works
struct BandEntry {
  double v;
  uint8_t ai, aj;
  int sign;  // 1 the diagonal, -1 a coupling, 0 none
  __device__ __forceinline__ void load(const BandArgs &A, int m, int i, int j, int jj, int kk) {
    const int q = min(i, m - 1);
    const double *p = A.c;
    sign = j == i ? 1 : 0;
    if (kk > 0 && j == i - 1) p = A.b, sign = -1;
    if (jj > 0 && j == i - A.nz) p = A.s, sign = -1;
    if (i >= A.ny * A.nz && j == i - A.ny * A.nz) p = A.w, sign = -1;
    if (i >= m) sign = 0;
    v = p[q];
    ai = aj = 1;
    if (A.act) {
      ai = A.act[q];
      aj = A.act[min(j, m - 1)];
    }
  }
  __device__ __forceinline__ double value() const {
    return !ai || !aj || sign == 0 ? 0.0 : sign > 0 ? v : -v;
  }
  // a diagonal entry: a pivot up to this is taken for 0
  __device__ __forceinline__ double least() const {
    return ai && sign ? 1e-10 * fabs(v) : 1.0e300;
  }
};

// Threads [0, bw] divide the column and store it, the last 256 bring in the row
// that enters the window (loads only, a step ahead: a wave that also stores
// would wait for its stores), all of them subtract the products, U each (their
// places in the window relative to the step stay).
template <int U>
static __global__ __launch_bounds__(kBandThreads) void k_band_chol(BandArgs A) {
  extern __shared__ __align__(16) char band_lds[];
  double *const W = reinterpret_cast<double *>(band_lds);
  __shared__ double col[kBandMax + 1], least[kBandMax + 1];
  const int m = A.nx * A.ny * A.nz, bw = A.bw, n = bw + 1, t = (int)threadIdx.x;
  const int te = t - (kBandThreads - 256);
  for (int i = t >> 5; i < n; i += 32)
    for (int j = t & 31; j <= i; j += 32) {
      BandEntry e;
      e.load(A, m, i, j, i / A.nz % A.ny, i % A.nz);
      W[i * (i + 1) / 2 + j] = e.value();
      if (i == j) least[i] = e.least();
    }
  int di[U], dj[U];  // this thread's products; past the last: none (dj 0)
#pragma unroll
  for (int u = 0; u < U; u++) {
    int row = 0, at = t + u * kBandThreads;  // pair `at` of (1, 1), (2, 1), (2, 2), ...
    if (at < bw * n / 2) {
      row = (int)((sqrtf(8.0f * (float)at + 1.0f) - 1.0f) * 0.5f);
      while (row * (row + 1) / 2 > at) row--;
      while ((row + 1) * (row + 2) / 2 <= at) row++;
      di[u] = row + 1;
      dj[u] = at - row * (row + 1) / 2 + 1;
    } else {
      di[u] = dj[u] = 0;
    }
  }
  // the entering row's place along y and z
  int jj = n / A.nz % A.ny, kk = n % A.nz;
  BandEntry in;
  in.load(A, m, n, 1 + min(max(te, 0), bw), jj, kk);
  __syncthreads();
  int sk = 0;  // slot of k
  for (int k = 0; k < m; k++) {
    if (t <= bw) {
      const double piv = W[band_at(sk, sk)];
      const int st = sk + t < n ? sk + t : sk + t - n;
      const double x = W[band_at(st, sk)];
      const bool pinned = piv <= least[sk];
      const double d = pinned ? 0.0 : sqrt(piv);
      double v = 0.0;
      if (!pinned && k + t < m) v = t == 0 ? d : x / d;
      col[t] = v;
      A.Lc[(size_t)k * n + t] = v;
      if (k + t < m) A.Lr[(size_t)(k + t) * n + t] = v;
      if (pinned) {  // its row drops out too (this thread wrote these entries)
        A.Lr[(size_t)k * n + t] = 0.0;
        if (k >= t) A.Lc[(size_t)(k - t) * n + t] = 0.0;
      }
    }
    __syncthreads();
    int at[U];
    double w[U], li[U], lj[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int si = sk + di[u] < n ? sk + di[u] : sk + di[u] - n;
      const int sj = sk + dj[u] < n ? sk + dj[u] : sk + dj[u] - n;
      at[u] = band_at(si, sj);
      w[u] = W[at[u]];
      li[u] = col[di[u]];
      lj[u] = col[dj[u]];
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (dj[u]) W[at[u]] = w[u] - li[u] * lj[u];
    // row k + bw + 1 takes the place of row k
    if (te >= 0 && te <= bw) {
      W[band_at(sk, sk + 1 + te < n ? sk + 1 + te : sk + 1 + te - n)] = in.value();
      if (te == bw) least[sk] = in.least();
      kk = kk + 1 < A.nz ? kk + 1 : 0;
      if (kk == 0) jj = jj + 1 < A.ny ? jj + 1 : 0;
      in.load(A, m, k + 1 + n, k + 2 + te, jj, kk);
    }
    __syncthreads();
    sk = sk + 1 < n ? sk + 1 : 0;
  }
}

// column blockIdx.x of the inverse to Bt (as a row), its sum to cm.  A lane
// holds the Q entries of L's column (row) it applies, the next ones under way;
// a diagonal entry of 0 marks a pinned cell.
template <int Q>
static __global__ __launch_bounds__(64) void k_band_inverse(BandArgs A, double *Bt, double *cm) {
  extern __shared__ __align__(16) char band_lds[];
  double *const y = reinterpret_cast<double *>(band_lds);
  const int m = A.nx * A.ny * A.nz, bw = A.bw, n = bw + 1;
  const int t = (int)threadIdx.x, col = (int)blockIdx.x;
  const bool live = A.Lc[(size_t)col * n] != 0.0;
  for (int i = t; i < m; i += 64) y[i] = live && i == col ? 1.0 : 0.0;
  __syncthreads();
  // forward from the column's own row, then back, in steps of dir
  auto solve = [&](const double *L, int i0, int dir, int steps) {
    double a[Q], nx[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) nx[q] = L[(size_t)i0 * n + min(t + 64 * q, bw)];
    for (int s = 0, i = i0; s < steps; s++, i += dir) {
      const int in = s + 1 < steps ? i + dir : i, room = dir > 0 ? m - 1 - i : i;
#pragma unroll
      for (int q = 0; q < Q; q++) {
        a[q] = nx[q];
        nx[q] = L[(size_t)in * n + min(t + 64 * q, bw)];
      }
      const double d = __shfl(a[0], 0);
      const double v = d != 0.0 ? y[i] / d : 0.0;
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const int e = t + 64 * q;
        if (e > bw || e > room) continue;
        const int at = i + dir * e;
        y[at] = e == 0 ? v : y[at] - a[q] * v;
      }
      __syncthreads();
    }
  };
  if (live) {
    solve(A.Lc, col, 1, m - col);
    solve(A.Lr, m - 1, -1, m);
  }
  for (int i = t; i < m; i += 64) Bt[(size_t)col * m + i] = y[i];
  if (t == 0) {
    double sum = 0.0;
#pragma unroll 8
    for (int i = 0; i < m; i++) sum += y[i];
    cm[col] = sum;
  }
}

// sums of the inverse's rows
static __global__ __launch_bounds__(64) void k_band_rows(int m, const double *Bt, double *rm) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= m) return;
  double sum = 0.0;
#pragma unroll 8
  for (int j = 0; j < m; j++) sum += Bt[(size_t)j * m + i];
  rm[i] = sum;
}

// B row by row (G) from its columns
static __global__ __launch_bounds__(kBlock) void k_band_turn(int m, const double *Bt, double *G) {
  __shared__ double tile[16][17];
  const int nt = (m + 15) / 16, ti = (int)blockIdx.x / nt * 16, tj = (int)blockIdx.x % nt * 16;
  const int x = threadIdx.x & 15, z = threadIdx.x >> 4;
  if (tj + z < m && ti + x < m) tile[z][x] = Bt[(size_t)(tj + z) * m + ti + x];
  __syncthreads();
  if (ti + z < m && tj + x < m) G[(size_t)(ti + z) * m + tj + x] = tile[x][z];
}

// The sum of B's entries one after another, as a loop over them gives it, by
// one workgroup.  While the running sum s stays between two powers of two it is
// a multiple of one unit u, and adding b rounds b to a multiple of u, whatever
// s is (a tie apart, which goes to the even neighbour of the sum): the
// additions are then whole numbers and can be taken in any order.  A pass takes
// 8192 entries up to the first one that is a tie or leaves the interval, adds
// that one to the sum in floating point, and the next pass goes on behind it.
// While there is no such interval yet (the sum is 0 through the rows of solid
// cells before the first active one) a pass skips zeros, which leave the sum as
// it is, and adds up to 64 entries one by one: 48^3 with its first half solid,
// a new matrix in 7.1 ms where 64 zeros at a time took 29.5.
// Measured: 0.27 ms for the 2^18 entries of 8^3 cells, 1.7 ms for the 3.0 M of
// 12^3 (one after another: 4 ns each).
constexpr int kTotalPer = 8;
static __global__ __launch_bounds__(1024) void k_band_total(long long n, const double *B,
                                                            double *total) {
  __shared__ double s_sum, head[64];
  __shared__ long long s_pos, wsum[16];
  __shared__ int s_bad;
  const int t = (int)threadIdx.x, lane = t & 63, wid = t >> 6;
  if (t == 0) {
    s_sum = 0.0;
    s_pos = 0;
  }
  __syncthreads();
  constexpr double kLo = 4503599627370496.0, kHi = 9007199254740992.0;  // 2^52, 2^53
  for (;;) {
    const long long pos = s_pos;
    const double s = s_sum;
    if (pos >= n) break;
    if (t == 0) s_bad = 1024 * kTotalPer;
    double b[kTotalPer];
#pragma unroll
    for (int q = 0; q < kTotalPer; q++) {
      const long long at = pos + t * kTotalPer + q;
      b[q] = at < n ? B[at] : 0.0;
    }
    // the first entries, and a sum that is not a normal positive number: singly
    if (pos < 64 || !(s >= 1e-290 && s <= 1e290)) {
      int first = 1024 * kTotalPer;
#pragma unroll
      for (int q = kTotalPer - 1; q >= 0; q--) first = b[q] != 0.0 ? t * kTotalPer + q : first;
      __syncthreads();
      if (first < 1024 * kTotalPer) atomicMin(&s_bad, first);
      __syncthreads();
      const long long from = pos + s_bad;
      const int some = s_bad < 1024 * kTotalPer ? (int)min((long long)64, n - from) : 0;
      if (t < some) head[t] = B[from + t];
      __syncthreads();
      if (t == 0) {
        double v = s;
        for (int q = 0; q < some; q++) v += head[q];
        s_sum = v;
        s_pos = from + some;
      }
      __syncthreads();
      continue;
    }
    const int e = (int)(__double_as_longlong(s) >> 52) - 1023;  // s in [2^e, 2^(e + 1))
    const double up = __longlong_as_double((long long)(52 - e + 1023) << 52);
    const double u = __longlong_as_double((long long)(e - 52 + 1023) << 52);
    long long mine = 0;
    int bad = 1024 * kTotalPer;  // the first entry of this thread that cannot be a whole number
#pragma unroll
    for (int q = kTotalPer - 1; q >= 0; q--) {
      const double x = b[q] * up, r = rint(x);
      const bool whole = fabs(x) < kLo && fabs(x - r) != 0.5;
      if (!whole) bad = t * kTotalPer + q;
      mine += whole ? (long long)r : 0;
    }
    // units before this thread's entries
    long long inc = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const long long o = __shfl_up(inc, d);
      if (lane >= d) inc += o;
    }
    if (lane == 63) wsum[wid] = inc;
    __syncthreads();
    long long before = (long long)(s * up) + inc - mine;
    for (int q = 0; q < wid; q++) before += wsum[q];
    long long run = before;
#pragma unroll
    for (int q = 0; q < kTotalPer; q++) {
      const int at = t * kTotalPer + q;
      if (at >= bad) continue;
      run += (long long)rint(b[q] * up);
      if (!((double)run > kLo && (double)run < kHi)) bad = at;
    }
    if (bad < 1024 * kTotalPer) atomicMin(&s_bad, bad);
    __syncthreads();
    const int first = s_bad;
    if (first == 1024 * kTotalPer) {
      if (t == 1023) {
        s_sum = (double)run * u;
        s_pos = pos + 1024 * kTotalPer;
      }
    } else if (first / kTotalPer == t) {
      long long at = before;
      double add = 0.0;
#pragma unroll
      for (int q = 0; q < kTotalPer; q++) {
        if (q < first % kTotalPer) at += (long long)rint(b[q] * up);
        if (q == first % kTotalPer) add = b[q];
      }
      s_sum = (double)at * u + add;
      s_pos = pos + first + 1;
    }
    __syncthreads();
  }
  if (t == 0) *total = s_sum;
}

// G = B with the means of its rows and columns taken off, 0 off the active cells
static __global__ __launch_bounds__(kBlock) void k_band_project(int m, const uint8_t *act,
                                                                const double *rm,
                                                                const double *cm,
                                                                const double *total, double *G) {
  __shared__ double sm[kWaves][1];
  double na[1] = {0.0};
  for (int i = threadIdx.x; i < m; i += kBlock) na[0] += !act || act[i] ? 1.0 : 0.0;
  block_sum<1>(na, sm);
  const int i = (int)blockIdx.x;
  const double r = rm[i] / na[0], mean = *total / (na[0] * na[0]);
  const bool on = !act || act[i];
  for (int j = threadIdx.x; j < m; j += kBlock) {
    double &v = G[(size_t)i * m + j];
    v = on && (!act || act[j]) ? v - r - cm[j] / na[0] + mean : 0.0;
  }
}

}  // namespace psb
