// svd.hip -- sector SVD with global truncation (qtensor_op.cpp:1097-1453).
//
// Per mid-QN sector q (flux of the left indices, ascending QN order) the
// reference assembles a dense matrix from the blocks (rows: left position
// tuples in lexicographic order, columns: right tuples), takes its SVD,
// absorbs S into V (MoveFromLeft) or U (MoveFromRight), sorts all singular
// values globally (descending), keeps them while 1 - cumsum(s^2/sum s^2)
// >= cutoff (stopping at exact zeros, capping at K) and slices U, S, V.
//
// Device form (all FP64):
//   1. bookkeeping kernels: per-block sector keys, sorted unique row / column
//      tuple lists, sector sizes and row / column offsets;
//   2. gather of the blocks into packed sector matrices;
//   3. Gram matrix per sector on the grouped MFMA GEMM: A*A^T for
//      MoveFromLeft (the left factor U is what must be orthonormal),
//      A^T*A for MoveFromRight;
//   4. Jacobi eigensolver per sector: one workgroup for up to 64 rows, block
//      Jacobi over workgroups above;  s = sqrt(max(lambda, 0));
//   5. truncation on the device: per-sector rank-K cap, sum of s^2 and the
//      sequential cumsum rule in one thread, in the reference's order;
//   6. the absorbed factor as a second grouped GEMM (U^T A or A V), then the
//      slicing of U, V and S into blocks.
#include <algorithm>
#include <type_traits>
#include <cmath>
#include <cstring>
#include <numeric>

#include "ttg_device.h"
#include "ttg_internal.h"
#include "ttg_jacobi.h"
#include "ttg_plan.h"

namespace ttg {

__device__ inline uint32_t qcode_s(int q0, int q1) {
  return ((uint32_t)(q0 + 32768) << 16) | (uint32_t)(q1 + 32768);
}

// 1a. keys: (q << 32 | left tuple), (q << 32 | right tuple)
__global__ void k_svd_keys(MetaView A, int nleft, uint64_t* kl, uint64_t* kr, int* ids) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= A.nblocks) return;
  const int* qi = A.qi + (size_t)b * A.rank;
  int q0 = 0, q1 = 0;
  uint64_t l = 0, r = 0;
  for (int j = 0; j < A.rank; j++) {
    if (j < nleft) {
      const int* e = A.idx + 3 * (A.idx_off[j] + qi[j]);
      int sg = A.arrow[j] == 0 ? 1 : -1;   // qtensor_op.cpp:1129-1133
      q0 += sg * e[0];
      q1 += sg * e[1];
      l = l * A.nsec[j] + qi[j];
    } else {
      r = r * A.nsec[j] + qi[j];
    }
  }
  uint64_t qc = (uint64_t)qcode_s(q0, q1) << 32;
  kl[b] = qc | l;
  kr[b] = qc | r;
  ids[b] = b;
}

// size (product of sector dims) of a tuple over indices [j0, j1)
__device__ inline int64_t tuple_size(const MetaView& A, int j0, int j1, uint64_t key) {
  int64_t s = 1;
  for (int j = j1 - 1; j >= j0; j--) {
    int p = (int)(key % A.nsec[j]);
    key /= A.nsec[j];
    s *= A.idx[3 * (A.idx_off[j] + p) + 2];
  }
  return s;
}

struct SvdTab {
  uint64_t *uL, *uR;          // unique sorted keys
  int64_t *lsz, *loff;        // per uL entry: size, row offset inside its sector
  int64_t *rsz, *roff;        // per uR entry
  int *qL0, *qL1, *qR0, *qR1; // per sector ranges
  int64_t *rows, *cols;       // per sector
  uint32_t* qc;               // per sector QN code
  int64_t* hdr;               // [nuL, nuR, nQ]
};

// 1b. unique lists, sector table, offsets (one workgroup)
__global__ void __launch_bounds__(1024) k_svd_unique(MetaView A, int nleft, const uint64_t* sl,
                                                     const uint64_t* sr, int n, SvdTab t) {
  __shared__ int64_t lds[32];
  int64_t carry = 0;
  for (int base = 0; base < n; base += 1024) {   // unique left
    int i = base + threadIdx.x;
    int f = i < n && (i == 0 || sl[i] != sl[i - 1]);
    int64_t tot;
    int64_t pos = block_excl_scan<1024>((int64_t)f, lds, &tot);
    if (f) t.uL[carry + pos] = sl[i];
    carry += tot;
  }
  __syncthreads();
  const int nuL = (int)carry;
  carry = 0;
  for (int base = 0; base < n; base += 1024) {   // unique right
    int i = base + threadIdx.x;
    int f = i < n && (i == 0 || sr[i] != sr[i - 1]);
    int64_t tot;
    int64_t pos = block_excl_scan<1024>((int64_t)f, lds, &tot);
    if (f) t.uR[carry + pos] = sr[i];
    carry += tot;
  }
  __syncthreads();
  const int nuR = (int)carry;
  carry = 0;
  for (int base = 0; base < nuL; base += 1024) {  // sectors from uL
    int i = base + threadIdx.x;
    int f = i < nuL && (i == 0 || (t.uL[i] >> 32) != (t.uL[i - 1] >> 32));
    int64_t tot;
    int64_t pos = block_excl_scan<1024>((int64_t)f, lds, &tot);
    if (f) t.qL0[carry + pos] = i;
    carry += tot;
  }
  __syncthreads();
  const int nQ = (int)carry;
  for (int q = threadIdx.x; q < nQ; q += 1024) {
    int l0 = t.qL0[q], l1 = q + 1 < nQ ? t.qL0[q + 1] : nuL;
    t.qL1[q] = l1;
    uint64_t qc = t.uL[l0] >> 32;
    t.qc[q] = (uint32_t)qc;
    t.qR0[q] = lower_bound_u64(t.uR, nuR, qc << 32);
    t.qR1[q] = lower_bound_u64(t.uR, nuR, (qc + 1) << 32);
  }
  __syncthreads();
  // per-entry sizes and offsets inside the sector (sequential per sector)
  for (int q = threadIdx.x; q < nQ; q += 1024) {
    int64_t o = 0;
    for (int i = t.qL0[q]; i < t.qL1[q]; i++) {
      int64_t s = tuple_size(A, 0, nleft, t.uL[i] & 0xffffffffull);
      t.lsz[i] = s;
      t.loff[i] = o;
      o += s;
    }
    t.rows[q] = o;
    o = 0;
    for (int i = t.qR0[q]; i < t.qR1[q]; i++) {
      int64_t s = tuple_size(A, nleft, A.rank, t.uR[i] & 0xffffffffull);
      t.rsz[i] = s;
      t.roff[i] = o;
      o += s;
    }
    t.cols[q] = o;
  }
  if (threadIdx.x == 0) {
    t.hdr[0] = nuL;
    t.hdr[1] = nuR;
    t.hdr[2] = nQ;
  }
}

// 2. gather blocks into sector matrices (column-major rows_q x cols_q)
__global__ void k_svd_gather(MetaView A, int nleft, const double* __restrict__ a, SvdTab t,
                             int nuL, int nuR, int nQ, const int64_t* moff,
                             double* __restrict__ mat) {
  for (int b = blockIdx.x; b < A.nblocks; b += gridDim.x) {
    const int* qi = A.qi + (size_t)b * A.rank;
    int q0 = 0, q1 = 0;
    uint64_t l = 0, r = 0;
    for (int j = 0; j < A.rank; j++) {
      if (j < nleft) {
        const int* e = A.idx + 3 * (A.idx_off[j] + qi[j]);
        int sg = A.arrow[j] == 0 ? 1 : -1;
        q0 += sg * e[0];
        q1 += sg * e[1];
        l = l * A.nsec[j] + qi[j];
      } else {
        r = r * A.nsec[j] + qi[j];
      }
    }
    const uint64_t qc = (uint64_t)qcode_s(q0, q1) << 32;
    const int il = lower_bound_u64(t.uL, nuL, qc | l);
    const int ir = lower_bound_u64(t.uR, nuR, qc | r);
    // sector of il
    int lo = 0, hi = nQ;
    while (lo < hi) {
      int m = (lo + hi) >> 1;
      if (t.qL0[m] <= il) lo = m + 1;
      else hi = m;
    }
    const int q = lo - 1;
    const int64_t rows = t.rows[q];
    const int64_t ls = t.lsz[il], rs = t.rsz[ir];
    double* dst = mat + moff[q] + t.loff[il] + rows * t.roff[ir];
    const double* src = a + A.off[b];
    const int64_t n = ls * rs;
#pragma unroll 8
    for (int64_t e = threadIdx.x; e < n; e += blockDim.x) {
      const int64_t i = e % ls, j = e / ls;
      dst[i + rows * j] = src[e];
    }
  }
}

// 4. sectors of up to 64 rows: one workgroup per sector sweeps (ttg_jacobi.h)
// the matrix, padded with zeros to 16, 32 or 64 (the padding never rotates), in
// LDS until a sweep holds no significant rotation: |a_pq| above 1e-12 of
// sqrt(a_pp a_qq) (an off-diagonal d moves eigenvalues by ~d^2 / gap, so
// the eigenvalues are exact to ~1e-24 relative) and above 1e-14 of the
// largest diagonal, and then for up to kJacExtra sweeps without that floor, until
// one holds none by the relative test alone.  (The rounding noise in the null space of a
// rank-deficient sector's Gram matrix never passes the relative test alone.  A
// graded matrix, as a site's whose columns carry the singular values of its
// neighbour, has small singular values that are no noise.)
//
// Sectors of more than 16 rows go through a pivoted Cholesky factorisation
// P^T G P = R^T R first (as the large ones, 4c): the iteration then runs on
// G' = R R^T, r x r, which is nearly diagonal and holds no null space, and
// V = R^T W Lambda^(-1/2), corrected to first order for the remainder that the
// factorisation leaves out and made orthonormal to rounding by Gram-Schmidt steps
// (2e-15 where the rotations alone gave 2e-14).  The matrix stays in the registers of the
// 8 waves (8 rows each), every wave keeps the remaining diagonal and finds the pivot for
// itself, and one row a step passes through LDS.  On the sectors of an m = 100 state (up to 60
// rows, rank-deficient) k_jacobi took 445 us and takes 95, at m = 333 531 and 250.
// Why the correction: the remainder's diagonal is below kPcTol = 4.5 roundings of the
// largest, and left out it moved the vectors near a cutoff of 1e-9 more than the rounding
// of the Gram matrix does: the factors of states of m = 40 to 200 were off by 0.80e-12
// (of the state's norm, geometric mean over 160 states) where the plain iteration's are by
// 0.54e-12; with it they are by 0.29e-12, and k_jacobi takes 95 us at m = 100 instead of 89.
// The route is taken when the r columns are all that the selection can use, and all above
// kLrFix of the largest: r >= kq, the values kept before truncation, with no pivot among
// them below kLrCond of the largest diagonal, or a cutoff above kLrCutoff.  (A cutoff c
// keeps a value of weight w only if what follows weighs more than c in all, so the least
// kept value is above c / 10 unless more than ten values share the tail; what the
// factorisation leaves out weighs 64 kPcTol at most.)
constexpr double kJacFloor = 1e-14;   // convergence floor relative to the largest diagonal
constexpr double kPcTol = 1e-15;      // a remaining diagonal below this of the largest ends the factorisation
constexpr double kLrFix = 1e-12;      // least eigenvalue (of the largest) whose vector is corrected for the remainder
constexpr double kLrCutoff = 10 * kLrFix;
constexpr double kLrCond = 1e-8;
constexpr int kSvdMaxN = 8192;        // largest sector

// LDS of k_jacobi
struct JacLds {
  double s[kJS];                 // the matrix, later W^T
  double qts[2 * 4 * kJQt];
  double r[kJS];                 // rows of R
  double row[2][kJW];            // pivot row of a step, in turn; later the eigenvalues
  double dmax;
  int sig;
};

// Pivoted Cholesky of a matrix of up to 64 rows in the registers of 8 waves: x[s] is
// element (8 wave + s, lane), d the remaining diagonal of index `lane`, kept by every
// wave, `open` an index not yet taken.  Row k of R goes to r[k kJP + ..], the index of
// step k to lane k's `order`; ends after n steps or when stop(k, pivot) says so, and
// returns the steps; x is then what remains of the matrix at the open indices.  Ties go
// to the lower index.  `row`: two rows of LDS.
template <class Stop>
__device__ __forceinline__ int cholesky64(double (&x)[8], double d, bool& open, int n, double* r, double (*row)[kJW],
                                          int wave, int lane, int& order, Stop stop) {
  int k = 0;
  order = 0;
  for (; k < n; k++) {
    const double v = open ? d : -1.0;
    double m = v;
    m = fmax(m, lane_xor<1>(m));
    m = fmax(m, lane_xor<2>(m));
    m = fmax(m, lane_xor<4>(m));
    m = fmax(m, lane_xor<8>(m));
    m = fmax(m, lane_xor<16>(m));
    m = fmax(m, lane_xor<32>(m));
    if (stop(k, m)) break;   // the same in every wave
    const int p = __builtin_ctzll(__ballot(v == m));
    double* rk = row[k & 1];
    if (wave == p >> 3)
#pragma unroll
      for (int s = 0; s < 8; s++)
        if ((p & 7) == s) rk[lane] = x[s];
    const double inv = jac_rsqrt(m);
    __syncthreads();
    const double rv = open ? (lane == p ? m : rk[lane]) * inv : 0.0;
    open = open && lane != p;
    if (lane == k) order = p;
    if (wave == 0) r[k * kJP + lane] = rv;
    d = fma(-rv, rv, d);
    typedef int i2 __attribute__((ext_vector_type(2)));
    const i2 w = __builtin_bit_cast(i2, rv);
#pragma unroll
    for (int s = 0; s < 8; s++) {
      i2 u;
      u[0] = __builtin_amdgcn_readlane(w[0], 8 * wave + s);
      u[1] = __builtin_amdgcn_readlane(w[1], 8 * wave + s);
      x[s] = fma(-__builtin_bit_cast(double, u), rv, x[s]);
    }
  }
  __syncthreads();
  return k;
}

// Pivoted Cholesky of G0 (n x n): rows of R to L.r (zero beyond row r and column
// n); returns r, in `good` the rows with pivots above kLrCond of the largest
// diagonal, and in x rows 8 wave .. 8 wave + 7 of the remainder G0 - R^T R.  dg: the
// diagonal, scaled by 2^-ex as the matrix is on its way in.
__device__ __forceinline__ int jac_cholesky(JacLds& L, int n, const double* G0, double dg, int ex, int wave, int lane,
                                            int& good, double (&x)[8]) {
#pragma unroll
  for (int s = 0; s < 8; s++) {
    const int i = 8 * wave + s;
    x[s] = i < n && lane < n ? __builtin_amdgcn_ldexp(0.5 * (G0[i + (int64_t)n * lane] + G0[lane + (int64_t)n * i]), -ex)
                             : 0.0;
  }
  for (int e = threadIdx.x; e < kJS; e += kJThreads) L.r[e] = 0.0;
  __syncthreads();
  double tol = 0.0, fair = 0.0;
  int order, g = 0;
  bool open = lane < n;
  const int r = cholesky64(x, dg, open, n, L.r, L.row, wave, lane, order,
                           [&](int k, double m) {
                             if (k == 0) {
                               tol = kPcTol * m;
                               fair = kLrCond * m;
                             }
                             if (!(m > tol)) return true;
                             g += m > fair;   // (the pivots descend)
                             return false;
                           });
  good = g;
  const uint64_t left = __ballot(open);
#pragma unroll
  for (int s = 0; s < 8; s++) x[s] = open && (left >> (8 * wave + s) & 1) ? x[s] : 0.0;
  return r;
}

// G' = R R^T into L.s (16 NPR square)
template <int NPR>
__device__ __forceinline__ void jac_gram(JacLds& L, int n, int wave, int lane) {
  const int j = lane & 15, g = lane >> 4;
  for (int t = wave; t < NPR * (NPR + 1) / 2; t += 8) {
    int b = 0;
    while ((b + 1) * (b + 2) / 2 <= t) b++;
    const int a = t - b * (b + 1) / 2;   // a <= b
    jac_v4d r = {0.0, 0.0, 0.0, 0.0};
    for (int k = 0; k < n; k += 4)
      r = __builtin_amdgcn_mfma_f64_16x16x4f64(L.r[(16 * a + j) * kJP + k + g], L.r[(16 * b + j) * kJP + k + g], r, 0,
                                               0, 0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int i = 16 * a + g + 4 * s, c = 16 * b + j;
      L.s[i * kJP + c] = r[s];
      L.s[c * kJP + i] = r[s];
    }
  }
}

// Eigenpairs of the matrix G0 (n x n, r = 0) or of G' (r x r, from L.r) and from
// them those of G0, both scaled by 2^-ex.  rem: the remainder's rows (jac_cholesky).
template <int NPR>
__device__ __forceinline__ void jacobi_sector(JacLds& L, int n, int r, int ex, const double* G0, const double (&rem)[8],
                                              double* Vg, double* ev, int max_sweeps, double floor_rel, int wave,
                                              int lane) {
  constexpr int W = 16 * NPR;
  const int tid = threadIdx.x;
  double* S = L.s;
  if (r == 0) {
#pragma unroll 8
    for (int e = tid; e < W * W; e += kJThreads) {
      const int i = e % W, j = e / W;
      S[j * kJP + i] =
          (i < n && j < n) ? __builtin_amdgcn_ldexp(0.5 * (G0[i + (int64_t)n * j] + G0[j + (int64_t)n * i]), -ex) : 0.0;
    }
  } else {
    jac_gram<NPR>(L, n, wave, lane);
    floor_rel = 0.0;   // the relative test alone
  }
  double vt[2 * NPR][2];
  jac_identity<NPR>(vt, wave, lane);
  __syncthreads();
  if (wave == 0) {   // largest diagonal element: the scale of the convergence floor
    double m = lane < W ? fabs(S[lane * kJP + lane]) : 0.0;
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if (lane == 0) L.dmax = m;
  }
  int par = 0, extra = 0;
  double floor_abs = -1.0;
  for (int sweep = 0; sweep < max_sweeps; sweep++) {
    if (tid == 0) L.sig = 0;
    __syncthreads();
    if (sweep == 0) floor_abs = floor_rel * L.dmax;
    jac_sweep<NPR>(S, L.qts, vt, wave, lane, par, floor_abs, &L.sig);
    __syncthreads();
    // every thread reads the flag before thread 0 may clear it for the next
    // sweep: the barrier between the read and the reset keeps the decision
    // uniform over the workgroup
    const int rotated = L.sig;
    __syncthreads();
    if (extra ? !rotated || extra == kJacExtra : !rotated && floor_abs == 0.0) break;
    if (extra || !rotated) {   // the floor's own end: without it from here
      floor_abs = 0.0;
      extra++;
    }
  }
  if (r == 0) {
    for (int i = tid; i < n; i += kJThreads) ev[i] = __builtin_amdgcn_ldexp(S[i * kJP + i], ex);
    if (wave >= 4) {   // V(i, c) = V^T(c, i): consecutive lanes down a column of V
      const int i = 16 * (wave - 4) + (lane & 15);
#pragma unroll
      for (int b = 0; b < 2 * NPR; b++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int c = 8 * b + (lane >> 4) + 4 * h;
          if (i < n && c < n) Vg[i + (int64_t)n * c] = vt[b][h];
        }
    }
    return;
  }
  // V = R^T W Lambda^(-1/2); columns c >= r are zero, with eigenvalue zero
  double *lam = L.row[0], *out = L.row[1];
  if (tid < kJW) out[tid] = lam[tid] = tid < r ? S[tid * kJP + tid] : 0.0;
  __syncthreads();
  if (wave >= 4 && wave < 4 + NPR) {
#pragma unroll
    for (int b = 0; b < 2 * NPR; b++)
#pragma unroll
      for (int h = 0; h < 2; h++) S[(8 * b + (lane >> 4) + 4 * h) * kJP + 16 * (wave - 4) + (lane & 15)] = vt[b][h];
  }
  __syncthreads();
  // tiles (a, b) of V^T: rows c, columns i; X = V^T (r rows) afterwards in L.r
  const int j = lane & 15, g = lane >> 4, nt = (n + 15) / 16;
  constexpr int kMine = (NPR * 4 + 7) / 8;   // tiles a wave can have
  jac_v4d v[kMine];
#pragma unroll
  for (int u = 0; u < kMine; u++) {
    const int t = wave + 8 * u, a = t % NPR, b = t / NPR;
    v[u] = {0.0, 0.0, 0.0, 0.0};
    if (t < NPR * nt) {
#pragma unroll
      for (int k = 0; k < W; k += 4)
        v[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[(16 * a + j) * kJP + k + g], L.r[(k + g) * kJP + 16 * b + j], v[u],
                                                    0, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const double l = lam[16 * a + g + 4 * s];
        v[u][s] *= l > 0.0 ? 1.0 / sqrt(l) : 0.0;
      }
    }
  }
  auto put = [&]() {   // X = v
#pragma unroll
    for (int u = 0; u < kMine; u++) {
      const int t = wave + 8 * u, a = t % NPR, b = t / NPR;
      if (t < NPR * nt)
#pragma unroll
        for (int s = 0; s < 4; s++) L.r[(16 * a + g + 4 * s) * kJP + 16 * b + j] = v[u][s];
    }
  };
  __syncthreads();
  put();
  // The remainder E that the factorisation left out moves the vectors by E X / lambda
  // to first order, and the eigenvalues by x_c^T E x_c: half of what it adds to |x_c|^2,
  // times lambda_c.
  const double least = kLrFix * L.dmax;
  const bool fix = r < n;
  if (fix) {
#pragma unroll
    for (int s = 0; s < 8; s++) S[(8 * wave + s) * kJP + lane] = rem[s];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMine; u++) {
      const int t = wave + 8 * u, a = t % NPR, b = t / NPR;
      if (t >= NPR * nt) continue;
      jac_v4d y = {0.0, 0.0, 0.0, 0.0};
      for (int k = 0; k < n; k += 4)
        y = __builtin_amdgcn_mfma_f64_16x16x4f64(L.r[(16 * a + j) * kJP + k + g], S[(k + g) * kJP + 16 * b + j], y, 0, 0,
                                                 0);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const double l = lam[16 * a + g + 4 * s];
        v[u][s] += l > least ? y[s] / l : 0.0;
      }
    }
    __syncthreads();
    put();
  }
  __syncthreads();
  // X is orthonormal to the rounding of R^T W, eps sqrt(lambda_1 / lambda_c), and to E / lambda:
  // a Gram-Schmidt step in the order of the eigenvalues squares that,
  // X <- C X, C(c, a) = -(X X^T)(c, a) for lambda_a > lambda_c, (3 - |x_c|^2) / 2 at c
  for (int round = fix ? 3 : 1; round > 0; round--) {
    for (int t = wave; t < NPR * (NPR + 1) / 2; t += 8) {
      int b = 0;
      while ((b + 1) * (b + 2) / 2 <= t) b++;
      const int a = t - b * (b + 1) / 2;
      jac_v4d m = {0.0, 0.0, 0.0, 0.0};
      for (int k = 0; k < n; k += 4)
        m = __builtin_amdgcn_mfma_f64_16x16x4f64(L.r[(16 * a + j) * kJP + k + g], L.r[(16 * b + j) * kJP + k + g], m, 0,
                                                 0, 0);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int i = 16 * a + g + 4 * s, c = 16 * b + j;
        const double li = lam[i], lc = lam[c];
        const bool first = li > lc || (li == lc && i < c);   // x_i is corrected before x_c
        S[c * kJP + i] = i == c ? 1.5 - 0.5 * m[s] : first ? -m[s] : 0.0;
        if (i != c) S[i * kJP + c] = first ? 0.0 : -m[s];
        else if (round == 3 && lc > least) out[c] = lc * (0.5 + 0.5 * m[s]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMine; u++) {
      const int t = wave + 8 * u, a = t % NPR, b = t / NPR;
      v[u] = {0.0, 0.0, 0.0, 0.0};
      if (t >= NPR * nt) continue;
#pragma unroll
      for (int k = 0; k < W; k += 4)
        v[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[(16 * a + j) * kJP + k + g], L.r[(k + g) * kJP + 16 * b + j], v[u],
                                                    0, 0, 0);
    }
    if (round > 1) {
      __syncthreads();
      put();
      __syncthreads();
    }
  }
  if (tid < n) ev[tid] = __builtin_amdgcn_ldexp(out[tid], ex);
#pragma unroll
  for (int u = 0; u < kMine; u++) {
    const int t = wave + 8 * u, a = t % NPR, b = t / NPR;
    if (t < NPR * nt)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int c = 16 * a + g + 4 * s, i = 16 * b + j;
        if (i < n && c < n) Vg[i + (int64_t)n * c] = v[u][s];
      }
  }
  for (int e = tid; e < n * (n - W); e += kJThreads) Vg[(int64_t)n * W + e] = 0.0;
}

// kq: the eigenpairs a sector can use (null: every one, no factorisation);
// drop: fewer will do, the others are below the cutoff
__global__ void __launch_bounds__(kJThreads)
k_jacobi(const int* __restrict__ nq, const int* __restrict__ kq, int drop, const int64_t* __restrict__ goff,
         const double* __restrict__ Gin, double* __restrict__ Vout, double* __restrict__ evals,
         const int64_t* __restrict__ eoff, int max_sweeps, int nmax_here, double floor_rel) {
  __shared__ __attribute__((aligned(16))) JacLds L;
  const int q = blockIdx.x;
  const int n = nq[q];
  if (n == 0 || n > nmax_here) return;   // larger sectors: block Jacobi
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double* G0 = Gin + goff[q];      // full n x n column-major
  double* Vg = Vout + goff[q];           // eigenvectors, the same layout
  double* ev = evals + eoff[q];
  const double dg = lane < n ? G0[lane * (int64_t)(n + 1)] : 0.0;
  // (even: R's scale is a power of two as well)
  const int ex = __builtin_amdgcn_frexp_exp(wave_all(fabs(dg), [](double a, double b) { return fmax(a, b); })) & ~1;
  int r = 0;
  double rem[8] = {};
  if (kq && n > 16) {
    int good;
    r = jac_cholesky(L, n, G0, __builtin_amdgcn_ldexp(dg, -ex), ex, wave, lane, good, rem);
    if (!drop && good < kq[q]) r = 0;
  }
  const int w = r ? r : n;
  if (w <= 16) jacobi_sector<1>(L, n, r, ex, G0, rem, Vg, ev, max_sweeps, floor_rel, wave, lane);
  else if (w <= 32) jacobi_sector<2>(L, n, r, ex, G0, rem, Vg, ev, max_sweeps, floor_rel, wave, lane);
  else jacobi_sector<4>(L, n, r, ex, G0, rem, Vg, ev, max_sweeps, floor_rel, wave, lane);
}

// 4b. Sectors larger than kJacBlockMin: two-sided block Jacobi.  The padded
// Gram matrix (N = n rounded up to 64, zero padding never rotates) is cut into
// 32-wide blocks; a round pairs the blocks (circle method) and
//   k_bjac_solve  diagonalises every 64 x 64 subproblem G[I+J, I+J] in LDS
//                 (one inner cyclic sweep) into Q_IJ, its eigenpairs sorted
//                 in descending order, and
//   k_bjac_apply  updates G <- P^T G P (upper tiles, mirrored: G stays
//                 exactly symmetric) and V <- V P, P = diag(Q_IJ), as 64 x 64
//                 tile products on the FP64 matrix cores,
// so a round moves G and V through memory once instead of once per scalar
// rotation.  A sweep (nbk - 1 rounds) leaves a sector active while any
// subproblem held an off-diagonal element above 1e-12 sqrt(g_ii g_jj) and
// above the sector's floor, 1e-14 of the largest diagonal, and for up to kJacExtra
// sweeps more while some are above the relative test.  A subproblem with
// none leaves Q_IJ = I and marks its pair unrotated; the
// tile products of a round skip the tiles whose pairs were both unrotated.
constexpr int kJacBlockMin = kJW;
constexpr int kBJ = 32;                // block width; subproblems are 2 kBJ
constexpr int kSub = 2 * kBJ;

typedef double bj_v4d __attribute__((ext_vector_type(4)));

struct BJSector {
  int n, N, nbk, q;                    // size, padded size, blocks, sector id
  int64_t gp, qp;                      // offsets of padded G / V and of the pair Q's
  double floor;                        // off-diagonal size below which nothing rotates
  int pb;                              // index of the sector's first pair in the pair list
  int ex;                              // G is held scaled by 2^-ex (its largest diagonal below 1)
};

// circle method over m = 2 npair indices: pair k of round r (a < b)
__device__ inline void circle_pair(int m, int r, int k, int& a, int& b) {
  const int m1 = m - 1;
  if (k == 0) { a = r % m1; b = m1; }
  else { a = (r + k) % m1; b = (r - k + m1) % m1; }
  if (a > b) { const int t = a; a = b; b = t; }
}
// subproblem entry t (0..63) of pair k of round r is global index
// (t < kBJ ? a : b) * kBJ + t % kBJ, (a, b) = circle_pair(nbk, r, k)

// Gp: the padded matrix scaled by a power of two (ex), Vp: identity; and
// sec[li].floor = floor_rel max_i |G_ii|, scaled
__global__ void __launch_bounds__(256) k_bjac_init(BJSector* sec, int nsec, const int64_t* goff, const double* G,
                                                   double* Gp, double* Vp, double floor_rel) {
  __shared__ double red[4];
  const int li = blockIdx.y;
  if (li >= nsec) return;
  const int n = sec[li].n, N = sec[li].N;
  const int64_t gp = sec[li].gp;
  const double* g = G + goff[sec[li].q];
  double mx = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) mx = fmax(mx, fabs(g[i + (int64_t)n * i]));
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  const int ex = __builtin_amdgcn_frexp_exp(mx);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sec[li].floor = floor_rel * __builtin_amdgcn_ldexp(mx, -ex);
    sec[li].ex = ex;
  }
  const int64_t NN = (int64_t)N * N;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < NN;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int i = (int)(e % N), j = (int)(e / N);
    Gp[gp + e] = (i < n && j < n) ? __builtin_amdgcn_ldexp(0.5 * (g[i + (int64_t)n * j] + g[j + (int64_t)n * i]), -ex)
                                  : 0.0;
    Vp[gp + e] = i == j ? 1.0 : 0.0;
  }
}

// one workgroup per (sector, pair): the 64 x 64 subproblem, one cyclic sweep
// (ttg_jacobi.h)
static_assert(kSub == kJW, "a subproblem is one Jacobi matrix");
__global__ void __launch_bounds__(kJThreads)
k_bjac_solve(const BJSector* sec, const int2* items, int nitems, int r, const int* active, int* flag,
             int* rotated, const double* Gp, double* Qp) {
  __shared__ __attribute__((aligned(16))) double lds[kJLds];
  __shared__ int perm[kSub], cnt[kSub];
  __shared__ int sig, sweep_sig;   // (the sweep's own flag: sig is the test's before it)
  const int2 it = items[blockIdx.x];
  const int li = it.x, k = it.y;
  const BJSector S = sec[li];
  if (!active[li] || r >= S.nbk - 1) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double* M = lds;
  double* Qts = lds + kJS;
  // the pair's two blocks (uniform): subproblem entry t is global index
  // (t < 32 ? ba : bb) * 32 + t % 32; the sector's own indices (global index
  // < n) are entries [0, na) and [32, 32 + nbb)
  int ba, bb;
  circle_pair(S.nbk, r, k, ba, bb);
  const int na = min(max(S.n - kBJ * ba, 0), kBJ), nbb = min(max(S.n - kBJ * bb, 0), kBJ);
  auto gidx = [&](int t) { return (t >= kBJ ? bb : ba) * kBJ + (t & (kBJ - 1)); };
  auto own = [&](int t) { return t < kBJ ? t < na : t - kBJ < nbb; };
  if (tid == 0) sig = 0;
  if (tid < kSub) cnt[tid] = 0;
  {
    // all of a thread's loads are issued before the first LDS store (a loop
    // with one load per iteration would wait one memory latency per entry)
    constexpr int kPer = kSub * kSub / kJThreads;
    double gv[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
      const int e = tid + kJThreads * u, i = e % kSub, j = e / kSub;   // G is exactly symmetric
      gv[u] = Gp[S.gp + gidx(i) + (int64_t)S.N * gidx(j)];
    }
#pragma unroll
    for (int u = 0; u < kPer; u++) {
      const int e = tid + kJThreads * u, i = e % kSub, j = e / kSub;
      M[j * kJP + i] = gv[u];
    }
  }
  __syncthreads();
  {
    // significance test of this subproblem (before rotating), bit 0: |v| > 1e-12
    // sqrt(g_pp g_qq), compared squared, bit 1: above the floor as well; thread t's
    // columns p are all t % 64 (so one diagonal load), its rows q = t / 64 + 8 i
    const int p = tid % kSub;
    const double gpp = M[p * kJP + p];
    bool any = false, big = false;
    for (int q = tid / kSub; q < kSub; q += kJThreads / kSub) {
      if (p == q) continue;
      const double v = M[q * kJP + p];
      const bool here = v * v > (kJacRel * kJacRel) * fabs(gpp * M[q * kJP + q]);
      any |= here;
      big |= here & (fabs(v) > S.floor);
    }
    if (any) atomicOr(&sig, big ? 3 : 1);
  }
  __syncthreads();
  double* Qg = Qp + S.qp + (int64_t)k * kSub * kSub;   // column-major 64 x 64
  if (!sig) {   // already diagonal: Q = I
    for (int e = tid; e < kSub * kSub; e += kJThreads) Qg[e] = (e % kSub == e / kSub) ? 1.0 : 0.0;
    if (tid == 0) rotated[blockIdx.x] = 0;
    return;
  }
  if (tid == 0) {
    atomicOr(&flag[li], sig);
    rotated[blockIdx.x] = 1;
  }
  double vt[8][2];
  jac_identity<4>(vt, wave, lane);
  int par = 0;
  jac_sweep<4>(M, Qts, vt, wave, lane, par, S.floor, &sweep_sig);
  // Eigenpairs in descending order (the larger values to the pair's lower
  // block): a fixed order keeps values from swapping between blocks from
  // round to round, which otherwise holds the outer iteration at a linear rate.
  // Only the sector's own indices are ordered, over their own positions; a
  // padding index (global index >= n, never rotated) keeps its column, so no
  // eigenvector moves into the padding that k_bjac_finish drops.
  {
    // rank of own entry x among the own entries (descending eigenvalue,
    // ties to the lower entry), counted by the eight waves over an eighth of
    // the entries each
    const int x = tid % kSub, part = tid / kSub;
    if (own(x)) {
      const double d = M[x * kJP + x];
      int c = 0;
#pragma unroll
      for (int u = 8 * part; u < 8 * part + 8; u++) {
        const double du = M[u * kJP + u];
        c += own(u) && ((du > d) || (du == d && u < x));
      }
      if (c) atomicAdd(&cnt[x], c);
    }
  }
  __syncthreads();
  if (tid < kSub) {
    // the rank-th own entry in ascending order: own entries are [0, na) then
    // [32, 32 + nbb)
    const int x = tid;
    int dst = x;
    if (own(x)) {
      const int rk = cnt[x];
      dst = rk < na ? rk : kBJ + (rk - na);
    }
    perm[x] = dst;   // column of Q for the eigenvector of entry x
  }
  __syncthreads();
  if (wave >= 4) {   // Q(i, perm(c)) = V^T(c, i)
    const int i = 16 * (wave - 4) + (lane & 15);
#pragma unroll
    for (int b = 0; b < 8; b++)
#pragma unroll
      for (int h = 0; h < 2; h++) Qg[i + kSub * perm[8 * b + (lane >> 4) + 4 * h]] = vt[b][h];
  }
}

// tile products of a round on v_mfma_f64_16x16x4 (lane l holds A[l%16][l/16],
// B[l/16][l%16]; result register r holds D[l/16 + 4r][l%16]).  Wave w
// computes rows 16w..16w+15 of the 64 x 64 result; the operand all waves
// share is staged in LDS, the per-wave operand is read from memory.
//   kind 0 (a <= b): X = Qa^T T, R = X Qb for T = G[Ia, Ib]; R written to
//                    G[Ia, Ib] and mirrored into G[Ib, Ia];
//   kind 1: R^T = Qb^T T^T for T = V[rows 64a..64a+63, Ib]: V <- V Qb, the
//           transposed product so that lanes store down V's columns.
constexpr int kTLd = kSub + 1;
__global__ void __launch_bounds__(256) k_bjac_apply(const BJSector* sec, const int4* items, int nitems,
                                                    int r, const int* active, const int* rotated,
                                                    double* Gp, double* Vp, const double* Qp) {
  __shared__ double Bs[kSub * kTLd];
  __shared__ double Xs[kSub * kTLd];
  const int4 it = items[blockIdx.x];
  const int li = it.x;
  const BJSector S = sec[li];
  if (!active[li] || r >= S.nbk - 1) return;
  const int kind = it.w, a = it.y, b = it.z;
  const bool rb = rotated[S.pb + b] != 0;
  const bool ra = kind == 0 && rotated[S.pb + a] != 0;
  if (!ra && !rb) return;   // both factors are the identity
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int l16 = lane & 15, l4 = lane >> 4;
  // global indices of the entries of pairs a and b (their blocks computed once)
  int a0, a1, b0, b1;
  circle_pair(S.nbk, r, a, a0, a1);
  circle_pair(S.nbk, r, b, b0, b1);
  auto ga = [&](int t) { return (t >= kBJ ? a1 : a0) * kBJ + (t & (kBJ - 1)); };
  auto gb = [&](int t) { return (t >= kBJ ? b1 : b0) * kBJ + (t & (kBJ - 1)); };
  const double* qa = Qp + S.qp + (int64_t)a * kSub * kSub;
  const double* qb = Qp + S.qp + (int64_t)b * kSub * kSub;
  double af[16];
  bj_v4d acc[4];
  if (kind == 1) {
    double* V = Vp + S.gp;
#pragma unroll
    for (int s = 0; s < 16; s++) af[s] = qb[(4 * s + l4) + kSub * (16 * w + l16)];   // Qb^T
    double tv[16];   // Bs[k][ii] = V(64a + ii, gj(k)): all loads issued, then the LDS stores
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int e = tid + 256 * u, ii = e % kSub, kk = e / kSub;
      tv[u] = V[(int64_t)(a * kSub + ii) + (int64_t)S.N * gb(kk)];
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int e = tid + 256 * u, ii = e % kSub, kk = e / kSub;
      Bs[kk * kTLd + ii] = tv[u];
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < 4; f++) acc[f] = bj_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 16; s++)
#pragma unroll
      for (int f = 0; f < 4; f++)
        acc[f] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[s], Bs[(4 * s + l4) * kTLd + 16 * f + l16], acc[f],
                                                      0, 0, 0);
#pragma unroll
    for (int rr = 0; rr < 4; rr++) {
      const int64_t col = (int64_t)S.N * gb(16 * w + l4 + 4 * rr);
#pragma unroll
      for (int f = 0; f < 4; f++) V[col + a * kSub + 16 * f + l16] = acc[f][rr];
    }
    return;
  }
  double* G = Gp + S.gp;
#pragma unroll
  for (int s = 0; s < 16; s++) af[s] = qa[(4 * s + l4) + kSub * (16 * w + l16)];   // Qa^T
  {
    double tv[16], xv[16];   // all loads issued, then the LDS stores
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int e = tid + 256 * u, kk = e % kSub, j = e / kSub;
      tv[u] = G[ga(kk) + (int64_t)S.N * gb(j)];
      xv[u] = qb[kk + kSub * j];
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int e = tid + 256 * u, kk = e % kSub, j = e / kSub;
      Bs[kk * kTLd + j] = tv[u];
      Xs[kk * kTLd + j] = xv[u];
    }
  }
  __syncthreads();
#pragma unroll
  for (int f = 0; f < 4; f++) acc[f] = bj_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < 16; s++)
#pragma unroll
    for (int f = 0; f < 4; f++)
      acc[f] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[s], Bs[(4 * s + l4) * kTLd + 16 * f + l16], acc[f],
                                                    0, 0, 0);
  __syncthreads();   // every wave is done reading T
#pragma unroll
  for (int f = 0; f < 4; f++)
#pragma unroll
    for (int rr = 0; rr < 4; rr++) Bs[(16 * w + l4 + 4 * rr) * kTLd + 16 * f + l16] = acc[f][rr];
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 16; s++) af[s] = Bs[(16 * w + l16) * kTLd + 4 * s + l4];   // X rows of wave w
#pragma unroll
  for (int f = 0; f < 4; f++) acc[f] = bj_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < 16; s++)
#pragma unroll
    for (int f = 0; f < 4; f++)
      acc[f] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[s], Xs[(4 * s + l4) * kTLd + 16 * f + l16], acc[f],
                                                    0, 0, 0);
#pragma unroll
  for (int rr = 0; rr < 4; rr++) {
    const int gi = ga(16 * w + l4 + 4 * rr);
#pragma unroll
    for (int f = 0; f < 4; f++) {
      const int gj = gb(16 * f + l16);
      G[gi + (int64_t)S.N * gj] = acc[f][rr];
      if (a != b) G[gj + (int64_t)S.N * gi] = acc[f][rr];   // G stays symmetric
    }
  }
}

// end of an outer sweep: a sector stays active (1) while its sweep rotated
// anything above the floor, then (2, 3, ..) for kJacExtra sweeps while it rotates
// anything; the flags start over for the next sweep; *any = some sector active
__global__ void __launch_bounds__(256) k_bjac_sweep_end(int nsec, int* flag, int* act, int* any) {
  __shared__ int s_any;
  if (threadIdx.x == 0) s_any = 0;
  __syncthreads();
  int a = 0;
  for (int li = threadIdx.x; li < nsec; li += blockDim.x) {
    const int f = flag[li], was = act[li];
    const int now = !f || was == 0 ? 0 : was == 1 ? (f & 2 ? 1 : 2) : was < 1 + kJacExtra ? was + 1 : 0;
    act[li] = now;
    flag[li] = 0;
    a |= now;
  }
  if (a) atomicOr(&s_any, 1);
  __syncthreads();
  if (threadIdx.x == 0) *any = s_any;
}

__global__ void k_bjac_finish(const BJSector* sec, int nsec, const int64_t* goff,
                              const int64_t* eoff, const double* Gp, const double* Vp,
                              double* Vout, double* evals) {
  const int li = blockIdx.y;
  if (li >= nsec) return;
  const BJSector S = sec[li];
  const int64_t nn = (int64_t)S.n * S.n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nn;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int i = (int)(e % S.n), j = (int)(e / S.n);
    Vout[goff[S.q] + e] = Vp[S.gp + i + (int64_t)S.N * j];
    if (i == j) evals[eoff[S.q] + i] = __builtin_amdgcn_ldexp(Gp[S.gp + i + (int64_t)S.N * i], S.ex);
  }
}

// host driver of the block Jacobi over the sectors `big` (sizes nq)
static int block_jacobi(const std::vector<int>& big, const std::vector<int>& nq, const int64_t* d_goff,
                        const int64_t* d_eoff, const double* G, double* Vev, double* ev,
                        hipStream_t s, int max_sweeps, double floor_rel) {
  PhaseTimer _phase("block_jacobi");
  const int ns = (int)big.size();
  std::vector<BJSector> sec(ns);
  std::vector<int2> pitems;
  std::vector<int4> titems;
  int64_t gp = 0, qp = 0;
  int maxr = 0;
  for (int li = 0; li < ns; li++) {
    const int q = big[li], n = nq[q];
    const int N = (n + kSub - 1) / kSub * kSub;
    const int nbk = N / kBJ, npair = nbk / 2;
    sec[li] = BJSector{n, N, nbk, q, gp, qp, 0.0, (int)pitems.size(), 0};
    gp += (int64_t)N * N;
    qp += (int64_t)npair * kSub * kSub;
    maxr = std::max(maxr, nbk - 1);
    for (int k = 0; k < npair; k++) pitems.push_back(int2{li, k});
    for (int a = 0; a < npair; a++)
      for (int b = a; b < npair; b++) titems.push_back(int4{li, a, b, 0});   // a <= b, mirrored
    for (int rc = 0; rc < N / kSub; rc++)
      for (int b = 0; b < npair; b++) titems.push_back(int4{li, rc, b, 1});
  }
  Scratch sc;
  BJSector* d_sec = sc.get<BJSector>(ns);
  int2* d_pit = sc.get<int2>(pitems.size());
  int4* d_tit = sc.get<int4>(titems.size());
  double* Gp = sc.get<double>(gp);
  double* Vp = sc.get<double>(gp);
  double* Qp = sc.get<double>(qp);
  int* act = sc.get<int>(ns);
  int* flag = sc.get<int>(ns);
  int* rot = sc.get<int>(pitems.size());
  int* anyd = sc.get<int>(1);
  TTG_TRY(sc.ok("svd: block Jacobi"));
  {
    UploadBatch up;
    TTG_TRY(h2d_vec(d_sec, sec));
    TTG_TRY(h2d_vec(d_pit, pitems));
    TTG_TRY(h2d_vec(d_tit, titems));
    TTG_TRY(h2d_vec(act, std::vector<int>(ns, 1)));
    TTG_TRY(h2d_vec(flag, std::vector<int>(ns, 0)));
    TTG_TRY(up.flush());
  }
  hipLaunchKernelGGL(k_bjac_init, dim3(64, ns), dim3(256), 0, s, d_sec, ns, d_goff, G, Gp, Vp, floor_rel);
  // Outer sweeps.  The active flags move on the device (k_bjac_sweep_end),
  // so the host reads the "any sector active" word only from the sweep at
  // which the previous call of the same kind (LR-reduced or plain Gram
  // matrices) converged, less two: a sweep after convergence finds every
  // sector inactive and its launches return at once.
  static int prev_sweeps[2] = {0, 0};
  int& prev = prev_sweeps[floor_rel > 0 ? 1 : 0];
  const int first_check = std::max(0, prev - 2);
  int sweep = 0;
  for (; sweep < max_sweeps; sweep++) {
    for (int r = 0; r < maxr; r++) {
      hipLaunchKernelGGL(k_bjac_solve, dim3((unsigned)pitems.size()), dim3(kJThreads), 0, s, d_sec, d_pit,
                         (int)pitems.size(), r, act, flag, rot, Gp, Qp);
      hipLaunchKernelGGL(k_bjac_apply, dim3((unsigned)titems.size()), dim3(256), 0, s, d_sec, d_tit,
                         (int)titems.size(), r, act, rot, Gp, Vp, Qp);
    }
    hipLaunchKernelGGL(k_bjac_sweep_end, dim3(1), dim3(256), 0, s, ns, flag, act, anyd);
    if (sweep < first_check && sweep + 1 < max_sweeps) continue;
    int any = 0;
    const D2HPiece pc{&any, anyd, sizeof(int)};
    TTG_TRY(d2h_wait(&pc, 1));
    if (!any) break;
  }
  prev = std::min(sweep, 16);
  hipLaunchKernelGGL(k_bjac_finish, dim3(64, ns), dim3(256), 0, s, d_sec, ns, d_goff, d_eoff, Gp, Vp,
                     Vev, ev);
  TTG_HIP(hipGetLastError());
  return 0;   // the scratch goes back to the pool in stream order
}

// 4c. LR preconditioning of the large sectors.  A sector's Gram matrix of
// a DMRG state is numerically rank-deficient (a few hundred of its rows
// carry weight), and that of a site to be canonicalised when it has more rows on
// the isometric side than on the other; the Jacobi iteration on G spends most of
// its sweeps decoupling that null space from the rest.  A pivoted Cholesky
// factorisation P^T G P = R^T R stops at the numerical rank r (largest
// remaining diagonal below 1e-15 of the largest diagonal) and gives
// G' = R R^T (r x r, the same nonzero eigenvalues, no null space).  Jacobi
// on G' with the relative convergence test alone (no absolute floor: G' is
// positive definite) converges in about a third of the sweeps, at size r,
// and G's eigenvectors follow as X = R^T W Lambda^(-1/2), orthonormal to the
// relative accuracy of W and to eps sqrt(lambda_1 / lambda_c); one Gram-Schmidt
// step in the order of the eigenvalues makes that 2e-15 (1e-12 before).  The
// n - r null-space columns are left zero with eigenvalue 0: a zero singular value
// is never kept when cutoff > 0 (qtensor_op.cpp:1294-1300).  Without a cutoff
// the rule is: the r columns cover the kq values asked for, and no pivot among them
// is below kLrCond of the largest diagonal, or kLrCondOpen when the factorisation
// leaves indices out (r < n: nothing corrects for the remainder here); otherwise the sector's
// Gram matrix is formed again and solved by block Jacobi.  The smallest singular values of
// 130 x 65 and 600 x 300 sectors were off by 6e-15 and 8e-14 of the largest (block Jacobi:
// 4e-14, 2e-13) with pivots from 2e-4, by 6e-14 and 3e-13 from 3e-6, and by 2e-12 from 1e-7.
// (A site of m = 701: 11 sweeps of 5 rounds on G, 7 of 3 on G', 2600 to 1870 us.)
// R is stored by original column index (row k of R at k n + j), so neither
// G' nor V needs the permutation.
//   k_pchol_init   d = diag(G), dmax per sector
//   k_pchol_panel  the next up to 64 pivots, from a 64 x 64 principal submatrix
//   k_pchol_update their rows of R, and G <- G - R_panel^T R_panel
constexpr int kPcThreads = 512;
constexpr int kPcNbMax = 64;   // candidates of a panel: a wave's lanes
struct PcSector {
  int n, q;
  int kq;         // eigenpairs the selection can use
  int pad;
  int64_t goff;   // G (trailing matrix, overwritten) and R, n x n each
  int64_t doff;   // remaining diagonal, pivots in order, step of each column (-1: none), n each
};
struct PcState {
  double dmax;    // largest diagonal of G
  double least;   // smallest of the first kq pivots
  int rank;       // -1: not finished
  int k0, k1;     // rows of R that the last panel wrote
  int panels, pad;
};

__global__ void __launch_bounds__(kPcThreads) k_pchol_init(const PcSector* ps, const double* G, double* d,
                                                           int* pos, PcState* st) {
  __shared__ double red[kPcThreads / 64];
  const PcSector P = ps[blockIdx.x];
  double mx = 0.0;
  for (int j = threadIdx.x; j < P.n; j += blockDim.x) {
    const double v = G[P.goff + j + (int64_t)P.n * j];
    d[P.doff + j] = v;
    pos[P.doff + j] = -1;
    mx = fmax(mx, v);
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) m = fmax(m, red[w]);
    st[blockIdx.x] = PcState{m, m, -1, 0, 0, 0, 0};
  }
}

// A panel takes its pivots from the (up to) 64 largest remaining diagonals at
// its start: k_pchol_panel, one workgroup a sector, factorises that 64 x 64
// principal submatrix in registers (cholesky64), and k_pchol_update forms the
// panel's rows of R by forward substitution, column by column, where it needs
// them, and takes R_panel^T R_panel from the trailing matrix.  The panel ends early
// when its best candidate is below kPcLoose of the largest diagonal that is
// not a candidate (which only decrease): a pivot is never less than that part
// of the largest remaining one, and a panel has one pivot at least (1/32 took 11 panels
// where this takes 16, but an element of R may be the square root of that above
// its pivot: the smallest kept values' vectors were up to 2.4 times less accurate, and
// are as accurate as with the largest pivot in every step here).  A step of the
// panel is a chain of latencies, about 0.3 us; with whole rows of R formed in every
// step, by one workgroup, it was 2.5 us, whether the pivot's column came from
// memory or from LDS.  Sectors of up to 388 rows (m = 1500, rank 248): 16 panels of 20.1 us
// and 16 updates of 14.1, before 9 of 69.3 and 9 of 12.2.
// the remaining diagonal is held in LDS, beside 39 KB of fixed size
static_assert(sizeof(double) * kSvdMaxN + 40 * 1024 <= 160 * 1024, "the largest sector's diagonal fits");
constexpr double kPcLoose = 0.125;
constexpr double kLrCondOpen = 1e-4;
// state of one panel for the update: column k of the substitution at L[64 k ..]
// (elements t > k, and 1 / the diagonal at k)
constexpr int kPcL = kPcNbMax * kPcNbMax;

__global__ void __launch_bounds__(kJThreads) k_pchol_panel(const PcSector* ps, const double* A, const double* dg,
                                                           int* piv, int* pos, double* Lg, PcState* st) {
  extern __shared__ __attribute__((aligned(16))) double pc_lds[];   // d (n): -1 for pivots taken
  __shared__ double s_r[kJS], s_row[2][kJW], s_dc[kPcNbMax], s_max[8];
  __shared__ int s_cand[kPcNbMax], s_cnt[2][8];
  const PcSector P = ps[blockIdx.x];
  PcState& T = st[blockIdx.x];
  const int n = P.n, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k0 = T.k1;
  const bool finished = T.rank >= 0;
  __syncthreads();
  if (finished) {                      // nothing for the update either
    if (tid == 0) T.k0 = k0;
    return;
  }
  double* d = pc_lds;
  double top = -1.0;
  for (int j = tid; j < n; j += kJThreads) {
    const double v = pos[P.doff + j] >= 0 ? -1.0 : dg[P.doff + j];
    d[j] = v;
    top = fmax(top, v);
  }
  for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o));
  if (lane == 0) s_max[wave] = top;
  for (int e = tid; e < kJS; e += kJThreads) s_r[e] = 0.0;
  if (tid < kPcNbMax) s_dc[tid] = -1.0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; w++) top = fmax(top, s_max[w]);
  const double tol = kPcTol * T.dmax;
  // Candidates: those above the smallest step of a scale of quarter octaves that at
  // most 64 open columns reach, found by bisection between the threshold and the
  // largest diagonal; then some of the next step until there are 64.
  int turn = 0;
  auto total = [&](int mine) {         // the sum of a wave-uniform count over the waves
    if (lane == 0) s_cnt[turn][wave] = mine;
    __syncthreads();
    int c = 0;
#pragma unroll
    for (int w = 0; w < 8; w++) c += s_cnt[turn][w];
    turn ^= 1;
    return c;
  };
  auto key = [](double v) { return v > 0.0 ? (int)(__builtin_bit_cast(uint64_t, v) >> 50) : -1; };
  auto reach = [&](int k) {
    int c = 0;
    for (int j0 = 64 * wave; j0 < n; j0 += kJThreads) c += __popcll(__ballot(j0 + lane < n && key(d[j0 + lane]) >= k));
    return total(c);
  };
  int lo = max(key(tol), 0), hi = key(top) + 1;   // reach(hi) <= 64; reach(lo) > 64, unless every column above the threshold is taken
  if (reach(lo) <= kPcNbMax) hi = lo;
  else
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (reach(mid) <= kPcNbMax) hi = mid;
      else lo = mid;
    }
  const bool rest = hi > lo;           // open columns above the threshold that are no candidates
  for (int pass = 0, base = 0; pass < (rest ? 2 : 1); pass++) {
    int mine = 0;
    for (int j0 = 64 * wave; j0 < n; j0 += kJThreads) {
      const int k = j0 + lane < n ? key(d[j0 + lane]) : -1;
      mine += __popcll(__ballot(pass == 0 ? k >= hi : k == lo));
    }
    const int* cnt = s_cnt[turn];
    const int all = total(mine);
    int at = base;
    for (int w = 0; w < wave; w++) at += cnt[w];
    for (int j0 = 64 * wave; j0 < n; j0 += kJThreads) {
      const int j = j0 + lane;
      const double v = j < n ? d[j] : -1.0;
      const int k = key(v);
      const bool in = pass == 0 ? k >= hi : k == lo;
      const uint64_t m = __ballot(in);
      const int c = at + __popcll(m & ((1ull << lane) - 1ull));
      if (in && c < kPcNbMax) {
        s_cand[c] = j;
        s_dc[c] = v;
      }
      at += __popcll(m);
    }
    base += all;
  }
  __syncthreads();
  // the largest open diagonal that is not a candidate is below the next step of the scale
  const double next = rest ? __builtin_bit_cast(double, (uint64_t)hi << 50) : 0.0;
  const double dc = s_dc[lane];
  const bool real = dc > 0.0;
  const int cand = real ? s_cand[lane] : 0, nc = __popcll(__ballot(real));
  double x[8];
#pragma unroll
  for (int s = 0; s < 8; s++) {
    const int i = 8 * wave + s;
    x[s] = i < nc && real ? A[P.goff + (int64_t)n * s_cand[i] + cand] : 0.0;
  }
  double least = T.least;
  bool small = nc == 0;
  int order;
  bool open = real;
  const int ks = cholesky64(x, dc, open, nc, s_r, s_row, wave, lane, order, [&](int k, double m) {
    small = !(m > tol);
    if (small || m < kPcLoose * next) return true;
    if (k0 + k < P.kq) least = fmin(least, m);
    return false;
  });
  double* L = Lg + (int64_t)kPcL * blockIdx.x;
#pragma unroll
  for (int s = 0; s < 8; s++) {
    const int k = 8 * wave + s, t = lane;
    const double v = s_r[k * kJP + order];   // R(k, pivot of step t)
    L[kPcNbMax * k + t] = k >= ks || t >= ks || t < k ? 0.0 : t == k ? 1.0 / v : v;
  }
  const int col = __shfl(cand, order);
  if (wave == 0 && lane < ks) {
    piv[P.doff + k0 + lane] = col;
    pos[P.doff + col] = k0 + lane;
  }
  if (tid == 0) {
    T.least = least;
    T.k0 = k0;
    T.k1 = k0 + ks;
    T.panels++;
    // nothing left, or nothing above the threshold among the candidates and the rest (with no
    // pivot taken the rest is at most a step of the scale above the candidates)
    if (k0 + ks >= n || (small && (ks == 0 || !(next > tol)))) T.rank = k0 + ks;
  }
}

// Rows of R of a panel for 64 columns: forward substitution, a thread per column
// (y in registers, the coefficients from LDS), and G[i, j] -= sum_k R[k, i] R[k, j], 64 x 64
// tiles on the FP64 matrix cores.  The workgroups on the diagonal write R and the
// remaining diagonal.  Rows of a column are zero after the step that takes it.
constexpr int kPcP = 66;   // LDS pitch of a row of R: 64 columns
__device__ __forceinline__ void pc_rows(const double* __restrict__ Acol, int64_t n, const int* __restrict__ piv,
                                        const double* L, int ks, double (&y)[kPcNbMax]) {
  // steps and rows in groups of 8; groups beyond ks are skipped, and steps beyond it in
  // the last group have zero coefficients
#pragma unroll
  for (int tb = 0; tb < kPcNbMax; tb += 8) {
    if (tb < ks) {
#pragma unroll
      for (int t = tb; t < tb + 8; t++) y[t] = Acol[n * piv[min(t, ks - 1)]];
    }
  }
#pragma unroll
  for (int kb = 0; kb < kPcNbMax; kb += 8) {
    if (kb < ks) {
#pragma unroll
      for (int tb = kb; tb < kPcNbMax; tb += 8) {
        if (tb < ks) {
#pragma unroll
          for (int k = kb; k < kb + 8; k++) {
            if (tb == kb) y[k] *= L[kPcNbMax * k + k];
#pragma unroll
            for (int t = tb == kb ? k + 1 : tb; t < tb + 8; t++) y[t] = fma(-L[kPcNbMax * k + t], y[k], y[t]);
          }
        }
      }
    }
  }
}
__global__ void __launch_bounds__(256) k_pchol_update(const PcSector* ps, const PcState* st, const int* piv,
                                                      const int* pos, const double* __restrict__ Lg, double* A,
                                                      double* R, double* dg) {
  // the coefficients and, when every row is formed, the rows (two workgroups a CU)
  __shared__ __attribute__((aligned(16))) double lds[2 * kPcNbMax * kPcP];
  const PcSector P = ps[blockIdx.y];
  const int n = P.n, nt = (n + 63) / 64;
  const int bi = blockIdx.x % nt, bj = blockIdx.x / nt;
  const int k0 = st[blockIdx.y].k0, ks = st[blockIdx.y].k1 - k0;
  const bool finished = st[blockIdx.y].rank >= 0;
  if (bj >= nt || ks == 0 || (finished && bi != bj)) return;   // (a finished sector needs no trailing matrix)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  {
    const double* src = Lg + (int64_t)kPcL * blockIdx.y;
    const int rows = (ks + 7) & ~7;
    for (int e = threadIdx.x; e < kPcNbMax * rows; e += 256) lds[e] = src[e];
  }
  __syncthreads();
  const bool mine = wave < (bi == bj ? 1 : 2);
  double y[kPcNbMax];
  const int cc = min(64 * (wave ? bj : bi) + lane, n - 1);
  if (mine) pc_rows(A + P.goff + cc, n, piv + P.doff + k0, lds, ks, y);
  __syncthreads();
  if (mine) {
    const int taken = pos[P.doff + cc], last = taken >= 0 ? taken - k0 : kPcNbMax;
    double* Y = lds + wave * kPcNbMax * kPcP + lane;
#pragma unroll
    for (int t = 0; t < kPcNbMax; t++)
      if (t < ((ks + 3) & ~3)) Y[t * kPcP] = t <= last ? y[t] : 0.0;
  }
  __syncthreads();
  const double* Yi = lds;
  const double* Yj = lds + (bi == bj ? 0 : kPcNbMax * kPcP);
  if (bi == bj)
    for (int t = wave; t < ks; t += 4)
      if (64 * bi + lane < n) R[P.goff + (int64_t)(k0 + t) * n + 64 * bi + lane] = Yi[t * kPcP + lane];
  if (finished) return;
  // wave w: rows 16 w .. 16 w + 15 of the tile, its four 16-column pieces; D[l/16 + 4 r][l%16]
  const int j = lane & 15, g = lane >> 4;
  jac_v4d acc[4] = {};
  for (int k = 0; k < ks; k += 4) {    // (rows of Y beyond ks are zero)
    const double a = Yj[(k + g) * kPcP + 16 * wave + j];
#pragma unroll
    for (int u = 0; u < 4; u++)
      acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, Yi[(k + g) * kPcP + 16 * u + j], acc[u], 0, 0, 0);
  }
  // columns that are pivots stay as they are: other workgroups read them here, and
  // nothing reads them later
  bool open[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int col = 64 * bj + 16 * wave + g + 4 * r;
    open[r] = col < n && pos[P.doff + col] < 0;
  }
#pragma unroll
  for (int u = 0; u < 4; u++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = 64 * bi + 16 * u + j, col = 64 * bj + 16 * wave + g + 4 * r;
      if (row < n && open[r]) {
        double* e = A + P.goff + row + (int64_t)n * col;
        const double v = *e - acc[u][r];
        *e = v;
        if (row == col) dg[P.doff + row] = v;
      }
    }
}

// X (in G's place): columns c < r of R^T W scaled by 1 / sqrt(lambda_c), eigenvalue lambda_c;
// columns c >= r of V: zero, eigenvalue 0
__global__ void k_lr_scale(const PcSector* ps, const int* rk, const int64_t* eoff2, const double* ev2,
                           const int64_t* eoff, double* X, double* Vev, double* ev) {
  const PcSector P = ps[blockIdx.y];
  const int n = P.n, r = rk[blockIdx.y];
  const int c = blockIdx.x;
  if (c >= n) return;
  const double lam = c < r ? ev2[eoff2[blockIdx.y] + c] : 0.0;
  const double sc = lam > 0.0 ? 1.0 / sqrt(lam) : 0.0;
  double* col = (c < r ? X : Vev) + P.goff + (int64_t)n * c;
  for (int i = threadIdx.x; i < n; i += blockDim.x) col[i] = c < r ? col[i] * sc : 0.0;
  if (threadIdx.x == 0) ev[eoff[P.q] + c] = lam;
}

// The Gram-Schmidt coefficients of X from M = X^T X (r x r): column c of V is X C_c,
// C(a, c) = -M(a, c) for lambda_a > lambda_c, (3 - M(c, c)) / 2 at c
__global__ void __launch_bounds__(256) k_lr_order(const int* rk, const int64_t* goff2, const int64_t* eoff2,
                                                  const double* ev2, const double* M, double* C) {
  const int r = rk[blockIdx.y], c = blockIdx.x;
  if (c >= r) return;
  const double* lam = ev2 + eoff2[blockIdx.y];
  const int64_t o = goff2[blockIdx.y] + (int64_t)r * c;
  const double lc = lam[c];
  for (int a = threadIdx.x; a < r; a += 256) {
    const double la = lam[a], m = M[o + a];
    C[o + a] = a == c ? 1.5 - 0.5 * m : (la > lc || (la == lc && a < c)) ? -m : 0.0;
  }
}

// 5a. per sector: eigen order (descending), top-k singular values in the
// reference's sector / descending order, selected eigenvectors packed
// ordering key of a value: NaN compares as -inf, so that rank counts over
// any input form a permutation
__device__ inline double rank_key(double v) { return v == v ? v : -INFINITY; }

// every sector's Gram diagonal finite (a Gram matrix's entries are bounded by
// its diagonal, and a NaN input reaches the diagonal); *bad = 1 otherwise
__global__ void __launch_bounds__(256) k_svd_finite(int nQ, const int* nq, const int64_t* goff,
                                                    const double* G, int* bad) {
  const int q = blockIdx.x;
  if (q >= nQ) return;
  const int n = nq[q];
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    if (!isfinite(G[goff[q] + i + (int64_t)n * i])) *bad = 1;
}

// 5a. per sector: the rank of each eigenvalue (descending, ties by index; a
// NaN ranks as -inf, so the ranks are a permutation for any input), the kept
// singular values in rank order and the eigenpair index of each kept rank.
// One thread per eigenvalue (grid: sectors x 256-value groups); the sector's
// eigenvalues pass through LDS in chunks, so every comparison reads one
// broadcast LDS value.
constexpr int kRankChunk = 2048;
__global__ void __launch_bounds__(256) k_svd_select(const int* nq, const int* kq,
                                                    const int64_t* eoff, const double* evals,
                                                    const int64_t* soff, double* svals,
                                                    int* ssec, int* selidx) {
  __shared__ double chunk[kRankChunk];
  const int q = blockIdx.x;
  const int n = nq[q], k = kq[q];
  if ((int)blockIdx.y * 256 >= n) return;   // the whole workgroup: before any barrier
  const int i = blockIdx.y * 256 + threadIdx.x;
  const double* ev = evals + eoff[q];
  const double v = i < n ? rank_key(ev[i]) : 0.0;
  int r = 0;
  for (int c0 = 0; c0 < n; c0 += kRankChunk) {
    const int cn = min(kRankChunk, n - c0);
    __syncthreads();
#pragma unroll 8
    for (int e = threadIdx.x; e < cn; e += 256) chunk[e] = rank_key(ev[c0 + e]);
    __syncthreads();
    for (int j = 0; j < cn; j++) {
      const double u = chunk[j];
      r += (u > v) || (u == v && c0 + j < i);
    }
  }
  if (i < n && r < k) {
    svals[soff[q] + r] = sqrt(fmax(v, 0.0));
    ssec[soff[q] + r] = q;
    selidx[soff[q] + r] = i;
  }
}

// the selected eigenvectors packed in rank order, Esel_q(:, r) = V_q(:, selidx_q[r]):
// workgroups over (sector, columns), consecutive threads on consecutive rows
__global__ void __launch_bounds__(256) k_svd_gather_sel(const int* nq, const int* kq,
                                                        const int64_t* goff, const double* V,
                                                        const int64_t* soff, const int* selidx,
                                                        const int64_t* selo, double* Esel) {
  const int q = blockIdx.x;
  const int n = nq[q], k = kq[q];
  for (int r = blockIdx.y; r < k; r += gridDim.y) {
    const double* src = V + goff[q] + (int64_t)n * selidx[soff[q] + r];
    double* dst = Esel + selo[q] + (int64_t)n * r;
    for (int row = threadIdx.x; row < n; row += blockDim.x) dst[row] = src[row];
  }
}

// 5b. truncation (qtensor_op.cpp:1280-1301): nm and cumsum are summed
// sequentially in the reference's order; the global order is a stable
// descending sort (the reference's std::sort is unstable on ties).
// 5b. global descending order of all singular values (ties by position,
// a stable sort as the reference's pairCompare sort over (sector, desc) order).
// Each sector's values are already non-increasing (k_svd_select), so the rank
// of value v at position j of sector q is j, plus the values >= v of the
// sectors before q (they come first on ties), plus the values > v of the
// sectors after it: one binary search per other sector instead of a pass
// over all values.
__device__ inline int count_ge(const double* a, int n, double v) {   // a non-increasing
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] >= v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}
__device__ inline int count_gt(const double* a, int n, double v) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] > v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}
__global__ void __launch_bounds__(256) k_svd_rank(int T, int nQ, const int64_t* __restrict__ soff,
                                                  const double* __restrict__ svals, int* __restrict__ order,
                                                  double* __restrict__ sorted) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T) return;
  const double v = svals[i];
  int lo = 0, hi = nQ;   // sector q of i: the last q with soff[q] <= i
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (soff[mid] <= i) lo = mid;
    else hi = mid;
  }
  const int q = lo;
  int r = i - (int)soff[q];
  for (int o = 0; o < nQ; o++) {
    if (o == q) continue;
    const double* a = svals + soff[o];
    const int n = (int)(soff[o + 1] - soff[o]);
    r += o < q ? count_ge(a, n, v) : count_gt(a, n, v);
  }
  order[r] = i;
  sorted[r] = v;
}

// 5c. the reference's keep loop (qtensor_op.cpp:1294-1300), sequential in its
// summation order: nm over (sector, descending) order, cumsum over the sorted
// values
constexpr int kTrChunk = 2048;   // values staged in LDS per pass of the serial loops
constexpr int kTrPer = kTrChunk / 256;   // staged values per thread (launched with 256 threads)
// The serial loops add precomputed terms: every thread forms its values'
// square s*s (for nm) and s*s/nm (for cumsum), each rounded as the
// reference's expressions round them, and one thread adds them in order, so
// the sums are the reference's and the serial chain holds no multiply or
// divide.
__global__ void __launch_bounds__(256) k_svd_truncate(int T, int nQ, const double* svals, const int* ssec,
                                                      const int* order, const double* sorted, double cutoff,
                                                      int64_t K, int* newdim, double* out) {
  __shared__ double val[kTrChunk];
  __shared__ double term[kTrChunk];
  __shared__ double s_nm, s_cum;
  __shared__ long long s_acc;
  __shared__ int s_done;
  const int tid = threadIdx.x;
  // nm: the sum of squares in the (sector, descending) order
  double nm = 0.0;
  for (int c0 = 0; c0 < T; c0 += kTrChunk) {
    const int cn = min(kTrChunk, T - c0);
    {   // a thread's loads are all issued before its stores
      double v[kTrPer];
#pragma unroll
      for (int u = 0; u < kTrPer; u++) {
        const int e = tid + 256 * u;
        v[u] = e < cn ? svals[c0 + e] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < kTrPer; u++) {
        const int e = tid + 256 * u;
        if (e < cn) term[e] = v[u] * v[u];
      }
    }
    __syncthreads();
    if (tid == 0) {
      // unrolled so that the LDS reads run ahead of the (ordered) adds
#pragma unroll 8
      for (int e = 0; e < cn; e++) nm += term[e];
    }
    __syncthreads();
  }
  if (tid == 0) { s_nm = nm; s_cum = 0.0; s_acc = 0; s_done = 0; }
  __syncthreads();
  nm = s_nm;
  // the keep loop over the sorted values, in order, chunk by chunk
  for (int c0 = 0; c0 < T; c0 += kTrChunk) {
    if (s_done) break;   // read after a barrier: the same value in every thread
    const int cn = min(kTrChunk, T - c0);
    {
      double v[kTrPer];
#pragma unroll
      for (int u = 0; u < kTrPer; u++) {
        const int e = tid + 256 * u;
        v[u] = e < cn ? sorted[c0 + e] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < kTrPer; u++) {
        const int e = tid + 256 * u;
        if (e < cn) {
          val[e] = v[u];
          term[e] = v[u] * v[u] / nm;
        }
      }
    }
    __syncthreads();
    if (tid == 0) {
      double cumsum = s_cum;
      long long acc = s_acc;
      int done = 0;
#pragma unroll 8
      for (int e = 0; e < cn; e++) {
        cumsum += term[e];
        if (val[e] == 0. && cutoff != 0.) { done = 1; break; }
        acc += 1;
        if ((1 - cumsum < cutoff && cutoff != 0.) || (acc >= K && K != 0)) { done = 1; break; }
      }
      s_cum = cumsum;
      s_acc = acc;
      s_done = done;
    }
    __syncthreads();
  }
  // kept values per sector: the first acc entries of the sorted order
  const long long acc = s_acc;
  for (long long i = tid; i < acc; i += blockDim.x) {
    const int oi = order[i];
    const int q = (oi >= 0 && oi < T) ? ssec[oi] : -1;
    if (q >= 0 && q < nQ) atomicAdd(&newdim[q], 1);   // unreachable otherwise: order and ssec are complete
  }
  if (tid == 0) {
    out[0] = fmax(1 - s_cum, 0.0);
    out[1] = (double)acc;
  }
}

// 6a. block lists of U (left..., mid) and V (mid, right...) and S (mid)
__global__ void __launch_bounds__(1024) k_svd_emit(MetaView A, int nleft, SvdTab t, int nQ,
                                                   const int* newdim, const int* midnum,
                                                   int* uqi, int64_t* uoff, int* vqi,
                                                   int64_t* voff) {
  __shared__ int64_t lds[32];
  const int nuL = (int)t.hdr[0], nuR = (int)t.hdr[1];
  const int rU = nleft + 1, rV = A.rank - nleft + 1;
  // U: entries of uL whose sector keeps values, in (sector, left) order
  int64_t cb = 0, co = 0;
  for (int base = 0; base < nuL; base += 1024) {
    int i = base + threadIdx.x;
    int q = -1;
    int64_t f = 0, sz = 0;
    if (i < nuL) {
      int lo = 0, hi = nQ;
      while (lo < hi) { int m = (lo + hi) >> 1; if (t.qL0[m] <= i) lo = m + 1; else hi = m; }
      q = lo - 1;
      f = newdim[q] > 0;
      sz = f ? t.lsz[i] * newdim[q] : 0;
    }
    int64_t tb, ts;
    int64_t pb = block_excl_scan<1024>(f, lds, &tb);
    int64_t ps = block_excl_scan<1024>(sz, lds, &ts);
    if (f) {
      uint64_t key = t.uL[i] & 0xffffffffull;
      for (int j = nleft - 1; j >= 0; j--) { uqi[(cb + pb) * rU + j] = (int)(key % A.nsec[j]); key /= A.nsec[j]; }
      uqi[(cb + pb) * rU + nleft] = midnum[q];
      uoff[cb + pb] = co + ps;
    }
    cb += tb;
    co += ts;
  }
  if (threadIdx.x == 0) uoff[cb] = co;
  __syncthreads();
  cb = 0;
  co = 0;
  for (int base = 0; base < nuR; base += 1024) {
    int i = base + threadIdx.x;
    int64_t f = 0, sz = 0;
    int q = -1;
    if (i < nuR) {
      const uint64_t qc = t.uR[i] >> 32;
      int lo = 0, hi = nQ;
      while (lo < hi) { int m = (lo + hi) >> 1; if (t.qc[m] < qc) lo = m + 1; else hi = m; }
      q = lo;
      f = newdim[q] > 0;
      sz = f ? t.rsz[i] * newdim[q] : 0;
    }
    int64_t tb, ts;
    int64_t pb = block_excl_scan<1024>(f, lds, &tb);
    int64_t ps = block_excl_scan<1024>(sz, lds, &ts);
    if (f) {
      uint64_t key = t.uR[i] & 0xffffffffull;
      vqi[(cb + pb) * rV] = midnum[q];
      for (int j = A.rank - 1; j >= nleft; j--) {
        vqi[(cb + pb) * rV + 1 + (j - nleft)] = (int)(key % A.nsec[j]);
        key /= A.nsec[j];
      }
      voff[cb + pb] = co + ps;
    }
    cb += tb;
    co += ts;
  }
  if (threadIdx.x == 0) voff[cb] = co;
}

// 6b. slice sector matrices into blocks.  U_q (rows x k, ld rows) ->
// U blocks (lsize x k);  W_q (k x cols, ld k) -> V blocks (k x rsize).
// Workgroups over (sector, columns): a column of a block is contiguous on
// both sides.
__global__ void __launch_bounds__(256) k_svd_scatter(SvdTab t, int nQ, const int* newdim,
                                                     const int* ublk0, const int* vblk0,
                                                     const int64_t* uoffs, const int64_t* voffs,
                                                     const double* Umat, const int64_t* umo,
                                                     const double* Wmat, const int64_t* wmo,
                                                     double* Ud, double* Vd) {
  const int q = blockIdx.x;
  const int k = newdim[q];
  if (k == 0) return;
  const int64_t rows = t.rows[q];
  int ub = ublk0[q];
  for (int i = t.qL0[q]; i < t.qL1[q]; i++, ub++) {
    const int ls = (int)t.lsz[i];
    const int64_t lo = t.loff[i];
    for (int c = blockIdx.y; c < k; c += gridDim.y) {
      double* dst = Ud + uoffs[ub] + (int64_t)ls * c;
      const double* src = Umat + umo[q] + lo + rows * c;
      for (int r = threadIdx.x; r < ls; r += blockDim.x) dst[r] = src[r];
    }
  }
  int vb = vblk0[q];
  for (int i = t.qR0[q]; i < t.qR1[q]; i++, vb++) {
    const int rs = (int)t.rsz[i];
    const int64_t co = t.roff[i];
    for (int c = blockIdx.y; c < rs; c += gridDim.y) {
      double* dst = Vd + voffs[vb] + (int64_t)k * c;
      const double* src = Wmat + wmo[q] + (int64_t)k * (co + c);
      for (int r = threadIdx.x; r < k; r += blockDim.x) dst[r] = src[r];
    }
  }
}

// the unabsorbed factor without a product: W_q = E^T (k x cols) for
// MoveFromRight, by 32 x 32 tiles through LDS (reads along E's columns,
// writes along W's columns); tiles over (sector, tile index)
constexpr int kTT = 32;
__global__ void __launch_bounds__(256) k_svd_transpose(int nQ, const int* nq, const int* newdim,
                                                       const int64_t* selo, const double* E,
                                                       const int64_t* wmo, double* W) {
  __shared__ double tile[kTT][kTT + 1];
  const int q = blockIdx.x;
  const int n = nq[q], k = newdim[q];
  const int ti = (n + kTT - 1) / kTT, tc = (k + kTT - 1) / kTT;
  const int x = threadIdx.x % kTT, y0 = threadIdx.x / kTT;   // 32 x 8 threads
  for (int tt = blockIdx.y; tt < ti * tc; tt += gridDim.y) {
    const int i0 = (tt % ti) * kTT, c0 = (tt / ti) * kTT;
    __syncthreads();
    for (int y = y0; y < kTT; y += 8)   // E(i0 + x, c0 + y)
      if (i0 + x < n && c0 + y < k) tile[y][x] = E[selo[q] + (i0 + x) + (int64_t)n * (c0 + y)];
    __syncthreads();
    for (int y = y0; y < kTT; y += 8)   // W(c0 + x, i0 + y) = E(i0 + y, c0 + x)
      if (c0 + x < k && i0 + y < n) W[wmo[q] + (c0 + x) + (int64_t)k * (i0 + y)] = tile[x][y];
  }
}

// U_q = the first k columns of Esel_q (rows x kq, ld rows) for MoveFromLeft
__global__ void __launch_bounds__(256) k_svd_copy_sel(int nQ, const int64_t* rowsq, const int* newdim,
                                                      const int64_t* selo, const double* E,
                                                      const int64_t* umo, double* U) {
  const int q = blockIdx.x;
  const int64_t tot = rowsq[q] * newdim[q];
  for (int64_t e = (int64_t)blockIdx.y * blockDim.x + threadIdx.x; e < tot;
       e += (int64_t)gridDim.y * blockDim.x)
    U[umo[q] + e] = E[selo[q] + e];
}

__global__ void k_svd_svals(int nQ, const int* newdim, const int64_t* soff, const double* svals,
                            const int64_t* sout_off, double* S) {
  const int q = blockIdx.x;
  for (int i = threadIdx.x; i < newdim[q]; i += blockDim.x) S[sout_off[q] + i] = svals[soff[q] + i];
}

// grouped GEMM over sectors with host-built tasks
struct HostGemm {
  std::vector<GemmTask> tasks;
  std::vector<CBlock> cblk;
};

static int run_host_gemm(HostGemm& hg, const double* A, const double* B, double* C) {
  if (hg.cblk.empty()) return 0;
  ttg_plan_s p;
  p.prec = TTG_FP64;
  p.cfg = TILE_64x64;
  const int TK = tk_of(p.prec);
  for (CBlock& b : hg.cblk) {   // k-tile offsets of each block's walk
    int kt = 0;
    for (int t = b.t0; t < b.t1; t++) {
      GemmTask& g = hg.tasks[t];
      g.kt0 = kt;
      kt += (g.K / g.ek0) * ((g.ek0 + TK - 1) / TK);
    }
    b.nkt = kt;
  }
  p.ntasks = (int64_t)hg.tasks.size();
  const GemmTask& g0 = hg.tasks[0];
  p.a_mcontig = g0.sam0 == 1;
  p.b_kcontig = g0.sbk0 == 1;
  p.d_tasks = dalloc<GemmTask>(hg.tasks.size());
  p.d_cblk = dalloc<CBlock>(hg.cblk.size());
  TTG_REQUIRE(p.d_tasks && p.d_cblk, (std::string("svd: ") + ttg_last_error()).c_str());
  hipStream_t s = stream();
  UploadBatch up;
  TTG_TRY(h2d_vec(p.d_tasks, hg.tasks));
  TTG_TRY(h2d_vec(p.d_cblk, hg.cblk));
  TTG_TRY(build_tiles(p, hg.cblk));
  TTG_TRY(up.flush());
  TTG_TRY(gemm_launch(p, A, B, C, true, s));
  return 0;   // p's destructor returns the device arrays to the pool (stream-ordered reuse)
}

static GemmTask gtask(int64_t a_off, int64_t b_off, int em0, int64_t sam0, int ek0, int64_t sak0,
                      int64_t sbk0, int en0, int64_t sbn0, int K) {
  GemmTask g{};
  g.a_off = a_off; g.b_off = b_off;
  g.em0 = em0; g.sam0 = sam0; g.sam1 = 0;
  g.ek0 = ek0; g.sak0 = sak0; g.sak1 = 0; g.sbk0 = sbk0; g.sbk1 = 0;
  g.en0 = en0; g.sbn0 = sbn0; g.sbn1 = 0;
  g.K = K;
  g.nk1 = K / ek0;
  return g;
}

// host arrays uploaded as one copy into one scratch allocation: add() the
// arrays, upload(), then at<T>(offset) gives each array's device address
class Pack {
 public:
  template <class T>
  size_t add(const std::vector<T>& v) {
    const size_t off = (bytes_.size() + 15) & ~size_t(15);
    bytes_.resize(off + sizeof(T) * std::max<size_t>(v.size(), 1));
    if (!v.empty()) memcpy(bytes_.data() + off, v.data(), sizeof(T) * v.size());
    return off;
  }
  int upload(Scratch& sc, const char* what) {
    d_ = sc.get<char>(std::max<size_t>(bytes_.size(), 1));
    TTG_TRY(sc.ok(what));
    return h2d(d_, bytes_.data(), bytes_.size());
  }
  template <class T>
  T* at(size_t off) const {
    return (T*)(d_ + off);
  }

 private:
  std::vector<char> bytes_;
  char* d_ = nullptr;
};

// eigenpairs of the large sectors `big` through the LR step (see 4c); without
// `drop`, the sectors that the step cannot serve go to `plain`
static int lr_eigen(const std::vector<int>& big, const std::vector<int>& nq, const std::vector<int>& kq, bool drop,
                    std::vector<int>& plain, const std::vector<int64_t>& goff,
                    const std::vector<int64_t>& eoff, const int64_t* d_eoff, int64_t gtotal, double* G,
                    double* Vev, double* ev, hipStream_t s) {
  PhaseTimer _phase("lr_eigen");
  const int ns = (int)big.size();
  std::vector<PcSector> ps(ns);
  int nmax = 0;
  int64_t dtot = 0;
  for (int li = 0; li < ns; li++) {
    const int q = big[li];
    ps[li] = PcSector{nq[q], q, kq[q], 0, goff[q], dtot};
    dtot += nq[q];
    nmax = std::max(nmax, nq[q]);
  }
  const size_t lds = sizeof(double) * nmax;
  Scratch sc;
  PcSector* d_ps = sc.get<PcSector>(ns);
  double* R = sc.get<double>(gtotal);
  double* dg = sc.get<double>(dtot);
  int* piv = sc.get<int>(dtot);
  int* pos = sc.get<int>(dtot);
  double* Lg = sc.get<double>((size_t)kPcL * ns);
  PcState* d_st = sc.get<PcState>(ns);
  TTG_TRY(sc.ok("svd: LR step"));
  TTG_TRY(h2d_vec(d_ps, ps));
  hipLaunchKernelGGL(k_pchol_init, dim3(ns), dim3(kPcThreads), 0, s, d_ps, G, dg, pos, d_st);
  TTG_HIP(hipFuncSetAttribute((const void*)k_pchol_panel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds));
  const int nt = (nmax + 63) / 64;
  // Panels are launched up to one more than the previous call needed, then
  // the ranks are read back, and while a sector is running some more follow
  // (a finished sector's launches exit at once, but each launch still costs
  // a few microseconds).
  static int prev_panels = 0;
  int more = prev_panels > 0 ? prev_panels + 1 : (nmax + kPcNbMax - 1) / kPcNbMax;
  std::vector<PcState> pst(ns);
  for (int done = 0; done <= nmax; done += more, more = 4) {   // every panel takes a pivot or ends its sector
    for (int i = 0; i < more; i++) {
      hipLaunchKernelGGL(k_pchol_panel, dim3(ns), dim3(kJThreads), lds, s, d_ps, G, dg, piv, pos, Lg, d_st);
      hipLaunchKernelGGL(k_pchol_update, dim3(nt * nt, ns), dim3(256), 0, s, d_ps, d_st, piv, pos, Lg, G, R, dg);
    }
    const D2HPiece pc{pst.data(), d_st, sizeof(PcState) * ns};
    TTG_TRY(d2h_wait(&pc, 1));
    bool running = false;
    for (const PcState& t : pst) running |= t.rank < 0;
    if (!running) break;
  }
  prev_panels = 0;
  for (const PcState& t : pst) prev_panels = std::max(prev_panels, t.panels);
  std::vector<int> r2(ns);
  std::vector<int64_t> goff2(ns + 1, 0), eoff2(ns + 1, 0);
  bool any_small = false;
  std::vector<int> big2;
  for (int li = 0; li < ns; li++) {
    TTG_REQUIRE(pst[li].rank >= 0, "svd: the pivoted Cholesky factorisation did not end");
    int r = pst[li].rank;
    const double cond = r < ps[li].n ? kLrCondOpen : kLrCond;
    if (!drop && (r < ps[li].kq || pst[li].least < cond * pst[li].dmax)) {
      plain.push_back(big[li]);
      r = 0;
    }
    r2[li] = r;
    goff2[li + 1] = goff2[li] + (int64_t)r * r;
    eoff2[li + 1] = eoff2[li] + r;
    if (r > kJacBlockMin) big2.push_back(li);
    else if (r > 0) any_small = true;
  }
  double* G2 = sc.get<double>(std::max<int64_t>(1, goff2[ns]));
  double* W2 = sc.get<double>(std::max<int64_t>(1, goff2[ns]));
  double* ev2 = sc.get<double>(std::max<int64_t>(1, eoff2[ns]));
  TTG_TRY(sc.ok("svd: LR step"));
  Pack pk;
  const size_t o_r2 = pk.add(r2), o_goff2 = pk.add(goff2), o_eoff2 = pk.add(eoff2);
  TTG_TRY(pk.upload(sc, "svd: LR step"));
  int* d_r2 = pk.at<int>(o_r2);
  int64_t* d_goff2 = pk.at<int64_t>(o_goff2);
  int64_t* d_eoff2 = pk.at<int64_t>(o_eoff2);
  // G' = R R^T: A(k, j) = R[k n + j], B(j, k') = R[k' n + j]
  {
    HostGemm hg;
    for (int li = 0; li < ns; li++) {
      const int n = ps[li].n, r = r2[li];
      if (r == 0) continue;
      hg.tasks.push_back(gtask(ps[li].goff, ps[li].goff, r, n, n, 1, 1, r, n, n));
      const int t = (int)hg.tasks.size() - 1;
      hg.cblk.push_back(CBlock{goff2[li], r, r, t, t + 1});
    }
    TTG_TRY(run_host_gemm(hg, R, R, G2));
  }
  // eigenpairs of G' (relative convergence test only)
  if (any_small) {
    hipLaunchKernelGGL(k_jacobi, dim3(ns), dim3(kJThreads), 0, s, d_r2, (const int*)nullptr, 0, d_goff2, G2, W2, ev2, d_eoff2, 40,
                       kJacBlockMin, 0.0);
    TTG_HIP(hipGetLastError());
  }
  if (!big2.empty()) TTG_TRY(block_jacobi(big2, r2, d_goff2, d_eoff2, G2, W2, ev2, s, 40, 0.0));
  // X = R^T W Lambda^(-1/2), in G's place: A(j, k) = R[k n + j], B(k, c) = W[k + r c];
  // M = X^T X, in G2's: A(c, i) = X[i + n c], B(i, a) = X[i + n a];
  // V = X C: A(i, a) = X[i + n a], B(a, c) = C[a + r c]
  HostGemm hx, hm, hv;
  for (int li = 0; li < ns; li++) {
    const int n = ps[li].n, r = r2[li];
    if (r == 0) continue;
    const int t = (int)hx.tasks.size();
    hx.tasks.push_back(gtask(ps[li].goff, goff2[li], n, 1, r, n, 1, r, r, r));
    hx.cblk.push_back(CBlock{ps[li].goff, n, r, t, t + 1});
    hm.tasks.push_back(gtask(ps[li].goff, ps[li].goff, r, n, n, 1, 1, r, n, n));
    hm.cblk.push_back(CBlock{goff2[li], r, r, t, t + 1});
    hv.tasks.push_back(gtask(ps[li].goff, goff2[li], n, 1, r, n, 1, r, r, r));
    hv.cblk.push_back(CBlock{ps[li].goff, n, r, t, t + 1});
  }
  TTG_TRY(run_host_gemm(hx, R, W2, G));
  hipLaunchKernelGGL(k_lr_scale, dim3(nmax, ns), dim3(256), 0, s, d_ps, d_r2, d_eoff2, ev2, d_eoff, G, Vev, ev);
  TTG_TRY(run_host_gemm(hm, G, G, G2));
  hipLaunchKernelGGL(k_lr_order, dim3(nmax, ns), dim3(256), 0, s, d_r2, d_goff2, d_eoff2, ev2, G2, W2);
  TTG_HIP(hipGetLastError());
  return run_host_gemm(hv, G, W2, Vev);
}

}  // namespace ttg

using namespace ttg;

extern "C" int ttg_svd(ttg_tensor A, int nleft, int direction, double cutoff, int64_t K,
                       ttg_tensor* Uout, ttg_tensor* Sout, ttg_tensor* Vout, double* trunc_err,
                       int64_t* kept) {
  PhaseTimer _phase("ttg_svd");
  TTG_REQUIRE(A && Uout && Sout && Vout, "svd: null argument");
  const TMeta& m = *A->m;
  TTG_REQUIRE(nleft >= 1 && nleft < m.rank, "svd: need at least one left and one right index");
  TTG_REQUIRE(direction == TTG_MOVE_FROM_LEFT || direction == TTG_MOVE_FROM_RIGHT, "svd: direction");
  double rl = 1, rr = 1;
  for (int j = 0; j < m.rank; j++) (j < nleft ? rl : rr) *= m.nsec[j];
  TTG_REQUIRE(rl < 4294967295.0 && rr < 4294967295.0, "svd: sector-tuple key exceeds 32 bits");
  hipStream_t s = stream();
  const int nb = m.nblocks;
  TTG_REQUIRE(nb > 0, "svd: tensor without blocks");
  // ---- 1. bookkeeping
  Scratch sc;   // every buffer below goes back to the pool on return
  uint64_t *kl = sc.get<uint64_t>(nb), *kr = sc.get<uint64_t>(nb);
  uint64_t *sl = sc.get<uint64_t>(nb), *sr = sc.get<uint64_t>(nb);
  int *ids = sc.get<int>(nb), *sid = sc.get<int>(nb);
  SvdTab t{};
  t.uL = sc.get<uint64_t>(nb); t.uR = sc.get<uint64_t>(nb);
  t.lsz = sc.get<int64_t>(nb); t.loff = sc.get<int64_t>(nb);
  t.rsz = sc.get<int64_t>(nb); t.roff = sc.get<int64_t>(nb);
  // the header and the per-sector tables the host reads, in one allocation
  // (read back with one copy): hdr[4], rows, cols (int64), qc, qL0, qL1,
  // qR0, qR1 (32-bit), nb entries each
  const size_t nbp = ((size_t)nb + 31) & ~size_t(31);
  const size_t tab_bytes = 32 + nbp * (2 * sizeof(int64_t) + 5 * sizeof(int));
  char* tabs = sc.get<char>(tab_bytes);
  TTG_TRY(sc.ok("svd"));
  t.hdr = (int64_t*)tabs;
  t.rows = (int64_t*)(tabs + 32);
  t.cols = t.rows + nbp;
  t.qc = (uint32_t*)(t.cols + nbp);
  t.qL0 = (int*)(t.qc + nbp);
  t.qL1 = t.qL0 + nbp;
  t.qR0 = t.qL1 + nbp;
  t.qR1 = t.qR0 + nbp;
  const unsigned g1 = (nb + 255) / 256;
  hipLaunchKernelGGL(k_svd_keys, dim3(g1), dim3(256), 0, s, m.view(), nleft, kl, kr, ids);
  hipLaunchKernelGGL(k_sort_keys, dim3(g1), dim3(256), 0, s, kl, ids, nb, sl, sid);
  hipLaunchKernelGGL(k_sort_keys, dim3(g1), dim3(256), 0, s, kr, ids, nb, sr, sid);
  hipLaunchKernelGGL(k_svd_unique, dim3(1), dim3(1024), 0, s, m.view(), nleft, sl, sr, nb, t);
  std::vector<char> htab(tab_bytes);
  {
    const D2HPiece pc{htab.data(), tabs, tab_bytes};
    TTG_TRY(d2h_wait(&pc, 1));
  }
  int64_t hdr[4];
  memcpy(hdr, htab.data(), sizeof(hdr));
  const int nuL = (int)hdr[0], nuR = (int)hdr[1], nQ = (int)hdr[2];
  TTG_REQUIRE(nQ >= 0 && nQ <= nb, "svd: bad sector count");
  auto tab = [&](const void* dptr, auto* dst, size_t elem) {
    memcpy(dst, htab.data() + ((const char*)dptr - tabs), elem * nQ);
  };
  std::vector<int64_t> rows(nQ), cols(nQ);
  std::vector<uint32_t> qcs(nQ);
  std::vector<int> qL0(nQ), qL1(nQ), qR0(nQ), qR1(nQ);
  tab(t.rows, rows.data(), sizeof(int64_t));
  tab(t.cols, cols.data(), sizeof(int64_t));
  tab(t.qc, qcs.data(), sizeof(uint32_t));
  tab(t.qL0, qL0.data(), sizeof(int));
  tab(t.qL1, qL1.data(), sizeof(int));
  tab(t.qR0, qR0.data(), sizeof(int));
  tab(t.qR1, qR1.data(), sizeof(int));
  // ---- host layout of the per-sector work arrays
  const bool fromLeft = direction == TTG_MOVE_FROM_LEFT;
  std::vector<int64_t> moff(nQ + 1, 0), goff(nQ + 1, 0), eoff(nQ + 1, 0);
  std::vector<int> nq(nQ), kq(nQ);
  for (int q = 0; q < nQ; q++) {
    const int64_t n = fromLeft ? rows[q] : cols[q];
    TTG_REQUIRE(n <= kSvdMaxN, "svd: sector larger than 8192");
    nq[q] = (int)n;
    int kd = (int)std::min(rows[q], cols[q]);
    kq[q] = K > 0 ? (int)std::min<int64_t>(K, kd) : kd;   // rank-K SVD per sector
    moff[q + 1] = moff[q] + rows[q] * cols[q];
    goff[q + 1] = goff[q] + n * n;
    eoff[q + 1] = eoff[q] + n;
  }
  std::vector<int64_t> soff(nQ + 1, 0), selo(nQ + 1, 0);
  for (int q = 0; q < nQ; q++) {
    soff[q + 1] = soff[q] + kq[q];
    selo[q + 1] = selo[q] + (int64_t)nq[q] * kq[q];
  }
  double* mat = sc.get<double>(moff[nQ]);
  double* G = sc.get<double>(goff[nQ]);
  double* Vev = sc.get<double>(goff[nQ]);
  double* ev = sc.get<double>(eoff[nQ]);
  double* Esel = sc.get<double>(selo[nQ]);
  int* selidx = sc.get<int>(soff[nQ]);
  double* svals = sc.get<double>(soff[nQ]);
  int* ssec = sc.get<int>(soff[nQ]);
  int* order = sc.get<int>(soff[nQ]);
  double* ssorted = sc.get<double>(soff[nQ]);
  double* tout = sc.get<double>(2);
  TTG_TRY(sc.ok("svd"));
  Pack pk;
  const size_t o_moff = pk.add(moff), o_goff = pk.add(goff), o_eoff = pk.add(eoff),
               o_soff = pk.add(soff), o_selo = pk.add(selo), o_nq = pk.add(nq), o_kq = pk.add(kq),
               o_nd = pk.add(std::vector<int>(nQ, 0)), o_bad = pk.add(std::vector<int>(1, 0));
  TTG_TRY(pk.upload(sc, "svd"));
  int64_t* d_moff = pk.at<int64_t>(o_moff);
  int64_t* d_goff = pk.at<int64_t>(o_goff);
  int64_t* d_eoff = pk.at<int64_t>(o_eoff);
  int64_t* d_soff = pk.at<int64_t>(o_soff);
  int64_t* d_selo = pk.at<int64_t>(o_selo);
  int* d_nq = pk.at<int>(o_nq);
  int* d_kq = pk.at<int>(o_kq);
  int* newdim = pk.at<int>(o_nd);   // zero
  int* bad = pk.at<int>(o_bad);     // zero
  // ---- 2. gather
  fill_f64(mat, moff[nQ], 0.0);
  hipLaunchKernelGGL(k_svd_gather, dim3(std::min(nb, 4096)), dim3(256), 0, s, m.view(), nleft,
                     A->d_data, t, nuL, nuR, nQ, d_moff, mat);
  // ---- 3. Gram on MFMA
  auto gram = [&](const std::vector<int>& of) {
    HostGemm hg;
    for (int q : of) {
      const int n = nq[q], t = (int)hg.tasks.size();
      const int64_t r = rows[q], c = cols[q];
      if (fromLeft)   // G = A A^T : A(m=i, k=j) = mat[i + r j]; B(k=j, n=i') = mat[i' + r j]
        hg.tasks.push_back(gtask(moff[q], moff[q], (int)r, 1, (int)c, r, r, (int)r, 1, (int)c));
      else            // G = A^T A : A(m=j, k=i) = mat[i + r j]; B(k=i, n=j') = mat[i + r j']
        hg.tasks.push_back(gtask(moff[q], moff[q], (int)c, r, (int)r, 1, 1, (int)c, r, (int)r));
      hg.cblk.push_back(CBlock{goff[q], n, n, t, t + 1});
    }
    return run_host_gemm(hg, mat, mat, G);
  };
  {
    std::vector<int> every(nQ);
    std::iota(every.begin(), every.end(), 0);
    TTG_TRY(gram(every));
  }
  // a sector whose Gram matrix overflowed (entries of A above ~1e154) or that
  // holds a NaN has no meaningful eigenpairs: fail before the eigensolver
  {
    int hbad = 0;
    hipLaunchKernelGGL(k_svd_finite, dim3(nQ), dim3(256), 0, s, nQ, d_nq, d_goff, G, bad);
    const D2HPiece pc{&hbad, bad, sizeof(int)};
    TTG_TRY(d2h_wait(&pc, 1));
    TTG_REQUIRE(!hbad, "svd: a sector's Gram matrix is not finite (tensor entries above ~1e154, or NaN)");
  }
  // ---- 4. eigensolver
  std::vector<int> big;
  int nsmall = 0;
  for (int q = 0; q < nQ; q++) {
    if (nq[q] > kJacBlockMin) { big.push_back(q); continue; }
    nsmall = std::max(nsmall, nq[q]);
  }
  // The small sectors' one-workgroup Jacobi runs on the side stream, beside
  // the large sectors' solver on the main stream: the two read and write
  // disjoint sector ranges of G, Vev and ev.
  bool forked = false;
  if (nsmall > 0) {
    hipStream_t js = s;
    if (!big.empty()) {
      TTG_TRY(side_fork(&js));
      forked = true;
    }
    hipLaunchKernelGGL(k_jacobi, dim3(nQ), dim3(kJThreads), 0, js, d_nq, d_kq, (int)(cutoff > kLrCutoff), d_goff, G, Vev, ev, d_eoff, 40,
                       kJacBlockMin, kJacFloor);
    TTG_HIP(hipGetLastError());
  }
  // large sectors: the LR step, and without a cutoff (every value is kept) block
  // Jacobi on G, formed again, for those it cannot serve
  int brc = 0;
  std::vector<int> plain;
  if (!big.empty()) {
    const std::string last = ttg_last_error();
    const uint64_t refused = pool_refusals();
    brc = lr_eigen(big, nq, kq, cutoff > 0, plain, goff, eoff, d_eoff, goff[nQ], G, Vev, ev, s);
    if (brc && !(cutoff > 0) && pool_refusals() != refused) {   // no room for its arrays
      plain = big;
      brc = 0;
      set_error(last);
    }
  }
  if (!brc && !plain.empty()) {
    brc = gram(plain);
    if (!brc) brc = block_jacobi(plain, nq, d_goff, d_eoff, G, Vev, ev, s, 40, kJacFloor);
  }
  if (forked) {
    // join before anything else, the error path included: the scratch the
    // side stream reads goes back to the pool when this call returns
    const int jrc = side_join();
    if (brc || jrc) (void)hipStreamSynchronize(s);
    TTG_TRY(jrc);
  }
  TTG_TRY(brc);
  // ---- 5. selection and truncation
  {
    int nmax = 1, kmax = 1;
    for (int q = 0; q < nQ; q++) { nmax = std::max(nmax, nq[q]); kmax = std::max(kmax, kq[q]); }
    hipLaunchKernelGGL(k_svd_select, dim3(nQ, (nmax + 255) / 256), dim3(256), 0, s, d_nq, d_kq, d_eoff, ev,
                       d_soff, svals, ssec, selidx);
    hipLaunchKernelGGL(k_svd_gather_sel, dim3(nQ, std::min(kmax, 64)), dim3(256), 0, s, d_nq, d_kq, d_goff,
                       Vev, d_soff, selidx, d_selo, Esel);
  }
  {
    const int T = (int)soff[nQ];
    if (T > 0)
      hipLaunchKernelGGL(k_svd_rank, dim3((T + 255) / 256), dim3(256), 0, s, T, nQ, d_soff, svals, order,
                         ssorted);
    hipLaunchKernelGGL(k_svd_truncate, dim3(1), dim3(256), 0, s, T, nQ, svals, ssec, order, ssorted,
                       cutoff, K, newdim, tout);
  }
  std::vector<int> nd(nQ);
  double th[2];
  {
    const D2HPiece pc[2] = {{nd.data(), newdim, sizeof(int) * nQ}, {th, tout, sizeof(th)}};
    TTG_TRY(d2h_wait(pc, 2));
  }
  if (trunc_err) *trunc_err = th[0];
  if (kept) *kept = (int64_t)th[1];
  // ---- 6. outputs: index tables (left..., mid) (mid, right...) (mid)
  std::vector<int> midnum(nQ, -1);
  std::vector<int> mq, md;
  int nm = 0;
  for (int q = 0; q < nQ; q++)
    if (nd[q] > 0) {
      midnum[q] = nm++;
      mq.push_back((int)(qcs[q] >> 16) - 32768);
      mq.push_back((int)(qcs[q] & 0xffff) - 32768);
      md.push_back(nd[q]);
    }
  TTG_REQUIRE(nm > 0, "svd: no singular value kept");
  std::vector<std::pair<const TMeta*, int>> lsrc, rsrc;
  for (int j = 0; j < nleft; j++) lsrc.push_back({&m, j});
  for (int j = nleft; j < m.rank; j++) rsrc.push_back({&m, j});
  MetaPtr mid;
  int arrOut = 1, arrIn = 0;
  UploadBatch up;   // the tables of the results, in one launch
  TTG_TRY(meta_shell(1, &arrOut, &nm, mq.data(), md.data(), &mid));
  MetaPtr midIn;
  TTG_TRY(meta_shell(1, &arrIn, &nm, mq.data(), md.data(), &midIn));
  auto concat = [](const std::vector<std::pair<const TMeta*, int>>& a) { return a; };
  std::vector<std::pair<const TMeta*, int>> usrc = concat(lsrc), vsrc{{midIn.get(), 0}};
  usrc.push_back({mid.get(), 0});
  vsrc.insert(vsrc.end(), rsrc.begin(), rsrc.end());
  MetaPtr Um = meta_from_indices(usrc), Vm = meta_from_indices(vsrc);
  TTG_REQUIRE(Um && Vm, "svd: meta allocation failed");
  int nUb = 0, nVb = 0;
  int64_t Utot = 0, Vtot = 0, Stot = 0;
  std::vector<int> ublk0(nQ, 0), vblk0(nQ, 0);
  std::vector<int64_t> sout(nQ + 1, 0);
  for (int q = 0; q < nQ; q++) {
    ublk0[q] = nUb;
    vblk0[q] = nVb;
    sout[q + 1] = sout[q] + nd[q];
    if (nd[q] == 0) continue;
    nUb += qL1[q] - qL0[q];
    nVb += qR1[q] - qR0[q];
    Utot += rows[q] * nd[q];
    Vtot += cols[q] * nd[q];
    Stot += nd[q];
  }
  TTG_TRY(meta_alloc_blocks(*Um, nUb, (size_t)Utot));
  TTG_TRY(meta_alloc_blocks(*Vm, nVb, (size_t)Vtot));
  TTG_TRY(meta_alloc_blocks(*mid, nm, (size_t)Stot));
  {
    std::vector<int> sqi(nm);
    std::iota(sqi.begin(), sqi.end(), 0);
    std::vector<int64_t> soffv(nm + 1, 0);
    for (int q = 0, k = 0; q < nQ; q++)
      if (nd[q] > 0) { soffv[k + 1] = soffv[k] + nd[q]; k++; }
    TTG_TRY(h2d_vec(mid->d_qi, sqi));
    TTG_TRY(h2d_vec(mid->d_off, soffv));
  }
  Pack pko;
  const size_t o_mid = pko.add(midnum), o_ub0 = pko.add(ublk0), o_vb0 = pko.add(vblk0), o_sout = pko.add(sout);
  TTG_TRY(pko.upload(sc, "svd"));
  std::vector<int64_t> umo(nQ + 1, 0), wmo(nQ + 1, 0);
  for (int q = 0; q < nQ; q++) {
    umo[q + 1] = umo[q] + rows[q] * nd[q];
    wmo[q + 1] = wmo[q] + (int64_t)nd[q] * cols[q];
  }
  Pack pkm;
  const size_t o_umo = pkm.add(umo), o_wmo = pkm.add(wmo);
  TTG_TRY(pkm.upload(sc, "svd"));
  int64_t* d_umo = pkm.at<int64_t>(o_umo);
  int64_t* d_wmo = pkm.at<int64_t>(o_wmo);
  TTG_TRY(up.flush());
  int* d_mid = pko.at<int>(o_mid);
  int* d_ub0 = pko.at<int>(o_ub0);
  int* d_vb0 = pko.at<int>(o_vb0);
  int64_t* d_sout = pko.at<int64_t>(o_sout);
  hipLaunchKernelGGL(k_svd_emit, dim3(1), dim3(1024), 0, s, m.view(), nleft, t, nQ, newdim, d_mid,
                     Um->d_qi, Um->d_off, Vm->d_qi, Vm->d_off);
  ttg_tensor U, V, Sv;
  TTG_TRY(tensor_from_meta(Um, false, &U));
  std::unique_ptr<ttg_tensor_s> Uown(U);
  TTG_TRY(tensor_from_meta(Vm, false, &V));
  std::unique_ptr<ttg_tensor_s> Vown(V);
  TTG_TRY(tensor_from_meta(mid, false, &Sv));
  std::unique_ptr<ttg_tensor_s> Sown(Sv);
  hipLaunchKernelGGL(k_svd_svals, dim3(nQ), dim3(64), 0, s, nQ, newdim, d_soff, svals, d_sout, Sv->d_data);
  // absorbed factor: MoveFromLeft  W = E^T A (k x cols), U = E (rows x k)
  //                  MoveFromRight U = A E (rows x k),   W = E^T (k x cols)
  double* Umat = sc.get<double>(umo[nQ]);
  double* Wmat = sc.get<double>(wmo[nQ]);
  TTG_TRY(sc.ok("svd"));
  {
    HostGemm hg;
    for (int q = 0; q < nQ; q++) {
      if (nd[q] == 0) continue;
      const int64_t r = rows[q], c = cols[q], n = nq[q];
      const int k = nd[q];
      if (fromLeft)   // W(i, j) = sum_a E(a, i) A(a, j): A-op E^T (m=i,k=a) = E[a + n i]
        hg.tasks.push_back(gtask(selo[q], moff[q], k, n, (int)r, 1, 1, (int)c, r, (int)r));
      else            // U(i, j) = sum_a A(i, a) E(a, j)
        hg.tasks.push_back(gtask(moff[q], selo[q], (int)r, 1, (int)c, r, 1, k, n, (int)c));
      const int tix = (int)hg.tasks.size() - 1;
      hg.cblk.push_back(fromLeft ? CBlock{wmo[q], k, (int)c, tix, tix + 1}
                                 : CBlock{umo[q], (int)r, k, tix, tix + 1});
    }
    TTG_TRY(fromLeft ? run_host_gemm(hg, Esel, mat, Wmat) : run_host_gemm(hg, mat, Esel, Umat));
  }
  if (fromLeft) {   // U_q = E restricted to k columns: Esel already (n = rows) x k, ld rows
    hipLaunchKernelGGL(k_svd_copy_sel, dim3(nQ, 32), dim3(256), 0, s, nQ, t.rows, newdim, d_selo, Esel,
                       d_umo, Umat);
  } else {
    hipLaunchKernelGGL(k_svd_transpose, dim3(nQ, 64), dim3(256), 0, s, nQ, d_nq, newdim, d_selo, Esel,
                       d_wmo, Wmat);
  }
  hipLaunchKernelGGL(k_svd_scatter, dim3(nQ, 64), dim3(256), 0, s, t, nQ, newdim, d_ub0, d_vb0, Um->d_off,
                     Vm->d_off, Umat, d_umo, Wmat, d_wmo, U->d_data, V->d_data);
  TTG_HIP(hipGetLastError());   // the outputs are written in stream order; the scratch returns to the pool
  *Uout = Uown.release();
  *Vout = Vown.release();
  *Sout = Sown.release();
  return 0;
}
