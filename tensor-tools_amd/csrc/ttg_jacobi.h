// ttg_jacobi.h -- one cyclic Jacobi sweep over a symmetric matrix of up to
// 64 x 64, held by one workgroup of 8 waves: the inner solver of the sector
// SVD (svd.hip), for small sectors (swept until converged) and for the 64 x 64
// subproblems of the block Jacobi (one sweep each).
//
// The matrix is cut into 8-wide blocks.  A step pairs the blocks (block b with
// b ^ D, D = 1 .. blocks - 1: every pair of blocks meets once), and
//   1. wave w rotates the 16 x 16 tile of pair w alone: 8 rounds of 8
//      disjoint rotations over the pairs across the two blocks (in the first
//      step also the 7 rounds of pairs inside them), accumulating Q_w;
//   2. the tiles off the pairs' diagonal become Q_a^T T Q_b on
//      v_mfma_f64_16x16x4 (upper tiles, mirrored);
//   3. V^T <- Q^T V^T, held in the registers of the other four waves, which
//      do it while step 1 of the next step runs.
// Every pair of indices is rotated once per sweep, as in the round-robin order
// of 63 rounds of 32 rotations, but 49 of the 63 rounds touch one wave's
// 16 x 16 tile (no workgroup barrier), and the rest of the matrix moves
// through LDS 7 times per sweep instead of 63.  What bounds it is the chain of
// a round: the rotation, one cross-lane copy, the exchange of the 2 x 2 blocks.  A
// 64 x 64 subproblem of the block Jacobi, with its load and eigenvalue order, took
// 61.2 us as 63 rounds through LDS and takes 29.3.
//
// Lane layout of v_mfma_f64_16x16x4 (lane l: A[l%16][l/16], B[l/16][l%16],
// result register r: D[l/16 + 4r][l%16]): a tile T held as T[l/16 + 4s][l%16]
// is the A operand of T^T Q, whose result is X = Q_a^T T in the A layout of the
// second product X Q_b, so both products chain in registers; Q enters every
// product as Qt[l%16][l/16 + 4s].
#pragma once
#include "ttg_device.h"
#include "ttg_internal.h"

namespace ttg {

constexpr int kJW = 64;                    // largest matrix
constexpr int kJThreads = 512;             // waves 0-3: rotations and tiles; 4-7: V^T
// LDS row pitches (doubles): rows step 16 banks (S) and 40 banks (Qt), so the
// 2 x 2 blocks of a round and the MFMA operands spread over all banks
constexpr int kJP = 72, kJQ = 20;
constexpr int kJS = kJW * kJP;             // doubles of S
constexpr int kJQt = 16 * kJQ;             // doubles of one pair's Q^T
constexpr int kJLds = kJS + 2 * 4 * kJQt;  // S and two buffers of four Q^T

typedef double jac_v4d __attribute__((ext_vector_type(4)));

// LDS operations of one wave complete in order; this keeps the compiler's
// order between a round's writes and the next round's reads
__device__ __forceinline__ void jac_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Jacobi rotation for a_pq of [[app, apq], [apq, aqq]]: rows/columns
// (p, q) <- (c x_p - s x_q, s x_p + c x_q), t = s/c the smaller root of
// t^2 + 2 theta t - 1 = 0, theta = (aqq - app) / (2 apq).  The angle only has to
// shrink a_pq, so t is computed in single precision (relative error ~1e-7: what
// is left of a_pq is that far below it, and the next sweep rotates it); c and s
// are a rotation to full double precision: c = (1 + t^2)^(-1/2) from the
// single-precision estimate with one third-order step (2^-21 -> 2^-64),
// s = t c.  aqq - app and 2 apq are scaled by a power of two, so any finite input
// is in range; a ratio below 2^-126 rotates nothing.
__device__ __forceinline__ void jac_rotation(double app, double aqq, double apq, double& c, double& s) {
  const double d = aqq - app, b = 2.0 * apq;
  const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(d), fabs(b)));
  const float df = (float)__builtin_amdgcn_ldexp(d, ex), bf = (float)__builtin_amdgcn_ldexp(b, ex);
  const float den = fabsf(df) + __builtin_amdgcn_sqrtf(fmaf(df, df, bf * bf));
  float t = bf * __builtin_amdgcn_rcpf(den);
  t = df < 0.f ? -t : t;
  t = bf == 0.f ? 0.f : t;   // nothing to rotate (0 / 0 when d is zero too)
  const double td = t;
  const double x = fma(td, td, 1.0), y = (double)__builtin_amdgcn_rsqf(fmaf(t, t, 1.f));
  const double e = fma(-x * y, y, 1.0);
  c = fma(y * e, fma(0.375, e, 0.5), y);
  s = td * c;
}

// x^(-1/2) for x > 0 of any size: the hardware estimate (better than 2^-20) of
// the value scaled by a power of four, and two Newton steps
__device__ __forceinline__ double jac_rsqrt(double x) {
  const int ex = __builtin_amdgcn_frexp_exp(x) & ~1;
  const double m = __builtin_amdgcn_ldexp(x, -ex);
  double y = __builtin_amdgcn_rsq(m);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const double e = fma(-m * y, y, 1.0);
    y = fma(0.5 * y, e, y);
  }
  return __builtin_amdgcn_ldexp(y, -(ex >> 1));
}

constexpr double kJacRel = 1e-12;   // an off-diagonal below this of sqrt(a_pp a_qq) is converged

// (compared squared: the callers scale a matrix by a power of two until its largest
// diagonal is about 1.  A Gram matrix has the squares of a tensor's entries, and its own
// squares leave the range of a double when those are below 1e-80 or above 1e77)
__device__ __forceinline__ bool jac_significant(double app, double aqq, double apq, double floor_abs) {
  return apq * apq > (kJacRel * kJacRel) * fabs(app * aqq) && fabs(apq) > floor_abs;
}
// Sweeps without the floor after one in which nothing above it had to rotate, as long as
// something above the relative test does.  In a rank-deficient matrix that is the null space's rounding
// noise, for ever.  In a graded one it is the small indices, which are resolved to their own
// relative accuracy: their singular values were off by up to 1e-3 of themselves when the
// iteration stopped at the floor, by 1e-5 to 1e-12 after one sweep more, and no more than by the
// Gram matrix's rounding after two (12 to 64 rows, singular values falling by 4 to 20 decades).
constexpr int kJacExtra = 2;

// One wave's 16 x 16 tile in its registers: lane (k1, k2) = (l / 8, l % 8)
// holds the 2 x 2 block of pairs k1 and k2, and in Q^T the rows of pair k1 at
// columns k2 and k2 + 8.
struct JacBlk {
  double x00, x01, x10, x11;   // S at rows p1, q1 and columns p2, q2
  double u0, u1, v0, v1;       // Q^T at row p1 (u) and q1 (v)
};

// One round: lane 9 k = (k, k) holds pair k's own block and computes its
// rotation; every lane takes the rotations of its two pairs from there.
__device__ __forceinline__ void jac_round(JacBlk& t, int k1, int k2, double floor_abs, bool& sig) {
  sig |= k1 == k2 && jac_significant(t.x00, t.x11, t.x01, floor_abs);
  double c, s;
  jac_rotation(t.x00, t.x11, t.x01, c, s);
  const double c1 = __shfl(c, 9 * k1), s1 = __shfl(s, 9 * k1), c2 = __shfl(c, 9 * k2), s2 = __shfl(s, 9 * k2);
  // rows, then columns
  const double y00 = c1 * t.x00 - s1 * t.x10, y01 = c1 * t.x01 - s1 * t.x11;
  const double y10 = s1 * t.x00 + c1 * t.x10, y11 = s1 * t.x01 + c1 * t.x11;
  t.x00 = c2 * y00 - s2 * y01;
  t.x01 = s2 * y00 + c2 * y01;
  t.x10 = c2 * y10 - s2 * y11;
  t.x11 = s2 * y10 + c2 * y11;
  const double u0 = t.u0, u1 = t.u1;
  t.u0 = c1 * u0 - s1 * t.v0;
  t.u1 = c1 * u1 - s1 * t.v1;
  t.v0 = s1 * u0 + c1 * t.v0;
  t.v1 = s1 * u1 + c1 * t.v1;
}

// The 8 rounds across the two blocks: pairs (i, 8 + (i ^ e)) with e in Gray code
// order, so the rows and columns of the second block move by one lane bit
// (D = the bit that changes) from round to round, and those of the first stay.
template <int D>
__device__ __forceinline__ void jac_move(JacBlk& t) {
  t.x01 = lane_xor<D>(t.x01);
  t.x11 = lane_xor<8 * D>(lane_xor<D>(t.x11));
  t.x10 = lane_xor<8 * D>(t.x10);
  t.v0 = lane_xor<8 * D>(t.v0);
  t.v1 = lane_xor<8 * D>(t.v1);
}
constexpr int kJacLastE = 4;   // the last e of 0, 1, 3, 2, 6, 7, 5, 4

// the block of a round whose pairs are rows (P, Q) of S and (p, q) of Q^T
__device__ __forceinline__ void jac_load(JacBlk& t, const double* S, const double* Qt, int k2, int P1, int Q1, int P2,
                                         int Q2, int p1, int q1) {
  t.x00 = S[P1 * kJP + P2];
  t.x01 = S[P1 * kJP + Q2];
  t.x10 = S[Q1 * kJP + P2];
  t.x11 = S[Q1 * kJP + Q2];
  t.u0 = Qt[p1 * kJQ + k2];
  t.u1 = Qt[p1 * kJQ + k2 + 8];
  t.v0 = Qt[q1 * kJQ + k2];
  t.v1 = Qt[q1 * kJQ + k2 + 8];
}
__device__ __forceinline__ void jac_store(const JacBlk& t, double* S, double* Qt, int k2, int P1, int Q1, int P2,
                                          int Q2, int p1, int q1) {
  S[P1 * kJP + P2] = t.x00;
  S[P1 * kJP + Q2] = t.x01;
  S[Q1 * kJP + P2] = t.x10;
  S[Q1 * kJP + Q2] = t.x11;
  Qt[p1 * kJQ + k2] = t.u0;
  Qt[p1 * kJQ + k2 + 8] = t.u1;
  Qt[q1 * kJQ + k2] = t.v0;
  Qt[q1 * kJQ + k2 + 8] = t.v1;
}

// rotations of the tile of blocks at rows o0 and o1: inside the blocks when
// `inside` (through LDS: these 7 rounds come once per sweep), then across them
__device__ __forceinline__ void jac_tile(double* S, double* Qt, int o0, int o1, bool inside, int lane,
                                         double floor_abs, bool& sig) {
  const int k1 = lane >> 3, k2 = lane & 7;
  JacBlk t;
  if (inside) {   // pairs (i, i ^ d), d < 8: four in each block
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int e = lane + 64 * u;
      Qt[(e >> 4) * kJQ + (e & 15)] = (e >> 4) == (e & 15) ? 1.0 : 0.0;
    }
    jac_wave_fence();
#pragma unroll 1
    for (int d = 1; d < 8; d++) {
      const int hb = 31 - __builtin_clz(d), low = (1 << hb) - 1;
      const int p1 = ((k1 & ~low) << 1) | (k1 & low), q1 = p1 ^ d;
      const int p2 = ((k2 & ~low) << 1) | (k2 & low), q2 = p2 ^ d;
      const int b1 = p1 < 8 ? o0 : o1 - 8, b2 = p2 < 8 ? o0 : o1 - 8;
      jac_load(t, S, Qt, k2, b1 + p1, b1 + q1, b2 + p2, b2 + q2, p1, q1);
      jac_wave_fence();
      jac_round(t, k1, k2, floor_abs, sig);
      jac_store(t, S, Qt, k2, b1 + p1, b1 + q1, b2 + p2, b2 + q2, p1, q1);
      jac_wave_fence();
    }
    jac_load(t, S, Qt, k2, o0 + k1, o1 + k1, o0 + k2, o1 + k2, k1, 8 + k1);
  } else {
    jac_load(t, S, Qt, k2, o0 + k1, o1 + k1, o0 + k2, o1 + k2, k1, 8 + k1);
    t.u0 = t.v1 = k1 == k2 ? 1.0 : 0.0;
    t.u1 = t.v0 = 0.0;
  }
  jac_wave_fence();
  jac_round(t, k1, k2, floor_abs, sig);
  jac_move<1>(t);
  jac_round(t, k1, k2, floor_abs, sig);
  jac_move<2>(t);
  jac_round(t, k1, k2, floor_abs, sig);
  jac_move<1>(t);
  jac_round(t, k1, k2, floor_abs, sig);
  jac_move<4>(t);
  jac_round(t, k1, k2, floor_abs, sig);
  jac_move<1>(t);
  jac_round(t, k1, k2, floor_abs, sig);
  jac_move<2>(t);
  jac_round(t, k1, k2, floor_abs, sig);
  jac_move<1>(t);
  jac_round(t, k1, k2, floor_abs, sig);
  jac_store(t, S, Qt, k2, o0 + k1, o1 + (k1 ^ kJacLastE), o0 + k2, o1 + (k2 ^ kJacLastE), k1, 8 + (k1 ^ kJacLastE));
}

// pair k of step D: blocks b and b ^ D, b the k-th block with D's highest bit clear
__host__ __device__ constexpr int jac_b0(int D, int k) {
  int low = 1;
  while (2 * low <= D) low *= 2;
  return ((k & ~(low - 1)) << 1) | (k & (low - 1));
}

// V^T <- diag(Q)^T V^T for the pairs of step D (compile-time, so that the
// blocks of V^T stay in registers)
template <int NPR, int D>
__device__ __forceinline__ void jac_vt(const double* Qb, double (&vt)[2 * NPR][2], int j, int g) {
#pragma unroll
  for (int k = 0; k < NPR; k++) {
    const int b0 = jac_b0(D, k), b1 = b0 ^ D;
    double q[4];
#pragma unroll
    for (int s = 0; s < 4; s++) q[s] = Qb[k * kJQt + j * kJQ + g + 4 * s];
    jac_v4d r = {0.0, 0.0, 0.0, 0.0};
    r = __builtin_amdgcn_mfma_f64_16x16x4f64(q[0], vt[b0][0], r, 0, 0, 0);
    r = __builtin_amdgcn_mfma_f64_16x16x4f64(q[1], vt[b0][1], r, 0, 0, 0);
    r = __builtin_amdgcn_mfma_f64_16x16x4f64(q[2], vt[b1][0], r, 0, 0, 0);
    r = __builtin_amdgcn_mfma_f64_16x16x4f64(q[3], vt[b1][1], r, 0, 0, 0);
    vt[b0][0] = r[0];
    vt[b0][1] = r[1];
    vt[b1][0] = r[2];
    vt[b1][1] = r[3];
  }
}

// V^T = I
template <int NPR>
__device__ __forceinline__ void jac_identity(double (&vt)[2 * NPR][2], int wave, int lane) {
#pragma unroll
  for (int b = 0; b < 2 * NPR; b++)
#pragma unroll
    for (int h = 0; h < 2; h++)
      vt[b][h] = 8 * b + (lane >> 4) + 4 * h == 16 * (wave - 4) + (lane & 15) ? 1.0 : 0.0;
}

// One sweep over 16 NPR indices; *sig_flag = 1 if any rotation was
// significant.  All 512 threads call it; S holds the matrix, complete in LDS;
// Qts two buffers of four Q^T, used in turn (par).  Waves 4 .. 3 + NPR hold
// V^T: vt[b][h] of lane l is V^T[8 b + l/16 + 4 h][16 (wave - 4) + l%16]; their
// last products run past the sweep's last barrier and read buffer par ^ 1 only.
// The steps are a loop for the rotations and tiles (their code stays in the
// instruction cache); only the V^T products are expanded per step.
template <int NPR>
__device__ __forceinline__ void jac_sweep(double* S, double* Qts, double (&vt)[2 * NPR][2], int wave, int lane,
                                          int& par, double floor_abs, int* sig_flag) {
  const int j = lane & 15, g = lane >> 4;
#pragma unroll 1
  for (int D = 1; D < 2 * NPR; D++) {
    double* Qb = Qts + par * 4 * kJQt;
    par ^= 1;
    if (wave < NPR) {
      const int b0 = jac_b0(D, wave);
      bool sig = false;
      jac_tile(S, Qb + wave * kJQt, 8 * b0, 8 * (b0 ^ D), D == 1, lane, floor_abs, sig);
      if (sig) *sig_flag = 1;
    }
    __syncthreads();   // the step's Q are complete and the pairs' own tiles rotated
    if (NPR > 1) {
      // tiles (a, b), a < b, of the pairs, a wave each: 1 for NPR = 2, 6 for NPR = 4
      constexpr int nt = NPR * (NPR - 1) / 2;
      if (const int t = wave; t < nt) {
        const int a = t == 1 ? 2 : t == 3 || t == 5 ? 1 : 0;
        const int b = t == 0 ? 1 : t == 2 || t == 5 ? 2 : 3;
        const int a0 = 8 * jac_b0(D, a), a1 = a0 ^ (8 * D);
        const int b0 = 8 * jac_b0(D, b), b1 = b0 ^ (8 * D);
        const int cj = j < 8 ? b0 + j : b1 + j - 8;
        double T[4], qa[4], qb[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
          const int ri = s < 2 ? a0 + g + 4 * s : a1 + g + 4 * s - 8;
          T[s] = S[ri * kJP + cj];
          qa[s] = Qb[a * kJQt + j * kJQ + g + 4 * s];
          qb[s] = Qb[b * kJQt + j * kJQ + g + 4 * s];
        }
        jac_v4d x = {0.0, 0.0, 0.0, 0.0}, r = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; s++) x = __builtin_amdgcn_mfma_f64_16x16x4f64(T[s], qa[s], x, 0, 0, 0);   // (Qa^T T)^T
#pragma unroll
        for (int s = 0; s < 4; s++) r = __builtin_amdgcn_mfma_f64_16x16x4f64(x[s], qb[s], r, 0, 0, 0);
#pragma unroll
        for (int s = 0; s < 4; s++) {
          const int ri = s < 2 ? a0 + g + 4 * s : a1 + g + 4 * s - 8;
          S[ri * kJP + cj] = r[s];
          S[cj * kJP + ri] = r[s];   // S stays symmetric
        }
      }
    }
    __syncthreads();
    if (wave >= 4 && wave - 4 < NPR) {
      if (D == 1) jac_vt<NPR, 1>(Qb, vt, j, g);
      if constexpr (NPR >= 2) {
        if (D == 2) jac_vt<NPR, 2>(Qb, vt, j, g);
        else if (D == 3) jac_vt<NPR, 3>(Qb, vt, j, g);
      }
      if constexpr (NPR == 4) {
        if (D == 4) jac_vt<NPR, 4>(Qb, vt, j, g);
        else if (D == 5) jac_vt<NPR, 5>(Qb, vt, j, g);
        else if (D == 6) jac_vt<NPR, 6>(Qb, vt, j, g);
        else if (D == 7) jac_vt<NPR, 7>(Qb, vt, j, g);
      }
    }
  }
}

}  // namespace ttg
