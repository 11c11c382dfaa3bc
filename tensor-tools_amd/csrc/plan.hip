// plan.hip -- device QN-sector bookkeeping for C = A * B (qtensor.cpp:523-734).
//
// The reference builds, on the host, per mid-QN q the ordered sets of A's
// free-index position tuples (left), B's free tuples (right) and B's
// contracted tuples (mid), creates one result block per (q, right, left) in
// (ascending q, lexicographic right, lexicographic left) order, and runs one
// block GEMM per mid tuple whose A and B blocks both exist.  Here every set
// is a sorted array of 64-bit keys built on the device:
//   (qcode << 32 | tuple)   with qcode order = QN_t_2 order (util/QN.h:100)
//   tuple = mixed-radix number of the positions, first position most
//           significant, so integer order = std::set<uint_vec> order.
// The planning kernels produce the result block list, its packed offsets, the
// task list in the reference loop order and the grouped-GEMM tile list.
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "ttg_device.h"
#include "ttg_internal.h"
#include "ttg_plan.h"

namespace ttg {

__device__ inline uint32_t qcode(int q0, int q1) {
  return ((uint32_t)(q0 + 32768) << 16) | (uint32_t)(q1 + 32768);
}

// Sorted keys and groups of one plan (device scratch, nmax entries each).
// q is a function of the left tuple, so the blocks of A with one left tuple are
// a run of sSA, in ascending mid order: the candidates of every result block
// with that left tuple, in the reference's mid order.
struct PlanSets {
  uint64_t *kUL, *kSA, *kUR, *kSB;   // keys by block (the path of many blocks)
  uint64_t *sUL, *sSA, *sUR, *sSB;   // sorted: (q, left), (left, mid), (q, right), (mid, right)
  int *svSA, *svUR, *svSB;           // block ids in those orders
  uint64_t *uL, *uR;                 // unique (q, left), (q, right)
  int *lsa0, *lcnt, *lpre;           // per left tuple: first entry of sSA, blocks, blocks of all earlier ones (nuL + 1)
  int *rrep;                         // per right tuple: one block of B that has it
  int *qL0, *qL1, *qR0, *qR1;        // per q: ranges of uL and uR
  int64_t *qbase, *qcand;            // per q: first result block, first candidate (nQ + 1)
};

__device__ inline void plan_key_a(const MetaView& A, const PairSpec& ps, int i, uint64_t& ul, uint64_t& sa) {
  const int* qi = A.qi + (size_t)i * A.rank;
  int q0 = 0, q1 = 0;
  uint64_t left = 0, mid = 0;
  for (int j = 0; j < ps.nfa; j++) {
    int p = ps.fa[j], s = qi[p];
    const int* e = A.idx + 3 * (A.idx_off[p] + s);
    int sg = A.arrow[p] == 0 ? 1 : -1;          // Inward +, Outward - (:617-621)
    q0 += sg * e[0];
    q1 += sg * e[1];
    left = left * A.nsec[p] + s;
  }
  for (int t = 0; t < ps.np; t++) {
    int p = ps.pa[t];
    mid = mid * A.nsec[p] + qi[p];
  }
  ul = ((uint64_t)qcode(q0, q1) << 32) | left;
  sa = (left << 32) | mid;
}
__device__ inline void plan_key_b(const MetaView& B, const PairSpec& ps, int i, uint64_t& ur, uint64_t& sb) {
  const int* qi = B.qi + (size_t)i * B.rank;
  int q0 = 0, q1 = 0;
  uint64_t right = 0, mid = 0;
  for (int j = 0; j < ps.nfb; j++) {
    int p = ps.fb[j], s = qi[p];
    const int* e = B.idx + 3 * (B.idx_off[p] + s);
    int sg = B.arrow[p] == 0 ? -1 : 1;          // Inward -, Outward + (:629-633)
    q0 += sg * e[0];
    q1 += sg * e[1];
    right = right * B.nsec[p] + s;
  }
  for (int t = 0; t < ps.np; t++) {
    int p = ps.pb[t];
    mid = mid * B.nsec[p] + qi[p];
  }
  ur = ((uint64_t)qcode(q0, q1) << 32) | right;
  sb = (mid << 32) | right;
}

// ---- groups of the sorted keys (one workgroup) ---------------------------
constexpr int kPlanThreads = 1024;   // most threads of the one-workgroup planning kernels

// rank of the calling thread's set flag among the workgroup's, and the count
__device__ inline int block_rank(bool f, int* lds, int* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const uint64_t m = __ballot(f);
  if (lane == 0) lds[w] = __popcll(m);
  __syncthreads();
  int base = 0, tot = 0;
  for (int k = 0; k < nw; k++) {
    const int c = lds[k];
    base += k < w ? c : 0;
    tot += c;
  }
  __syncthreads();
  *total = tot;
  return base + __popcll(m & ((1ull << lane) - 1ull));
}
// exclusive prefix sum over the workgroup
__device__ inline int64_t block_prefix(int64_t v, int64_t* lds, int64_t* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int64_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) lds[w] = x;
  __syncthreads();
  int64_t base = 0, tot = 0;
  for (int k = 0; k < nw; k++) {
    const int64_t c = lds[k];
    base += k < w ? c : 0;
    tot += c;
  }
  __syncthreads();
  *total = tot;
  return base + x - v;
}

// Unique left and right tuples, q groups, and the first result block and first
// candidate of every group.  The sorted keys are read from, and the unique
// ones written to, LDS or global memory (cuL may be sUL, cuR may be sUR); the
// other results go to w's global arrays and the header to both headers.
__device__ __forceinline__ void plan_groups(const uint64_t* sUL, const uint64_t* sSA, const uint64_t* sUR, const int* svUR,
                                            uint64_t* cuL, uint64_t* cuR, int nA, int nB, const PlanSets& w,
                                            int* lds_i, int64_t* lds_l, PlanHdr* hdr, PlanHdr* host) {
  const int nt = blockDim.x, tid = threadIdx.x;
  int nuL = 0, nuR = 0, nQ = 0;
  int64_t blocks_before = 0;   // blocks of A before the chunk
  for (int base = 0; base < nA; base += nt) {
    const int i = base + tid;
    const uint64_t key = i < nA ? sUL[i] : 0;
    const bool f = i < nA && (i == 0 || key != sUL[i - 1]);
    int tot;
    const int pos = nuL + block_rank(f, lds_i, &tot);
    int cnt = 0, a0 = 0;
    if (f) {
      const uint64_t left = key & 0xffffffffull;
      a0 = lower_bound_u64(sSA, nA, left << 32);
      cnt = lower_bound_u64(sSA, nA, (left + 1) << 32) - a0;
    }
    int64_t all;
    const int64_t pre = block_prefix(cnt, lds_l, &all);
    if (f) {
      cuL[pos] = key;
      w.lsa0[pos] = a0;
      w.lcnt[pos] = cnt;
      w.lpre[pos] = (int)(blocks_before + pre);
    }
    nuL += tot;
    blocks_before += all;
  }
  for (int base = 0; base < nB; base += nt) {
    const int i = base + tid;
    const uint64_t key = i < nB ? sUR[i] : 0;
    const bool f = i < nB && (i == 0 || key != sUR[i - 1]);
    int tot;
    const int pos = nuR + block_rank(f, lds_i, &tot);   // (its barriers: every read of the chunk comes before a write)
    if (f) {
      cuR[pos] = key;
      w.uR[pos] = key;
      w.rrep[pos] = svUR[i];
    }
    nuR += tot;
  }
  if (tid == 0) w.lpre[nuL] = (int)blocks_before;
  __syncthreads();
  // q groups of the left tuples (ascending q; A's mid-QN set, :622-623)
  for (int base = 0; base < nuL; base += nt) {
    const int i = base + tid;
    const bool f = i < nuL && (i == 0 || (cuL[i] >> 32) != (cuL[i - 1] >> 32));
    int tot;
    const int pos = nQ + block_rank(f, lds_i, &tot);
    if (f) w.qL0[pos] = i;
    nQ += tot;
  }
  __syncthreads();
  int64_t nblk = 0, ncand = 0;
  for (int base = 0; base < nQ; base += nt) {
    const int t = base + tid;
    int64_t cnt = 0, cand = 0;
    if (t < nQ) {
      const int l0 = w.qL0[t], l1 = t + 1 < nQ ? w.qL0[t + 1] : nuL;
      const uint64_t qc = cuL[l0] >> 32;
      const int r0 = lower_bound_u64(cuR, nuR, qc << 32), r1 = lower_bound_u64(cuR, nuR, (qc + 1) << 32);
      w.qL1[t] = l1;
      w.qR0[t] = r0;
      w.qR1[t] = r1;
      cnt = (int64_t)(l1 - l0) * (r1 - r0);
      cand = (int64_t)(w.lpre[l1] - w.lpre[l0]) * (r1 - r0);
    }
    int64_t tot, tot2;
    const int64_t pb = block_prefix(cnt, lds_l, &tot), pc = block_prefix(cand, lds_l, &tot2);
    if (t < nQ) {
      w.qbase[t] = nblk + pb;
      w.qcand[t] = ncand + pc;
    }
    nblk += tot;
    ncand += tot2;
  }
  if (tid == 0) {
    w.qbase[nQ] = nblk;
    w.qcand[nQ] = ncand;
    hdr->nQ = host->nQ = nQ;
    hdr->nblocksC = host->nblocksC = nblk;
    hdr->ncand = host->ncand = ncand;
  }
}

// ---- up to kPlanSmall blocks per operand: keys, sorts and groups in one
// workgroup's LDS (one launch and 12 us where the three kernels below take
// 23 us and two launch gaps at a few hundred blocks).  The four key arrays
// are sorted together by bitonic networks of P entries, P the power of two
// above both block counts.
constexpr int kPlanSmall = 1024;
__global__ void __launch_bounds__(kPlanThreads) k_plan_small(MetaView A, MetaView B, PairSpec ps, int P, PlanSets w,
                                                             PlanHdr* hdr, PlanHdr* host) {
  __shared__ uint64_t K[4][kPlanSmall];   // (q, left), (left, mid), (q, right), (mid, right)
  __shared__ int V[3][kPlanSmall];        // block ids of the last three
  __shared__ int lds_i[kPlanThreads / 64];
  __shared__ int64_t lds_l[kPlanThreads / 64];
  const int tid = threadIdx.x, nA = A.nblocks, nB = B.nblocks;
  for (int i = tid; i < P; i += blockDim.x) {
    uint64_t ul = ~0ull, sa = ~0ull, ur = ~0ull, sb = ~0ull;   // above every key: a tuple's half is below 2^32 - 1
    if (i < nA) plan_key_a(A, ps, i, ul, sa);
    if (i < nB) plan_key_b(B, ps, i, ur, sb);
    K[0][i] = ul;
    K[1][i] = sa;
    K[2][i] = ur;
    K[3][i] = sb;
    V[0][i] = V[1][i] = V[2][i] = i;
  }
  const int half = P >> 1, hs = 31 - __builtin_clz(half | 1);   // half = 1 << hs (P >= 2)
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      __syncthreads();
      for (int c = tid; c < 4 * half; c += blockDim.x) {
        const int a = c >> hs, e = c & (half - 1);
        const int i = 2 * e - (e & (j - 1)), l = i + j;
        const uint64_t x = K[a][i], y = K[a][l];
        // equal keys keep block order (a repeated block is found at its first id)
        const bool after = x > y || (x == y && a > 0 && V[a - 1][i] > V[a - 1][l]);
        if (after == ((i & k) == 0)) {
          K[a][i] = y;
          K[a][l] = x;
          if (a > 0) {
            const int t = V[a - 1][i];
            V[a - 1][i] = V[a - 1][l];
            V[a - 1][l] = t;
          }
        }
      }
    }
  __syncthreads();
  for (int i = tid; i < nA; i += blockDim.x) {
    w.sSA[i] = K[1][i];
    w.svSA[i] = V[0][i];
  }
  for (int i = tid; i < nB; i += blockDim.x) {
    w.sSB[i] = K[3][i];
    w.svSB[i] = V[2][i];
  }
  plan_groups(K[0], K[1], K[2], V[1], K[0], K[2], nA, nB, w, lds_i, lds_l, hdr, host);
}

// ---- more blocks: keys, stable rank sort (grid.y selects the array), groups
__global__ void k_plan_keys(MetaView A, MetaView B, PairSpec ps, PlanSets w) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < A.nblocks) plan_key_a(A, ps, i, w.kUL[i], w.kSA[i]);
  if (i < B.nblocks) plan_key_b(B, ps, i, w.kUR[i], w.kSB[i]);
}

struct SortJob {
  const uint64_t* in;
  uint64_t* out;
  int* vout;   // ids of the sorted entries, or null
  int n;
};
struct SortJobs { SortJob j[4]; };

__global__ void __launch_bounds__(256) k_rank_sort(SortJobs jobs) {
  const SortJob& J = jobs.j[blockIdx.y];
  __shared__ uint64_t tile[256];
  const int i = blockIdx.x * 256 + threadIdx.x;
  if ((int)(blockIdx.x * 256) >= J.n) return;
  const uint64_t key = i < J.n ? J.in[i] : 0;
  int rank = 0;
  for (int base = 0; base < J.n; base += 256) {
    __syncthreads();
    if (base + (int)threadIdx.x < J.n) tile[threadIdx.x] = J.in[base + threadIdx.x];
    __syncthreads();
    const int lim = min(256, J.n - base);
    for (int t = 0; t < lim; t++) {
      uint64_t o = tile[t];
      rank += (o < key) || (o == key && base + t < i);
    }
  }
  if (i < J.n) {
    J.out[rank] = key;
    if (J.vout) J.vout[rank] = i;
  }
}

__global__ void __launch_bounds__(kPlanThreads) k_plan_groups(int nA, int nB, PlanSets w, PlanHdr* hdr, PlanHdr* host) {
  __shared__ int lds_i[kPlanThreads / 64];
  __shared__ int64_t lds_l[kPlanThreads / 64];
  plan_groups(w.sUL, w.sSA, w.sUR, w.svUR, w.uL, w.uR, nA, nB, w, lds_i, lds_l, hdr, host);
}

// ---- per result block: tuple, dims, task enumeration ---------------------
// what the scan kernel and the host need of a result block
struct BlkStat {
  int64_t t0;          // first task slot
  int64_t opmax;       // largest operand block (elements) of its tasks
  double flops;
  int M, N, nt, nkt;   // nt tasks, nkt k-tiles
  int ktmax, bad;      // largest K; a task with more than two strides per dimension
  int votes[4];        // tasks with unit stride: A m, A k, B k, B n
};

// fold (extent, stride) components in order: extent-1 ones are dropped,
// contiguous runs merged; n counts the components, the first two are kept.
// 32 bits: an operand block of 2^28 elements or more is refused (opmax).
struct Fold {
  int n = 0;
  unsigned e0 = 1, ce = 0, cs = 0, s0 = 0, s1 = 0;   // ce: extent of the open component (0: none)
  __device__ __forceinline__ void close() {
    const bool open = ce != 0;
    e0 = open && n == 0 ? ce : e0;
    s0 = open && n == 0 ? cs : s0;
    s1 = open && n == 1 ? cs : s1;
    n += open;
    ce = 0;
  }
  __device__ __forceinline__ void add(unsigned ext, unsigned st) {
    if (ext == 1) return;
    if (ce != 0 && st == ce * cs) { ce *= ext; return; }
    close();
    ce = ext;
    cs = st;
  }
};
// the same for K, whose components have a stride in each operand
struct FoldK {
  int n = 0;
  unsigned e0 = 1, ce = 0, ca = 0, cb = 0, a0 = 0, a1 = 0, b0 = 0, b1 = 0;
  __device__ __forceinline__ void close() {
    const bool open = ce != 0, first = open && n == 0, second = open && n == 1;
    e0 = first ? ce : e0;
    a0 = first ? ca : a0;
    b0 = first ? cb : b0;
    a1 = second ? ca : a1;
    b1 = second ? cb : b1;
    n += open;
    ce = 0;
  }
  __device__ __forceinline__ void add(unsigned ext, unsigned sa, unsigned sb) {
    if (ext == 1) return;
    if (ce != 0 && sa == ce * ca && sb == ce * cb) { ce *= ext; return; }
    close();
    ce = ext;
    ca = sa;
    cb = sb;
  }
};
// extent and stride of index p (uniform, runtime) of a block of extents d:
// products of selects, so the array stays in registers
__device__ __forceinline__ unsigned ext_of(const unsigned (&d)[MAXR], int p) {
  unsigned r = 1;
#pragma unroll
  for (int j = 0; j < MAXR; j++) r *= j == p ? d[j] : 1u;
  return r;
}
__device__ __forceinline__ unsigned stride_of(const unsigned (&d)[MAXR], int p) {
  unsigned r = 1;
#pragma unroll
  for (int j = 0; j < MAXR - 1; j++) r *= j < p ? d[j] : 1u;
  return r;
}

__device__ inline int64_t wave_sum_i64(int64_t v) {
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
  return v;
}
__device__ inline int wave_sum_i32(int v) {
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
  return v;
}
__device__ inline double wave_sum_f64(double v) {
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
  return v;
}
__device__ inline int64_t wave_max_i64(int64_t v) {
  for (int d = 32; d >= 1; d >>= 1) {
    const int64_t o = __shfl_xor(v, d);
    v = o > v ? o : v;
  }
  return v;
}

// One wave per result block (q -> right -> left).  Its candidates are A's
// blocks with its left tuple, in ascending mid order (qtensor.cpp:696-722); the
// lanes take 64 at a time and look up the B block (mid, right).  The tasks of
// the block are written one after another from its first candidate slot, each
// at the prefix sum of the matches before it, so the tasks, their k-tile
// offsets and the counts come out of one pass.  The B keys are staged in LDS
// when they fit (stage_b): the lookups are a chain of dependent loads.
constexpr int kPlanStageB = 4096;
__global__ void __launch_bounds__(256) k_plan_blocks(MetaView A, MetaView B, PairSpec ps, PlanSets w, int stage_b,
                                                     const PlanHdr* hdr, BlkStat* stat, int* c_qi, GemmTask* tasks,
                                                     int* tuples, int TK) {
  extern __shared__ uint64_t lds_sb[];
  const int nB = B.nblocks;
  if (stage_b) {
    for (int i = threadIdx.x; i < nB; i += 256) lds_sb[i] = w.sSB[i];
    __syncthreads();
  }
  const int lane = threadIdx.x & 63;
  const int b = (int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6);
  const int nQ = (int)hdr->nQ;
  if (b >= hdr->nblocksC) return;   // the whole wave
  // q group containing b: the last t with qbase[t] <= b
  int t = -1;
  for (int i = 0; i < nQ; i += 64)
    t += __popcll(__ballot(i + lane < nQ && w.qbase[i + lane] <= b));
  const int local = (int)(b - w.qbase[t]);
  const int l0 = w.qL0[t], nL = w.qL1[t] - l0;
  const int ri = local / nL, l = l0 + local % nL, r = w.qR0[t] + ri;
  const int sa0 = w.lsa0[l], cnt = w.lcnt[l];
  const int64_t t0 = w.qcand[t] + (int64_t)ri * (w.lpre[l0 + nL] - w.lpre[l0]) + (w.lpre[l] - w.lpre[l0]);
  const uint32_t right = (uint32_t)w.uR[r];
  const int rep = w.rrep[r];
  unsigned freeA = 0, freeB = 0;   // uniform
  for (int j = 0; j < ps.nfa; j++) freeA |= 1u << ps.fa[j];
  for (int j = 0; j < ps.nfb; j++) freeB |= 1u << ps.fb[j];
  const int rankC = ps.nfa + ps.nfb;
  int64_t N = 1;
  {
    int k = ps.nfa;
#pragma unroll
    for (int j = 0; j < MAXR; j++)
      if ((freeB >> j) & 1) {
        const int s = B.qi[(size_t)rep * B.rank + j];
        N *= B.idx[3 * (B.idx_off[j] + s) + 2];
        if (lane == 0) c_qi[(size_t)b * rankC + k] = s;
        k++;
      }
  }
  int64_t M = 1;
  int nt = 0, kt = 0;   // tasks and k-tiles of the block so far (uniform)
  double fl = 0.0;
  int votes[4] = {0, 0, 0, 0}, ktmax = 0, bad = 0;
  int64_t opmax = 0;
  for (int c0 = 0; c0 < cnt; c0 += 64) {
    const int ca = c0 + lane;
    bool valid = false;
    GemmTask g{};
    int64_t K = 1;
    int ktl = 0, ablk = 0, bblk = 0;
    if (ca < cnt) {
      ablk = w.svSA[sa0 + ca];
      const uint64_t akey = w.sSA[sa0 + ca];
      const bool again = ca > 0 && w.sSA[sa0 + ca - 1] == akey;   // a repeated block counts once
      const uint64_t key = (akey << 32) | right;                  // (mid, right)
      unsigned dA[MAXR];
      int qA[MAXR];
#pragma unroll
      for (int j = 0; j < MAXR; j++) qA[j] = j < A.rank ? A.qi[(size_t)ablk * A.rank + j] : 0;
#pragma unroll
      for (int j = 0; j < MAXR; j++) dA[j] = j < A.rank ? A.idx[3 * (A.idx_off[j] + qA[j]) + 2] : 1;
      M = 1;
#pragma unroll
      for (int j = 0; j < MAXR; j++) M *= (freeA >> j) & 1 ? dA[j] : 1;
      if (ca == 0) {
        int k = 0;
#pragma unroll
        for (int j = 0; j < MAXR; j++)
          if ((freeA >> j) & 1) c_qi[(size_t)b * rankC + k++] = qA[j];
      }
      const uint64_t* sb = stage_b ? lds_sb : w.sSB;
      const int ib = lower_bound_u64(sb, nB, key);
      if (!again && ib < nB && sb[ib] == key) {
        valid = true;
        bblk = w.svSB[ib];
        unsigned dB[MAXR];
#pragma unroll
        for (int j = 0; j < MAXR; j++)
          dB[j] = j < B.rank ? B.idx[3 * (B.idx_off[j] + B.qi[(size_t)bblk * B.rank + j]) + 2] : 1;
        g.a_off = A.off[ablk];
        g.b_off = B.off[bblk];
        Fold fm, fn;
        unsigned sA = 1, sB = 1;   // strides of the stored (unpermuted) blocks
#pragma unroll
        for (int j = 0; j < MAXR; j++) {
          if ((freeA >> j) & 1) fm.add(dA[j], sA);
          if ((freeB >> j) & 1) fn.add(dB[j], sB);
          sA *= dA[j];
          sB *= dB[j];
        }
        fm.close();
        fn.close();
        g.em0 = fm.e0; g.sam0 = fm.s0; g.sam1 = fm.s1;
        g.en0 = fn.e0; g.sbn0 = fn.s0; g.sbn1 = fn.s1;
        // the contraction order forwards, and reversed: taken when it folds
        // better, or when it puts the longer component first (the GEMM walks k
        // in chunks of the first component, so a short first component wastes
        // chunk slots)
        FoldK fk, fr;
        for (int p = 0; p < ps.np; p++) {
          const int z = ps.np - 1 - p;
          const unsigned ext = ext_of(dB, ps.pb[p]);
          K *= ext;
          fk.add(ext, stride_of(dA, ps.pa[p]), stride_of(dB, ps.pb[p]));
          fr.add(ext_of(dB, ps.pb[z]), stride_of(dA, ps.pa[z]), stride_of(dB, ps.pb[z]));
        }
        fk.close();
        fr.close();
        const bool rev = (fk.n > 2 && fr.n <= 2) || (fk.n == 2 && fr.n == 2 && fr.e0 > fk.e0);
        g.ek0 = rev ? fr.e0 : fk.e0;
        g.sak0 = rev ? fr.a0 : fk.a0;
        g.sak1 = rev ? fr.a1 : fk.a1;
        g.sbk0 = rev ? fr.b0 : fk.b0;
        g.sbk1 = rev ? fr.b1 : fk.b1;
        g.K = (int)K;
        g.nk1 = (int)(K / g.ek0);
        if (fm.n > 2 || fn.n > 2 || (rev ? fr.n : fk.n) > 2) bad = 1;
        ktl = g.nk1 * ((g.ek0 + TK - 1) / TK);   // K walk in TK-wide chunks of the first k component (gemm.hip)
        votes[0] += g.sam0 == 1 || M == 1;
        votes[1] += g.sak0 == 1 || K == 1;
        votes[2] += g.sbk0 == 1 || K == 1;
        votes[3] += g.sbn0 == 1 || N == 1;
        ktmax = max(ktmax, (int)K);
        const int64_t oa = M * K, ob = K * N;
        opmax = oa > opmax ? oa : opmax;
        opmax = ob > opmax ? ob : opmax;
        fl += 2.0 * (double)M * (double)N * (double)K;
      }
    }
    // position and k-tile offset: exclusive prefix sums over the lanes
    const uint64_t vm = __ballot(valid);
    const int pos = __popcll(vm & ((1ull << lane) - 1ull));
    int incl = ktl;
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d);
      if (lane >= d) incl += y;
    }
    if (valid) {
      g.kt0 = kt + incl - ktl;
      tasks[t0 + nt + pos] = g;
      int* tu = tuples + 6 * (t0 + nt + pos);
      tu[0] = b; tu[1] = ablk; tu[2] = bblk; tu[3] = (int)M; tu[4] = (int)N; tu[5] = (int)K;
    }
    nt += __popcll(vm);
    kt += __shfl(incl, 63);
  }
  fl = wave_sum_f64(fl);
  for (int v = 0; v < 4; v++) votes[v] = wave_sum_i32(votes[v]);
  for (int d = 32; d >= 1; d >>= 1) {
    ktmax = max(ktmax, __shfl_xor(ktmax, d));
    bad = max(bad, __shfl_xor(bad, d));
  }
  opmax = wave_max_i64(opmax);
  if (lane == 0)   // lane 0 holds the block's first candidate, so its M
    stat[b] = BlkStat{t0, opmax, fl, (int)M, (int)N, nt, kt, ktmax, bad, {votes[0], votes[1], votes[2], votes[3]}};
}

// ---- scan over the result blocks (one workgroup) --------------------------
// Packed offsets and the block table, on the device and in pinned host memory
// (hcb, when the table is read back that way), the result's index table, and
// the totals.  The per-shape totals of the tile choice are a wave's each.
__global__ void __launch_bounds__(kPlanThreads) k_plan_scan(MetaView A, MetaView B, PairSpec ps, const BlkStat* stat,
                                                            int TK, int64_t* c_off, int* c_idx, CBlock* cblk,
                                                            CBlock* hcb, PlanHdr* hdr, PlanHdr* host) {
  __shared__ int64_t lds[kPlanThreads / 64];
  __shared__ PlanHdr H;
  const int n = (int)hdr->nblocksC, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  for (int k = tid; k < (int)(sizeof(PlanHdr) / 8); k += blockDim.x) ((int64_t*)&H)[k] = 0;
  __syncthreads();
  if (tid == 0) {
    H.nQ = hdr->nQ;
    H.nblocksC = n;
    H.ncand = hdr->ncand;
  }
  int64_t total = 0, nt = 0, opmax = 0;
  int vote[4] = {0, 0, 0, 0}, nkt = 0, nmax = 0, ktmax = 0, bad = 0;
  double fl = 0.0;
  for (int base = 0; base < n; base += blockDim.x) {
    const int i = base + tid;
    BlkStat s{};
    if (i < n) s = stat[i];
    int64_t tot;
    const int64_t off = total + block_prefix((int64_t)s.M * s.N, lds, &tot);
    if (i < n) {
      const CBlock cb{off, s.M, s.N, (int)s.t0, (int)(s.t0 + s.nt), s.nkt, 0};
      c_off[i] = off;
      cblk[i] = cb;
      if (hcb) hcb[i] = cb;
      nt += s.nt;
      fl += s.flops;
      nkt = max(nkt, s.nkt);
      if (s.nt) nmax = max(nmax, s.N);
      ktmax = max(ktmax, s.ktmax);
      opmax = s.opmax > opmax ? s.opmax : opmax;
      bad |= s.bad;
      for (int v = 0; v < 4; v++) vote[v] += s.votes[v];
    }
    total += tot;
  }
  // the workgroup's totals: a wave's by shuffles, the waves' by LDS atomics
  // (integers and maxima; the FLOP count is a sum of whole numbers)
  nt = wave_sum_i64(nt);
  fl = wave_sum_f64(fl);
  opmax = wave_max_i64(opmax);
  for (int v = 0; v < 4; v++) vote[v] = wave_sum_i32(vote[v]);
  for (int d = 32; d >= 1; d >>= 1) {
    nkt = max(nkt, __shfl_xor(nkt, d));
    nmax = max(nmax, __shfl_xor(nmax, d));
    ktmax = max(ktmax, __shfl_xor(ktmax, d));
    bad |= __shfl_xor(bad, d);
  }
  typedef unsigned long long u64;
  if (lane == 0) {
    atomicAdd((u64*)&H.ntasks, (u64)nt);
    atomicAdd(&H.flops, fl);
    atomicMax((u64*)&H.kmax, (u64)((int64_t)nkt * TK));
    atomicMax((u64*)&H.nmax, (u64)nmax);
    atomicMax((u64*)&H.ktmax, (u64)ktmax);
    atomicMax((u64*)&H.opmax, (u64)opmax);
    for (int v = 0; v < 4; v++) atomicAdd((u64*)&H.votes[v], (u64)vote[v]);
    if (bad) atomicAdd((u64*)&H.err, 1ull);
  }
  // tile-choice totals: wave w takes shapes w, w + nw, ...
  for (int c = wave; c < TILE_NCFG; c += nw) {
    const int TM = cfg_tm(c), TN = cfg_tn(c);
    int64_t tiles = 0;
    double padded = 0.0;
    for (int i = lane; i < n; i += 64) {
      const int tm = (stat[i].M + TM - 1) / TM, tn = (stat[i].N + TN - 1) / TN;
      tiles += (int64_t)tm * tn;
      padded += (double)(tm * TM) * (double)(tn * TN) * ((double)stat[i].nkt * TK);
    }
    tiles = wave_sum_i64(tiles);
    padded = wave_sum_f64(padded);
    if (lane == 0) {
      H.tiles[c] = tiles;
      H.padded[c] = padded;
    }
  }
  // the result's sectors: A's free indices, then B's
  {
    int o = 0;
    for (int j = 0; j < ps.nfa + ps.nfb; j++) {
      const MetaView& S = j < ps.nfa ? A : B;
      const int p = j < ps.nfa ? ps.fa[j] : ps.fb[j - ps.nfa], len = 3 * S.nsec[p];
      for (int e = tid; e < len; e += blockDim.x) c_idx[o + e] = S.idx[3 * S.idx_off[p] + e];
      o += len;
    }
  }
  if (tid == 0) {
    c_off[n] = total;
    H.totalC = total;
  }
  __syncthreads();
  for (int k = tid; k < (int)(sizeof(PlanHdr) / 8); k += blockDim.x) ((int64_t*)host)[k] = ((const int64_t*)&H)[k];
}

}  // namespace ttg

ttg_plan_s::~ttg_plan_s() {
  ttg::dfree(d_tasks);
  ttg::dfree(d_cblk);
  ttg::dfree(d_tiles);   // d_groups lies in the same allocation
  ttg::dfree(d_part);
  ttg::dfree(d_tuples);
}

namespace ttg {

// Tile-shape autotuner (analytic).  For tile shape c a workgroup's k-tile
// costs, per wave (one wave per SIMD):
//   mfma  = fragments x MFMA cycles per k-tile (FP64 f64 16x16x4: 64 cycles,
//           4 per 16 k; FP32 f32 16x16x4: 32; split-BF16: three 16-cycle
//           16x16x32 per 32 k),
//   issue = 4 cycles x the staging / address / LDS instructions of the tile's
//           load slots (about 6 per FP64/FP32 element, 8 per split-BF16
//           element including the hi/lo split) plus fragment loads and loop,
//   lat   = global-load latency (kLatency) shared by the occ workgroups a CU
//           keeps resident (occupancy of the actual kernel instantiation).
// A CU retires one workgroup k-tile per max(mfma, issue, lat / occ) cycles;
// each work item adds its first load and its epilogue.  The launch takes
// max(total work over the CUs, the longest item after split-K run at the
// single-workgroup rate max(mfma, issue, lat)).
// Split-K (build_tiles) cuts the longest walk into at most kMaxSplit pieces.
constexpr int kMinPiece = 8;   // fewest k-tiles one split piece owns
constexpr double kLatency = 2000.0;

static int choose_cfg(const PlanHdr& h, int prec, int ncu, bool am, bool bk) {
  const int TK = tk_of(prec);
  int best = 0;
  double bestc = 1e300;
  for (int c = 0; c < TILE_NCFG; c++) {
    const double TM = cfg_tm(c), TN = cfg_tn(c);
    const double wm = TN == 16 ? 4 : 2, wn = 4 / wm;
    const double fm = TM / (16 * wm), fn = TN / (16 * wn);
    double mfma, issue;
    if (prec == TTG_BF16X3) {
      mfma = fm * fn * 3 * 16;
      const double slots = std::ceil(TM * TK / 8 / 256.0) + std::ceil(TN * TK / 8 / 256.0);
      issue = 4.0 * (slots * 8 * 8 + 4 * (fm + fn) + 24);
    } else {
      mfma = fm * fn * (TK / 4) * (prec == TTG_FP64 ? 64.0 : 32.0);
      const double slots = (TM + TN) * TK / 256.0;
      issue = 4.0 * (6 * slots + 2 * (fm + fn) + 24);
    }
    const double occ = gemm_occupancy(prec, c, am, bk);
    const double per_ktile = std::max(std::max(mfma, issue), kLatency / occ);
    const double single = std::max(std::max(mfma, issue), kLatency);
    const double ktiles = h.padded[c] / (TM * TN * (double)TK);
    const double item = kLatency + TM * TN / 256.0 * 16.0;   // first load + epilogue stores
    const double work = (ktiles * per_ktile + (double)h.tiles[c] * item / occ) / ncu;
    const double kwalk = (double)h.kmax / TK;
    const double longest = std::max(kwalk / kMaxSplit, std::min(kwalk, (double)kMinPiece));
    const double critical = longest * single + item;
    const double cost = std::max(work, critical);
    if (cost < bestc) {
      bestc = cost;
      best = c;
    }
  }
  return best;
}

// Work list of a plan.  Every output block is cut into TM x TN tiles; a tile
// whose k walk is longer than `piece` k-tiles is split into S <= kMaxSplit
// consecutive k ranges, each written to its own partial slot and summed in
// slot order by the reduction pass (deterministic).  `piece` is the whole
// walk over 6 x the CU count, so the longest item is short against the
// launch while the partial tiles (written, then read by the reduction) stay
// few: the m=2048 operator's FP64 stage 3 takes 77 us, 80-85 us at 4 x and
// 78-79 us at 8 x and 12 x; the m=8192 operator is unchanged within 3%.
int build_tiles(ttg_plan_s& p, const std::vector<CBlock>& cb) {
  const int TM = cfg_tm(p.cfg), TN = cfg_tn(p.cfg);
  const int64_t G = 3 * (int64_t)rt().num_cu;
  int64_t work = 0;
  for (const CBlock& b : cb)
    work += (int64_t)((b.M + TM - 1) / TM) * ((b.N + TN - 1) / TN) * std::max(b.nkt, 1);
  const int64_t piece = std::max<int64_t>(kMinPiece, (work + 2 * G - 1) / (2 * G));
  std::vector<Tile> tiles;
  std::vector<SplitGroup> groups;
  int64_t nslots = 0;
  for (size_t c = 0; c < cb.size(); c++) {
    const CBlock& b = cb[c];
    if (p.cfg == TILE_SKINNY) {   // row chunks, whole walk, no split
      for (int m0 = 0; m0 < b.M; m0 += TM) tiles.push_back(Tile{(int)c, m0, 0, 0, b.nkt, -1});
      continue;
    }
    const int S = (int)std::min<int64_t>(kMaxSplit, std::max<int64_t>(1, (b.nkt + piece - 1) / piece));
    for (int m0 = 0; m0 < b.M; m0 += TM)
      for (int n0 = 0; n0 < b.N; n0 += TN) {
        if (S == 1) {
          tiles.push_back(Tile{(int)c, m0, n0, 0, b.nkt, -1});
          continue;
        }
        groups.push_back(SplitGroup{(int)c, m0, n0, (int)nslots, S, 0});
        for (int sp = 0; sp < S; sp++)
          tiles.push_back(Tile{(int)c, m0, n0, (int)((int64_t)b.nkt * sp / S),
                               (int)((int64_t)b.nkt * (sp + 1) / S), (int)(nslots + sp)});
        nslots += S;
      }
  }
  TTG_REQUIRE(tiles.size() < (size_t)INT32_MAX && nslots < INT32_MAX, "plan: work list too long");
  // Longest walks first (a counting sort, stable): workgroups are dispatched in
  // list order as others end, so the last ones to start are the short ones.
  // Items of equal walks stay in output-block creation order (q -> right ->
  // left): the tiles of one block share A rows, and consecutive blocks share B
  // blocks, through an XCD's L2.
  if (p.cfg != TILE_SKINNY) {
    int most = 0;
    for (const Tile& t : tiles) most = std::max(most, t.kt1 - t.kt0);
    std::vector<int> at(most + 2, 0);
    for (const Tile& t : tiles) at[most - (t.kt1 - t.kt0) + 1]++;
    for (int k = 1; k <= most + 1; k++) at[k] += at[k - 1];
    std::vector<Tile> order(tiles.size());
    for (const Tile& t : tiles) order[at[most - (t.kt1 - t.kt0)]++] = t;
    tiles.swap(order);
  }
  p.ntiles = (int)tiles.size();
  p.ngroups = (int)groups.size();
  p.nslots = nslots;
  // tiles and reduction groups share one allocation and one upload
  const size_t tbytes = sizeof(Tile) * tiles.size(), goff = (tbytes + 255) & ~size_t(255);
  const size_t gbytes = sizeof(SplitGroup) * groups.size();
  p.d_tiles = (Tile*)dmalloc(goff + std::max<size_t>(gbytes, sizeof(SplitGroup)));
  p.d_groups = p.d_tiles ? (SplitGroup*)((char*)p.d_tiles + goff) : nullptr;
  const size_t acc = p.prec == TTG_FP64 ? sizeof(double) : sizeof(float);
  p.d_part = nslots ? dmalloc((size_t)nslots * TM * TN * acc) : nullptr;
  TTG_REQUIRE(p.d_tiles && (p.d_part || !nslots), "plan: work list allocation failed");
  const H2DPiece pc[2] = {{tiles.data(), 0, tbytes}, {groups.data(), goff, gbytes}};
  TTG_TRY(h2d_pieces(p.d_tiles, pc, 2));
  return 0;
}

// replace a plan's work list by one for tile shape cfg (an MFMA shape)
int rebuild_tiles(ttg_plan_s& p, int cfg) {
  TTG_REQUIRE(cfg >= 0 && cfg < TILE_ALL, "plan: bad tile shape");
  if ((int)p.hcb.size() != p.nblocksC) {
    p.hcb.resize(p.nblocksC);
    const D2HPiece pc{p.hcb.data(), p.d_cblk, sizeof(CBlock) * p.nblocksC};
    TTG_TRY(d2h_wait(&pc, 1));
  }
  dfree(p.d_tiles); dfree(p.d_part);   // d_groups lies in d_tiles' allocation
  p.d_tiles = nullptr; p.d_groups = nullptr; p.d_part = nullptr;
  p.ngroups = 0;
  p.nslots = 0;
  p.cfg = cfg;
  p.tiles_pending = false;
  return build_tiles(p, p.hcb);
}

// k-tile offsets of every task of a block's k walk, and the block's k-tile
// count, for k-tile depth TK (one thread per output block)
__global__ void __launch_bounds__(256) k_plan_ktiles(int nblocks, CBlock* cblk, GemmTask* tasks, int TK) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblocks) return;
  const CBlock cb = cblk[b];
  int kt = 0;
  for (int t = cb.t0; t < cb.t1; t++) {
    const GemmTask& g = tasks[t];
    tasks[t].kt0 = kt;
    kt += (g.K / g.ek0) * ((g.ek0 + TK - 1) / TK);
  }
  cblk[b].nkt = kt;
}

int plan_clone(const ttg_plan_s& src, int prec, ttg_plan* out) {
  TTG_REQUIRE(prec == TTG_FP64 || prec == TTG_FP32 || prec == TTG_BF16X3, "unknown precision");
  std::unique_ptr<ttg_plan_s> p(new ttg_plan_s());
  p->A = src.A;
  p->B = src.B;
  p->C = src.C;
  p->ps = src.ps;
  p->prec = prec;
  p->nblocksC = src.nblocksC;
  p->ntasks = src.ntasks;
  p->ncand = src.ncand;
  p->flops = src.flops;
  p->cfg = src.cfg;   // packed_in / split_out start false: the new operator sets them
  p->a_mcontig = src.a_mcontig;
  p->b_kcontig = src.b_kcontig;
  const int64_t nt = p->ncand;
  const int64_t nb = std::max<int64_t>(1, p->nblocksC);
  p->d_tasks = dalloc<GemmTask>(nt);
  p->d_cblk = dalloc<CBlock>(nb);
  p->d_tuples = dalloc<int>(6 * nt);
  TTG_REQUIRE(p->d_tasks && p->d_cblk && p->d_tuples, (std::string("plan: ") + ttg_last_error()).c_str());
  hipStream_t s = stream();
  const DevPiece cp[3] = {{p->d_tasks, src.d_tasks, sizeof(GemmTask) * nt},
                          {p->d_cblk, src.d_cblk, sizeof(CBlock) * nb},
                          {p->d_tuples, src.d_tuples, sizeof(int) * 6 * nt}};
  TTG_TRY(dev_copy(cp, 3));
  if (tk_of(prec) != tk_of(src.prec) && p->nblocksC > 0)
    hipLaunchKernelGGL(k_plan_ktiles, dim3((p->nblocksC + 255) / 256), dim3(256), 0, s, p->nblocksC,
                       p->d_cblk, p->d_tasks, tk_of(prec));
  if (tk_of(prec) == tk_of(src.prec) && (int)src.hcb.size() == p->nblocksC) {
    p->hcb = src.hcb;   // the same k-tile counts
  } else {
    p->hcb.resize(p->nblocksC);
    const D2HPiece pc{p->hcb.data(), p->d_cblk, sizeof(CBlock) * (size_t)p->nblocksC};
    TTG_TRY(d2h_wait(&pc, 1));
  }
  TTG_TRY(build_tiles(*p, p->hcb));
  *out = p.release();
  return 0;
}

// pinned host memory that the planning kernels write: two headers (group
// pass, scan pass) and the block table of plans of up to kPlanHostBlocks
// blocks.  Allocated once for the process: plans are built one at a time, and
// every read of it follows a stream sync.
constexpr int kPlanHostBlocks = 8192;
struct PlanHost {
  PlanHdr groups, scan;
  CBlock cb[kPlanHostBlocks];
};
static PlanHost* plan_host() {
  static PlanHost* h = nullptr;
  if (!h && hipHostMalloc((void**)&h, sizeof(PlanHost)) != hipSuccess) {
    (void)hipGetLastError();
    h = nullptr;
  }
  return h;
}

int plan_build(const MetaPtr& A, const MetaPtr& B, int np, const int* pa, const int* pb, int prec,
               int force_cfg, ttg_plan* out, bool defer_tiles) {
  PhaseTimer _phase("plan_build");
  TTG_TRY(ensure_init());
  TTG_REQUIRE(np >= 0 && np <= A->rank && np <= B->rank, "plan: bad pair count");
  PairSpec ps{};
  ps.np = np;
  std::vector<bool> usedA(A->rank, false), usedB(B->rank, false);
  for (int p = 0; p < np; p++) {
    TTG_REQUIRE(pa[p] >= 0 && pa[p] < A->rank && pb[p] >= 0 && pb[p] < B->rank,
                "plan: pair position out of range");
    TTG_REQUIRE(!usedA[pa[p]] && !usedB[pb[p]], "plan: index paired twice");
    usedA[pa[p]] = usedB[pb[p]] = true;
    ps.pa[p] = pa[p];
    ps.pb[p] = pb[p];
    // the pair must be the same index seen from both sides (tag match)
    TTG_REQUIRE(A->nsec[pa[p]] == B->nsec[pb[p]], "plan: paired indices differ in sectors");
    for (int s = 0; s < A->nsec[pa[p]]; s++)
      TTG_REQUIRE(A->q0(pa[p], s) == B->q0(pb[p], s) && A->q1(pa[p], s) == B->q1(pb[p], s) &&
                      A->dim(pa[p], s) == B->dim(pb[p], s),
                  "plan: paired indices differ in sectors");
  }
  for (int j = 0; j < A->rank; j++) if (!usedA[j]) ps.fa[ps.nfa++] = j;
  for (int j = 0; j < B->rank; j++) if (!usedB[j]) ps.fb[ps.nfb++] = j;
  TTG_REQUIRE(ps.nfa + ps.nfb <= MAXR, "plan: result rank exceeds 8");
  auto radix_ok = [](const TMeta& m, const int* pos, int n) {
    double r = 1;
    for (int j = 0; j < n; j++) r *= m.nsec[pos[j]];
    return r < 4294967295.0;
  };
  TTG_REQUIRE(radix_ok(*A, ps.fa, ps.nfa) && radix_ok(*B, ps.fb, ps.nfb) && radix_ok(*A, ps.pa, np),
              "plan: sector-tuple key exceeds 32 bits");

  const int nA = A->nblocks, nB = B->nblocks;
  hipStream_t s = stream();
  // scratch (returned to the pool on every exit path)
  Scratch sc;
  PlanSets w{};
  const int nmax = std::max(1, std::max(nA, nB));
  const bool small = nmax <= kPlanSmall;
  for (uint64_t** k : {&w.sUL, &w.sSA, &w.sUR, &w.sSB, &w.uL, &w.uR}) *k = sc.get<uint64_t>(nmax);
  for (int** v : {&w.svSA, &w.svUR, &w.svSB, &w.lsa0, &w.lcnt, &w.rrep, &w.qL0, &w.qL1, &w.qR0, &w.qR1})
    *v = sc.get<int>(nmax);
  w.lpre = sc.get<int>(nmax + 1);
  w.qbase = sc.get<int64_t>(nmax + 1);
  w.qcand = sc.get<int64_t>(nmax + 1);
  if (!small)
    for (uint64_t** k : {&w.kUL, &w.kSA, &w.kUR, &w.kSB}) *k = sc.get<uint64_t>(nmax);
  PlanHdr* d_hdr = sc.get<PlanHdr>(1);
  TTG_TRY(sc.ok("plan"));
  PlanHost* host = plan_host();
  TTG_REQUIRE(host, "plan: pinned host memory allocation failed");
  // One host wait when every (A, B) block pair could be a result block or a
  // task without much memory: the arrays take that size.  Otherwise the counts
  // are read back first.
  constexpr int64_t kPlanPairs = 4096;
  const bool one_wait = (int64_t)nA * nB <= kPlanPairs;
  int64_t nbcap = std::max<int64_t>(1, (int64_t)nA * nB), ncap = nbcap;

  if (small) {
    int P = 2;
    while (P < nmax) P *= 2;
    hipLaunchKernelGGL(k_plan_small, dim3(1), dim3(std::min(kPlanThreads, std::max(256, P))), 0, s, A->view(), B->view(),
                       ps, P, w, d_hdr, &host->groups);
  } else {
    hipLaunchKernelGGL(k_plan_keys, dim3((nmax + 255) / 256), dim3(256), 0, s, A->view(), B->view(), ps, w);
    SortJobs jobs;
    jobs.j[0] = {w.kUL, w.sUL, nullptr, nA};
    jobs.j[1] = {w.kSA, w.sSA, w.svSA, nA};
    jobs.j[2] = {w.kUR, w.sUR, w.svUR, nB};
    jobs.j[3] = {w.kSB, w.sSB, w.svSB, nB};
    hipLaunchKernelGGL(k_rank_sort, dim3((nmax + 255) / 256, 4), dim3(256), 0, s, jobs);
    hipLaunchKernelGGL(k_plan_groups, dim3(1), dim3(kPlanThreads), 0, s, nA, nB, w, d_hdr, &host->groups);
  }
  if (!one_wait) {
    TTG_HIP(hipStreamSynchronize(s));
    TTG_REQUIRE(host->groups.nblocksC < (1 << 30), "plan: too many result blocks");
    TTG_REQUIRE(host->groups.ncand < (1 << 30), "plan: too many block pairs");
    nbcap = std::max<int64_t>(1, host->groups.nblocksC);
    ncap = std::max<int64_t>(1, host->groups.ncand);
  }

  // result structure (its index table is written by the scan kernel)
  std::vector<std::pair<const TMeta*, int>> cidx;
  for (int j = 0; j < ps.nfa; j++) cidx.push_back({A.get(), ps.fa[j]});
  for (int j = 0; j < ps.nfb; j++) cidx.push_back({B.get(), ps.fb[j]});
  MetaPtr C = meta_from_indices(cidx, false);
  if (!C) return 1;
  TTG_TRY(meta_alloc_blocks(*C, (int)nbcap, 0));
  BlkStat* stat = sc.get<BlkStat>(nbcap);
  TTG_TRY(sc.ok("plan"));
  // the task list is emitted with the counts, into slots by candidate
  std::unique_ptr<ttg_plan_s> p(new ttg_plan_s());
  p->d_tasks = dalloc<GemmTask>(ncap);
  p->d_cblk = dalloc<CBlock>(nbcap);
  p->d_tuples = dalloc<int>(6 * ncap);
  if (!p->d_tasks || !p->d_cblk || !p->d_tuples) {
    set_error(std::string("plan: ") + ttg_last_error());
    return 1;
  }
  const int stage_b = nB <= kPlanStageB;
  hipLaunchKernelGGL(k_plan_blocks, dim3((unsigned)((nbcap + 3) / 4)), dim3(256), stage_b ? sizeof(uint64_t) * nB : 0, s,
                     A->view(), B->view(), ps, w, stage_b, d_hdr, stat, C->d_qi, p->d_tasks, p->d_tuples, tk_of(prec));
  const bool hcb_pinned = nbcap <= kPlanHostBlocks;
  hipLaunchKernelGGL(k_plan_scan, dim3(1), dim3(nbcap <= 256 ? 256 : kPlanThreads), 0, s, A->view(), B->view(), ps, stat,
                     tk_of(prec), C->d_off, C->d_idx, p->d_cblk, hcb_pinned ? host->cb : nullptr, d_hdr, &host->scan);
  TTG_HIP(hipGetLastError());
  TTG_HIP(hipStreamSynchronize(s));
  const PlanHdr* h_hdr = &host->scan;
  const int64_t nblocksC = h_hdr->nblocksC;
  C->nblocks = (int)nblocksC;
  p->ncand = std::max<int64_t>(1, h_hdr->ncand);
  p->hcb.resize(nblocksC);
  if (hcb_pinned) {
    std::copy(host->cb, host->cb + nblocksC, p->hcb.begin());
  } else {
    const D2HPiece pc{p->hcb.data(), p->d_cblk, sizeof(CBlock) * (size_t)nblocksC};
    TTG_TRY(d2h_wait(&pc, 1));
  }
  TTG_REQUIRE(!h_hdr->err, "plan: operand layout needs more than two strides per GEMM dimension");
  C->total = (size_t)h_hdr->totalC;
  // the GEMM's 32-bit byte offsets per block
  TTG_REQUIRE(h_hdr->opmax < (int64_t(1) << 28), "plan: an operand block exceeds 2^28 elements");

  p->A = A;
  p->B = B;
  p->C = C;
  p->ps = ps;
  p->prec = prec;
  p->nblocksC = (int)nblocksC;
  p->ntasks = h_hdr->ntasks;
  p->flops = h_hdr->flops;
  p->a_mcontig = h_hdr->votes[0] >= h_hdr->votes[1];
  p->b_kcontig = h_hdr->votes[2] >= h_hdr->votes[3];
  if (force_cfg < 0) {   // TTG_TILE_CFG=<n> pins every plan's tile shape (tuning runs)
    const char* e = getenv("TTG_TILE_CFG");
    if (e && *e) force_cfg = atoi(e);
  }
  const bool skinny_ok = h_hdr->nmax <= kSkinnyN && h_hdr->ktmax <= kSkinnyK;
  if (force_cfg == TILE_SKINNY && skinny_ok) p->cfg = TILE_SKINNY;
  else if (force_cfg >= 0 && force_cfg < TILE_NCFG) p->cfg = force_cfg;
  else if (force_cfg > TILE_SKINNY && force_cfg < TILE_ALL) p->cfg = force_cfg;
  else p->cfg = skinny_ok ? TILE_SKINNY
                          : choose_cfg(*h_hdr, prec, rt().num_cu, p->a_mcontig, p->b_kcontig);
  if (defer_tiles) p->tiles_pending = true;
  else TTG_TRY(build_tiles(*p, p->hcb));
  *out = p.release();
  return 0;
}

}  // namespace ttg

using namespace ttg;

extern "C" {

int ttg_contract_plan(ttg_tensor A, ttg_tensor B, int npairs, const int* pa, const int* pb, int prec,
                      ttg_plan* out) {
  TTG_REQUIRE(A && B && out, "contract_plan: null argument");
  TTG_REQUIRE(prec == TTG_FP64 || prec == TTG_FP32 || prec == TTG_BF16X3, "unknown precision");
  return plan_build(A->m, B->m, npairs, pa, pb, prec, -1, out);
}

int ttg_plan_info(ttg_plan p, int* nblocks, int64_t* ntasks, double* flops) {
  TTG_REQUIRE(p, "null plan");
  if (nblocks) *nblocks = p->nblocksC;
  if (ntasks) *ntasks = p->ntasks;
  if (flops) *flops = p->flops;
  return 0;
}

int ttg_plan_tasks_download(ttg_plan p, int* tasks6) {
  TTG_REQUIRE(p, "null plan");
  // a block's tasks start at its first candidate's slot: packed here
  std::vector<int> all(6 * (size_t)p->ncand);
  if (p->ntasks)
    TTG_HIP(hipMemcpyAsync(all.data(), p->d_tuples, sizeof(int) * all.size(), hipMemcpyDeviceToHost, stream()));
  TTG_HIP(hipStreamSynchronize(stream()));
  if (p->ntasks)
    for (const CBlock& b : p->hcb)
      tasks6 = std::copy(all.begin() + 6 * (size_t)b.t0, all.begin() + 6 * (size_t)b.t1, tasks6);
  return 0;
}

int ttg_plan_new_output(ttg_plan p, ttg_tensor* C) {
  TTG_REQUIRE(p, "null plan");
  return tensor_from_meta(p->C, false, C);
}

int ttg_contract_exec(ttg_plan p, ttg_tensor A, ttg_tensor B, ttg_tensor C) {
  TTG_REQUIRE(p && A && B && C, "contract_exec: null argument");
  // the plan's task offsets are only valid for the block lists it was built on
  TTG_REQUIRE(same_meta(A->m, p->A) && same_meta(B->m, p->B) && same_meta(C->m, p->C),
              "contract_exec: tensors do not have the block lists the plan was built on");
  if (p->prec == TTG_FP64) {
    TTG_TRY(gemm_launch(*p, A->d_data, B->d_data, C->d_data, true, stream()));
  } else {
    const float *a32, *b32;
    TTG_TRY(tensor_f32(A, &a32));
    TTG_TRY(tensor_f32(B, &b32));
    TTG_TRY(gemm_launch(*p, a32, b32, C->d_data, true, stream()));
  }
  mark_written(C);
  return 0;
}

int ttg_plan_free(ttg_plan p) {
  delete p;
  return 0;
}

int ttg_contract(ttg_tensor A, ttg_tensor B, int npairs, const int* pa, const int* pb, int prec,
                 ttg_tensor* C) {
  PhaseTimer _phase("ttg_contract");
  ttg_plan p = nullptr;
  TTG_TRY(ttg_contract_plan(A, B, npairs, pa, pb, prec, &p));
  int r = ttg_plan_new_output(p, C);
  if (r == 0) r = ttg_contract_exec(p, A, B, *C);
  delete p;
  return r;
}

}  // extern "C"
