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

// One operand of a contraction as the planning kernels read it, made on the host:
// kernel arguments lie in host memory, and a list of positions that is walked in
// them is a chain of slow loads.
struct OperandSpec {
  const int *idx, *qi;
  const int64_t* off;
  int nblocks, rank, nf, np;
  unsigned free;               // bit j: index j is not contracted
  int start[MAXR];             // of index j's sectors in idx
  unsigned wf[MAXR], wm[MAXR]; // place values of index j in the free and in the contracted tuple
  int sign[MAXR];              // of index j's QN in q: +1, -1, or 0 (contracted)
  int pair[MAXR];              // index of pair p
};

// Sorted keys and groups of one plan (device scratch, nmax entries each).
// q is a function of the left tuple, so the blocks of A with one left tuple are
// a run of SA, in ascending mid order: the candidates of every result block
// with that left tuple, in the reference's mid order.  What a result block
// needs of a block, a tuple or a q group is one record: its address depends on the
// record before, and every such step is a load that misses to memory (about
// 0.9 us).
struct PlanRec {          // a block of A or B
  uint64_t key;           // (left, mid) or (mid, right)
  int64_t off;            // of its data
  int id, ext;            // ext: product of the free extents
  unsigned e0, s0, s1;    // the free indices folded into one mixed-radix index (Fold)
  int n, pad[2];
  unsigned dk[MAXR], sk[MAXR];   // extent and stride of the index of pair p
};
struct PlanL {            // a left tuple: first entry of SA, blocks, blocks of all earlier ones
  int sa0, cnt, lpre, pad;
};
struct PlanR {            // a right tuple, one block of B that has it, and its extent
  unsigned right;
  int rep;
  int64_t N;
};
struct PlanQ {            // a q group
  int64_t base, cand;     // first result block, first candidate
  int l0, nL, r0;         // first left tuple, left tuples, first right tuple
  int lpre, wid;          // L[l0].lpre, candidates per right tuple
  int pad[3];
};
struct PlanSets {
  uint64_t *kUL, *kSA, *kUR, *kSB;   // keys by block (the path of many blocks)
  uint64_t *sUL, *sSA, *sUR, *sSB;   // sorted: (q, left), (left, mid), (q, right), (mid, right)
  int *svSA, *svUR, *svSB;           // block ids in those orders
  uint64_t *uL, *uR;                 // unique (q, left), (q, right) (the path of many blocks)
  int* qL0;                          // first left tuple of every q (the path of many blocks)
  PlanRec *SA, *SB;                  // blocks in the orders of sSA and sSB
  PlanL* L;                          // (one more: the total in lpre)
  PlanR* R;
  PlanQ* Q;
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

// keys of block i: (q, free tuple), the free and the contracted tuple; with REC its
// record as well, but for the key
template <bool REC>
__device__ __forceinline__ void plan_block(const OperandSpec& M, int i, uint64_t& uq, unsigned& fr, unsigned& mid,
                                           PlanRec& r, int64_t& ext) {
  int s[MAXR], e0[MAXR], e1[MAXR];
  unsigned d[MAXR];
  if (REC) r.off = M.off[i];
#pragma unroll
  for (int j = 0; j < MAXR; j++) s[j] = j < M.rank ? M.qi[(size_t)i * M.rank + j] : 0;
#pragma unroll
  for (int j = 0; j < MAXR; j++) {
    const int* e = M.idx + (j < M.rank ? 3 * (M.start[j] + s[j]) : 0);
    e0[j] = e1[j] = 0;
    d[j] = 1;
    if (j < M.rank) {
      e0[j] = e[0];
      e1[j] = e[1];
      d[j] = e[2];
    }
  }
  int q0 = 0, q1 = 0;
  fr = mid = 0;
  ext = 1;
#pragma unroll
  for (int j = 0; j < MAXR; j++) {
    q0 += M.sign[j] * e0[j];
    q1 += M.sign[j] * e1[j];
    fr += M.wf[j] * (unsigned)s[j];
    mid += M.wm[j] * (unsigned)s[j];
    ext *= (M.free >> j) & 1 ? d[j] : 1u;
  }
  uq = ((uint64_t)qcode(q0, q1) << 32) | fr;
  if (REC) {
    Fold f;
    unsigned st[MAXR], acc = 1;   // strides of the stored (unpermuted) block
#pragma unroll
    for (int j = 0; j < MAXR; j++) {
      st[j] = acc;
      if ((M.free >> j) & 1) f.add(d[j], acc);
      acc *= d[j];
    }
    f.close();
    r.id = i;
    r.ext = (int)min(ext, (int64_t)0x7fffffff);   // (a block of 2^28 elements is refused, opmax)
    r.e0 = f.e0;
    r.s0 = f.s0;
    r.s1 = f.s1;
    r.n = f.n;
#pragma unroll
    for (int p = 0; p < MAXR; p++) {
      r.dk[p] = 1;
      r.sk[p] = 0;
      if (p < M.np)
#pragma unroll
        for (int j = 0; j < MAXR; j++) {
          r.dk[p] = j == M.pair[p] ? d[j] : r.dk[p];
          r.sk[p] = j == M.pair[p] ? st[j] : r.sk[p];
        }
    }
  }
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

// ---- up to kPlanSmall blocks per operand: keys, sorts and groups in one
// workgroup's LDS, a thread per block.  The four key arrays are sorted in runs of 64, a
// run a wave in its registers (a key's place is the number of keys below it), and
// the runs merged by binary searches in the other runs.  The q groups follow from
// three prefix sums, of values packed into one word.  At 168 blocks the sort took
// 50000 cycles as bitonic networks in LDS and takes 12000, the groups 13000 and 9000; what
// bounds the rest is the keys' two dependent loads (6000 to 9000): 24 us before, 16 now,
// 12.8 at 10 blocks.
constexpr int kPlanSmall = 1024;
struct PlanLds {
  uint64_t K[4][kPlanSmall];         // (q, left), (left, mid), (q, right), (mid, right); ~0 beyond the blocks
  uint64_t S[4][kPlanSmall];         // runs; later the unique keys
  unsigned short V[kPlanSmall], W[4][kPlanSmall];      // block ids of (q, right); of S
  unsigned short place[2][kPlanSmall];                 // of every block in SA and SB
  int64_t N[kPlanSmall];             // free extent of B's blocks
  int lpre[kPlanSmall + 1], qL0[kPlanSmall];
  uint64_t sums[kPlanThreads / 64];
};

// exclusive prefix sum of packed fields over the workgroup, and the total
__device__ __forceinline__ uint64_t plan_scan64(uint64_t v, uint64_t* sums, uint64_t* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  uint64_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  __syncthreads();
  if (lane == 63) sums[w] = x;
  __syncthreads();
  uint64_t base = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < kPlanThreads / 64; k++) {
    const uint64_t c = k < nw ? sums[k] : 0;
    base += k < w ? c : 0;
    tot += c;
  }
  *total = tot;
  return base + x - v;
}

// keys below a (and below b) of an ascending array of P entries, P a power of two
__device__ __forceinline__ void plan_count2(const uint64_t* k, int P, uint64_t a, uint64_t b, int& ca, int& cb) {
  ca = cb = 0;
  for (int s = P >> 1; s > 0; s >>= 1) {
    const uint64_t x = k[ca + s - 1], y = k[cb + s - 1];
    ca += x < a ? s : 0;
    cb += y < b ? s : 0;
  }
  const uint64_t x = k[ca], y = k[cb];
  ca += x < a;
  cb += y < b;
}

__global__ void __launch_bounds__(kPlanThreads) k_plan_small(OperandSpec A, OperandSpec B, PlanSets w, PlanHdr* hdr,
                                                             PlanHdr* host) {
  __shared__ PlanLds L;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
  const int nA = A.nblocks, nB = B.nblocks;
  const int runs = (max(max(nA, nB), 1) + 63) >> 6;   // of 64 keys
  int P = 64;
  while (P < 64 * runs) P *= 2;
  PlanRec ra{}, rb{};                 // of blocks tid of A and B
  {
    uint64_t k[4] = {~0ull, ~0ull, ~0ull, ~0ull};     // above every key: a tuple's half is below 2^32 - 1
    unsigned f, m;
    int64_t ext;
    if (tid < nA) {
      plan_block<true>(A, tid, k[0], f, m, ra, ext);
      k[1] = ra.key = (uint64_t)f << 32 | m;          // (left, mid)
    }
    if (tid < nB) {
      plan_block<true>(B, tid, k[2], f, m, rb, ext);
      k[3] = rb.key = (uint64_t)m << 32 | f;          // (mid, right)
      L.N[tid] = ext;
    }
    for (int i = tid; i < P; i += blockDim.x)
#pragma unroll
      for (int a = 0; a < 4; a++) L.K[a][i] = i == tid ? k[a] : ~0ull;
  }
  __syncthreads();
  for (int t = wave; t < 4 * runs; t += nw) {
    const int a = t & 3, i = (t >> 2) * 64 + lane;
    const uint64_t key = L.K[a][i];
    const unsigned lo = (unsigned)key, hi = (unsigned)(key >> 32);
    // keys of the run below this one; equal keys keep block order, and so does the
    // padding, behind all n keys
    const int n = min(64, max(0, (a < 2 ? nA : nB) - (t >> 2) * 64));
    int c = 0;
    for (int e0 = 0; e0 < n; e0 += 8) {
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int e = e0 + u;
        const uint64_t o = (uint64_t)(unsigned)__builtin_amdgcn_readlane((int)hi, e) << 32 |
                           (unsigned)__builtin_amdgcn_readlane((int)lo, e);
        c += (o < key) | ((o == key) & (e < lane));
      }
    }
    if (lane >= n) c = lane;
    L.S[a][(t >> 2) * 64 + c] = key;
    L.W[a][(t >> 2) * 64 + c] = (unsigned short)i;
  }
  __syncthreads();
  for (int t = wave; t < 4 * runs; t += nw) {
    const int a = t & 3, run = t >> 2;
    const uint64_t key = L.S[a][64 * run + lane];
    int c = lane;
    for (int o = 0; o < runs; o++) {
      if (o == run) continue;
      // keys of run o before this one: below it, or equal in an earlier run
      const uint64_t lim = o < run ? key + 1 : key;   // (~0, padding: it goes last in any order, handled below)
      const uint64_t* r = &L.S[a][64 * o];
      int n = 0;
#pragma unroll
      for (int s = 32; s > 0; s >>= 1) n += r[n + s - 1] < lim ? s : 0;
      n += r[n] < lim;
      c += n;
    }
    if (key != ~0ull) {
      L.K[a][c] = key;
      const unsigned short id = L.W[a][64 * run + lane];
      if (a == 2) L.V[c] = id;
      else if (a) L.place[a >> 1][id] = (unsigned short)c;
    }
  }
  for (int i = tid; i < P; i += blockDim.x) {         // (places of no key)
    if (i >= nA) L.K[0][i] = L.K[1][i] = ~0ull;
    if (i >= nB) L.K[2][i] = L.K[3][i] = ~0ull;
  }
  __syncthreads();
  if (tid < nA) w.SA[L.place[0][tid]] = ra;
  if (tid < nB) {
    w.SB[L.place[1][tid]] = rb;
    w.sSB[L.place[1][tid]] = rb.key;
  }
  // unique left and right tuples, and the blocks of A of every left one
  const uint64_t kl = tid < nA ? L.K[0][tid] : ~0ull, kr = tid < nB ? L.K[2][tid] : ~0ull;
  const bool fl = tid < nA && (tid == 0 || kl != L.K[0][tid - 1]);
  const bool fr = tid < nB && (tid == 0 || kr != L.K[2][tid - 1]);
  int a0 = 0, a1 = 0;
  if (fl) plan_count2(L.K[1], P, (kl & 0xffffffffull) << 32, ((kl & 0xffffffffull) + 1) << 32, a0, a1);
  uint64_t tot;
  const uint64_t pre = plan_scan64((uint64_t)fl | (uint64_t)fr << 16 | (uint64_t)(a1 - a0) << 32, L.sums, &tot);
  const int nuL = (int)(tot & 0xffff), nuR = (int)(tot >> 16 & 0xffff), all = (int)(tot >> 32);
  uint64_t *cuL = L.S[0], *cuR = L.S[2];
  if (fl) {
    const int l = (int)(pre & 0xffff), lp = (int)(pre >> 32);
    cuL[l] = kl;
    L.lpre[l] = lp;
    w.L[l] = PlanL{a0, a1 - a0, lp, 0};
  }
  if (fr) {
    const int r = (int)(pre >> 16 & 0xffff), rep = L.V[tid];
    cuR[r] = kr;
    w.R[r] = PlanR{(unsigned)kr, rep, L.N[rep]};
  }
  if (tid == 0) L.lpre[nuL] = all;
  if (tid >= nuR && tid < P) cuR[tid] = ~0ull;   // (the workgroup has P threads at least)
  __syncthreads();
  // q groups of the left tuples (ascending q; A's mid-QN set, :622-623)
  const bool fq = tid < nuL && (tid == 0 || (cuL[tid] >> 32) != (cuL[tid - 1] >> 32));
  const int qi = (int)plan_scan64(fq, L.sums, &tot), nQ = (int)tot;
  if (fq) L.qL0[qi] = tid;
  __syncthreads();
  PlanQ q{};
  uint64_t mine = 0;
  if (tid < nQ) {
    q.l0 = L.qL0[tid];
    const int l1 = tid + 1 < nQ ? L.qL0[tid + 1] : nuL;
    const uint64_t qc = cuL[q.l0] >> 32;
    q.nL = l1 - q.l0;
    int r1;
    plan_count2(cuR, P, qc << 32, qc == 0xffffffffull ? ~0ull : (qc + 1) << 32, q.r0, r1);
    const int nR = r1 - q.r0;
    q.lpre = L.lpre[q.l0];
    q.wid = L.lpre[l1] - q.lpre;
    mine = (uint64_t)(q.nL * nR) | (uint64_t)(q.wid * nR) << 32;   // both at most nA * nB <= 2^20
  }
  const uint64_t at = plan_scan64(mine, L.sums, &tot);
  if (tid < nQ) {
    q.base = (int64_t)(at & 0xffffffffull);
    q.cand = (int64_t)(at >> 32);
    w.Q[tid] = q;
  }
  if (tid == 0) {
    hdr->nQ = nQ;
    hdr->nblocksC = (int64_t)(tot & 0xffffffffull);
    hdr->ncand = (int64_t)(tot >> 32);
    hdr->done = 0;
    if (host) {
      host->nblocksC = hdr->nblocksC;
      host->ncand = hdr->ncand;
    }
  }
}

// ---- more blocks: keys, stable rank sort (grid.y selects the array), groups
__global__ void k_plan_keys(OperandSpec A, OperandSpec B, PlanSets w) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  PlanRec none;
  unsigned f, m;
  int64_t ext;
  if (i < A.nblocks) {
    plan_block<false>(A, i, w.kUL[i], f, m, none, ext);
    w.kSA[i] = (uint64_t)f << 32 | m;
  }
  if (i < B.nblocks) {
    plan_block<false>(B, i, w.kUR[i], f, m, none, ext);
    w.kSB[i] = (uint64_t)m << 32 | f;
  }
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

// Unique left and right tuples, q groups, and the first result block and first
// candidate of every group, by one workgroup (the path of many blocks).
__global__ void __launch_bounds__(kPlanThreads) k_plan_groups(OperandSpec B, int nA, int nB, PlanSets w,
                                                              PlanHdr* hdr, PlanHdr* host) {
  __shared__ int lds_i[kPlanThreads / 64];
  __shared__ int64_t lds_l[kPlanThreads / 64];
  const uint64_t *sUL = w.sUL, *sSA = w.sSA, *sUR = w.sUR;
  uint64_t *cuL = w.uL, *cuR = w.uR;
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
      w.L[pos] = PlanL{a0, cnt, (int)(blocks_before + pre), 0};
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
      const int rep = w.svUR[i];
      uint64_t uq;
      unsigned f, m;
      PlanRec none;
      int64_t N;
      plan_block<false>(B, rep, uq, f, m, none, N);
      w.R[pos] = PlanR{(unsigned)key, rep, N};
    }
    nuR += tot;
  }
  if (tid == 0) w.L[nuL].lpre = (int)blocks_before;
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
    PlanQ q{};
    if (t < nQ) {
      q.l0 = w.qL0[t];
      const int l1 = t + 1 < nQ ? w.qL0[t + 1] : nuL;
      const uint64_t qc = cuL[q.l0] >> 32;
      q.nL = l1 - q.l0;
      q.r0 = lower_bound_u64(cuR, nuR, qc << 32);
      const int nR = lower_bound_u64(cuR, nuR, (qc + 1) << 32) - q.r0;
      q.lpre = w.L[q.l0].lpre;
      q.wid = w.L[l1].lpre - q.lpre;
      cnt = (int64_t)q.nL * nR;
      cand = (int64_t)q.wid * nR;
    }
    int64_t tot, tot2;
    const int64_t pb = block_prefix(cnt, lds_l, &tot), pc = block_prefix(cand, lds_l, &tot2);
    if (t < nQ) {
      q.base = nblk + pb;
      q.cand = ncand + pc;
      w.Q[t] = q;
    }
    nblk += tot;
    ncand += tot2;
  }
  if (tid == 0) {
    hdr->nQ = nQ;
    hdr->nblocksC = host->nblocksC = nblk;
    hdr->ncand = host->ncand = ncand;
    hdr->done = 0;
  }
}

// the records of the sorted blocks
__global__ void __launch_bounds__(256) k_plan_recs(OperandSpec A, OperandSpec B, PlanSets w) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  auto rec = [&](const OperandSpec& M, int id, uint64_t key) {
    PlanRec r{};
    uint64_t uq;
    unsigned f, m;
    int64_t ext;
    plan_block<true>(M, id, uq, f, m, r, ext);
    r.key = key;
    return r;
  };
  if (i < A.nblocks) w.SA[i] = rec(A, w.svSA[i], w.sSA[i]);
  if (i < B.nblocks) w.SB[i] = rec(B, w.svSB[i], w.sSB[i]);
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
  int left, pad;       // left tuple
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
template <class T>
__device__ __forceinline__ T wave_sum(T v) {
  return wave_all(v, [](T a, T b) { return a + b; });
}
template <class T>
__device__ __forceinline__ T wave_max(T v) {
  return wave_all(v, [](T a, T b) { return a > b ? a : b; });
}

// What the scan and the tile choice need of the result blocks, one workgroup: packed
// offsets and the block table, on the device and in pinned host memory (hcb, when
// the table is read back that way), the result's index table, and the totals.  Writes
// to host memory come last: a barrier would wait for them.
struct ScanLds {
  int64_t sums[kPlanThreads / 64];
  PlanHdr H;
  int M[kPlanThreads], N[kPlanThreads], kt[kPlanThreads];   // of the first chunk of blocks
};
struct ScanOut {
  int64_t* c_off;
  int* c_idx;
  CBlock *cblk, *hcb;
  PlanHdr* host;
  const int* seg[MAXR];   // the result's index table: pieces of the operands' ones
  int len[MAXR];          // (ints)
};
__device__ __forceinline__ void plan_scan(ScanLds& L, const BlkStat* stat, int TK, const ScanOut& out, int64_t nQ, int n,
                                          int64_t ncand) {
  PlanHdr& H = L.H;
  {   // the index table, its loads before its stores
    int v[MAXR], *to = out.c_idx;
#pragma unroll
    for (int j = 0; j < MAXR; j++) v[j] = (int)threadIdx.x < out.len[j] ? out.seg[j][threadIdx.x] : 0;
#pragma unroll
    for (int j = 0; j < MAXR; j++) {
      if ((int)threadIdx.x < out.len[j]) to[threadIdx.x] = v[j];
      for (int e = threadIdx.x + blockDim.x; e < out.len[j]; e += blockDim.x) to[e] = out.seg[j][e];
      to += out.len[j];
    }
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  for (int k = tid; k < (int)(sizeof(PlanHdr) / 8); k += blockDim.x) ((int64_t*)&H)[k] = 0;
  __syncthreads();
  if (tid == 0) {
    H.nQ = nQ;
    H.nblocksC = n;
    H.ncand = ncand;
  }
  int64_t total = 0, nt = 0, opmax = 0;
  int64_t vote[4] = {0, 0, 0, 0};
  int nkt = 0, nmax = 0, ktmax = 0, bad = 0;
  double fl = 0.0;
  CBlock first{};   // of the first chunk, for the host (all of it up to a block a thread)
  for (int base = 0; base < n; base += blockDim.x) {
    const int i = base + tid;
    BlkStat s{};
    if (i < n) s = stat[i];
    int64_t tot;
    const int64_t off = total + block_prefix((int64_t)s.M * s.N, L.sums, &tot);
    if (i < n) {
      const CBlock cb{off, s.M, s.N, (int)s.t0, (int)(s.t0 + s.nt), s.nkt, s.left};
      out.c_off[i] = off;
      out.cblk[i] = cb;
      if (base == 0) first = cb;
      else if (out.hcb) out.hcb[i] = cb;
      nt += s.nt;
      fl += s.flops;
      nkt = max(nkt, s.nkt);
      if (s.nt) nmax = max(nmax, s.N);
      ktmax = max(ktmax, s.ktmax);
      opmax = s.opmax > opmax ? s.opmax : opmax;
      bad |= s.bad;
      for (int v = 0; v < 4; v++) vote[v] += s.votes[v];
    }
    if (base == 0) {
      L.M[tid] = s.M;
      L.N[tid] = s.N;
      L.kt[tid] = s.nkt;
    }
    total += tot;
  }
  __syncthreads();
  // the workgroup's totals: a wave's by lane exchanges, the waves' by LDS atomics
  // (integers and maxima; the FLOP count is a sum of whole numbers)
  nt = wave_sum(nt);
  fl = wave_sum(fl);
  opmax = wave_max(opmax);
  for (int v = 0; v < 4; v++) vote[v] = wave_sum(vote[v]);
  nkt = wave_max(nkt);
  nmax = wave_max(nmax);
  ktmax = wave_max(ktmax);
  bad = wave_max(bad);
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
    auto add = [&](int M, int N, int kt) {
      const int tm = (M + TM - 1) / TM, tn = (N + TN - 1) / TN;
      tiles += (int64_t)tm * tn;
      padded += (double)(tm * TM) * (double)(tn * TN) * ((double)kt * TK);
    };
    for (int i = lane; i < min(n, (int)blockDim.x); i += 64) add(L.M[i], L.N[i], L.kt[i]);
    for (int i = blockDim.x + lane; i < n; i += 64) add(stat[i].M, stat[i].N, stat[i].nkt);
    tiles = wave_sum(tiles);
    padded = wave_sum(padded);
    if (lane == 0) {
      H.tiles[c] = tiles;
      H.padded[c] = padded;
    }
  }
  if (tid == 0) {
    out.c_off[n] = total;
    H.totalC = total;
  }
  __syncthreads();
  for (int k = tid; k < (int)(sizeof(PlanHdr) / 8); k += blockDim.x) ((int64_t*)out.host)[k] = ((const int64_t*)&H)[k];
  if (out.hcb && tid < n) out.hcb[tid] = first;
}

// One wave per result block (q -> right -> left), the workgroups striding over
// them.  A block's candidates are A's blocks with its left tuple, in ascending mid
// order (qtensor.cpp:696-722); the lanes take 64 at a time and look up the B block
// (mid, right).  The tasks of the block are written one after another from its
// first candidate slot, each at the prefix sum of the matches before it, so the
// tasks, their k-tile offsets and the counts come out of one pass.  The B keys are
// staged in LDS when they fit (stage_b): the lookups are a chain of dependent
// loads.  What bounds it is that chain: four loads that miss (q group, tuple, blocks of A
// and of B), 20000 cycles with the launch, the records written, 15000 for the scan.  The
// workgroup that finishes last goes on with the scan, for `fuse` blocks or fewer (16.9 us at
// 170 blocks for both; 15.8 and 9.1 as two kernels, and the gap between them): kPlanFuse
// of them when the host has read the count, and whatever a plan of one wait comes
// to (kPlanPairs), as the host does not know it.  A longer list goes to k_plan_scan's
// 1024 threads.
constexpr int kPlanStageB = 4096;
constexpr int kPlanGrid = 512;      // most workgroups of k_plan_blocks
constexpr int64_t kPlanFuse = 2048;
__global__ void __launch_bounds__(256) k_plan_blocks(OperandSpec A, OperandSpec B, PlanSets w, int stage_b,
                                                     PlanHdr* hdr, BlkStat* stat, int* c_qi, GemmTask* tasks,
                                                     int* tuples, int TK, int64_t fuse, ScanOut out) {
  extern __shared__ uint64_t lds_sb[];
  __shared__ ScanLds L;
  __shared__ bool last;
  const int nB = B.nblocks, lane = threadIdx.x & 63;
  const int nQ = (int)hdr->nQ;
  const int64_t nblk = hdr->nblocksC;
  const int groups = (int)max((int64_t)1, min((nblk + 3) / 4, (int64_t)gridDim.x));   // workgroups with work
  if ((int)blockIdx.x >= groups) return;
  if (stage_b) {
    for (int i = threadIdx.x; i < nB; i += 256) lds_sb[i] = w.sSB[i];
    __syncthreads();
  }
  const int rankC = A.nf + B.nf, np = A.np;
  // lane k: the result's index k as an index of A or B
  int from = 0;
  {
    int k = 0;
#pragma unroll
    for (int j = 0; j < MAXR; j++)
      if ((A.free >> j) & 1) from = lane == k++ ? j : from;
#pragma unroll
    for (int j = 0; j < MAXR; j++)
      if ((B.free >> j) & 1) from = lane == k++ ? j : from;
  }
  const int wave0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  for (int64_t bb = wave0; bb < nblk; bb += 4 * (int64_t)groups) {
    const int b = (int)bb;
    // q group containing b: the last with base <= b
    PlanQ q{};
    for (int i = 0; i < nQ; i += 64) {
      PlanQ mine{};
      if (i + lane < nQ) mine = w.Q[i + lane];
      const uint64_t m = __ballot(i + lane < nQ && mine.base <= b);
      if (!m) break;
      const int t = __popcll(m) - 1;
      q.base = (int64_t)__builtin_amdgcn_readlane((int)mine.base, t);   // at most b
      q.cand = (int64_t)(unsigned)__builtin_amdgcn_readlane((int)mine.cand, t) |
               (int64_t)__builtin_amdgcn_readlane((int)(mine.cand >> 32), t) << 32;
      q.l0 = __builtin_amdgcn_readlane(mine.l0, t);
      q.nL = __builtin_amdgcn_readlane(mine.nL, t);
      q.r0 = __builtin_amdgcn_readlane(mine.r0, t);
      q.lpre = __builtin_amdgcn_readlane(mine.lpre, t);
      q.wid = __builtin_amdgcn_readlane(mine.wid, t);
      if (t < 63) break;
    }
    const int local = (int)(b - q.base), ri = local / q.nL;
    const PlanL l = w.L[q.l0 + local % q.nL];
    const PlanR r = w.R[q.r0 + ri];
    const int64_t t0 = q.cand + (int64_t)ri * q.wid + (l.lpre - q.lpre);
    const int sa0 = l.sa0, cnt = l.cnt;
    const uint32_t right = r.right;
    const int64_t N = r.N;
    int64_t M = 1;
    int ablk0 = 0;        // lane 0: the first candidate's block of A
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
        const PlanRec a = w.SA[sa0 + ca];
        const uint64_t akey = a.key;
        const bool again = ca > 0 && w.SA[sa0 + ca - 1].key == akey;   // a repeated block counts once
        const uint64_t key = (akey << 32) | right;                     // (mid, right)
        ablk = a.id;
        if (c0 == 0) ablk0 = ablk;
        M = a.ext;
        const uint64_t* sb = stage_b ? lds_sb : w.sSB;
        const int ib = lower_bound_u64(sb, nB, key);
        if (!again && ib < nB && sb[ib] == key) {
          valid = true;
          const PlanRec o = w.SB[ib];
          bblk = o.id;
          g.a_off = a.off;
          g.b_off = o.off;
          g.em0 = a.e0; g.sam0 = a.s0; g.sam1 = a.s1;
          g.en0 = o.e0; g.sbn0 = o.s0; g.sbn1 = o.s1;
          // the contraction order forwards, and reversed: taken when it folds
          // better, or when it puts the longer component first (the GEMM walks k
          // in chunks of the first component, so a short first component wastes
          // chunk slots)
          FoldK fk, fr;
#pragma unroll
          for (int p = 0; p < MAXR; p++)
            if (p < np) {
              K *= o.dk[p];
              fk.add(o.dk[p], a.sk[p], o.sk[p]);
            }
#pragma unroll
          for (int p = MAXR - 1; p >= 0; p--)
            if (p < np) fr.add(o.dk[p], a.sk[p], o.sk[p]);
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
          if (a.n > 2 || o.n > 2 || (rev ? fr.n : fk.n) > 2) bad = 1;
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
    // the block's tuple (loads that nothing waits for)
    if (lane < rankC) {
      const int ab = __builtin_amdgcn_readfirstlane(ablk0);
      c_qi[(size_t)b * rankC + lane] =
          lane < A.nf ? A.qi[(size_t)ab * A.rank + from] : B.qi[(size_t)r.rep * B.rank + from];
    }
    fl = wave_sum(fl);
    for (int v = 0; v < 4; v++) votes[v] = wave_sum(votes[v]);
    ktmax = wave_max(ktmax);
    bad = wave_max(bad);
    opmax = wave_max(opmax);
    if (lane == 0)   // lane 0 holds the block's first candidate, so its M
      stat[b] = BlkStat{t0, opmax, fl, (int)M, (int)N, nt, kt, ktmax, bad, {votes[0], votes[1], votes[2], votes[3]},
                        q.l0 + local % q.nL, 0};
  }
  if (nblk > fuse) return;   // k_plan_scan follows
  // Every wave waits for its own stores: a barrier orders them within the
  // workgroup only, and what thread 0 waits for before the counter are its own wave's
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(&hdr->done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)groups - 1;
  __syncthreads();
  if (last)
    plan_scan(L, stat, TK, out, nQ, (int)nblk, hdr->ncand);
}

__global__ void __launch_bounds__(kPlanThreads) k_plan_scan(const BlkStat* stat, int TK, const PlanHdr* hdr,
                                                            ScanOut out) {
  __shared__ ScanLds L;
  plan_scan(L, stat, TK, out, hdr->nQ, (int)hdr->nblocksC, hdr->ncand);
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
// (6 per FP64/FP32 element is what 8-byte loads took; with the kernel's 16-byte slots it
// takes fewer, so the model sees the wide shapes a little dearer than they are.  The shapes
// 96x64 and 64x96 are not in it: operators time them, tune_stage.)
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
  // The vector kernel's items: row chunks, whole walk, no split.  The result blocks of
  // one left tuple read the same rows of the same blocks of A (2.8 times each in
  // the MPO stage of an H_eff).  An A larger than the Infinity Cache is read from
  // memory every time, so there their items for a chunk of rows stand together:
  // they run at one time and, the list being dealt to the XCDs in runs, behind one L2
  // (1.76 GB at m = 8192: 1325 to 1111 us).  A smaller A comes from that cache
  // in any order (96 MB: 71.0 and 71.2 us; as FP32, 41.7 and 44.4).
  constexpr size_t kInfinityCache = size_t(256) << 20;
  p.by_rows = p.cfg == TILE_SKINNY && p.A &&
              p.A->total * (p.prec == TTG_FP64 ? sizeof(double) : sizeof(float)) > kInfinityCache;
  if (p.by_rows) {
    std::vector<int> order(cb.size());
    for (size_t c = 0; c < cb.size(); c++) order[c] = (int)c;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return cb[x].left < cb[y].left; });
    for (size_t i = 0, e; i < order.size(); i = e) {
      int most = 0;
      for (e = i; e < order.size() && cb[order[e]].left == cb[order[i]].left; e++) most = std::max(most, cb[order[e]].M);
      for (int m0 = 0; m0 < most; m0 += TM)
        for (size_t k = i; k < e; k++)
          if (m0 < cb[order[k]].M) tiles.push_back(Tile{order[k], m0, 0, 0, cb[order[k]].nkt, -1});
    }
  }
  for (size_t c = 0; c < cb.size() && !p.by_rows; c++) {
    const CBlock& b = cb[c];
    if (p.cfg == TILE_SKINNY) {
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

// A's QNs count Inward + and Outward - (qtensor.cpp:617-621), B's the other way
// round (:629-633): `inward` is the sign of an Inward index
static OperandSpec operand_spec(const TMeta& m, int nf, const int* f, int np, const int* pair, int inward) {
  OperandSpec o{};
  o.idx = m.d_idx;
  o.qi = m.d_qi;
  o.off = m.d_off;
  o.nblocks = m.nblocks;
  o.rank = m.rank;
  o.nf = nf;
  o.np = np;
  for (int j = 0; j < m.rank; j++) o.start[j] = m.idx_off[j];
  unsigned w = 1;
  for (int k = nf - 1; k >= 0; k--) {   // the first index is the most significant
    o.free |= 1u << f[k];
    o.sign[f[k]] = m.arrow[f[k]] == 0 ? inward : -inward;
    o.wf[f[k]] = w;
    w *= (unsigned)m.nsec[f[k]];
  }
  w = 1;
  for (int k = np - 1; k >= 0; k--) {
    o.pair[k] = pair[k];
    o.wm[pair[k]] = w;
    w *= (unsigned)m.nsec[pair[k]];
  }
  return o;
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
  w.sSB = sc.get<uint64_t>(nmax);
  w.SA = sc.get<PlanRec>(nmax);
  w.SB = sc.get<PlanRec>(nmax);
  w.L = sc.get<PlanL>(nmax + 1);
  w.R = sc.get<PlanR>(nmax);
  w.Q = sc.get<PlanQ>(nmax);
  if (!small) {
    for (uint64_t** k : {&w.kUL, &w.kSA, &w.kUR, &w.kSB, &w.sUL, &w.sSA, &w.sUR, &w.uL, &w.uR}) *k = sc.get<uint64_t>(nmax);
    for (int** v : {&w.svSA, &w.svUR, &w.svSB, &w.qL0}) *v = sc.get<int>(nmax);
  }
  const OperandSpec va = operand_spec(*A, ps.nfa, ps.fa, np, ps.pa, 1), vb = operand_spec(*B, ps.nfb, ps.fb, np, ps.pb, -1);
  PlanHdr* d_hdr = sc.get<PlanHdr>(1);
  TTG_TRY(sc.ok("plan"));
  PlanHost* host = plan_host();
  TTG_REQUIRE(host, "plan: pinned host memory allocation failed");
  // One host wait when every (A, B) block pair could be a result block or a
  // task without much memory: the arrays take that size.  Otherwise the counts
  // are read back first.
  constexpr int64_t kPlanPairs = 8192;
  const bool one_wait = (int64_t)nA * nB <= kPlanPairs;
  int64_t nbcap = std::max<int64_t>(1, (int64_t)nA * nB), ncap = nbcap;

  if (small) {
    // a thread per block, and a wave per run to sort
    const int waves = std::min(kPlanThreads / 64, 4 * ((nmax + 63) / 64));
    hipLaunchKernelGGL(k_plan_small, dim3(1), dim3(64 * waves), 0, s, va, vb, w, d_hdr,
                       one_wait ? nullptr : &host->groups);
  } else {
    hipLaunchKernelGGL(k_plan_keys, dim3((nmax + 255) / 256), dim3(256), 0, s, va, vb, w);
    SortJobs jobs;
    jobs.j[0] = {w.kUL, w.sUL, nullptr, nA};
    jobs.j[1] = {w.kSA, w.sSA, w.svSA, nA};
    jobs.j[2] = {w.kUR, w.sUR, w.svUR, nB};
    jobs.j[3] = {w.kSB, w.sSB, w.svSB, nB};
    hipLaunchKernelGGL(k_rank_sort, dim3((nmax + 255) / 256, 4), dim3(256), 0, s, jobs);
    hipLaunchKernelGGL(k_plan_groups, dim3(1), dim3(kPlanThreads), 0, s, vb, nA, nB, w, d_hdr, &host->groups);
    hipLaunchKernelGGL(k_plan_recs, dim3((nmax + 255) / 256), dim3(256), 0, s, va, vb, w);
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
  const bool hcb_pinned = nbcap <= kPlanHostBlocks;
  ScanOut so{C->d_off, C->d_idx, p->d_cblk, hcb_pinned ? host->cb : nullptr, &host->scan, {}, {}};
  for (int j = 0; j < ps.nfa + ps.nfb; j++) {
    const TMeta& m = j < ps.nfa ? *A : *B;
    const int k = j < ps.nfa ? ps.fa[j] : ps.fb[j - ps.nfa];
    so.seg[j] = m.d_idx + 3 * m.idx_off[k];
    so.len[j] = 3 * m.nsec[k];
  }
  // the scan by the last workgroup, unless a table of this size wants more threads (in a
  // plan of one wait nbcap is only a bound, mostly far above the count)
  const bool fused = nbcap <= kPlanFuse || one_wait;
  hipLaunchKernelGGL(k_plan_blocks, dim3((unsigned)std::min<int64_t>((nbcap + 3) / 4, kPlanGrid)), dim3(256),
                     stage_b ? sizeof(uint64_t) * nB : 0, s, va, vb, w, stage_b, d_hdr, stat, C->d_qi,
                     p->d_tasks, p->d_tuples, tk_of(prec), fused ? nbcap : 0, so);
  if (!fused)
    hipLaunchKernelGGL(k_plan_scan, dim3(1), dim3(kPlanThreads), 0, s, stat, tk_of(prec), d_hdr, so);
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
