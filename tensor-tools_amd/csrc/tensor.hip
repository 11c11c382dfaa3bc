// tensor.hip -- device tensor store and the packed-block vector operations.
#include <algorithm>
#include <cstring>

#include "ttg_internal.h"
#include "ttg_device.h"

namespace ttg {

// ---------------------------------------------------------------- meta
TMeta::~TMeta() {
  if (!base) {
    dfree(d_idx);
    dfree(d_qi);
    dfree(d_off);
  }
  dfree(d_lut);
}

MetaView TMeta::view() const {
  MetaView v;
  v.rank = rank;
  v.nblocks = nblocks;
  for (int j = 0; j < MAXR; j++) {
    v.arrow[j] = arrow[j];
    v.nsec[j] = nsec[j];
    v.idx_off[j] = idx_off[j];
  }
  v.idx = d_idx;
  v.qi = d_qi;
  v.off = d_off;
  return v;
}

bool TMeta::same_indices(const TMeta& o) const {
  if (rank != o.rank) return false;
  for (int j = 0; j < rank; j++)
    if (arrow[j] != o.arrow[j] || nsec[j] != o.nsec[j]) return false;
  return h_idx == o.h_idx;
}

static int upload_idx(TMeta& m) {
  m.d_idx = dalloc<int>(m.h_idx.size());
  TTG_REQUIRE(m.d_idx, "meta: device allocation failed");
  return h2d_vec(m.d_idx, m.h_idx);
}

int meta_shell(int rank, const int* arrows, const int* nsec, const int* qn, const int* qdim,
               MetaPtr* out) {
  TTG_TRY(ensure_init());
  TTG_REQUIRE(rank >= 0 && rank <= MAXR, "tensor rank out of range (max 8)");
  auto m = std::make_shared<TMeta>();
  m->rank = rank;
  int off = 0;
  for (int j = 0; j < rank; j++) {
    TTG_REQUIRE(arrows[j] == 0 || arrows[j] == 1, "arrow must be 0 (Inward) or 1 (Outward)");
    TTG_REQUIRE(nsec[j] >= 1, "every index needs at least one sector");
    m->arrow[j] = arrows[j];
    m->nsec[j] = nsec[j];
    m->idx_off[j] = off;
    for (int s = 0; s < nsec[j]; s++) {
      int a = qn[2 * (off + s)], b = qn[2 * (off + s) + 1], d = qdim[off + s];
      TTG_REQUIRE(d >= 1, "sector dimension must be >= 1");
      TTG_REQUIRE(a > -32768 && a < 32767 && b > -32768 && b < 32767, "QN component out of range");
      if (s > 0) {
        int pa = qn[2 * (off + s - 1)], pb = qn[2 * (off + s - 1) + 1];
        TTG_REQUIRE(std::make_pair(pa, pb) < std::make_pair(a, b),
                    "index sectors must be sorted by QN and distinct");
      }
      m->h_idx.push_back(a);
      m->h_idx.push_back(b);
      m->h_idx.push_back(d);
    }
    off += nsec[j];
  }
  m->idx_off[rank] = off;
  TTG_TRY(upload_idx(*m));
  *out = m;
  return 0;
}

MetaPtr meta_from_indices(const std::vector<std::pair<const TMeta*, int>>& src, bool upload) {
  auto m = std::make_shared<TMeta>();
  m->rank = (int)src.size();
  int off = 0;
  for (int j = 0; j < m->rank; j++) {
    const TMeta* s = src[j].first;
    int k = src[j].second;
    m->arrow[j] = s->arrow[k];
    m->nsec[j] = s->nsec[k];
    m->idx_off[j] = off;
    for (int t = 0; t < s->nsec[k]; t++) {
      m->h_idx.push_back(s->q0(k, t));
      m->h_idx.push_back(s->q1(k, t));
      m->h_idx.push_back(s->dim(k, t));
    }
    off += s->nsec[k];
  }
  m->idx_off[m->rank] = off;
  if (upload) {
    if (upload_idx(*m) != 0) return nullptr;
  } else {
    m->d_idx = dalloc<int>(m->h_idx.size());
    if (!m->d_idx) {
      set_error(std::string("meta: ") + ttg_last_error());
      return nullptr;
    }
  }
  return m;
}

int meta_alloc_blocks(TMeta& m, int nblocks, size_t total) {
  m.nblocks = nblocks;
  m.total = total;
  m.d_qi = dalloc<int>((size_t)nblocks * std::max(m.rank, 1));
  m.d_off = dalloc<int64_t>((size_t)nblocks + 1);
  TTG_REQUIRE(m.d_qi && m.d_off, "meta: device allocation failed");
  return 0;
}

}  // namespace ttg

ttg_tensor_s::~ttg_tensor_s() {
  ttg::dfree(d_data);
  ttg::dfree(d_f32);
}

namespace ttg {

int tensor_from_meta(const MetaPtr& m, bool zero, ttg_tensor* out) {
  ttg_tensor t = new ttg_tensor_s();
  t->m = m;
  t->d_data = dalloc<double>(m->total);
  if (!t->d_data) {
    delete t;
    set_error(std::string("tensor: ") + ttg_last_error());   // the pool's reason
    return 1;
  }
  if (zero && m->total)
    fill_f64(t->d_data, m->total, 0.0);
  *out = t;
  return 0;
}

bool same_structure(ttg_tensor a, ttg_tensor b) { return same_meta(a->m, b->m); }

bool same_meta(const MetaPtr& a, const MetaPtr& b) {
  if (a == b) return true;
  if (!a || !b) return false;
  TMeta &x = *a, &y = *b;
  if (x.nblocks != y.nblocks || x.total != y.total || !x.same_indices(y)) return false;
  // compare block lists on the host (small)
  const size_t n = (size_t)x.nblocks * x.rank;
  D2HPiece pc[2];
  int np = 0;
  for (TMeta* m : {&x, &y})
    if (m->h_qi.size() != n) {
      m->h_qi.resize(n);
      pc[np++] = {m->h_qi.data(), m->d_qi, n * sizeof(int)};
    }
  if (np && d2h_wait(pc, np) != 0) {
    for (int i = 0; i < np; i++) (pc[i].dst == x.h_qi.data() ? x : y).h_qi.clear();
    set_error("block list comparison: device copy failed");
    return false;
  }
  return x.h_qi == y.h_qi;
}

// ---------------------------------------------------------------- kernels
__global__ void k_fill(double* __restrict__ d, size_t n, double v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    d[i] = v;
}

__global__ void k_random(double* __restrict__ d, size_t n, uint64_t seed) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    uint64_t z = seed + (uint64_t)(i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    d[i] = (double)(z >> 11) * (1.0 / 9007199254740992.0);
  }
}

__global__ void k_to_f32(const double* __restrict__ s, float* __restrict__ d, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    d[i] = (float)s[i];
}

__global__ void k_scale(double* __restrict__ d, size_t n, double a) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    d[i] *= a;
}

__global__ void k_axpy(double a, const double* __restrict__ x, double* __restrict__ y, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    y[i] += a * x[i];
}

struct LinArgs {
  const double* x[8];
  double c[8];
  int n;
};
__global__ void k_lincomb(LinArgs a, double* __restrict__ y, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int k = 0; k < a.n; k++) s += a.c[k] * a.x[k][i];
    y[i] = s;
  }
}

// Deterministic dot: 512 partial sums (number c takes elements 256 c .. 256 c +
// 255 of every stretch of 512 * 256), added in a fixed tree by the workgroup that
// finishes last, which writes the result to pinned host memory.  A workgroup
// forms four partial sums: what is paid besides the reading is one agent-scope
// fence and counter update a workgroup, and 512 workgroups of 256 threads took
// 13.3 us for 2 x 8 MB where these take 7.3.  Workgroups without elements are not
// launched; their partial sums are zero.  (As two kernels and a copy of the
// result a dot took 16 us of the stream, most of it between the three.)
constexpr int kDotGrid = 128, kDotParts = 512;
__global__ void __launch_bounds__(1024) k_dot(const double* __restrict__ x, const double* __restrict__ y, size_t n,
                                              double* part, unsigned* done, double* out) {
  __shared__ double red[16];
  __shared__ bool last;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  auto wave_sum = [](double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
  };
  double s = 0.0;
  constexpr size_t S = (size_t)kDotParts * 256;
  size_t i = blockIdx.x * (size_t)1024 + tid;
  for (; i + 7 * S < n; i += 8 * S) {   // eight pairs of loads under way at once
    double a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      a[j] = x[i + j * S];
      b[j] = y[i + j * S];
    }
#pragma unroll
    for (int j = 0; j < 8; j++) s += a[j] * b[j];
  }
  for (; i < n; i += S) s += x[i] * y[i];
  s = wave_sum(s);
  if (lane == 0) red[w] = s;
  __syncthreads();
  if (w == 0) {
    if (lane < 4)
      __hip_atomic_store(&part[4 * blockIdx.x + lane],
                         (red[4 * lane] + red[4 * lane + 2]) + (red[4 * lane + 1] + red[4 * lane + 3]),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (lane == 0)
      last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  if (w < 8) {
    const double v =
        tid < 4 * (int)gridDim.x ? __hip_atomic_load(&part[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
    const double r = wave_sum(v);
    if (lane == 0) red[w] = r;
  }
  __syncthreads();
  if (w == 0) {
    const double r = wave_sum(lane < 8 ? red[lane] : 0.0);
    if (lane == 0) {
      *out = r;
      *done = 0;   // for the next call, which the stream orders after this one
    }
  }
}

// x . y into *out once the stream is done
static int dev_dot(const double* x, const double* y, size_t n, double* out) {
  static double* scratch = nullptr;   // partial sums and the counter
  static double* host = nullptr;
  if (!scratch) {
    scratch = dalloc<double>(kDotParts + 1);
    TTG_REQUIRE(scratch, "dot scratch allocation failed");
    fill_f64(scratch, kDotParts + 1, 0.0);
  }
  if (!host) TTG_HIP(hipHostMalloc((void**)&host, sizeof(double)));
  const unsigned g = (unsigned)std::max<size_t>(1, std::min<size_t>((n + 1023) / 1024, kDotGrid));
  hipLaunchKernelGGL(k_dot, dim3(g), dim3(1024), 0, stream(), x, y, n, scratch, (unsigned*)(scratch + kDotParts), host);
  TTG_HIP(hipGetLastError());
  TTG_HIP(hipStreamSynchronize(stream()));
  *out = *host;
  return 0;
}

static unsigned grid_for(size_t n) {
  size_t g = (n + 255) / 256;
  if (g > 4096) g = 4096;
  if (g < 1) g = 1;
  return (unsigned)g;
}

void fill_f64(double* d, size_t n, double v) {
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(256), 0, stream(), d, n, v);
}

// Copies between buffers of the device and pinned host memory: one launch for
// up to kCopyPieces of them, 16 bytes a lane (the library's buffers are aligned to
// that; single bytes at the end and for any other address).  A
// planning call or an SVD makes a dozen copies of a few hundred bytes, and a
// hipMemcpyAsync is a launch too (2.9 us of the GPU, as one of these is) that
// costs the host more: the Davidson call at m=1024 took 2281 us with 73 of them and
// takes 1808 us with 15 launches of k_copy, a 20-site sweep at m=48 107 and 98 ms
// (4270 and 2407).
// (It stands here, beside kernels that every program launches: a source file's kernels
// are loaded at the first launch of one of them, some milliseconds.)
__global__ void __launch_bounds__(256) k_copy(CopyArgs a) {
  const int p = blockIdx.y;
  char* __restrict__ d = a.dst[p];
  const char* __restrict__ s = a.src[p];
  const size_t n = a.bytes[p];
  const size_t i0 = blockIdx.x * (size_t)256 + threadIdx.x, step = gridDim.x * (size_t)256;
  const unsigned low = (unsigned)((size_t)d | (size_t)s);
  size_t done = 0;
  if ((low & 15) == 0) {
    for (size_t i = i0; i < n / 16; i += step) ((uint4*)d)[i] = ((const uint4*)s)[i];
    done = n & ~size_t(15);
  }
  for (size_t i = done + i0; i < n; i += step) d[i] = s[i];
}

int copy_pieces(const CopyArgs& a, unsigned g, int n) {
  hipLaunchKernelGGL(k_copy, dim3(g, n), dim3(256), 0, stream(), a);
  TTG_HIP(hipGetLastError());
  return 0;
}

// the same sectors and block list with every arrow flipped (qtensor::dag,
// qtensor.cpp:1575-1581): a new structure object on the same device tables,
// which nothing writes once a structure is complete
int meta_dag(const MetaPtr& o, MetaPtr* out) {
  auto m = std::make_shared<TMeta>();
  m->rank = o->rank;
  m->nblocks = o->nblocks;
  m->total = o->total;
  m->h_idx = o->h_idx;
  m->h_qi = o->h_qi;
  for (int j = 0; j <= MAXR; j++) m->idx_off[j] = o->idx_off[j];
  for (int j = 0; j < o->rank; j++) {
    m->arrow[j] = 1 - o->arrow[j];
    m->nsec[j] = o->nsec[j];
  }
  m->d_idx = o->d_idx;
  m->d_qi = o->d_qi;
  m->d_off = o->d_off;
  m->base = o->base ? o->base : o;
  *out = m;
  return 0;
}

int tensor_f32(ttg_tensor t, const float** out) {
  if (!t->d_f32) {
    t->d_f32 = dalloc<float>(t->m->total);
    TTG_REQUIRE(t->d_f32, "f32 shadow allocation failed");
  }
  if (t->f32_version != t->version) {
    hipLaunchKernelGGL(k_to_f32, dim3(grid_for(t->m->total)), dim3(256), 0, stream(), t->d_data,
                       t->d_f32, t->m->total);
    t->f32_version = t->version;
  }
  *out = t->d_f32;
  return 0;
}

// ---------------------------------------------------------------- initBlock
// One workgroup walks the sector combinations in chunks of 1024 (index 0
// fastest), flags zero-flux tuples and compacts them with a block scan.
// Writes (nblocks, total) to hdr, in pinned host memory, and, if there are
// arrays for them, qi and offsets.
__global__ void __launch_bounds__(1024) k_init_blocks(MetaView m, int64_t ncomb,
                                                      int* __restrict__ qi_out,
                                                      int64_t* __restrict__ off_out,
                                                      int64_t* __restrict__ hdr) {
  __shared__ int64_t scan_lds[2 * 32];
  int64_t carry_n = 0, carry_s = 0;
  for (int64_t base = 0; base < ncomb; base += 1024) {
    int64_t i = base + threadIdx.x;
    int legal = 0;
    int64_t size = 0;
    int pos[MAXR];
    if (i < ncomb) {
      int64_t r = i;
      int f0 = 0, f1 = 0;
      size = 1;
      for (int j = 0; j < m.rank; j++) {
        int p = (int)(r % m.nsec[j]);
        r /= m.nsec[j];
        pos[j] = p;
        const int* e = m.idx + 3 * (m.idx_off[j] + p);
        int sg = m.arrow[j] == 0 ? 1 : -1;
        f0 += sg * e[0];
        f1 += sg * e[1];
        size *= e[2];
      }
      legal = (f0 == 0 && f1 == 0);
      if (!legal) size = 0;
    }
    int64_t tot_n, tot_s;
    int64_t pn = block_excl_scan<1024>((int64_t)legal, scan_lds, &tot_n);
    int64_t ps = block_excl_scan<1024>(size, scan_lds + 32, &tot_s);
    if (qi_out && legal) {
      int64_t b = carry_n + pn;
      for (int j = 0; j < m.rank; j++) qi_out[b * m.rank + j] = pos[j];
      off_out[b] = carry_s + ps;
    }
    carry_n += tot_n;
    carry_s += tot_s;
  }
  if (threadIdx.x == 0) {
    hdr[0] = carry_n;
    hdr[1] = carry_s;
    if (qi_out) off_out[carry_n] = carry_s;
  }
}

}  // namespace ttg

using namespace ttg;

extern "C" {

int ttg_tensor_create(int rank, const int* arrows, const int* nsec, const int* qn,
                      const int* qdim, int nblocks, const int* block_qi, ttg_tensor* out) {
  PhaseTimer _phase("ttg_tensor_create");
  MetaPtr m;
  UploadBatch up;
  TTG_TRY(meta_shell(rank, arrows, nsec, qn, qdim, &m));
  TTG_REQUIRE(nblocks >= 0, "nblocks < 0");
  std::vector<int64_t> off(nblocks + 1, 0);
  for (int b = 0; b < nblocks; b++) {
    int64_t sz = 1;
    for (int j = 0; j < rank; j++) {
      int p = block_qi[b * rank + j];
      TTG_REQUIRE(p >= 0 && p < nsec[j], "block sector position out of range");
      sz *= m->dim(j, p);
    }
    off[b + 1] = off[b] + sz;
  }
  TTG_TRY(meta_alloc_blocks(*m, nblocks, (size_t)off[nblocks]));
  if (nblocks) TTG_TRY(h2d(m->d_qi, block_qi, sizeof(int) * (size_t)nblocks * rank));
  TTG_TRY(h2d_vec(m->d_off, off));
  TTG_TRY(up.flush());
  TTG_TRY(tensor_from_meta(m, true, out));
  return 0;
}

int ttg_tensor_init_blocks(int rank, const int* arrows, const int* nsec, const int* qn,
                           const int* qdim, ttg_tensor* out) {
  PhaseTimer _phase("ttg_tensor_init_blocks");
  MetaPtr m;
  TTG_TRY(meta_shell(rank, arrows, nsec, qn, qdim, &m));
  int64_t ncomb = 1;
  for (int j = 0; j < rank; j++) {
    ncomb *= nsec[j];
    TTG_REQUIRE(ncomb < ((int64_t)1 << 40), "initBlock: too many sector combinations");
  }
  // up to kInitOnce combinations the tables take that many entries and one
  // launch fills them; above that a first launch counts
  constexpr int64_t kInitOnce = 4096;
  static int64_t* hdr = nullptr;
  if (!hdr) TTG_HIP(hipHostMalloc((void**)&hdr, 2 * sizeof(int64_t)));
  const bool once = ncomb <= kInitOnce;
  if (once) TTG_TRY(meta_alloc_blocks(*m, (int)ncomb, 0));
  hipLaunchKernelGGL(k_init_blocks, dim3(1), dim3(1024), 0, stream(), m->view(), ncomb, m->d_qi, m->d_off, hdr);
  TTG_HIP(hipGetLastError());
  TTG_HIP(hipStreamSynchronize(stream()));
  TTG_REQUIRE(hdr[0] < (1 << 30), "initBlock: too many blocks");
  if (once) {
    m->nblocks = (int)hdr[0];
    m->total = (size_t)hdr[1];
  } else {
    TTG_TRY(meta_alloc_blocks(*m, (int)hdr[0], (size_t)hdr[1]));
    hipLaunchKernelGGL(k_init_blocks, dim3(1), dim3(1024), 0, stream(), m->view(), ncomb, m->d_qi, m->d_off, hdr);
  }
  return tensor_from_meta(m, true, out);
}

int ttg_tensor_upload(ttg_tensor t, const double* host, size_t n) {
  PhaseTimer _phase("ttg_tensor_upload");
  TTG_REQUIRE(t && n == t->m->total, "upload: size mismatch");
  if (n) TTG_HIP(hipMemcpyAsync(t->d_data, host, n * sizeof(double), hipMemcpyHostToDevice, stream()));
  TTG_HIP(hipStreamSynchronize(stream()));
  mark_written(t);
  return 0;
}

int ttg_tensor_download(ttg_tensor t, double* host, size_t n) {
  PhaseTimer _phase("ttg_tensor_download");
  TTG_REQUIRE(t && n == t->m->total, "download: size mismatch");
  if (n) TTG_HIP(hipMemcpyAsync(host, t->d_data, n * sizeof(double), hipMemcpyDeviceToHost, stream()));
  TTG_HIP(hipStreamSynchronize(stream()));
  return 0;
}

int ttg_tensor_info(ttg_tensor t, int* rank, int* nblocks, size_t* total) {
  TTG_REQUIRE(t, "null tensor");
  if (rank) *rank = t->m->rank;
  if (nblocks) *nblocks = t->m->nblocks;
  if (total) *total = t->m->total;
  return 0;
}

int ttg_tensor_meta_download(ttg_tensor t, int* block_qi, int64_t* offsets) {
  TTG_REQUIRE(t, "null tensor");
  const TMeta& m = *t->m;
  if (block_qi && m.nblocks)
    TTG_HIP(hipMemcpyAsync(block_qi, m.d_qi, sizeof(int) * (size_t)m.nblocks * m.rank,
                           hipMemcpyDeviceToHost, stream()));
  if (offsets)
    TTG_HIP(hipMemcpyAsync(offsets, m.d_off, sizeof(int64_t) * ((size_t)m.nblocks + 1),
                           hipMemcpyDeviceToHost, stream()));
  TTG_HIP(hipStreamSynchronize(stream()));
  return 0;
}

int ttg_tensor_index_download(ttg_tensor t, int j, int* nsec, int* qn, int* qdim) {
  TTG_REQUIRE(t && j >= 0 && j < t->m->rank, "index_download: bad index");
  const TMeta& m = *t->m;
  if (nsec) *nsec = m.nsec[j];
  for (int s = 0; s < m.nsec[j]; s++) {
    if (qn) { qn[2 * s] = m.q0(j, s); qn[2 * s + 1] = m.q1(j, s); }
    if (qdim) qdim[s] = m.dim(j, s);
  }
  return 0;
}

int ttg_tensor_dag(ttg_tensor t) {
  PhaseTimer _phase("ttg_tensor_dag");
  TTG_REQUIRE(t, "null tensor");
  MetaPtr m;
  TTG_TRY(meta_dag(t->m, &m));
  t->m = m;
  return 0;
}

int ttg_same_blocks(ttg_tensor a, ttg_tensor b, int* same) {
  TTG_REQUIRE(a && b && same, "same_blocks: null argument");
  *same = same_structure(a, b) ? 1 : 0;
  return 0;
}

int ttg_tensor_copy(ttg_tensor src, ttg_tensor* out) {
  PhaseTimer _phase("ttg_tensor_copy");
  TTG_REQUIRE(src, "null tensor");
  TTG_TRY(tensor_from_meta(src->m, false, out));
  const DevPiece pc{(*out)->d_data, src->d_data, src->m->total * sizeof(double)};
  return dev_copy(&pc, 1);
}

int ttg_tensor_free(ttg_tensor t) {
  delete t;
  return 0;
}

int ttg_tensor_fill(ttg_tensor t, double v) {
  TTG_REQUIRE(t, "null tensor");
  fill_f64(t->d_data, t->m->total, v);
  mark_written(t);
  return 0;
}

int ttg_tensor_set_random(ttg_tensor t, uint64_t seed) {
  TTG_REQUIRE(t, "null tensor");
  size_t n = t->m->total;
  hipLaunchKernelGGL(k_random, dim3(grid_for(n)), dim3(256), 0, stream(), t->d_data, n, seed);
  mark_written(t);
  return 0;
}

// ---------------------------------------------------------------- vector ops
int ttg_dot(ttg_tensor x, ttg_tensor y, double* out) {
  PhaseTimer _phase("ttg_dot");
  TTG_REQUIRE(x && y, "null tensor");
  TTG_REQUIRE(same_structure(x, y), "dot: tensors have different block lists");
  return dev_dot(x->d_data, y->d_data, x->m->total, out);
}

int ttg_nrm2(ttg_tensor x, double* out) {
  PhaseTimer _phase("ttg_nrm2");
  TTG_REQUIRE(x, "null tensor");
  double s;
  TTG_TRY(dev_dot(x->d_data, x->d_data, x->m->total, &s));
  *out = std::sqrt(s);
  return 0;
}

int ttg_scale(ttg_tensor x, double a) {
  TTG_REQUIRE(x, "null tensor");
  hipLaunchKernelGGL(k_scale, dim3(grid_for(x->m->total)), dim3(256), 0, stream(), x->d_data,
                     x->m->total, a);
  mark_written(x);
  return 0;
}

int ttg_axpy(double a, ttg_tensor x, ttg_tensor y) {
  TTG_REQUIRE(x && y, "null tensor");
  TTG_REQUIRE(same_structure(x, y), "axpy: tensors have different block lists");
  hipLaunchKernelGGL(k_axpy, dim3(grid_for(x->m->total)), dim3(256), 0, stream(), a, x->d_data,
                     y->d_data, x->m->total);
  mark_written(y);
  return 0;
}

int ttg_lincomb(int nx, const ttg_tensor* xs, const double* c, ttg_tensor y) {
  PhaseTimer _phase("ttg_lincomb");
  TTG_REQUIRE(nx >= 1 && nx <= 8, "lincomb: 1..8 operands");
  LinArgs a;
  a.n = nx;
  for (int k = 0; k < nx; k++) {
    TTG_REQUIRE(xs[k] && same_structure(xs[k], y), "lincomb: block lists differ");
    a.x[k] = xs[k]->d_data;
    a.c[k] = c[k];
  }
  hipLaunchKernelGGL(k_lincomb, dim3(grid_for(y->m->total)), dim3(256), 0, stream(), a, y->d_data,
                     y->m->total);
  mark_written(y);
  return 0;
}

}  // extern "C"
