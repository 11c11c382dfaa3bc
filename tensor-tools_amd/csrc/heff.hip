// heff.hip -- lazy effective Hamiltonian y = prime(-1)[((L*x)*W12)*R]
// (big_qtensor::product, big_qtensor.cpp:23-40) as three planned grouped
// GEMM stages on the library stream.
//
// The three stage plans are built once per operator (the block structure of
// L, W12, R and x does not change inside a Davidson call).  Stage outputs
// T1 and T2 are materialised in HBM: FP64 for TTG_FP64, FP32 for the
// reduced-precision forms (whose operands are FP32 shadows of L, W12 and R
// made once per operator).  The split-BF16 form keeps the operands of its
// two MFMA stages (L, x, T2, R) as pre-split words (bf16 hi << 16 | bf16
// lo, the same 4 bytes per element): L and R are split once per operator,
// x by the apply's first kernel and T2 by the vector-ALU stage that writes
// it, so the MFMA stages only regroup halves where they would split.  The
// first stage reads x and the last one writes y in FP64 in x's block layout:
// every output block's offset is remapped to the offset of the same sector
// tuple in x, so y and x share one block list and the Davidson vector ops stay
// plain packed-array BLAS-1.
//
// An apply launches its stages directly (three to six kernels).  As a captured
// graph it needed x and y copied in and out of fixed buffers: two copies and
// a graph launch cost 12-25 us per apply, and capturing and instantiating the
// graph cost an operator more than the launches of the few products it serves.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <map>
#include <set>
#include <tuple>

#include "ttg_device.h"
#include "ttg_internal.h"
#include "ttg_plan.h"

struct ttg_heff_s {
  ttg_plan p[3] = {nullptr, nullptr, nullptr};
  ttg::MetaPtr xm;               // x / y block structure
  int prec = TTG_FP64;
  ttg_tensor L = nullptr, W = nullptr, R = nullptr;   // not owned (reference: raw pointers)
  void* T1 = nullptr;
  void* T2 = nullptr;
  // reduced-form operand copies: FP32, or split-BF16 words when packed
  void *Lr = nullptr, *Rr = nullptr, *xr = nullptr;
  float* W32 = nullptr;
  bool packed = false;
  bool covers = false;           // the last stage writes every block of y
  double flops = 0;
  ~ttg_heff_s() {
    for (auto* q : p) delete q;
    ttg::dfree(T1); ttg::dfree(T2);
    ttg::dfree(Lr); ttg::dfree(W32); ttg::dfree(Rr); ttg::dfree(xr);
  }
};

namespace ttg {

__global__ void k_cvt_f32(const double* __restrict__ s, float* __restrict__ d, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    d[i] = (float)s[i];
}

static unsigned grid_n(size_t n) {
  size_t g = (n + 255) / 256;
  return (unsigned)std::max<size_t>(1, std::min<size_t>(g, 4096));
}

// point every output block of the last stage at the same tuple's offset in x
__global__ void k_remap(MetaView c, const uint64_t* xkeys, const int* xids, int nx,
                        const int64_t* xoff, const int* xqi_dims_dummy, CBlock* cblk, int* err) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= c.nblocks) return;
  uint64_t k = 0;
  for (int j = 0; j < c.rank; j++) k = k * c.nsec[j] + c.qi[(size_t)b * c.rank + j];
  int p = lower_bound_u64(xkeys, nx, k);
  if (p >= nx || xkeys[p] != k) {
    atomicAdd(err, 1);
    return;
  }
  int xb = xids[p];
  if (xoff[xb + 1] - xoff[xb] != (int64_t)cblk[b].M * cblk[b].N) {
    atomicAdd(err, 1);
    return;
  }
  cblk[b].c_off = xoff[xb];
}

static int remap_to_x(ttg_plan p3, const MetaPtr& xm) {
  PhaseTimer _phase("remap_to_x");
  hipStream_t s = stream();
  const int nx = xm->nblocks, nc = p3->C->nblocks;
  Scratch sc;
  uint64_t* keys = sc.get<uint64_t>(std::max(nx, 1));
  uint64_t* skeys = sc.get<uint64_t>(std::max(nx, 1));
  int* ids = sc.get<int>(std::max(nx, 1));
  int* sids = sc.get<int>(std::max(nx, 1));
  int* err = sc.get<int>(1);
  TTG_TRY(sc.ok("heff"));
  int herr = 0;
  TTG_TRY(h2d(err, &herr, sizeof(int)));
  if (nx) {
    hipLaunchKernelGGL(k_tuple_keys, dim3((nx + 255) / 256), dim3(256), 0, s, xm->view(), keys, ids);
    hipLaunchKernelGGL(k_sort_keys, dim3((nx + 255) / 256), dim3(256), 0, s, keys, ids, nx, skeys, sids);
  }
  if (nc)
    hipLaunchKernelGGL(k_remap, dim3((nc + 255) / 256), dim3(256), 0, s, p3->C->view(), skeys, sids,
                       nx, xm->d_off, (const int*)nullptr, p3->d_cblk, err);
  {
    const D2HPiece pc{&herr, err, sizeof(int)};
    TTG_TRY(d2h_wait(&pc, 1));
  }
  TTG_REQUIRE(herr == 0, "heff: the product has blocks outside x's block list "
                         "(give x the full legal block list, ttg_tensor_init_blocks)");
  return 0;
}

// Measured tile-shape choice for an MFMA stage of an operator: each
// candidate tile shape's work list is built and its launch timed (HIP events
// on the library stream) on the stage's own operands; the fastest shape is
// kept.  The choice is cached by a coarse signature of the stage (precision,
// stage, rounded log2 flops and tasks, operand layout and format), so the
// operators of neighbouring DMRG bonds reuse it without timing.  Stages the
// planner gave the vector-ALU kernel, stages below kTuneMinFlops (their
// launches are short whatever the shape) and pinned shapes (TTG_TILE_CFG)
// keep the analytic choice.  A plan built with its work list deferred gets
// the list here, for the shape kept.
struct TuneKey {
  int prec, stage, lfl, lnt, layout;
  bool operator<(const TuneKey& o) const {
    return std::tie(prec, stage, lfl, lnt, layout) < std::tie(o.prec, o.stage, o.lfl, o.lnt, o.layout);
  }
};
static std::map<TuneKey, int> g_tuned;
constexpr double kTuneMinFlops = 2e8;

int tune_stage(ttg_plan p, int stage, const void* A, const void* B, void* C, bool out_f64,
               hipStream_t s) {
  PhaseTimer _phase("tune_stage");
  auto keep = [&]() { return p->tiles_pending ? rebuild_tiles(*p, p->cfg) : 0; };
  if (p->cfg == TILE_SKINNY || p->ntasks == 0 || p->flops < kTuneMinFlops) return keep();
  const char* e = getenv("TTG_TILE_CFG");
  if (e && *e) return keep();
  const TuneKey key{p->prec, stage, (int)std::lround(std::log2(std::max(p->flops, 1.0))),
                    (int)std::lround(std::log2((double)std::max<int64_t>(p->ntasks, 1))),
                    (p->a_mcontig ? 1 : 0) | (p->b_kcontig ? 2 : 0) | (p->packed_in ? 4 : 0)};
  auto it = g_tuned.find(key);
  if (it != g_tuned.end()) return it->second == p->cfg ? keep() : rebuild_tiles(*p, it->second);
  int best = p->cfg;
  float best_ms = 1e30f;
  // candidates: the analytic choice and the shapes that were fastest, in some
  // precision, on a stage of the m=512 to m=8192 operators with many small or
  // few large sectors
  std::vector<int> cand{p->cfg};
  for (int c : {TILE_32x32, TILE_64x32, TILE_32x64, TILE_96x32, TILE_64x64, TILE_96x64, TILE_64x96, TILE_128x64}) {
    // (two more shapes cost a split-BF16 operator 3 ms of kernel loading and are
    // never its fastest)
    if (p->prec == TTG_BF16X3 && (c == TILE_96x64 || c == TILE_64x96)) continue;
    if (c != p->cfg) cand.push_back(c);
  }
  // One timed launch per candidate, all queued before one wait.  A kernel
  // instantiation's first launch in the process (code object load) is run
  // untimed first, and the first candidate twice.  Work lists are rebuilt
  // between candidates in stream order (their uploads queue behind the
  // launches that read the old ones).
  static std::set<int> warmed;
  std::vector<hipEvent_t> ev(2 * cand.size(), nullptr);
  auto release = [&]() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  };
  for (size_t i = 0; i < cand.size(); i++) {
    if (hipEventCreate(&ev[2 * i]) != hipSuccess || hipEventCreate(&ev[2 * i + 1]) != hipSuccess) {
      release();
      set_error("heff: event creation failed");
      return 1;
    }
  }
  for (size_t i = 0; i < cand.size(); i++) {
    const int c = cand[i];
    const int kid = c | (p->prec << 5) | (p->a_mcontig ? 128 : 0) | (p->b_kcontig ? 256 : 0) |
                    (out_f64 ? 512 : 0) | (p->packed_in ? 1024 : 0);
    // (the first candidate's extra launch: it is not timed on an idle GPU's
    // lower clock)
    const int warm = i == 0 ? 2 : (warmed.count(kid) ? 0 : 1);
    int wr = rebuild_tiles(*p, c);
    for (int k = 0; k < warm && !wr; k++) wr = gemm_launch(*p, A, B, C, out_f64, s);
    if (wr ||
        hipEventRecord(ev[2 * i], s) != hipSuccess || gemm_launch(*p, A, B, C, out_f64, s) ||
        hipEventRecord(ev[2 * i + 1], s) != hipSuccess) {
      release();
      set_error(std::string("heff: tile timing failed: ") + ttg_last_error());
      return 1;
    }
    warmed.insert(kid);
  }
  if (hipEventSynchronize(ev.back()) != hipSuccess) {
    release();
    set_error("heff: tile timing failed");
    return 1;
  }
  for (size_t i = 0; i < cand.size(); i++) {
    float ms = 0;
    if (hipEventElapsedTime(&ms, ev[2 * i], ev[2 * i + 1]) == hipSuccess && ms < best_ms) {
      best_ms = ms;
      best = cand[i];
    }
  }
  release();
  g_tuned[key] = best;
  return rebuild_tiles(*p, best);
}

// operands, output and output type (FP64 or not) of stage st of y = H x
struct StageIO {
  const void* a;
  const void* b;
  void* c;
  bool f64;
};
static StageIO stage_io(ttg_heff h, int st, const double* x, double* y) {
  if (h->prec == TTG_FP64) {
    if (st == 0) return {h->L->d_data, x, h->T1, true};
    if (st == 1) return {h->T1, h->W->d_data, h->T2, true};
    return {h->T2, h->R->d_data, y, true};
  }
  if (st == 0) return {h->Lr, h->xr, h->T1, false};
  if (st == 1) return {h->T1, h->W32, h->T2, false};
  return {h->T2, h->Rr, y, true};
}

// n FP64 values into a reduced form's operand format (FP32 or split words)
static void reduce_copy(const ttg_heff h, const double* src, void* dst, size_t n, hipStream_t s) {
  if (h->packed) split_words(src, (unsigned*)dst, n, s);
  else hipLaunchKernelGGL(k_cvt_f32, dim3(grid_n(n)), dim3(256), 0, s, src, (float*)dst, n);
}

// y = H x.  x is read by the first stage (or its conversion) only and y written
// by the last one only, so they may be the same array.
static int run(ttg_heff h, const double* x, double* y, hipStream_t s) {
  if (h->prec != TTG_FP64) reduce_copy(h, x, h->xr, h->xm->total, s);
  for (int st = 0; st < 3; st++) {
    if (st == 2 && !h->covers) fill_f64(y, h->xm->total, 0.0);   // blocks of y no stage writes are zero
    const StageIO io = stage_io(h, st, x, y);
    TTG_TRY(gemm_launch(*h->p[st], io.a, io.b, io.c, io.f64, s));
  }
  return 0;
}

// the same for tensors: a y that is one of the operator's own operands is
// written after the last stage has read them
static int apply(ttg_heff h, ttg_tensor x, ttg_tensor y, hipStream_t s) {
  if (y != h->L && y != h->W && y != h->R) return run(h, x->d_data, y->d_data, s);
  Scratch sc;
  double* t = sc.get<double>(h->xm->total);
  TTG_TRY(sc.ok("heff_apply"));
  TTG_TRY(run(h, x->d_data, t, s));
  const DevPiece pc{y->d_data, t, h->xm->total * sizeof(double)};
  return dev_copy(&pc, 1);
}

// intermediates, reduced-form operand copies (FP32 or split words) and, with
// `tune`, the measured tile shapes (on the values of x_like) of an operator
// whose three plans exist; 1 with the error set on failure (the caller
// deletes h)
static int heff_finish(ttg_heff h, const double* x_like, bool tune) {
  const bool red = h->prec != TTG_FP64;
  const size_t es = red ? sizeof(float) : sizeof(double);
  h->covers = h->p[2]->C->nblocks == h->xm->nblocks;   // distinct tuples, each remapped to a block of x
  h->T1 = dmalloc(std::max<size_t>(1, h->p[0]->C->total) * es);
  h->T2 = dmalloc(std::max<size_t>(1, h->p[1]->C->total) * es);
  if (!h->T1 || !h->T2) {
    set_error("heff: allocation failed");
    return 1;
  }
  hipStream_t s = stream();
  if (red) {
    // split words need the vector-ALU kernel to write T2 (it does for the
    // MPO stage's narrow sector dimensions) and MFMA kernels to read L, x, T2
    // and R (small operators can give those stages the vector-ALU kernel,
    // which reads FP32); otherwise the form stays FP32
    h->packed = h->prec == TTG_BF16X3 && h->p[1]->cfg == TILE_SKINNY && h->p[0]->cfg != TILE_SKINNY &&
                h->p[2]->cfg != TILE_SKINNY;
    h->p[0]->packed_in = h->p[2]->packed_in = h->p[1]->split_out = h->packed;
    h->xr = dmalloc(std::max<size_t>(1, h->xm->total) * 4);
    h->Lr = dmalloc(std::max<size_t>(1, h->L->m->total) * 4);
    h->Rr = dmalloc(std::max<size_t>(1, h->R->m->total) * 4);
    h->W32 = dalloc<float>(std::max<size_t>(1, h->W->m->total));
    if (!h->xr || !h->Lr || !h->Rr || !h->W32) {
      set_error("heff: allocation failed");
      return 1;
    }
    reduce_copy(h, h->L->d_data, h->Lr, h->L->m->total, s);
    reduce_copy(h, h->R->d_data, h->Rr, h->R->m->total, s);
    hipLaunchKernelGGL(k_cvt_f32, dim3(grid_n(h->W->m->total)), dim3(256), 0, s, h->W->d_data, h->W32,
                       h->W->m->total);
  }
  if (tune) {   // measured tile shapes of the MFMA stages
    Scratch sc;
    double* y = sc.get<double>(h->xm->total);
    TTG_TRY(sc.ok("heff"));
    for (int st = 0; st < 3; st++) {
      const StageIO io = stage_io(h, st, x_like, y);
      if (tune_stage(h->p[st], st, io.a, io.b, io.c, io.f64, s)) return 1;
    }
  }
  return 0;
}

}  // namespace ttg

using namespace ttg;

extern "C" {

int ttg_heff_create(ttg_tensor L, ttg_tensor W12, ttg_tensor R, ttg_tensor x_like,
                    const int* pairs3, int prec, ttg_heff* out) {
  PhaseTimer _phase("ttg_heff_create");
  TTG_REQUIRE(L && W12 && R && x_like && out, "heff_create: null argument");
  TTG_REQUIRE(prec == TTG_FP64 || prec == TTG_FP32 || prec == TTG_BF16X3, "unknown precision");
  ttg_heff h = new ttg_heff_s();
  h->prec = prec;
  h->L = L; h->W = W12; h->R = R;
  h->xm = x_like->m;
  const int* pp = pairs3;
  MetaPtr lhs[3] = {L->m, nullptr, nullptr};
  MetaPtr rhs[3] = {x_like->m, W12->m, R->m};
  for (int s = 0; s < 3; s++) {
    int np = *pp++;
    std::vector<int> pa(np), pb(np);
    for (int i = 0; i < np; i++) { pa[i] = *pp++; pb[i] = *pp++; }
    MetaPtr a = s == 0 ? lhs[0] : h->p[s - 1]->C;
    // work lists deferred: heff_finish builds each for its measured shape
    int r = plan_build(a, rhs[s], np, pa.data(), pb.data(), prec, -1, &h->p[s], true);
    if (r) { delete h; return r; }
    h->flops += h->p[s]->flops;
  }
  // the last stage's result indices must be x's (after prime(-1))
  if (!h->p[2]->C->same_indices(*h->xm)) {
    delete h;
    set_error("heff: L*x*W12*R does not reproduce x's index sectors");
    return 1;
  }
  if (remap_to_x(h->p[2], h->xm) || heff_finish(h, x_like->d_data, true)) {
    delete h;
    return 1;
  }
  *out = h;
  return 0;
}

int ttg_heff_create_twin(ttg_heff src, int prec, ttg_heff* out) {
  PhaseTimer _phase("ttg_heff_create_twin");
  TTG_REQUIRE(src && out, "heff_create_twin: null argument");
  TTG_REQUIRE(prec == TTG_FP64 || prec == TTG_FP32 || prec == TTG_BF16X3, "unknown precision");
  ttg_heff h = new ttg_heff_s();
  h->prec = prec;
  h->L = src->L; h->W = src->W; h->R = src->R;
  h->xm = src->xm;
  h->flops = src->flops;
  for (int st = 0; st < 3; st++) {
    if (plan_clone(*src->p[st], prec, &h->p[st])) {
      delete h;
      return 1;
    }
  }
  // the source's tile shapes (a twin serves a few products: timing candidate
  // shapes for it would cost more than it saves)
  if (heff_finish(h, nullptr, false)) {
    delete h;
    return 1;
  }
  *out = h;
  return 0;
}

int ttg_heff_new_output(ttg_heff h, ttg_tensor* y) {
  TTG_REQUIRE(h, "null heff");
  return tensor_from_meta(h->xm, true, y);
}

int ttg_heff_apply(ttg_heff h, ttg_tensor x, ttg_tensor y) {
  PhaseTimer _phase("ttg_heff_apply");
  TTG_REQUIRE(h && x && y, "heff_apply: null argument");
  TTG_REQUIRE(same_meta(x->m, h->xm) && same_meta(y->m, h->xm),
              "heff_apply: x/y do not have the operator's block list");
  TTG_TRY(apply(h, x, y, stream()));
  mark_written(y);
  return 0;
}

int ttg_heff_info(ttg_heff h, double* flops, int64_t* ntasks3, double* stage_flops3) {
  TTG_REQUIRE(h, "null heff");
  if (flops) *flops = h->flops;
  for (int s = 0; s < 3; s++) {
    if (ntasks3) ntasks3[s] = h->p[s]->ntasks;
    if (stage_flops3) stage_flops3[s] = h->p[s]->flops;
  }
  return 0;
}

int ttg_heff_time(ttg_heff h, ttg_tensor x, ttg_tensor y, int n, double* ms) {
  TTG_REQUIRE(h && x && y && n > 0 && ms, "heff_time: bad argument");
  TTG_REQUIRE(same_meta(x->m, h->xm) && same_meta(y->m, h->xm),
              "heff_time: x/y do not have the operator's block list");
  hipStream_t s = stream();
  hipEvent_t e0, e1;
  TTG_HIP(hipEventCreate(&e0));
  TTG_HIP(hipEventCreate(&e1));
  TTG_HIP(hipEventRecord(e0, s));
  for (int i = 0; i < n; i++) TTG_TRY(apply(h, x, y, s));
  TTG_HIP(hipEventRecord(e1, s));
  TTG_HIP(hipEventSynchronize(e1));
  float t = 0;
  TTG_HIP(hipEventElapsedTime(&t, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  mark_written(y);
  *ms = t / n;
  return 0;
}

int ttg_heff_stage_time(ttg_heff h, ttg_tensor x, int n, double* ms3) {
  TTG_REQUIRE(h && x && n > 0 && ms3, "heff_stage_time: bad argument");
  TTG_REQUIRE(same_meta(x->m, h->xm), "heff_stage_time: x does not have the operator's block list");
  hipStream_t s = stream();
  Scratch sc;
  double* y = sc.get<double>(h->xm->total);
  TTG_TRY(sc.ok("heff_stage_time"));
  if (h->prec != TTG_FP64) reduce_copy(h, x->d_data, h->xr, h->xm->total, s);
  hipEvent_t ev[4];
  for (auto& e : ev) TTG_HIP(hipEventCreate(&e));
  float acc[3] = {0, 0, 0};
  for (int it = 0; it < n; it++) {
    TTG_HIP(hipEventRecord(ev[0], s));
    for (int st = 0; st < 3; st++) {
      const StageIO io = stage_io(h, st, x->d_data, y);
      TTG_TRY(gemm_launch(*h->p[st], io.a, io.b, io.c, io.f64, s));
      TTG_HIP(hipEventRecord(ev[st + 1], s));
    }
    TTG_HIP(hipEventSynchronize(ev[3]));
    for (int k = 0; k < 3; k++) {
      float t = 0;
      TTG_HIP(hipEventElapsedTime(&t, ev[k], ev[k + 1]));
      acc[k] += t;
    }
  }
  for (auto& e : ev) (void)hipEventDestroy(e);
  for (int k = 0; k < 3; k++) ms3[k] = acc[k] / n;
  return 0;
}

int ttg_heff_tiles(ttg_heff h, int* tile_cfg3, int* ntiles3) {
  TTG_REQUIRE(h, "null heff");
  for (int k = 0; k < 3; k++) {
    if (tile_cfg3) tile_cfg3[k] = h->p[k]->cfg;
    if (ntiles3) ntiles3[k] = h->p[k]->ntiles;
  }
  return 0;
}

int ttg_heff_stage_plan(ttg_heff h, int stage, ttg_plan* out) {
  TTG_REQUIRE(h && out && stage >= 0 && stage < 3, "heff_stage_plan: bad argument");
  *out = h->p[stage];
  return 0;
}

int ttg_heff_free(ttg_heff h) {
  delete h;   // its buffers go back to the pool, whose reuse is ordered by the stream
  return 0;
}

}  // extern "C"
