// MI355X (gfx950) hierarchical-matrix matvec engine and its C-ABI.
//
// One matvec y = H x is two to five kernels on the caller's stream:
//   k_gather   x -> xt[0:n]   (permutation of matvecOriginal, hmat.cc:586-593,
//                              or a copy; converts to the factor precision)
//   k_slab     pass 1: t = W x   (W_k = B_k), each row written through the
//              row map into xt[xt_t : ...]
//              (small operators: k_slab_gather does both)
//   k_slab     pass 2: y = F x + U t, each y row written once, with the
//              permutation of matvecOriginal (hmat.cc:618-626) fused in
// Slabs that are split over several workgroups: the last of them adds the
// partial sums, or in passes of many workgroups a k_reduce after the pass.
// Every byte of the factor data is streamed once per matvec with 16-byte
// non-temporal vector loads; x and t are re-read from L2 / MALL.  See
// layout.h for the slab format.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../../include/bigwham_hip.h"
#include "layout.h"
#include "recompress.h"

// Scratch of bw_hip_matvec_noalloc: x gathered in the factor precision and
// the rank vector t (xt), then the partial sums of both passes, in one fixed
// array per GPU (each GPU that loads this library holds its own copy until
// the process ends).  Host code never passes `scratch` itself to a kernel: its
// device address on each GPU comes from hipGetSymbolAddress (noalloc_bind).
static __device__ __align__(256) unsigned char scratch[BW_NOALLOC_SCRATCH_BYTES];

namespace {

thread_local std::string g_err;

bool verbose() {
  static const bool v = [] {
    const char* e = std::getenv("BIGWHAM_VERBOSE");
    return e && e[0] && e[0] != '0';
  }();
  return v;
}

int fail(int code, const std::string& m) {
  g_err = m;
  return code;
}

#define HIPCHK(expr)                                                              \
  do {                                                                            \
    hipError_t e_ = (expr);                                                       \
    if (e_ != hipSuccess)                                                         \
      return fail(BW_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_));    \
  } while (0)

#include "slab_kernels.h"
#include "batched_kernels.h"

// Waves per workgroup of the batched kernels: 8 are 4-15 % slower (32 right-hand
// sides, FP64, 24 300 DoF: 307 us against 293; FP32, 49 152 DoF: 357 / 331).
constexpr int kBatchWaves = 4;

// ---------------------------------------------------------------------------

// One work-item list of a pass on the device.
struct DevItems {
  bwl::WorkItem* wis = nullptr;
  bwl::Reduce* reds = nullptr;  // one per split slab
  int nwi = 0, nred = 0;
  int ncount = 0;               // counters of split slabs (bwl::ItemList)
  XcdSplit xs = {};
  int blocks = 0;               // workgroups of a launch
  int64_t part_elems = 0;

  // bytes of the scratch for `cols` columns, and the counters within it
  size_t part_bytes(int cols, int es) const { return (part_elems * cols * es + 15) / 16 * 16; }
  size_t scratch_bytes(int cols, int es) const { return part_bytes(cols, es) + ncount * sizeof(int32_t); }
  // the counters: a null pointer always goes with ncount = 0
  int32_t* counters(void* part, int cols, int es) const {
    if (ncount == 0) return nullptr;
    return reinterpret_cast<int32_t*>(static_cast<unsigned char*>(part) + part_bytes(cols, es));
  }
  SplitSums sums(void* part, int cols, int es) const { return {reds, counters(part, cols, es)}; }
  bool reduce_launch() const { return nred > ncount; }
};

struct DevPass {
  DevItems single, batched, wide;  // wide: rounds of 64 columns, if rowtab
  int gather_cols = 0;        // pass 1: longest work item's columns if it may gather x itself
  int32_t* gidx = nullptr;
  int32_t* rowmap = nullptr;  // pass 1: t entry of every slab row
  int64_t* rowtab = nullptr;  // pass 1, windows: where every slab row lies (bwl::Program::rowtab)
  void* data = nullptr;
  int64_t data_bytes = 0;

  // where the partial sums of `wide` begin in the batched scratch
  size_t wide_offset(int cols, int es) const {
    return (batched.scratch_bytes(cols, es) + 255) / 256 * 256;
  }
};

// The read-only device layout of one operator (H or H^T) at one precision.
// Everything a matvec writes lives in an OpScratch instead, one per stream.
struct DevOp {
  bool present = false;
  int elem = 8;  // bytes
  DevPass p1, p2;
  int64_t xt_size = 0;
  int64_t xt_t = 0;     // first t entry in xt
  int64_t t_total = 0;  // t entries
  int64_t n_in = 0, n_out = 0;
  const int64_t* perm_in = nullptr;   // device, n_in / dof
  const int64_t* perm_out = nullptr;  // device, n_out / dof
  int64_t stream_bytes = 0;
  int unroll[2] = {8, 8};     // loads in flight per lane in k_slab (4, 8 or 16), per pass
};

// What one matvec of an operator writes: xt (x gathered in the factor
// precision, then t = B x), the partial sums of split work items of both
// passes with the counters of their split slabs behind them (zero between
// launches), and the same for the batched products (xt_size x xb_cols input and
// rank rows, partial sums x xb_cols).  xt is zero where no kernel writes (the
// gap after x and the tail after t, which padded column groups read); the
// batched gather writes those rows of xb itself.
struct OpScratch {
  void* xt = nullptr;
  void* part[2] = {nullptr, nullptr};
  void* xb = nullptr;
  void* partb[2] = {nullptr, nullptr};
  int xb_cols = 0;  // widest round the batched scratch holds
};

// The scratch of one stream (or of one captured graph): per operator, plus
// the staging vectors of host-pointer calls and the full permuted output of a
// selection.  Calls on different streams use different StreamCtx, so they
// may run concurrently on one handle.
struct StreamCtx {
  hipStream_t stream = nullptr;
  OpScratch op[2][2];  // [adjoint][fp32]
  double* x_stage = nullptr;
  double* y_stage = nullptr;
  double* x_pin = nullptr;  // pinned, read and written by the kernels
  double* y_pin = nullptr;
  double* y_full = nullptr;
  std::vector<void*> allocs;
};

// Allocation-failure hook for tests of the cleanup paths: with the
// environment variable BWHIP_FAIL_ALLOC_AT=k (k >= 1), the k-th device or
// pinned-host allocation made by one C-ABI call asks the runtime for more than
// any machine has, and fails there as if the memory were exhausted.  The count
// restarts at every call that allocates.
// BWHIP_FAIL_FILL_AT=k fails the k-th zero fill of fresh scratch in the same way.
thread_local int64_t g_alloc_seq = 0;
thread_local int64_t g_alloc_fail_at = 0;
thread_local int64_t g_fill_seq = 0;
thread_local int64_t g_fill_fail_at = 0;

void arm_alloc_hook() {
  g_alloc_seq = 0;
  const char* e = std::getenv("BWHIP_FAIL_ALLOC_AT");
  g_alloc_fail_at = e ? std::atoll(e) : 0;
  g_fill_seq = 0;
  const char* f = std::getenv("BWHIP_FAIL_FILL_AT");
  g_fill_fail_at = f ? std::atoll(f) : 0;
}

// Bytes to ask for where a caller needs `bytes`.
size_t alloc_bytes(size_t bytes) {
  const bool fires = g_alloc_fail_at > 0 && ++g_alloc_seq == g_alloc_fail_at;
  return fires ? size_t(1) << 50 : std::max<size_t>(bytes, 16);
}

// hipMalloc of at least 16 bytes, recorded in `allocs`; BW_ENOMEM on failure.
// A failure is reported here and may be handled by the caller: it must not stay
// the thread's last error, which the checks after later launches (here and in
// the caller's other libraries) would take for theirs.
int dev_alloc(void** p, size_t bytes, std::vector<void*>* allocs, const char* what) {
  *p = nullptr;
  const hipError_t e = hipMalloc(p, alloc_bytes(bytes));
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return fail(BW_ENOMEM, std::string(what) + ": hipMalloc: " + hipGetErrorString(e));
  }
  allocs->push_back(*p);
  return BW_OK;
}

int host_pinned_alloc(void** p, size_t bytes, const char* what) {
  *p = nullptr;
  if (hipHostMalloc(p, alloc_bytes(bytes)) != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return fail(BW_ENOMEM, std::string(what) + ": hipHostMalloc failed");
  }
  return BW_OK;
}

// Work-item bytes for the next create; 0 = sized from the matrix (layout.cpp).
std::atomic<int64_t> g_wi_bytes64{0};
std::atomic<int64_t> g_wi_bytes32{0};
std::atomic<int> g_stack_rows{64};
// Relative tolerance of the FP32 copy's low-rank recompression (0: off).
std::atomic<double> g_fp32_rank_tol{0.0};

int upload_items(const bwl::ItemList& il, DevItems* di, std::vector<void*>* allocs) {
  di->nwi = static_cast<int>(il.wis.size());
  di->nred = static_cast<int>(il.reds.size());
  di->ncount = il.counters;
  di->part_elems = il.part_elems;
  for (int x = 0; x <= bwl::kXcds; ++x) di->xs.s[x] = il.xcd[x];
  di->blocks = il.blocks();
  int rc;
  if ((rc = dev_alloc(reinterpret_cast<void**>(&di->wis), il.wis.size() * sizeof(bwl::WorkItem),
                      allocs, "create")) ||
      (rc = dev_alloc(reinterpret_cast<void**>(&di->reds), il.reds.size() * sizeof(bwl::Reduce),
                      allocs, "create")))
    return rc;
  if (!il.wis.empty())
    HIPCHK(hipMemcpy(di->wis, il.wis.data(), il.wis.size() * sizeof(bwl::WorkItem),
                     hipMemcpyHostToDevice));
  if (!il.reds.empty())
    HIPCHK(hipMemcpy(di->reds, il.reds.data(), il.reds.size() * sizeof(bwl::Reduce),
                     hipMemcpyHostToDevice));
  return BW_OK;
}

template <typename T>
int upload_pass(const bwl::Layout& L, const bwl::Program& P, DevPass* dp, hipStream_t st,
                std::vector<void*>* allocs) {
  auto dalloc = [&](void** p, size_t bytes) -> int { return dev_alloc(p, bytes, allocs, "create"); };
  int rc;
  if ((rc = upload_items(P.single, &dp->single, allocs)) ||
      (rc = upload_items(P.batched, &dp->batched, allocs)))
    return rc;
  if (!P.rowtab.empty() && (rc = upload_items(P.wide, &dp->wide, allocs))) return rc;
  if ((rc = dalloc(reinterpret_cast<void**>(&dp->gidx), P.gidx.size() * sizeof(int32_t)))) return rc;
  if (!P.rowmap.empty()) {
    if ((rc = dalloc(reinterpret_cast<void**>(&dp->rowmap), P.rowmap.size() * sizeof(int32_t))))
      return rc;
    HIPCHK(hipMemcpy(dp->rowmap, P.rowmap.data(), P.rowmap.size() * sizeof(int32_t),
                     hipMemcpyHostToDevice));
  }
  if (!P.rowtab.empty()) {
    if ((rc = dalloc(reinterpret_cast<void**>(&dp->rowtab), P.rowtab.size() * sizeof(int64_t))))
      return rc;
    HIPCHK(hipMemcpy(dp->rowtab, P.rowtab.data(), P.rowtab.size() * sizeof(int64_t),
                     hipMemcpyHostToDevice));
  }
  dp->data_bytes = P.data_elems * static_cast<int64_t>(sizeof(T));
  if ((rc = dalloc(&dp->data, static_cast<size_t>(dp->data_bytes)))) return rc;
  if (!P.gidx.empty())
    HIPCHK(hipMemcpy(dp->gidx, P.gidx.data(), P.gidx.size() * sizeof(int32_t), hipMemcpyHostToDevice));
  // data: fill slabs into pinned staging chunks and stream them up
  const int32_t nslab = static_cast<int32_t>(P.slabs.size());
  if (nslab == 0) return BW_OK;
  int64_t max_slab = 0;
  for (const auto& s : P.slabs) max_slab = std::max<int64_t>(max_slab, s.ngroups * s.rows * L.opt.vec_elems);
  // no larger than the pass: pinning 2 x 256 MiB takes 5 ms, most of the upload
  // of a small operator
  const int64_t chunk_elems = std::max<int64_t>(
      max_slab, std::min<int64_t>(P.data_elems, (int64_t(256) << 20) / static_cast<int64_t>(sizeof(T))));
  T* stage[2] = {nullptr, nullptr};
  if ((rc = host_pinned_alloc(reinterpret_cast<void**>(&stage[0]), chunk_elems * sizeof(T),
                              "create: upload staging")))
    return rc;
  if ((rc = host_pinned_alloc(reinterpret_cast<void**>(&stage[1]), chunk_elems * sizeof(T),
                              "create: upload staging"))) {
    (void)hipHostFree(stage[0]);
    return rc;
  }
  hipEvent_t done[2] = {nullptr, nullptr};
  if (hipEventCreate(&done[0]) != hipSuccess || hipEventCreate(&done[1]) != hipSuccess) {
    if (done[0]) (void)hipEventDestroy(done[0]);
    (void)hipHostFree(stage[0]);
    (void)hipHostFree(stage[1]);
    return fail(BW_EHIP, "upload: hipEventCreate");
  }
  const unsigned hc = std::max(1u, std::thread::hardware_concurrency());
  const int nthreads = static_cast<int>(std::min(hc, 32u));
  int buf = 0;
  bool pending[2] = {false, false};
  int32_t s = 0;
  int status = BW_OK;
  while (s < nslab) {
    int32_t e = s;
    int64_t elems = 0;
    while (e < nslab) {
      const int64_t se = P.slabs[e].ngroups * P.slabs[e].rows * L.opt.vec_elems;
      if (elems + se > chunk_elems && e > s) break;
      elems += se;
      ++e;
    }
    if (pending[buf]) {
      // the copy out of this staging buffer must be complete before refilling it
      const hipError_t we = hipEventSynchronize(done[buf]);
      pending[buf] = false;
      if (we != hipSuccess) {
        status = fail(BW_EHIP, std::string("upload: ") + hipGetErrorString(we));
        break;
      }
    }
    T* dst = stage[buf];
    // parallel fill over slabs of this chunk
    std::atomic<int32_t> next{s};
    auto worker = [&]() {
      while (true) {
        const int32_t i = next.fetch_add(8);
        if (i >= e) break;
        const int32_t j = std::min(e, i + 8);
        bwl::fill_slabs<T>(L, P, i, j, dst + (P.slabs[i].data_off - P.slabs[s].data_off));
      }
    };
    std::vector<std::thread> ths;
    for (int t = 1; t < nthreads; ++t) ths.emplace_back(worker);
    worker();
    for (auto& t : ths) t.join();
    hipError_t ce = hipMemcpyAsync(static_cast<T*>(dp->data) + P.slabs[s].data_off, dst,
                                   elems * sizeof(T), hipMemcpyHostToDevice, st);
    if (ce != hipSuccess) {
      status = fail(BW_EHIP, std::string("upload: ") + hipGetErrorString(ce));
      break;
    }
    const hipError_t re = hipEventRecord(done[buf], st);
    if (re != hipSuccess) {
      status = fail(BW_EHIP, std::string("upload: ") + hipGetErrorString(re));
      break;
    }
    pending[buf] = true;
    buf ^= 1;
    if (verbose() && nslab >= 10 && (e * 10 / nslab) != (s * 10 / nslab))
      std::fprintf(stderr, "[bwhip] upload %d / %d slabs\n", e, nslab);
    s = e;
  }
  // every copy has ended (or failed) before the staging buffers are freed
  const hipError_t se = hipStreamSynchronize(st);
  if (se != hipSuccess && status == BW_OK)
    status = fail(BW_EHIP, std::string("upload: ") + hipGetErrorString(se));
  (void)hipEventDestroy(done[0]);
  (void)hipEventDestroy(done[1]);
  (void)hipHostFree(stage[0]);
  (void)hipHostFree(stage[1]);
  return status;
}

}  // namespace

// One direction of a selection operator (0: H, 1: H^T).
struct SelDir {
  int64_t* in_src = nullptr;  // point of each scattered input in the caller's vector
  int64_t* in_dst = nullptr;  // its permuted point (repeated indices: the last one wins)
  int64_t n_pairs = 0;
  int64_t n_in = 0;           // points in the caller's input vector
  int64_t* out_dst = nullptr; // permuted point of each output point
  int64_t n_out = 0;
};

struct SelInfo {
  bool on = false;
  int ordering = BW_ORDER_ORIGINAL;
  SelDir dir[2];
};

struct bw_hip_handle {
  int device = 0;
  int dof = 1;
  int64_t n_row_pts = 0, n_col_pts = 0;
  int64_t nb_entries = 0;
  // algorithmic entries of the factors each precision streams: FR blocks,
  // left factors A, right factors B, and the total rank T ([fp32])
  int64_t entries[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  double fp32_rank_tol = 0.0;
  DevOp op[2][2];  // [adjoint][fp32]
  int64_t* perm0 = nullptr;
  int64_t* perm1 = nullptr;
  std::vector<double> diag_perm, diag_orig;
  std::vector<void*> allocs;
  int64_t device_bytes = 0;
  SelInfo sel;
  // Scratch per stream, allocated on a stream's first call (the null stream's
  // at creation).  stage_elems: doubles of each host-pointer staging vector;
  // yfull_elems: doubles of a selection's full permuted output (0: none).
  std::vector<std::unique_ptr<StreamCtx>> ctxs;
  int64_t stage_elems = 0;
  int64_t yfull_elems = 0;
  // Kernel timing: two alternating sets of events between the kernels of a
  // matvec; a set is read (and accumulated) only when reused two calls later,
  // so timing never stalls the launch pipeline.
  bool timing = false;
  hipEvent_t evs[2][6] = {};
  hipEvent_t* ev = evs[0];
  bool pending[2] = {false, false};
  int cur = 0;
  double sum_ms[6] = {0, 0, 0, 0, 0, 0};
  int64_t n_timed = 0;
  std::mutex mu;  // host-side state (timing ring, lazily allocated batch buffers)
};

namespace {

// Pass 1 gathers x itself where its longest work item's input fits this much
// LDS (two workgroups stay on a compute unit) and the pass is at most this
// long: the gather launch it saves is 3.3 us where launches bound the call and
// 1-2 us behind a longer pass, while reading x through the permutation once per
// work item grows with the pass (16 M entries 68.3 -> 66.0 us a matvec, 46 M
// 157.0 -> 157.2, FP32 43 M 91.6 -> 92.1).
constexpr size_t kGatherLds = 48 << 10;
constexpr int64_t kGatherEntries = 24 << 20;

template <typename T>
int build_op(bw_hip_handle* hd, const bw_flat_hmat* h, bool adjoint, hipStream_t st) {
  DevOp& op = hd->op[adjoint ? 1 : 0][sizeof(T) == 4 ? 1 : 0];
  bwl::OpView view;
  bwl::make_view(h, adjoint, &view);
  bwl::LayoutOptions opt;
  opt.vec_elems = Vec<T>::V;
  opt.elem_bytes = sizeof(T);
  opt.wi_bytes = sizeof(T) == 8 ? g_wi_bytes64.load() : g_wi_bytes32.load();
  opt.stack_rows = g_stack_rows.load();
  bwl::Layout L;
  bwl::build_layout(view, opt, &L);
  std::string msg;
  int rc = bwl::check_layout_limits(L, &msg);
  if (rc) return fail(rc, "create: " + msg);
  if ((rc = upload_pass<T>(L, L.pass1, &op.p1, st, &hd->allocs))) return rc;
  if ((rc = upload_pass<T>(L, L.pass2, &op.p2, st, &hd->allocs))) return rc;
  op.elem = sizeof(T);
  int cols = 0;  // columns of the longest pass-1 work item
  for (const bwl::WorkItem& w : L.pass1.single.wis) cols = std::max(cols, w.ngroups * opt.vec_elems);
  if (cols * sizeof(T) <= kGatherLds && L.pass1.data_elems <= kGatherEntries)
    op.p1.gather_cols = cols;
  op.xt_size = L.xt_size;
  op.xt_t = L.xt_t;
  op.t_total = L.view.t_total;
  op.n_in = static_cast<int64_t>(h->dof) * view.n_col_pts;
  op.n_out = static_cast<int64_t>(h->dof) * view.n_row_pts;
  op.perm_in = adjoint ? hd->perm0 : hd->perm1;
  op.perm_out = adjoint ? hd->perm1 : hd->perm0;
  op.stream_bytes = (L.pass1.data_elems + L.pass2.data_elems) * static_cast<int64_t>(sizeof(T));
  hd->device_bytes += op.p1.data_bytes + op.p2.data_bytes + L.xt_size * sizeof(T) +
                      (L.pass1.single.part_elems + L.pass2.single.part_elems) * sizeof(T) +
                      (op.p1.single.nwi + op.p1.batched.nwi + op.p2.single.nwi + op.p2.batched.nwi) *
                          sizeof(bwl::WorkItem) +
                      (L.pass1.gidx.size() + L.pass2.gidx.size()) * sizeof(int32_t) +
                      L.pass1.rowtab.size() * sizeof(int64_t);
  op.present = true;
  return BW_OK;
}

// Frees the allocations a failed ensure_* call made after `mark`.
int undo_allocs(StreamCtx* ctx, size_t mark, int rc) {
  for (size_t i = mark; i < ctx->allocs.size(); ++i) (void)hipFree(ctx->allocs[i]);
  ctx->allocs.resize(mark);
  return rc;
}

// Zeroes fresh scratch and waits for it, so that no kernel of any stream can
// see it before the zeros land.  (hipMemset of device memory returns before
// it completes, on the null stream, which does not order non-blocking
// streams such as torch's.)
hipError_t zero_now(void* p, size_t bytes) {
  if (g_fill_fail_at > 0 && ++g_fill_seq == g_fill_fail_at) return hipErrorUnknown;
  hipError_t e = hipMemsetAsync(p, 0, bytes, nullptr);
  if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
  return e;
}

// Zeroes the split-slab counters of fresh scratch.
hipError_t zero_counters(const DevItems& di, void* part, int cols, int es) {
  if (di.ncount == 0) return hipSuccess;
  return zero_now(di.counters(part, cols, es), di.ncount * sizeof(int32_t));
}

// Allocates what `ctx` lacks for operator [adj][fp32]: the single-vector
// scratch, and with `batched` the batched one.  xt is zeroed here, once
// (synchronously, before any kernel of the context can use it): the kernels
// only ever write x and t entries, so the gap and tail stay zero.
// A failure frees what it leaves incomplete; the single-vector scratch that was
// complete by then (allocated and zeroed, held by `s`) stays for later calls.
int ensure_op_scratch(bw_hip_handle* hd, StreamCtx* ctx, int adj, int fp32, bool batched) {
  const DevOp& op = hd->op[adj][fp32];
  OpScratch& s = ctx->op[adj][fp32];
  const size_t es = op.elem;
  const size_t mark = ctx->allocs.size();
  int rc;
  if (!s.xt) {
    void* xt = nullptr;
    void* part[2] = {nullptr, nullptr};
    // whole 2 MiB pages, so that no other allocation shares a page with the
    // vectors that this stream's kernels write
    const size_t pages = (op.xt_size * es + (size_t(2) << 20) - 1) >> 21;
    if ((rc = dev_alloc(&xt, pages << 21, &ctx->allocs, "scratch"))) return undo_allocs(ctx, mark, rc);
    for (int p = 0; p < 2; ++p)
      if ((rc = dev_alloc(&part[p], (p ? op.p2 : op.p1).single.scratch_bytes(1, es), &ctx->allocs,
                          "scratch")))
        return undo_allocs(ctx, mark, rc);
    hipError_t e = zero_now(xt, op.xt_size * es);
    for (int p = 0; p < 2 && e == hipSuccess; ++p)
      e = zero_counters((p ? op.p2 : op.p1).single, part[p], 1, es);
    if (e != hipSuccess)
      return undo_allocs(ctx, mark, fail(BW_EHIP, std::string("scratch: zero fill: ") + hipGetErrorString(e)));
    s.xt = xt;
    s.part[0] = part[0];
    s.part[1] = part[1];
  }
  if (batched && !s.xb) {
    // FP32 calls of more than 32 columns run 64 at a time where the scratch and
    // the kernels' 32-bit offsets allow it; everything else needs 32 columns
    int cols = fp32 && op.xt_size * 64 <= static_cast<int64_t>(UINT32_MAX) ? 64 : 32;
    for (;; cols = 32) {
      const size_t mark_b = ctx->allocs.size();
      void* xb = nullptr;
      void* partb[2] = {nullptr, nullptr};
      rc = dev_alloc(&xb, static_cast<size_t>(op.xt_size) * cols * es, &ctx->allocs, "scratch");
      for (int p = 0; p < 2 && !rc; ++p)
        rc = dev_alloc(&partb[p], (p ? op.p2 : op.p1).wide_offset(cols, es) +
                                      (p ? op.p2 : op.p1).wide.scratch_bytes(cols, es),
                       &ctx->allocs, "scratch");
      if (rc) {
        undo_allocs(ctx, mark_b, rc);
        if (cols > 32) continue;
        return rc;
      }
      for (int p = 0; p < 2; ++p) {
        const DevPass& dp = p ? op.p2 : op.p1;
        hipError_t e = zero_counters(dp.batched, partb[p], cols, es);
        if (e == hipSuccess)
          e = zero_counters(dp.wide, static_cast<unsigned char*>(partb[p]) + dp.wide_offset(cols, es),
                            cols, es);
        if (e != hipSuccess)
          return undo_allocs(ctx, mark_b, fail(BW_EHIP, std::string("scratch: zero fill: ") + hipGetErrorString(e)));
      }
      s.xb = xb;
      s.partb[0] = partb[0];
      s.partb[1] = partb[1];
      s.xb_cols = cols;
      break;
    }
  }
  return BW_OK;
}

// Vectors of host-pointer calls.  Up to kPinnedEntries they pass through
// pinned memory that the kernels themselves read and write: copies from and
// to pageable memory cost 15-20 us of a small call (two such copies and two
// small kernels, 800 entries: 30.8 us; through pinned memory 14.9; 16 000: 36.0
// and 22.9; 100 000: 86 and 74).  Results of at most kDirectEntries are stored
// in pinned memory by pass 2, scattered by the permutation (800 entries: 14.9
// us, 16.2 through device memory and a copy kernel; 4 000: 19.8 and 17.9).
// Pass 1 gathers x from pinned memory up to kPinnedGather entries (host calls
// of 800 entries: 22.7 us against 24.4 with a gather launch, 4 599: 42.9 / 49.6,
// 8 000: 40.4 / 36.8).
constexpr int64_t kPinnedEntries = 128 * 1024, kDirectEntries = 1024, kPinnedGather = 6 * 1024;

// Staging vectors of host-pointer calls and a selection's full output.
int ensure_ctx_vectors(bw_hip_handle* hd, StreamCtx* ctx, bool staging) {
  const size_t mark = ctx->allocs.size();
  const size_t bytes = hd->stage_elems * sizeof(double);
  const bool pinned = hd->stage_elems <= kPinnedEntries;
  int rc;
  if (staging && !ctx->y_stage) {
    void *xs = nullptr, *ys = nullptr;
    if ((!pinned && (rc = dev_alloc(&xs, bytes, &ctx->allocs, "scratch"))) ||
        (rc = dev_alloc(&ys, bytes, &ctx->allocs, "scratch")))
      return undo_allocs(ctx, mark, rc);
    if (pinned) {
      // one allocation, x then y
      void* hp = nullptr;
      const size_t xb = (bytes + 255) / 256 * 256;
      if ((rc = host_pinned_alloc(&hp, xb + std::max<size_t>(bytes, 16), "scratch")))
        return undo_allocs(ctx, mark, rc);
      ctx->x_pin = static_cast<double*>(hp);
      ctx->y_pin = reinterpret_cast<double*>(static_cast<unsigned char*>(hp) + xb);
    }
    ctx->x_stage = static_cast<double*>(xs);
    ctx->y_stage = static_cast<double*>(ys);
  }
  if (hd->yfull_elems > 0 && !ctx->y_full) {
    const size_t mark_y = ctx->allocs.size();
    void* yf = nullptr;
    if ((rc = dev_alloc(&yf, hd->yfull_elems * sizeof(double), &ctx->allocs, "scratch")))
      return undo_allocs(ctx, mark_y, rc);
    ctx->y_full = static_cast<double*>(yf);
  }
  return BW_OK;
}

void free_ctx(StreamCtx* ctx) {
  for (void* p : ctx->allocs) (void)hipFree(p);
  ctx->allocs.clear();
  if (ctx->x_pin) (void)hipHostFree(ctx->x_pin);
  ctx->x_pin = ctx->y_pin = nullptr;
}

// The context of `stream` (created empty on its first use); caller holds hd->mu.
StreamCtx* stream_ctx(bw_hip_handle* hd, hipStream_t stream) {
  for (auto& c : hd->ctxs)
    if (c->stream == stream) return c.get();
  hd->ctxs.emplace_back(new StreamCtx());
  hd->ctxs.back()->stream = stream;
  return hd->ctxs.back().get();
}

void compute_diagonal(bw_hip_handle* hd, const bw_flat_hmat* h) {
  const int64_t d = h->dof;
  const int64_t npt = std::max(h->n_row_pts, h->n_col_pts);
  hd->diag_perm.assign(d * npt, 0.0);
  for (int64_t k = 0; k < h->n_fr; ++k) {
    const int64_t* c = h->fr_pattern + 6 * k;
    const int64_t i0 = c[1], j0 = c[2], iend = c[3], jend = c[4];
    const bool lower = (i0 > j0) && (i0 > jend) && (iend > j0) && (iend > jend);
    const bool upper = (i0 < j0) && (i0 < jend) && (iend < j0) && (iend < jend);
    if (lower || upper) continue;
    const int64_t m = d * (iend - i0), n = d * (jend - j0);
    const double* F = h->fr_blocks[k];
    for (int64_t j = 0; j < n; ++j) {
      const int64_t i = j + d * j0 - d * i0;
      if (i >= 0 && i < m) hd->diag_perm[i + d * i0] = F[i + j * m];
    }
  }
  hd->diag_orig.assign(d * npt, 0.0);
  for (int64_t i = 0; i < npt && i < h->n_col_pts; ++i)
    for (int64_t j = 0; j < d; ++j) hd->diag_orig[d * h->perm1[i] + j] = hd->diag_perm[d * i + j];
}

template <typename T, typename OutT, int PASS>
void launch_slab(const DevPass& dp, int unroll, hipStream_t st, const T* xin, OutT* out, T* part,
                 const int64_t* perm, int dof) {
  // 8 waves per workgroup: 4 leave more small workgroups to start and end (the
  // 120 000-DoF 3DR0 operator: pass 1 545 us against 509, pass 2 647 / 638),
  // 16 leave one workgroup per compute unit (mode-1, 25 600 DoF: 44 us / 39).
  // Two buffers of 8 loads; 16 leave a third fewer waves and are slower
  // everywhere (pass 1: 550 us), so an unroll of 16 runs as 8.
  constexpr int W = 8;
  const DevItems& di = dp.single;
#define BW_SLAB(U)                                                                              \
  hipLaunchKernelGGL((k_slab<T, OutT, U, PASS, W>), dim3(di.blocks), dim3(64 * W), 0, st, di.wis, \
                     di.xs, dp.gidx, static_cast<const T*>(dp.data), xin, out, part,               \
                     di.sums(part, 1, sizeof(T)), perm, dof,                                        \
                     dp.rowmap)
  if (unroll == 4)
    BW_SLAB(4);
  else
    BW_SLAB(8);
#undef BW_SLAB
}

// Pass 1 with the gather of x in the same launch (DevPass::gather_cols > 0).
template <typename T>
void launch_slab_gather(const DevPass& dp, int unroll, hipStream_t st, const double* x, T* xt,
                        int64_t n_in, T* part, const int64_t* perm, int dof) {
  constexpr int W = 8;
  const DevItems& di = dp.single;
  // a multiple of 8, so that work items keep their XCD
  const int ngather =
      static_cast<int>(std::min<int64_t>(256, (n_in + 8 * 64 * W - 1) / (8 * 64 * W) * 8));
  const size_t lds = (dp.gather_cols + 64 * W) * sizeof(T);
#define BW_SLAB(U)                                                                             \
  hipLaunchKernelGGL((k_slab_gather<T, U, W>), dim3(ngather + di.blocks), dim3(64 * W), lds, st, \
                     di.wis, di.xs, dp.gidx, static_cast<const T*>(dp.data), x, xt,             \
                     static_cast<int>(n_in), perm, dof, ngather, dp.gather_cols, part,          \
                     di.sums(part, 1, sizeof(T)), dp.rowmap)
  if (unroll == 4)
    BW_SLAB(4);
  else
    BW_SLAB(8);
#undef BW_SLAB
}

// Zero fill of xt's gap after x and its tail after t and of both passes'
// counters, for scratch that other operators may have used before (the
// no-allocation entry point).
template <typename T>
__global__ __launch_bounds__(256) void k_zero_ranges(T* __restrict__ xt, int64_t a0, int64_t a1,
                                                     int64_t b0, int64_t b1,
                                                     int32_t* __restrict__ c1, int n1,
                                                     int32_t* __restrict__ c2, int n2) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < a1 - a0) {
    xt[a0 + i] = T(0);
    return;
  }
  i -= a1 - a0;
  if (i < b1 - b0) {
    xt[b0 + i] = T(0);
    return;
  }
  i -= b1 - b0;
  if (i < n1)
    c1[i] = 0;
  else if (i - n1 < n2)
    c2[i - n1] = 0;
}

// The two to five (selection: four to six) kernels of one matvec on stream st,
// writing only the scratch `s` (and y_full for a selection).
template <typename T>
int launch_matvec(bw_hip_handle* hd, DevOp& op, const OpScratch& s, double* y_full,
                  const double* xd, double* yd, int ordering, hipStream_t st,
                  const SelDir* sd = nullptr, bool timed = true, bool x_pinned = false) {
  const bool orig = !sd && ordering == BW_ORDER_ORIGINAL;
  const int dof = hd->dof;
  T* xt = static_cast<T*>(s.xt);
  T* part1 = static_cast<T*>(s.part[0]);
  T* part2 = static_cast<T*>(s.part[1]);
  double* const y_user = yd;
  if (sd) yd = y_full;  // the passes write the full permuted y
  const bool timing = timed && hd->timing;
  // pass 1 gathers x, unless that reads a long x many times from host memory
  const bool fused = !sd && op.p1.gather_cols > 0 && (!x_pinned || op.n_in <= kPinnedGather);
  if (timing) (void)hipEventRecord(hd->ev[0], st);
  if (sd) {
    if (sd->n_pairs > 0) {
      const int blocks = static_cast<int>((sd->n_pairs * dof + 255) / 256);
      hipLaunchKernelGGL(k_scatter_sel<T>, dim3(blocks), dim3(256), 0, st, xd, xt, sd->in_src,
                         sd->in_dst, sd->n_pairs, dof);
    }
  } else if (!fused) {
    const int64_t n = op.n_in;
    const int blocks = static_cast<int>((n + 255) / 256);
    hipLaunchKernelGGL(k_gather<T>, dim3(blocks), dim3(256), 0, st, xd, xt, n,
                       orig ? op.perm_in : nullptr, dof);
  }
  if (timing) (void)hipEventRecord(hd->ev[1], st);
  if (fused) {
    launch_slab_gather<T>(op.p1, op.unroll[0], st, xd, xt, op.n_in, part1,
                          orig ? op.perm_in : nullptr, dof);
  } else if (op.p1.single.nwi > 0) {
    launch_slab<T, T, 1>(op.p1, op.unroll[0], st, xt, xt, part1, nullptr, dof);
  }
  if (timing) (void)hipEventRecord(hd->ev[2], st);
  if (op.p1.single.reduce_launch())
    hipLaunchKernelGGL((k_reduce<T, T>), dim3(op.p1.single.nred), dim3(64), 0, st,
                       op.p1.single.reds, op.p1.single.nred, part1, xt, nullptr, dof, op.p1.rowmap);
  if (timing) (void)hipEventRecord(hd->ev[3], st);
  if (op.p2.single.nwi > 0) {
    launch_slab<T, double, 2>(op.p2, op.unroll[1], st, xt, yd, part2, orig ? op.perm_out : nullptr,
                              dof);
  }
  if (timing) (void)hipEventRecord(hd->ev[4], st);
  if (op.p2.single.reduce_launch())
    hipLaunchKernelGGL((k_reduce<T, double>), dim3(op.p2.single.nred), dim3(64), 0, st,
                       op.p2.single.reds, op.p2.single.nred, part2, yd, orig ? op.perm_out : nullptr, dof, nullptr);
  if (sd && sd->n_out > 0) {
    const int blocks = static_cast<int>((sd->n_out * dof + 255) / 256);
    hipLaunchKernelGGL(k_gather_sel, dim3(blocks), dim3(256), 0, st, yd, y_user, sd->out_dst,
                       sd->n_out, dof);
  }
  if (timing) (void)hipEventRecord(hd->ev[5], st);
  HIPCHK(hipGetLastError());
  return BW_OK;
}

int accumulate_timing(bw_hip_handle* hd, int set) {
  hipEvent_t* e = hd->evs[set];
  HIPCHK(hipEventSynchronize(e[5]));
  float ms;
  for (int i = 0; i < 5; ++i) {
    HIPCHK(hipEventElapsedTime(&ms, e[i], e[i + 1]));
    hd->sum_ms[i] += ms;
  }
  HIPCHK(hipEventElapsedTime(&ms, e[0], e[5]));
  hd->sum_ms[5] += ms;
  hd->n_timed += 1;
  hd->pending[set] = false;
  return BW_OK;
}

int do_matvec(bw_hip_handle* hd, bool adjoint, const double* x, double* y, int ordering,
              int precision, int on_device, void* stream) {
  if (!hd || !x || !y) return fail(BW_EINVAL, "matvec: null argument");
  if (ordering != BW_ORDER_PERMUTED && ordering != BW_ORDER_ORIGINAL)
    return fail(BW_EINVAL, "matvec: ordering must be 0 (permuted) or 1 (original)");
  if (precision != BW_PREC_FP64 && precision != BW_PREC_FP32)
    return fail(BW_EINVAL, "matvec: precision must be BW_PREC_FP64 or BW_PREC_FP32");
  const int adj = adjoint ? 1 : 0, f32 = precision == BW_PREC_FP32 ? 1 : 0;
  DevOp& op = hd->op[adj][f32];
  if (!op.present)
    return fail(BW_ENOTSUP, adjoint ? "rmatvec: adjoint / precision not built for this handle"
                                    : "matvec: precision not built for this handle");
  const SelDir* sd = nullptr;
  if (hd->sel.on) {
    if (ordering != hd->sel.ordering)
      return fail(BW_ENOTSUP, "matvec: this selection was created for the other ordering");
    sd = &hd->sel.dir[adj];
  }
  const int64_t n_in = sd ? hd->dof * sd->n_in : op.n_in;
  const int64_t n_out = sd ? hd->dof * sd->n_out : op.n_out;
  std::lock_guard<std::mutex> lock(hd->mu);
  arm_alloc_hook();
  hipStream_t st = static_cast<hipStream_t>(stream);
  HIPCHK(hipSetDevice(hd->device));
  StreamCtx* ctx = stream_ctx(hd, st);
  int rc;
  if ((rc = ensure_op_scratch(hd, ctx, adj, f32, false)) ||
      (rc = ensure_ctx_vectors(hd, ctx, !on_device)))
    return rc;
  const double* xd = x;
  double* yd = y;
  const bool pinned = !on_device && ctx->x_pin;
  // a selection stores its rows in order
  const bool direct = pinned && (sd || n_out <= kDirectEntries);
  if (!on_device) {
    if (pinned) {
      std::memcpy(ctx->x_pin, x, n_in * sizeof(double));
      xd = ctx->x_pin;
    } else {
      HIPCHK(hipMemcpyAsync(ctx->x_stage, x, n_in * sizeof(double), hipMemcpyHostToDevice, st));
      xd = ctx->x_stage;
    }
    yd = direct ? ctx->y_pin : ctx->y_stage;
  }
  if (hd->timing) {
    const int set = hd->cur;
    if (hd->pending[set]) {
      int rc0 = accumulate_timing(hd, set);
      if (rc0) return rc0;
    }
    hd->ev = hd->evs[set];
  }
  const OpScratch& s = ctx->op[adj][f32];
  rc = f32 ? launch_matvec<float>(hd, op, s, ctx->y_full, xd, yd, ordering, st, sd, true, pinned)
           : launch_matvec<double>(hd, op, s, ctx->y_full, xd, yd, ordering, st, sd, true, pinned);
  if (rc) return rc;
  if (hd->timing) {
    hd->pending[hd->cur] = true;
    hd->cur ^= 1;
  }
  if (pinned) {
    if (!direct && n_out > 0) {
      hipLaunchKernelGGL(k_copy, dim3(static_cast<unsigned>((n_out + 255) / 256)), dim3(256), 0, st,
                         ctx->y_stage, ctx->y_pin, n_out);
      HIPCHK(hipGetLastError());
    }
    HIPCHK(hipStreamSynchronize(st));
    std::memcpy(y, ctx->y_pin, n_out * sizeof(double));
  } else if (!on_device) {
    HIPCHK(hipMemcpyAsync(y, ctx->y_stage, n_out * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
  }
  return BW_OK;
}

// Device address of `scratch` on each GPU (index: device ordinal), taken
// once per device by noalloc_bind with that device current; nullptr until
// then, or if hipGetSymbolAddress failed there (noalloc_err holds why).
std::mutex g_noalloc_mu;
std::vector<void*> g_noalloc_ptr;
std::vector<std::string> g_noalloc_err;

// Called by every create on its device (current).  A failure only disables
// bw_hip_matvec_noalloc on that device; the other entry points never use
// the array.
void noalloc_bind(int device) {
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (static_cast<int>(g_noalloc_ptr.size()) <= device) {
    g_noalloc_ptr.resize(device + 1, nullptr);
    g_noalloc_err.resize(device + 1);
  }
  if (g_noalloc_ptr[device]) return;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    (void)hipGetLastError();  // handled: only this entry point is lost
    g_noalloc_err[device] = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
    return;
  }
  g_noalloc_ptr[device] = p;
}

int noalloc_matvec(bw_hip_handle* hd, const double* x, double* y, int ordering, int precision,
                   void* stream) {
  if (!hd || !x || !y) return fail(BW_EINVAL, "matvec_noalloc: null argument");
  if (ordering != BW_ORDER_PERMUTED && ordering != BW_ORDER_ORIGINAL)
    return fail(BW_EINVAL, "matvec_noalloc: ordering must be 0 (permuted) or 1 (original)");
  if (precision != BW_PREC_FP64 && precision != BW_PREC_FP32)
    return fail(BW_EINVAL, "matvec_noalloc: precision must be BW_PREC_FP64 or BW_PREC_FP32");
  if (hd->sel.on) return fail(BW_ENOTSUP, "matvec_noalloc: not available on a selection");
  const int f32 = precision == BW_PREC_FP32 ? 1 : 0;
  DevOp& op = hd->op[0][f32];
  if (!op.present) return fail(BW_ENOTSUP, "matvec_noalloc: precision not built for this handle");
  // xt, then the partial sums of pass 1 and pass 2, each 256-byte aligned
  const auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  const int64_t off1 = up(op.xt_size * op.elem);
  const int64_t off2 = off1 + up(op.p1.single.scratch_bytes(1, op.elem));
  const int64_t need = off2 + up(op.p2.single.scratch_bytes(1, op.elem));
  int64_t limit = BW_NOALLOC_SCRATCH_BYTES;
  if (const char* e = std::getenv("BWHIP_NOALLOC_LIMIT")) {
    const long long v = std::atoll(e);
    if (v > 0 && v < limit) limit = v;  // tests of the size check may only lower it
  }
  if (need > limit)
    return fail(BW_ESHAPE, "matvec_noalloc: this operator needs " + std::to_string(need) +
                               " bytes of scratch; the fixed array holds " + std::to_string(limit) +
                               " (use bw_hip_matvec)");
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (hd->device < static_cast<int>(g_noalloc_ptr.size())) base = g_noalloc_ptr[hd->device];
    if (!base)
      return fail(BW_EHIP, "matvec_noalloc: no scratch address on this device: " +
                               (hd->device < static_cast<int>(g_noalloc_err.size())
                                    ? g_noalloc_err[hd->device]
                                    : std::string("not bound")));
  }
  std::lock_guard<std::mutex> lock(hd->mu);
  hipStream_t st = static_cast<hipStream_t>(stream);
  HIPCHK(hipSetDevice(hd->device));
  unsigned char* b = static_cast<unsigned char*>(base);
  OpScratch s;
  s.xt = b;
  s.part[0] = b + off1;
  s.part[1] = b + off2;
  // Padded column groups read xt past x (the gap) and past t (the tail), so
  // those must hold zeros; an earlier call on this GPU may have left other
  // values there.  x and t are rewritten by every call, and every partial
  // sum is written before it is read; the split slabs' counters start at zero.
  // A fill kernel, not hipMemsetAsync,
  // so the call can be captured into a graph.
  const int64_t na = op.xt_t - op.n_in, nb = op.xt_size - (op.xt_t + op.t_total);
  const DevItems &d1 = op.p1.single, &d2 = op.p2.single;
  int32_t* const c1 = d1.counters(s.part[0], 1, op.elem);
  int32_t* const c2 = d2.counters(s.part[1], 1, op.elem);
  const int zblocks = static_cast<int>((na + nb + d1.ncount + d2.ncount + 255) / 256);
  if (zblocks > 0) {
    if (f32)
      hipLaunchKernelGGL(k_zero_ranges<float>, dim3(zblocks), dim3(256), 0, st,
                         static_cast<float*>(s.xt), op.n_in, op.xt_t, op.xt_t + op.t_total,
                         op.xt_size, c1, d1.ncount, c2, d2.ncount);
    else
      hipLaunchKernelGGL(k_zero_ranges<double>, dim3(zblocks), dim3(256), 0, st,
                         static_cast<double*>(s.xt), op.n_in, op.xt_t, op.xt_t + op.t_total,
                         op.xt_size, c1, d1.ncount, c2, d2.ncount);
  }
  return f32 ? launch_matvec<float>(hd, op, s, nullptr, x, y, ordering, st, nullptr, false)
             : launch_matvec<double>(hd, op, s, nullptr, x, y, ordering, st, nullptr, false);
}

}  // namespace

extern "C" {

int bw_hip_matvec_noalloc(bw_hip_handle* hd, const double* x, double* y, int ordering,
                          int precision, void* stream) {
  return noalloc_matvec(hd, x, y, ordering, precision, stream);
}

const char* bw_hip_last_error(void) { return g_err.c_str(); }

int bw_hip_set_tuning(int64_t wi64, int64_t wi32) {
  if (wi64 < 0 || wi32 < 0) return fail(BW_EINVAL, "set_tuning: negative size");
  g_wi_bytes64 = wi64;
  g_wi_bytes32 = wi32;
  return BW_OK;
}

int bw_hip_set_fp32_rank_tolerance(double rel_tol) {
  if (!(rel_tol >= 0.0) || !(rel_tol < 1.0))
    return fail(BW_EINVAL, "set_fp32_rank_tolerance: tolerance must be in [0, 1)");
  g_fp32_rank_tol = rel_tol;
  return BW_OK;
}

int bw_hip_entries(bw_hip_handle* hd, int precision, int64_t* e_full, int64_t* e_left,
                   int64_t* e_right, int64_t* total_rank) {
  if (!hd) return fail(BW_EINVAL, "entries: null handle");
  if (precision != BW_PREC_FP64 && precision != BW_PREC_FP32)
    return fail(BW_EINVAL, "entries: precision must be BW_PREC_FP64 or BW_PREC_FP32");
  const int64_t* e = hd->entries[precision == BW_PREC_FP32 ? 1 : 0];
  if (e_full) *e_full = e[0];
  if (e_left) *e_left = e[1];
  if (e_right) *e_right = e[2];
  if (total_rank) *total_rank = e[3];
  return BW_OK;
}

int bw_hip_set_stacking(int stack_rows) {
  if (stack_rows < 0 || stack_rows > 64) return fail(BW_EINVAL, "set_stacking: rows must be 0-64");
  g_stack_rows = stack_rows;
  return BW_OK;
}

void bw_hip_destroy(bw_hip_handle* hd) {
  if (!hd) return;
  (void)hipSetDevice(hd->device);
  (void)hipDeviceSynchronize();
  for (auto& c : hd->ctxs) free_ctx(c.get());
  for (void* p : hd->allocs) (void)hipFree(p);
  for (auto& set : hd->evs)
    for (auto& e : set)
      if (e) (void)hipEventDestroy(e);
  delete hd;
}

}  // extern "C"

namespace bwl {
int compose_flat(const bw_flat_hmat* const* hs, int n, bw_flat_composite* c, std::string* msg);
}

namespace {

// The null stream's single-vector scratch and staging, allocated up front
// (most callers use that stream; other streams get theirs on first use).
int prepare_null_stream(bw_hip_handle* hd) {
  StreamCtx* ctx0 = stream_ctx(hd, nullptr);
  int rc;
  for (int adj = 0; adj < 2; ++adj)
    for (int f32 = 0; f32 < 2; ++f32)
      if (hd->op[adj][f32].present && (rc = ensure_op_scratch(hd, ctx0, adj, f32, false))) return rc;
  return ensure_ctx_vectors(hd, ctx0, true);
}

int create_impl(const bw_flat_hmat* h, long double expected_area, int precision_mask, int flags,
                int device, bw_hip_handle** out, bool prepare_ctx0 = true) {
  if (!out) return fail(BW_EINVAL, "create: null output pointer");
  *out = nullptr;
  std::string msg;
  int rc = bwl::validate_flat(h, &msg, expected_area);
  if (rc) return fail(rc, "create: " + msg);
  if ((precision_mask & (BW_PREC_FP64 | BW_PREC_FP32)) == 0 ||
      (precision_mask & ~(BW_PREC_FP64 | BW_PREC_FP32)))
    return fail(BW_EINVAL, "create: precision_mask must combine BW_PREC_FP64 / BW_PREC_FP32");
  if (flags & ~BW_FLAG_ADJOINT) return fail(BW_EINVAL, "create: unknown flag");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return fail(BW_EHIP, "create: no HIP device available");
  auto* hd = new bw_hip_handle();
  if (device < 0) {
    if (hipGetDevice(&hd->device) != hipSuccess) hd->device = 0;
  } else {
    hd->device = device;
  }
  auto cleanup = [&](int code) {
    bw_hip_destroy(hd);
    return code;
  };
  if (hipSetDevice(hd->device) != hipSuccess) return cleanup(fail(BW_EHIP, "create: hipSetDevice"));
  noalloc_bind(hd->device);  // once per device: the address of bw_hip_matvec_noalloc's array
  hd->dof = h->dof;
  hd->n_row_pts = h->n_row_pts;
  hd->n_col_pts = h->n_col_pts;
  const int64_t d = h->dof;
  auto dmal = [&](void** p, size_t bytes) -> int { return dev_alloc(p, bytes, &hd->allocs, "create"); };
  if ((rc = dmal(reinterpret_cast<void**>(&hd->perm0), h->n_row_pts * sizeof(int64_t)))) return cleanup(rc);
  if ((rc = dmal(reinterpret_cast<void**>(&hd->perm1), h->n_col_pts * sizeof(int64_t)))) return cleanup(rc);
  hd->stage_elems = d * std::max(h->n_row_pts, h->n_col_pts);
  if (hipMemcpy(hd->perm0, h->perm0, h->n_row_pts * sizeof(int64_t), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(hd->perm1, h->perm1, h->n_col_pts * sizeof(int64_t), hipMemcpyHostToDevice) != hipSuccess)
    return cleanup(fail(BW_EHIP, "create: permutation upload"));
  // the FP32 copy may stream recompressed low-rank factors
  bwl::RecompressedFlat rf;
  const bw_flat_hmat* h32 = h;
  hd->fp32_rank_tol = g_fp32_rank_tol.load();
  if ((precision_mask & BW_PREC_FP32) && hd->fp32_rank_tol > 0.0) {
    std::string rmsg;
    if ((rc = bwl::recompress_flat(h, hd->fp32_rank_tol, &rf, &rmsg, expected_area)))
      return cleanup(fail(rc, "create: recompression: " + rmsg));
    h32 = &rf.flat;
  }
  for (int f32 = 0; f32 < 2; ++f32) {
    const bw_flat_hmat* hp = f32 ? h32 : h;
    int64_t* e = hd->entries[f32];
    for (int64_t k = 0; k < hp->n_fr; ++k) {
      const int64_t* c = hp->fr_pattern + 6 * k;
      e[0] += d * (c[3] - c[1]) * d * (c[4] - c[2]);
    }
    for (int64_t k = 0; k < hp->n_lr; ++k) {
      const int64_t* c = hp->lr_pattern + 6 * k;
      e[1] += d * (c[3] - c[1]) * c[5];
      e[2] += c[5] * d * (c[4] - c[2]);
      e[3] += c[5];
    }
  }
  hipStream_t st;
  if (hipStreamCreate(&st) != hipSuccess) return cleanup(fail(BW_EHIP, "create: hipStreamCreate"));
  for (int adj = 0; adj < 2; ++adj) {
    if (adj && !(flags & BW_FLAG_ADJOINT)) continue;
    if (precision_mask & BW_PREC_FP64) {
      rc = build_op<double>(hd, h, adj != 0, st);
      if (rc) {
        (void)hipStreamDestroy(st);
        return cleanup(rc);
      }
    }
    if (precision_mask & BW_PREC_FP32) {
      rc = build_op<float>(hd, h32, adj != 0, st);
      if (rc) {
        (void)hipStreamDestroy(st);
        return cleanup(rc);
      }
    }
  }
  (void)hipStreamDestroy(st);
  // nbOfEntries (hmat.cc:299-312)
  int64_t E = 0;
  for (int64_t k = 0; k < h->n_fr; ++k) {
    const int64_t* c = h->fr_pattern + 6 * k;
    E += d * (c[3] - c[1]) * d * (c[4] - c[2]);
  }
  for (int64_t k = 0; k < h->n_lr; ++k) {
    const int64_t* c = h->lr_pattern + 6 * k;
    E += d * (c[3] - c[1]) * c[5] + c[5] * d * (c[4] - c[2]);
  }
  hd->nb_entries = E;
  compute_diagonal(hd, h);
  for (auto& set : hd->evs)
    for (auto& e : set)
      if (hipEventCreate(&e) != hipSuccess) return cleanup(fail(BW_EHIP, "create: hipEventCreate"));
  if (prepare_ctx0 && (rc = prepare_null_stream(hd))) return cleanup(rc);
  *out = hd;
  return BW_OK;
}

}  // namespace

// A captured matvec.  It owns its scratch, so replays never race with
// eager calls on the handle (two replays of one graph must be ordered).
struct bw_hip_graph {
  int device = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  StreamCtx ctx;
};

extern "C" {

int bw_hip_create(const bw_flat_hmat* h, int precision_mask, int flags, int device,
                  bw_hip_handle** out) {
  arm_alloc_hook();
  return create_impl(h, -1.0L, precision_mask, flags, device, out);
}

int bw_hip_create_multi(const bw_flat_hmat* const* hs, int n_mats, int precision_mask, int flags,
                        int device, bw_hip_handle** out, int64_t* row_off, int64_t* col_off) {
  if (!out) return fail(BW_EINVAL, "create_multi: null output pointer");
  *out = nullptr;
  arm_alloc_hook();
  bw_flat_composite* c = nullptr;
  int rc = bw_flat_compose(hs, n_mats, &c);
  if (rc) return fail(rc, std::string("create_multi: ") + bw_flat_compose_last_error());
  const bw_flat_hmat* f = bw_flat_composite_view(c);
  long double area = 0.0L;
  for (int m = 0; m < n_mats; ++m)
    area += static_cast<long double>(hs[m]->n_row_pts) * hs[m]->n_col_pts;
  rc = create_impl(f, area, precision_mask, flags, device, out);
  if (!rc) bw_flat_composite_offsets(c, row_off, col_off);
  bw_flat_composite_free(c);
  return rc;
}

int bw_hip_create_selection(const bw_flat_hmat* h, const int64_t* rows, int64_t n_rows,
                            const int64_t* cols, int64_t n_cols, int ordering,
                            int precision_mask, int flags, int device, bw_hip_handle** out) {
  if (!out) return fail(BW_EINVAL, "create_selection: null output pointer");
  *out = nullptr;
  arm_alloc_hook();
  std::string msg;
  int rc = bwl::validate_flat(h, &msg);
  if (rc) return fail(rc, "create_selection: " + msg);
  if (!rows || !cols || n_rows <= 0 || n_cols <= 0)
    return fail(BW_EINVAL, "create_selection: empty row or column selection");
  if (ordering != BW_ORDER_PERMUTED && ordering != BW_ORDER_ORIGINAL)
    return fail(BW_EINVAL, "create_selection: ordering must be 0 (permuted) or 1 (original)");
  for (int64_t i = 0; i < n_rows; ++i)
    if (rows[i] < 0 || rows[i] >= h->n_row_pts)
      return fail(BW_EINVAL, "create_selection: row index out of bounds");
  for (int64_t i = 0; i < n_cols; ++i)
    if (cols[i] < 0 || cols[i] >= h->n_col_pts)
      return fail(BW_EINVAL, "create_selection: column index out of bounds");
  // selected points in the permuted numbering (HmatSelection::blockSelection,
  // hmat_selection.cc:44-77): the inverse permutation for original indices
  std::vector<int64_t> inv0(h->n_row_pts), inv1(h->n_col_pts);
  for (int64_t i = 0; i < h->n_row_pts; ++i) inv0[h->perm0[i]] = i;
  for (int64_t i = 0; i < h->n_col_pts; ++i) inv1[h->perm1[i]] = i;
  const bool orig = ordering == BW_ORDER_ORIGINAL;
  std::vector<int64_t> prow(n_rows), pcol(n_cols);
  for (int64_t i = 0; i < n_rows; ++i) prow[i] = orig ? inv0[rows[i]] : rows[i];
  for (int64_t i = 0; i < n_cols; ++i) pcol[i] = orig ? inv1[cols[i]] : cols[i];
  // prefix counts of marked points: a block is kept if its row range holds a
  // selected row and its column range a selected column (hmat_selection.cc:82-128)
  std::vector<int64_t> rcnt(h->n_row_pts + 1, 0), ccnt(h->n_col_pts + 1, 0);
  {
    std::vector<char> mr(h->n_row_pts, 0), mc(h->n_col_pts, 0);
    for (int64_t p : prow) mr[p] = 1;
    for (int64_t p : pcol) mc[p] = 1;
    for (int64_t i = 0; i < h->n_row_pts; ++i) rcnt[i + 1] = rcnt[i] + mr[i];
    for (int64_t i = 0; i < h->n_col_pts; ++i) ccnt[i + 1] = ccnt[i] + mc[i];
  }
  auto keep = [&](const int64_t* c) {
    return rcnt[c[3]] > rcnt[c[1]] && ccnt[c[4]] > ccnt[c[2]];
  };
  std::vector<int64_t> fr_pat, lr_pat;
  std::vector<const double*> fr_ptr, lr_a, lr_b;
  long double area = 0.0L;
  for (int64_t k = 0; k < h->n_fr; ++k) {
    const int64_t* c = h->fr_pattern + 6 * k;
    if (!keep(c)) continue;
    fr_pat.insert(fr_pat.end(), c, c + 6);
    fr_ptr.push_back(h->fr_blocks[k]);
    area += static_cast<long double>(c[3] - c[1]) * (c[4] - c[2]);
  }
  for (int64_t k = 0; k < h->n_lr; ++k) {
    const int64_t* c = h->lr_pattern + 6 * k;
    if (!keep(c)) continue;
    lr_pat.insert(lr_pat.end(), c, c + 6);
    lr_a.push_back(h->lr_A[k]);
    lr_b.push_back(h->lr_B[k]);
    area += static_cast<long double>(c[3] - c[1]) * (c[4] - c[2]);
  }
  bw_flat_hmat sub = *h;
  sub.n_fr = static_cast<int64_t>(fr_ptr.size());
  sub.fr_pattern = sub.n_fr ? fr_pat.data() : nullptr;
  sub.fr_blocks = sub.n_fr ? fr_ptr.data() : nullptr;
  sub.n_lr = static_cast<int64_t>(lr_a.size());
  sub.lr_pattern = sub.n_lr ? lr_pat.data() : nullptr;
  sub.lr_A = sub.n_lr ? lr_a.data() : nullptr;
  sub.lr_B = sub.n_lr ? lr_b.data() : nullptr;
  bw_hip_handle* hd = nullptr;
  rc = create_impl(&sub, area, precision_mask, flags, device, &hd, false);
  if (rc) return rc;
  // scatter pairs with repeated targets reduced to the last occurrence, as
  // HmatSelection::matvec overwrites x_full (hmat_selection.cc:197-205)
  auto pairs = [](const std::vector<int64_t>& dst, std::vector<int64_t>* s, std::vector<int64_t>* d) {
    std::vector<int64_t> order(dst.size());
    for (size_t i = 0; i < dst.size(); ++i) order[i] = static_cast<int64_t>(i);
    std::stable_sort(order.begin(), order.end(),
                     [&](int64_t a, int64_t b) { return dst[a] < dst[b]; });
    for (size_t k = 0; k < order.size(); ++k)
      if (k + 1 == order.size() || dst[order[k + 1]] != dst[order[k]]) {
        s->push_back(order[k]);
        d->push_back(dst[order[k]]);
      }
  };
  auto up = [&](const std::vector<int64_t>& v, int64_t** dp) -> int {
    int rc1 = dev_alloc(reinterpret_cast<void**>(dp), v.size() * sizeof(int64_t), &hd->allocs,
                        "create_selection");
    if (rc1) return rc1;
    if (!v.empty() &&
        hipMemcpy(*dp, v.data(), v.size() * sizeof(int64_t), hipMemcpyHostToDevice) != hipSuccess)
      return fail(BW_EHIP, "create_selection: upload");
    return BW_OK;
  };
  const std::vector<int64_t>* in_of[2] = {&pcol, &prow};
  const std::vector<int64_t>* out_of[2] = {&prow, &pcol};
  for (int dir = 0; dir < 2; ++dir) {
    SelDir& sd = hd->sel.dir[dir];
    std::vector<int64_t> s_src, s_dst;
    pairs(*in_of[dir], &s_src, &s_dst);
    if ((rc = up(s_src, &sd.in_src)) || (rc = up(s_dst, &sd.in_dst)) ||
        (rc = up(*out_of[dir], &sd.out_dst))) {
      bw_hip_destroy(hd);
      return rc;
    }
    sd.n_pairs = static_cast<int64_t>(s_src.size());
    sd.n_in = static_cast<int64_t>(in_of[dir]->size());
    sd.n_out = static_cast<int64_t>(out_of[dir]->size());
  }
  // every stream's scratch holds the full permuted output of the selected
  // blocks; host-pointer staging must hold the selection vectors, which
  // repeated indices can make longer than the full ones
  const int64_t nfull = h->dof * std::max(h->n_row_pts, h->n_col_pts);
  hd->yfull_elems = nfull;
  hd->stage_elems = std::max(nfull, h->dof * std::max(n_rows, n_cols));
  if ((rc = prepare_null_stream(hd))) {
    bw_hip_destroy(hd);
    return rc;
  }
  hd->sel.on = true;
  hd->sel.ordering = ordering;
  hd->n_row_pts = n_rows;
  hd->n_col_pts = n_cols;
  *out = hd;
  return BW_OK;
}

int bw_hip_matvec(bw_hip_handle* hd, const double* x, double* y, int ordering, int precision,
                  int on_device, void* stream) {
  return do_matvec(hd, false, x, y, ordering, precision, on_device, stream);
}

int bw_hip_rmatvec(bw_hip_handle* hd, const double* x, double* y, int ordering, int precision,
                   int on_device, void* stream) {
  return do_matvec(hd, true, x, y, ordering, precision, on_device, stream);
}

}  // extern "C"

namespace {

// Checks of the batched entry points; on success *op is the operator used.
// X(i, j) = X[i * xr + j * xc] (input index i, right-hand side j); Y likewise
// with (yr, yc).  Column-major is (1, ld), row-major (nrhs, 1).
int check_batched(bw_hip_handle* hd, bool adjoint, int nrhs, const double* X, int64_t xr,
                  int64_t xc, const double* Y, int64_t yr, int64_t yc, int ordering, int precision,
                  bool leading_dims, DevOp** op_out) {
  if (!hd || !X || !Y || nrhs <= 0) return fail(BW_EINVAL, "matvec_batched: bad argument");
  if (xr < 1 || xc < 1 || yr < 1 || yc < 1)
    return fail(BW_ESHAPE, "matvec_batched: strides must be positive");
  if (hd->sel.on) return fail(BW_ENOTSUP, "matvec_batched: not available for a selection");
  if (ordering != BW_ORDER_PERMUTED && ordering != BW_ORDER_ORIGINAL)
    return fail(BW_EINVAL, "matvec_batched: bad ordering");
  if (precision != BW_PREC_FP64 && precision != BW_PREC_FP32)
    return fail(BW_EINVAL, "matvec_batched: bad precision");
  DevOp& op = hd->op[adjoint ? 1 : 0][precision == BW_PREC_FP32 ? 1 : 0];
  if (!op.present)
    return fail(BW_ENOTSUP, adjoint ? "rmatvec_batched: adjoint / precision not built"
                                    : "matvec_batched: precision not built");
  if (leading_dims && (xc < op.n_in || yc < op.n_out))
    return fail(BW_ESHAPE, "matvec_batched: leading dimension too small");
  // the MFMA kernels index the 32-wide input rows with 32-bit offsets
  if (op.xt_size * 32 > static_cast<int64_t>(UINT32_MAX))
    return fail(BW_ESHAPE, "matvec_batched: input plus rank entries exceed 2^32 / 32");
  // distinct outputs must not share an address: columns apart by at least a
  // column's extent, or rows apart by at least a row's
  if (!(yc >= op.n_out * yr || yr >= static_cast<int64_t>(nrhs) * yc))
    return fail(BW_ESHAPE, "matvec_batched: output strides overlap");
  *op_out = &op;
  return BW_OK;
}

// The MFMA kernel of one pass of a round of NB columns, and the reduction of
// its split slabs if that is a launch of its own.
template <int PASS, int NB, typename T>
void launch_batched_pass(const DevPass& dp, hipStream_t st, const T* xb, void* part, int cols,
                         BatchOut<T> o) {
  const bool wide = PASS == 1 && NB == 64 && dp.rowtab;
  const DevItems& di = wide ? dp.wide : dp.batched;
  if (wide) part = static_cast<unsigned char*>(part) + dp.wide_offset(cols, sizeof(T));
  o.part = static_cast<T*>(part);
  o.sp = di.sums(part, cols, sizeof(T));
  const dim3 grid(di.blocks), block(64 * kBatchWaves);
  const T* data = static_cast<const T*>(dp.data);
  if (di.nwi > 0) {
#define BW_MFMA32(WIN)                                                                           \
  hipLaunchKernelGGL((k_slab_mfma32<PASS, NB / 32, kBatchWaves, WIN>), grid, block, 0, st, di.wis, \
                     di.xs, dp.gidx, data, xb, dp.rowtab, o)
    if constexpr (sizeof(T) == 4 && NB >= 32) {
      if constexpr (PASS == 1 && NB == 64) {
        if (wide)
          BW_MFMA32(true);
        else
          BW_MFMA32(false);
      } else {
        BW_MFMA32(false);
      }
    } else {
      hipLaunchKernelGGL((k_slab_mfma16<T, PASS, NB / 16, kBatchWaves>), grid, block, 0, st, di.wis,
                         di.xs, dp.gidx, data, xb, o);
    }
#undef BW_MFMA32
  }
  if (di.reduce_launch())
    hipLaunchKernelGGL((k_reduce_b<PASS, NB, T>), dim3(di.nred), dim3(256), 0, st, di.reds,
                       di.nred, o);
}

// One round: columns 0 .. nk - 1 (nk <= NB) of X and Y, writing only the
// batched scratch `s`.
template <typename T, int NB>
int launch_round(bw_hip_handle* hd, const DevOp& op, const OpScratch& s, int nk, const double* X,
                 int64_t xr, int64_t xc, double* Y, int64_t yr, int64_t yc, bool orig,
                 hipStream_t st) {
  const int dof = hd->dof;
  const int64_t* pin = orig ? op.perm_in : nullptr;
  T* xb = static_cast<T*>(s.xb);
  const GatherRows g{op.n_in, op.xt_t, op.xt_t + op.t_total, op.xt_size};
  // row-major input (unit column stride, even row stride, 16-byte aligned
  // rows): the vector gather
  const bool rowmajor = xc == 1 && xr % 2 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0;
  const int rows = rowmajor ? 256 / (NB / 4) : 256 / NB;  // per workgroup
  const dim3 gblocks(static_cast<unsigned>((g.count() + rows - 1) / rows));
  if (rowmajor)
    hipLaunchKernelGGL((k_gather_b4<T, NB>), gblocks, dim3(256), 0, st, X, xr, nk, xb, g, pin, dof);
  else
    hipLaunchKernelGGL((k_gather_b<T, NB>), gblocks, dim3(256), 0, st, X, xr, xc, nk, xb, g, pin,
                       dof);
  BatchOut<T> o1{};
  o1.tout = xb;
  o1.nk = NB;
  o1.dof = dof;
  o1.rowmap = op.p1.rowmap;
  BatchOut<T> o2{};
  o2.Y = Y;
  o2.yr = yr;
  o2.yc = yc;
  o2.nk = nk;
  o2.yvec = yc == 1 && yr % 2 == 0 && reinterpret_cast<uintptr_t>(Y) % 16 == 0;
  o2.perm = orig ? op.perm_out : nullptr;
  o2.dof = dof;
  launch_batched_pass<1, NB>(op.p1, st, xb, s.partb[0], s.xb_cols, o1);
  launch_batched_pass<2, NB>(op.p2, st, xb, s.partb[1], s.xb_cols, o2);
  HIPCHK(hipGetLastError());
  return BW_OK;
}

// Y = H X on stream st in rounds of 64 (FP32), 32 or 16 columns.
template <typename T>
int launch_batched(bw_hip_handle* hd, const DevOp& op, const OpScratch& s, int nrhs,
                   const double* X, int64_t xr, int64_t xc, double* Y, int64_t yr, int64_t yc,
                   int ordering, hipStream_t st) {
  const bool orig = ordering == BW_ORDER_ORIGINAL;
  for (int k0 = 0; k0 < nrhs;) {
    const int left = nrhs - k0;
    const double* Xk = X + static_cast<int64_t>(k0) * xc;
    double* Yk = Y + static_cast<int64_t>(k0) * yc;
    int rc, nk;
    if (sizeof(T) == 4 && left > 32 && s.xb_cols >= 64) {
      nk = std::min(64, left);
      rc = launch_round<float, 64>(hd, op, s, nk, Xk, xr, xc, Yk, yr, yc, orig, st);
    } else if (left > 16) {
      nk = std::min(32, left);
      rc = launch_round<T, 32>(hd, op, s, nk, Xk, xr, xc, Yk, yr, yc, orig, st);
    } else {
      nk = left;
      rc = launch_round<T, 16>(hd, op, s, nk, Xk, xr, xc, Yk, yr, yc, orig, st);
    }
    if (rc) return rc;
    k0 += nk;
  }
  return BW_OK;
}

int batched_impl(bw_hip_handle* hd, bool adjoint, int nrhs, const double* X, int64_t xr,
                 int64_t xc, double* Y, int64_t yr, int64_t yc, int ordering, int precision,
                 void* stream, bool leading_dims = false) {
  DevOp* op = nullptr;
  int rc = check_batched(hd, adjoint, nrhs, X, xr, xc, Y, yr, yc, ordering, precision,
                         leading_dims, &op);
  if (rc) return rc;
  std::lock_guard<std::mutex> lock(hd->mu);
  arm_alloc_hook();
  HIPCHK(hipSetDevice(hd->device));
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int adj = adjoint ? 1 : 0, f32 = precision == BW_PREC_FP32 ? 1 : 0;
  StreamCtx* ctx = stream_ctx(hd, st);
  if ((rc = ensure_op_scratch(hd, ctx, adj, f32, true))) return rc;
  const OpScratch& s = ctx->op[adj][f32];
  return f32 ? launch_batched<float>(hd, *op, s, nrhs, X, xr, xc, Y, yr, yc, ordering, st)
             : launch_batched<double>(hd, *op, s, nrhs, X, xr, xc, Y, yr, yc, ordering, st);
}

// Captures launch(stream, ctx) on a private stream into a new graph that owns
// ctx (already holding its scratch).  Caller holds hd->mu.
template <typename F>
int capture_graph(bw_hip_handle* hd, std::unique_ptr<bw_hip_graph> g, F launch,
                  bw_hip_graph** out) {
  hipStream_t cs;
  const hipError_t ec = hipStreamCreateWithFlags(&cs, hipStreamNonBlocking);
  if (ec != hipSuccess) {
    free_ctx(&g->ctx);
    return fail(BW_EHIP, std::string("graph_create: ") + hipGetErrorString(ec));
  }
  const bool timing = hd->timing;
  hd->timing = false;  // no event records inside the graph
  hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
  int rc = BW_OK;
  hipGraph_t graph = nullptr;
  if (e == hipSuccess) {
    rc = launch(cs, g->ctx);
    hipError_t e2 = hipStreamEndCapture(cs, &graph);
    if (!rc && e2 != hipSuccess) rc = fail(BW_EHIP, std::string("graph_create: ") + hipGetErrorString(e2));
  } else {
    rc = fail(BW_EHIP, std::string("graph_create: ") + hipGetErrorString(e));
  }
  hd->timing = timing;
  (void)hipStreamDestroy(cs);
  if (!rc) {
    g->graph = graph;
    e = hipGraphInstantiate(&g->exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) rc = fail(BW_EHIP, std::string("graph_create: instantiate: ") + hipGetErrorString(e));
  }
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    free_ctx(&g->ctx);
    return rc;
  }
  *out = g.release();
  return BW_OK;
}

}  // namespace

extern "C" {

int bw_hip_graph_create(bw_hip_handle* hd, const double* x, double* y, int ordering,
                        int precision, int adjoint, bw_hip_graph** out) {
  if (!hd || !x || !y || !out) return fail(BW_EINVAL, "graph_create: null argument");
  *out = nullptr;
  if (ordering != BW_ORDER_PERMUTED && ordering != BW_ORDER_ORIGINAL)
    return fail(BW_EINVAL, "graph_create: ordering must be 0 (permuted) or 1 (original)");
  if (precision != BW_PREC_FP64 && precision != BW_PREC_FP32)
    return fail(BW_EINVAL, "graph_create: precision must be BW_PREC_FP64 or BW_PREC_FP32");
  const int adj = adjoint ? 1 : 0, f32 = precision == BW_PREC_FP32 ? 1 : 0;
  DevOp& op = hd->op[adj][f32];
  if (!op.present) return fail(BW_ENOTSUP, "graph_create: adjoint / precision not built");
  const SelDir* sd = hd->sel.on ? &hd->sel.dir[adj] : nullptr;
  if (sd && ordering != hd->sel.ordering)
    return fail(BW_ENOTSUP, "graph_create: this selection was created for the other ordering");
  std::lock_guard<std::mutex> lock(hd->mu);
  arm_alloc_hook();
  HIPCHK(hipSetDevice(hd->device));
  std::unique_ptr<bw_hip_graph> g(new bw_hip_graph());
  g->device = hd->device;
  int rc;
  if ((rc = ensure_op_scratch(hd, &g->ctx, adj, f32, false)) ||
      (rc = ensure_ctx_vectors(hd, &g->ctx, false))) {
    free_ctx(&g->ctx);
    return rc;
  }
  return capture_graph(hd, std::move(g), [&](hipStream_t cs, StreamCtx& ctx) {
    const OpScratch& s = ctx.op[adj][f32];
    return f32 ? launch_matvec<float>(hd, op, s, ctx.y_full, x, y, ordering, cs, sd)
               : launch_matvec<double>(hd, op, s, ctx.y_full, x, y, ordering, cs, sd);
  }, out);
}

int bw_hip_graph_create_batched(bw_hip_handle* hd, int adjoint, int nrhs, const double* X,
                                int64_t x_row_stride, int64_t x_col_stride, double* Y,
                                int64_t y_row_stride, int64_t y_col_stride, int ordering,
                                int precision, bw_hip_graph** out) {
  if (!out) return fail(BW_EINVAL, "graph_create_batched: null argument");
  *out = nullptr;
  DevOp* op = nullptr;
  int rc = check_batched(hd, adjoint != 0, nrhs, X, x_row_stride, x_col_stride, Y, y_row_stride,
                         y_col_stride, ordering, precision, false, &op);
  if (rc) return rc;
  std::lock_guard<std::mutex> lock(hd->mu);
  arm_alloc_hook();
  HIPCHK(hipSetDevice(hd->device));
  const int adj = adjoint ? 1 : 0, f32 = precision == BW_PREC_FP32 ? 1 : 0;
  std::unique_ptr<bw_hip_graph> g(new bw_hip_graph());
  g->device = hd->device;
  if ((rc = ensure_op_scratch(hd, &g->ctx, adj, f32, true))) {
    free_ctx(&g->ctx);
    return rc;
  }
  return capture_graph(hd, std::move(g), [&](hipStream_t cs, StreamCtx& ctx) {
    const OpScratch& s = ctx.op[adj][f32];
    return f32 ? launch_batched<float>(hd, *op, s, nrhs, X, x_row_stride, x_col_stride, Y,
                                       y_row_stride, y_col_stride, ordering, cs)
               : launch_batched<double>(hd, *op, s, nrhs, X, x_row_stride, x_col_stride, Y,
                                        y_row_stride, y_col_stride, ordering, cs);
  }, out);
}

int bw_hip_graph_launch(bw_hip_graph* g, void* stream) {
  if (!g) return fail(BW_EINVAL, "graph_launch: null graph");
  HIPCHK(hipSetDevice(g->device));
  HIPCHK(hipGraphLaunch(g->exec, static_cast<hipStream_t>(stream)));
  return BW_OK;
}

void bw_hip_graph_destroy(bw_hip_graph* g) {
  if (!g) return;
  (void)hipSetDevice(g->device);
  (void)hipDeviceSynchronize();
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  free_ctx(&g->ctx);
  delete g;
}

int bw_hip_stream_release(bw_hip_handle* hd, void* stream) {
  if (!hd) return fail(BW_EINVAL, "stream_release: null handle");
  std::lock_guard<std::mutex> lock(hd->mu);
  HIPCHK(hipSetDevice(hd->device));
  hipStream_t st = static_cast<hipStream_t>(stream);
  for (size_t i = 0; i < hd->ctxs.size(); ++i) {
    if (hd->ctxs[i]->stream != st) continue;
    HIPCHK(hipStreamSynchronize(st));
    free_ctx(hd->ctxs[i].get());
    hd->ctxs.erase(hd->ctxs.begin() + static_cast<std::ptrdiff_t>(i));
    return BW_OK;
  }
  return BW_OK;
}

int bw_hip_matvec_batched(bw_hip_handle* hd, int nrhs, const double* X, int64_t ldx, double* Y,
                          int64_t ldy, int ordering, int precision, void* stream) {
  return batched_impl(hd, false, nrhs, X, 1, ldx, Y, 1, ldy, ordering, precision, stream, true);
}

int bw_hip_rmatvec_batched(bw_hip_handle* hd, int nrhs, const double* X, int64_t ldx, double* Y,
                           int64_t ldy, int ordering, int precision, void* stream) {
  return batched_impl(hd, true, nrhs, X, 1, ldx, Y, 1, ldy, ordering, precision, stream, true);
}

int bw_hip_matvec_batched_strided(bw_hip_handle* hd, int adjoint, int nrhs, const double* X,
                                  int64_t x_row_stride, int64_t x_col_stride, double* Y,
                                  int64_t y_row_stride, int64_t y_col_stride, int ordering,
                                  int precision, void* stream) {
  return batched_impl(hd, adjoint != 0, nrhs, X, x_row_stride, x_col_stride, Y, y_row_stride,
                      y_col_stride, ordering, precision, stream);
}

int bw_hip_diagonal(bw_hip_handle* hd, double* dg, int ordering) {
  if (!hd || !dg) return fail(BW_EINVAL, "diagonal: null argument");
  if (hd->sel.on) return fail(BW_ENOTSUP, "diagonal: not defined for a selection");
  if (ordering != BW_ORDER_PERMUTED && ordering != BW_ORDER_ORIGINAL)
    return fail(BW_EINVAL, "diagonal: bad ordering");
  const auto& v = ordering == BW_ORDER_ORIGINAL ? hd->diag_orig : hd->diag_perm;
  std::memcpy(dg, v.data(), v.size() * sizeof(double));
  return BW_OK;
}

int bw_hip_sizes(bw_hip_handle* hd, int64_t* n_rows, int64_t* n_cols, int64_t* nb_entries,
                 int64_t* device_bytes, int64_t* sb64, int64_t* sb32) {
  if (!hd) return fail(BW_EINVAL, "sizes: null handle");
  if (n_rows) *n_rows = hd->dof * hd->n_row_pts;
  if (n_cols) *n_cols = hd->dof * hd->n_col_pts;
  if (nb_entries) *nb_entries = hd->nb_entries;
  if (device_bytes) *device_bytes = hd->device_bytes;
  if (sb64) *sb64 = hd->op[0][0].present ? hd->op[0][0].stream_bytes : 0;
  if (sb32) *sb32 = hd->op[0][1].present ? hd->op[0][1].stream_bytes : 0;
  return BW_OK;
}

int bw_hip_set_unroll(bw_hip_handle* hd, int unroll_fp64, int unroll_fp32) {
  if (!hd) return fail(BW_EINVAL, "set_unroll: null handle");
  std::lock_guard<std::mutex> lock(hd->mu);
  for (int u : {unroll_fp64, unroll_fp32})
    if (u != 0 && u != 4 && u != 8 && u != 16)
      return fail(BW_EINVAL, "set_unroll: unroll must be 4, 8 or 16 (0 keeps the current one)");
  for (int adj = 0; adj < 2; ++adj)
    for (int pass = 0; pass < 2; ++pass) {
      if (unroll_fp64) hd->op[adj][0].unroll[pass] = unroll_fp64;
      if (unroll_fp32) hd->op[adj][1].unroll[pass] = unroll_fp32;
    }
  return BW_OK;
}

int bw_hip_set_unroll_pass(bw_hip_handle* hd, int precision_mask, int pass, int unroll) {
  if (!hd) return fail(BW_EINVAL, "set_unroll_pass: null handle");
  std::lock_guard<std::mutex> lock(hd->mu);
  if (pass != 1 && pass != 2) return fail(BW_EINVAL, "set_unroll_pass: pass must be 1 or 2");
  if (unroll != 4 && unroll != 8 && unroll != 16)
    return fail(BW_EINVAL, "set_unroll_pass: unroll must be 4, 8 or 16");
  if (precision_mask <= 0 || (precision_mask & ~(BW_PREC_FP64 | BW_PREC_FP32)))
    return fail(BW_EINVAL, "set_unroll_pass: bad precision mask");
  for (int adj = 0; adj < 2; ++adj) {
    if (precision_mask & BW_PREC_FP64) hd->op[adj][0].unroll[pass - 1] = unroll;
    if (precision_mask & BW_PREC_FP32) hd->op[adj][1].unroll[pass - 1] = unroll;
  }
  return BW_OK;
}

int bw_hip_set_mfma_schedule(bw_hip_handle* hd, int precision_mask, int schedule) {
  if (!hd) return fail(BW_EINVAL, "set_mfma_schedule: null handle");
  std::lock_guard<std::mutex> lock(hd->mu);
  if (schedule < 0 || schedule > 15) return fail(BW_EINVAL, "set_mfma_schedule: schedule must be 0-15");
  if (precision_mask <= 0 || (precision_mask & ~(BW_PREC_FP64 | BW_PREC_FP32)))
    return fail(BW_EINVAL, "set_mfma_schedule: bad precision mask");
  return BW_OK;
}

int bw_hip_set_timing(bw_hip_handle* hd, int enable) {
  if (!hd) return fail(BW_EINVAL, "set_timing: null handle");
  std::lock_guard<std::mutex> lock(hd->mu);
  for (int s = 0; s < 2; ++s)
    if (hd->pending[s]) HIPCHK(hipEventSynchronize(hd->evs[s][5]));
  hd->pending[0] = hd->pending[1] = false;
  hd->cur = 0;
  for (double& v : hd->sum_ms) v = 0.0;
  hd->n_timed = 0;
  hd->timing = enable != 0;
  return BW_OK;
}

int bw_hip_timing_stats(bw_hip_handle* hd, double* avg_ms6, int64_t* count) {
  if (!hd || !avg_ms6) return fail(BW_EINVAL, "timing_stats: null argument");
  std::lock_guard<std::mutex> lock(hd->mu);
  for (int s = 0; s < 2; ++s) {
    const int set = (hd->cur + s) & 1;  // oldest first
    if (hd->pending[set]) {
      int rc = accumulate_timing(hd, set);
      if (rc) return rc;
    }
  }
  for (int i = 0; i < 6; ++i) avg_ms6[i] = hd->n_timed ? hd->sum_ms[i] / hd->n_timed : 0.0;
  if (count) *count = hd->n_timed;
  return BW_OK;
}

}  // extern "C"
