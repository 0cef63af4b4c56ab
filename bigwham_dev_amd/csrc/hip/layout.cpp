// Slab-program construction (see layout.h for the scheme).
#include "layout.h"

#include <algorithm>
#include <climits>
#include <atomic>
#include <cmath>
#include <cstring>
#include <numeric>
#include <string>
#include <thread>

namespace bwl {

#define PAT(p, r, k) ((p)[(r) + 6 * static_cast<int64_t>(k)])

namespace {

int64_t align_up(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

}  // namespace

int validate_flat(const bw_flat_hmat* h, std::string* msg, long double expected_area,
                  bool need_lr_data) {
  if (!h) {
    *msg = "null bw_flat_hmat";
    return BW_EINVAL;
  }
  if (h->dof < 1 || h->dof > 8) {
    *msg = "dof must be in [1, 8]";
    return BW_EINVAL;
  }
  if (h->n_row_pts <= 0 || h->n_col_pts <= 0 || !h->perm0 || !h->perm1) {
    *msg = "empty matrix or missing permutation";
    return BW_EINVAL;
  }
  if (h->n_fr < 0 || h->n_lr < 0 || (h->n_fr > 0 && (!h->fr_pattern || !h->fr_blocks)) ||
      (h->n_lr > 0 && (!h->lr_pattern || (need_lr_data && (!h->lr_A || !h->lr_B))))) {
    *msg = "missing pattern or block pointers";
    return BW_EINVAL;
  }
  const int64_t d = h->dof;
  if (d * h->n_row_pts >= (int64_t(1) << 30) || d * h->n_col_pts >= (int64_t(1) << 30)) {
    *msg = "matrix too large for 32-bit row indices";
    return BW_ESHAPE;
  }
  auto check_perm = [&](const int64_t* p, int64_t n) {
    std::vector<char> seen(n, 0);
    for (int64_t i = 0; i < n; ++i) {
      if (p[i] < 0 || p[i] >= n || seen[p[i]]) return false;
      seen[p[i]] = 1;
    }
    return true;
  };
  if (!check_perm(h->perm0, h->n_row_pts) || !check_perm(h->perm1, h->n_col_pts)) {
    *msg = "permutation is not a bijection";
    return BW_ESHAPE;
  }
  long double area = 0.0L;
  for (int64_t k = 0; k < h->n_fr; ++k) {
    const int64_t i0 = PAT(h->fr_pattern, 1, k), j0 = PAT(h->fr_pattern, 2, k);
    const int64_t i1 = PAT(h->fr_pattern, 3, k), j1 = PAT(h->fr_pattern, 4, k);
    if (i0 < 0 || j0 < 0 || i1 <= i0 || j1 <= j0 || i1 > h->n_row_pts || j1 > h->n_col_pts ||
        !h->fr_blocks[k]) {
      *msg = "full-rank block " + std::to_string(k) + " out of range";
      return BW_ESHAPE;
    }
    area += static_cast<long double>(i1 - i0) * (j1 - j0);
  }
  for (int64_t k = 0; k < h->n_lr; ++k) {
    const int64_t i0 = PAT(h->lr_pattern, 1, k), j0 = PAT(h->lr_pattern, 2, k);
    const int64_t i1 = PAT(h->lr_pattern, 3, k), j1 = PAT(h->lr_pattern, 4, k);
    const int64_t r = PAT(h->lr_pattern, 5, k);
    if (i0 < 0 || j0 < 0 || i1 <= i0 || j1 <= j0 || i1 > h->n_row_pts || j1 > h->n_col_pts ||
        r < 0 || (need_lr_data && r > 0 && (!h->lr_A[k] || !h->lr_B[k]))) {
      *msg = "low-rank block " + std::to_string(k) + " out of range";
      return BW_ESHAPE;
    }
    area += static_cast<long double>(i1 - i0) * (j1 - j0);
  }
  if (expected_area < 0.0L) expected_area = static_cast<long double>(h->n_row_pts) * h->n_col_pts;
  if (area != expected_area) {
    *msg = "blocks do not tile the matrix";
    return BW_ESHAPE;
  }
  return BW_OK;
}

void make_view(const bw_flat_hmat* h, bool transposed, OpView* v) {
  v->h = h;
  v->transposed = transposed;
  v->dof = h->dof;
  v->n_row_pts = transposed ? h->n_col_pts : h->n_row_pts;
  v->n_col_pts = transposed ? h->n_row_pts : h->n_col_pts;
  const int rr0 = transposed ? 2 : 1, rr1 = transposed ? 4 : 3;
  const int cc0 = transposed ? 1 : 2, cc1 = transposed ? 3 : 4;
  v->fr_r0.resize(h->n_fr);
  v->fr_r1.resize(h->n_fr);
  v->fr_c0.resize(h->n_fr);
  v->fr_c1.resize(h->n_fr);
  for (int64_t k = 0; k < h->n_fr; ++k) {
    v->fr_r0[k] = PAT(h->fr_pattern, rr0, k);
    v->fr_r1[k] = PAT(h->fr_pattern, rr1, k);
    v->fr_c0[k] = PAT(h->fr_pattern, cc0, k);
    v->fr_c1[k] = PAT(h->fr_pattern, cc1, k);
  }
  v->lr_r0.resize(h->n_lr);
  v->lr_r1.resize(h->n_lr);
  v->lr_c0.resize(h->n_lr);
  v->lr_c1.resize(h->n_lr);
  v->lr_rank.resize(h->n_lr);
  for (int64_t k = 0; k < h->n_lr; ++k) {
    v->lr_r0[k] = PAT(h->lr_pattern, rr0, k);
    v->lr_r1[k] = PAT(h->lr_pattern, rr1, k);
    v->lr_c0[k] = PAT(h->lr_pattern, cc0, k);
    v->lr_c1[k] = PAT(h->lr_pattern, cc1, k);
    v->lr_rank[k] = PAT(h->lr_pattern, 5, k);
  }
  // t-space: low-rank blocks ordered by (row range, first column) so that the
  // blocks of one row cluster are adjacent and their runs merge in pass 2.
  std::vector<int64_t> order(h->n_lr);
  std::iota(order.begin(), order.end(), 0);
  std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) {
    if (v->lr_r0[a] != v->lr_r0[b]) return v->lr_r0[a] < v->lr_r0[b];
    if (v->lr_r1[a] != v->lr_r1[b]) return v->lr_r1[a] < v->lr_r1[b];
    if (v->lr_c0[a] != v->lr_c0[b]) return v->lr_c0[a] < v->lr_c0[b];
    return a < b;
  });
  v->toff.assign(h->n_lr, 0);
  int64_t t = 0;
  for (int64_t k : order) {
    v->toff[k] = t;
    t += v->lr_rank[k];
  }
  v->t_total = t;
}

const double* OpView::source(int32_t kind, int64_t k, int64_t row, int64_t col,
                             int64_t* rs, int64_t* cs) const {
  const int64_t d = dof;
  if (kind == 0) {
    // original block is (d*(i1-i0)) x (d*(j1-j0)), ld = rows
    const int64_t m_orig = transposed ? d * (fr_c1[k] - fr_c0[k]) : d * (fr_r1[k] - fr_r0[k]);
    const double* F = h->fr_blocks[k];
    if (!transposed) {
      *rs = 1;
      *cs = m_orig;
    } else {
      *rs = m_orig;
      *cs = 1;
    }
    return F + row * (*rs) + col * (*cs);
  }
  const int64_t r = lr_rank[k];
  const int64_t m_orig = transposed ? d * (lr_c1[k] - lr_c0[k]) : d * (lr_r1[k] - lr_r0[k]);
  const double* A = h->lr_A[k];
  const double* B = h->lr_B[k];
  if (kind == 1) {
    if (!transposed) {  // A (m x r), ld m
      *rs = 1;
      *cs = m_orig;
      return A + row + col * m_orig;
    }
    *rs = r;  // B^T: (i, a) = B[a + i*r]
    *cs = 1;
    return B + col + row * r;
  }
  if (!transposed) {  // B (r x n), ld r
    *rs = 1;
    *cs = r;
    return B + row + col * r;
  }
  *rs = m_orig;  // A^T: (a, j) = A[j + a*m]
  *cs = 1;
  return A + col + row * m_orig;
}

namespace {

struct RunBuilder {
  Program* P;
  void add_piece(int64_t zoff, int64_t ncols, int32_t kind, int64_t block) {
    if (ncols <= 0) return;
    if (!P->runs.empty() && open_) {
      RunDesc& last = P->runs.back();
      if (last.zoff + last.ncols == zoff) {
        last.ncols += ncols;
        P->pieces.push_back({block, kind, 0, ncols});
        last.piece_end = static_cast<int32_t>(P->pieces.size());
        return;
      }
    }
    RunDesc rd;
    rd.zoff = zoff;
    rd.ncols = ncols;
    rd.piece_beg = static_cast<int32_t>(P->pieces.size());
    P->pieces.push_back({block, kind, 0, ncols});
    rd.piece_end = static_cast<int32_t>(P->pieces.size());
    P->runs.push_back(rd);
    open_ = true;
  }
  void close() { open_ = false; }
  bool open_ = false;
};

void add_slabs(Program* P, int64_t total_rows, int max_rows, int64_t out_row0,
               int64_t src_row0, int32_t run_beg, int32_t run_end, int V) {
  if (total_rows <= 0) return;  // a slab with no runs still writes zeros
  int64_t ngroups = 0;
  for (int32_t r = run_beg; r < run_end; ++r) ngroups += (P->runs[r].ncols + V - 1) / V;
  const int64_t nsl = (total_rows + max_rows - 1) / max_rows;
  int64_t done = 0;
  for (int64_t s = 0; s < nsl; ++s) {
    const int64_t rows = (total_rows - done) / (nsl - s);
    SlabDesc sd{};
    sd.rows = static_cast<int32_t>(rows);
    sd.out_row0 = out_row0 + done;
    sd.src_row0 = src_row0 + done;
    sd.run_beg = run_beg;
    sd.run_end = run_end;
    sd.ngroups = ngroups;
    P->slabs.push_back(sd);
    done += rows;
  }
}

// Work-item sizes, in entries (bytes / element size, so that FP32 items hold as
// many entries as FP64 ones).  A work item is one workgroup's share of a slab.
// Measured on MI355X with 8-wave workgroups for the single-vector kernel:
// - below the bounds the launch's tail and the kernel's start dominate, above
//   them too few workgroups are left to balance: pass 2 of the 120 000-DoF
//   3DR0 operator (4.3 GB) takes 656 us at 1.5 MiB, 639 at 384 KiB and 650 at
//   256 KiB; the 21 000-DoF 3DT0 one (320 MB) 61 us at 384 KiB, 57 at 192-256
//   KiB and 75 with whole slabs (0.8 MiB).
constexpr int64_t kItemMin = 24 * 1024, kItemMax = 48 * 1024;
constexpr int64_t kItemShare = 4096;  // between the two: 1 / 4096 of the pass
// - the batched kernels (4-wave workgroups) pay for every split with NB-wide
//   partial rows: 32 right-hand sides on the 49 152-DoF 3DR0 operator take 306
//   us at 384 KiB (FP32), 314 at 256, 311 at 768 KiB.
//   Passes of fewer slabs than kMinSlabs leave compute units idle at that size
//   and are cut to about 384 items (1 728 DoF, FP64, 32 slabs of 90 K entries:
//   38.6 -> 27.5 us, FP32 31 -> 22.4; 6 912 DoF, 128 slabs: 84 -> 77; 1 / 512 of
//   the pass 81, 1 / 1024 81); from 253 slabs on the cut costs more than it
//   balances (16 cracks, FP32: 41.5 us whole, 42.8 cut).
constexpr int64_t kItemBatched = 96 * 1024, kItemBatchedMin = 16 * 1024, kBatchedItems = 384;
// Pass 1 of a small operator is cut by rows instead: a slab over a wide column
// cluster gets fewer rows (at least 16), so that it is one work item and the
// pass needs no reduction.  Its item size is 1 / 1500 of the pass, at least 48
// KiB (25 600-DoF mode-1 operator, 171 MB: 42.7 us at 1 / 512, 40.4 at 1 /
// 1024, 38.8 at 1 / 1500, 41.3 at 1 / 2048; 16 000-DoF 2DS0 operator, whole
// matvec: 26.6 us at 64 KiB, 22.8 at 48; 6 400-DoF mode-1 19.5 at 64 and 48,
// 20.5 at 32).
constexpr int64_t kPass1Share = 1500, kPass1MinBytes = 48 * 1024;
// Rounds of 64 columns read four times the bytes of a 16-row slab as input rows,
// and its 32-row tiles are half empty: from this size on they take pass 1 in
// windows of 64 rows over all slabs of a column cluster instead (whole products,
// slabs and windows: 470 and 426 us at 114 M entries in pass 1, 241 and 217 at
// 46 M, 117 and 115 at 15 M, 69.6 and 68.8 at 8 M; mode-1 263 and 254 at 40 M, 141
// and 136 at 17 M, but 80 and 87 at 8 M).  Narrower rounds lose by the split windows (16 columns 3-10 %, 32 columns
// -4 to +4 %), and FP64 takes 277 us in slabs, 288 in windows.
constexpr int64_t kWindowEntries = 12 << 20, kMaxWindowGroups = 1 << 20;
constexpr int64_t kSortEntries = 200 << 20;
// A pass wants at least this many workgroups (of 256 compute units); in pass 2,
// operators with fewer slabs that fit one work item each get slabs of fewer rows (4 000-
// DoF 2DS0 operator, pass 2: 64 slabs of 62 rows 12.0 us, 256 of 16 rows 10.7).
constexpr int64_t kMinSlabs = 192;
constexpr int kMinRows = 16;

// Cuts the slabs into work items of about wi_bytes each and deals them to the
// XCDs in eight contiguous ranges of about equal cost.  row_tile: rows that a
// kernel's work comes in (the MFMA tile; 1: cost is bytes).  sorted: costliest
// first within each XCD's range, so that a range ends on its small items.
// windows: the slabs are windows over P.rowtab.
void cut_items(const std::vector<SlabDesc>& slabs, const LayoutOptions& opt, int64_t wi_bytes,
               int row_tile, bool sorted, bool windows, ItemList* il) {
  const int V = opt.vec_elems;
  *il = ItemList{};
  int64_t part = 0;
  for (const SlabDesc& sd : slabs) {
    const int64_t bytes = sd.ngroups * sd.rows * V * opt.elem_bytes;
    int64_t nwi = std::max<int64_t>(1, (bytes + wi_bytes / 2) / wi_bytes);
    nwi = std::min<int64_t>(nwi, std::max<int64_t>(1, sd.ngroups));
    const int64_t per = std::max<int64_t>(1, (sd.ngroups + nwi - 1) / nwi);
    nwi = std::max<int64_t>(1, (sd.ngroups + per - 1) / per);
    for (int64_t w = 0; w < nwi; ++w) {
      const int64_t g0 = w * per;
      const int64_t g1 = std::min(sd.ngroups, g0 + per);
      WorkItem wi{};
      wi.data_off = windows ? g0 : sd.data_off + g0 * sd.rows * V;
      wi.gbeg = static_cast<int32_t>(sd.gbeg + g0);
      wi.ngroups = static_cast<int32_t>(g1 - g0);
      wi.rows = sd.rows;
      wi.out_row = static_cast<int32_t>(sd.out_row0);
      wi.part_off = nwi == 1 ? -1 : static_cast<int32_t>(part + w * sd.rows);
      wi.red = static_cast<int32_t>(il->reds.size());
      il->wis.push_back(wi);
    }
    if (nwi > 1) {
      const Reduce rd{static_cast<int32_t>(sd.out_row0), sd.rows, static_cast<int32_t>(part),
                      static_cast<int32_t>(nwi)};
      il->reds.push_back(rd);
      part += nwi * sd.rows;
    }
  }
  il->part_elems = part;
  if (static_cast<int64_t>(il->wis.size()) <= kInKernelItems)
    il->counters = static_cast<int32_t>(il->reds.size());
  // balanced XCD ranges: cut the WI list where the running cost crosses x/8 of
  // the total (the nearer side of the crossing)
  const int64_t nwi = static_cast<int64_t>(il->wis.size());
  std::vector<int64_t> cum(nwi + 1, 0);
  auto cost = [&](const WorkItem& w) {
    return static_cast<int64_t>(w.ngroups) * ((w.rows + row_tile - 1) / row_tile * row_tile) + 1;
  };
  for (int64_t i = 0; i < nwi; ++i) cum[i + 1] = cum[i] + cost(il->wis[i]);
  il->xcd[0] = 0;
  for (int x = 1; x < kXcds; ++x) {
    const long double target = static_cast<long double>(cum[nwi]) * x / kXcds;
    int64_t i = std::lower_bound(cum.begin(), cum.end(), static_cast<int64_t>(target)) - cum.begin();
    if (i > 0 && target - cum[i - 1] < cum[std::min(i, nwi)] - target) --i;
    il->xcd[x] = static_cast<int32_t>(std::max<int64_t>(il->xcd[x - 1], std::min(i, nwi)));
  }
  il->xcd[kXcds] = static_cast<int32_t>(nwi);
  if (sorted)
    for (int x = 0; x < kXcds; ++x)
      std::stable_sort(il->wis.begin() + il->xcd[x], il->wis.begin() + il->xcd[x + 1],
                       [&](const WorkItem& a, const WorkItem& b) { return cost(a) > cost(b); });
}

// Places the slabs' data and column groups, and cuts both work-item lists.
// Pass 1's items differ most in size (24 KiB to its bound) and run costliest
// first (30 000-DoF 3DR0 operator: pass 1 97 us in slab order, 90 sorted), up to
// kSortEntries: in slab order neighbours share input entries, which is worth
// more on long passes (600 000-DoF 3DT0, FP64 3.45 ms against 3.56).  Pass 2's
// single-vector items are alike, and slab order is 1 % faster on the 120 000-DoF
// operator.  The batched
// kernels run 6-8 % faster sorted (327 -> 306 us, FP32, 49 152 DoF).
void finalize_program(Program* P, const LayoutOptions& opt, int64_t wi_single, bool sort_single) {
  const int V = opt.vec_elems;
  int64_t data = 0;
  P->gidx.clear();
  for (SlabDesc& sd : P->slabs) {
    sd.data_off = data;
    sd.gbeg = static_cast<int32_t>(P->gidx.size());
    for (int32_t r = sd.run_beg; r < sd.run_end; ++r) {
      const RunDesc& rd = P->runs[r];
      const int64_t ng = (rd.ncols + V - 1) / V;
      for (int64_t g = 0; g < ng; ++g) P->gidx.push_back(static_cast<int32_t>(rd.zoff + g * V));
    }
    data += sd.ngroups * sd.rows * V;
  }
  P->data_elems = data;
  const bool tuned = opt.wi_bytes > 0;
  cut_items(P->slabs, opt, tuned ? opt.wi_bytes : wi_single, 1, sort_single, false, &P->single);
  auto batched_bytes = [&](size_t slabs) {
    if (tuned) return opt.wi_bytes;
    return opt.elem_bytes * (static_cast<int64_t>(slabs) >= kMinSlabs
                                 ? kItemBatched
                                 : std::min(kItemBatched, std::max(kItemBatchedMin, data / kBatchedItems)));
  };
  const int row_tile = opt.elem_bytes == 8 ? 16 : 32;
  cut_items(P->slabs, opt, batched_bytes(P->slabs.size()), row_tile, true, false, &P->batched);
  P->wide = ItemList{};
  P->rowtab.clear();
  if (opt.elem_bytes != 4 || tuned || P->rowmap.empty() || data < kWindowEntries) return;
  // the rows of a window lie within 192 rows of slabs: 32-bit offsets
  for (const SlabDesc& sd : P->slabs)
    if (sd.ngroups >= kMaxWindowGroups) return;
  // Windows of up to 64 rows over the slabs of one column cluster, whose rows
  // follow each other in the row map.
  std::vector<SlabDesc> win;
  size_t i = 0;
  while (i < P->slabs.size()) {
    const SlabDesc& a = P->slabs[i];
    const RunDesc& ra = P->runs[a.run_beg];
    int64_t rows = 0;
    for (; i < P->slabs.size(); ++i) {
      const SlabDesc& sd = P->slabs[i];
      const RunDesc& rd = P->runs[sd.run_beg];
      if (rd.zoff != ra.zoff || rd.ncols != ra.ncols) break;
      for (int32_t r = 0; r < sd.rows; ++r)
        P->rowtab.push_back((sd.data_off / V + r) << 8 | sd.rows);
      rows += sd.rows;
    }
    for (int64_t r = 0; r < rows; r += 64) {
      SlabDesc w = a;
      w.rows = static_cast<int32_t>(std::min<int64_t>(64, rows - r));
      w.out_row0 = a.out_row0 + r;
      win.push_back(w);
    }
  }
  cut_items(win, opt, batched_bytes(win.size()), row_tile, true, true, &P->wide);
}

}  // namespace

void build_layout(const OpView& v, const LayoutOptions& opt, Layout* L) {
  L->view = v;
  L->opt = opt;
  const int V = opt.vec_elems;
  const int64_t d = v.dof;
  const int64_t ncols_dof = d * v.n_col_pts;
  L->xt_t = align_up(ncols_dof + 64, 64);  // gap: padded x groups never reach t
  L->xt_size = align_up(L->xt_t + v.t_total, 64) + 64;
  const int64_t nlr = static_cast<int64_t>(v.lr_rank.size());
  const int64_t nfr = static_cast<int64_t>(v.fr_r0.size());

  // ---- pass 1: t_k = W_k x_{J_k}.  Blocks with the same column cluster
  // share their input, so their rows are stacked into slabs of at most
  // max_rows rows; a slab row writes its t entry through rowmap.
  {
    Program& P = L->pass1;
    P = Program{};
    P.out_rows = v.t_total;
    int64_t entries = 0;
    for (int64_t k = 0; k < nlr; ++k) entries += v.lr_rank[k] * d * (v.lr_c1[k] - v.lr_c0[k]);
    const int64_t max_item = kItemMax * opt.elem_bytes;
    const int64_t item =
        std::max<int64_t>(kPass1MinBytes, entries * opt.elem_bytes / kPass1Share);
    const bool by_rows = opt.wi_bytes == 0 && item < max_item;
    // most rows of a slab over `cols` columns
    auto rows_for = [&](int64_t cols) -> int64_t {
      if (!by_rows) return opt.max_rows;
      const int64_t r = item * 3 / 2 / (cols * opt.elem_bytes) / kMinRows * kMinRows;
      return std::min<int64_t>(opt.max_rows, std::max<int64_t>(kMinRows, r));
    };
    std::vector<int64_t> order;
    order.reserve(nlr);
    for (int64_t k = 0; k < nlr; ++k)
      if (v.lr_rank[k] > 0) order.push_back(k);
    std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) {
      if (v.lr_c0[a] != v.lr_c0[b]) return v.lr_c0[a] < v.lr_c0[b];
      if (v.lr_c1[a] != v.lr_c1[b]) return v.lr_c1[a] < v.lr_c1[b];
      return v.toff[a] < v.toff[b];
    });
    RunBuilder rb{&P};
    size_t i = 0;
    while (i < order.size()) {
      size_t j = i;  // [i, j): one column cluster
      while (j < order.size() && v.lr_c0[order[j]] == v.lr_c0[order[i]] &&
             v.lr_c1[order[j]] == v.lr_c1[order[i]])
        ++j;
      const int64_t c0 = v.lr_c0[order[i]], ncols = d * (v.lr_c1[order[i]] - c0);
      const int64_t maxr = rows_for(ncols);
      // each factor's rows cut into ceil(r / maxr) chunks of even height (a
      // rank of 90 gives 45 + 45, not 64 + 26), packed first-fit decreasing
      std::vector<StackPart> chunks;
      for (size_t q = i; q < j; ++q) {
        const int64_t r = v.lr_rank[order[q]];
        const int64_t nsl = (r + maxr - 1) / maxr;
        for (int64_t c = 0, r0 = 0; c < nsl; ++c) {
          const int64_t n = (r - r0) / (nsl - c);
          chunks.push_back({order[q], static_cast<int32_t>(r0), static_cast<int32_t>(n)});
          r0 += n;
        }
      }
      std::stable_sort(chunks.begin(), chunks.end(),
                       [](const StackPart& a, const StackPart& b) { return a.nrows > b.nrows; });
      std::vector<std::vector<StackPart>> bins;
      std::vector<int64_t> fill;
      for (const StackPart& c : chunks) {
        size_t b = 0;
        if (c.nrows > opt.stack_rows)
          b = bins.size();  // a chunk this tall keeps a slab of its own
        while (b < bins.size() && (fill[b] + c.nrows > maxr || bins[b][0].nrows > opt.stack_rows))
          ++b;
        if (b == bins.size()) {
          bins.emplace_back();
          fill.push_back(0);
        }
        bins[b].push_back(c);
        fill[b] += c.nrows;
      }
      for (size_t b = 0; b < bins.size(); ++b) {
        SlabDesc sd{};
        sd.rows = static_cast<int32_t>(fill[b]);
        sd.out_row0 = static_cast<int64_t>(P.rowmap.size());
        sd.stack_beg = static_cast<int32_t>(P.stack.size());
        for (const StackPart& c : bins[b]) {
          P.stack.push_back(c);
          for (int32_t a = 0; a < c.nrows; ++a)
            P.rowmap.push_back(static_cast<int32_t>(L->xt_t + v.toff[c.block] + c.row0 + a));
        }
        sd.stack_end = static_cast<int32_t>(P.stack.size());
        rb.close();
        sd.run_beg = static_cast<int32_t>(P.runs.size());
        rb.add_piece(d * c0, ncols, 2, bins[b][0].block);
        sd.run_end = static_cast<int32_t>(P.runs.size());
        sd.src_row0 = 0;
        sd.ngroups = (ncols + V - 1) / V;
        P.slabs.push_back(sd);
      }
      i = j;
    }
    finalize_program(&P, opt, by_rows ? 4 * item : max_item, entries <= kSortEntries);
  }

  // ---- pass 2: row intervals
  {
    Program& P = L->pass2;
    P = Program{};
    P.out_rows = d * v.n_row_pts;
    std::vector<int64_t> bps;
    bps.reserve(2 * (nfr + nlr) + 2);
    bps.push_back(0);
    bps.push_back(v.n_row_pts);
    for (int64_t k = 0; k < nfr; ++k) {
      bps.push_back(v.fr_r0[k]);
      bps.push_back(v.fr_r1[k]);
    }
    for (int64_t k = 0; k < nlr; ++k) {
      bps.push_back(v.lr_r0[k]);
      bps.push_back(v.lr_r1[k]);
    }
    std::sort(bps.begin(), bps.end());
    bps.erase(std::unique(bps.begin(), bps.end()), bps.end());
    const int64_t nint = static_cast<int64_t>(bps.size()) - 1;
    auto interval_of = [&](int64_t pt) {
      return static_cast<int64_t>(std::upper_bound(bps.begin(), bps.end(), pt) - bps.begin()) - 1;
    };
    std::vector<std::vector<int64_t>> frl(nint), lrl(nint);
    for (int64_t k = 0; k < nfr; ++k)
      for (int64_t q = interval_of(v.fr_r0[k]); q < nint && bps[q] < v.fr_r1[k]; ++q) frl[q].push_back(k);
    for (int64_t k = 0; k < nlr; ++k) {
      if (v.lr_rank[k] == 0) continue;
      for (int64_t q = interval_of(v.lr_r0[k]); q < nint && bps[q] < v.lr_r1[k]; ++q) lrl[q].push_back(k);
    }
    int64_t entries = 0;
    for (int64_t k = 0; k < nfr; ++k)
      entries += d * (v.fr_r1[k] - v.fr_r0[k]) * d * (v.fr_c1[k] - v.fr_c0[k]);
    for (int64_t k = 0; k < nlr; ++k) entries += v.lr_rank[k] * d * (v.lr_r1[k] - v.lr_r0[k]);
    const int64_t item = opt.elem_bytes * std::min<int64_t>(
        kItemMax, std::max<int64_t>(kItemMin, entries / kItemShare));
    int64_t nslab = 0;  // slabs of full height
    for (int64_t q = 0; q < nint; ++q)
      nslab += (d * (bps[q + 1] - bps[q]) + opt.max_rows - 1) / opt.max_rows;
    int64_t max_rows = opt.max_rows;
    if (opt.wi_bytes == 0 && nslab < kMinSlabs &&
        entries * opt.elem_bytes / nslab < item * 3 / 2)
      max_rows = std::max<int64_t>(kMinRows, opt.max_rows * nslab / kMinSlabs / kMinRows * kMinRows);
    RunBuilder rb{&P};
    for (int64_t q = 0; q < nint; ++q) {
      auto& fl = frl[q];
      std::sort(fl.begin(), fl.end(), [&](int64_t a, int64_t b) {
        return v.fr_c0[a] != v.fr_c0[b] ? v.fr_c0[a] < v.fr_c0[b] : a < b;
      });
      auto& ll = lrl[q];
      std::sort(ll.begin(), ll.end(), [&](int64_t a, int64_t b) { return v.toff[a] < v.toff[b]; });
      rb.close();
      const int32_t rbeg = static_cast<int32_t>(P.runs.size());
      for (int64_t k : fl) rb.add_piece(d * v.fr_c0[k], d * (v.fr_c1[k] - v.fr_c0[k]), 0, k);
      rb.close();
      for (int64_t k : ll) rb.add_piece(L->xt_t + v.toff[k], v.lr_rank[k], 1, k);
      const int32_t rend = static_cast<int32_t>(P.runs.size());
      const int64_t rows = d * (bps[q + 1] - bps[q]);
      add_slabs(&P, rows, static_cast<int>(max_rows), d * bps[q], d * bps[q], rbeg, rend, V);
    }
    finalize_program(&P, opt, item, false);
  }
}

template <typename T>
void fill_slabs(const Layout& L, const Program& P, int32_t s_beg, int32_t s_end, T* out) {
  const OpView& v = L.view;
  const int V = L.opt.vec_elems;
  const int64_t d = v.dof;
  const int64_t base_off = P.slabs[s_beg].data_off;
  for (int32_t s = s_beg; s < s_end; ++s) {
    const SlabDesc& sd = P.slabs[s];
    const int64_t R = sd.rows;
    T* slab = out + (sd.data_off - base_off);
    std::memset(slab, 0, sizeof(T) * static_cast<size_t>(sd.ngroups * R * V));
    int64_t gcur = 0;  // first group of the current run
    for (int32_t r = sd.run_beg; r < sd.run_end; ++r) {
      const RunDesc& rd = P.runs[r];
      T* runp = slab + gcur * R * V;
      int64_t col = 0;  // column within the run
      if (sd.stack_end > sd.stack_beg) {
        // pass 1: one run over the shared columns, rows from stacked W_k
        int64_t rbase = 0;
        for (int32_t q = sd.stack_beg; q < sd.stack_end; ++q) {
          const StackPart& sp = P.stack[q];
          int64_t rs, cs;
          const double* src = v.source(2, sp.block, sp.row0, 0, &rs, &cs);
          for (int64_t c = 0; c < rd.ncols; ++c) {
            T* dst = runp + (c / V) * R * V + (c % V) + rbase * V;
            const double* sc = src + c * cs;
            for (int64_t a = 0; a < sp.nrows; ++a) dst[a * V] = static_cast<T>(sc[a * rs]);
          }
          rbase += sp.nrows;
        }
        gcur += (rd.ncols + V - 1) / V;
        continue;
      }
      for (int32_t pi = rd.piece_beg; pi < rd.piece_end; ++pi) {
        const Piece& pc = P.pieces[pi];
        int64_t row_local;
        if (pc.kind == 2)
          row_local = sd.src_row0;
        else if (pc.kind == 0)
          row_local = sd.src_row0 - d * v.fr_r0[pc.block];
        else
          row_local = sd.src_row0 - d * v.lr_r0[pc.block];
        int64_t rs, cs;
        const double* src = v.source(pc.kind, pc.block, row_local, pc.col0, &rs, &cs);
        for (int64_t c = 0; c < pc.ncols; ++c, ++col) {
          T* dst = runp + (col / V) * R * V + (col % V);
          const double* sc = src + c * cs;
          for (int64_t i = 0; i < R; ++i) dst[i * V] = static_cast<T>(sc[i * rs]);
        }
      }
      gcur += (rd.ncols + V - 1) / V;
    }
  }
}

template void fill_slabs<double>(const Layout&, const Program&, int32_t, int32_t, double*);
template void fill_slabs<float>(const Layout&, const Program&, int32_t, int32_t, float*);

int check_layout_limits(const Layout& L, std::string* msg) {
  const int64_t lim = INT32_MAX;
  if (L.xt_size >= lim) {
    *msg = "input and rank vectors too long for 32-bit offsets";
    return BW_ESHAPE;
  }
  if (L.view.n_row_pts * L.view.dof >= lim) {
    *msg = "too many rows for 32-bit row indices";
    return BW_ESHAPE;
  }
  for (const Program* P : {&L.pass1, &L.pass2}) {
    if (static_cast<int64_t>(P->gidx.size()) >= lim || P->single.part_elems >= lim ||
        P->batched.part_elems >= lim || P->wide.part_elems >= lim || static_cast<int64_t>(P->rowmap.size()) >= lim ||
        static_cast<int64_t>(P->single.wis.size()) >= lim / 4 ||
        static_cast<int64_t>(P->batched.wis.size()) >= lim / 4 ||
        static_cast<int64_t>(P->wide.wis.size()) >= lim / 4) {
      *msg = "matrix too large for 32-bit layout descriptors";
      return BW_ESHAPE;
    }
  }
  return BW_OK;
}

int64_t layout_stored_entries(const Layout& L) { return L.pass1.data_elems + L.pass2.data_elems; }

}  // namespace bwl
