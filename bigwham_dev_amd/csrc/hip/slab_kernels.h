// Device code of the single-vector matvec: gather, slab dot products, reduce.
// Included by engine.hip only (inside its anonymous namespace).
#pragma once

typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef float flt4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Vec;
template <>
struct Vec<double> {
  static constexpr int V = 2;
  typedef dbl2 type;
};
template <>
struct Vec<float> {
  static constexpr int V = 4;
  typedef flt4 type;
};

// Workgroups are dispatched round-robin over the 8 XCDs of the MI355X
// (workgroup b runs on XCD b % 8).  Each XCD gets a contiguous range of work
// items of about equal bytes (neighbouring row clusters share x entries in
// that XCD's L2, and no XCD is left with the tail).  Returns the work item of
// this workgroup, or -1.
struct XcdSplit {
  int32_t s[bwl::kXcds + 1];
};

__device__ __forceinline__ int xcd_work_item(const XcdSplit& xs, unsigned block) {
  const int x = block % bwl::kXcds;
  const int w = xs.s[x] + static_cast<int>(block / bwl::kXcds);
  return w < xs.s[x + 1] ? w : -1;
}

template <typename T>
__global__ __launch_bounds__(256) void k_gather(const double* __restrict__ x,
                                                T* __restrict__ xt, int64_t n,
                                                const int64_t* __restrict__ perm, int dof) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t src = i;
  if (perm) {
    const int64_t p = i / dof;
    src = dof * perm[p] + (i - p * dof);
  }
  xt[i] = static_cast<T>(x[src]);
}

// Result of a host-pointer call to pinned memory, in order.
__global__ __launch_bounds__(256) void k_copy(const double* __restrict__ src,
                                              double* __restrict__ dst, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

template <typename OutT>
__device__ __forceinline__ int64_t out_index(int64_t idx, const int64_t* perm, int dof) {
  if (!perm) return idx;
  // row indices fit in 32 bits (checked when the layout is built)
  const int i = static_cast<int>(idx);
  const int p = i / dof;
  return dof * perm[p] + (i - p * dof);
}

// Where a slab's input entries come from.  `off(g)` gives the offset of column
// group g and `at(off, v)` entry v of it; `ready()` is called once per wave,
// after its first factor loads have been requested and before the first `at`.
//
// From xt through the group offsets; tall slabs have wave-uniform offsets
// (scalar loads).
template <typename T, bool TALL>
struct XtInput {
  const int32_t* __restrict__ gi;
  const T* __restrict__ xin;

  __device__ __forceinline__ int off(int g) const { return gi[g]; }
  __device__ __forceinline__ T at(int o, int v) const {
    // unsigned: no sign extension of the loaded offset is placed (and waited
    // for) next to its load
    if constexpr (TALL)
      return xin[static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(o)) + v];
    else
      return xin[o + v];
  }
  __device__ __forceinline__ void ready() const {}
};

// From LDS, where ready() puts the work item's whole input: the entries
// z0 .. z0 + ncol - 1 of the permuted x, read from the caller's vector (pass 1
// of small operators; a pass-1 slab's columns are one run).
template <typename T, int THREADS>
struct StagedInput {
  static constexpr int V = Vec<T>::V;
  T* lds;
  int g0;  // the wave's first group within the work item
  const double* __restrict__ x;
  const int64_t* __restrict__ perm;
  int dof;
  int n_in, z0, ncol;

  __device__ __forceinline__ int off(int g) const { return (g0 + g) * V; }
  __device__ __forceinline__ T at(int o, int v) const { return lds[o + v]; }
  __device__ __forceinline__ void ready() const {
    for (int c = threadIdx.x; c < ncol; c += THREADS) {
      const int z = z0 + c;  // past x: the zeros that xt holds there
      lds[c] = z < n_in ? static_cast<T>(x[out_index<T>(z, perm, dof)]) : T(0);
    }
    __syncthreads();
  }
};

// The accumulators of a lane: for even and odd groups one each (FP64) or one
// per entry of a group (FP32), so that the chains of FP32 additions are an
// eighth of the lane's columns.  Errors of FP32 products against 64 bits over
// 800-120 000 DoF: two accumulators 0.86-1.14e-7, these 0.84-1.07e-7 in the same
// time; sixteen are no better and 1 % slower.
template <typename T>
constexpr int kAccs = sizeof(T) == 4 ? 4 : 1;

template <typename T>
__device__ __forceinline__ T sum_acc(const T (&acc)[2][kAccs<T>]) {
  if constexpr (kAccs<T> == 1) return acc[0][0] + acc[1][0];
  else
    return ((acc[0][0] + acc[0][1]) + (acc[0][2] + acc[0][3])) +
           ((acc[1][0] + acc[1][1]) + (acc[1][2] + acc[1][3]));
}

// Dot products of a wave's column groups with more than 32 rows: one column
// group per step for the whole wavefront.  U: 16-byte loads in flight per lane.
template <typename T, int U, typename In>
__device__ __forceinline__ T dot_tall(const typename Vec<T>::type* __restrict__ p, int R, int ng,
                                      const In& in) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  constexpr int A = kAccs<T>;
  T acc[2][A] = {};
  // Full batches of U groups through two register buffers: the loads of
  // batch b + 1 go out before the FMAs of batch b, so a batch's loads are in
  // flight while the previous one is consumed.  The loop body issues the same
  // loads on every trip and the last one or two batches are peeled, so the
  // waits the compiler places are the same on every path.
  const int nfull = ng / U;
  if (nfull > 0) {
    VT a[U], b[U];
    int za[U], zb[U];
    auto load = [&](int g0, VT (&buf)[U], int (&zz)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) zz[u] = in.off(g0 + u);
#pragma unroll
      for (int u = 0; u < U; ++u) buf[u] = __builtin_nontemporal_load(p + (g0 + u) * R);
    };
    auto use = [&](const VT (&buf)[U], const int (&zz)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int v = 0; v < V; ++v) {
          acc[u & 1][v % A] += buf[u][v] * in.at(zz[u], v);
        }
    };
    load(0, a, za);
    __builtin_amdgcn_sched_barrier(0);
    in.ready();
    int bt = 0;
    for (; bt + 2 < nfull; bt += 2) {
      __builtin_amdgcn_sched_barrier(0);
      load((bt + 1) * U, b, zb);
      __builtin_amdgcn_sched_barrier(0);
      use(a, za);
      __builtin_amdgcn_sched_barrier(0);
      load((bt + 2) * U, a, za);
      __builtin_amdgcn_sched_barrier(0);
      use(b, zb);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (bt + 2 == nfull) {
      load((bt + 1) * U, b, zb);
      __builtin_amdgcn_sched_barrier(0);
      use(a, za);
      __builtin_amdgcn_sched_barrier(0);
      use(b, zb);
    } else {
      use(a, za);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // The last, partial batch in one memory round trip: 4 or U loads (clamped
  // to the last group, in bounds), of which the first rem are used.
  const int g = nfull * U, rem = ng - g;
  auto tail = [&](auto N) {
    constexpr int n = decltype(N)::value;
    VT a[n];
    int z[n];
#pragma unroll
    for (int u = 0; u < n; ++u) z[u] = in.off(g + min(u, rem - 1));
#pragma unroll
    for (int u = 0; u < n; ++u) a[u] = __builtin_nontemporal_load(p + (g + min(u, rem - 1)) * R);
    if (nfull == 0) in.ready();
#pragma unroll
    for (int u = 0; u < n; ++u)
      if (u < rem) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
          acc[u & 1][v % A] += a[u][v] * in.at(z[u], v);
        }
      }
  };
  if (rem > 4)
    tail(std::integral_constant<int, U>{});
  else if (rem > 0)
    tail(std::integral_constant<int, 4>{});
  return sum_acc<T>(acc);
}

// Dot products of a wave's column groups with at most 32 rows: nsplit = 64 / R
// groups at a time (lane = split * R + row; `p` points at the lane's row), U
// of them per step.  As in dot_tall, a step's loads (factors and input
// entries) go out before the FMAs of the step before, through two register
// buffers; the input offsets are loaded two steps ahead, so that one memory
// round trip covers a step.  Offsets and groups past the end are clamped (in
// bounds) and not used.
template <typename T, int U, typename In>
__device__ __forceinline__ T dot_short(const typename Vec<T>::type* __restrict__ p, int R,
                                       int nsplit, int split, int ng, const In& in) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  constexpr int A = kAccs<T>;
  T acc[2][A] = {};
  const int step = U * nsplit;
  const int n = (ng + step - 1) / step;
  VT a[U], b[U];
  T xa[U][V], xb[U][V];
  int za[U], zb[U];
  auto load_z = [&](int s, int (&z)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) z[u] = in.off(min(s * step + split + u * nsplit, ng - 1));
  };
  auto load_a = [&](int s, VT (&f)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      f[u] = __builtin_nontemporal_load(p + min(s * step + split + u * nsplit, ng - 1) * R);
  };
  auto load_x = [&](int s, T (&x)[U][V], int (&z)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) x[u][v] = in.at(z[u], v);
    load_z(s + 2, z);
  };
  auto use = [&](const VT (&f)[U], const T (&x)[U][V]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        acc[u & 1][v % A] += f[u][v] * x[u][v];
      }
  };
  auto use_last = [&](const VT (&f)[U], const T (&x)[U][V]) {  // step n - 1
#pragma unroll
    for (int u = 0; u < U; ++u)
      if ((n - 1) * step + split + u * nsplit < ng) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
          acc[u & 1][v % A] += f[u][v] * x[u][v];
        }
      }
  };
  load_z(0, za);
  load_z(1, zb);
  load_a(0, a);
  __builtin_amdgcn_sched_barrier(0);
  in.ready();
  load_x(0, xa, za);
  int s = 0;
  for (; s + 2 < n; s += 2) {
    __builtin_amdgcn_sched_barrier(0);
    load_a(s + 1, b);
    load_x(s + 1, xb, zb);
    __builtin_amdgcn_sched_barrier(0);
    use(a, xa);
    __builtin_amdgcn_sched_barrier(0);
    load_a(s + 2, a);
    load_x(s + 2, xa, za);
    __builtin_amdgcn_sched_barrier(0);
    use(b, xb);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (s + 2 == n) {
    load_a(s + 1, b);
    load_x(s + 1, xb, zb);
    __builtin_amdgcn_sched_barrier(0);
    use(a, xa);
    __builtin_amdgcn_sched_barrier(0);
    use_last(b, xb);
  } else {
    use_last(a, xa);
  }
  return sum_acc<T>(acc);
}

// Adds the column splits of a wave onto lanes 0..R-1, in split order.
template <typename T>
__device__ __forceinline__ T fold_splits(T acc, int R, int nsplit, int split, int lane) {
  for (int s = 1; s < nsplit; ++s) {
    const T o = __shfl(acc, lane + s * R, 64);
    if (split == 0) acc += o;
  }
  return acc;
}

// Split slabs of passes of few work items (the others: k_reduce).  Each work
// item of one stores its partial sums, waits until they have arrived, and counts itself in; the one that finds all others
// counted adds the partial sums in work-item order, stores the rows and sets
// the counter back to zero for the next launch.  The work items of a slab can
// run on different XCDs, whose L2s are not coherent: partial sums and counters
// are only ever touched by agent-scope atomic accesses, which go past the L2.
// They are relaxed: a release or acquire at agent scope would write back and
// invalidate a whole L2, and the wait below is the order that is needed (a
// store that has been acknowledged is visible to every later agent-scope load).
// No work item waits for another.
struct SplitSums {
  const bwl::Reduce* reds;
  int32_t* count;  // one per split slab, zero between launches; nullptr: k_reduce adds them
};

template <typename P>
__device__ __forceinline__ void part_store(P* p, P v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename P>
__device__ __forceinline__ P part_load(const P* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until this wave's stores have been acknowledged.
__device__ __forceinline__ void stores_arrived() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Counts a work item in (one lane); true for the last of nparts.
__device__ __forceinline__ bool count_in(int32_t* count, int nparts) {
  return __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nparts - 1;
}

// The waves' sums of a work item added in wave order from LDS, and its rows
// stored by the first wave (`orow`: the lane's output row, requested before
// the stream).
template <typename T, typename OutT, int W>
__device__ __forceinline__ void wave_sum_put(T acc, T (*red)[64], const bwl::WorkItem& wi,
                                             int wave, int lane, int64_t orow, OutT* out, T* part,
                                             const SplitSums& sp) {
  const int R = wi.rows;
  if (wave > 0 && lane < R) red[wave][lane] = acc;
  __syncthreads();
  if (wave > 0 || lane >= R) return;
#pragma unroll
  for (int k = 1; k < W; ++k) acc += red[k][lane];
  if (wi.part_off >= 0) {
    if (!sp.count) {  // added by k_reduce
      part[wi.part_off + lane] = acc;
      return;
    }
    const bwl::Reduce rd = sp.reds[wi.red];
    part_store(part + wi.part_off + lane, acc);
    stores_arrived();
    int last = 0;
    if (lane == 0) last = count_in(sp.count + wi.red, rd.nparts);
    if (!__builtin_amdgcn_readfirstlane(last)) return;
    // four interleaved sums over the parts, eight loads in flight; the order
    // of the additions is fixed, so the result is deterministic
    const T* p = part + rd.part_off + lane;
    T s[4] = {0, 0, 0, 0};
    int q = 0;
    for (; q + 8 <= rd.nparts; q += 8) {
      T v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = part_load(p + (q + k) * R);
#pragma unroll
      for (int k = 0; k < 8; ++k) s[k & 3] += v[k];
    }
    for (; q + 4 <= rd.nparts; q += 4) {
      T v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = part_load(p + (q + k) * R);
#pragma unroll
      for (int k = 0; k < 4; ++k) s[k] += v[k];
    }
    T v[3] = {0, 0, 0};
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (q + k < rd.nparts) v[k] = part_load(p + (q + k) * R);
#pragma unroll
    for (int k = 0; k < 3; ++k) s[0] += v[k];
    acc = (s[0] + s[1]) + (s[2] + s[3]);
    if (lane == 0) part_store(sp.count + wi.red, int32_t{0});
  }
  out[orow] = static_cast<OutT>(acc);
}

// One workgroup of W waves per work item: the waves take equal contiguous
// shares of its column groups, and the first wave adds their sums from LDS in
// wave order, so a slab needs a partial-sum buffer and a reduce launch only
// where it is longer than what one workgroup should stream.  Bound by the
// factor stream.  One wave per work item, 32 768 of them and two reduce
// launches against this: 4 000-DoF 2DS0 operator (15 MB) 23 -> 15 us a matvec,
// 3 072-DoF 3DR0 (51 MB) 34 -> 20, 25 600-DoF mode-1 H and H^T (0.85 GB) 219
// -> 163, 120 000-DoF 3DR0 (7.7 GB) 1 178 -> 1 136 (6.75 TB/s), 600 000-DoF
// 3DT0 (53 GB) 7 906 -> 7 780 us.
// T: factor / accumulation type; OutT: output type (T for pass 1, double
// for pass 2); U: unroll depth (independent 16-byte loads in flight per lane);
// PASS only names the two launches apart in profiles.
template <typename T, typename OutT, int U, int PASS, int W>
__global__ __launch_bounds__(64 * W) void k_slab(const bwl::WorkItem* __restrict__ wis,
                                                 XcdSplit xs, const int32_t* __restrict__ gidx,
                                                 const T* __restrict__ data,
                                                 const T* __restrict__ xin,
                                                 OutT* __restrict__ out, T* __restrict__ part,
                                                 SplitSums sp,
                                                 const int64_t* __restrict__ perm, int dof,
                                                 const int32_t* __restrict__ rowmap) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  __shared__ T red[W][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int w = xcd_work_item(xs, blockIdx.x);
  if (w < 0) return;
  const bwl::WorkItem wi = wis[w];
  const int R = wi.rows;
  // this wave's share of the column groups
  const int per = (wi.ngroups + W - 1) / W;
  const int g0 = min(wave * per, wi.ngroups);
  const int ng = min(per, wi.ngroups - g0);
  const VT* __restrict__ base =
      reinterpret_cast<const VT*>(data + wi.data_off + static_cast<int64_t>(g0) * R * V);
  const int32_t* __restrict__ gi = gidx + wi.gbeg + g0;
  int64_t orow = 0;
  if (wave == 0 && (wi.part_off < 0 || sp.count) && lane < R) {
    // pass 1 rows go to their t entries through the row map
    const int64_t r = rowmap ? rowmap[wi.out_row + lane] : static_cast<int64_t>(wi.out_row) + lane;
    orow = out_index<OutT>(r, perm, dof);
  }
  T acc = 0;
  if (R > 32) {
    if (lane < R && ng > 0) acc = dot_tall<T, U>(base + lane, R, ng, XtInput<T, true>{gi, xin});
  } else {
    const int nsplit = 64 / R;
    const int split = lane / R;
    if (split < nsplit && ng > 0)
      acc = dot_short<T, 4>(base + (lane - split * R), R, nsplit, split, ng,
                            XtInput<T, false>{gi, xin});
    acc = fold_splits(acc, R, nsplit, split, lane);
  }
  wave_sum_put<T, OutT, W>(acc, red, wi, wave, lane, orow, out, part, sp);
}

// Pass 1 of small operators together with the gather of x: the first
// `ngather` workgroups write the permuted x to xt for pass 2, the others take
// the work items and stage their own input from the caller's vector in LDS
// (lds_cols entries), behind the first factor loads.  A launch less where
// launches count: 4 000-DoF 2DS0 operator 15.7 -> 12.6 us a matvec, 3 072-DoF
// 3DR0 19.6 -> 16.2.
template <typename T, int U, int W>
__global__ __launch_bounds__(64 * W) void k_slab_gather(
    const bwl::WorkItem* __restrict__ wis, XcdSplit xs, const int32_t* __restrict__ gidx,
    const T* __restrict__ data, const double* __restrict__ x, T* __restrict__ xt, int n_in,
    const int64_t* __restrict__ perm, int dof, int ngather, int lds_cols, T* __restrict__ part,
    SplitSums sp,
    const int32_t* __restrict__ rowmap) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  extern __shared__ __align__(16) unsigned char smem[];
  T* const stage = reinterpret_cast<T*>(smem);
  T(*const red)[64] = reinterpret_cast<T(*)[64]>(stage + lds_cols);
  if (blockIdx.x < static_cast<unsigned>(ngather)) {
    for (int i = blockIdx.x * (64 * W) + threadIdx.x; i < n_in; i += ngather * (64 * W))
      xt[i] = static_cast<T>(x[out_index<T>(i, perm, dof)]);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int w = xcd_work_item(xs, blockIdx.x - ngather);
  if (w < 0) return;
  const bwl::WorkItem wi = wis[w];
  const int R = wi.rows;
  const int per = (wi.ngroups + W - 1) / W;
  const int g0 = min(wave * per, wi.ngroups);
  const int ng = min(per, wi.ngroups - g0);
  const VT* __restrict__ base =
      reinterpret_cast<const VT*>(data + wi.data_off + static_cast<int64_t>(g0) * R * V);
  int64_t orow = 0;
  if (wave == 0 && (wi.part_off < 0 || sp.count) && lane < R) orow = rowmap[wi.out_row + lane];
  const StagedInput<T, 64 * W> in{stage, g0, x, perm, dof, n_in, gidx[wi.gbeg], wi.ngroups * V};
  T acc = 0;
  // every wave passes ready() once, in uniform control flow (its barrier):
  // lanes without a row of their own repeat a loaded one and are not stored
  if (ng == 0) {
    in.ready();
  } else if (R > 32) {
    acc = dot_tall<T, U>(base + min(lane, R - 1), R, ng, in);
  } else {
    const int nsplit = 64 / R;
    const int split = min(lane / R, nsplit - 1);
    acc = dot_short<T, 4>(base + min(lane - split * R, R - 1), R, nsplit, split, ng, in);
    acc = fold_splits(acc, R, nsplit, lane / R, lane);
  }
  wave_sum_put<T, T, W>(acc, red, wi, wave, lane, orow, xt, part, sp);
}

template <typename T, typename OutT>
__global__ __launch_bounds__(64) void k_reduce(const bwl::Reduce* __restrict__ reds, int nred,
                                               const T* __restrict__ part, OutT* out,
                                               const int64_t* __restrict__ perm, int dof,
                                               const int32_t* __restrict__ rowmap) {
  const int r = blockIdx.x;
  if (r >= nred) return;
  const bwl::Reduce rd = reds[r];
  const int t = threadIdx.x;
  if (t >= rd.rows) return;
  // four interleaved partial sums keep four loads in flight; the order of
  // the additions is fixed, so the result is deterministic
  const T* p = part + rd.part_off + t;
  const int R = rd.rows;
  T s0 = 0, s1 = 0, s2 = 0, s3 = 0;
  int q = 0;
  for (; q + 4 <= rd.nparts; q += 4) {
    s0 += p[(q + 0) * R];
    s1 += p[(q + 1) * R];
    s2 += p[(q + 2) * R];
    s3 += p[(q + 3) * R];
  }
  for (; q < rd.nparts; ++q) s0 += p[q * R];
  const T s = (s0 + s1) + (s2 + s3);
  const int64_t orow = rowmap ? rowmap[rd.out_row + t] : static_cast<int64_t>(rd.out_row) + t;
  out[out_index<OutT>(orow, perm, dof)] = static_cast<OutT>(s);
}

// Sub-matrix selection: the input is scattered into the (zeroed) x part of xt
// at the permuted points of the selected columns, and the output gathered
// from a full permuted y at the selected rows.
template <typename T>
__global__ __launch_bounds__(256) void k_scatter_sel(const double* __restrict__ x,
                                                     T* __restrict__ xt,
                                                     const int64_t* __restrict__ src,
                                                     const int64_t* __restrict__ dst, int64_t n,
                                                     int dof) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n * dof) return;
  const int64_t p = i / dof;
  const int64_t c = i - p * dof;
  xt[dof * dst[p] + c] = static_cast<T>(x[dof * src[p] + c]);
}

__global__ __launch_bounds__(256) void k_gather_sel(const double* __restrict__ yfull,
                                                    double* __restrict__ y,
                                                    const int64_t* __restrict__ dst, int64_t n,
                                                    int dof) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n * dof) return;
  const int64_t p = i / dof;
  y[i] = yfull[dof * dst[p] + (i - p * dof)];
}
