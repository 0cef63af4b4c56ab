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

__device__ __forceinline__ int xcd_work_item(const XcdSplit& xs) {
  const int x = blockIdx.x % bwl::kXcds;
  const int w = xs.s[x] + static_cast<int>(blockIdx.x / bwl::kXcds);
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

template <typename OutT>
__device__ __forceinline__ int64_t out_index(int64_t idx, const int64_t* perm, int dof) {
  if (!perm) return idx;
  // row indices fit in 32 bits (checked when the layout is built)
  const int i = static_cast<int>(idx);
  const int p = i / dof;
  return dof * perm[p] + (i - p * dof);
}

// Dot products of a wave's column groups with more than 32 rows: one column
// group per step for the whole wavefront, so the group offset and the input
// entries are wave-uniform (scalar loads).  U: 16-byte loads in flight per lane.
template <typename T, int U>
__device__ __forceinline__ T dot_tall(const typename Vec<T>::type* __restrict__ p, int R,
                                      const int32_t* __restrict__ gi, int ng,
                                      const T* __restrict__ xin) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  T acc0 = 0, acc1 = 0;
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
      for (int u = 0; u < U; ++u) zz[u] = gi[g0 + u];
#pragma unroll
      for (int u = 0; u < U; ++u) buf[u] = __builtin_nontemporal_load(p + (g0 + u) * R);
    };
    auto use = [&](const VT (&buf)[U], const int (&zz)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // unsigned: no sign extension of the loaded offset is placed
        // (and waited for) next to its load
        const uint32_t z = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(zz[u]));
#pragma unroll
        for (int v = 0; v < V; ++v) {
          if (u & 1)
            acc1 += buf[u][v] * xin[z + v];
          else
            acc0 += buf[u][v] * xin[z + v];
        }
      }
    };
    load(0, a, za);
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
  // The last, partial batch in one memory round trip: 4, 8 or U loads
  // (clamped to the last group, in bounds), of which the first rem are used.
  const int g = nfull * U, rem = ng - g;
  auto tail = [&](auto N) {
    constexpr int n = decltype(N)::value;
    VT a[n];
    int z[n];
#pragma unroll
    for (int u = 0; u < n; ++u) z[u] = gi[g + min(u, rem - 1)];
#pragma unroll
    for (int u = 0; u < n; ++u) a[u] = __builtin_nontemporal_load(p + (g + min(u, rem - 1)) * R);
#pragma unroll
    for (int u = 0; u < n; ++u) {
      const uint32_t zu = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(z[u]));
      if (u < rem) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
          if (u & 1)
            acc1 += a[u][v] * xin[zu + v];
          else
            acc0 += a[u][v] * xin[zu + v];
        }
      }
    }
  };
  if (rem > 8)
    tail(std::integral_constant<int, (U > 8 ? U : 8)>{});
  else if (rem > 4)
    tail(std::integral_constant<int, (U > 4 ? 8 : 4)>{});
  else if (rem > 0)
    tail(std::integral_constant<int, 4>{});
  return acc0 + acc1;
}

// Dot products of a wave's column groups with at most 32 rows: nsplit = 64 / R
// groups at a time (lane = split * R + row; `p` points at the lane's row), U
// of them per step.  As in dot_tall, a step's loads (factors and input
// entries) go out before the FMAs of the step before, through two register
// buffers; the input offsets are loaded two steps ahead, so that one memory
// round trip covers a step.  Offsets and groups past the end are clamped (in
// bounds) and not used.
template <typename T, int U>
__device__ __forceinline__ T dot_short(const typename Vec<T>::type* __restrict__ p, int R,
                                       int nsplit, int split, const int32_t* __restrict__ gi,
                                       int ng, const T* __restrict__ xin) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  T acc0 = 0, acc1 = 0;
  const int step = U * nsplit;
  const int n = (ng + step - 1) / step;
  VT a[U], b[U];
  T xa[U][V], xb[U][V];
  int za[U], zb[U];
  auto load_z = [&](int s, int (&z)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) z[u] = gi[min(s * step + split + u * nsplit, ng - 1)];
  };
  auto load = [&](int s, VT (&f)[U], T (&x)[U][V], int (&z)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      f[u] = __builtin_nontemporal_load(p + min(s * step + split + u * nsplit, ng - 1) * R);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) x[u][v] = xin[z[u] + v];
    load_z(s + 2, z);
  };
  auto use = [&](const VT (&f)[U], const T (&x)[U][V]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        if (u & 1)
          acc1 += f[u][v] * x[u][v];
        else
          acc0 += f[u][v] * x[u][v];
      }
  };
  auto use_last = [&](const VT (&f)[U], const T (&x)[U][V]) {  // step n - 1
#pragma unroll
    for (int u = 0; u < U; ++u)
      if ((n - 1) * step + split + u * nsplit < ng) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
          if (u & 1)
            acc1 += f[u][v] * x[u][v];
          else
            acc0 += f[u][v] * x[u][v];
        }
      }
  };
  load_z(0, za);
  load_z(1, zb);
  load(0, a, xa, za);
  int s = 0;
  for (; s + 2 < n; s += 2) {
    __builtin_amdgcn_sched_barrier(0);
    load(s + 1, b, xb, zb);
    __builtin_amdgcn_sched_barrier(0);
    use(a, xa);
    __builtin_amdgcn_sched_barrier(0);
    load(s + 2, a, xa, za);
    __builtin_amdgcn_sched_barrier(0);
    use(b, xb);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (s + 2 == n) {
    load(s + 1, b, xb, zb);
    __builtin_amdgcn_sched_barrier(0);
    use(a, xa);
    __builtin_amdgcn_sched_barrier(0);
    use_last(b, xb);
  } else {
    use_last(a, xa);
  }
  return acc0 + acc1;
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
                                                 const int64_t* __restrict__ perm, int dof,
                                                 const int32_t* __restrict__ rowmap) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int w = xcd_work_item(xs);
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
  // output row of this lane, requested before the stream
  int64_t orow = 0;
  if (wave == 0 && wi.part_off < 0 && lane < R) {
    // pass 1 rows go to their t entries through the row map
    const int64_t r = rowmap ? rowmap[wi.out_row + lane] : static_cast<int64_t>(wi.out_row) + lane;
    orow = out_index<OutT>(r, perm, dof);
  }
  T acc = 0;
  if (R > 32) {
    if (lane < R && ng > 0) acc = dot_tall<T, U>(base + lane, R, gi, ng, xin);
  } else {
    const int nsplit = 64 / R;
    const int split = lane / R;
    if (split < nsplit && ng > 0)
      acc = dot_short<T, 4>(base + (lane - split * R), R, nsplit, split, gi, ng, xin);
    // fold the column splits onto lanes 0..R-1, in split order
    for (int s = 1; s < nsplit; ++s) {
      const T o = __shfl(acc, lane + s * R, 64);
      if (split == 0) acc += o;
    }
  }
  if constexpr (W > 1) {
    __shared__ T red[W][64];
    if (wave > 0 && lane < R) red[wave][lane] = acc;
    __syncthreads();
    if (wave > 0) return;
    if (lane < R) {
#pragma unroll
      for (int k = 1; k < W; ++k) acc += red[k][lane];
    }
  }
  if (lane >= R) return;
  if (wi.part_off < 0)
    out[orow] = static_cast<OutT>(acc);
  else  // split slab: the partial sums are added in work-item order by k_reduce
    part[wi.part_off + lane] = acc;
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
