// Device code of the batched matvec (many right-hand sides on MFMA).
// Included by engine.hip only (inside its anonymous namespace), after
// slab_kernels.h.
//
// The slab layout serves as the A operand without change.  NB is the width of
// the gathered input XB[z][NB] (row-major) and of t; a call runs its columns
// in rounds of NB, columns past nk are zero and never stored.  Rounds of 16
// columns move half the input rows and partial sums of 32 (24 300 DoF, 32 and
// 16 columns: FP64 275 and 237 us, FP32 157 and 132); in FP32 a round of 64
// streams the factors once for twice the columns (314 -> 217, 49 152 DoF 590 ->
// 426), and wins from 33 columns on (295 + 257 -> 426).  FP64 stays at 32: its
// time goes with the columns (158 us for one vector).
//
// What bounds them: reads from L2 (53-75 G requests a second up to 32 columns and
// in the single-vector kernel, input rows 40-50 % of them); at 64 columns 46-55 G,
// with the FP32 matrix instructions busy 47-68 % of the time.
//
// A workgroup of W waves takes one work item: the waves take contiguous
// shares of its k-steps, each with a full set of accumulators, and the sums
// over the waves go through LDS, 32 rows at a time, added in wave order.  So
// a slab's 32-wide partial rows reach memory once per workgroup and not once
// per wave, and not at all where a slab is one work item.
#pragma once

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double dblx4 __attribute__((ext_vector_type(4)));

// Rows of XB that a gather writes: x rows 0 .. n - 1, and zeros in the gap up
// to row t0 and in the tail t1 .. size - 1, which padded column groups read.
// (Every call writes them, so that rounds of different widths share a buffer.)
struct GatherRows {
  int64_t n, t0, t1, size;

  int64_t count() const { return t0 + (size - t1); }
  __device__ __forceinline__ int64_t row(int64_t i) const { return i < t0 ? i : t1 + (i - t0); }
};

template <typename T, int NB>
__global__ __launch_bounds__(256) void k_gather_b(const double* __restrict__ X, int64_t xr,
                                                  int64_t xc, int nrhs, T* __restrict__ XB,
                                                  GatherRows g, const int64_t* __restrict__ perm,
                                                  int dof) {
  const int64_t i = g.row(static_cast<int64_t>(blockIdx.x) * (256 / NB) + threadIdx.x / NB);
  const int c = threadIdx.x % NB;
  if (i >= g.size) return;
  T v = 0;
  if (i < g.n && c < nrhs) {
    int64_t src = i;
    if (perm) {
      const int64_t p = i / dof;
      src = dof * perm[p] + (i - p * dof);
    }
    v = static_cast<T>(X[src * xr + c * xc]);
  }
  XB[i * NB + c] = v;
}

// The same gather for a row-major X (unit column stride, even row stride,
// 16-byte aligned): NB / 4 threads per row, four columns each, two 16-byte
// loads and one 16-byte (FP32) or two (FP64) stores per thread.
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_gather_b4(const double* __restrict__ X, int64_t xr,
                                                   int nrhs, T* __restrict__ XB, GatherRows g,
                                                   const int64_t* __restrict__ perm, int dof) {
  constexpr int TPR = NB / 4;  // threads per row
  const int64_t i = g.row(static_cast<int64_t>(blockIdx.x) * (256 / TPR) + threadIdx.x / TPR);
  const int c0 = 4 * (threadIdx.x % TPR);
  if (i >= g.size) return;
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  if (i < g.n) {
    int64_t src = i;
    if (perm) {
      const int64_t p = i / dof;
      src = dof * perm[p] + (i - p * dof);
    }
    const double* __restrict__ row = X + src * xr + c0;
    if (c0 + 4 <= nrhs) {
      const dbl2 a = *reinterpret_cast<const dbl2*>(row);
      const dbl2 b = *reinterpret_cast<const dbl2*>(row + 2);
      v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (c0 + k < nrhs) v[k] = row[k];
    }
  }
  T* dst = XB + i * NB + c0;
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<flt4*>(dst) = flt4{static_cast<float>(v[0]), static_cast<float>(v[1]),
                                         static_cast<float>(v[2]), static_cast<float>(v[3])};
  } else {
    *reinterpret_cast<dbl2*>(dst) = dbl2{v[0], v[1]};
    *reinterpret_cast<dbl2*>(dst + 2) = dbl2{v[2], v[3]};
  }
}

// Where a batched pass writes: pass 1 t (row through rowmap, NB values per
// row), pass 2 Y (row through the point permutation; row stride yr, column
// stride yc; yvec: unit column stride and 16-byte aligned rows).
template <typename T>
struct BatchOut {
  T* tout;
  double* Y;
  int64_t yr, yc;
  int nk;
  int yvec;
  T* part;
  SplitSums sp;
  const int64_t* perm;
  int dof;
  const int32_t* rowmap;
};

template <int PASS, typename T>
__device__ __forceinline__ int64_t batched_row(const BatchOut<T>& o, int idx) {
  if (PASS == 1) return o.rowmap[idx];
  return out_index<double>(idx, o.perm, o.dof);
}

// Stores 16 bytes of sums: columns c .. c + V - 1 of output row `row`.
template <int PASS, int NB, typename T>
__device__ __forceinline__ void batched_put(const BatchOut<T>& o, int64_t row, int c,
                                            typename Vec<T>::type v) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  if (PASS == 1) {
    *reinterpret_cast<VT*>(o.tout + row * NB + c) = v;
    return;
  }
  if (o.yvec && c + V <= o.nk) {
    double* y = o.Y + row * o.yr + c;
#pragma unroll
    for (int k = 0; k < V; k += 2)
      *reinterpret_cast<dbl2*>(y + k) = dbl2{static_cast<double>(v[k]), static_cast<double>(v[k + 1])};
    return;
  }
#pragma unroll
  for (int k = 0; k < V; ++k)
    if (c + k < o.nk) o.Y[row * o.yr + (c + k) * o.yc] = static_cast<double>(v[k]);
}

// 16 bytes of partial sums, as two 8-byte atomic accesses.
template <typename T>
__device__ __forceinline__ void part_put(T* p, typename Vec<T>::type v) {
  typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
  const u64x2 u = __builtin_bit_cast(u64x2, v);
  part_store(reinterpret_cast<uint64_t*>(p), static_cast<uint64_t>(u.x));
  part_store(reinterpret_cast<uint64_t*>(p) + 1, static_cast<uint64_t>(u.y));
}

template <typename T>
__device__ __forceinline__ typename Vec<T>::type part_get(const T* p) {
  typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
  const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
  return __builtin_bit_cast(typename Vec<T>::type, u64x2{part_load(q), part_load(q + 1)});
}

// The end of a split slab's work item, by every thread of the workgroup after
// its partial sums are stored: the last work item of the slab adds them, a
// thread summing one 16-byte vector of right-hand sides of one row over the
// parts, in part order, four parts in flight.
template <int PASS, int NB, int W, typename T>
__device__ __forceinline__ void sum_parts(const bwl::WorkItem& wi, const BatchOut<T>& o) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  constexpr int VPR = NB / V;
  if (wi.part_off < 0 || !o.sp.count) return;
  __shared__ int last;
  const bwl::Reduce rd = o.sp.reds[wi.red];
  stores_arrived();
  __syncthreads();  // of every wave
  if (threadIdx.x == 0) last = count_in(o.sp.count + wi.red, rd.nparts);
  __syncthreads();
  if (!last) return;
  const T* __restrict__ base = o.part + static_cast<int64_t>(rd.part_off) * NB;
  const int nvec = rd.rows * VPR;
  for (int e = threadIdx.x; e < nvec; e += 64 * W) {
    const int64_t row = batched_row<PASS>(o, rd.out_row + e / VPR);
    const T* p = base + static_cast<int64_t>(e) * V;
    const int64_t stride = static_cast<int64_t>(nvec) * V;
    VT sum = {};
    int q = 0;
    for (; q + 4 <= rd.nparts; q += 4) {
      const VT a = part_get(p + (q + 0) * stride);
      const VT b = part_get(p + (q + 1) * stride);
      const VT c = part_get(p + (q + 2) * stride);
      const VT d = part_get(p + (q + 3) * stride);
      sum += a;
      sum += b;
      sum += c;
      sum += d;
    }
    VT v[3] = {};
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (q + k < rd.nparts) v[k] = part_get(p + (q + k) * stride);
#pragma unroll
    for (int k = 0; k < 3; ++k) sum += v[k];
    batched_put<PASS, NB>(o, row, (e % VPR) * V, sum);
  }
  if (threadIdx.x == 0) part_store(o.sp.count + wi.red, int32_t{0});
}

// Sums the W images lds[wave][32][NB] (rows r0 .. r0 + 31 of the work item,
// written by the waves before the call) in wave order and stores the rows
// below R.  Every thread of the workgroup calls it.
template <int PASS, int NB, int W, typename T>
__device__ __forceinline__ void wave_sum_store(const T* lds, const bwl::WorkItem& wi, int r0,
                                               const BatchOut<T>& o) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  constexpr int VPR = NB / V;         // 16-byte vectors per row
  constexpr int N = 32 * VPR;         // vectors of one image
  constexpr int T0 = 64 * W;
  constexpr int E = (N + T0 - 1) / T0;
  int64_t orow[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int q = e * T0 + static_cast<int>(threadIdx.x);
    const int row = min(r0 + q / VPR, wi.rows - 1);  // clamped, in bounds
    orow[e] = wi.part_off < 0 ? batched_row<PASS>(o, wi.out_row + row) : 0;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int q = e * T0 + static_cast<int>(threadIdx.x);
    const int row = r0 + q / VPR, c = (q % VPR) * V;
    if (q >= N || row >= wi.rows) continue;
    VT s = *reinterpret_cast<const VT*>(lds + q * V);
#pragma unroll
    for (int k = 1; k < W; ++k) s += *reinterpret_cast<const VT*>(lds + k * 32 * NB + q * V);
    if (wi.part_off < 0) {
      batched_put<PASS, NB>(o, orow[e], c, s);
    } else {
      T* pp = o.part + (static_cast<int64_t>(wi.part_off) + row) * NB + c;
      if (o.sp.count)
        part_put(pp, s);
      else  // read once by k_reduce_b: nontemporal
        __builtin_nontemporal_store(s, reinterpret_cast<VT*>(pp));
    }
  }
}

// Where a lane's two rows of a 32-row-tile item lie: the 16-byte vectors of
// column group g + half (at most the last).
//
// The rows of a slab.
struct SlabRows {
  int R, ng, row0, row1;
  __device__ __forceinline__ int2 vectors(int g, int half) const {
    const int b = min(g + half, ng - 1) * R;
    return {b + row0, b + row1};
  }
};

// A window of up to 64 rows over all slabs of a pass-1 column cluster (they read
// the same input), each row with the offset and the stride of its own slab from
// the row table (Program::rowtab).  The layout makes windows only where these
// numbers fit (less than 2^20 groups a slab).
struct WindowRows {
  int ng;
  int off0, str0, off1, str1;
  __device__ __forceinline__ int2 vectors(int g, int half) const {
    const int c = min(g + half, ng - 1);
    return {__mul24(c, str0) + off0, __mul24(c, str1) + off1};
  }
};

// FP32, v_mfma_f32_32x32x2f32: lanes 0-31 read rows 0-31 of column group g,
// lanes 32-63 rows 0-31 of group g + 1, 16 bytes (4 columns) each; element s
// of a lane's vector is A[row][k] of MFMA step s, with k = lane / 32
// selecting the group.  The accumulator holds rows x right-hand sides:
// element j of lane l is row 8*(j/4) + 4*(l/32) + j%4, column l % 32.
//
// The loads run through a ring of D register buffers in the order they are
// consumed (KU group pairs per step): the MFMAs of buffer j run, then buffer
// j is refilled with the step D ahead, so D - 1 steps are in flight.  Loads
// and MFMAs are unconditional, so the loop body is one basic block with the
// same waits on every path: past the last step the loads read clamped,
// in-bounds addresses and the MFMAs get B = 0.
//
// The B operands are staged through LDS: a column group's four input rows
// (4 NB contiguous floats) arrive as NC 16-byte loads per lane of its
// half-wave, are written to the wave's own LDS slot and read back in the MFMA
// layout one step ahead of their MFMAs.  LDS operations of a wave run in
// order, so a read sees the write before it.
template <int NC, int KU, int D, bool TWO, typename Rows>
__device__ __forceinline__ void mfma32_stream(const flt4* __restrict__ base,
                                              const int32_t* __restrict__ gi,
                                              const float* __restrict__ XB, int ng, const Rows& rows, int half,
                                              int r0, float* slot, floatx16 (&acc)[2][NC]) {
  constexpr int NB = 32 * NC;
  constexpr int G = 2 * KU;  // groups per step
  const int nsteps = (ng + G - 1) / G;
  flt4 a0[D][KU], a1[D][KU];
  flt4 bq[D][KU][NC];  // this lane's 16-byte pieces of the four input rows of group 2u + half
  int zz[D][KU];       // input offset of group 2u + half for the step buffer k gets next
  float bn[KU][4][NC]; // B of the next step to multiply, read back from LDS
  auto gz = [&](int step, int u) { return gi[min(step * G + 2 * u + half, ng - 1)]; };
  auto load = [&](int step, const int (&z)[KU], flt4 (&x0)[KU], flt4 (&x1)[KU],
                  flt4 (&bb)[KU][NC]) {
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int2 at = rows.vectors(step * G + 2 * u, half);
      x0[u] = __builtin_nontemporal_load(base + at.x);
      if (TWO) x1[u] = __builtin_nontemporal_load(base + at.y);
      // rows z .. z + 3 of XB are contiguous and 128-byte aligned; 32-bit
      // offsets (xt_size * NB < 2^32, checked by the host)
      const uint32_t zo = static_cast<uint32_t>(z[u]) * NB + 4 * r0;
#pragma unroll
      for (int c = 0; c < NC; ++c) bb[u][c] = *reinterpret_cast<const flt4*>(XB + zo + 128 * c);
    }
  };
  auto stage_b = [&](const flt4 (&bb)[KU][NC]) {
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        *reinterpret_cast<flt4*>(slot + (2 * u + half) * 4 * NB + 128 * c + 4 * r0) = bb[u][c];
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          bn[u][s][c] = slot[(2 * u + half) * 4 * NB + s * NB + 32 * c + r0];
  };
  // Sums of one trip of the ring (D steps): the first MFMA of a trip starts
  // them from zero, and they are added to acc when the trip is over.  Short
  // chains instead of a wave's whole share keep the FP32 rounding error of long
  // work items down (49 152-DoF 3DR0, 32 right-hand sides: 1.06e-7 against 64
  // bits with chains of 12 MFMAs; one chain per wave 2.5e-7).
  floatx16 p[2][NC];
  auto compute = [&](int step, bool first, const flt4 (&x0)[KU], const flt4 (&x1)[KU]) {
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const bool ok = step * G + 2 * u + half < ng;
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const float bv = ok ? bn[u][s][c] : 0.0f;
          const bool zero = first && u == 0 && s == 0;
          p[0][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(x0[u][s], bv,
                                                         zero ? floatx16{0} : p[0][c], 0, 0, 0);
          if (TWO)
            p[1][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(x1[u][s], bv,
                                                           zero ? floatx16{0} : p[1][c], 0, 0, 0);
        }
    }
  };
#pragma unroll
  for (int k = 0; k < D; ++k)
#pragma unroll
    for (int u = 0; u < KU; ++u) zz[k][u] = gz(k, u);
#pragma unroll
  for (int k = 0; k < D; ++k) {
    __builtin_amdgcn_sched_barrier(0);
    load(k, zz[k], a0[k], a1[k], bq[k]);
#pragma unroll
    for (int u = 0; u < KU; ++u) zz[k][u] = gz(k + D, u);
  }
  __builtin_amdgcn_sched_barrier(0);
  stage_b(bq[0]);
  for (int s0 = 0; s0 < nsteps; s0 += D) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int s = s0 + j;
      __builtin_amdgcn_sched_barrier(0);
      compute(s, j == 0, a0[j], a1[j]);  // past the last step: B = 0, adds nothing
      __builtin_amdgcn_sched_barrier(0);
      stage_b(bq[(j + 1) % D]);
      __builtin_amdgcn_sched_barrier(0);
      load(s + D, zz[j], a0[j], a1[j], bq[j]);
#pragma unroll
      for (int u = 0; u < KU; ++u) zz[j][u] = gz(s + 2 * D, u);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      acc[0][c] += p[0][c];
      if (TWO) acc[1][c] += p[1][c];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

// WIN: the items are windows (pass 1 of long operators, rounds of 64 columns).
template <int PASS, int NC, int W, bool WIN>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(NC > 1 ? 2 : 3))) void
k_slab_mfma32(const bwl::WorkItem* __restrict__ wis, XcdSplit xs,
              const int32_t* __restrict__ gidx, const float* __restrict__ data,
              const float* __restrict__ XB, const int64_t* __restrict__ rowtab, BatchOut<float> o) {
  // The ring: one group pair per step, three steps (2, 3 and 4 steps: 24 300 DoF,
  // 100 columns 454, 447 and 457 us; 16 cracks, 32 columns 52.7, 49.1 and 47.9;
  // 49 152 DoF, 32 columns 302, 306 and 307; two pairs, three steps 457, 54.2, 317)
  constexpr int NB = 32 * NC, KU = 1, D = 3, G = 4;
  __shared__ __align__(16) float lds[W * 32 * NB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int w = xcd_work_item(xs, blockIdx.x);
  if (w < 0) return;
  const bwl::WorkItem wi = wis[w];
  const int R = __builtin_amdgcn_readfirstlane(wi.rows);
  // this wave's share of the column groups
  const int nst = (wi.ngroups + G - 1) / G;
  const int g0 = __builtin_amdgcn_readfirstlane(G * (nst * wave / W));
  const int ng = __builtin_amdgcn_readfirstlane(min(wi.ngroups, G * (nst * (wave + 1) / W)) - g0);
  const int half = lane >> 5;  // which group of the pair
  const int r0 = lane & 31;
  const int32_t* __restrict__ gi = gidx + __builtin_amdgcn_readfirstlane(wi.gbeg) + g0;
  floatx16 acc[2][NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[0][c] = acc[1][c] = floatx16{0};
  float* mine = lds + wave * 32 * NB;  // the wave's B slot, then its image of the sums
  const bool two = R > 32;
  auto run = [&](const flt4* __restrict__ base, const auto& rows) {
    if (ng <= 0) return;
    if (two)
      mfma32_stream<NC, KU, D, true>(base, gi, XB, ng, rows, half, r0, mine, acc);
    else
      mfma32_stream<NC, KU, D, false>(base, gi, XB, ng, rows, half, r0, mine, acc);
  };
  const int row0 = min(r0, R - 1), row1 = min(r0 + 32, R - 1);
  if constexpr (WIN) {
    const int64_t* __restrict__ tab = rowtab + wi.out_row;
    const int64_t e0 = tab[row0], e1 = tab[row1], e = tab[0] >> 8;
    const int64_t first =
        static_cast<int64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(e >> 32))) << 32 |
        static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(e)));
    const int s0 = e0 & 0xff, s1 = e1 & 0xff;
    const int g = static_cast<int>(wi.data_off) + g0;  // the wave's first group
    const WindowRows rows{ng, static_cast<int>((e0 >> 8) - first) + g * s0, s0,
                          static_cast<int>((e1 >> 8) - first) + g * s1, s1};
    run(reinterpret_cast<const flt4*>(data) + first, rows);
  } else {
    run(reinterpret_cast<const flt4*>(data + wi.data_off) + static_cast<int64_t>(g0) * R,
        SlabRows{R, ng, row0, row1});
  }
  auto put = [&](const floatx16 (&a)[NC]) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int j = 0; j < 16; ++j)
        mine[(8 * (j >> 2) + 4 * half + (j & 3)) * NB + 32 * c + r0] = a[c][j];
  };
  put(acc[0]);
  wave_sum_store<PASS, NB, W>(lds, wi, 0, o);
  if (two) {
    __syncthreads();  // the first image has been read
    put(acc[1]);
    wave_sum_store<PASS, NB, W>(lds, wi, 32, o);
  }
  sum_parts<PASS, NB, W>(wi, o);
}

// 16-row tiles: v_mfma_f64_16x16x4f64 and v_mfma_f32_16x16x4f32.  One k-step
// covers four column groups: as a tile's A operand lane l holds the 16-byte
// vector of row l % 16 in group 4 step + l / 16, and element s of it is A[i][k]
// of MFMA s with i = l % 16, k = l / 16; B[k][n] = XB[z(group) + s][n], n = l % 16
// (+ 16 per column tile).
template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> {
  typedef dblx4 acc_t;
  // element r of a lane's accumulator is row l / 16 + 4 r (measured on gfx950
  // with one-hot operands), column l % 16
  static __device__ __forceinline__ int row(int kq, int r) { return kq + 4 * r; }
  static __device__ __forceinline__ acc_t mfma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma16<float> {
  typedef floatx4 acc_t;
  static __device__ __forceinline__ int row(int kq, int r) { return 4 * kq + r; }
  static __device__ __forceinline__ acc_t mfma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// The k-steps of a wave for a slab of NT 16-row tiles (NT a template argument,
// so the loop body is one basic block); ring of D buffers as in mfma32_stream.
template <typename T, int NT, int NC, int D>
__device__ __forceinline__ void mfma16_stream(const typename Vec<T>::type* __restrict__ base,
                                              const int32_t* __restrict__ gi,
                                              const T* __restrict__ XB, int ng, int R, int kq,
                                              int i16, typename Mfma16<T>::acc_t (&acc)[4][NC]) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  constexpr int NB = 16 * NC;
  int rowc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) rowc[t] = min(16 * t + i16, R - 1);
  const int nsteps = (ng + 3) >> 2;
  VT a[D][NT];
  T b[D][NC][V];
  int zz[D];  // input offset of the step buffer q is refilled with next
  auto gz = [&](int step) { return gi[min(4 * step + kq, ng - 1)]; };
  auto load = [&](int step, int z, VT (&aa)[NT], T (&bb)[NC][V]) {
    const int ga = min(4 * step + kq, ng - 1);
#pragma unroll
    for (int t = 0; t < NT; ++t) aa[t] = __builtin_nontemporal_load(base + ga * R + rowc[t]);
    const uint32_t zo = static_cast<uint32_t>(z) * NB + i16;  // < 2^32, checked by the host
#pragma unroll
    for (int s = 0; s < V; ++s)
#pragma unroll
      for (int c = 0; c < NC; ++c) bb[c][s] = XB[zo + s * NB + 16 * c];
  };
  // FP32: sums of two steps, added to acc after them (short chains, as in
  // mfma32_stream: 900-DoF mode-1, 5 right-hand sides, errors against 64 bits
  // 1.4e-7 with chains of a whole trip)
  constexpr bool kTrip = sizeof(T) == 4;
  typename Mfma16<T>::acc_t p[kTrip ? NT : 1][NC];
  auto flush = [&]() {
    if constexpr (kTrip) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[t][c] += p[t][c];
    }
  };
  auto compute = [&](int step, bool first, const VT (&aa)[NT], const T (&bb)[NC][V]) {
    const bool ok = 4 * step + kq < ng;
#pragma unroll
    for (int s = 0; s < V; ++s)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const T bv = ok ? bb[c][s] : T(0);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          if constexpr (kTrip)
            p[t][c] = Mfma16<T>::mfma(
                aa[t][s], bv, first && s == 0 ? typename Mfma16<T>::acc_t{0, 0, 0, 0} : p[t][c]);
          else
            acc[t][c] = Mfma16<T>::mfma(aa[t][s], bv, acc[t][c]);
        }
      }
  };
#pragma unroll
  for (int q = 0; q < D; ++q) zz[q] = gz(q);
#pragma unroll
  for (int q = 0; q < D; ++q) {
    __builtin_amdgcn_sched_barrier(0);
    load(q, zz[q], a[q], b[q]);
    zz[q] = gz(q + D);
  }
  for (int s0 = 0; s0 < nsteps; s0 += D) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int st = s0 + j;
      __builtin_amdgcn_sched_barrier(0);
      compute(st, j % 2 == 0, a[j], b[j]);  // past the last step: B = 0, adds nothing
      __builtin_amdgcn_sched_barrier(0);
      load(st + D, zz[j], a[j], b[j]);
      zz[j] = gz(st + 2 * D);
      if (j % 2 == 1 || j == D - 1) {
        __builtin_amdgcn_sched_barrier(0);
        flush();
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

template <typename T, int PASS, int NC, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(3))) void
k_slab_mfma16(const bwl::WorkItem* __restrict__ wis, XcdSplit xs,
              const int32_t* __restrict__ gidx, const T* __restrict__ data,
              const T* __restrict__ XB, BatchOut<T> o) {
  typedef typename Vec<T>::type VT;
  constexpr int NB = 16 * NC, D = sizeof(T) * NC > 8 ? 3 : 4;
  __shared__ __align__(16) T lds[W * 32 * NB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int w = xcd_work_item(xs, blockIdx.x);
  if (w < 0) return;
  const bwl::WorkItem wi = wis[w];
  const int R = wi.rows;
  const int nst = (wi.ngroups + 3) >> 2;
  const int g0 = __builtin_amdgcn_readfirstlane(4 * (nst * wave / W));
  const int ng = __builtin_amdgcn_readfirstlane(min(wi.ngroups, 4 * (nst * (wave + 1) / W)) - g0);
  const int kq = lane >> 4, i16 = lane & 15;
  const VT* __restrict__ base =
      reinterpret_cast<const VT*>(data + wi.data_off) + static_cast<int64_t>(g0) * R;
  const int32_t* __restrict__ gi = gidx + wi.gbeg + g0;
  const int ntile = (R + 15) >> 4;  // 16-row tiles in use, wave-uniform
  typename Mfma16<T>::acc_t acc[4][NC];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[t][c] = typename Mfma16<T>::acc_t{0, 0, 0, 0};
  if (ng > 0) {
    switch (ntile) {
      case 1: mfma16_stream<T, 1, NC, D>(base, gi, XB, ng, R, kq, i16, acc); break;
      case 2: mfma16_stream<T, 2, NC, D>(base, gi, XB, ng, R, kq, i16, acc); break;
      case 3: mfma16_stream<T, 3, NC, D>(base, gi, XB, ng, R, kq, i16, acc); break;
      default: mfma16_stream<T, 4, NC, D>(base, gi, XB, ng, R, kq, i16, acc);
    }
  }
  T* mine = lds + wave * 32 * NB;
  auto put = [&](int t0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          mine[(16 * t + Mfma16<T>::row(kq, r)) * NB + 16 * c + i16] =
              t0 == 0 ? acc[t][c][r] : acc[2 + t][c][r];
  };
  put(0);
  wave_sum_store<PASS, NB, W>(lds, wi, 0, o);
  if (R > 32) {
    __syncthreads();  // the first image has been read
    put(2);
    wave_sum_store<PASS, NB, W>(lds, wi, 32, o);
  }
  sum_parts<PASS, NB, W>(wi, o);
}

// One workgroup per split slab; a thread sums one 16-byte vector of
// right-hand sides of one row over the parts, in part order, four parts in
// flight (nontemporal loads: each partial row is read once).
template <int PASS, int NB, typename T>
__global__ __launch_bounds__(256) void k_reduce_b(const bwl::Reduce* __restrict__ reds, int nred,
                                                  BatchOut<T> o) {
  typedef typename Vec<T>::type VT;
  constexpr int V = Vec<T>::V;
  constexpr int VPR = NB / V;
  const int r = blockIdx.x;
  if (r >= nred) return;
  const bwl::Reduce rd = reds[r];
  const VT* __restrict__ base_p =
      reinterpret_cast<const VT*>(o.part + static_cast<int64_t>(rd.part_off) * NB);
  const int nvec = rd.rows * VPR;
  const int64_t stride = nvec;
  for (int e = threadIdx.x; e < nvec; e += blockDim.x) {
    VT sum = {};
    int q = 0;
    for (; q + 4 <= rd.nparts; q += 4) {
      const VT a = __builtin_nontemporal_load(&base_p[(q + 0) * stride + e]);
      const VT b = __builtin_nontemporal_load(&base_p[(q + 1) * stride + e]);
      const VT c = __builtin_nontemporal_load(&base_p[(q + 2) * stride + e]);
      const VT d = __builtin_nontemporal_load(&base_p[(q + 3) * stride + e]);
      sum += a;
      sum += b;
      sum += c;
      sum += d;
    }
    for (; q < rd.nparts; ++q) sum += __builtin_nontemporal_load(&base_p[q * stride + e]);
    batched_put<PASS, NB>(o, batched_row<PASS>(o, rd.out_row + e / VPR), (e % VPR) * V, sum);
  }
}
