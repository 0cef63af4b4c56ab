// Orthogonalisation step of the device GMRES (the caller side of the matvec;
// the reference leaves it to scipy on the host,
// interfaces/python/bigwham4py/bigwham4py.py:362-380).
//
// bw_hip_orthogonalize makes (a copy of) w orthogonal to the k basis vectors V[0..k-1] by
// classical Gram-Schmidt with one re-orthogonalisation pass, and normalises it
// into the next basis vector: four kernels on the caller's stream
//   k_dots          partial dot products V w over chunks of the vectors
//   k_project<1>    w -= V h1 on the chunk, then its partial products V w
//   k_project<2>    w -= V h2 on the chunk, then its partial square norm
//   k_normalize     next = w / ||w||, and the Hessenberg column
// Every kernel adds the partial sums of the one before by itself, in a fixed
// order, so no kernel is spent on reductions.  Bound by reading V twice (its
// chunk comes from L2 the second time in each projection) and, on small
// vectors, by the launches: as torch products the step took eleven launches,
// and a solve on 4 800 DoF (43 iterations) 4.65 ms; with these four, and the
// whole next iteration queued before the host waits, 2.67 ms (16 us a step).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../../include/bigwham_hip.h"

namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr int kMaxChunk = 4096;  // entries of a chunk (LDS)
constexpr int kMaxVectors = 1024;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s, 64);
  return v;
}

// part[j * nb + block] = V[j] . ws over the block's chunk; one wave per vector.
__device__ __forceinline__ void chunk_dots(const double* __restrict__ V, int64_t ldv,
                                           const double* ws, int m, int k, int nb,
                                           double* __restrict__ part) {
  const int lane = threadIdx.x & 63;
  for (int j = threadIdx.x >> 6; j < k; j += kWaves) {
    const double* __restrict__ v = V + j * ldv;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    int i = lane;
    for (; i + 192 < m; i += 256) {
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] += v[i + 64 * q] * ws[i + 64 * q];
    }
    for (; i < m; i += 64) s[0] += v[i] * ws[i];
    const double t = wave_sum((s[0] + s[1]) + (s[2] + s[3]));
    if (lane == 0) part[static_cast<int64_t>(j) * nb + blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(kThreads) void k_dots(const double* __restrict__ V, int64_t ldv,
                                                   const double* __restrict__ w, int64_t n, int k,
                                                   int chunk, int nb, double* __restrict__ part) {
  __shared__ double ws[kMaxChunk];
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * chunk;
  const int m = static_cast<int>(min(static_cast<int64_t>(chunk), n - i0));
  for (int i = threadIdx.x; i < m; i += kThreads) ws[i] = w[i0 + i];
  __syncthreads();
  chunk_dots(V + i0, ldv, ws, m, k, nb, part);
}

// u = w - V h, with h the sums of part_in (u and w may be the same vector).
// STEP 1: part_out = partial products V u, h = h1.
// STEP 2: part_out = partial square norms of u, h = h1 + h2.
template <int STEP>
__global__ __launch_bounds__(kThreads) void k_project(const double* __restrict__ V, int64_t ldv,
                                                      const double* w, double* u, int64_t n, int k,
                                                      int chunk, int nb,
                                                      const double* __restrict__ part_in,
                                                      double* __restrict__ part_out,
                                                      double* __restrict__ h) {
  __shared__ double ws[kMaxChunk];
  __shared__ double hs[kMaxVectors];
  __shared__ double red[kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int j = wave; j < k; j += kWaves) {
    double s = 0.0;
    for (int b = lane; b < nb; b += 64) s += part_in[static_cast<int64_t>(j) * nb + b];
    s = wave_sum(s);
    if (lane == 0) {
      hs[j] = s;
      if (blockIdx.x == 0) h[j] = STEP == 1 ? s : h[j] + s;
    }
  }
  __syncthreads();
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * chunk;
  const int m = static_cast<int>(min(static_cast<int64_t>(chunk), n - i0));
  double sq = 0.0;
  for (int i = threadIdx.x; i < m; i += kThreads) {
    const double* __restrict__ v = V + i0 + i;
    double s = w[i0 + i];
    int j = 0;
    for (; j + 8 <= k; j += 8) {
      double a[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) a[q] = v[(j + q) * ldv];
#pragma unroll
      for (int q = 0; q < 8; ++q) s -= hs[j + q] * a[q];
    }
    for (; j < k; ++j) s -= hs[j] * v[j * ldv];
    u[i0 + i] = s;
    if (STEP == 1)
      ws[i] = s;
    else
      sq += s * s;
  }
  if (STEP == 1) {
    __syncthreads();
    chunk_dots(V + i0, ldv, ws, m, k, nb, part_out);
  } else {
    sq = wave_sum(sq);
    if (lane == 0) red[wave] = sq;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) t += red[q];
      part_out[blockIdx.x] = t;
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_normalize(const double* __restrict__ w, int64_t n,
                                                        int k, int nb,
                                                        const double* __restrict__ part,
                                                        const double* __restrict__ h,
                                                        double* __restrict__ next,
                                                        double* __restrict__ col) {
  __shared__ double norm;
  if (threadIdx.x < 64) {
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += 64) s += part[b];
    s = wave_sum(s);
    if (threadIdx.x == 0) norm = sqrt(s);
  }
  __syncthreads();
  const double hn = norm;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i < n) next[i] = w[i] / hn;
  if (blockIdx.x == 0)
    for (int j = threadIdx.x; j <= k; j += kThreads) col[j] = j < k ? h[j] : hn;
}

// Makes a device current for a scope.  The step stands in for torch operations
// on vectors of any device, which leave the caller's current device as it is.
struct CurrentDevice {
  int before = -1;
  bool ok;

  explicit CurrentDevice(int device) {
    ok = hipGetDevice(&before) == hipSuccess && (before == device || hipSetDevice(device) == hipSuccess);
    if (before == device) before = -1;  // nothing to put back
  }
  ~CurrentDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
  CurrentDevice(const CurrentDevice&) = delete;
  CurrentDevice& operator=(const CurrentDevice&) = delete;
};

// Chunks: at least 256 entries, about 512 workgroups, at most kMaxChunk.
int chunk_of(int64_t n) {
  const int64_t c = std::max<int64_t>(256, (n + 511) / 512);
  return static_cast<int>(std::min<int64_t>(kMaxChunk, (c + 63) / 64 * 64));
}

}  // namespace

extern "C" {

int bw_hip_orthogonalize_work(int64_t n, int k, int64_t* elems) {
  if (!elems || n <= 0 || k <= 0) return BW_EINVAL;
  if (k > kMaxVectors || (n + kThreads - 1) / kThreads > INT32_MAX) return BW_ESHAPE;
  const int64_t nb = (n + chunk_of(n) - 1) / chunk_of(n);
  *elems = n + (2 * static_cast<int64_t>(k) + 1) * nb + k;
  return BW_OK;
}

int bw_hip_orthogonalize(int device, int64_t n, int k, const double* V, int64_t ldv,
                         const double* w, double* next, double* col, double* work, int64_t work_elems,
                         void* stream) {
  int64_t need = 0;
  const int rc = bw_hip_orthogonalize_work(n, k, &need);
  if (rc) return rc;
  if (!V || !w || !next || !col || !work || ldv < n) return BW_EINVAL;
  if (work_elems < need) return BW_ESHAPE;
  const CurrentDevice current(device);
  if (!current.ok) return BW_EHIP;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int chunk = chunk_of(n);
  const int nb = static_cast<int>((n + chunk - 1) / chunk);
  double* u = work;                                // w as it is projected
  double* a = u + n;                               // partial products of w
  double* b = a + static_cast<int64_t>(k) * nb;    // of w after the first projection
  double* c = b + static_cast<int64_t>(k) * nb;    // partial square norms
  double* h = c + nb;
  hipLaunchKernelGGL(k_dots, dim3(nb), dim3(kThreads), 0, st, V, ldv, w, n, k, chunk, nb, a);
  hipLaunchKernelGGL(k_project<1>, dim3(nb), dim3(kThreads), 0, st, V, ldv, w, u, n, k, chunk,
                     nb, a, b, h);
  hipLaunchKernelGGL(k_project<2>, dim3(nb), dim3(kThreads), 0, st, V, ldv, u, u, n, k, chunk,
                     nb, b, c, h);
  const int64_t blocks = (n + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(k_normalize, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, st, u, n,
                     k, nb, c, h, next, col);
  return hipGetLastError() == hipSuccess ? BW_OK : BW_EHIP;
}

}  // extern "C"
