// k_util.hip -- fills and exclusive scans used by the expansion pipeline.
// No hipMemset on the expansion stream: every clear is a kernel, so the
// pipeline stays capturable in a HIP graph.
#include <hip/hip_runtime.h>

#include "dp_internal.h"

namespace {

__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
    p[t] = v;
}

__global__ void k_begin(long long* __restrict__ counters, int n, int32_t* __restrict__ a, int64_t na,
                        int32_t* __restrict__ b, int64_t nb, dp_marks marks) {
  dp_mark(marks);
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  if (t0 < n) counters[t0] = 0;
  for (int64_t t = t0; t < na; t += step) a[t] = 0;
  for (int64_t t = t0; t < nb; t += step) b[t] = 0;
}

// One workgroup, each thread a contiguous chunk: the chunk sums scanned with
// wave shuffles and one exchange of the 16 wave sums (a step-by-step scan
// of 1024 sums in LDS paid 20 barriers, 4.7 us at 4096 elements against 3.0).
__global__ __launch_bounds__(1024) void k_scan_small(const int32_t* src, int32_t* dst, int64_t n,
                                                     int32_t* total, int64_t cap, long long* counters, int slot) {
  __shared__ long long s[16];
  const int t = threadIdx.x, lane = t % 64;
  const int64_t chunk = (n + 1023) / 1024;
  const int64_t b = t * chunk;
  const int64_t e = b + chunk < n ? b + chunk : n;
  long long sum = 0;
  for (int64_t k = b; k < e; ++k) sum += src[k];
  long long incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const long long u = __shfl_up(incl, d, 64);
    if (lane >= d) incl += u;
  }
  if (lane == 63) s[t / 64] = incl;
  __syncthreads();
  long long run = incl - sum;
  for (int k = 0; k < t / 64; ++k) run += s[k];
  for (int64_t k = b; k < e; ++k) {
    int32_t v = src[k];
    dst[k] = (int32_t)run;
    run += v;
  }
  if (t == 1023) {
    long long tot = run;  // thread 1023 owns the last chunk
    dst[n] = (int32_t)tot;
    if (total) *total = (int32_t)(tot < cap ? tot : cap);
    if (slot >= 0) counters[slot] = tot;
    if (tot > cap) counters[DPC_OVERFLOW] = 1;
  }
}

// Row-major pinned host memory ([n][nx], then n values of g) into component
// arrays: one launch of a few us, read over the host link.
__global__ void k_upload_rows(const double* __restrict__ src, int32_t n, int nx, int32_t ncap,
                              double* __restrict__ nodes, double* __restrict__ g) {
  const int64_t total = (int64_t)n * (nx + (g ? 1 : 0));
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const double v = src[t];
    if (t < (int64_t)n * nx) nodes[(t % nx) * (int64_t)ncap + t / nx] = v;
    else g[t - (int64_t)n * nx] = v;
  }
}

__global__ void k_put_counters(const long long* __restrict__ c, int n, long long* __restrict__ host) {
  if ((int)threadIdx.x < n) host[threadIdx.x] = c[threadIdx.x];
}

// The results of pairs [q0, q0 + n) as the caller's arrays hold them, written
// straight into pinned host memory: no final state, g or h but of a FREE pair
// before its node's cap (NaN otherwise), no goal index past the cap.
__global__ __launch_bounds__(256) void k_pack_pairs(dp_pack a) {
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < a.n; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q = a.q0 + t;
    const int8_t v = a.verdict[q], r = a.res[q];
    const bool capped = r == DP_R_CAPPED, has = v == DP_V_FREE && !capped;
    if (a.o_node) a.o_node[t] = a.node[q];
    if (a.o_prim) a.o_prim[t] = a.prim[q];
    if (a.o_verdict) a.o_verdict[t] = v;
    if (a.o_firstk) a.o_firstk[t] = a.firstk[q];
    if (a.o_goal) a.o_goal[t] = capped ? -1 : a.goal[q];
    if (a.o_res) a.o_res[t] = r;
    if (a.o_g) a.o_g[t] = has ? a.g[q] : __longlong_as_double(0x7ff8000000000000ll);
    if (a.o_h) a.o_h[t] = has ? a.h[q] : __longlong_as_double(0x7ff8000000000000ll);
  }
  if (a.o_final) {
    const int nx = a.nx;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < a.n * nx;
         t += (int64_t)gridDim.x * blockDim.x) {
      const int64_t i = t / nx, q = a.q0 + i;
      const int k = (int)(t - i * nx);
      const bool has = a.verdict[q] == DP_V_FREE && a.res[q] != DP_R_CAPPED;
      a.o_final[t] = has ? a.fin[(int64_t)k * a.pcap + q] : __longlong_as_double(0x7ff8000000000000ll);
    }
  }
}

}  // namespace

void dp_upload_rows(const double* src, int32_t n, int nx, int32_t cap, double* rows, double* g, hipStream_t s) {
  k_upload_rows<<<dp_grid_blocks((int64_t)n * (nx + 1), 256, 1024), 256, 0, s>>>(src, n, nx, cap, rows, g);
}
void dp_put_counters(dp_ctx* c, hipStream_t s) {
  static_assert(DPC_COUNT <= 64, "one wave copies the counters");
  k_put_counters<<<1, 64, 0, s>>>(c->d_counters, DPC_COUNT, c->h_pinned);
}
void dp_pack_pairs(const dp_pack& a, hipStream_t s) {
  k_pack_pairs<<<dp_grid_blocks(a.n * (a.o_final ? a.nx : 1), 256, 2048), 256, 0, s>>>(a);
}

void dp_fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t s) {
  if (n <= 0) return;
  k_fill_i32<<<dp_grid_blocks(n, 256, 4096), 256, 0, s>>>(p, n, v);
}

void dp_begin(long long* counters, int32_t* a, int64_t na, int32_t* b, int64_t nb, dp_marks marks, hipStream_t s) {
  k_begin<<<dp_grid_blocks(na + nb, 256, 2048), 256, 0, s>>>(counters, DPC_COUNT, a, na, b, nb, marks);
}

void dp_scan_small(const int32_t* src, int32_t* dst, int64_t n, int32_t* total, int64_t cap, long long* counters,
                   int slot, hipStream_t s) {
  k_scan_small<<<1, 1024, 0, s>>>(src, dst, n, total, cap, counters, slot);
}

// Growth frees a buffer earlier kernels of the batch may still read, so the
// device is drained first (growth happens on the first batches only).
int dp_ensure_i32(int32_t** p, int64_t* cap, int64_t need) {
  if (*cap >= need && *p) return DP_OK;
  dp_bump_epoch();
  DP_HIP_RET(hipDeviceSynchronize());
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  DP_HIP_RET(hipMalloc(p, sizeof(int32_t) * (size_t)(need > 0 ? need : 1)));
  *cap = need;
  return DP_OK;
}

int dp_ensure_f64(double** p, int64_t* cap, int64_t need) {
  if (*cap >= need && *p) return DP_OK;
  dp_bump_epoch();
  DP_HIP_RET(hipDeviceSynchronize());
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  DP_HIP_RET(hipMalloc(p, sizeof(double) * (size_t)(need > 0 ? need : 1)));
  *cap = need;
  return DP_OK;
}

int dp_ensure_u64(uint64_t** p, int64_t* cap, int64_t need) {
  if (*cap >= need && *p) return DP_OK;
  dp_bump_epoch();
  DP_HIP_RET(hipDeviceSynchronize());
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *cap = 0;
  DP_HIP_RET(hipMalloc(p, sizeof(uint64_t) * (size_t)(need > 0 ? need : 1)));
  *cap = need;
  return DP_OK;
}
