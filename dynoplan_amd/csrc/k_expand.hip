// k_expand.hip -- gfx950 kernels of the batched db-A* expansion.
//
// Pipeline of one dp_expand (all on one stream, no host round trip):
//   k_begin           counters, counts and grid cells cleared, one launch
//   k_app_blk         applicability query nearestR(c, alpha*delta) over primitive
//                     start states (Expander::expand_lazy, dbastar.hpp:270-312),
//                     brute force with exact early rejections, one bit mask per
//                     64 primitives, counted (k_app_count with a pair order per
//                     node)
//   k_app_fill        the masks as the (node, primitive) pair list; up to 1024
//                     nodes it scans the counts itself
//   k_check_planar    one lane per pair, then one lane per (state, obstacle) or
//                     visited candidate: translate (transform_primitive),
//                     is_state_valid on every state, swept-box cull of the
//                     node's obstacles in LDS, SAT per state, first offending
//                     index (check_lazy_trajectory, dbastar.cpp:391-490),
//                     check_goal (:492-512), g/h (:833-847), duplicate test
//                     against the visited grid (:850-854), contenders counted
//                     into their grid cells
//   k_grid.hip        contender grid, earlier-conflict lists and the ordered
//                     duplicate / branching-cap resolution (:856-918)
#include <hip/hip_runtime.h>
#include <float.h>
#include <limits.h>

#include <cmath>

#include "dp_internal.h"

namespace {

constexpr int kWaves = 4;  // waves per workgroup of the check kernels

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------------------
// applicability (T_m->nearestR over primitive start states)
// ------------------------------------------------------------------------
// Exact rejections ahead of dp_within for the applicability scan: each test
// shows d(a, b) > r from one metric term (the terms are non-negative and
// IEEE addition is monotone), reading a few components only.
struct app_bounds {
  double T_p, T_v, T_w;  // squared-sum bounds of dp_pos_bound's form for the position,
                         // velocity and rate terms (quadrotor; INFINITY when unused)
  double c_q;            // quadrotor: |q_a . q_b| < c_q implies w1 * angle > r
};

template <int NX>
__device__ __forceinline__ bool app_reject(const dp_dev_sys& S, const app_bounds& B, const double* a,
                                           const double* start, int32_t P, int32_t j, double r) {
  if constexpr (NX == 13) {
    double dot = a[3] * start[(int64_t)3 * P + j];
    dot = dot + a[4] * start[(int64_t)4 * P + j];
    dot = dot + a[5] * start[(int64_t)5 * P + j];
    dot = dot + a[6] * start[(int64_t)6 * P + j];
    if (fabs(dot) < B.c_q) return true;
    double s = 0.0;
#pragma unroll
    for (int c = 10; c < 13; ++c) {
      const double d = a[c] - start[(int64_t)c * P + j];
      s = c == 10 ? d * d : s + d * d;
    }
    return s > B.T_w;
  } else {
    // the heading term (unicycles, car): w1 * so2 alone
    return S.w[1] * dp_so2(a[2], start[(int64_t)2 * P + j]) > r;
  }
}

// kAppParts waves per node, each over a share of the primitives, 64 per
// step: the applicable ones are recorded as a bit mask per 64 primitives
// (mask[i * words + j / 64]) and counted into app[i] (cleared before); the
// fill pass turns the masks into the (node, primitive) pair list without
// evaluating the metric again.
constexpr int kAppParts = 4;

// With a pair order (order != nullptr, [rows][P]) bit r of node i's mask is
// primitive order[(i % rows) * P + r]: the pairs come out in that order.
template <int NX>
__global__ __launch_bounds__(64) void k_app_count(const dp_dev_sys* __restrict__ Sp, app_bounds B,
                                                  const double* __restrict__ nodes, int32_t Ncap, int32_t N,
                                                  const double* __restrict__ start, int32_t P, double r_app,
                                                  const int32_t* __restrict__ order, int32_t rows,
                                                  int32_t* __restrict__ app, uint64_t* __restrict__ mask) {
  const dp_dev_sys& S = *Sp;
  const int32_t i = blockIdx.x / kAppParts, part = blockIdx.x % kAppParts;
  if (i >= N) return;
  const int lane = threadIdx.x;
  const int32_t words = (P + 63) / 64;
  const int32_t w0 = (int32_t)((int64_t)words * part / kAppParts), w1 = (int32_t)((int64_t)words * (part + 1) / kAppParts);
  const int32_t* row = order ? order + (int64_t)(i % rows) * P : nullptr;
  double a[NX];
#pragma unroll
  for (int c = 0; c < NX; ++c) a[c] = dp_is_offset_dim(S, c) ? 0.0 : nodes[(int64_t)c * Ncap + i];
  int32_t cnt = 0;
  for (int32_t j0 = 64 * w0; j0 < P && j0 < 64 * w1; j0 += 64) {
    const int32_t r = j0 + lane;
    const int32_t j = row && r < P ? row[r] : r;
    bool hit = false;
    if (r < P && !app_reject<NX>(S, B, a, start, P, j, r_app)) {
      double b[NX];
#pragma unroll
      for (int c = 0; c < NX; ++c) b[c] = start[(int64_t)c * P + j];
      hit = dp_within(S, a, b, r_app);
    }
    const uint64_t m = __ballot(hit);
    if (lane == 0) mask[(int64_t)i * words + j0 / 64] = m;
    cnt += __popcll(m);
  }
  if (lane == 0 && cnt) atomicAdd(&app[i], cnt);
}

// The same query for kAppNodes nodes per wave (a shared pair order or
// none): each lane loads its primitive's key once per 64-primitive chunk and
// tests it against every node of the group, so the keys stream from L2 once
// per group instead of once per node.  The exact early rejections run for
// all (node, primitive) combinations; the combinations they leave go to a
// wave-local queue and the full metric runs on them 64 at a time, packed,
// instead of on every chunk that has at least one such lane.  Bit r of node
// i's mask word w is set exactly when k_app_count would set it.
constexpr int kAppNodes = 16;

// Exact rejections of the blocked query, evaluated in FP32 on FP32 copies of
// the keys and node states, with margins that cover FP32 rounding (about
// 1e-6 relative on the quantities compared, against 1e-4 of margin): a pair
// rejected here is rejected by the FP64 metric too.  Quadrotor: the attitude
// term is w1 * acos(|q_a . q_b|), and for unit quaternions acos(|q_a . q_b|)
// >= |q_a - sign(q_a . q_b) q_b| (the chord 2 sin(theta / 2) <= theta); every
// other term is non-negative, so w1 * chord + w3 * |w_a - w_b| above the
// radius proves d > r.  That leaves about 0.3% more pairs than are
// applicable for the FP64 metric, against about 3x with the attitude bound
// alone.  Planar systems: the heading term alone.
struct app_bounds32 {
  float c_q;      // quadrotor: |dot| below it rejects
  float T_w;      // quadrotor: squared rate difference above it rejects
  float w1, w3;   // metric weights of the attitude / heading and rate terms
  float R;        // quadrotor: chord bound above it rejects; planar: heading term above it rejects
};

// Stage 1, for every (node, primitive) of a chunk: quadrotor |dot| >= c_q;
// planar systems: the heading term.
template <int NX>
__device__ __forceinline__ bool app_pass1(const app_bounds32& B, const float* a, const float* k) {
  if constexpr (NX == 13) {
    float dot = a[3] * k[3];
    dot = dot + a[4] * k[4];
    dot = dot + a[5] * k[5];
    dot = dot + a[6] * k[6];
    return !(fabsf(dot) < B.c_q);
  } else {
    float d = fabsf(a[2] - k[2]);
    d = d > 3.14159265f ? 6.28318531f - d : d;
    return !(B.w1 * d > B.R);
  }
}

// Stage 2, quadrotor only, on the stage-1 survivors (packed): the chord and
// rate bound.
__device__ __forceinline__ bool app_pass2_quad(const app_bounds32& B, const float* a, const float* k) {
  float dot = a[3] * k[3];
  dot = dot + a[4] * k[4];
  dot = dot + a[5] * k[5];
  dot = dot + a[6] * k[6];
  const float sg = dot < 0.0f ? -1.0f : 1.0f;
  // sums of squared differences with their FP32 error bounds: each term
  // (a - k)^2 is off by at most 8e-7 (a^2 + k^2) (inputs rounded to FP32,
  // one subtraction, one product, the sum); 2e-6 (a^2 + k^2) is taken off
  float c2 = 0.0f, s = 0.0f, ec = 0.0f, es = 0.0f;
#pragma unroll
  for (int c = 3; c < 7; ++c) {
    const float d = a[c] - sg * k[c];
    c2 = c2 + d * d;
    ec = ec + (a[c] * a[c] + k[c] * k[c]);
  }
#pragma unroll
  for (int c = 10; c < 13; ++c) {
    const float d = a[c] - k[c];
    s = s + d * d;
    es = es + (a[c] * a[c] + k[c] * k[c]);
  }
  const float c2_lo = fmaxf(c2 - 2e-6f * ec, 0.0f), s_lo = fmaxf(s - 2e-6f * es, 0.0f);
  if (s_lo > B.T_w) return false;
  return !(B.w1 * sqrtf(c2_lo) + B.w3 * sqrtf(s_lo) > B.R);
}

template <int NX>
__global__ __launch_bounds__(64) void k_app_blk(const dp_dev_sys* __restrict__ Sp, app_bounds32 B,
                                                const double* __restrict__ nodes, int32_t Ncap, int32_t N,
                                                const double* __restrict__ keys, const float* __restrict__ keys32,
                                                int32_t P, double r_app, const int32_t* __restrict__ row,
                                                int32_t parts, int32_t* __restrict__ app,
                                                uint64_t* __restrict__ mask) {
  __shared__ double s_a[kAppNodes * NX];
  __shared__ float s_a32[kAppNodes * NX];
  __shared__ float s_k[NX * 64];
  __shared__ uint16_t s_q[kAppNodes * 64];
  __shared__ uint16_t s_q2[kAppNodes * 64];
  __shared__ unsigned long long s_m[kAppNodes];
  const dp_dev_sys& S = *Sp;
  const int32_t grp = blockIdx.x / parts, part = blockIdx.x % parts;
  const int32_t i0 = grp * kAppNodes;
  if (i0 >= N) return;
  const int32_t nb = N - i0 < kAppNodes ? N - i0 : kAppNodes;
  const int lane = threadIdx.x;
  const uint64_t lt = (1ull << lane) - 1ull;
  const int32_t words = (P + 63) / 64;
  const int32_t w0 = (int32_t)((int64_t)words * part / parts), w1 = (int32_t)((int64_t)words * (part + 1) / parts);
  for (int t = lane; t < kAppNodes * NX; t += 64) {
    const int b = t / NX, c = t % NX;
    s_a[t] = b < nb && !dp_is_offset_dim(S, c) ? nodes[(int64_t)c * Ncap + i0 + b] : 0.0;
    s_a32[t] = (float)s_a[t];
  }
  if (lane < kAppNodes) s_m[lane] = 0ull;
  wave_lds_sync();
  int32_t cnt = 0;  // lane b < nb: node i0 + b
  for (int32_t w = w0; w < w1; ++w) {
    const int32_t r = w * 64 + lane;
    // every lane loads (past P, the last primitive's key, then unused): a
    // load under a condition would be waited for on its own, component
    // after component
    const int32_t rc = r < P ? r : P - 1;
    const int32_t j = row ? row[rc] : rc;
    float k[NX];
#pragma unroll
    for (int c = 0; c < NX; ++c) k[c] = keys32[(int64_t)c * P + j];
#pragma unroll
    for (int c = 0; c < NX; ++c) {
      k[c] = r < P ? k[c] : 0.0f;
      s_k[c * 64 + lane] = k[c];
    }
    // stage 1 for every node of the group; survivors queued
    int qn = 0;
    for (int b = 0; b < nb; ++b) {
      const bool pass = r < P && app_pass1<NX>(B, s_a32 + b * NX, k);
      const uint64_t m = __ballot(pass);
      if (pass) s_q[qn + __popcll(m & lt)] = (uint16_t)((b << 6) | lane);
      qn += __popcll(m);
    }
    wave_lds_sync();
    const uint16_t* q = s_q;
    if constexpr (NX == 13) {
      // stage 2 on the packed survivors
      int qn2 = 0;
      for (int e0 = 0; e0 < qn; e0 += 64) {
        const int e = e0 + lane;
        bool pass = false;
        int ent = 0;
        if (e < qn) {
          ent = s_q[e];
          const int b = ent >> 6, lj = ent & 63;
          float kk[NX];
#pragma unroll
          for (int c = 0; c < NX; ++c) kk[c] = s_k[c * 64 + lj];
          pass = app_pass2_quad(B, s_a32 + b * NX, kk);
        }
        const uint64_t m = __ballot(pass);
        if (pass) s_q2[qn2 + __popcll(m & lt)] = (uint16_t)ent;
        qn2 += __popcll(m);
      }
      wave_lds_sync();
      q = s_q2;
      qn = qn2;
    }
    // the full metric on the survivors, 64 at a time
    for (int e0 = 0; e0 < qn; e0 += 64) {
      const int e = e0 + lane;
      if (e < qn) {
        const int ent = q[e];
        const int b = ent >> 6, lj = ent & 63;
        const int32_t jj = row ? row[w * 64 + lj] : w * 64 + lj;
        double kk[NX];
#pragma unroll
        for (int c = 0; c < NX; ++c) kk[c] = keys[(int64_t)c * P + jj];
        if (dp_within(S, s_a + b * NX, kk, r_app)) atomicOr(&s_m[b], 1ull << lj);
      }
    }
    wave_lds_sync();
    if (lane < nb) {
      const unsigned long long m = s_m[lane];
      mask[(int64_t)(i0 + lane) * words + w] = m;
      cnt += __popcll(m);
      s_m[lane] = 0ull;
    }
    wave_lds_sync();
  }
  if (lane < nb && cnt) atomicAdd(&app[i0 + lane], cnt);
}


// The masks as the (node, primitive) pair list, one wave per node, 64 mask
// words at a time: each lane expands its own word's set bits into LDS at the
// word's offset (an exclusive scan of the counts across the lanes), then the
// wave copies the batch out with full-width stores.
//
// Up to kFillScan nodes the wave sums the counts of the nodes before its own
// itself (at most 16 loads per lane) and writes the node's offset: no scan
// launch.  The quadrotor's FP32 pass also gets the node's pairs reordered
// from here (qperm: (pair, primitive)), those whose primitive leaves the
// attitude / rate bounds first (BOUNDS whatever the translation: short
// rollouts, no collision tests), each group in canonical order: with one bit
// per primitive the two groups' places are bit counts of the masks, where a
// kernel that looked every pair's primitive up took 16 us (1.13M pairs).
constexpr int32_t kFillScan = 1024;

struct fill_args {
  int32_t N, P;
  const int32_t* cnt;      // pairs per node
  int32_t* app;            // offsets: read, or written when scan is set
  int32_t scan;
  const uint64_t* mask;
  const int32_t* order;
  int32_t rows;
  int32_t* pnode;
  int32_t* pprim;
  int64_t pair_cap;
  int32_t* total;
  long long* counters;
  const uint64_t* qshort;  // quadrotor FP32 pass (else null): bit j: the primitive's rates leave the bounds
  int2* qperm;
  int32_t* nshort;
  int32_t* chunks;         // 64-pair chunks of the two groups
};

template <bool kRow>
__global__ __launch_bounds__(64) void k_app_fill(fill_args a) {
  __shared__ int32_t s_p[64 * 64];
  const int32_t i = blockIdx.x;
  if (i >= a.N) return;
  const int lane = threadIdx.x;
  const int32_t words = (a.P + 63) / 64;
  const int32_t* row = kRow ? a.order + (int64_t)(i % a.rows) * a.P : nullptr;
  int64_t q0;
  if (a.scan) {
    long long sum = 0;
    for (int32_t k = lane; k < i; k += 64) sum += a.cnt[k];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d, 64);
    q0 = sum;
    if (lane == 0) {
      a.app[i] = (int32_t)sum;
      if (i == a.N - 1) {
        const long long tot = sum + a.cnt[i];
        a.app[a.N] = (int32_t)tot;
        *a.total = (int32_t)(tot < a.pair_cap ? tot : a.pair_cap);
        a.counters[DPC_PAIRS] = tot;
        if (tot > a.pair_cap) a.counters[DPC_OVERFLOW] = 1;
      }
    }
  } else {
    q0 = a.app[i];
  }
  // first places of the short and the long group
  int64_t ws = q0, wl = q0;
  if (a.qshort) {
    int32_t ns = 0;
    for (int32_t w = lane; w < words; w += 64) ns += __popcll(a.mask[(int64_t)i * words + w] & a.qshort[w]);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) ns += __shfl_xor(ns, d, 64);
    wl = q0 + ns;
    if (lane == 0) {
      // pairs past the capacity are dropped at the end of the list
      const int64_t end = q0 + a.cnt[i] < a.pair_cap ? q0 + a.cnt[i] : a.pair_cap;
      const int32_t n = end > q0 ? (int32_t)(end - q0) : 0;
      a.nshort[i] = n < a.cnt[i] ? 0 : ns;
      a.chunks[i] = n < a.cnt[i] ? 0 : (ns + 63) / 64 + (n - ns + 63) / 64;
    }
  }
  for (int32_t wb = 0; wb < words; wb += 64) {
    const int32_t wl_ = wb + lane;
    uint64_t m = wl_ < words ? a.mask[(int64_t)i * words + wl_] : 0ull;
    const uint64_t sh = a.qshort && wl_ < words ? a.qshort[wl_] : 0ull;
    int32_t incl = __popcll(m), sinc = __popcll(m & sh);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t v = __shfl_up(incl, o), u = __shfl_up(sinc, o);
      if (lane >= o) {
        incl += v;
        sinc += u;
      }
    }
    int32_t pos = incl - __popcll(m);
    int32_t sp = sinc - __popcll(m & sh), lp = pos - sp;
    const uint64_t m0 = m;
    while (m) {
      s_p[pos++] = wl_ * 64 + (__ffsll((long long)m) - 1);
      m &= m - 1ull;
    }
    wave_lds_sync();
    const int32_t total = __builtin_amdgcn_readlane(incl, 63);
    for (int32_t k = lane; k < total; k += 64) {
      const int64_t q = q0 + k;
      if (q < a.pair_cap) {
        const int32_t r = s_p[k];
        a.pnode[q] = i;
        if constexpr (kRow) a.pprim[q] = row[r];
        else a.pprim[q] = r;
      }
    }
    if (a.qshort) {
      // the same bits again into the two groups
      const int64_t first = q0 + incl - __popcll(m0);
      int32_t k = 0;
      for (m = m0; m; m &= m - 1ull, ++k) {
        const int bit = __ffsll((long long)m) - 1;
        const bool is_short = (sh >> bit) & 1ull;
        const int64_t at = is_short ? ws + sp++ : wl + lp++;
        if (at < a.pair_cap) a.qperm[at] = make_int2((int32_t)(first + k), wl_ * 64 + bit);
      }
      const int32_t st = __builtin_amdgcn_readlane(sinc, 63);
      ws += st;
      wl += total - st;
    }
    q0 += total;
    wave_lds_sync();
  }
}

}  // namespace

// Arguments of the check kernels (passed by value in the kernarg segment).
struct dp_check_args {
  const dp_dev_sys* sys;
  const double* nodes;
  int32_t Ncap;
  const double* gpar;
  const int32_t* off;
  const double* st;
  int32_t S;
  const double4* st4;    // [boxes][S] per state: (x, y, cos, sin) of the body, then the trailer's (offset x, y, cos, sin)
  const double* prec;    // [P][DP_PREC] what a pair reads of its primitive
  double reach[4];       // union of the swept boxes relative to a node (lo x, hi x, lo y, hi y)
  int32_t ppw;           // pairs per wave, 2 to 64 (0: from the pair count)
  int32_t P;
  const int32_t* goalidx;
  int32_t num_goal, check_goal;
  const double* obs;
  int32_t nobs;
  const double* vis;
  int64_t vstride;
  int64_t nv, nv_sorted;
  const int32_t* vstart;
  dp_grid_geom grid;
  const int32_t* pnode;
  const int32_t* pprim;
  const int32_t* total;
  int8_t* verdict;
  int32_t* firstk;
  int32_t* goal_out;
  int8_t* res;
  int8_t* flags;
  double* fin;
  int64_t pcap;
  double* gout;
  double* hout;
  double goal[DP_MAX_NX];
  double goal_bound, r_dup, cdf;
  int32_t surrogate;  // pairs already marked DP_V_SURROGATE_REJECT are skipped
  long long* counters;
  // tdbastar's reverse search: placement offset = node - last position of
  // the primitive, new state = first placed state
  int32_t backward;
  // tdbastar constraints: times [ncon], then states [ncon][nx]
  int32_t ncon;
  const double* con;
  double con_delta;
  // dbrrt selection: no goal check or duplicate test, resolution DP_R_NONE
  int32_t select;
  // contender grid: cell counts, and each contender's cell and place in it
  // (count null: not counted here)
  int32_t* cont_count;
  int32_t* cont_cell;
  int32_t* cont_place;
  dp_marks marks;
};

namespace {

template <int NX>
__device__ __forceinline__ void load_translated(const dp_check_args& a, int64_t sidx, double ox, double oy, double* s) {
  s[0] = a.st[sidx] + ox;
  s[1] = a.st[(int64_t)a.S + sidx] + oy;
#pragma unroll
  for (int c = 2; c < NX; ++c) s[c] = a.st[(int64_t)c * a.S + sidx];
}

// Flattened items of a wave: segments of 0 or more items, numbered one after
// another and dealt to the 64 lanes in turn.  A bitmap of the segments' first
// items gives an item's segment by a bit count, kItemWindow items at a time.
constexpr int kItemWindow = 4096;
constexpr int kPairItems = 1 << 20;  // visited candidates of a pair past which it is a list of its own

// Per-wave LDS of k_check_planar: 9.5 KB for three components, 10.5 KB for
// five.  A workgroup takes four of them, 0.9 KB of constants and 40 bytes per
// obstacle, so three workgroups fit a CU (as many as the registers allow) up
// to some 370 obstacles, with five components up to 270, and two up to 950.
template <int NX>
struct check_wave {
  uint64_t head[kItemWindow / 64];
  // bounds and collision: per segment (a pair with states to test)
  int32_t pre[64];           // its first item
  int32_t st0[64];           // first state of the pair's primitive (complemented: bounds to be tested too)
  int32_t bad[64], col[64];  // first offending / colliding state so far (constraints: bad = first violated one)
  uint64_t mask[64];         // obstacles of the staged chunk that meet the pair's swept box
  double ox[64], oy[64];     // placement offset
  union {
    struct {
      int32_t len[64], reach[64];
      float g[64];
    } con;                   // constraints: per pair to test
    struct {
      double x[NX][64];      // state of the new node, per lane
      int2 run[10 * 64];      // per non-empty run: the pair's lane, sorted position minus first item
    } vis;
  };
};
static_assert(sizeof(check_wave<3>) == 9728 && sizeof(check_wave<4>) == 10240 && sizeof(check_wave<5>) == 10752,
              "the figures above");

__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(v, d, 64);
    if (lane >= d) v += u;
  }
  return v;
}

// Calls set(window start) for each window of items (it marks the first items
// of the segments in head[], relative to the window), then item(segment, f)
// for every item f < T of it.
template <typename Set, typename Item>
__device__ __forceinline__ void for_items(uint64_t* head, int T, int lane, Set&& set, Item&& item) {
  const uint64_t le = (2ull << lane) - 1ull;
  int base = -1;
  for (int w0 = 0; w0 < T; w0 += kItemWindow) {
    head[lane] = 0ull;
    wave_lds_sync();
    set(w0);
    wave_lds_sync();
    for (int r = 0; r < 64 && w0 + 64 * r < T; ++r) {
      const uint64_t h = head[r];
      const int f = w0 + 64 * r + lane;
      if (f < T) item(base + (int)__popcll(h & le), f);
      base += __builtin_amdgcn_readfirstlane((int)__popcll(h));
    }
    wave_lds_sync();
  }
}

__device__ __forceinline__ void mark_item(uint64_t* head, int f, int w0) {
  const int r = f - w0;
  if (r >= 0 && r < kItemWindow) atomicOr((unsigned long long*)&head[r >> 6], 1ull << (r & 63));
}

// Planar translate systems (unicycle1/2, car+trailer), FP64.  A wave takes
// a.ppw consecutive pairs, one per lane, and spreads what varies in length
// between pairs (states against obstacles, constraints, visited candidates)
// over all 64 lanes as one flattened list, so that a pair's length costs its
// share and the loads of 64 items are in flight together.
//
// It is bound by the latency of its chains of dependent loads (pair ->
// primitive record -> states; final state -> cell starts -> candidates) at
// three waves per SIMD.  A split of LPP lanes per pair, each lane one state,
// did the once-per-pair work LPP times and ran every group to its longest
// primitive.  Measured, 1.95M pairs of 5-30 states, 200 boxes, 100k visited:
// 32 lanes per pair (the old rule for that length) 2.03 ms, the best split
// (4) 0.69 ms, this form 0.32 ms, of which states against boxes 0.10, the
// visited set 0.10, setting up and writing the pairs the rest.  0.50M car
// pairs, 300 boxes: 1.07 -> 0.18 ms.
//
// Pairs per wave without a setting: about 2304 waves (9 per CU) over the
// batch, read on the device.  Fewer pairs per wave leave fewer states to
// one wave but idle lanes in the once-per-pair part: 24k pairs 64 / 16 / 4
// per wave 50 / 33 / 58 us, 143k pairs 56 / 79 / 153 us.
template <int NX>
__global__ __launch_bounds__(256) void k_check_planar(dp_check_args a) {
  extern __shared__ double smem[];
  // the system constants in LDS: read from global memory after the loop's
  // stores, each would be a load the wave waits for
  __shared__ dp_dev_sys s_sys;
  __shared__ check_wave<NX> s_wave[kWaves];
  const dp_dev_sys& S = s_sys;
  const int nobs = a.nobs;
  dp_mark(a.marks);
  // a.ppw 0: about 9 waves per CU over the batch's pairs, 4 to 64 pairs each
  int ppw = a.ppw;
  if (ppw == 0) {
    const int want = *a.total / 2304;
    ppw = want <= 4 ? 4 : want <= 8 ? 8 : want <= 16 ? 16 : want <= 32 ? 32 : 64;
  }
  if ((int64_t)blockIdx.x * kWaves * ppw >= (int64_t)*a.total) return;  // uniform per block
  double* s_obs = smem;  // [nobs][4]
  for (int t = threadIdx.x; t < 4 * nobs; t += blockDim.x) s_obs[t] = a.obs[t];
  static_assert(sizeof(dp_dev_sys) % sizeof(double) == 0, "copied as doubles");
  for (int t = threadIdx.x; t < (int)(sizeof(dp_dev_sys) / sizeof(double)); t += blockDim.x)
    reinterpret_cast<double*>(&s_sys)[t] = reinterpret_cast<const double*>(a.sys)[t];
  // the workgroup's counts, added to the batch counters once per workgroup
  __shared__ unsigned long long s_cnt[5];
  if (threadIdx.x < 5) s_cnt[threadIdx.x] = 0ull;
  __syncthreads();

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  check_wave<NX>& W = s_wave[wave];
  int16_t* list = (int16_t*)(smem + 4 * nobs) + (int64_t)wave * nobs;  // obstacles near the node being checked
  const uint64_t lt = (1ull << lane) - 1ull;
  const int32_t total = *a.total;
  const double Tdup = dp_pos_bound(S, a.r_dup), Tgoal = dp_pos_bound(S, a.goal_bound);
  int c_b = 0, c_c = 0, c_f = 0, c_k = 0, c_x = 0;

  for (int64_t q0 = ((int64_t)blockIdx.x * kWaves + wave) * ppw; q0 < total; q0 += (int64_t)gridDim.x * kWaves * ppw) {
    const int64_t q = q0 + lane;
    const bool vp = lane < ppw && q < total && !(a.surrogate && a.verdict[q] == DP_V_SURROGATE_REJECT);
    int32_t i = 0, j = 0, st0 = 0, L1 = 0;
    double ox = 0.0, oy = 0.0;
    const double* rec = a.prec;
    // ---- is_state_valid on every translated state -----------------------
    // First from the primitive's component ranges: with the translation
    // rounded the same way, (min + offset) >= lo and (max + offset) <= hi
    // bound every translated state (rounding is monotone); other components
    // compare their range directly.  Only pairs not cleared this way scan
    // their states for the first offending index.
    bool clear = true;
    double bx0 = 0, bx1 = 0, by0 = 0, by1 = 0;
    double tx0 = 0, tx1 = 0, ty0 = 0, ty1 = 0;  // range of the placed positions
    if (vp) {
      i = a.pnode[q];
      j = a.pprim[q];
      rec = a.prec + (int64_t)j * DP_PREC;
      const int2 sl = *reinterpret_cast<const int2*>(rec + DP_PREC_S0);
      st0 = sl.x;
      L1 = sl.y;
      ox = a.nodes[i];
      oy = a.nodes[(int64_t)a.Ncap + i];
      if (a.backward) {  // offset - motion->traj.states.back().head(2), tdbastar.hpp:193-196
        ox = ox - rec[DP_PREC_LAST];
        oy = oy - rec[DP_PREC_LAST + 1];
      }
      bx0 = (rec[0] + ox) - DP_SWEEP_PAD;
      bx1 = (rec[1] + ox) + DP_SWEEP_PAD;
      by0 = (rec[2] + oy) - DP_SWEEP_PAD;
      by1 = (rec[3] + oy) + DP_SWEEP_PAD;
#pragma unroll
      for (int c = 0; c < NX; ++c) {
        const double o = c == 0 ? ox : (c == 1 ? oy : 0.0);
        const double mn = rec[DP_PREC_RANGE + 2 * c], mx = rec[DP_PREC_RANGE + 2 * c + 1];
        const double tmn = c < 2 ? mn + o : mn, tmx = c < 2 ? mx + o : mx;
        clear = clear & (tmn >= S.lo[c]) & (tmx <= S.hi[c]);
        if (c == 0) tx0 = tmn, tx1 = tmx;
        if (c == 1) ty0 = tmn, ty1 = tmx;
      }
    }
    int first_bad = INT_MAX, first_col = INT_MAX;

    // ---- bounds and collision, node by node of the wave's pairs ----------
    for (uint64_t todo = __ballot(vp); todo;) {
      const int src = __ffsll((long long)todo) - 1;
      const int32_t node = __builtin_amdgcn_readlane(i, src);
      const bool mine = vp && i == node;
      todo &= ~__ballot(mine);
      // Obstacles that can touch any of the node's primitives: every swept
      // box lies inside the union box `reach` and both tests round the same
      // way, so the list holds every obstacle that a pair's own box meets.
      int nlist = 0;
      {
        const double nox = a.nodes[node], noy = a.nodes[(int64_t)a.Ncap + node];
        const double rx0 = (a.reach[0] + nox) - DP_SWEEP_PAD, rx1 = (a.reach[1] + nox) + DP_SWEEP_PAD;
        const double ry0 = (a.reach[2] + noy) - DP_SWEEP_PAD, ry1 = (a.reach[3] + noy) + DP_SWEEP_PAD;
        for (int ob = 0; ob < nobs; ob += 64) {
          const int o = ob + lane;
          bool hit = false;
          if (o < nobs) {
            const double* b = s_obs + 4 * o;
            hit = !(b[0] + b[2] < rx0 || b[0] - b[2] > rx1 || b[1] + b[3] < ry0 || b[1] - b[3] > ry1);
          }
          const uint64_t m = __ballot(hit);
          if (hit) list[nlist + __popcll(m & lt)] = (int16_t)o;
          nlist += __popcll(m);
        }
      }
      wave_lds_sync();
      // 64 obstacles of the list at a time, one bit each
      for (int c0 = 0; c0 == 0 || c0 < nlist; c0 += 64) {
        const int nc = nlist - c0 < 64 ? nlist - c0 : 64;
        uint64_t mask = 0ull;
        for (int t = 0; t < nc; ++t) {
          const double* b = s_obs + 4 * list[c0 + t];
          const bool hit = !(b[0] + b[2] < bx0 || b[0] - b[2] > bx1 || b[1] + b[3] < by0 || b[1] - b[3] > by1);
          mask |= hit ? 1ull << t : 0ull;
        }
        const bool scan = mine && (mask != 0ull || (c0 == 0 && !clear));
        const int n = scan ? L1 : 0;
        const int incl = wave_incl_scan(n, lane);
        const int T = __builtin_amdgcn_readlane(incl, 63);
        const int seg = __popcll(__ballot(scan) & lt);
        if (scan) {
          W.pre[seg] = incl - n;
          W.mask[seg] = mask;
          W.st0[seg] = clear ? st0 : ~st0;
          W.ox[seg] = ox;
          W.oy[seg] = oy;
          W.bad[seg] = INT_MAX;
          W.col[seg] = INT_MAX;
        }
        for_items(
            W.head, T, lane,
            [&](int w0) {
              if (scan) mark_item(W.head, incl - n, w0);
            },
            [&](int p, int f) {
              const int k = f - W.pre[p];
              const int32_t s0 = W.st0[p];
              const int64_t sidx = (int64_t)(s0 < 0 ? ~s0 : s0) + k;
              const double4 s4 = a.st4[sidx];
              const double x = s4.x + W.ox[p], y = s4.y + W.oy[p];
              if (s0 < 0 && c0 == 0) {
                bool bad = !((x >= S.lo[0]) & (x <= S.hi[0])) | !((y >= S.lo[1]) & (y <= S.hi[1]));
#pragma unroll
                for (int c = 2; c < NX; ++c) {
                  const double v = a.st[(int64_t)c * a.S + sidx];
                  bad = bad | !((v >= S.lo[c]) & (v <= S.hi[c]));
                }
                if (bad) atomicMin(&W.bad[p], k);
              }
              bool col = false;
              const uint64_t m0 = W.mask[p];
              for (uint64_t m = m0; m && !col; m &= m - 1ull) {
                const double* b = s_obs + 4 * list[c0 + __ffsll((long long)m) - 1];
                col = dp_obb_aabb(x, y, s4.z, s4.w, S.body_hl, S.body_hw, b[0], b[1], b[2], b[3]);
              }
              if constexpr (NX == 4) {  // the trailer's box, at its offset from the state position
                if (m0 && !col) {
                  const double4 t4 = a.st4[(int64_t)a.S + sidx];
                  const double cx = x + t4.x, cy = y + t4.y;
                  for (uint64_t m = m0; m && !col; m &= m - 1ull) {
                    const double* b = s_obs + 4 * list[c0 + __ffsll((long long)m) - 1];
                    col = dp_obb_aabb(cx, cy, t4.z, t4.w, S.trailer_hl, S.trailer_hw, b[0], b[1], b[2], b[3]);
                  }
                }
              }
              if (col) atomicMin(&W.col[p], k);
            });
        if (scan) {
          first_bad = min(first_bad, W.bad[seg]);
          first_col = min(first_col, W.col[seg]);
        }
        wave_lds_sync();
      }
    }
    int8_t vd = first_bad != INT_MAX ? DP_V_BOUNDS : (first_col != INT_MAX ? DP_V_COLLIDE : DP_V_FREE);

    // ---- tdbastar constraints on a valid pair (tdbastar.cpp:408-443) -----
    // (pair, constraint) items; the first violated constraint in list order
    // wins.
    if (a.ncon > 0) {
      const bool nc = vp && vd == DP_V_FREE;
      bool reaches = false;
      float gf = 0.0f;
      if (nc) {
        double s[NX];
        load_translated<NX>(a, (int64_t)st0 + (a.backward ? L1 - 1 : 0), ox, oy, s);
        reaches = dp_distance(S, s, a.goal) <= a.con_delta;
        gf = (float)a.gpar[i];  // best_node_gScore is passed as float
      }
      // state that constraint ci selects for a pair, or -1
      auto con_state = [&](int ci, float g_f, bool reach, int len) {
        const float toff = (float)(a.con[ci] - (double)g_f);
        const int ti = (int)lround((double)toff / S.dt);
        int k = -1;
        if (reach && ti >= len - 1) k = len - 1;
        if (ti >= 0 && ti < len - 1) k = ti;
        return k;
      };
      const uint64_t ncm = __ballot(nc);
      const int np = __popcll(ncm), seg = __popcll(ncm & lt);
      if (nc) {  // the pairs to test, packed
        W.st0[seg] = st0;
        W.ox[seg] = ox;
        W.oy[seg] = oy;
        W.bad[seg] = INT_MAX;  // first violated constraint
        W.con.len[seg] = L1;
        W.con.reach[seg] = reaches ? 1 : 0;
        W.con.g[seg] = gf;
      }
      wave_lds_sync();
      for (int64_t f = lane; f < (int64_t)np * a.ncon; f += 64) {
        const int p = (int)(f / a.ncon), ci = (int)(f % a.ncon);
        if (W.bad[p] < ci) continue;  // an earlier one is violated
        const int k = con_state(ci, W.con.g[p], W.con.reach[p] != 0, W.con.len[p]);
        if (k < 0) continue;
        double s[NX], cs[NX];
        load_translated<NX>(a, (int64_t)W.st0[p] + k, W.ox[p], W.oy[p], s);
#pragma unroll
        for (int c = 0; c < NX; ++c) cs[c] = a.con[a.ncon + (int64_t)ci * NX + c];
        if (dp_distance(S, s, cs) <= a.con_delta) atomicMin(&W.bad[p], ci);
      }
      wave_lds_sync();
      if (nc && W.bad[seg] != INT_MAX) {
        vd = DP_V_CONSTRAINT;
        first_col = con_state(W.bad[seg], gf, reaches, L1);
      }
      wave_lds_sync();
    }

    // ---- FREE: check_goal, g, h, duplicate vs visited --------------------
    const bool fr = vp && vd == DP_V_FREE;
    int chosen = -1;
    if (a.check_goal && !a.select && fr) {
      // The position range of the placed states against the goal: beyond the
      // bound no state can reach it (the differences and their squares round
      // monotonically, dp_pos_bound covers the root), so most pairs load none
      // of the goal states.
      const double dx = fmax(fmax(tx0 - a.goal[0], a.goal[0] - tx1), 0.0);
      const double dy = fmax(fmax(ty0 - a.goal[1], a.goal[1] - ty1), 0.0);
      double s2 = dx * dx;
      s2 = s2 + dy * dy;
      if (!(s2 > Tgoal))
        for (int gk = 0; gk < a.num_goal && chosen == -1; ++gk) {
          const int idx = a.goalidx[(int64_t)gk * a.P + j];
          double s[NX];
          load_translated<NX>(a, (int64_t)st0 + idx, ox, oy, s);
          if (dp_within(S, s, a.goal, a.goal_bound)) chosen = idx;
        }
    }
    double xf[NX];
    double gq = 0.0, hq = 0.0;
    if (fr) {
      // the new node's state: the last placed state, or the first for the
      // reverse search (check_goal, tdbastar.cpp:453-458)
      double nd[NX], t0[NX];
#pragma unroll
      for (int c = 0; c < NX; ++c) {
        const double o = c == 0 ? ox : oy;
        nd[c] = a.nodes[(int64_t)c * a.Ncap + i];
        const double first = rec[DP_PREC_START + c], last = rec[DP_PREC_LAST + c];
        t0[c] = c < 2 ? first + o : first;
        xf[c] = a.backward ? t0[c] : (c < 2 ? last + o : last);
      }
      if (chosen != -1) load_translated<NX>(a, (int64_t)st0 + chosen, ox, oy, xf);
      hq = dp_lower_bound_time(S, xf, a.goal);
      const double cm = chosen != -1 ? chosen * S.dt : (L1 - 1) * S.dt;
      gq = a.gpar[i] + cm + a.cdf * dp_lower_bound_time(S, nd, t0);
    } else {
#pragma unroll
      for (int c = 0; c < NX; ++c) xf[c] = 0.0;
    }
    bool dupv = false;
    if (a.nv > 0 && !a.select && __ballot(fr)) {
      // the 9 runs of each final state's 27-cell block (dp_grid_run_any's
      // rules), their bounds loaded together, and the unsorted tail
      int32_t rb[10], rn[10];
      int K = 0, nr = 0;
#pragma unroll
      for (int k = 0; k < 10; ++k) rb[k] = rn[k] = 0;
      if (fr) {
        const dp_grid_geom& G = a.grid;
        int32_t c[3];
        dp_cell_coords(G, xf, c);
        const int32_t x0 = c[0] > 0 ? c[0] - 1 : 0, x1 = c[0] + 1 < G.dims[0] ? c[0] + 1 : G.dims[0] - 1;
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          const int32_t n1 = c[1] + k % 3 - 1, d2 = k / 3 - 1;
          int32_t n2 = c[2] + d2;
          bool ok = n1 >= 0 && n1 < G.dims[1];
          if (G.dims[2] == 1) {
            ok = ok && d2 == 0;
            n2 = 0;
          } else if (G.periodic2) {
            n2 = n2 < 0 ? n2 + G.dims[2] : (n2 >= G.dims[2] ? n2 - G.dims[2] : n2);
          } else {
            ok = ok && n2 >= 0 && n2 < G.dims[2];
          }
          const int64_t row = ok ? ((int64_t)n2 * G.dims[1] + n1) * G.row : 0;
          rb[k] = a.vstart[ok ? row + x0 : 0];
          rn[k] = a.vstart[ok ? row + x1 + 1 : 0];
        }
        rb[9] = (int32_t)a.nv_sorted;
        rn[9] = (int32_t)a.nv;
#pragma unroll
        for (int k = 0; k < 10; ++k) {
          rn[k] -= rb[k];
          K += rn[k];
          nr += rn[k] > 0 ? 1 : 0;
        }
      }
      W.bad[lane] = 0;
#pragma unroll
      for (int c = 0; c < NX; ++c) W.vis.x[c][lane] = xf[c];
      // The items of 64 pairs are numbered in 31 bits.  A pair of more than
      // kPairItems candidates (a set of that many states within a block) could
      // take the sum past them: then the wave's pairs go one after another.
      const bool alone = __ballot(K > kPairItems) != 0;
      for (uint64_t left = alone ? __ballot(K > 0) : 1ull; left; left &= left - 1ull) {
        const bool in = !alone || lane == __ffsll((long long)left) - 1;
        const int n = in ? K : 0, runs = in ? nr : 0;
        const int incl = wave_incl_scan(n, lane), run0 = wave_incl_scan(runs, lane) - runs;
        const int T = __builtin_amdgcn_readlane(incl, 63);
        if (in) {
          int f = incl - n, at = run0;
#pragma unroll
          for (int k = 0; k < 10; ++k)
            if (rn[k] > 0) {
              W.vis.run[at++] = make_int2(lane, rb[k] - f);
              f += rn[k];
            }
        }
        for_items(
            W.head, T, lane,
            [&](int w0) {
              if (!in) return;
              int f = incl - n;
#pragma unroll
              for (int k = 0; k < 10; ++k)
                if (rn[k] > 0) {
                  mark_item(W.head, f, w0);
                  f += rn[k];
                }
            },
            [&](int run, int f) {
              const int2 r = W.vis.run[run];
              double x[NX];
#pragma unroll
              for (int c = 0; c < NX; ++c) x[c] = W.vis.x[c][r.x];
              if (dp_within_col_pf<NX>(S, x, a.vis, a.vstride, (int64_t)f + r.y, a.r_dup, Tdup)) W.bad[r.x] = 1;
            });
      }
      dupv = fr && W.bad[lane] != 0;
      wave_lds_sync();
    }
    if (vp) {
      a.verdict[q] = vd;
      a.firstk[q] = vd == DP_V_BOUNDS ? first_bad : (vd == DP_V_COLLIDE || vd == DP_V_CONSTRAINT ? first_col : -1);
      a.goal_out[q] = chosen;
      a.res[q] = fr && !a.select ? DP_R_UNDECIDED : DP_R_NONE;
      a.flags[q] = (int8_t)((dupv ? 1 : 0) | (chosen != -1 ? 2 : 0));
      if (fr) {
#pragma unroll
        for (int c = 0; c < NX; ++c) a.fin[(int64_t)c * a.pcap + q] = xf[c];
        a.gout[q] = gq;
        a.hout[q] = hq;
        if (a.cont_count && (chosen != -1 || !dupv))
          dp_count_contender(a.grid, xf, q, a.cont_count, a.cont_cell, a.cont_place);
      }
    }
    c_b += __popcll(__ballot(vp && vd == DP_V_BOUNDS));
    c_c += __popcll(__ballot(vp && vd == DP_V_COLLIDE));
    c_x += __popcll(__ballot(vp && vd == DP_V_CONSTRAINT));
    c_f += __popcll(__ballot(fr));
    c_k += __popcll(__ballot(vp && vd != DP_V_BOUNDS));
  }
  if (lane == 0) {
    if (c_x) atomicAdd(&s_cnt[0], (unsigned long long)c_x);
    if (c_b) atomicAdd(&s_cnt[1], (unsigned long long)c_b);
    if (c_c) atomicAdd(&s_cnt[2], (unsigned long long)c_c);
    if (c_f) atomicAdd(&s_cnt[3], (unsigned long long)c_f);
    if (c_k) atomicAdd(&s_cnt[4], (unsigned long long)c_k);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int slot[5] = {DPC_CONSTRAINT, DPC_BOUNDS, DPC_COLLIDE, DPC_FREE, DPC_CHECKED};
    for (int k = 0; k < 5; ++k)
      if (s_cnt[k]) atomicAdd((unsigned long long*)&a.counters[slot[k]], s_cnt[k]);
  }
}

// dbrrt's choice per node (dbrrt.cpp:627-660): among the node's FREE pairs,
// in pair order, the first with the smallest distance(last placed state,
// target) below DBL_MAX (the reference starts from
// numeric_limits<double>::max() and keeps a candidate only when d < min), or
// the first FREE one with choose_first.  Writes the pair index (-1: none) and
// [last state, first state, distance, g, h].  Bounded by four dependent loads
// per chunk of pairs, so a node's chunks go to four waves at once (one wave per
// node, chunk after chunk: 30 us for 1000 nodes of 175 pairs; this 20).
constexpr int kSelectWaves = 4;
template <int NX>
__global__ __launch_bounds__(64 * kSelectWaves) void k_select(dp_check_args a, const int32_t* __restrict__ app, int32_t N,
                                               const double* __restrict__ targets, const double* __restrict__ cost,
                                               double cost_jump, int32_t choose_first, int32_t* __restrict__ sel_q,
                                               int32_t* __restrict__ sel_prim, double* __restrict__ sel) {
  dp_mark(a.marks);
  const dp_dev_sys& S = *a.sys;
  const int32_t i = blockIdx.x;
  if (i >= N) return;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  __shared__ double wave_d[kSelectWaves];
  __shared__ int32_t wave_q[kSelectWaves];
  const int32_t tot = *a.total;
  const int32_t b = app[i] < tot ? app[i] : tot;
  const int32_t e = app[i + 1] < tot ? app[i + 1] : tot;
  double tg[NX];
#pragma unroll
  for (int c = 0; c < NX; ++c) tg[c] = targets[(int64_t)c * a.Ncap + i];
  const double ox = a.nodes[i], oy = a.nodes[(int64_t)a.Ncap + i];
  double best_d = DBL_MAX;
  int32_t best_q = -1;
  for (int32_t cb = b + 64 * wave; cb < e; cb += 64 * kSelectWaves) {
    const int32_t q = cb + lane;
    double d = DBL_MAX;
    bool ok = false;
    if (q < e && a.verdict[q] == DP_V_FREE) {
      const int32_t j = a.pprim[q];
      double x[NX];
      load_translated<NX>(a, (int64_t)a.off[j + 1] - 1, ox, oy, x);
      d = dp_distance(S, x, tg);
      ok = d < DBL_MAX;  // NaN and +inf never enter
    }
    if (choose_first) {
      const uint64_t m = __ballot(ok);
      if (m) {
        const int src = __ffsll((long long)m) - 1;
        best_d = __shfl(d, src);
        best_q = cb + src;
        break;
      }
      continue;
    }
    // first minimum of the chunk: (d, q) lexicographic over the lanes that qualify
    double md = ok ? d : DBL_MAX;
    int32_t mq = ok ? q : INT_MAX;
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) {
      const double od = __shfl_xor(md, w);
      const int32_t oq = __shfl_xor(mq, w);
      if (od < md || (od == md && oq < mq)) {
        md = od;
        mq = oq;
      }
    }
    if (mq != INT_MAX && md < best_d) {  // strictly below every earlier chunk's minimum
      best_d = md;
      best_q = mq;
    }
  }
  // the waves' choices: the smallest distance, then the lowest pair (with
  // choose_first the lowest pair)
  if (lane == 0) {
    wave_d[wave] = best_d;
    wave_q[wave] = best_q;
  }
  __syncthreads();
  if (wave != 0) return;
  best_q = -1;
#pragma unroll
  for (int w = 0; w < kSelectWaves; ++w) {
    const double d = wave_d[w];
    const int32_t q = wave_q[w];
    if (q < 0) continue;
    const bool better = best_q < 0 || (choose_first ? q < best_q : d < best_d || (d == best_d && q < best_q));
    if (better) {
      best_d = d;
      best_q = q;
    }
  }
  if (lane == 0) {
    sel_q[i] = best_q;
    sel_prim[i] = best_q >= 0 ? a.pprim[best_q] : -1;
  }
  double* o = sel + (int64_t)i * (2 * NX + 3);
  if (best_q < 0) {
    if (lane < 2 * NX + 3) o[lane] = NAN;
    return;
  }
  if (lane == 0) {
    const int32_t j = a.pprim[best_q];
    double x[NX], x0[NX], nd[NX];
    load_translated<NX>(a, (int64_t)a.off[j + 1] - 1, ox, oy, x);
    load_translated<NX>(a, (int64_t)a.off[j], ox, oy, x0);
#pragma unroll
    for (int c = 0; c < NX; ++c) nd[c] = a.nodes[(int64_t)c * a.Ncap + i];
#pragma unroll
    for (int c = 0; c < NX; ++c) {
      o[c] = x[c];
      o[NX + c] = x0[c];
    }
    o[2 * NX] = best_d;
    o[2 * NX + 1] = a.gpar[i] + cost[j] + cost_jump * dp_lower_bound_time(S, nd, x0);  // dbrrt.cpp:645-648
    o[2 * NX + 2] = dp_lower_bound_time(S, x, a.goal);                                  // dbrrt.cpp:641-642
  }
}

}  // namespace

// ==========================================================================
// host-side pipeline
// ==========================================================================

template <typename F>
static int dispatch_nx(int nx, F&& f) {
  switch (nx) {
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 5: return f(std::integral_constant<int, 5>{});
    case 13: return f(std::integral_constant<int, 13>{});
  }
  dp_set_error("unsupported nx");
  return DP_ERR_ARG;
}

// Applicability count only: the exact number of pairs of the uploaded nodes
// lands in counters[DPC_PAIRS] (buffers are sized from it).
// Exact rejection bounds of the applicability scan for radius r.
static app_bounds make_app_bounds(const dp_ctx* c, double r) {
  app_bounds B{INFINITY, INFINITY, INFINITY, -1.0};
  const dp_system_desc& d = c->desc;
  auto sq = [&](double w) {
    if (!(w > 0.0)) return (double)INFINITY;
    const double t = r / w;
    return t * t * (1.0 + 1e-9);
  };
  B.T_p = sq(d.dist_w[0]);
  if (d.system == DP_SYS_QUADROTOR) {
    B.T_v = sq(d.dist_w[2]);
    B.T_w = sq(d.dist_w[3]);
    // w1 * acos(|dot|) > r when |dot| < cos(r / w1); the 1e-9 margin covers
    // libm's cos and the few ulps of the device's acos series
    if (d.dist_w[1] > 0.0 && r / d.dist_w[1] < 1.5) B.c_q = std::cos(r / d.dist_w[1]) - 1e-9;
  }
  return B;
}

// Applicability masks and counts of the uploaded nodes (app is clear).
template <int NX>
static void launch_app(dp_ctx* c, const app_bounds& B, double r_app, hipStream_t s);

// Applicability radius: alpha * delta as the float product of dbastar.cpp:585-586,
// or dbrrt's Expander radius (options_dbrrt.delta) for dp_expand_select.
static double app_radius(const dp_ctx* c, const dp_expand_params* p) {
  return c->select_mode ? c->select_radius : (double)(p->alpha * p->delta);
}

// Margins of the FP32 rejections (app_bounds32): relative 1e-4 on the
// compared quantities, absolute 1e-6 on top.
static app_bounds32 make_app_bounds32(const dp_ctx* c, double r) {
  const dp_system_desc& d = c->desc;
  app_bounds32 B{-1.0f, INFINITY, (float)d.dist_w[1], (float)d.dist_w[3], INFINITY};
  if (d.system == DP_SYS_QUADROTOR) {
    if (d.dist_w[1] > 0.0 && r / d.dist_w[1] < 1.5) B.c_q = (float)(std::cos(r / d.dist_w[1]) - 1e-5);
    if (d.dist_w[3] > 0.0) B.T_w = (float)((r / d.dist_w[3]) * (r / d.dist_w[3]) * (1.0 + 1e-4) + 1e-6);
    B.R = (float)(r * (1.0 + 1e-4) + 1e-6);
  } else {
    B.R = (float)(r * (1.0 + 1e-4) + d.dist_w[1] * 1e-6 + 1e-6);
  }
  return B;
}

// Primitive parts per node of the blocked applicability: about 4096 waves
// over the (node group, part) grid, at most one part per mask word.
static int32_t app_parts(const dp_ctx* c) {
  const int32_t groups = (c->N + kAppNodes - 1) / kAppNodes;
  const int32_t words = (c->P + 63) / 64;
  int32_t parts = (4096 + groups - 1) / groups;
  return parts < 1 ? 1 : (parts > words ? words : parts);
}
static bool app_per_node_order(const dp_ctx* c) { return c->d_order && c->order_rows > 1; }

template <int NX>
static void launch_app(dp_ctx* c, const app_bounds& B, double r_app, hipStream_t s) {
  const int32_t N = c->N;
  const double* keys = c->forward ? c->d_start : c->d_last;
  if (app_per_node_order(c)) {  // a pair order per node: one wave per node part
    k_app_count<NX><<<N * kAppParts, 64, 0, s>>>(c->d_sys, B, c->d_nodes, c->N_cap, N, keys, c->P, r_app, c->d_order,
                                                 c->order_rows, c->d_app_cnt, c->d_app_mask);
    return;
  }
  const int32_t groups = (N + kAppNodes - 1) / kAppNodes;
  const int32_t parts = app_parts(c);
  const float* keys32 = c->forward ? c->d_start32 : c->d_last32;
  k_app_blk<NX><<<groups * parts, 64, 0, s>>>(c->d_sys, make_app_bounds32(c, r_app), c->d_nodes, c->N_cap, N, keys,
                                              keys32, c->P, r_app, c->d_order, parts, c->d_app_cnt, c->d_app_mask);
}

int dp_launch_count(dp_ctx* c, const dp_expand_params* p, hipStream_t s) {
  const double r_app = app_radius(c, p);
  const int32_t N = c->N;
  const app_bounds B = make_app_bounds(c, r_app);
  dp_fill_i32(c->d_app_cnt, N, 0, s);
  return dispatch_nx(c->desc.nx, [&](auto NXc) -> int {
    constexpr int NX = decltype(NXc)::value;
    launch_app<NX>(c, B, r_app, s);
    dp_scan_small(c->d_app_cnt, c->d_app, N, c->d_total, c->pair_cap, c->d_counters, DPC_PAIRS, s);
    DP_HIP_RET(hipGetLastError());
    return DP_OK;
  });
}

// Start and end events are skipped while a multi-instance graph is captured.
#define DP_EV(ev_, s_) \
  do { \
    if (!c->no_events) DP_HIP_RET(hipEventRecord(ev_, s_)); \
  } while (0)

// Pairs per wave of the planar check: 128 / lanes_per_pair when that is set, so
// that the settings 2 to 64 span what the rule on the pair count chooses from
// (with 64 / lanes a tuned shape stopped at 32 pairs: 0.42 ms against 0.32 for
// 1.95M pairs).
static int32_t planar_pairs_per_wave(const dp_ctx* c) {
  return c->tiles.lanes_per_pair > 0 ? 128 / c->tiles.lanes_per_pair : 0;
}

int dp_launch_expand(dp_ctx* c, const dp_expand_params* p, hipStream_t s) {
  const int nx = c->desc.nx;
  const int32_t N = c->N;
  const double r_app = app_radius(c, p);                                 // dbastar.cpp:585-586 (float product)
  const double r_dup = (1. - (double)p->alpha) * (double)p->delta;      // dbastar.cpp:852
  const double goal_bound = p->delta_factor_goal * (double)p->delta;    // dbastar.cpp:827

  if (!c->select_mode && (c->grid_dirty || c->grid_radius != r_dup || !dp_tail_fits(c))) {
    int rc = dp_launch_visited_rebuild(c, r_dup, s);
    if (rc) return rc;
  }
  if (!c->select_mode) c->nv_ready = c->nv;

  // The check stage counts the contenders into their grid cells as it finds
  // them; limit 0 takes pairs out again after it (k_precap_first), so there
  // they are counted later.
  const bool small = dp_small_batch(c, p);
  const bool count = !c->select_mode && p->limit_branching_factor != 0 && !small;
  int rc = c->select_mode || small ? DP_OK : dp_ensure_cont_grid(c);
  if (rc) return rc;
  c->counts_fresh = false;
  DP_EV(c->ev[0], s);
  dp_begin(c->d_counters, c->d_app_cnt, c->app_ready ? 0 : N, c->d_cont_count, count ? c->grid.nslots : 0, dp_stage(c, 1u << 0), s);
  const app_bounds B = make_app_bounds(c, r_app);
  rc = dispatch_nx(nx, [&](auto NXc) -> int {
    constexpr int NX = decltype(NXc)::value;
    // counted already when the batch did not fit its pair arrays outright
    // (1000 nodes x 5000 primitives: 15 us of a steering selection's 234)
    if (!c->app_ready) launch_app<NX>(c, B, r_app, s);
    fill_args f{};
    f.N = N;
    f.P = c->P;
    f.cnt = c->d_app_cnt;
    f.app = c->d_app;
    f.scan = N <= kFillScan ? 1 : 0;
    f.mask = c->d_app_mask;
    f.order = c->d_order;
    f.rows = c->order_rows;
    f.pnode = c->d_pnode;
    f.pprim = c->d_pprim;
    f.pair_cap = c->pair_cap;
    f.total = c->d_total;
    f.counters = c->d_counters;
    // the FP32 pass's order needs the primitive of a mask bit: with a caller's
    // order the pairs are split afterwards
    if (NX == 13 && p->fp32_rollout && !c->d_order) {
      f.qshort = c->d_qshort;
      f.qperm = reinterpret_cast<int2*>(c->d_qperm);
      f.nshort = c->d_nshort;
      f.chunks = c->d_chunk;
    }
    if (!f.scan) dp_scan_small(c->d_app_cnt, c->d_app, N, c->d_total, c->pair_cap, c->d_counters, DPC_PAIRS, s);
    if (c->d_order) k_app_fill<true><<<N, 64, 0, s>>>(f);
    else k_app_fill<false><<<N, 64, 0, s>>>(f);
    return DP_OK;
  });
  if (rc) return rc;
  if (p->use_surrogate) {
    if (!c->mlp.w || (p->use_surrogate == 1 && !c->mlp.ready)) {
      dp_set_error("use_surrogate needs a trained and calibrated surrogate");
      return DP_ERR_STATE;
    }
    if (c->desc.system == DP_SYS_QUADROTOR) {
      dp_set_error("the surrogate is defined for planar systems");
      return DP_ERR_ARG;
    }
    rc = dp_launch_surrogate(c, p->use_surrogate == 1, s);
    if (rc) return rc;
  }
  dp_check_args a{};
  a.sys = c->d_sys;
  a.nodes = c->d_nodes;
  a.Ncap = c->N_cap;
  a.gpar = c->d_gpar;
  a.off = c->d_off;
  a.st = c->d_st;
  a.S = c->S;
  a.st4 = reinterpret_cast<const double4*>(c->d_st4);
  a.prec = c->d_prec;
  for (int k = 0; k < 4; ++k) a.reach[k] = c->forward ? c->reach_box[k] : c->reach_box_bwd[k];
  a.P = c->P;
  a.goalidx = c->d_goalidx;
  a.num_goal = p->num_check_goal;
  a.check_goal = p->check_intermediate_goal && p->num_check_goal > 0;
  a.obs = c->d_obs;
  a.nobs = c->nb;
  a.vis = c->d_vis_sorted;
  a.vstride = c->nv_cap;
  a.nv = c->nv;
  a.nv_sorted = c->nv_sorted;
  a.vstart = c->d_vis_start;
  a.grid = c->grid;
  a.pnode = c->d_pnode;
  a.pprim = c->d_pprim;
  a.total = c->d_total;
  a.verdict = c->d_verdict;
  a.firstk = c->d_firstk;
  a.goal_out = c->d_goal;
  a.res = c->d_res;
  a.flags = c->d_flags;
  a.fin = c->d_final;
  a.pcap = c->pair_cap;
  a.gout = c->d_g;
  a.hout = c->d_h;
  for (int k = 0; k < DP_MAX_NX; ++k) a.goal[k] = k < nx ? p->goal[k] : 0.0;
  a.goal_bound = goal_bound;
  a.r_dup = r_dup;
  a.cdf = p->cost_delta_factor;
  a.surrogate = p->use_surrogate ? 1 : 0;
  a.counters = c->d_counters;
  a.backward = c->forward ? 0 : 1;
  a.ncon = c->select_mode ? 0 : c->ncon;
  a.con = c->d_con;
  a.con_delta = (double)p->delta;
  a.select = c->select_mode ? 1 : 0;
  if (c->select_mode) a.nv = a.nv_sorted = 0;
  a.cont_count = count ? c->d_cont_count : nullptr;
  a.cont_cell = c->d_cont_cell;
  a.cont_place = c->d_conf_ov;

  if (c->desc.system == DP_SYS_QUADROTOR) {
    rc = dp_launch_quad(c, p, goal_bound, r_dup, count, s);
    if (rc) return rc;
    rc = small ? dp_launch_resolve_small(c, p, r_dup, s) : dp_launch_resolve(c, p, r_dup, count, s);
    if (rc) return rc;
    DP_EV(c->ev[1], s);
    c->timing_valid = !c->no_events && !c->defer_walk;
    return DP_OK;
  }
  a.ppw = planar_pairs_per_wave(c);
  a.marks = dp_stage(c, p->use_surrogate ? (1u << 1) | (1u << 5) : (1u << 4) | (1u << 1) | (1u << 5));
  // LDS: the obstacles plus one list of obstacles near a node per wave
  const size_t lds = (sizeof(double) * 4 + sizeof(int16_t) * kWaves) * (size_t)c->nb;
  // The pair count is on the device; size the grid from the bound N*P.
  const int32_t least = a.ppw > 0 ? a.ppw : 4;
  const int64_t groups = ((int64_t)N * c->P + least - 1) / least;
  const int blocks = dp_grid_blocks(groups, kWaves, c->tiles.check_blocks);
  rc = dispatch_nx(nx, [&](auto NXc) -> int {
    constexpr int NX = decltype(NXc)::value;
    if constexpr (NX == 13) {
      return DP_ERR_ARG;
    } else {
      k_check_planar<NX><<<blocks, 256, lds, s>>>(a);
      return DP_OK;
    }
  });
  if (rc) return rc;
  DP_HIP_RET(hipGetLastError());

  if (c->select_mode) {
    rc = dispatch_nx(nx, [&](auto NXc) -> int {
      constexpr int NX = decltype(NXc)::value;
      if constexpr (NX == 13) {
        return DP_ERR_ARG;
      } else {
        a.marks = dp_stage(c, (1u << 6) | (1u << 2) | (1u << 7));
        int32_t* sel_q = reinterpret_cast<int32_t*>(c->d_sel + (int64_t)(2 * nx + 3) * c->sel_cap);
        k_select<NX><<<N, 64 * kSelectWaves, 0, s>>>(a, c->d_app, N, c->d_targets, c->d_cost, c->select_cost_jump,
                                      c->select_first, sel_q, sel_q + c->sel_cap, c->d_sel);
        return DP_OK;
      }
    });
    if (rc) return rc;
    DP_HIP_RET(hipGetLastError());
    DP_EV(c->ev[1], s);
    c->timing_valid = !c->no_events && !c->defer_walk;
    return DP_OK;
  }
  rc = small ? dp_launch_resolve_small(c, p, r_dup, s) : dp_launch_resolve(c, p, r_dup, count, s);
  if (rc) return rc;
  DP_EV(c->ev[1], s);
  c->timing_valid = !c->no_events && !c->defer_walk;
  return DP_OK;
}
