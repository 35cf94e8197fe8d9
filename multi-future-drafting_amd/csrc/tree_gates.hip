// Gates of a Gated-DeltaNet layer over a draft tree, for gfx950.
//
// Follows inference/hf/qwen35_tree.py:77-79: beta = sigmoid(float(b)),
// g = -exp(float(A_log)) * softplus(float(a) + float(dt_bias)) (torch's softplus: x above 20 is returned
// as is, else log1p(exp(x))), and G = anc @ g, the log decay summed over the node's ancestors and itself.
// The reference forms G with a dense [n, n] x [n, H] product; here a workgroup takes one request's nodes with four
// heads: the softplus of every (node, head) and every node's root path (parents precede children, so the walk up the
// parent pointers ends at the root) go to LDS, then each (node, head) thread sums g over the path from the root down.
#include "mfd_common.h"

namespace {

constexpr int MAX_WALK = 4096;  // parent steps before a malformed (cyclic) tree is rejected

struct GatesArgs {
  const void* a;
  const void* b;
  int ab_bf16;
  int64_t ab_st;  // row stride of a and b (elements)
  const float* A_log;
  const float* dt_bias;
  const int32_t* parents;
  const int8_t* anc8;
  const int32_t* cu_nodes;
  int R, N, H;
  float* g_cum;
  float* beta;
  int32_t* err;
};

__device__ __forceinline__ float load_ab(const void* p, int ab_bf16, int64_t idx) {
  return ab_bf16 ? bf2f(reinterpret_cast<const uint16_t*>(p)[idx]) : reinterpret_cast<const float*>(p)[idx];
}

__device__ __forceinline__ float softplus_torch(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// What bounds it: latency, that of two trips to memory (offsets, then parents and projections) and of the chain of a
// few hundred dependent operations of softplus and sigmoid, which the two waves per SIMD of a CU's one workgroup do not
// hide: so the softplus is formed once per (node, head), by all threads at once. 8 trees of 128 nodes, 32 heads:
// 5.5 us; 11 us with g formed again for every descendant, 16.8 us for threads that walked in memory, once per summed
// ancestor.
constexpr int NT = 512;
constexpr int HB = 4;       // heads per workgroup: 64 workgroups for 8 requests of 32 heads
constexpr int NMAX = 1024;  // nodes of a request held in LDS; those of a larger one go to workgroups that walk in memory
constexpr int NB = NT / HB; // nodes of such a workgroup
constexpr int PATH = 16;    // path entries held in LDS; deeper nodes walk again per ancestor

__device__ __forceinline__ float beta_of(const GatesArgs& a, int node, int h) {
  return 1.f / (1.f + expf(-load_ab(a.b, a.ab_bf16, (int64_t)node * a.ab_st + h)));
}
__device__ __forceinline__ float softplus_of(const GatesArgs& a, int node, int h, float dt) {
  return softplus_torch(load_ab(a.a, a.ab_bf16, (int64_t)node * a.ab_st + h) + dt);
}
// (The sum over a path takes each g = scale * softplus as the product of an FMA, rounded once with the sum.)

// One (node, head) of a request of more than NMAX nodes, by one thread that walks the parents in memory.
__device__ void walk_in_memory(const GatesArgs& a, int node, int h) {
  int lo = 0, hi = a.cu_nodes ? a.R - 1 : 0;  // the request: cu_nodes is sorted
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.cu_nodes[mid] <= node) lo = mid; else hi = mid - 1;
  }
  const int ns = a.cu_nodes ? a.cu_nodes[lo] : 0;
  if ((a.cu_nodes && lo + 1 < a.R ? a.cu_nodes[lo + 1] : a.N) - ns <= NMAX || node < ns) return;
  const int i = node - ns;
  const float dt = a.dt_bias[h], scale = -expf(a.A_log[h]);
  // parent of a request-local node: from the parents, or the largest strict ancestor in anc8
  auto parent_of = [&](int c) -> int {
    if (a.parents) return a.parents[ns + c];
    const int8_t* row = a.anc8 + (int64_t)c * a.N;
    int j = c - 1;
    while (j >= 0 && row[j] == 0) --j;
    return j;
  };
  const int64_t at = (int64_t)node * a.H + h;
  a.beta[at] = beta_of(a, node, h);
  int d = 0;
  for (int cur = i; cur >= 0; ++d) {
    const int p = parent_of(cur);
    if (p >= cur || d >= MAX_WALK) {
      if (a.err) atomicOr(a.err, MFD_DEVERR_NOT_TOPOLOGICAL);
      a.g_cum[at] = __builtin_nanf("");
      return;
    }
    cur = p;
  }
  float G = 0.f;
  for (int s = d - 1; s >= 0; --s) {  // s = steps from the node up to the summed ancestor
    int cur = i;
    for (int q = 0; q < s; ++q) cur = parent_of(cur);
    G = fmaf(scale, softplus_of(a, ns + cur, h, dt), G);
  }
  a.g_cum[at] = G;
}

// Workgroups 0 .. R hblocks - 1: one per request of at most NMAX nodes and four heads. Then, in batches that can hold a
// larger request, one per NB nodes of the batch and four heads for the nodes of such requests: 1400 nodes, 32 heads
// take 88 of them (15 us; 144 us by the eight workgroups of the request and its heads).
__global__ __launch_bounds__(NT) void tree_gates_kernel(GatesArgs a) {
  __shared__ float sp[NMAX][HB];  // softplus of every (node, head)
  __shared__ int16_t par[NMAX], depth[NMAX];
  __shared__ uint16_t path[NMAX][PATH];  // [s] = the s-th ancestor (0 = the node itself), request-local
  const int tid = threadIdx.x;
  const int hblocks = (a.H + HB - 1) / HB;
  const int r = blockIdx.x / hblocks;
  const int h = (blockIdx.x - r * hblocks) * HB + (tid & (HB - 1));
  const bool live = h < a.H;
  if (__builtin_expect(r >= a.R, 0)) {
    const int node = (r - a.R) * NB + tid / HB;
    if (live && node < a.N) walk_in_memory(a, node, h);
    return;
  }
  const float dt = live ? a.dt_bias[h] : 0.f, A_log = live ? a.A_log[h] : 0.f;
  // (scalar loads)
  const auto cu = (const __attribute__((address_space(4))) int32_t*)a.cu_nodes;
  const int ns = cu ? cu[r] : 0;
  const int n = (cu && r + 1 < a.R ? cu[r + 1] : a.N) - ns;  // the last request ends the batch
  if (n > NMAX) return;
  const float scale = -expf(A_log);
  if (a.parents) {
    // clamped to 16 bits: everything from the node on is malformed alike, everything negative ends the walk
    for (int i = tid; i < n; i += NT) par[i] = (int16_t)max(-1, min(a.parents[ns + i], NMAX));
  } else {
    // the largest strict ancestor in anc8: a wave per row, 64 entries at a time from the end, four rows' reads in flight
    const int lane = tid & 63;
    for (int i0 = (tid >> 6) * 4; i0 < n; i0 += NT / 16) {
      int p[4] = {-1, -1, -1, -1};
      for (int e = min(i0 + 3, n - 1); e > 0; e -= 256) {
        int8_t x[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int j = e - 256 + 64 * q + lane;
            x[u][q] = (j >= 0 && j < i0 + u && i0 + u < n) ? a.anc8[(int64_t)(i0 + u) * a.N + j] : (int8_t)0;
          }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int q = 3; q >= 0; --q) {
            const uint64_t m = __builtin_amdgcn_ballot_w64(x[u][q] != 0);
            if (p[u] < 0 && m) p[u] = e - 256 + 64 * q + 63 - __builtin_clzll(m);
          }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (lane == u && i0 + u < n) par[i0 + u] = (int16_t)p[u];
    }
  }
  for (int t = tid; t < n * HB; t += NT) {
    const int i = t / HB;
    if (live) {
      a.beta[(int64_t)(ns + i) * a.H + h] = beta_of(a, ns + i, h);
      sp[i][tid & (HB - 1)] = softplus_of(a, ns + i, h, dt);
    }
  }
  __syncthreads();
  // nodes on every node's root path, -1 for a malformed one
  for (int i = tid; i < n; i += NT) {
    int d = 0;
    for (int cur = i; cur >= 0; ++d) {
      if (d < PATH) path[i][d] = (uint16_t)cur;
      const int p = par[cur];
      if (p >= cur) {
        d = -1;
        break;
      }
      cur = p;
    }
    depth[i] = (int16_t)d;
  }
  __syncthreads();
  for (int t = tid; t < n * HB; t += NT) {
    if (!live) break;
    const int i = t / HB;
    const int d = depth[i];
    float G = 0.f;
    if (d < 0) {
      if (a.err) atomicOr(a.err, MFD_DEVERR_NOT_TOPOLOGICAL);
      G = __builtin_nanf("");
    } else if (d <= PATH) {
      // all reads in flight before the first sum, each pinned outside its select (left free, the compiler puts every
      // read and sum behind a branch of its own)
      float x[PATH];
#pragma unroll
      for (int s = PATH - 1; s >= 0; --s) x[s] = sp[path[i][s < d ? s : 0]][tid & (HB - 1)];
#pragma unroll
      for (int s = PATH - 1; s >= 0; --s) {
        asm volatile("" : "+v"(x[s]));
        const float with = fmaf(scale, x[s], G);
        G = s < d ? with : G;
      }
    } else {
      for (int s = d - 1; s >= 0; --s) {  // s = steps from the node up to the summed ancestor
        int cur = i;
        for (int q = 0; q < s; ++q) cur = par[cur];
        G = fmaf(scale, sp[cur][tid & (HB - 1)], G);
      }
    }
    a.g_cum[(int64_t)(ns + i) * a.H + h] = G;
  }
}

}  // namespace

extern "C" int mfd_tree_gates(const void* a_proj, const void* b_proj, int ab_bf16, int64_t ab_row_stride,
                              const float* A_log, const float* dt_bias, const int32_t* parents, const int8_t* anc8,
                              const int32_t* cu_nodes, int R, int N, int H, float* g_cum, float* beta,
                              int32_t* err_flag, void* stream) {
  if (R < 1 || N < 0 || H < 1 || ab_row_stride < H)
    return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_tree_gates: bad sizes R=%d N=%d H=%d stride=%lld", R, N, H,
                         (long long)ab_row_stride);
  if (!cu_nodes && R != 1) return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_tree_gates: cu_nodes required for R > 1");
  if (!parents && (!anc8 || R != 1))
    return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_tree_gates: parents required unless R == 1 and anc8 given");
  if (N == 0) return MFD_OK;
  if (!a_proj || !b_proj || !A_log || !dt_bias || !g_cum || !beta)
    return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_tree_gates: null tensor pointer");
  GatesArgs args{a_proj, b_proj, ab_bf16 ? 1 : 0, ab_row_stride, A_log, dt_bias, parents, anc8, cu_nodes, R, N, H,
                 g_cum, beta, err_flag};
  const int64_t blocks = ((int64_t)R + (N > NMAX ? (N + NB - 1) / NB : 0)) * ((H + HB - 1) / HB);
  if (blocks > 0x7FFFFFFF) return mfd_set_error(MFD_ERR_UNSUPPORTED, "mfd_tree_gates: too many requests x heads");
  hipLaunchKernelGGL(tree_gates_kernel, dim3((unsigned)blocks), dim3(NT), 0, static_cast<hipStream_t>(stream), args);
  MFD_CHECK_LAUNCH();
  return MFD_OK;
}
