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
// hide: so the softplus is formed once per (node, head), by all threads at once. 8 trees of 128 nodes, 32 heads: 5.5 us;
// 11 us with g formed again for every descendant, 16.8 us for threads that walked in memory, once per summed ancestor.
constexpr int NT = 512;
constexpr int HB = 4;       // heads per workgroup: 64 workgroups for 8 requests of 32 heads
constexpr int NMAX = 1024;  // nodes of a request held in LDS; a larger request's threads walk in memory
constexpr int PATH = 16;    // path entries held in LDS; deeper nodes walk again per ancestor

__global__ __launch_bounds__(NT) void tree_gates_kernel(GatesArgs a) {
  __shared__ float sp[NMAX][HB];  // softplus of every (node, head)
  __shared__ int16_t par[NMAX];
  __shared__ uint16_t path[NMAX][PATH];  // [s] = the s-th ancestor (0 = the node itself), request-local
  const int tid = threadIdx.x;
  const int hblocks = (a.H + HB - 1) / HB;
  const int r = blockIdx.x / hblocks;
  const int h = (blockIdx.x - r * hblocks) * HB + (tid & (HB - 1));
  const int ns = a.cu_nodes ? a.cu_nodes[r] : 0;
  const int n = (a.cu_nodes && r + 1 < a.R ? a.cu_nodes[r + 1] : a.N) - ns;  // the last request ends the batch
  const bool live = h < a.H;
  const float dt = live ? a.dt_bias[h] : 0.f, scale = live ? -expf(a.A_log[h]) : 0.f;
  // (the sum over a path takes each g = scale * softplus as the product of an FMA, rounded once with the sum)
  auto softplus_at = [&](int i) -> float {
    return softplus_torch(load_ab(a.a, a.ab_bf16, (int64_t)(ns + i) * a.ab_st + h) + dt);
  };
  // parent of a request-local node in memory: from the parents, or the largest strict ancestor in anc8
  auto parent_of = [&](int i) -> int {
    if (a.parents) return a.parents[ns + i];
    const int8_t* row = a.anc8 + (int64_t)i * a.N;
    int j = i - 1;
    while (j >= 0 && row[j] == 0) --j;
    return j;
  };
  const bool staged = n <= NMAX;
  if (staged) {
    if (a.parents) {
      // clamped to 16 bits: everything from the node on is malformed alike, everything negative ends the walk
      for (int i = tid; i < n; i += NT) par[i] = (int16_t)max(-1, min(a.parents[ns + i], NMAX));
    } else {
      // a wave per row, 64 entries at a time from the end, four rows' reads in flight
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
  }
  for (int t = tid; t < n * HB; t += NT) {
    const int i = t / HB;
    if (live) {
      const int64_t at = (int64_t)(ns + i) * a.H + h;
      a.beta[at] = 1.f / (1.f + expf(-load_ab(a.b, a.ab_bf16, (int64_t)(ns + i) * a.ab_st + h)));
      if (staged) sp[i][tid & (HB - 1)] = softplus_at(i);
    }
  }
  __syncthreads();
  auto up = [&](int i) -> int { return staged ? (int)par[i] : parent_of(i); };
  // nodes on the root path of a node, -1 for a malformed one
  auto depth_of = [&](int i, bool store) -> int {
    int d = 0;
    for (int cur = i; cur >= 0; ++d) {
      if (store && d < PATH) path[i][d] = (uint16_t)cur;
      const int p = up(cur);
      if (p >= cur || d >= MAX_WALK) return -1;
      cur = p;
    }
    return d;
  };
  __shared__ int16_t depth[NMAX];
  if (staged) {
    for (int i = tid; i < n; i += NT) depth[i] = (int16_t)depth_of(i, true);
    __syncthreads();
  }
  for (int t = tid; t < n * HB; t += NT) {
    if (!live) break;
    const int i = t / HB;
    const int d = staged ? (int)depth[i] : depth_of(i, false);
    float G = 0.f;
    if (d < 0) {
      if (a.err) atomicOr(a.err, MFD_DEVERR_NOT_TOPOLOGICAL);
      G = __builtin_nanf("");
    } else if (staged && d <= PATH) {
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
        for (int q = 0; q < s; ++q) cur = up(cur);
        G = fmaf(scale, staged ? sp[cur][tid & (HB - 1)] : softplus_at(cur), G);
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
  const int64_t blocks = (int64_t)R * ((H + HB - 1) / HB);
  if (blocks > 0x7FFFFFFF) return mfd_set_error(MFD_ERR_UNSUPPORTED, "mfd_tree_gates: too many requests x heads");
  hipLaunchKernelGGL(tree_gates_kernel, dim3((unsigned)blocks), dim3(NT), 0, static_cast<hipStream_t>(stream), args);
  MFD_CHECK_LAUNCH();
  return MFD_OK;
}
