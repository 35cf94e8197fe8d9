// Draft LM-head product of the draft top-k head (DDTreeDraftTopK: logits = hidden @ weight^T over the
// drafted rows, inference/sglang/patches/sglang-v0.5.22-mfd.patch:1523-1532) for gfx950, and the head's
// single entry point (the product, then the logits step of logits_topk.hip on its output).
//
// The product streams the weight (vocabulary x hidden, bf16, read once per 128 drafted rows: 778 MB at a
// 151936-token vocabulary and hidden 2560) against the drafted rows, which every workgroup shares. Three forms, by
// the drafted rows and the vocabulary rows a CU gets (draft_head_gemm): the k-split form (few drafted rows, or a
// vocabulary so small that one wave's walk over k would be the whole time), the wide form (more than 128 rows per CU)
// and, between them, the pass form described here.
//  * The vocabulary is split evenly over the grid's workgroups (one per CU; ranges of a multiple of 8 rows),
//    each taking its range in passes of 128 weight rows against all (up to 128) drafted rows.
//  * Both operands stream through LDS in 64-k stages (128 weight rows and 128 drafted rows, 128 bytes each,
//    32 KB per stage) in a ring of four stages. Two producer waves issue the direct-to-LDS loads (every load
//    instruction moves 8 whole rows x 128 contiguous bytes), up to three stages ahead; four consumer waves
//    split each pass's 128 x 128 outputs 2 x 2, a consumer computing 64 weight rows x 64 drafted rows as
//    4 x 4 v_mfma_f32_16x16x32_bf16 tiles (fp32 accumulators, 64 registers). The waves hand stages over
//    through LDS counters with bounded polling, so the consumers never stall on load issue and the producers
//    never wait for products: each producer counts the stages whose loads it has seen land, each consumer
//    the stages it has released, and a wave waits until every counter of the other side reaches the stage
//    (one shared count could be reached by a wave running two stages ahead while another lags). A wait that
//    runs out (it never should) turns the workgroup's remaining outputs into NaN instead of hanging.
//  * 16-byte chunk c of staged row r sits at slot c ^ ((r >> 1) & 7) of the row, so the 16 lanes of each
//    quarter of an operand read hit distinct banks.
//  * The drafted-row stream restarts at k = 0 for every pass: stage v of a workgroup is pass v / (K / 64),
//    k-chunk v % (K / 64). Rows past the end of a pass (the last one) read the pass's last row; rows past M
//    read row M - 1; neither is stored. A pass's outputs are rounded to bf16 (round to nearest even, as the
//    library GEMM of the reference) and stored when its last stage is done.

#include "mfd_common.h"

namespace {

constexpr int NC = 4;                 // consumer waves (2 x 2 over a pass's outputs)
constexpr int NP = 2;                 // producer waves
constexpr int NT = (NC + NP) * 64;
constexpr int MT = 128;               // drafted rows of one launch
constexpr int PT = 128;               // weight rows per pass
constexpr int KS = 64;                // k per stage
constexpr int SROW = KS * 2;          // bytes of a staged row
constexpr int WBLK = PT * SROW;       // weight block of a stage (16 KB)
constexpr int HBLK = MT * SROW;       // drafted-row block of a stage (16 KB)
constexpr int SBUF = WBLK + HBLK;     // a stage: weight block, then drafted-row block
constexpr int NBUF = 4;               // stages in the ring (128 KB)
constexpr int DPW = WBLK / 1024 / NP; // 1-KB weight loads per producer per stage (8)
constexpr int DPH = HBLK / 1024 / NP; // 1-KB drafted-row loads per producer per stage (8)
constexpr int SMEM = NBUF * SBUF + 48;  // + the hand-over counters (16-byte aligned groups) and the failure flag
constexpr int SPIN = 1 << 22;         // polls before a hand-over wait gives up (about 0.3 s: far beyond any real wait)

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct HeadArgs {
  const uint16_t* hidden;  // drafted row m at hidden + (m / rpg) * group_stride + (m % rpg) * row_stride
  int64_t row_stride, group_stride;
  int rpg;
  int row0;                // the launch's drafted rows are row0 .. row0 + M - 1
  const uint16_t* w;       // [N][K] row-major
  uint16_t* out;           // [M][out_stride], row 0 = drafted row row0
  int64_t out_stride;
  int M, N, K;
  int nwg;                 // workgroups of the grid
};

// First vocabulary row of workgroup g: an even split of N rows over nwg workgroups, rounded down to a multiple
// of 8 (non-decreasing in g; workgroup nwg starts at N).
__host__ __device__ __forceinline__ int wg_row0(int g, int N, int nwg) {
  return g >= nwg ? N : (int)(((int64_t)g * N / nwg) & ~(int64_t)7);
}

// One direct-to-LDS load (global_load_lds_dwordx4): lane l's 16 bytes at base + off land at LDS byte address
// lds_byte + 16 l (base and lds_byte wave-uniform). Inline asm: the compiler does not count it among its own
// loads; the producer waits for it explicitly.
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds_byte) {
  const uint32_t l = __builtin_amdgcn_readfirstlane(lds_byte);
  const uint64_t bb = (uint64_t)(uintptr_t)base;
  const uint64_t bs = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(bb >> 32)) << 32) |
                      (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)bb);
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(l), "v"(off), "s"(bs) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Wait until each of the NCNT (2 or 4) LDS counters at c (16-byte aligned, read together) reaches target.
// Bounded: a wait that runs out (it never should) sets the workgroup's failure flag and returns, so the kernel
// always completes and the workgroup's remaining outputs are written as NaN instead of values computed from
// stale operands.
template <int NCNT>
__device__ __forceinline__ void wait_all(const int* c, int target, int* fail) {
  static_assert(NCNT == 2 || NCNT == 4, "counter groups of 2 or 4");
  for (int it = 0; it < SPIN; ++it) {
    int lo;
    // through an LDS pointer: a generic (flat) load would also wait for the wave's global loads in flight
    if constexpr (NCNT == 2) {
      const u32x2 x = *(const __attribute__((address_space(3))) volatile u32x2*)c;
      lo = min((int)x[0], (int)x[1]);
    } else {
      const u32x4 x = *(const __attribute__((address_space(3))) volatile u32x4*)c;
      lo = min(min((int)x[0], (int)x[1]), min((int)x[2], (int)x[3]));
    }
    if (__builtin_amdgcn_readfirstlane(lo) >= target) {
      // LDS performs a wave's operations in issue order, so the stage reads (or direct-to-LDS loads) issued
      // after this poll follow it; only the compiler must not move them above it (a workgroup-scope acquire
      // fence would also wait for the producer's loads in flight)
      asm volatile("" ::: "memory");
      return;
    }
    // no sleep between polls: a hand-over is due within a few hundred cycles, and sleeping measured slower
  }
  if ((threadIdx.x & 63) == 0) __atomic_store_n(fail, 1, __ATOMIC_RELAXED);
}
__device__ __forceinline__ void signal_count(int* c) {
  if ((threadIdx.x & 63) == 0) __atomic_fetch_add(c, 1, __ATOMIC_RELEASE);
}
// A consumer's release of a stage: LDS performs a wave's operations in issue order, so a counter update issued
// after the stage's reads lands after them; no wait for the reads' data is needed.
__device__ __forceinline__ void signal_after_reads(int* c) {
  asm volatile("" ::: "memory");
  if ((threadIdx.x & 63) == 0) __atomic_fetch_add(c, 1, __ATOMIC_RELAXED);
}

__global__ __launch_bounds__(NT) void draft_head_kernel(HeadArgs a) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  int* ready = reinterpret_cast<int*>(smem + NBUF * SBUF);  // [NP]: stages producer p has seen land
  int* done = ready + 4;                                     // [NC]: stages consumer c has released
  int* fail = ready + 8;                                     // set by a hand-over wait that ran out
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R0 = wg_row0(blockIdx.x, a.N, a.nwg);
  const int rows = wg_row0(blockIdx.x + 1, a.N, a.nwg) - R0;
  if (rows <= 0) return;
  const int K = a.K;
  const int SK = K / KS;                   // stages per pass
  const int npass = (rows + PT - 1) / PT;
  const int S = npass * SK;
  if (tid < 9) ready[tid] = 0;
  __syncthreads();

  if (w >= NC) {
    // ---------------------------------------------------------- producer p: half of each block's rows
    const int p = w - NC;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
    // load i fills block rows 64 p + 8 i + lane / 8 (weight and drafted-row blocks alike), at slot lane % 8
    // (chunk (lane % 8) ^ ((row >> 1) & 7))
    uint32_t hoff[DPH], wrow[DPW], wchunk[DPW], woff[DPW];
#pragma unroll
    for (int i = 0; i < DPH; ++i) {
      const int row = 64 * p + 8 * i + (lane >> 3);
      const int c = (lane & 7) ^ ((row >> 1) & 7);
      const int m = a.row0 + min(row, a.M - 1);
      hoff[i] = (uint32_t)(((int64_t)(m / a.rpg) * a.group_stride + (int64_t)(m % a.rpg) * a.row_stride + 8 * c) * 2);
    }
#pragma unroll
    for (int i = 0; i < DPW; ++i) {
      const int row = 64 * p + 8 * i + (lane >> 3);
      wrow[i] = (uint32_t)row;
      wchunk[i] = (uint32_t)(16 * ((lane & 7) ^ ((row >> 1) & 7)));
    }
    int lp = -1, lkc = SK - 1;
    const uint16_t* wp = a.w;
    for (int v = 0; v < S; ++v) {
      if (++lkc == SK) {  // next pass: its weight rows, the last one repeated past the range
        lkc = 0;
        ++lp;
        wp = a.w + ((int64_t)R0 + (int64_t)PT * lp) * K;
        const int last = min(PT, rows - PT * lp) - 1;
#pragma unroll
        for (int i = 0; i < DPW; ++i) woff[i] = (uint32_t)min((int)wrow[i], last) * (uint32_t)(2 * K) + wchunk[i];
      }
      // publish stage v - (NBUF - 1) as soon as it has landed (at most NBUF - 2 later stages in flight),
      // before waiting for the slot of stage v, so a slow slot never delays a ready stage
      if (v >= NBUF - 1) {
        wait_vmcnt<(DPW + DPH) * (NBUF - 2)>();
        signal_count(ready + p);
      }
      if (v >= NBUF) wait_all<NC>(done, v - NBUF + 1, fail);  // every consumer has released the slot's last stage
      const uint32_t dst = lds0 + (uint32_t)(v % NBUF) * SBUF;
      const uint32_t kb = (uint32_t)lkc * SROW;
#pragma unroll
      for (int i = 0; i < DPW; ++i) dma16(wp, woff[i] + kb, dst + (uint32_t)(64 * p) * SROW + 1024u * i);
#pragma unroll
      for (int i = 0; i < DPH; ++i) dma16(a.hidden, hoff[i] + kb, dst + WBLK + (uint32_t)(64 * p) * SROW + 1024u * i);
    }
    wait_vmcnt<0>();
    for (int v = max(S - (NBUF - 1), 0); v < S; ++v) signal_count(ready + p);
    return;
  }

  // -------------------------------------------------------------------- consumer: outputs 64 wa .., 64 wb ..
  const int wa = w & 1, wb = w >> 1;
  const int l16 = lane & 15, g4 = lane >> 4;
  // operand fragments of step st: row (block row base) + l16, chunk 4 st + g4
  uint32_t boff[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) boff[st] = (uint32_t)(l16 * SROW + (((4 * st + g4) ^ ((l16 >> 1) & 7)) << 4));

  f32x4 acc[4][4];
#pragma unroll
  for (int o = 0; o < 4; ++o)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[o][j] = (f32x4){};
  auto read_ops = [&](int v, int st, bf16x8 (&fa)[4], bf16x8 (&fb)[4]) __attribute__((always_inline)) {
    const uint8_t* base = smem + (v % NBUF) * SBUF;
#pragma unroll
    for (int o = 0; o < 4; ++o)
      fa[o] = *reinterpret_cast<const bf16x8*>(base + (64 * wa + 16 * o) * SROW + boff[st]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      fb[j] = *reinterpret_cast<const bf16x8*>(base + WBLK + (64 * wb + 16 * j) * SROW + boff[st]);
  };
  auto mfma16x16 = [&](const bf16x8 (&fa)[4], const bf16x8 (&fb)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int o = 0; o < 4; ++o)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[o][j] = mfma16(fa[o], fb[j], acc[o][j]);
  };
  // C register r of accumulator (o, j): weight row 64 wa + 16 o + 4 g4 + r of the pass, drafted row
  // 64 wb + 16 j + l16
  auto epilogue = [&](int pass) __attribute__((always_inline)) {
    const int nloc = PT * pass + 64 * wa + 4 * g4;  // the lane's first row within the workgroup's range
    const bool failed = __builtin_amdgcn_readfirstlane(__atomic_load_n(fail, __ATOMIC_RELAXED)) != 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = 64 * wb + 16 * j + l16;
      if (m < a.M) {
        uint16_t* orow = a.out + (int64_t)m * a.out_stride + R0;
#pragma unroll
        for (int o = 0; o < 4; ++o) {
          const int n = nloc + 16 * o;
          const f32x4 c = acc[o][j];
          u32x2 pk = {__builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){c[0], c[1]}, bf16x2)),
                      __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){c[2], c[3]}, bf16x2))};
          if (failed) pk = (u32x2){0x7FC07FC0u, 0x7FC07FC0u};  // bf16 quiet NaNs
          if (n + 4 <= rows) {
            *reinterpret_cast<u32x2*>(orow + n) = pk;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < rows) orow[n + e] = (uint16_t)(pk[e >> 1] >> (16 * (e & 1)));
          }
        }
      }
    }
#pragma unroll
    for (int o = 0; o < 4; ++o)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[o][j] = (f32x4){};
  };

  // Stage v: step 1's operands are read while step 0's products run; then, once stage v + 1 has landed, its
  // step-0 operands are read while step 1's products run (the last stage reads an unused slot instead, never
  // used); stage v is released once all of its reads are issued. Two register sets alternate for the step-0
  // operands (unrolled by two).
  bf16x8 fa0[2][4], fb0[2][4], fa1[4], fb1[4];
  wait_all<NP>(ready, 1, fail);
  read_ops(0, 0, fa0[0], fb0[0]);
  int ckc = 0, cp = 0;  // pass and k-chunk of the stage computed
  auto stage = [&](int v, int par) __attribute__((always_inline)) {
    read_ops(v, 1, fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    mfma16x16(fa0[par], fb0[par]);
    __builtin_amdgcn_sched_barrier(0);
    wait_all<NP>(ready, min(v + 2, S), fail);
    read_ops(v + 1, 0, fa0[par ^ 1], fb0[par ^ 1]);
    __builtin_amdgcn_sched_barrier(0);
    mfma16x16(fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    signal_after_reads(done + w);
    if (++ckc == SK) {
      epilogue(cp);
      ckc = 0;
      ++cp;
    }
  };
  int v = 0;
  for (; v + 1 < S; v += 2) {
    stage(v, 0);
    stage(v + 1, 1);
  }
  if (v < S) stage(v, 0);
}


// C registers of a tile pair to bf16 and out: weight rows n .. n + 3 of the range, drafted row's output at orow.
__device__ __forceinline__ void store4(uint16_t* orow, int n, int rows, const f32x4& c) {
  const u32x2 pk = {__builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){c[0], c[1]}, bf16x2)),
                    __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){c[2], c[3]}, bf16x2))};
  if (n + 4 <= rows) {
    *reinterpret_cast<u32x2*>(orow + n) = pk;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < rows) orow[n + e] = (uint16_t)(pk[e >> 1] >> (16 * (e & 1)));
  }
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const uint16_t* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ bf16x8 buffer_load8(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t soff) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, off, soff, 0));
}
// Byte offset of the launch's drafted row r (rows past the last repeat it).
__device__ __forceinline__ uint32_t drafted_off(const HeadArgs& a, int r) {
  const int m = a.row0 + min(r, a.M - 1);
  return (uint32_t)(((int64_t)(m / a.rpg) * a.group_stride + (int64_t)(m % a.rpg) * a.row_stride) * 2);
}

// ---- Wide form, for workgroup ranges of more than one 128-row pass. The pass form reads all drafted rows again for
//      every pass; here a workgroup holds accumulators for its whole range (up to WRMAX rows) and walks k once.
//      Bound by the weight's way from memory.
//  * Eight waves (two per SIMD) share the range's 16-row tiles evenly, each up to VTW neighbouring ones against all
//    128 drafted rows (8 tiles): 8 VTW v_mfma_f32_16x16x32_bf16 accumulators (160 registers at VTW 5). VTW follows
//    the range, so that a short one does not carry the registers and the code of a long one.
//  * The weight goes straight to registers, 64 k (128 bytes of a row) at a time: a fragment takes 64 bytes of each of
//    its 16 rows, and both halves of the row's 128-byte line are loaded back to back, after the products that last
//    read the registers. (Stages of 32 k through LDS fetched every line from L2 twice, the second half long after the
//    first had left the CU's cache: 182 us at 151936 x 2560 x 120, 4.27 TB/s; so 163 us, 4.77 TB/s.)
//    Rows past the range read as zero by the buffer's bound.
//  * The drafted rows are in LDS as blocks of 256 k (512 bytes a row, 64 KB), double buffered by direct-to-LDS loads,
//    one barrier per block; 16-byte chunk c of row r sits at c ^ (r & 15), so the 16 rows of a fragment read hit
//    distinct banks.
namespace wide {
constexpr int NW = 8;
constexpr int NTH = NW * 64;
constexpr int WRMAX = NW * 5 * 16;       // weight rows per workgroup (640)
constexpr int MTL = MT / 16;             // drafted-row tiles (8)
constexpr int KSW = 32;                  // k per step
constexpr int HS = 8;                    // steps per drafted block
constexpr int HRB = HS * KSW * 2;        // bytes of a drafted row's block (512)
constexpr int HBW = MT * HRB;            // drafted block (64 KB)
constexpr int SMEMW = 2 * HBW;
}  // namespace wide

template <int VTW>
__global__ __launch_bounds__(wide::NTH) __attribute__((amdgpu_waves_per_eu(2, 2))) void draft_head_wide_kernel(
    HeadArgs a) {
  using namespace wide;
  static_assert(VTW >= 2 && VTW <= 5, "tiles of a wave");
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R0 = wg_row0(blockIdx.x, a.N, a.nwg);
  const int rows = wg_row0(blockIdx.x + 1, a.N, a.nwg) - R0;
  if (rows <= 0) return;
  const int K = a.K;
  const int S = K / KSW;  // even
  const int l16 = lane & 15, g4 = lane >> 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // drafted block b (k 256 b ..): a load moves two rows of 512 bytes (past the last k: its last chunk, never read)
  auto issue_h = [&](int b) __attribute__((always_inline)) {
    const uint32_t slot = lds0 + (uint32_t)(b & 1) * HBW;
#pragma unroll
    for (int i = 0; i < MT / 2 / NW; ++i) {
      const int r = 2 * (i * NW + w) + (lane >> 5);
      const int c = (lane & 31) ^ (r & 15);
      const int kc = min(b * (HS * KSW) + 8 * c, K - 8);
      dma16(a.hidden, drafted_off(a, r) + 2u * (uint32_t)kc, slot + (uint32_t)(2 * (i * NW + w)) * HRB);
    }
  };
  // this wave's tiles t0 .. t0 + vtv - 1 of the range's
  const int T = (rows + 15) / 16;
  const int t0 = __builtin_amdgcn_readfirstlane(w * T / NW);
  const int vtv = __builtin_amdgcn_readfirstlane((w + 1) * T / NW) - t0;
  const __amdgpu_buffer_rsrc_t rs = buffer_of(a.w + (int64_t)R0 * K, (uint32_t)rows * (uint32_t)K * 2u);
  const uint32_t woff = ((uint32_t)(16 * t0 + l16) * (uint32_t)K + 8u * g4) * 2u;
  const uint32_t tstep = 32u * (uint32_t)K;  // bytes from a tile to the next
  f32x4 acc[VTW][MTL];
#pragma unroll
  for (int i = 0; i < VTW; ++i)
#pragma unroll
    for (int j = 0; j < MTL; ++j) acc[i][j] = (f32x4){};
  bf16x8 wf[2][VTW];
  // (i < vtv: the tile and step offset stays below the buffer's size, which the bounds check needs)
  auto load_w = [&](int v, int i) __attribute__((always_inline)) -> bf16x8 {
    return buffer_load8(rs, woff, (uint32_t)i * tstep + (uint32_t)(min(v, S - 1) * (KSW * 2)));
  };
  issue_h(0);
#pragma unroll
  for (int i = 0; i < VTW; ++i) {
    if (i >= vtv) break;
    wf[0][i] = load_w(0, i);
    wf[1][i] = load_w(1, i);
  }
  for (int b = 0; b * HS < S; ++b) {
    // the block's direct loads have landed: 2 vtv weight loads or more are younger
    if (vtv == VTW)
      wait_vmcnt<2 * VTW>();
    else if (vtv == VTW - 1)
      wait_vmcnt<2 * (VTW - 1)>();
    else
      wait_vmcnt<0>();
    __syncthreads();  // in every wave; and block b - 1 is read, so its half is free
    if ((b + 1) * HS < S) issue_h(b + 1);
    const uint8_t* base = smem + (b & 1) * HBW;
    const int end = min((b + 1) * HS, S);
#pragma unroll 1
    for (int v = b * HS; v < end; v += 2) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const uint32_t c0 = (uint32_t)(((v + p) & (HS - 1)) * 4 + g4);
        bf16x8 hf[MTL];
#pragma unroll
        for (int j = 0; j < MTL; ++j)
          hf[j] = *reinterpret_cast<const bf16x8*>(base + (16 * j + l16) * HRB + ((c0 ^ (uint32_t)l16) << 4));
#pragma unroll
        for (int i = 0; i < VTW; ++i) {
          if (i >= vtv) break;
#pragma unroll
          for (int j = 0; j < MTL; ++j) acc[i][j] = mfma16(wf[p][i], hf[j], acc[i][j]);
          if (p == 1) {
            wf[0][i] = load_w(v + 2, i);
            wf[1][i] = load_w(v + 3, i);
          }
        }
      }
    }
  }
  // C register r of accumulator (i, j): weight row 16 (t0 + i) + 4 g4 + r of the range, drafted row 16 j + l16
#pragma unroll
  for (int j = 0; j < MTL; ++j) {
    const int m = 16 * j + l16;
    if (m >= a.M) continue;
    uint16_t* orow = a.out + (int64_t)m * a.out_stride + R0;
#pragma unroll
    for (int i = 0; i < VTW; ++i)
      if (i < vtv) store4(orow, 16 * (t0 + i) + 4 * g4, rows, acc[i][j]);
  }
}

// ---- K-split form: a workgroup of four waves takes 16 VT weight rows against all of the launch's drafted rows (up to
//      16 MTL), each wave a quarter of k, the 64-k chunks w, w + 4, ..; the four partial sums meet in LDS and are added
//      in wave order. Nothing is shared before that, so no wave waits for another: both operands go straight to
//      registers (whole 128-byte lines, as in the wide form), one chunk ahead.
//      It pays where the drafted rows, read by every workgroup from L2, are few next to the weight, and where the
//      other forms have fewer tiles than waves and walk all of k in series: 8192 x 2560 weight rows x hidden, 120
//      drafted rows 34.8 (pass form) -> 26.6 us, 60 rows 33.3 -> 17.3, 15 rows 32.6 -> 14.7; 40000 x 2560, 15 rows
//      66 -> 43; 151936 x 2560, 15 rows 145.6 -> 139 (5.6 TB/s).
namespace ksplit {
constexpr int NW = 4;
constexpr int NTH = NW * 64;
constexpr int KC = 64;                   // k per chunk
}  // namespace ksplit

template <int VT, int MTL>
__global__ __launch_bounds__(ksplit::NTH) __attribute__((amdgpu_waves_per_eu(2, 2))) void draft_head_ksplit_kernel(
    HeadArgs a) {
  using namespace ksplit;
  constexpr int TT = VT * MTL;  // tiles: 1 KB of partial sums each per wave
  __shared__ f32x4 part[NW * TT * 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R0 = blockIdx.x * (16 * VT);
  const int rows = min(16 * VT, a.N - R0);
  const int K = a.K, P = K / KC;
  const int l16 = lane & 15, g4 = lane >> 4;
  const int last = (rows + 15) / 16 - 1;  // tiles past the last read it again and are not stored
  const __amdgpu_buffer_rsrc_t rw = buffer_of(a.w + (int64_t)R0 * K, (uint32_t)rows * (uint32_t)K * 2u);
  const __amdgpu_buffer_rsrc_t rh = buffer_of(a.hidden, 0xFFFFFFFFu);  // (offsets are of rows below M only)
  const uint32_t woff = ((uint32_t)l16 * (uint32_t)K + 8u * g4) * 2u;
  const uint32_t tstep = 32u * (uint32_t)K;
  uint32_t hoff[MTL];
#pragma unroll
  for (int j = 0; j < MTL; ++j) hoff[j] = drafted_off(a, 16 * j + l16) + 16u * g4;
  f32x4 acc[VT][MTL];
#pragma unroll
  for (int i = 0; i < VT; ++i)
#pragma unroll
    for (int j = 0; j < MTL; ++j) acc[i][j] = (f32x4){};
  bf16x8 wf[2][2][VT], hf[2][2][MTL];
  auto load = [&](int s, int p) __attribute__((always_inline)) {
    const uint32_t kb = (uint32_t)p * (KC * 2);
#pragma unroll
    for (int i = 0; i < VT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) wf[s][h][i] = buffer_load8(rw, woff, (uint32_t)min(i, last) * tstep + kb + 64 * h);
#pragma unroll
    for (int j = 0; j < MTL; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) hf[s][h][j] = buffer_load8(rh, hoff[j], kb + 64 * h);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto products = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < VT; ++i)
#pragma unroll
        for (int j = 0; j < MTL; ++j) acc[i][j] = mfma16(wf[s][h][i], hf[s][h][j], acc[i][j]);
  };
  if (w < P) load(0, w);
  for (int p = w; p < P; p += 2 * NW) {
    if (p + NW < P) load(1, p + NW);
    products(0);
    if (p + NW < P) {
      if (p + 2 * NW < P) load(0, p + 2 * NW);
      products(1);
    }
  }
#pragma unroll
  for (int i = 0; i < VT; ++i)
#pragma unroll
    for (int j = 0; j < MTL; ++j) part[(w * TT + i * MTL + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  for (int t = w; t < TT; t += NW) {
    const int i = t / MTL, m = 16 * (t % MTL) + l16;
    f32x4 c = part[t * 64 + lane];
#pragma unroll
    for (int x = 1; x < NW; ++x) {
      const f32x4 d = part[(x * TT + t) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] += d[e];
    }
    if (m < a.M) store4(a.out + (int64_t)m * a.out_stride + R0, 16 * i + 4 * g4, rows, c);
  }
}

template <int VT, int MTL>
void launch_ksplit(const HeadArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((draft_head_ksplit_kernel<VT, MTL>), dim3((a.N + 16 * VT - 1) / (16 * VT)), dim3(ksplit::NTH), 0,
                     stream, a);
}
// Rows of the most loaded CU when N rows go out in workgroups of 16 vt.
int64_t cu_rows(int N, int vt, int cus) {
  const int64_t wgs = ((int64_t)N + 16 * vt - 1) / (16 * vt);
  return (wgs + cus - 1) / cus * (16 * vt);
}
// The tile height that leaves the most loaded CU fewer rows; the taller where they are even (each workgroup reads the
// drafted rows once): 40000 rows x 2560, 15 drafted: 43 us with 64-row workgroups, 51 with 128; 32000: 31.5 and 30.7.
template <int VT, int MTL>
void launch_ksplit_tall_or_half(const HeadArgs& a, int cus, hipStream_t stream) {
  if (cu_rows(a.N, VT, cus) <= cu_rows(a.N, VT / 2, cus))
    launch_ksplit<VT, MTL>(a, stream);
  else
    launch_ksplit<VT / 2, MTL>(a, stream);
}

}  // namespace

static int draft_head_gemm(const uint16_t* hidden, int64_t row_stride, int rows_per_group, int64_t group_stride,
                           const uint16_t* weight, int M, int N, int K, uint16_t* out, int64_t out_stride,
                           void* stream, const char* who) {
  if (!hidden || !weight || !out) return mfd_set_error(MFD_ERR_INVALID_ARG, "%s: null pointer", who);
  if (M < 1 || N < 1 || K < 1 || rows_per_group < 1 || row_stride < 0 || group_stride < 0)
    return mfd_set_error(MFD_ERR_INVALID_ARG, "%s: bad sizes M=%d N=%d K=%d rows_per_group=%d", who, M, N, K,
                         rows_per_group);
  if (K % KS != 0)
    return mfd_set_error(MFD_ERR_UNSUPPORTED, "%s: needs K %% %d == 0 (K=%d)", who, KS, K);
  if (row_stride % 8 != 0 || group_stride % 8 != 0 || out_stride < N || out_stride % 4 != 0 ||
      (reinterpret_cast<uintptr_t>(hidden) & 15) || (reinterpret_cast<uintptr_t>(weight) & 15) ||
      (reinterpret_cast<uintptr_t>(out) & 7))
    return mfd_set_error(MFD_ERR_UNSUPPORTED,
                         "%s: drafted rows and weight need 16-byte alignment, output rows 8-byte alignment "
                         "(row_stride=%lld group_stride=%lld out_stride=%lld)",
                         who, (long long)row_stride, (long long)group_stride, (long long)out_stride);
  const int cus = mfd_num_cus();
  // one workgroup per CU (128 KB of LDS each), at least 128 weight rows each
  int nwg = std::max(1, std::min(cus, (N + PT - 1) / PT));
  if (((int64_t)N / nwg + 8) * K * 2 >= ((int64_t)1 << 32) ||
      ((int64_t)(M - 1) / rows_per_group * group_stride + (int64_t)rows_per_group * row_stride + K) * 2 >=
          ((int64_t)1 << 32))
    return mfd_set_error(MFD_ERR_UNSUPPORTED, "%s: N=%d K=%d M=%d too large for 32-bit offsets", who, N, K, M);
  // the wide form holds at most wide::WRMAX rows: longer ranges are cut again, to whole rounds of the CUs (one round of
  // the pass form reads the drafted rows eight times at 248320 x 2560: 313 us, two rounds so: 265)
  while (N / nwg + 8 > wide::WRMAX) nwg += cus;
  const int vtw = (N / nwg + 8 + 16 * wide::NW - 1) / (16 * wide::NW);  // tiles of a wave of the wide form
  {
    // the kernels' dynamic LDS limits, raised once per device
    int rc = mfd_set_max_lds(reinterpret_cast<const void*>(&draft_head_kernel), SMEM);
    if (rc == MFD_OK) rc = mfd_set_max_lds(reinterpret_cast<const void*>(&draft_head_wide_kernel<2>), wide::SMEMW);
    if (rc == MFD_OK) rc = mfd_set_max_lds(reinterpret_cast<const void*>(&draft_head_wide_kernel<3>), wide::SMEMW);
    if (rc == MFD_OK) rc = mfd_set_max_lds(reinterpret_cast<const void*>(&draft_head_wide_kernel<4>), wide::SMEMW);
    if (rc == MFD_OK) rc = mfd_set_max_lds(reinterpret_cast<const void*>(&draft_head_wide_kernel<5>), wide::SMEMW);
    if (rc != MFD_OK) return rc;
  }
  const hipStream_t st = static_cast<hipStream_t>(stream);
  // one launch per 128 drafted rows (each streams the weight once)
  for (int m0 = 0; m0 < M; m0 += MT) {
    HeadArgs a{hidden, row_stride, group_stride, rows_per_group, m0, weight, out + (int64_t)m0 * out_stride,
                out_stride, std::min(MT, M - m0), N, K, nwg};
    // The form (us at hidden 2560): k-split with up to 32 drafted rows at any vocabulary (28 rows: 32.5 against 36.6
    // in the pass form at 32000, 146.7 against 146.9 in the wide one at 151936), with up to 64 where a CU gets at most
    // 64 vocabulary rows (60 rows: 17.3 against 33.3 at 8192, 44.9 against 38.6 at 32000), with more where it gets at
    // most 32 (120 rows: 26.6 against 34.9 at 8192; 72 against 49.5 at 10000 x 4096): beyond, its reads of the
    // drafted rows outweigh the weight's. Else the pass form up to 128 rows per CU (32000: 41 against 49 in the wide
    // form) and the wide form above (34000: 51 against 72, 90000: 101 against 107).
    if (a.M <= 16)
      launch_ksplit_tall_or_half<8, 1>(a, cus, st);
    else if (a.M <= 32)
      launch_ksplit_tall_or_half<8, 2>(a, cus, st);
    else if (a.M <= 64 && N <= 64 * cus)
      launch_ksplit_tall_or_half<4, 4>(a, cus, st);
    else if (N <= 32 * cus)
      launch_ksplit_tall_or_half<2, 8>(a, cus, st);
    else if (N <= PT * cus)
      hipLaunchKernelGGL(draft_head_kernel, dim3(nwg), dim3(NT), SMEM, st, a);
    else if (vtw <= 2)
      hipLaunchKernelGGL(draft_head_wide_kernel<2>, dim3(nwg), dim3(wide::NTH), wide::SMEMW, st, a);
    else if (vtw == 3)
      hipLaunchKernelGGL(draft_head_wide_kernel<3>, dim3(nwg), dim3(wide::NTH), wide::SMEMW, st, a);
    else if (vtw == 4)
      hipLaunchKernelGGL(draft_head_wide_kernel<4>, dim3(nwg), dim3(wide::NTH), wide::SMEMW, st, a);
    else
      hipLaunchKernelGGL(draft_head_wide_kernel<5>, dim3(nwg), dim3(wide::NTH), wide::SMEMW, st, a);
    MFD_CHECK_LAUNCH();
  }
  return MFD_OK;
}

extern "C" int mfd_draft_head_gemm(const uint16_t* hidden, int64_t row_stride, int rows_per_group,
                                   int64_t group_stride, const uint16_t* weight, int M, int N, int K, uint16_t* out,
                                   int64_t out_stride, void* stream) {
  return draft_head_gemm(hidden, row_stride, rows_per_group, group_stride, weight, M, N, K, out, out_stride, stream,
                         "mfd_draft_head_gemm");
}

extern "C" int mfd_draft_topk_head(const uint16_t* hidden, int64_t row_stride, int rows_per_group,
                                   int64_t group_stride, const uint16_t* weight, int M, int N, int K,
                                   uint16_t* logits, int64_t logits_stride, int k, float* out_logp, void* out_ids,
                                   int ids_int64, float* out_logz, const int32_t* vocab_ids, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  if (M == 0) return MFD_OK;
  const int rc = draft_head_gemm(hidden, row_stride, rows_per_group, group_stride, weight, M, N, K, logits,
                                 logits_stride, stream, "mfd_draft_topk_head");
  if (rc != MFD_OK) return rc;
  return vocab_ids ? mfd_topk_logz_vocab(logits, M, N, logits_stride, k, out_logp, out_ids, ids_int64, out_logz,
                                         vocab_ids, workspace, workspace_bytes, stream)
                   : mfd_topk_logz(logits, M, N, logits_stride, k, out_logp, out_ids, ids_int64, out_logz, workspace,
                                   workspace_bytes, stream);
}
