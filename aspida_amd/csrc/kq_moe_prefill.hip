// kq_moe_prefill.hip -- the grouped MoE experts for several tokens at once as a
// grouped product over the experts' packed matrices, for every kind, on the
// arithmetic of kq_gemm.h.
//
// Per launch sequence of up to MOE_PREFILL_MAX_TOKENS tokens (LLM_MoE.Forward
// steps 4-5, src/llm/llm_moe.adb:249-299, for every token; the reference's
// prefill runs K-quant experts per token, gpu/gpu_matvec.cu:4237-4239):
//
//   moe_gx_prep     block 0: every (token, slot) job bucketed by expert (shared
//                   expert first), cut into groups of up to BP jobs; the other
//                   blocks: the tokens' activations as f16 hi / lo records, and
//                   the shared-expert gates
//   moe_gx_gate_up  per (group, 64 rows): gate and up rows of the group's expert
//                   against its jobs' tokens; h[job][row] = silu(gate) * up
//   moe_gx_hsplit   h as f16 hi / lo records, one row per job
//   moe_gx_down     per (group, 128 rows of dim): yk[job][row] = down . h[job]
//   moe_combine_mf  y[t] = sum_k top_w[t][k] yk[t, k] (ascending k) + g_t
//                   yk[t, shared] (kq_moe_mfma.hip)
//
// A group's weights are decoded once for all its jobs; a group of up to 32 jobs
// takes the one-block form of gx_columns, so a short group costs half a full
// one.  Within an expert's bucket the jobs' order is not fixed (atomic
// placement), but every output element is one job's own dot product over all
// columns in a fixed order, and the combine sums in ascending k: the results
// are deterministic.
//
// Bound by the matrix cores and the vector instructions around them (kq_gemm.h)
// from about 100 tokens, by the weights' latency below.  The Qwen3-MoE layer
// (2048x768, 128 experts and a shared one, top 8, Q4_K / Q6_K, router included):
// 1024 tokens 419 us (890 on 16x16x16 products of 64-job tiles), 512 265 (465),
// 256 179 (353), 128 162 (266), 64 153 (212 on two-job chunks); Q5_K / Q6_K 256
// tokens 190 (1457 on the vector ALUs).  At 1024 under the profiler, shortest of
// 20 launches: router 28, prep 11, gate/up 211, h split 13, down 139, combine 21.
#include <math.h>

#include <algorithm>

#include "kq_gemm.h"
#include "kq_kernels.h"
#include "kq_moe.h"

namespace kq {

struct GxMoe {
  MoeGroupedArgs g;     // weights, idx, top_w, x, sgi, y, h, yk, gsh
  uint8_t *ximg, *himg;  // records: [T][dim / 256], [T slots][I / 256]
  int* jobs;             // [T slots]: job = t slots + k, bucketed by expert position
  int4* units;           // [0].x = group count; [1 + c] = group c: {expert, first job (into jobs), job count, 0}
};

__device__ __forceinline__ int gx_expert_at(int p, int n_exp) { return p == 0 ? n_exp : p - 1; }

constexpr int PREP_THREADS = 1024;

__device__ __forceinline__ void gx_plan(const GxMoe& a, int BP) {
  __shared__ int cnt[MOE_MAX_EXP + 1], off[MOE_MAX_EXP + 2], coff[MOE_MAX_EXP + 2], cur[MOE_MAX_EXP + 1];
  const int T = a.g.T, top_k = a.g.top_k, ne = a.g.n_exp + 1, n = T * top_k, slots = top_k + 1, tid = threadIdx.x;
  for (int p = tid; p < ne; p += PREP_THREADS) cnt[p] = p == 0 ? T : 0;
  __syncthreads();
  for (int i = tid; i < n; i += PREP_THREADS) {
    const int e = a.g.idx[i];
    if (e >= 0 && e < a.g.n_exp) atomicAdd(&cnt[e + 1], 1);
  }
  __syncthreads();
  // Exclusive sums of the jobs and of the groups per position (one wave).
  if (tid < 64) {
    int rj = 0, rc = 0;
    for (int base = 0; base < ne; base += 64) {
      const int p = base + tid;
      const int c = p < ne ? cnt[p] : 0, g = (c + BP - 1) / BP;
      const int sj = wave_scan_add(c), sg = wave_scan_add(g);  // inclusive
      if (p < ne) {
        off[p] = rj + sj - c;
        coff[p] = rc + sg - g;
      }
      rj += __builtin_amdgcn_readlane(sj, 63);
      rc += __builtin_amdgcn_readlane(sg, 63);
    }
    if (tid == 0) {
      off[ne] = rj;
      coff[ne] = rc;
    }
  }
  __syncthreads();
  for (int p = tid; p < ne; p += PREP_THREADS) cur[p] = off[p];
  __syncthreads();
  for (int t = tid; t < T; t += PREP_THREADS) a.jobs[t] = t * slots + top_k;  // position 0: the shared expert
  for (int i = tid; i < n; i += PREP_THREADS) {
    const int e = a.g.idx[i];
    if (e >= 0 && e < a.g.n_exp) a.jobs[atomicAdd(&cur[e + 1], 1)] = (i / top_k) * slots + i % top_k;
  }
  const int groups = coff[ne];
  for (int c = tid; c < groups; c += PREP_THREADS) {
    int lo = 0, hi = ne - 1;  // the position p with coff[p] <= c < coff[p + 1]
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (coff[mid] <= c) lo = mid;
      else hi = mid - 1;
    }
    const int k = c - coff[lo];
    a.units[1 + c] = make_int4(gx_expert_at(lo, a.g.n_exp), off[lo] + k * BP, min(BP, cnt[lo] - k * BP), 0);
  }
  if (tid == 0) a.units[0] = make_int4(groups, 0, 0, 0);
}

// Thread t (0..31) of one record.
template <int SUMS>
__device__ __forceinline__ void gx_record(const float* x, uint8_t* rec, int t) {
  gx_split<SUMS>(x, t, [&](int f, int h) { return rec + f * 32 + h * 16; },
                 [&](int i, int h) { return rec + GX_RAUX + i * 32 + h * 16; }, rec + GX_RINV);
}

// The plan, the token records and the shared-expert gates g_t = sigmoid(sgi .
// x_t), or 1 without sgi (llm_moe.adb:285-293), are independent: one launch.
template <int SUMS>
__global__ __launch_bounds__(PREP_THREADS) void moe_gx_prep(GxMoe a, int BP, int split_blocks) {
  if (blockIdx.x == 0) {
    gx_plan(a, BP);
    return;
  }
  const int T = a.g.T, nd = a.g.dim / 256, b = blockIdx.x - 1;
  if (b < split_blocks) {
    const int q = b * (PREP_THREADS / 32) + (threadIdx.x >> 5), row = q / nd, s = q % nd;
    if (row < T)
      gx_record<SUMS>(a.g.x + (size_t)row * a.g.dim + 256 * s, a.ximg + (size_t)q * GX_REC, threadIdx.x & 31);
    return;
  }
  const int t = (b - split_blocks) * (PREP_THREADS / 64) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  float s = 0.f;
  if (a.g.sgi) {
    const float4* g4 = reinterpret_cast<const float4*>(a.g.sgi);
    const float4* x4 = reinterpret_cast<const float4*>(a.g.x + (size_t)t * a.g.dim);
    for (int i = lane; i < a.g.dim / 4; i += 64) {
      const float4 gv = g4[i], xv = x4[i];
      s = __builtin_fmaf(gv.x, xv.x, s);
      s = __builtin_fmaf(gv.y, xv.y, s);
      s = __builtin_fmaf(gv.z, xv.z, s);
      s = __builtin_fmaf(gv.w, xv.w, s);
    }
    s = wave_total(s);
  }
  if (lane == 0) a.g.gsh[t] = a.g.sgi ? 1.0f / (1.0f + expf(-s)) : 1.0f;
}

template <int SUMS>
__global__ __launch_bounds__(256) void moe_gx_hsplit(GxMoe a, int rows) {
  const int ni = a.g.I / 256, q = blockIdx.x * 8 + (threadIdx.x >> 5), row = q / ni, s = q % ni;
  if (row < rows) gx_record<SUMS>(a.g.h + (size_t)row * a.g.I + 256 * s, a.himg + (size_t)q * GX_REC, threadIdx.x & 31);
}

// The unit of workgroup b among N (groups times tiles): the shared expert's S
// first, dealt over the XCDs (workgroup b runs on XCD b % 8), then each XCD a
// run of consecutive units, so that the groups of one expert, which read the
// same weights, share an L2.  -1: none.
__device__ __forceinline__ int gx_unit(int b, int N, int S) {
  const int S8 = (S + 7) & ~7;
  if (b < S8) return b < S ? b : -1;
  const int per = (N - S + 7) >> 3, x = (b - S8) & 7, l = (b - S8) >> 3, u = S + x * per + l;
  return l < per && u < N ? u : -1;
}

template <int NV>
__device__ __forceinline__ GxRows<NV> gx_rows(const uint8_t* img, int rows, const int* list, const int4& G, int div,
                                              uint32_t stride, int lane) {
  GxRows<NV> X;
  X.img = gx_buffer(img, (size_t)rows * stride);
  X.h16 = 16 * (lane >> 5);
#pragma unroll
  for (int v = 0; v < NV; ++v) {  // past the group: its first job again
    const int k = 32 * v + (lane & 31);
    X.row[v] = (uint32_t)(list[G.y + (k < G.z ? k : 0)] / div) * stride;
  }
  return X;
}

// Waves 0 and 2 take the gate's, 1 and 3 the up projection's rows 0..31 and
// 32..63 of a tile; the up sums meet the gate's in LDS.
template <int KIND, int NV>
__device__ __forceinline__ void gx_gate_up(const GxMoe& a, const int4& G, int tile, uint8_t* lds, const int* jb) {
  const int nsb = a.g.dim / 256, slots = a.g.top_k + 1;
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), up = w & 1, rb = w >> 1;
  const int e = __builtin_amdgcn_readfirstlane(G.x);
  const uint8_t* W = e == a.g.n_exp ? (up ? a.g.sh_up : a.g.sh_gate)
                                    : (up ? a.g.up : a.g.gate) + (size_t)e * a.g.gu_stride;
  const GxRows<NV> X = gx_rows<NV>(a.ximg, a.g.T, a.jobs, G, slots, (uint32_t)nsb * GX_REC, lane);
  f16v acc[NV];
  gx_columns<KIND, NV>(W + (size_t)tile * nsb * GxW<KIND>::GB, 32 * rb, 0, nsb, X, lds, acc);
  __syncthreads();
  float* xch = reinterpret_cast<float*>(lds) + rb * NV * 16 * 64 + lane;
  if (up)
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int i = 0; i < 16; ++i) xch[(v * 16 + i) * 64] = acc[v][i];
  __syncthreads();
  if (up) return;
  float* out = a.g.h + 64 * tile + 32 * rb + n;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int job = jb[32 * v + (i & 3) + 8 * (i >> 2) + 4 * h];
      const float x = acc[v][i], y = (x / (1.0f + expf(-x))) * xch[(v * 16 + i) * 64];
      if (job >= 0) out[(size_t)job * a.g.I] = y;
    }
}

template <int KIND, int NV>
__device__ __forceinline__ void gx_down(const GxMoe& a, const int4& G, int blk, uint8_t* lds, const int* jb) {
  const int nsb = a.g.I / 256;
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = __builtin_amdgcn_readfirstlane(G.x), tile = 2 * blk + (w >> 1), row0 = 32 * (w & 1);
  const uint8_t* W = e == a.g.n_exp ? a.g.sh_down : a.g.down + (size_t)e * a.g.d_stride;
  const GxRows<NV> X = gx_rows<NV>(a.himg, a.g.T * (a.g.top_k + 1), a.jobs, G, 1, (uint32_t)nsb * GX_REC, lane);
  f16v acc[NV];
  gx_columns<KIND, NV>(W + (size_t)tile * nsb * GxW<KIND>::GB, row0, 0, nsb, X, lds, acc);
  float* out = a.g.yk + 64 * tile + row0 + n;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int job = jb[32 * v + (i & 3) + 8 * (i >> 2) + 4 * h];
      if (job >= 0) out[(size_t)job * a.g.dim] = acc[v][i];
    }
}

// NVM = 2: groups of up to 64 jobs; 1: up to 32, at a higher occupancy.
template <int KIND, int NVM, bool DOWN>
__global__ __launch_bounds__(256, NVM == 1 && KIND != Q8_0 ? 3 : 2) void moe_gx_expert(GxMoe a, int tiles, int shared_units) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  __shared__ int jb[32 * NVM];
  const int u = gx_unit(blockIdx.x, a.units[0].x * tiles, shared_units);
  if (u < 0) return;
  const int4 G = a.units[1 + u / tiles];
  const int tile = u % tiles;
  if (threadIdx.x < 32 * NVM) jb[threadIdx.x] = (int)threadIdx.x < G.z ? a.jobs[G.y + threadIdx.x] : -1;
  __syncthreads();
  if (NVM == 2 && G.z > 32) {
    if constexpr (DOWN) gx_down<KIND, NVM>(a, G, tile, lds, jb);
    else gx_gate_up<KIND, NVM>(a, G, tile, lds, jb);
  } else {
    if constexpr (DOWN) gx_down<KIND, 1>(a, G, tile, lds, jb);
    else gx_gate_up<KIND, 1>(a, G, tile, lds, jb);
  }
}

// ---- host side --------------------------------------------------------------

// Whether T tokens may take this path at all (moe_prefill_takes decides by the
// kinds and the experts).  Small experts are bound by launches, of which this
// path has two more: 1024x256, 16 experts, top 2 45 us against 35 at 48 tokens.
static bool gx_may_take(int T, int dim, int I) {
  return dim % 256 == 0 && I % 256 == 0 && (T >= 96 || (T >= 4 && (size_t)dim * I >= (size_t)1 << 19));
}

static size_t gx_round(size_t n) { return (n + 255) / 256 * 256; }

// Groups a plan can produce: ceil(jobs / BP) plus one partial group per
// non-empty position.
static size_t gx_max_groups(int T, int top_k, int n_exp, int bp) {
  const size_t jobs = (size_t)T * (top_k + 1);
  return (jobs + bp - 1) / bp + std::min<size_t>((size_t)n_exp, (size_t)T * top_k) + 1;
}

static uint8_t* gx_layout(GxMoe& a, uint8_t* p) {
  const size_t T = a.g.T, J = T * (a.g.top_k + 1), nd = a.g.dim / 256, ni = a.g.I / 256;
  auto take = [&](size_t bytes) {
    uint8_t* r = p;
    p += gx_round(bytes);
    return r;
  };
  a.ximg = take(T * nd * GX_REC);
  a.himg = take(J * ni * GX_REC);
  a.g.h = (float*)take(J * a.g.I * 4);
  a.g.yk = (float*)take(J * a.g.dim * 4);
  a.g.gsh = (float*)take(T * 4);
  a.jobs = (int*)take(J * 4);
  a.units = (int4*)take((1 + gx_max_groups(a.g.T, a.g.top_k, MOE_MAX_EXP, 32)) * 16);
  return p;
}

size_t moe_prefill_work_bytes(int T, int dim, int I, int top_k) {
  if (!gx_may_take(T, dim, I)) return 0;
  T = std::min(T, MOE_PREFILL_MAX_TOKENS);
  GxMoe a{};
  a.g.T = T; a.g.dim = dim; a.g.I = I; a.g.top_k = top_k;
  return (size_t)(gx_layout(a, nullptr) - (uint8_t*)nullptr);
}

// Expected jobs per routed expert from which groups hold up to 64 jobs instead
// of 32: a group of 33..64 then costs one decode of the weights instead of two,
// at two workgroups per CU instead of three.
constexpr double MOE_GX_WIDE = 24;

// The other paths' time grows with the jobs (chunks of two on the matrix cores
// for Q4_K / Q6_K, one job at a time on the vector ALUs for the other kinds),
// this one's mostly with the distinct experts, plus two more launches.  Times
// in us, this path / the other, per layer with the router on MI355X.
bool moe_prefill_takes(int T, int gu_kind, int down_kind, int dim, int I, int top_k, int n_exp) {
  // The records are addressed with 32-bit offsets.
  const size_t t = std::min(T, MOE_PREFILL_MAX_TOKENS);
  if (!gx_may_take(T, dim, I) || gu_kind < 0 || gu_kind > Q8_0 || down_kind < 0 || down_kind > Q8_0 || top_k < 1 || top_k > MOE_MAX_TOPK || n_exp < 1 || n_exp > MOE_MAX_EXP ||
      t * (top_k + 1) * (I / 256) * GX_REC >= (size_t)1 << 32 || t * (dim / 256) * GX_REC >= (size_t)1 << 32)
    return false;
  const long jobs = (long)T * top_k;
  // Q4_K / Q6_K: at 48 tokens 2048x768 with 128 experts, top 8 161 / 172; with
  // 60, top 4 91 / 99; with 16, top 2 63 / 69 (at 32: 150 / 126, 90 / 77, 63 /
  // 55).  Many jobs per expert pay earlier: 16 experts, top 8 61 / 67 at 16.
  // Fewer than about two per expert, the shared one's counted too, do not pay at
  // any T: a group then holds what two chunks do.  Experts alone, Q4_K / Q4_K
  // 2048x768: 128 experts, top 2 75 / 63 at 48 tokens, 87 / 83 at 72, 97 / 106 at
  // 95; top 3 88 / 79 at 48, 100 / 106 at 72; top 4 97 / 90 at 48, 105 / 111 at
  // 64; 256 experts, top 2 129 / 115 at 96, 153 / 144 at 128, 183 / 202 at 200.
  // Below 56 tokens three: 1024x512, 128 experts, top 5, Q4_K / Q6_K 51 / 49 at
  // 48, 51 / 53 at 56, and 64 experts, top 3, 1024x768 45 / 48 at 48.
  if (moe_mfma_kind(gu_kind) && moe_mfma_kind(down_kind))
    return (T >= 48 && 4 * (jobs + T) >= (T < 56 ? 12L : 9L) * n_exp) || (T >= 16 && jobs >= 6L * n_exp);
  // Others: 128 experts, top 8 at 16 tokens Q5_K/Q6_K 122 / 139, Q2_K/Q3_K 103 /
  // 110 (at 8: 96 / 90, 83 / 74); 16 experts, top 8 at 4 tokens Q5_K/Q6_K 54 / 66.
  return T >= 16 || jobs >= 2L * n_exp;
}

template <int KIND, int NVM, bool DOWN>
static hipError_t gx_expert(const GxMoe& a, size_t groups, int bp, int tiles, hipStream_t s) {
  const int shared = (a.g.T + bp - 1) / bp * tiles;
  const size_t units = std::max(groups * tiles, (size_t)shared);
  const size_t grid = (size_t)((shared + 7) & ~7) + (units - shared + 7) / 8 * 8;
  constexpr int lds = GxLds<KIND, NVM>::BYTES;
  // More than 64 KB of LDS has to be asked for.
  if (lds > 60 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(moe_gx_expert<KIND, NVM, DOWN>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((moe_gx_expert<KIND, NVM, DOWN>), dim3((unsigned)grid), dim3(256), lds, s, a, tiles, shared);
  return hipGetLastError();
}

template <bool DOWN>
static hipError_t gx_experts(const GxMoe& a, int kind, size_t groups, int bp, int tiles, hipStream_t s) {
#define KQ_GX(K) \
  case K: return bp == 64 ? gx_expert<K, 2, DOWN>(a, groups, bp, tiles, s) : gx_expert<K, 1, DOWN>(a, groups, bp, tiles, s);
  switch (kind) {
    KQ_GX(Q4_K) KQ_GX(Q6_K) KQ_GX(Q5_K) KQ_GX(Q3_K) KQ_GX(Q2_K) KQ_GX(Q8_0)
    default: return hipErrorInvalidValue;
  }
#undef KQ_GX
}

hipError_t launch_moe_prefill(const MoeGroupedArgs& g, int gu_kind, int down_kind, void* work, hipStream_t s) {
  if (g.T < 1 || g.T > MOE_PREFILL_MAX_TOKENS) return hipErrorInvalidValue;
  GxMoe a{};
  a.g = g;
  gx_layout(a, (uint8_t*)work);
  const int J = g.T * (g.top_k + 1), nd = g.dim / 256, ni = g.I / 256;
  const int bp = (double)g.T * g.top_k / g.n_exp > MOE_GX_WIDE ? 64 : 32;
  const size_t groups = gx_max_groups(g.T, g.top_k, g.n_exp, bp);
  const int split = (g.T * nd * 32 + PREP_THREADS - 1) / PREP_THREADS;
  const dim3 prep(1 + split + (g.T + PREP_THREADS / 64 - 1) / (PREP_THREADS / 64));
  switch (gx_sums(gu_kind)) {
    case 0: hipLaunchKernelGGL(moe_gx_prep<0>, prep, dim3(PREP_THREADS), 0, s, a, bp, split); break;
    case 1: hipLaunchKernelGGL(moe_gx_prep<1>, prep, dim3(PREP_THREADS), 0, s, a, bp, split); break;
    default: hipLaunchKernelGGL(moe_gx_prep<2>, prep, dim3(PREP_THREADS), 0, s, a, bp, split); break;
  }
  hipError_t e = gx_experts<false>(a, gu_kind, groups, bp, g.I / 64, s);
  if (e != hipSuccess) return e;
  const dim3 hs((J * ni + 7) / 8);
  switch (gx_sums(down_kind)) {
    case 0: hipLaunchKernelGGL(moe_gx_hsplit<0>, hs, dim3(256), 0, s, a, J); break;
    case 1: hipLaunchKernelGGL(moe_gx_hsplit<1>, hs, dim3(256), 0, s, a, J); break;
    default: hipLaunchKernelGGL(moe_gx_hsplit<2>, hs, dim3(256), 0, s, a, J); break;
  }
  e = gx_experts<true>(a, down_kind, groups, bp, g.dim / 128, s);
  if (e != hipSuccess) return e;
  return launch_moe_combine(a.g, s);
}

}  // namespace kq
