// kq_gemm.hip -- products of many vectors (prompts, large decode batches) over
// packed weights of every kind on the matrix cores: Y[b][out] = W X[b].
//
//   kq_gx_split   X as f16 hi / lo fragments per 32 vectors and column
//                 (kq_gemm.h), four workgroups each
//   kq_gemm       a workgroup of four waves per 128 rows x 32 or 64 vectors x a
//                 run of columns, each wave its own 32 rows: weights decoded in
//                 registers, activations shared through LDS;
//                 with the columns split, the last workgroup adds the sums
//
// Bound by the matrix cores and the vector instructions around them: Q4_K
// 28672x4096 x 512 takes 251 to 256 us, 0.95 PFLOP/s of f16 MFMA (hi and lo; a
// plain f16 library product of 8192^3 reaches 1.12), where eight launches of the
// 64-vector kernel took 546; Q6_K 5001x3584 x 333 49 us (457 on the one-pass
// kernel, 32 vectors a launch), Q6_K 4096x14336 x 64 38 us (115), Q5_K
// 14336x4096 x 16 20 us (109 on the vector kernel, 8 vectors a launch).
// Measured and not kept: decoding a stage ahead into LDS for two waves (tile
// 128 x 64 shared, 292 against 260 us) or four (128 x 128, 331): the waits at
// its barriers cost more than the instructions saved; 64 rows x 32 vectors a
// wave: 605 vector instructions per column against 380.
#include <algorithm>

#include "kq_gemm.h"
#include "kq_kernels.h"

namespace kq {

// 32 threads per vector, eight of a block's 32 vectors per workgroup.
template <int SUMS>
__global__ __launch_bounds__(256) void kq_gx_split(const float* __restrict__ X, int B, int in_dim,
                                                   uint8_t* __restrict__ img) {
  const int m = 8 * blockIdx.z + (threadIdx.x >> 5), t = threadIdx.x & 31, nsb = in_dim / 256;
  const int s = blockIdx.x, row = blockIdx.y * 32 + m;
  uint8_t* out = img + ((size_t)blockIdx.y * nsb + s) * GX_COL;
  gx_split<SUMS>(row < B ? X + (size_t)row * in_dim + 256 * s : nullptr, t,
                 [&](int f, int h) { return out + f * 1024 + (h * 32 + m) * 16; },
                 [&](int i, int h) { return out + GX_SUM + i * 1024 + (h * 32 + m) * 16; }, out + GX_AUX + 4 * m);
}

struct GemmArgs {
  const uint8_t *P, *img;
  float *Y, *part;  // part: [ks][groups][vgroups] tiles of sums
  unsigned* count;  // arrivals per (group, vector group), zero between launches
  int nsb, out_dim, B, tiles, groups, vblocks, vgroups, ks;
};

// Wave w of a workgroup takes rows 32 w .. 32 w + 31 of a 128-row group.
template <int KIND, int NV>
__global__ __launch_bounds__(256, NV == 1 ? 3 : 2) void kq_gemm(GemmArgs a) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  // Workgroups go to the 8 XCDs round robin: the vector groups of one (128
  // rows, column run) unit are consecutive workgroups of one XCD, so its
  // weights come from HBM once and from that XCD's L2 afterwards.
  const int local = blockIdx.x >> 3, vg = local % a.vgroups;
  const int unit = (local / a.vgroups) * 8 + (blockIdx.x & 7);
  if (unit >= a.groups * a.ks) return;
  const int group = unit % a.groups, kz = unit / a.groups;
  const int s0 = a.nsb * kz / a.ks, s1 = a.nsb * (kz + 1) / a.ks;
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int want = 2 * group + (w >> 1), tile = min(want, a.tiles - 1), row0 = 32 * (w & 1);
  const size_t vstride = (size_t)a.nsb * GX_COL;
  GxDense<NV> X;
#pragma unroll
  for (int v = 0; v < NV; ++v) X.img[v] = gx_buffer(a.img + min(NV * vg + v, a.vblocks - 1) * vstride, vstride);
  X.lo16 = 16 * lane;
  f16v acc[NV];
  gx_columns<KIND, NV>(a.P + (size_t)tile * a.nsb * GxW<KIND>::GB, row0, s0, s1, X, lds, acc);
  // Columns split over ks workgroups: each stores its sums (a tile's as
  // [v][i / 2][thread] pairs), the last to arrive adds the ks of them in
  // ascending order.  Agent-scope accesses and a counter, no fence, as in
  // kq_packed.h.
  if (a.ks > 1) {
    __shared__ unsigned is_last;
    constexpr size_t TILE = (size_t)NV * 16 * 256;
    const size_t ut = (size_t)group * a.vgroups + vg, nt = (size_t)a.groups * a.vgroups;
    unsigned long long* pt = reinterpret_cast<unsigned long long*>(a.part + ut * TILE) + threadIdx.x;
    unsigned long long* mine = pt + (size_t)kz * nt * (TILE / 2);
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float f0 = acc[v][i], f1 = acc[v][i + 1];
        __hip_atomic_store(mine + (8 * v + i / 2) * 256,
                           (unsigned long long)__builtin_bit_cast(uint32_t, f0) |
                               (unsigned long long)__builtin_bit_cast(uint32_t, f1) << 32,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    unsigned* count = a.count + ut * COUNTER_STRIDE;
    if (threadIdx.x == 0)
      is_last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(a.ks - 1);
    __syncthreads();
    if (!is_last) return;
    constexpr int U = 4;  // partials in flight
    for (int k0 = 0; k0 < a.ks; k0 += U) {
      unsigned long long x[U][NV * 8];
#pragma unroll
      for (int k = 0; k < U; ++k)
#pragma unroll
        for (int q = 0; q < NV * 8; ++q)
          x[k][q] = __hip_atomic_load(pt + (size_t)min(k0 + k, a.ks - 1) * nt * (TILE / 2) + q * 256, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (k0 + k < a.ks)
#pragma unroll
          for (int q = 0; q < NV * 8; ++q) {
            const float f0 = __builtin_bit_cast(float, (uint32_t)x[k][q]);
            const float f1 = __builtin_bit_cast(float, (uint32_t)(x[k][q] >> 32));
            acc[q / 8][2 * (q % 8)] = k0 + k == 0 ? f0 : acc[q / 8][2 * (q % 8)] + f0;
            acc[q / 8][2 * (q % 8) + 1] = k0 + k == 0 ? f1 : acc[q / 8][2 * (q % 8) + 1] + f1;
          }
    }
    if (threadIdx.x == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const int row = 64 * tile + row0 + (lane & 31);
  if (want >= a.tiles || row >= a.out_dim) return;
  float* dst = a.Y + row;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int b = 32 * (NV * vg + v) + (i & 3) + 8 * (i >> 2) + 4 * h;
      if (b < a.B) dst[(size_t)b * a.out_dim] = acc[v][i];
    }
}

// ---- host side --------------------------------------------------------------

// Columns are split over workgroups until the launch has two per CU of a 256-CU
// device, into runs of at least four columns where rows are long and at most
// 8 runs where they are not: the last workgroup of a tile reads every run's
// sums, about 1 us per four (4096^2, 8 vectors: 15.0, 12.9 and 14.9 us with at
// most 4, 8 and 16 runs; 14336x4096: 768 and 1024 workgroups 21.1 and 23.2 us
// against 21.6 on Q5_K at 4 vectors, 36.3 and 35.2 against 30.0 at 48).
constexpr int GEMM_WGS = 512;
constexpr int GEMM_RUNS = 8;

// Offsets within a vector block's image are 31 bits: rows of up to 58254
// columns.  The image of one call stays below 256 MB where 64 vectors do
// (512 vectors of up to 455 columns).
constexpr size_t GEMM_IMAGE = (size_t)256 << 20;

int gemm_step(int in_dim) {
  const int nsb = in_dim / 256;
  if (nsb > INT32_MAX / GX_COL) return 0;
  const size_t pairs = GEMM_IMAGE / ((size_t)2 * nsb * GX_COL);
  return 64 * (int)std::max<size_t>(1, std::min<size_t>(GEMM_STEP / 64, pairs));
}

static int gemm_nv(int batch) { return batch > 32 ? 2 : 1; }

static int gemm_ks(int in_dim, int out_dim, int batch) {
  const int per = 32 * gemm_nv(batch), wg = ((out_dim + 127) / 128) * ((batch + per - 1) / per);
  return std::max(1, std::min({in_dim / 256, GEMM_WGS / wg, std::max(GEMM_RUNS, in_dim / 1024)}));
}

static size_t gemm_image_bytes(int in_dim, int batch) {
  return (size_t)((batch + 31) / 32) * (in_dim / 256) * GX_COL;
}

size_t gemm_launch_bytes(int in_dim, int out_dim, int batch) {
  const int per = 32 * gemm_nv(batch), ks = gemm_ks(in_dim, out_dim, batch);
  const size_t tiles = (size_t)((out_dim + 127) / 128) * ((batch + per - 1) / per);
  return gemm_image_bytes(in_dim, batch) + (ks > 1 ? ks * tiles * 128 * per * sizeof(float) : 0);
}

// A split launch has at most GEMM_WGS workgroups of 128 x 64 sums, and never
// more runs than columns.
size_t gemm_workspace_bytes(int in_dim, int out_dim, int batch) {
  batch = std::min(batch, gemm_step(in_dim));
  if (batch < 1) return 0;
  const size_t cap = (size_t)GEMM_WGS * 128 * 64 * sizeof(float);
  const size_t all = (size_t)(in_dim / 256) * ((out_dim + 127) / 128) * 128 * ((batch + 63) / 64) * 64 * sizeof(float);
  return gemm_image_bytes(in_dim, batch) + std::min(cap, all);
}

// Where this path is ahead of the others.  Its time is nearly flat up to 32
// vectors, so the line lies at a batch that depends on how the other path of
// the kind splits the matrix; times in us, this path / the other, measured on
// MI355X with every launch of a product counted.
bool gemm_takes(int kind, int in_dim, int out_dim, int batch) {
  const int nsb = in_dim / 256, tiles = (out_dim + 63) / 64;
  if (!gemm_step(in_dim)) return false;
  const long units = (long)nsb * tiles;
  // Below 192 tiles (3/4 of a 256-CU device) the one-pass kernel takes 16-row
  // blocks and converts the activations once per 16 rows instead of per 64.
  const bool narrow = tiles < 192;
  if (kind == Q4_K || kind == Q6_K) {
    // More than one launch of the others (4096^2, 96 vectors: Q4_K 24.5 / 36.3,
    // Q6_K 27.6 / 54.5; 130x512, 70 vectors: 12.5 / 22).
    if (batch > 64) return true;
    if (kind == Q4_K) {
      // 33..64: 4096^2 19.8 / 20.6, 14336x4096 30.1 / 43.4, 1024x4096 18.8 /
      // 20.1, but 2048^2 15.8 / 14.1.
      if (batch > 32) return nsb >= 16;
      // 17..32: 14336x4096 20.5 / 25.3, 4096x8192 17.6 / 19.2, 8192x4096 16.0 /
      // 16.7, 4096^2 13.2 / 14.0, 1024x4096 12.5 / 12.6, but 2048^2 10.8 / 10.4;
      // on shorter rows many tiles only (18944x3584 22.1 / 33.9, 49152x2048 26.4 /
      // 34.2 at 17).
      if (batch > 16) return nsb >= 16 || units >= 3584;
      // Up to 16 only against 16-row blocks: 8192x4096 15.3 / 18.9 at 12,
      // 8192^2 21.3 / 29.2 at 8, 4096x14336 23.7 / 27.0 at 6, but 14336x4096
      // (64-row tiles) 19.2 / 15.0 at 8.
      if (batch > 8) return narrow && (units >= 2048 || nsb >= 48);
      return batch > 4 && narrow && (units >= 3584 || nsb >= 48);
    }
    // Q6_K 33..64: 14336x4096 35.2 / 88.6, 4096^2 21.1 / 27.6, 1024x2048 16.2 /
    // 25.4; the wave-per-column kernel is ahead on few tiles of long rows up to
    // 48 (1024x14336 at 33: 32.9 / 29.9, at 64: 33.2 / 40.4), and so are two
    // launches of the one-pass kernel on few tiles of two columns, which a split
    // into runs does not shorten (4096x512 at 33: 11.7 / 9.5, at 48 11.8 / 10.1,
    // at 52 11.8 / 12.1, but 16384x512 at 33 13.4 / 25.7; one column: 8.6 / 8.8,
    // three: 12.0 / 21.2).
    if (batch > 32) return batch > 48 || units > 1024 || (nsb < 32 && (nsb != 2 || units >= 256));
    // 17..32: 4096^2 15.0 / 19.9, 1024x4096 14.1 / 18.7, but 2048^2 12.1 / 11.1.
    if (batch > 16) return nsb >= 16;
    const bool split16 = narrow && tiles >= 128 && nsb >= 16;  // 8192x4096 18.0 / 19.8 at 6
    // 9..16: 14336x4096 23.8 / 27.2 and 1024x14336 21.8 / 33.2 at 12.  From 13 on
    // rows of more than 16 columns (4096x5120 17.0 / 22.8 at 13, 4096x6144 17.0 /
    // 17.1 at 14, 1024x8192 18.2 / 20.5 at 13); at 16 columns, one for each of the
    // one-pass kernel's waves, only where its 16-row blocks are more than the CUs
    // (6144x4096 17.2 / 24.7 at 15) or for 16 vectors (4096^2 14.3 / 16.0 at 16
    // but 14.5 / 12.2 at 13, 14.4 / 13.3 at 15).
    if (batch > 8)
      return units >= 3584 || nsb >= 48 || split16 || (batch > 12 && nsb >= 16 && (nsb > 16 || tiles > 64 || batch > 15));
    // 5..8: 28672x4096 36.5 / 41.3, 8192^2 25.8 / 34.0, 4096x14336 28.0 / 29.4,
    // but 14336x4096 23.6 / 22.6 and 4096x8192 20.3 / 18.9.
    if (batch > 4) return units >= 7168 || nsb >= 48 || split16;
    return batch > 2 && units >= 16384;  // 65536x4096 65.2 / 97.3 at 3, 60.6 / 60.7 at 2
  }
  // The others' path is the vector kernel, 8 vectors a launch: 4096^2 Q5_K
  // 14.0 / 43.5 at 16, Q8_0 14.2 / 20.3 at 8, Q2_K 13.5 / 17.6 at 8; at 5
  // vectors 14.0 / 16.4 (Q5_K), 13.8 / 13.3 (Q2_K).  Up to three launches of it
  // below 16 units stay there for their bits, not for the time: each row is the
  // batch-1 vector kernel's, on products that do not fill one workgroup a CU
  // either way (Q5_K 200x512 8.8 / 19.3 at 8, 9.1 / 57.6 at 24; 64x256 6.6 / 11.2
  // at 5).
  if (units < 16 && batch <= 24) return false;
  if (batch >= 8) return true;
  // 1024x14336 at 6: Q5_K 20.9 / 22.2, Q2_K 19.9 / 18.3, Q8_0 21.3 / 20.2.
  if (batch >= 5) return nsb < 32 || tiles >= 64;
  return batch == 4 && units >= 3584;  // 14336x4096: Q5_K 21.2 / 29.9, Q2_K 18.2 / 20.5, Q8_0 21.6 / 26.8
}

template <int KIND, int NV>
static hipError_t gemm_launch(const GemmArgs& a, hipStream_t s) {
  constexpr int lds = GxLds<KIND, NV>::BYTES;
  // More than 64 KB of LDS has to be asked for.
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kq_gemm<KIND, NV>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((kq_gemm<KIND, NV>), dim3((unsigned)((a.groups * a.ks + 7) / 8 * 8 * a.vgroups)), dim3(256), lds, s,
                     a);
  return hipGetLastError();
}

template <int KIND>
static hipError_t gemm_launch(const GemmArgs& a, int nv, hipStream_t s) {
  return nv == 2 ? gemm_launch<KIND, 2>(a, s) : gemm_launch<KIND, 1>(a, s);
}

hipError_t launch_gemm(int kind, const void* P, int in_dim, int out_dim, int batch, const float* X, float* Y, void* work,
                       unsigned* count, hipStream_t s) {
  if (batch < 1 || batch > gemm_step(in_dim)) return hipErrorInvalidValue;
  GemmArgs a{};
  a.P = (const uint8_t*)P;
  a.nsb = in_dim / 256;
  a.out_dim = out_dim;
  a.B = batch;
  a.tiles = (out_dim + 63) / 64;
  const int nv = gemm_nv(batch);
  a.groups = (out_dim + 127) / 128;
  a.vgroups = (batch + 32 * nv - 1) / (32 * nv);
  a.vblocks = (batch + 31) / 32;
  a.ks = gemm_ks(in_dim, out_dim, batch);
  a.img = (const uint8_t*)work;
  a.part = (float*)((uint8_t*)work + gemm_image_bytes(in_dim, batch));
  a.Y = Y;
  a.count = count;
  const dim3 gs((unsigned)a.nsb, (unsigned)a.vblocks, 4);
  switch (gx_sums(kind)) {
    case 0: hipLaunchKernelGGL(kq_gx_split<0>, gs, dim3(256), 0, s, X, batch, in_dim, (uint8_t*)work); break;
    case 1: hipLaunchKernelGGL(kq_gx_split<1>, gs, dim3(256), 0, s, X, batch, in_dim, (uint8_t*)work); break;
    default: hipLaunchKernelGGL(kq_gx_split<2>, gs, dim3(256), 0, s, X, batch, in_dim, (uint8_t*)work); break;
  }
  hipError_t e = hipErrorInvalidValue;
  switch (kind) {
    case Q4_K: e = gemm_launch<Q4_K>(a, nv, s); break;
    case Q6_K: e = gemm_launch<Q6_K>(a, nv, s); break;
    case Q5_K: e = gemm_launch<Q5_K>(a, nv, s); break;
    case Q3_K: e = gemm_launch<Q3_K>(a, nv, s); break;
    case Q2_K: e = gemm_launch<Q2_K>(a, nv, s); break;
    case Q8_0: e = gemm_launch<Q8_0>(a, nv, s); break;
  }
  return e;
}

}  // namespace kq
