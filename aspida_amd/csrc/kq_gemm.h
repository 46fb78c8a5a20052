// kq_gemm.h -- the matrix-core core of the many-vector products (kq_gemm.hip):
// one wave multiplies a 32-row block of packed weights with 32 or 64 activation
// vectors over a run of super-block columns, for every kind.
//
// MFMA shape.  v_mfma_f32_32x32x16_f16 with the activations as A (row m =
// vector) and the weights as B (column n = weight row): lane (n = l % 32,
// h = l / 32) holds eight K elements of its weight row, and D[m][n] lands in
// lane (n, h) register i with m = i % 4 + 8 (i / 4) + 4 h, so a lane's sixteen
// results share one weight row and its d / dmin are per-lane scalars.
//
// K order.  The order of the 256 elements of a super-block is free as long as
// both operands agree.  All kinds use the one their bytes give without moving
// a code between lanes: MFMA step ks = 2 u + b (u = 0..7, b = 0, 1), lane half
// h, position p holds element 32 u + 16 h + 8 b + GX_PERM[p].  A lane's codes
// of sub-block pair u are then 16 bytes of one 16-byte chunk of its own row
// (nibbles of chunk 1 + 2 (u / 2) + h for Q4_K), and the permutation is the
// (b0, b2), (b1, b3) byte pairs that two masks of a dword give.
//
// Numerics.  Codes times their integer sub-block scale enter as f16 where the
// product stays exact (Q4_K 945, Q5_K 1953, Q2_K 45, Q3_K 128); Q6_K's
// (q - 32) sc needs 13 bits and goes in as its f16 rounding plus the exact
// remainder (-1, 0 or 1); Q8_0 applies its f16 scale in f32 per 32 elements.
// The products are formed from the code bits as subnormals c * 2^-24 times
// sc * 2^10 (Q6_K 2^8), so they are normal numbers: the matrix cores align
// products by their operands' exponents, and small subnormals lose low bits
// (Q2_K 1.4e-6, Q3_K 5.5e-7, Q8_0 1.3e-6 of the result with them).  Activations are x S = hi + lo in f16, S a
// power of two per (vector, column).  hi and lo have chains of their own: the
// matrix cores round each 16-element step to f32 at the size of the running
// sum, so one chain taking both rounds twice as often (measured against 64
// bits over 256 elements: 1.5e-7 with hi and lo alternating, 1.07e-7 apart,
// 2.8e-7 for a sequential f32 sum; the split itself 4.4e-8).  Q5_K and Q2_K,
// whose code and min sums cancel most, have two chains of hi, one per half
// column (gx_halves); Q2_K's min sums, whose mins are as large as its codes,
// have three planes and are those of the split's own values.  Error over f64,
// without / with both / of the f32 vector kernel: Q5_K 4096x1024 x 16 1.31e-7 /
// 1.07e-7 / 1.25e-7, Q2_K 9.7e-8 / 8.8e-8 / 1.07e-7, with one activation of 1e4
// in 1024 Q5_K 1.37e-7 / 9.4e-8 / 1.48e-7, Q2_K 1.65e-7 / 1.20e-7 / 1.03e-7.
// Columns are added in groups of GX_GROUP, groups then among each other.
#pragma once
#include <type_traits>

#include "kq_gx_stages.h"
#include "kq_mmq.h"

namespace kq {

typedef float f16v __attribute__((ext_vector_type(16)));

// Activation image of one (32-vector block, super-block column): 32 fragments
// of 1 KB (step ks, plane p at (2 ks + p) KB; lane l's eight halves at 16 l),
// at GX_AUX 1 / S of the 32 vectors (f32) and from GX_SUM the min-term
// fragments (sums of 32: one, hi in the lower lane half and lo in the upper;
// sums of 16: three, hi, what it leaves as lo, and what both leave).
constexpr int GX_AUX = 32 * 1024;
constexpr int GX_SUM = GX_AUX + 1024;
constexpr int GX_COL = 36 * 1024;
constexpr int GX_STAGE = 8 * 1024;
constexpr int GX_GROUP = 8;

// Which sums the kind's min term takes: 0 none, 1 sums of 32, 2 sums of 16.
__host__ __device__ constexpr int gx_sums(int kind) { return kind == Q4_K || kind == Q5_K ? 1 : kind == Q2_K ? 2 : 0; }
// Their fragments.
__host__ __device__ constexpr int gx_sum_frags(int sums) { return sums == 2 ? 3 : sums; }
// Whether hi of a column's first half has a chain of its own.
__host__ __device__ constexpr bool gx_halves(int kind) { return kind == Q5_K || kind == Q2_K; }

__device__ __forceinline__ f16v mfma3216(h8 a, h8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f16v zero16() {
  f16v z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}
__device__ __forceinline__ h8 splat8(float v) {
  const _Float16 s = (_Float16)v;
  return h8{s, s, s, s, s, s, s, s};
}
// Packed 16-bit integers below 1024 as f16 (1024 + i as bits, less 1024).
__device__ __forceinline__ h8 gx_ints(uint32_t a, uint32_t b, uint32_t c, uint32_t d, float off = 0.f) {
  constexpr uint32_t K = 0x64006400u;
  return as_h8(a | K, b | K, c | K, d | K) - splat8(1024.f + off);
}
__device__ __forceinline__ uint32_t byte_of(uint32_t lo, uint32_t hi, int i) { return bfe(i < 4 ? lo : hi, 8 * (i & 3), 8); }

// A lane's share of one super-block column of a 32-row block: its `head`
// (scales; loaded a column ahead) and `body` (codes).  A 16-byte piece of its
// row holds both steps b = 0, 1 of a sub-block pair.  load_head / load_body(j)
// read the column at g for tile row `row`, pieces at chunk offset ro = 16 row;
// body(j) is what stage j (u = 2j, 2j + 1) was the last to use.  frag(u, b) is
// the B operand of step 2u + b.
template <int KIND> struct GxW;

__device__ __forceinline__ uint32_t first(const uint4& v, int b) { return b ? v.z : v.x; }
__device__ __forceinline__ uint32_t second(const uint4& v, int b) { return b ? v.w : v.y; }

// Q4_K and Q5_K scales and mins as bytes: s[0..3], s[4..7], m[0..3], m[4..7].
struct GxScaleMin {
  uint32_t s0, s1, m0, m1;
  __device__ __forceinline__ explicit GxScaleMin(const uint4& h)
      : s0(h.y & 0x3F3F3F3Fu), s1((h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u)), m0(h.z & 0x3F3F3F3Fu),
        m1(((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)) {}
  __device__ __forceinline__ h8 scale(int u, float unit) const { return splat8((float)byte_of(s0, s1, u) * unit); }
  // The eight mins in GX_PERM order.
  __device__ __forceinline__ h8 mins() const {
    return gx_ints(m0 & 0x003F003Fu, (m0 >> 8) & 0x003F003Fu, m1 & 0x003F003Fu, (m1 >> 8) & 0x003F003Fu);
  }
};

template <> struct GxW<Q4_K> {
  static constexpr int GB = 64 * 144;
  uint4 hd, hn;
  uint4 q[4];
  __device__ __forceinline__ void load_head(const uint8_t* g, int row, int, int) { hn = ld16(g + 16 * row); }
  __device__ __forceinline__ void next_head() { hd = hn; }
  __device__ __forceinline__ void load_body(const uint8_t* g, int ro, int h, int j) {
    q[j] = ld16(g + (1 + 2 * j + h) * 1024 + ro);
  }
  __device__ __forceinline__ h8 frag(const GxScaleMin& sm, int u, int b, int) const {
    const uint4& c = q[u >> 1];
    const uint32_t x = first(c, b), y = second(c, b), m = u & 1 ? 0x00F000F0u : 0x000F000Fu;
    return as_h8(x & m, (x >> 8) & m, y & m, (y >> 8) & m) * sm.scale(u, u & 1 ? 64.f : 1024.f);
  }
  __device__ __forceinline__ GxScaleMin scales() const { return GxScaleMin(hd); }
  __device__ __forceinline__ float d() const { return f16_ada(hd.x & 0xFFFFu); }
  __device__ __forceinline__ float dmin() const { return f16_ada(hd.x >> 16); }
};

template <> struct GxW<Q5_K> {
  static constexpr int GB = 64 * 176;
  uint4 hd, hn;
  uint4 qh, qhn, q[4];
  __device__ __forceinline__ void load_head(const uint8_t* g, int row, int ro, int h) {
    hn = ld16(g + 16 * row);
    qhn = ld16(g + (1 + h) * 1024 + ro);
  }
  __device__ __forceinline__ void next_head() {
    hd = hn;
    qh = qhn;
  }
  __device__ __forceinline__ void load_body(const uint8_t* g, int ro, int h, int j) {
    q[j] = ld16(g + (3 + 2 * j + h) * 1024 + ro);
  }
  __device__ __forceinline__ h8 frag(const GxScaleMin& sm, int u, int b, int) const {
    const uint4& c = q[u >> 1];
    const uint32_t x = first(c, b) >> (4 * (u & 1)), y = (second(c, b)) >> (4 * (u & 1));
    const uint32_t hx = first(qh, b), hy = second(qh, b);
    const uint32_t tx = u < 4 ? hx << (4 - u) : hx >> (u - 4), ty = u < 4 ? hy << (4 - u) : hy >> (u - 4);
    const h8 v = as_h8((x & 0x000F000Fu) | (tx & 0x00100010u), ((x >> 8) & 0x000F000Fu) | ((tx >> 8) & 0x00100010u),
                       (y & 0x000F000Fu) | (ty & 0x00100010u), ((y >> 8) & 0x000F000Fu) | ((ty >> 8) & 0x00100010u));
    return v * sm.scale(u, 1024.f);
  }
  __device__ __forceinline__ GxScaleMin scales() const { return GxScaleMin(hd); }
  __device__ __forceinline__ float d() const { return f16_ada(hd.x & 0xFFFFu); }
  __device__ __forceinline__ float dmin() const { return f16_ada(hd.x >> 16); }
};

// Q2_K: 16 (scale, min) nibble pairs in chunk 0, scale 2u + h of sub-block
// (u, h); codes 2 bits at shift 2 (u % 4) of chunk 1 + 2 (u / 4) + h.
template <> struct GxW<Q2_K> {
  static constexpr int GB = 64 * 84;
  struct S {
    uint4 s;
    __device__ __forceinline__ h8 scale(int u, int h) const {
      const uint32_t w = u < 2 ? s.x : u < 4 ? s.y : u < 6 ? s.z : s.w;
      return splat8((float)((w >> (16 * (u & 1) + 8 * h)) & 15u) * (1024.f / (1 << (2 * (u & 3)))));
    }
    // Mins 8h .. 8h + 7 in GX_PERM order.
    __device__ __forceinline__ h8 mins(int h) const {
      const uint32_t a = (h ? s.z : s.x) >> 4, b = (h ? s.w : s.y) >> 4;
      return gx_ints(a & 0x000F000Fu, (a >> 8) & 0x000F000Fu, b & 0x000F000Fu, (b >> 8) & 0x000F000Fu);
    }
  };
  uint4 sc, scn;
  uint4 q[2];
  uint32_t dd, ddn;
  __device__ __forceinline__ void load_head(const uint8_t* g, int row, int, int) {
    scn = ld16(g + 16 * row);
    ddn = ld4(g + 5 * 1024 + 4 * row);
  }
  __device__ __forceinline__ void next_head() {
    sc = scn;
    dd = ddn;
  }
  __device__ __forceinline__ void load_body(const uint8_t* g, int ro, int h, int j) {
    if (j & 1) q[j >> 1] = ld16(g + (1 + 2 * (j >> 1) + h) * 1024 + ro);
  }
  __device__ __forceinline__ h8 frag(const S& s, int u, int b, int h) const {
    const uint4& c = q[u >> 2];
    const uint32_t x = first(c, b), y = second(c, b), m = 0x00030003u << (2 * (u & 3));
    return as_h8(x & m, (x >> 8) & m, y & m, (y >> 8) & m) * s.scale(u, h);
  }
  __device__ __forceinline__ S scales() const { return {sc}; }
  __device__ __forceinline__ float d() const { return f16_ada(dd & 0xFFFFu); }
  __device__ __forceinline__ float dmin() const { return f16_ada(dd >> 16); }
};

// Q3_K: 6-bit scales of 16 elements, code = low2 + 4 hbit - 4; hmask bit u of
// chunk h, codes at shift 2 (u % 4) of chunk 2 + 2 (u / 4) + h.
template <> struct GxW<Q3_K> {
  static constexpr int GB = 64 * 110;
  struct S {
    uint32_t s[4];
    __device__ __forceinline__ h8 scale(int u, int h) const {
      return splat8((float)((int)((s[u >> 1] >> (16 * (u & 1) + 8 * h)) & 0xFFu) - 32) * 1024.f);
    }
  };
  uint4 hm, hmn, q[2];
  uint32_t a0, a1, a2, dd, b0, b1, b2, ddn;
  __device__ __forceinline__ void load_head(const uint8_t* g, int row, int ro, int h) {
    hmn = ld16(g + h * 1024 + ro);
    const uint8_t* sp = g + 6 * 1024 + 12 * row;
    b0 = ld4(sp);
    b1 = ld4(sp + 4);
    b2 = ld4(sp + 8);
    ddn = ld2(g + 6 * 1024 + 768 + 2 * row);
  }
  __device__ __forceinline__ void next_head() {
    hm = hmn;
    a0 = b0;
    a1 = b1;
    a2 = b2;
    dd = ddn;
  }
  __device__ __forceinline__ void load_body(const uint8_t* g, int ro, int h, int j) {
    if (j & 1) q[j >> 1] = ld16(g + (2 + 2 * (j >> 1) + h) * 1024 + ro);
  }
  __device__ __forceinline__ h8 frag(const S& s, int u, int b, int h) const {
    const uint4& c = q[u >> 2];
    const uint32_t x = first(c, b) >> (2 * (u & 3)), y = (second(c, b)) >> (2 * (u & 3));
    const uint32_t hx = first(hm, b), hy = second(hm, b);
    const uint32_t tx = u < 2 ? hx << (2 - u) : hx >> (u - 2), ty = u < 2 ? hy << (2 - u) : hy >> (u - 2);
    const h8 v = as_h8((x & 0x00030003u) | (tx & 0x00040004u), ((x >> 8) & 0x00030003u) | ((tx >> 8) & 0x00040004u),
                       (y & 0x00030003u) | (ty & 0x00040004u), ((y >> 8) & 0x00030003u) | ((ty >> 8) & 0x00040004u));
    return (v - splat8(4.f / 16777216.f)) * s.scale(u, h);
  }
  __device__ __forceinline__ S scales() const {
    return {{(a0 & 0x0F0F0F0Fu) | ((a2 & 0x03030303u) << 4), (a1 & 0x0F0F0F0Fu) | (((a2 >> 2) & 0x03030303u) << 4),
             ((a0 >> 4) & 0x0F0F0F0Fu) | (((a2 >> 4) & 0x03030303u) << 4),
             ((a1 >> 4) & 0x0F0F0F0Fu) | (((a2 >> 6) & 0x03030303u) << 4)}};
  }
  __device__ __forceinline__ float d() const { return f16_ada(dd); }
  __device__ __forceinline__ float dmin() const { return 0.f; }
};

// Q6_K: sub-block pair u = 4 hh + k takes low (k < 2) or high nibbles of chunk
// 4 hh + 2 (k % 2) + h, the two high bits at shift 2 k of chunk 8 + 2 hh + h,
// and the int8 scale 2 u + h.  frag gives the product's f16 rounding, rest
// what it leaves.
template <> struct GxW<Q6_K> {
  static constexpr int GB = 64 * 210;
  struct S {
    uint4 s;
    __device__ __forceinline__ h8 scale(int u, int h) const {
      const uint32_t w = u < 2 ? s.x : u < 4 ? s.y : u < 6 ? s.z : s.w;
      return splat8((float)(int8_t)((w >> (16 * (u & 1) + 8 * h)) & 0xFFu) * 256.f);
    }
  };
  uint4 sc, scn;
  uint4 qa[2], qb[2], qh[2];
  uint32_t dd, ddn;
  __device__ __forceinline__ void load_head(const uint8_t* g, int row, int, int) {
    scn = ld16(g + 12 * 1024 + 16 * row);
    ddn = ld2(g + 13 * 1024 + 2 * row);
  }
  __device__ __forceinline__ void next_head() {
    sc = scn;
    dd = ddn;
  }
  __device__ __forceinline__ void load_body(const uint8_t* g, int ro, int h, int j) {
    if (j & 1) {
      const int hh = j >> 1;
      qa[hh] = ld16(g + (4 * hh + h) * 1024 + ro);
      qb[hh] = ld16(g + (4 * hh + 2 + h) * 1024 + ro);
      qh[hh] = ld16(g + (8 + 2 * hh + h) * 1024 + ro);
    }
  }
  __device__ __forceinline__ static uint32_t codes(uint32_t ql, uint32_t qh, int k) {
    return ((ql >> (k < 2 ? 0 : 4)) & 0x0F0F0F0Fu) | ((k < 2 ? qh << (4 - 2 * k) : qh >> (2 * k - 4)) & 0x30303030u);
  }
  __device__ __forceinline__ h8 frag(const S& s, int u, int b, int h, h8& rest) const {
    const int hh = u >> 2, k = u & 3;
    const uint4 &c = k & 1 ? qb[hh] : qa[hh], &t = qh[hh];
    const uint32_t x = codes(first(c, b), first(t, b), k), y = codes(second(c, b), second(t, b), k);
    const h8 v = as_h8(x & 0x003F003Fu, (x >> 8) & 0x003F003Fu, y & 0x003F003Fu, (y >> 8) & 0x003F003Fu) -
                 splat8(32.f / 16777216.f);
    const h8 sv = s.scale(u, h), p = v * sv;
    rest = __builtin_elementwise_fma(v, sv, -p);
    return p;
  }
  __device__ __forceinline__ S scales() const { return {sc}; }
  __device__ __forceinline__ float d() const { return f16_ada(dd); }
  __device__ __forceinline__ float dmin() const { return 0.f; }
};

// Q8_0: codes of block u in chunks 2u + h, scales in chunk 16.
template <> struct GxW<Q8_0> {
  static constexpr int GB = 64 * 272;
  struct S {
    uint4 s;
    __device__ __forceinline__ float d(int u) const {
      const uint32_t w = u < 2 ? s.x : u < 4 ? s.y : u < 6 ? s.z : s.w;
      return f16_ada(u & 1 ? w >> 16 : w & 0xFFFFu);
    }
  };
  uint4 sc, scn;
  uint4 q[8];
  __device__ __forceinline__ void load_head(const uint8_t* g, int row, int, int) { scn = ld16(g + 16 * 1024 + 16 * row); }
  __device__ __forceinline__ void next_head() { sc = scn; }
  __device__ __forceinline__ void load_body(const uint8_t* g, int ro, int h, int j) {
    q[2 * j] = ld16(g + (4 * j + h) * 1024 + ro);
    q[2 * j + 1] = ld16(g + (4 * j + 2 + h) * 1024 + ro);
  }
  __device__ __forceinline__ h8 frag(const S&, int u, int b, int) const {
    const uint4& c = q[u];
    const uint32_t x = first(c, b) ^ 0x80808080u, y = (second(c, b)) ^ 0x80808080u;
    return gx_ints(x & 0x00FF00FFu, (x >> 8) & 0x00FF00FFu, y & 0x00FF00FFu, (y >> 8) & 0x00FF00FFu, 128.f);
  }
  __device__ __forceinline__ S scales() const { return {sc}; }
};

// ---- the activation split ------------------------------------------------------
//
// Thread t (0..31, consecutive lanes) of one vector's column at x (null: zeros):
// elements 8 t .. 8 t + 7, lane half h of fragments 4 u + 2 b (hi) and 4 u + 2 b
// + 1 (lo), t = 4 u + 2 h + b.  frag(f, h) is where the vector's 16 bytes of
// fragment f, lane half h go, sums(i, h) those of min-term fragment i, inv where
// 1 / S goes.
//
// Bound by the bytes, of which a wave's loads and stores cover whole lines: the
// 9216 x 768 split of the experts' h (28 MB in, 32 out) takes 13.6 us, 4.4 TB/s,
// where 32 elements a thread took 20; with four times the threads on the few
// vectors of a decode batch Q5_K 14336x4096 x 16 went from 21.4 to 20.4 us.
template <int SUMS, class F, class G>
__device__ __forceinline__ void gx_split(const float* x, int t, F&& frag, G&& sums, uint8_t* inv) {
  const int u = t >> 2, h = (t >> 1) & 1, b = t & 1;
  float4 x0 = make_float4(0.f, 0.f, 0.f, 0.f), x1 = x0;
  if (x) {
    x0 = reinterpret_cast<const float4*>(x + 8 * t)[0];
    x1 = reinterpret_cast<const float4*>(x + 8 * t)[1];
  }
  float a = fmaxf(fmaxf(fmaxf(fabsf(x0.x), fabsf(x0.y)), fmaxf(fabsf(x0.z), fabsf(x0.w))),
                  fmaxf(fmaxf(fabsf(x1.x), fabsf(x1.y)), fmaxf(fabsf(x1.z), fabsf(x1.w))));
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) a = fmaxf(a, __shfl_xor(a, o, 64));
  // S = 2^(14 - e) with a < 2^e, at most 2^116; 1 for a column of zeros.  Beside
  // an Inf 2^-114, at which no finite element becomes one too: Q3_K and Q8_0,
  // whose weight is one factor, then give the weight's sign times Inf.  The others
  // give NaN (Q6_K's rest is mostly 0, a sum's second plane Inf - Inf).
  int e = 0;
  const bool inf = __builtin_isinf(a);
  if (a > 0.f && !inf) (void)frexpf(a, &e);
  const int ex = inf ? -114 : a > 0.f ? min(14 - e, 116) : 0;
  const float S = ldexpf(1.f, ex);
  if (t == 0) *reinterpret_cast<float*>(inv) = ldexpf(1.f, -ex);
  // What hi leaves, at most 8; the clamp takes Inf - Inf.
  auto rest = [](float v, _Float16 hi) { return (_Float16)__builtin_amdgcn_fmed3f(v - (float)hi, -32.f, 32.f); };
  x0.x *= S; x0.y *= S; x0.z *= S; x0.w *= S;
  x1.x *= S; x1.y *= S; x1.z *= S; x1.w *= S;
  const h8 hi = {(_Float16)x0.x, (_Float16)x0.z, (_Float16)x0.y, (_Float16)x0.w,
                 (_Float16)x1.x, (_Float16)x1.z, (_Float16)x1.y, (_Float16)x1.w};
  const h8 lo = {rest(x0.x, hi[0]), rest(x0.z, hi[1]), rest(x0.y, hi[2]), rest(x0.w, hi[3]),
                 rest(x1.x, hi[4]), rest(x1.z, hi[5]), rest(x1.y, hi[6]), rest(x1.w, hi[7])};
  *reinterpret_cast<h8*>(frag(4 * u + 2 * b, h)) = hi;
  *reinterpret_cast<h8*>(frag(4 * u + 2 * b + 1, h)) = lo;
  // Position p of a fragment holds sub-block GX_PERM[p] = {0, 2, 1, 3, 4, 6, 5, 7}[p], its own inverse.
  auto put = [&](int c, int i, int half, float y) {
    const int p = (c & 4) | ((c & 1) << 1) | ((c >> 1) & 1);
    *reinterpret_cast<_Float16*>(sums(i, half) + 2 * p) = (_Float16)y;
  };
  if constexpr (SUMS != 0) {
    if constexpr (SUMS == 2) {  // of what hi and lo hold, so that code and min terms cancel on the same values
      x0 = make_float4((float)hi[0] + (float)lo[0], (float)hi[2] + (float)lo[2], (float)hi[1] + (float)lo[1],
                       (float)hi[3] + (float)lo[3]);
      x1 = make_float4((float)hi[4] + (float)lo[4], (float)hi[6] + (float)lo[6], (float)hi[5] + (float)lo[5],
                       (float)hi[7] + (float)lo[7]);
    }
    float y = ((x0.x + x0.y) + (x0.z + x0.w)) + ((x1.x + x1.y) + (x1.z + x1.w));
    y += __shfl_xor(y, 1, 64);
    if constexpr (SUMS == 1) y += __shfl_xor(y, 2, 64);
    y *= XSUM_UNIT;
    const float yh = (float)(_Float16)y;
    if constexpr (SUMS == 1) {
      if (b == 0) put(u, 0, h, h ? y - yh : yh);
    } else {
      const int c = 2 * u + h;
      const float yl = (float)(_Float16)(y - yh);
      put(c & 7, b, c >> 3, b ? yl : yh);
      if (b) put(c & 7, 2, c >> 3, (y - yh) - yl);
    }
  }
}

// ---- activations: global -> LDS ---------------------------------------------
//
// buffer_load ... lds moves 16 (or 4) bytes per lane into LDS (lane l's at the
// wave-uniform destination + 16 l) without passing through registers.  Loads
// return in order, so a wait for at most n outstanding ones covers every load
// with n later ones, and a barrier then covers the other waves'.  Buffer loads,
// because the compiler counts those exactly: after a global_load_lds it waits
// for every outstanding load before it uses any loaded weight.
typedef __amdgpu_buffer_rsrc_t gx_rsrc;
__device__ __forceinline__ gx_rsrc gx_buffer(const uint8_t* base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0, (int)(uint32_t)bytes, 0x00020000);
}
__device__ __forceinline__ void gx_dma16(gx_rsrc r, uint32_t lane_off, uint32_t off, uint32_t lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(uintptr_t)lds, 16, lane_off, off, 0, 0);
}
__device__ __forceinline__ void gx_dma4(gx_rsrc r, uint32_t lane_off, uint32_t off, uint32_t lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(uintptr_t)lds, 4, lane_off, off, 0, 0);
}
// At most N of this wave's global loads outstanding, its LDS accesses done,
// then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void gx_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
// The one before stage j (a constant once its loop is unrolled).
template <int KIND, int NV, bool LAST>
__device__ __forceinline__ void gx_stage_barrier(int j) {
  switch (j) {
    case 0: gx_wait_barrier<gx_stage_wait(KIND, NV, 0, LAST)>(); break;
    case 1: gx_wait_barrier<gx_stage_wait(KIND, NV, 1, LAST)>(); break;
    case 2: gx_wait_barrier<gx_stage_wait(KIND, NV, 2, LAST)>(); break;
    default: gx_wait_barrier<gx_stage_wait(KIND, NV, 3, LAST)>(); break;
  }
}
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
}
// Where a workgroup's activations come from: fragment f (0..31) and aux
// fragment i (0: the 32 vectors' 1 / S, then the sums) of vector block v in
// column s, moved into LDS at dst.
//
// GxDense: images of whole 32-vector blocks.
template <int NV> struct GxDense {
  gx_rsrc img[NV];
  uint32_t lo16;  // 16 * lane
  __device__ __forceinline__ void frag(int v, int s, int f, uint32_t dst) const {
    gx_dma16(img[v], lo16, s * GX_COL + f * 1024, dst);
  }
  __device__ __forceinline__ void aux(int v, int s, int i, uint32_t dst) const {
    if (i == 0) gx_dma4(img[v], lo16 >> 2, s * GX_COL + GX_AUX, dst);
    else gx_dma16(img[v], lo16, s * GX_COL + GX_SUM + 1024 * (i - 1), dst);
  }
};

// GxRows: any 32 rows of an image kept row by row (the MoE experts' jobs):
// record (row, column) holds the 32 fragments' 2 x 16 bytes of its vector (32 f
// + 16 h), at GX_RAUX the sums in fragment order and at GX_RINV 1 / S.
constexpr int GX_RAUX = 1024;
constexpr int GX_RINV = GX_RAUX + 96;
constexpr int GX_REC = 1152;
template <int NV> struct GxRows {
  gx_rsrc img;
  uint32_t row[NV];  // byte offset of lane l % 32's row in block v
  uint32_t h16;      // 16 * (lane / 32)
  __device__ __forceinline__ void frag(int v, int s, int f, uint32_t dst) const {
    gx_dma16(img, row[v] + h16, s * GX_REC + f * 32, dst);
  }
  __device__ __forceinline__ void aux(int v, int s, int i, uint32_t dst) const {
    if (i == 0) gx_dma4(img, row[v], s * GX_REC + GX_RINV, dst);
    else gx_dma16(img, row[v] + h16, s * GX_REC + GX_RAUX + 32 * (i - 1), dst);
  }
};

// LDS of a workgroup of NV vector blocks: the ring of stages, then two
// columns' aux (1 / S, 4 bytes a lane, and the min-term fragments).
template <int KIND, int NV> struct GxLds {
  static constexpr int INVB = 256, AUXB = INVB + gx_sum_frags(gx_sums(KIND)) * 1024;
  static constexpr int AUX0 = gx_ring(KIND, NV) * NV * GX_STAGE, BYTES = AUX0 + 2 * NV * AUXB;
  // Three workgroups (NV = 1) or two per CU in 160 KB, each with 1 KB for what a
  // kernel has of its own (the ring starts at a multiple of that).
  static_assert((NV == 1 ? 3 : 2) * (BYTES + 1024) <= 160 * 1024, "workgroups per CU");
};

// The columns [s0, s1) of 32 rows (rows row0 .. of the 64-row tile whose packed
// columns start at W) against NV 32-vector blocks of X: acc[v][i] is the sum for
// row row0 + l % 32 and vector i % 4 + 8 (i / 4) + 4 (l / 32) of block v.  The
// four waves of the workgroup share the staged activations: all call this with
// the same s0 < s1 and X; W, row0 and X's bases are wave-uniform.
//
// 32 rows x 64 vectors a wave: a weight fragment is decoded once for four
// MFMAs (six for Q6_K).  With two waves per SIMD a wave issues a vector
// instruction every ~8 cycles and an MFMA takes 32, so the vector instructions
// per MFMA set the time: a loop of MFMAs alone runs at 14.2 ns each, with 6
// vector instructions each at 17.5, with 10 at 24 ns.
template <int KIND, int NV, class SRC>
__device__ __forceinline__ void gx_columns(const uint8_t* W, int row0, int s0, int s1, const SRC& X, uint8_t* lds,
                                           f16v (&acc)[NV]) {
  using U = GxW<KIND>;
  using L = GxLds<KIND, NV>;
  constexpr int SUMS = gx_sums(KIND), GB = U::GB, AUXN = 1 + gx_sum_frags(SUMS);
  constexpr bool HALVES = gx_halves(KIND);
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t ring = __builtin_amdgcn_readfirstlane(lds_offset(lds)), lo16 = 16 * lane;
  constexpr int R = gx_ring(KIND, NV);
  const int last = 4 * (s1 - s0) - 1;  // stages
  // Stage g's 8 NV fragments, 2 NV per wave (past the end the last stage
  // again, into a slot nobody reads, so that every stage issues as many).
  auto dma_stage = [&](int g, int slot) {
    const int c = g < last ? g : last;
    const int s = s0 + (c >> 2), f = (c & 3) * 8 + 2 * w;
    const uint32_t dst = ring + slot * NV * GX_STAGE + 2 * w * 1024;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      X.frag(v, s, f, dst + v * GX_STAGE);
      X.frag(v, s, f + 1, dst + v * GX_STAGE + 1024);
    }
  };
  auto dma_aux = [&](int c) {  // of column s0 + c, one fragment per wave in turn
    const int s = s0 + c;
    const uint32_t dst = ring + L::AUX0 + (c & 1) * NV * L::AUXB;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int i = 0; i < AUXN; ++i)
        if (((v * AUXN + i) & 3) == w) X.aux(v, s, i, dst + v * L::AUXB + (i ? L::INVB + 1024 * (i - 1) : 0));
  };
  const int row = row0 + (lane & 31), ro = 16 * row;
  U wt;
  const uint8_t* g0 = W + (size_t)s0 * GB;
  dma_aux(0);
#pragma unroll
  for (int g = 0; g < R - 1; ++g) dma_stage(g, g);
  wt.load_head(g0, row, ro, h);
#pragma unroll
  for (int j = 0; j < 4; ++j) wt.load_body(g0, ro, h, j);
  // All of them (vmcnt 0): the loop's waits then count from here on both paths
  // into it, the compiler's for the weights as well as those below.
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0F70);
  asm volatile("" ::: "memory");
  int slot = 0, fill = R - 1;  // this stage's slot, the next one to fill
  f16v sum[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) sum[v] = acc[v] = zero16();
  // One column; the last one, a form of its own, has no next one's weights to
  // load.
  auto column = [&](const int c, auto is_last) {
    constexpr bool LAST = decltype(is_last)::value;
    wt.next_head();
    if constexpr (!LAST) {
      g0 += GB;
      wt.load_head(g0, row, ro, h);
    }
    const auto sc = wt.scales();
    f16v th[NV], tl[NV], t0[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) th[v] = tl[v] = zero16();
    if constexpr (HALVES)
#pragma unroll
      for (int v = 0; v < NV; ++v) t0[v] = zero16();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int g = 4 * c + j;
      // This wave's loads of stage g are done and its reads of stage g - 1;
      // then everyone's.
      gx_stage_barrier<KIND, NV, LAST>(j);
      const uint8_t* st = lds + slot * NV * GX_STAGE + lo16;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int u = 2 * j + t;
        if constexpr (KIND == Q8_0) {
          const h8 b0 = wt.frag(sc, u, 0, h), b1 = wt.frag(sc, u, 1, h);
          const float d = sc.d(u);
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            h8 a[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const h8*>(st + v * GX_STAGE + (4 * t + i) * 1024);
            f16v x = mfma3216(a[1], b0, zero16());
            x = mfma3216(a[3], b1, x);
            x = mfma3216(a[0], b0, x);
            x = mfma3216(a[2], b1, x);
#pragma unroll
            for (int i = 0; i < 16; ++i) th[v][i] = __builtin_fmaf(x[i], d, th[v][i]);
          }
          // Holds the next pair's LDS reads back: without it the compiler
          // spills 37 registers at NV = 2 in the products and up to 46 in the
          // experts, with it 8 and up to 17.
          __builtin_amdgcn_sched_barrier(0);
        } else {
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            h8 hi[NV], lo[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
              hi[v] = *reinterpret_cast<const h8*>(st + v * GX_STAGE + (4 * t + 2 * b) * 1024);
              lo[v] = *reinterpret_cast<const h8*>(st + v * GX_STAGE + (4 * t + 2 * b + 1) * 1024);
            }
            h8 q, rest;
            if constexpr (KIND == Q6_K) q = wt.frag(sc, u, b, h, rest);
            else q = wt.frag(sc, u, b, h);
#pragma unroll
            for (int v = 0; v < NV; ++v) tl[v] = mfma3216(lo[v], q, tl[v]);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
              f16v& t = HALVES && u < 4 ? t0[v] : th[v];
              t = mfma3216(hi[v], q, t);
            }
            if constexpr (KIND == Q6_K) {
#pragma unroll
              for (int v = 0; v < NV; ++v) tl[v] = mfma3216(hi[v], rest, tl[v]);
            }
          }
        }
      }
      if constexpr (!LAST) wt.load_body(g0, ro, h, j);
      if (!LAST && j == 1) dma_aux(c + 1);
      dma_stage(g + R - 1, fill);
      slot = slot + 1 == R ? 0 : slot + 1;
      fill = fill + 1 == R ? 0 : fill + 1;
    }
    // The column's d, mins and 1 / S.
    const uint8_t* ax = lds + L::AUX0 + (c & 1) * NV * L::AUXB;
    float d = 1.f, dm = 0.f;
    h8 m;
    if constexpr (KIND != Q8_0) d = wt.d() * (KIND == Q6_K ? 65536.f : 16384.f);
    if constexpr (SUMS != 0) dm = wt.dmin() * (-1.f / XSUM_UNIT);
    if constexpr (SUMS == 1) m = sc.mins();
    if constexpr (SUMS == 2) m = sc.mins(h);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const uint8_t* av = ax + v * L::AUXB;
      f4 inv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) inv[q] = *reinterpret_cast<const f4*>(av + 4 * (8 * q + 4 * h));
      f16v tm = zero16();
      if constexpr (SUMS != 0)
#pragma unroll
        for (int f = gx_sum_frags(SUMS) - 1; f >= 0; --f)  // the smallest first
          tm = mfma3216(*reinterpret_cast<const h8*>(av + L::INVB + 1024 * f + lo16), m, tm);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float t = th[v][i];
        if constexpr (KIND != Q8_0) {
          t = SUMS != 0 ? __builtin_fmaf(tl[v][i], d, tm[i] * dm) : tl[v][i] * d;
          t = __builtin_fmaf(th[v][i], d, t);
          if constexpr (HALVES) t = __builtin_fmaf(t0[v][i], d, t);
        }
        acc[v][i] = __builtin_fmaf(t, inv[i >> 2][i & 3], acc[v][i]);
      }
    }
    if ((c & (GX_GROUP - 1)) == GX_GROUP - 1) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        sum[v] += acc[v];
        acc[v] = zero16();
      }
    }
  };
  for (int c = 0; c < s1 - s0 - 1; ++c) column(c, std::false_type{});
  column(s1 - s0 - 1, std::true_type{});
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] += sum[v];
  // No load may reach LDS after the workgroup has ended.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace kq
