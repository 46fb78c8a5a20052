// kq_gx_stages.h -- how far a wave of the many-vector core (kq_gemm.h) runs
// ahead with its loads, and the wait counts that follow from it.  Plain
// constant expressions, so that a host build can check them.
//
// Per stage (64 elements of K, stage g = 4 c + j of column c) a wave issues, in
// this order: the loads of the next column's codes that replace what stage j
// used last (gx_body_loads), then the 2 NV activation fragments of stage g + R -
// 1 of a ring of R.  Head and 1 / S loads come on top and are not counted.
#pragma once
#include "kq_common.h"

namespace kq {

// 64-element stages (8 KB per vector block) in LDS: as many as leave room for
// three workgroups per CU (NV = 1) or two (NV = 2) beside the 1 / S and min
// sums; Q2_K's three fragments of sums take the room of one stage (with six,
// two workgroups fit: Q2_K / Q3_K experts at 64 tokens 138 us against 131 with
// five, Q2_K 14336x4096 x 16 17.7 against 17.4).
__host__ __device__ constexpr int gx_ring(int kind, int nv) { return nv == 1 ? (kind == Q2_K ? 5 : 6) : 4; }

// Code loads behind stage j: one, two for Q8_0, three in every other one for
// Q6_K, one in every other one for Q2_K and Q3_K.
__host__ __device__ constexpr int gx_body_loads(int kind, int j) {
  if (kind == Q8_0) return 2;
  if (kind == Q6_K) return j & 1 ? 3 : 0;
  if (kind == Q2_K || kind == Q3_K) return j & 1;
  return 1;
}

// How many of a wave's newest loads may still be out when stage j of a column
// begins, such that its fragments have arrived: what was issued after them, the
// fragments of the R - 2 stages that follow and the code loads behind the R - 2
// stages before.  Only loads that the compiler cannot drop are counted.  The
// fragments write LDS and always stay.  A code load stays where a column comes
// that uses it, so those issued in the last column itself (no next one) are not
// counted there.
__host__ __device__ constexpr int gx_stage_wait(int kind, int nv, int j, bool last) {
  const int ahead = gx_ring(kind, nv) - 2;
  int n = ahead * 2 * nv;
  for (int i = j - ahead; i < j; ++i)
    if (!last || i < 0) n += gx_body_loads(kind, i & 3);
  return n;
}

}  // namespace kq
