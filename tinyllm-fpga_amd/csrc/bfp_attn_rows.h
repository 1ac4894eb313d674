// Attention pieces for kernels in which a wave's lanes hold 64 positions (the
// scores) or 64 dimensions (the AV chains): the other operand of each product
// -- an element of q, a probability -- is the same for every lane.  It is kept
// 16 values to a register pair, one per lane of each 16-lane row, and read by
// the DPP row broadcast of v_fmac_f64, so it costs no LDS read, no scalar load
// and no lane read per product.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bfp_f64.h"

namespace bfp {

// The 64-vector x (LDS or global) as a wave keeps it: v[b] holds
// x[16 b + lane % 16].
struct RowVec {
  double v[4];
  __device__ __forceinline__ void load(const double *x) {
#pragma unroll
    for (int b = 0; b < 4; ++b) v[b] = x[16 * b + (threadIdx.x & 15)];
  }
};

// a[k] = fma(x[32 + i], y[32 + i], fma(x[i], y[i], 0)) for the eight i = L +
// 4 k (L < 4): the accumulators (r, L) and (r, L + 4), r < 4, of ddot64_skx.
// The s_nop covers the wait states between a write of x and a DPP read.
#define BFP_DOT_STEP(L, D0, D1, D2, D3)                                                                           \
  asm("s_nop 1\n\t"                                                                                               \
      "v_mov_b64 %0, 0\n\tv_mov_b64 %1, 0\n\tv_mov_b64 %2, 0\n\tv_mov_b64 %3, 0\n\t"                              \
      "v_mov_b64 %4, 0\n\tv_mov_b64 %5, 0\n\tv_mov_b64 %6, 0\n\tv_mov_b64 %7, 0\n\t"                              \
      "v_fmac_f64_dpp %0, %8, %12 row_newbcast:" D0 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %1, %8, %13 row_newbcast:" D1 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %2, %8, %14 row_newbcast:" D2 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %3, %8, %15 row_newbcast:" D3 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %4, %9, %16 row_newbcast:" D0 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %5, %9, %17 row_newbcast:" D1 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %6, %9, %18 row_newbcast:" D2 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %7, %9, %19 row_newbcast:" D3 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %0, %10, %20 row_newbcast:" D0 " row_mask:0xf bank_mask:0xf\n\t"                            \
      "v_fmac_f64_dpp %1, %10, %21 row_newbcast:" D1 " row_mask:0xf bank_mask:0xf\n\t"                            \
      "v_fmac_f64_dpp %2, %10, %22 row_newbcast:" D2 " row_mask:0xf bank_mask:0xf\n\t"                            \
      "v_fmac_f64_dpp %3, %10, %23 row_newbcast:" D3 " row_mask:0xf bank_mask:0xf\n\t"                            \
      "v_fmac_f64_dpp %4, %11, %24 row_newbcast:" D0 " row_mask:0xf bank_mask:0xf\n\t"                            \
      "v_fmac_f64_dpp %5, %11, %25 row_newbcast:" D1 " row_mask:0xf bank_mask:0xf\n\t"                            \
      "v_fmac_f64_dpp %6, %11, %26 row_newbcast:" D2 " row_mask:0xf bank_mask:0xf\n\t"                            \
      "v_fmac_f64_dpp %7, %11, %27 row_newbcast:" D3 " row_mask:0xf bank_mask:0xf"                                \
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(a[4]), "=&v"(a[5]), "=&v"(a[6]), "=&v"(a[7])    \
      : "v"(x.v[0]), "v"(x.v[1]), "v"(x.v[2]), "v"(x.v[3]), "v"(y[L]), "v"(y[L + 4]), "v"(y[L + 8]),              \
        "v"(y[L + 12]), "v"(y[L + 16]), "v"(y[L + 20]), "v"(y[L + 24]), "v"(y[L + 28]), "v"(y[L + 32]),           \
        "v"(y[L + 36]), "v"(y[L + 40]), "v"(y[L + 44]), "v"(y[L + 48]), "v"(y[L + 52]), "v"(y[L + 56]),           \
        "v"(y[L + 60]))

// np.dot(x, y) in the SkylakeX ddot order (ddot64_skx) of a wave-uniform x and
// each lane's own y.
__device__ __forceinline__ double ddot64_rows(const RowVec &x, const double (&y)[64]) {
  double s[4], a[8];
  auto fold = [&]() { return (((a[0] + a[1]) + (a[2] + a[3])) + (a[4] + a[5])) + (a[6] + a[7]); };
  BFP_DOT_STEP(0, "0", "4", "8", "12");
  s[0] = fold();
  BFP_DOT_STEP(1, "1", "5", "9", "13");
  s[1] = fold();
  BFP_DOT_STEP(2, "2", "6", "10", "14");
  s[2] = fold();
  BFP_DOT_STEP(3, "3", "7", "11", "15");
  s[3] = fold();
  return (s[0] + s[2]) + (s[1] + s[3]);
}
#undef BFP_DOT_STEP

// A K row of 64 mantissas at km (LDS, 16-byte aligned) with its four tile
// exponents packed in ke4, decoded exactly.
__device__ __forceinline__ void decode_row64(const int16_t *km, int ke4, double (&y)[64]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint4 u = *reinterpret_cast<const uint4 *>(km + 8 * j);
    const double s = ldexp(1.0, (int)(signed char)((ke4 >> (8 * (j >> 1))) & 0xff) - 15);
    const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) y[8 * j + i] = (double)(int)(short)((w[i >> 1] >> (16 * (i & 1))) & 0xffff) * s;
  }
}

// pr[k] = p(k) * v[k] (one rounding; an exact zero comes out +0), p(k) the
// value lane H * 8 + k of each row holds, k < 8.
#define BFP_AV_STEP(P0, P1, P2, P3, P4, P5, P6, P7)                                                               \
  asm("s_nop 1\n\t"                                                                                               \
      "v_mov_b64 %0, 0\n\tv_mov_b64 %1, 0\n\tv_mov_b64 %2, 0\n\tv_mov_b64 %3, 0\n\t"                              \
      "v_mov_b64 %4, 0\n\tv_mov_b64 %5, 0\n\tv_mov_b64 %6, 0\n\tv_mov_b64 %7, 0\n\t"                              \
      "v_fmac_f64_dpp %0, %8, %9 row_newbcast:" P0 " row_mask:0xf bank_mask:0xf\n\t"                              \
      "v_fmac_f64_dpp %1, %8, %10 row_newbcast:" P1 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %2, %8, %11 row_newbcast:" P2 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %3, %8, %12 row_newbcast:" P3 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %4, %8, %13 row_newbcast:" P4 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %5, %8, %14 row_newbcast:" P5 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %6, %8, %15 row_newbcast:" P6 " row_mask:0xf bank_mask:0xf\n\t"                             \
      "v_fmac_f64_dpp %7, %8, %16 row_newbcast:" P7 " row_mask:0xf bank_mask:0xf"                                 \
      : "=&v"(pr[0]), "=&v"(pr[1]), "=&v"(pr[2]), "=&v"(pr[3]), "=&v"(pr[4]), "=&v"(pr[5]), "=&v"(pr[6]),         \
        "=&v"(pr[7])                                                                                              \
      : "v"(p), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]))
template <int H>
__device__ __forceinline__ void av_products(double p, const double (&v)[8], double (&pr)[8]) {
  if constexpr (H == 0) BFP_AV_STEP("0", "1", "2", "3", "4", "5", "6", "7");
  else BFP_AV_STEP("8", "9", "10", "11", "12", "13", "14", "15");
}
#undef BFP_AV_STEP

// V rows decoded to float64 in LDS for the chains: blocks of ROWS_VB rows of 64
// values, two buffers.  Four waves produce a block: lane (row l / 8 of the
// wave's 8, 16-byte part l % 8), with the loads of the next ROWS_DEPTH blocks
// in flight (a block's chain is about 500 to 1200 cycles, less than one
// load's latency).
constexpr int ROWS_VB = 32;
constexpr int ROWS_DEPTH = 4;
struct VRing {
  uint4 m[ROWS_DEPTH];
  int e[ROWS_DEPTH];
};

// acc[i] += sum of p_i[t] V[t] for the rows t0 .. t0 + ROWS_VB - 1 in order
// (attn = sum_t p[t] * V[t], full.py:280-281), one dimension a lane: p_i[t]
// from LDS rows p[i] (0 from n[i] on: the products of those rows are +-0 and
// leave acc unchanged -- it starts at +0.0 and is never -0).
template <int NC>
__device__ __forceinline__ void av_block(const double *vb, const double *const (&p)[3], const int (&n)[3], int t0,
                                         double (&acc)[3]) {
  const int l = threadIdx.x & 63, l16 = l & 15;
  double pv[ROWS_VB / 16][NC], v[2][8];
  auto load = [&](int h) {
#pragma unroll
    for (int u = 0; u < 8; ++u) v[h & 1][u] = vb[(8 * h + u) * 64 + l];
  };
  load(0);
#pragma unroll
  for (int h = 0; h < ROWS_VB / 16; ++h)
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int t = t0 + 16 * h + l16;
      const double x = p[i][t < n[i] ? t : n[i] - 1];   // n[i] >= 1; no read in a branch
      pv[h][i] = t < n[i] ? x : 0.0;
    }
  // groups of 8 rows, the next group's reads in flight; the pairs' adds side
  // by side (each chain waits only on itself)
#pragma unroll
  for (int h = 0; h < ROWS_VB / 8; ++h) {
    if (h + 1 < ROWS_VB / 8) load(h + 1);
    double pr[NC][8];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      if (h & 1) av_products<1>(pv[h >> 1][i], v[h & 1], pr[i]);
      else av_products<0>(pv[h >> 1][i], v[h & 1], pr[i]);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int i = 0; i < NC; ++i) acc[i] = acc[i] + pr[i][u];
  }
}

}  // namespace bfp
