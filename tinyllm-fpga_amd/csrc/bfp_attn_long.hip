// The attention of one query head of one sequence in one workgroup, for KV
// capacities past the short forms' 512 positions
// (rtl/vc707/host/gen_smollm_blockfp_full.py:268-283).  The arithmetic is
// attn_body's -- the SkylakeX ddot order of the scores, numpy's softmax and
// pairwise sum, the ascending-t AV chain -- so the outputs are bit-identical
// to its long form's (k_attn<8, false>), which gives a head to four
// workgroups that each form every score and a quarter of the dimensions.
//   K    blocks of 512 rows through LDS (coalesced 16-byte loads); each wave
//        scores 64 of them, a decoded row a lane against the head's q
//        (ddot64_rows).  The next block's loads are issued before the scores,
//        but the compiler keeps them in scratch memory (the choice between
//        them and the current row is one of addresses, and so generic loads
//        one after another), so a block waits for them before its scores;
//   V    blocks of 32 rows decoded to float64 in LDS by waves 4-7, the loads
//        of four blocks in flight; wave 0 runs the 64 chains (av_block).
// A workgroup is a chain of dependent steps: about a third of it wave 0's
// 1500 products and adds at position 1500 (some 29 cycles a position: wave 0
// forms the products too, waves 1-3 are idle), the rest the K blocks' loads
// and scores and the softmax.  16 sequences at position 1500 (9 heads): 55.4
// us a launch against 69.6.
#include <stdint.h>

#include <algorithm>

#include "bfp.h"
#include "bfp_attn_rows.h"
#include "bfp_device.h"
#include "bfp_f64.h"
#include "bfp_internal.h"
#include "bfp_layer.h"

#include "bfp_layer_dev.h"

namespace bfp {

constexpr int AL_T = 512;
constexpr int AL_KS = 72;   // K row stride in LDS (int16), bank-spread
constexpr int AL_WORK = AL_T * (AL_KS * 2 + 4);
static_assert(AL_WORK >= 2 * ROWS_VB * 64 * 8, "the V buffers fit the K stage");

inline size_t attn_long_lds(int max_ctx) {
  return (size_t)(64 + PW_MAX_LEAVES + 8 + ((max_ctx + 1) & ~1)) * 8 + AL_WORK + 2 * (128 + 16);
}

__global__ __launch_bounds__(AL_T, 2) void k_attn_long(LayerArgs a) {
  extern __shared__ double dsm[];
  double *q = dsm;                                        // 64
  double *leaf = q + 64;                                  // PW_MAX_LEAVES
  double *red = leaf + PW_MAX_LEAVES;                     // 8
  double *sc = red + 8;                                   // max_ctx, rounded up to even
  double *work = sc + ((a.max_ctx + 1) & ~1);             // K stage / V blocks
  int16_t *kst = reinterpret_cast<int16_t *>(work);
  int8_t *kex = reinterpret_cast<int8_t *>(kst + AL_T * AL_KS);
  int16_t *kc = reinterpret_cast<int16_t *>(kex + 4 * AL_T);   // row pos: k (64), v (64) and their exponents
  int16_t *vc = kc + 64;
  int *kce = reinterpret_cast<int *>(vc + 64), *vce = kce + 4;  // packed in [0]
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int hq = blockIdx.x, b = blockIdx.y, grp = a.H_Q / a.H_KV, g = hq / grp;
  const int pos = cur_kv_pos(a), rpos = cur_pos(a), n = pos + 1;
  const long long kv_tok = (long long)a.H_KV * 64;
  int16_t *Km = a.k_m + (long long)b * a.max_ctx * kv_tok + g * 64;
  int8_t *Ke = a.k_e + (long long)b * a.max_ctx * (kv_tok / 16) + g * 4;
  int16_t *Vm = a.v_m + (long long)b * a.max_ctx * kv_tok + g * 64;
  int8_t *Ve = a.v_e + (long long)b * a.max_ctx * (kv_tok / 16) + g * 4;
  const int nq = a.D + 2 * a.KV, last = pos > 0 ? pos - 1 : 0;   // rows past pos - 1 are never used

  uint4 kr[8];
  int ke;
  auto load_k = [&](int k0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int t = min(k0 + (tid >> 3) + 64 * j, last);
      kr[j] = *reinterpret_cast<const uint4 *>(Km + t * kv_tok + 8 * (tid & 7));
    }
    ke = *reinterpret_cast<const int *>(Ke + min(k0 + tid, last) * (kv_tok / 16));
  };
  load_k(0);
  if (w < 3) {
    // RoPE of q (wave 0) and k (wave 1); v (wave 2) as it is
    const int i = w == 0 ? hq * 64 + l : (w == 1 ? a.D : a.D + a.KV) + g * 64 + l;
    int m = a.qkv_m[b * nq + i], e = a.qkv_e[b * (nq / 16) + (i >> 4)];
    if (w < 2) {
      const double *cs = a.rope_row ? a.rope_row : a.rope + (long long)rpos * 64;
      m = rope_lane(bfp_val(m, e), cs[2 * (l & 31)], cs[2 * (l & 31) + 1], e);
    }
    if (w == 0) {
      q[l] = bfp_val(m, e);
    } else {
      (w == 1 ? kc : vc)[l] = (int16_t)m;
      if ((l & 15) == 0) reinterpret_cast<int8_t *>(w == 1 ? kce : vce)[l >> 4] = (int8_t)e;
      if (hq % grp == 0) {   // one workgroup of the group stores the cache row
        int16_t *cm = (w == 1 ? Km : Vm) + pos * kv_tok;
        int8_t *ce = (w == 1 ? Ke : Ve) + pos * (kv_tok / 16);
        cm[l] = (int16_t)m;
        if ((l & 15) == 0) ce[l >> 4] = (int8_t)e;
      }
    }
  }
  lds_barrier();

  // scores[t] = float(np.dot(q, K[t])) / sqrt(HD)   (full.py:277-278)
  RowVec qv;
  qv.load(q);
  for (int k0 = 0; k0 < n; k0 += AL_T) {   // uniform
    if (k0) lds_barrier();   // the block before is read
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = (tid >> 3) + 64 * j;
      *reinterpret_cast<uint4 *>(kst + r * AL_KS + 8 * (tid & 7)) =
          k0 + r == pos ? *reinterpret_cast<const uint4 *>(kc + 8 * (tid & 7)) : kr[j];
    }
    *reinterpret_cast<int *>(kex + 4 * tid) = k0 + tid == pos ? kce[0] : ke;
    load_k(k0 + AL_T);
    lds_barrier();
    if (k0 + 64 * w < n) {   // uniform per wave
      double y[64];
      decode_row64(kst + tid * AL_KS, *reinterpret_cast<const int *>(kex + 4 * tid), y);
      const double s = ddot64_rows(qv, y) * a.score_mul;
      if (k0 + tid < n) sc[k0 + tid] = s;
    }
  }
  lds_barrier();

  // softmax_fp (full.py:245-247): e = exp(s - max); p = e / pairwise_sum(e)
  double mx = -INFINITY;
  for (int t = tid; t < n; t += AL_T) mx = fmax(mx, sc[t]);
  mx = fmax(mx, peer<32>(mx));
  mx = fmax(mx, peer<16>(mx));
  mx = fmax(mx, peer<8>(mx));
  mx = fmax(mx, peer<4>(mx));
  mx = fmax(mx, peer<2>(mx));
  mx = fmax(mx, peer<1>(mx));
  if (l == 0) red[w] = mx;
  lds_barrier();
  mx = red[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) mx = fmax(mx, red[i]);
  for (int t = tid; t < n; t += AL_T) sc[t] = exp_f64(sc[t] - mx);
  lds_barrier();
  const double sum = pairwise_sum_block(sc, n, leaf);
  for (int t = tid; t < n; t += AL_T) sc[t] = sc[t] / sum;
  lds_barrier();

  // attn = sum_t p[t] * V[t], ascending t from 0.0 (full.py:280-281)
  const int nvb = (n + ROWS_VB - 1) / ROWS_VB;
  if (w >= 4) {
    VRing R;
    auto load_v = [&](int k, uint4 &m, int &e) {
      const int t = min(k * ROWS_VB + 8 * (w - 4) + (l >> 3), last), p = l & 7;
      m = *reinterpret_cast<const uint4 *>(Vm + t * kv_tok + 8 * p);
      e = Ve[t * (kv_tok / 16) + (p >> 1)];
    };
    const uint4 vcp = *reinterpret_cast<const uint4 *>(vc + 8 * (l & 7));
    const int vcx = reinterpret_cast<const int8_t *>(vce)[(l & 7) >> 1];
#pragma unroll
    for (int d = 0; d < ROWS_DEPTH; ++d) load_v(d, R.m[d], R.e[d]);
    for (int k0 = 0; k0 < nvb; k0 += ROWS_DEPTH) {   // uniform
#pragma unroll
      for (int d = 0; d < ROWS_DEPTH; ++d) {
        const int k = k0 + d, r = 8 * (w - 4) + (l >> 3);
        if (k < nvb) {
          const bool cur = k * ROWS_VB + r == pos;
          const uint4 u = cur ? vcp : R.m[d];
          const double s = ldexp(1.0, (cur ? vcx : R.e[d]) - 15);
          const unsigned wd[4] = {u.x, u.y, u.z, u.w};
          double2 *o = reinterpret_cast<double2 *>(work + (k & 1) * (ROWS_VB * 64) + r * 64 + 8 * (l & 7));
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[i] = make_double2((double)(int)(short)(wd[i] & 0xffff) * s, (double)((int)wd[i] >> 16) * s);
        }
        load_v(k + ROWS_DEPTH, R.m[d], R.e[d]);
        if (k < nvb) lds_barrier();   // block k is in place, block k - 1 used
      }
    }
    return;
  }
  double acc[3] = {0.0, 0.0, 0.0};
  const double *pp[3] = {sc, sc, sc};
  const int pn[3] = {n, n, n};
  for (int k = 0; k < nvb; ++k) {
    lds_barrier();   // block k is in place
    if (w == 0) av_block<1>(work + (k & 1) * (ROWS_VB * 64), pp, pn, k * ROWS_VB, acc);
  }
  if (w == 0) {
    int e;
    const int m = quantize16_lanes(acc[0], e, true);   // tile_quantize(fp_quantize_vec(attn))
    const long long o = (long long)b * a.D + hq * 64 + l;
    a.att_m[o] = (int16_t)m;
    if ((l & 15) == 0) a.att_e[o >> 4] = (int8_t)e;
  }
}

int prepare_attn_long(int max_ctx) {
  return raise_lds_limit(reinterpret_cast<const void *>(k_attn_long), (int)attn_long_lds(max_ctx));
}

int launch_attn_long(const LayerArgs &a, hipStream_t s) {
  if (a.dump || a.HD != 64) return set_err(BFP_EINVAL, "attn_long: a stage dump or HD %d", a.HD);
  hipLaunchKernelGGL(k_attn_long, dim3(a.H_Q, a.batch), dim3(AL_T), attn_long_lds(a.max_ctx), s, a);
  return launch_status("attn");
}

}  // namespace bfp
