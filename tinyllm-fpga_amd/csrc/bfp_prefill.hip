// A prompt's positions through the layers as the rows of one batch.
//
// The token loop (rtl/vc707/host/gen_smollm_blockfp_full.py:426-443) feeds
// the prompt one token a step, and the head of those steps is not used
// before the last.  Within a layer the positions depend on one another only
// through the KV cache rows 0 .. p, which a pass writes for all its
// positions before any of them attends, so every position of a prompt can
// go through a layer together: the weights are read once for all of them,
// and a layer costs one chain of launches instead of one per position.
// Each row's arithmetic -- the engine's matvecs, the RMSNorm sums, the
// SkylakeX ddot scores, numpy's softmax sum, the ascending-t AV chain -- is
// the decode kernels', so the cache rows and outputs are bit-identical to
// the step-by-step loop's.  A 1000-token prompt and 24 tokens at SmolLM2's
// width and batch 1 take 36 ms so, of which the pass is 12, against 828 step by
// step; a layer of the 1000-row pass is 405 us: 151 of attention, 232 of
// matvecs.
#include <stdint.h>

#include <algorithm>

#include "bfp.h"
#include "bfp_device.h"
#include "bfp_f64.h"
#include "bfp_internal.h"
#include "bfp_prefill.h"

#include "bfp_attn_rows.h"
#include "bfp_layer_dev.h"

namespace bfp {

// ------------------------------------------------------------------- embed
// Row r's token embedding, quantised (full.py:411-412).
__global__ __launch_bounds__(256) void k_pf_embed(PrefillArgs a) {
  const int r = blockIdx.x, b = r / a.n, D = a.L.D;
  int tok = a.prompt[(long long)b * a.n_prompt + a.p0 + (r - b * a.n)];
  tok = tok < 0 ? 0 : (tok >= a.VOCAB ? a.VOCAB - 1 : tok);
  const float *row = a.embed + (long long)tok * D;
  for (int base = 0; base < D; base += blockDim.x) {
    const int i = base + threadIdx.x;
    const bool ok = i < D;
    int e;
    const int m = quantize16_lanes(ok ? (double)row[i] : 0.0, e);
    if (ok) {
      a.L.h_m[(long long)r * D + i] = (int16_t)m;
      if ((i & 15) == 0) a.L.h_e[(long long)r * (D / 16) + (i >> 4)] = (int8_t)e;
    }
  }
}

// -------------------------------------------------------------------- rope
// One 64-wide head of one row per wave: q heads rotated into qf (float64),
// k heads rotated into the cache, v heads copied into it (full.py:268-272).
constexpr int PF_ROPE_WAVES = 4;
__global__ __launch_bounds__(64 * PF_ROPE_WAVES) void k_pf_rope(PrefillArgs a) {
  const LayerArgs &L = a.L;
  const int nh = L.H_Q + 2 * L.H_KV, l = threadIdx.x & 63;
  const int job = blockIdx.x * PF_ROPE_WAVES + (threadIdx.x >> 6);
  const int rows = a.batch * a.n;
  const bool live = job < rows * nh;   // whole waves
  const int jc = live ? job : 0;
  const int r = jc / nh, hd = jc - r * nh;
  const int b = r / a.n, pos = a.p0 + (r - b * a.n);
  const int nq = L.D + 2 * L.KV, i = hd * 64 + l;
  int m = L.qkv_m[(long long)r * nq + i], e = L.qkv_e[(long long)r * (nq / 16) + (i >> 4)];
  if (hd < L.H_Q + L.H_KV) {   // q or k: rotate
    const double *cs = L.rope + (long long)pos * 64 + 2 * (l & 31);
    m = rope_lane(bfp_val(m, e), cs[0], cs[1], e);
  }
  if (!live) return;
  if (hd < L.H_Q) {
    a.qf[(long long)r * L.D + i] = bfp_val(m, e);
    return;
  }
  const bool isk = hd < L.H_Q + L.H_KV;
  const int g = hd - L.H_Q - (isk ? 0 : L.H_KV);
  const long long o = (((long long)b * L.max_ctx + pos) * L.H_KV + g) * 64 + l;
  (isk ? L.k_m : L.v_m)[o] = (int16_t)m;
  if ((l & 15) == 0) (isk ? L.k_e : L.v_e)[o >> 4] = (int8_t)e;
}

// --------------------------------------------------------------- attention
// A workgroup takes QT consecutive positions of one sequence and GH query
// heads of one KV group: NP = QT * GH (position, head) pairs over the same K
// and V rows.
//   scores   a block of 256 K rows goes through LDS (coalesced 16-byte
//            loads; the next block's are issued before the scores, but the
//            compiler keeps them in scratch memory, so they are waited for
//            there); lane t of a wave decodes K
//            row t once and forms that row's SkylakeX ddot with half of the
//            pairs' q (ddot64_rows);
//   softmax  one wave per pair, the whole row of scores in LDS, numpy's
//            pairwise sum on the wave (pairwise_sum_wave);
//   AV       V blocks of 32 rows decoded to float64 in LDS (two buffers) by
//            waves 4-7; waves 0-3 run the chains, one dimension a lane, NP / 4
//            pairs each (av_block).
// The LDS holds NP rows of scores, so NP is chosen by the longest context of
// the pass (pf_attn_shape).  What bounds it at long contexts is the vector
// unit: per pair and position two float64 products with their zeroed
// accumulators and the adds of ddot64_rows on a 64-lane wave, and three
// instructions of the chain.  1000 positions at SmolLM2's width: 153 us a layer
// (223 with q by scalar loads, p by lane reads and one V block in flight), of
// which the chains take 57, the scores 40 and the softmax 26; 64 sequences of
// 8: 30 (46), 5 of 23: 16 (27).
constexpr int PF_KB = 256;             // K rows per staged block
constexpr int PF_KS = 72;              // K row stride in LDS (int16), bank-spread
constexpr int PF_NP = 12;              // most pairs of a workgroup
constexpr int PF_SC_BYTES = 98304;     // most LDS for the scores
constexpr int PF_T = 512;
constexpr int PF_WORK = PF_KB * (PF_KS * 2 + 4) > 2 * ROWS_VB * 64 * 8 ? PF_KB * (PF_KS * 2 + 4) : 2 * ROWS_VB * 64 * 8;

struct PfAttnShape {
  int gh, ngh, qt, scl;   // heads a workgroup, workgroups a KV group, positions, score row length
  size_t lds;
};
inline PfAttnShape pf_attn_shape(int H_Q, int H_KV, int n, int ctx) {
  PfAttnShape s;
  const int grp = H_Q / H_KV;
  s.ngh = (grp + 2) / 3;                   // at most 3 heads a workgroup
  s.gh = (grp + s.ngh - 1) / s.ngh;
  s.scl = (ctx + 1) & ~1;
  const int np = std::min(PF_NP, std::max(s.gh, PF_SC_BYTES / (s.scl * 8)));
  s.qt = std::max(1, std::min(np / s.gh, n));
  s.lds = (size_t)s.qt * s.gh * s.scl * 8 + PF_WORK + 8 * PW_MAX_LEAVES * 8;
  return s;
}

// numpy's add-reduce of a[0..n) (1 <= n <= 4096, LDS) by one wave:
// pairwise_sum_block_g's leaves, 8 at a time, combined by pw_combine_wave.
__device__ __forceinline__ double pairwise_sum_wave(const double *a, int n, double *leaf) {
  const int l = threadIdx.x & 63, j = l & 7;
  const int ng = (n + 63) >> 6;
  for (int base = 0; base < ng; base += 8) {   // uniform
    const int gq = base + (l >> 3);
    const int e = min(gq * 64 + 63, n - 1);
    int flo = 0, fn = n;
    while (fn > 128) {
      int n2 = fn / 2;
      n2 -= n2 % 8;
      if (e < flo + n2) {
        fn = n2;
      } else {
        flo += n2;
        fn -= n2;
      }
    }
    const bool own = gq < ng && flo >= gq * 64;
    const int top = fn - fn % 8, end = flo + top;
    double x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int idx = flo + j + 8 * i;
      x[i] = a[own && idx < end ? idx : 0];
    }
    double r = x[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) r = flo + j + 8 * i < end ? r + x[i] : r;
    r = r + peer<1>(r);
    r = r + peer<2>(r);
    r = r + peer<4>(r);
    if (own && j == 7) {
      double res = r;
      if (fn < 8) {
        res = 0.0;
        for (int i = 0; i < fn; ++i) res += a[flo + i];
      } else {
        for (int i = top; i < fn; ++i) res += a[flo + i];
      }
      leaf[gq] = res;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  return 0.0 + pw_combine_wave(n, leaf);
}

__global__ __launch_bounds__(PF_T, 2) void k_pf_attn(PrefillArgs a, int gh, int ngh, int qt, int scl) {
  extern __shared__ double dsm[];
  const LayerArgs &L = a.L;
  const int np = qt * gh;
  double *sc = dsm;                                         // np x scl
  double *work = sc + np * scl;                             // K stage / V blocks
  double *leaf = work + PF_WORK / 8;                        // 8 x PW_MAX_LEAVES
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int grp = L.H_Q / L.H_KV;
  // blockIdx.x: (KV group, head part); y: position tiles, the longest first; z: sequence
  const int g = blockIdx.x / ngh, h0 = (blockIdx.x - g * ngh) * gh;
  const int nh = min(gh, grp - h0);                         // heads of this workgroup
  const int q0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * qt;
  const int nqt = min(qt, a.n - q0);                        // positions of this workgroup
  const int b = blockIdx.z, row0 = b * a.n + q0, pos0 = a.p0 + q0;
  const int nk = pos0 + nqt;                                // keys of the last position
  const int npl = nqt * nh;                                 // live pairs: pair i = (i / nh, i % nh)
  const long long kv_tok = (long long)L.H_KV * 64;
  const int16_t *Km = L.k_m + (long long)b * L.max_ctx * kv_tok + g * 64;
  const int8_t *Ke = L.k_e + (long long)b * L.max_ctx * (kv_tok / 16) + g * 4;
  const int16_t *Vm = L.v_m + (long long)b * L.max_ctx * kv_tok + g * 64;
  const int8_t *Ve = L.v_e + (long long)b * L.max_ctx * (kv_tok / 16) + g * 4;
  const double *qb = a.qf + (long long)row0 * L.D + (g * grp + h0) * 64;

  // scores[t] = float(np.dot(q, K[t])) / sqrt(HD)   (full.py:277-278)
  int16_t *kst = reinterpret_cast<int16_t *>(work);
  int8_t *kex = reinterpret_cast<int8_t *>(kst + PF_KB * PF_KS);
  constexpr int KL = PF_KB * 8 / PF_T;
  uint4 kr[KL];
  int ke;
  auto load_k = [&](int k0) {
#pragma unroll
    for (int j = 0; j < KL; ++j) {
      int t = k0 + (tid >> 3) + (PF_T / 8) * j;
      t = t < nk ? t : nk - 1;
      kr[j] = *reinterpret_cast<const uint4 *>(Km + t * kv_tok + 8 * (tid & 7));
    }
    const int te = min(k0 + (tid & (PF_KB - 1)), nk - 1);
    ke = *reinterpret_cast<const int *>(Ke + te * (kv_tok / 16));
  };
  auto q_ptr = [&](int i) {   // pair i's q
    const int qi = i / nh;
    return qb + (long long)qi * L.D + (i - qi * nh) * 64;
  };
  load_k(0);
  for (int k0 = 0; k0 < nk; k0 += PF_KB) {   // uniform
    if (k0) lds_barrier();   // the block before is read
#pragma unroll
    for (int j = 0; j < KL; ++j)
      *reinterpret_cast<uint4 *>(kst + ((tid >> 3) + (PF_T / 8) * j) * PF_KS + 8 * (tid & 7)) = kr[j];
    if (tid < PF_KB) *reinterpret_cast<int *>(kex + 4 * tid) = ke;
    load_k(k0 + PF_KB);      // past the end: the last row again
    lds_barrier();
    const int tl = 64 * (w & 3) + l, t = k0 + tl;
    const int i0 = w >> 2;
    if (k0 + 64 * (w & 3) < nk && i0 < npl) {   // uniform per wave
      RowVec q;
      q.load(q_ptr(i0));
      double y[64];
      decode_row64(kst + tl * PF_KS, *reinterpret_cast<const int *>(kex + 4 * tl), y);
      for (int i = i0; i < npl; i += 2) {
        const RowVec qc = q;
        q.load(q_ptr(i + 2 < npl ? i + 2 : i));   // in flight during this pair's products
        const double s = ddot64_rows(qc, y) * L.score_mul;
        if (t <= pos0 + i / nh) sc[i * scl + t] = s;
      }
    }
  }
  lds_barrier();

  // softmax_fp (full.py:245-247), one wave a pair
  for (int i = w; i < npl; i += 8) {
    double *sh = sc + i * scl;
    const int n = pos0 + i / nh + 1;
    double mx = -INFINITY;
    for (int t = l; t < n; t += 64) mx = fmax(mx, sh[t]);
    mx = fmax(mx, peer<32>(mx));
    mx = fmax(mx, peer<16>(mx));
    mx = fmax(mx, peer<8>(mx));
    mx = fmax(mx, peer<4>(mx));
    mx = fmax(mx, peer<2>(mx));
    mx = fmax(mx, peer<1>(mx));
    for (int t = l; t < n; t += 64) sh[t] = exp_f64(sh[t] - mx);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    const double sum = pairwise_sum_wave(sh, n, leaf + w * PW_MAX_LEAVES);
    for (int t = l; t < n; t += 64) sh[t] = sh[t] / sum;
  }
  lds_barrier();

  // attn = sum_t p[t] * V[t], ascending t from 0.0 (full.py:280-281)
  const int nvb = (nk + ROWS_VB - 1) / ROWS_VB;
  if (w >= 4) {
    // producers: block k's 32 rows, wave part w - 4 of 8 rows
    VRing R;
    auto load_v = [&](int k, uint4 &m, int &e) {
      const int t = min(k * ROWS_VB + 8 * (w - 4) + (l >> 3), nk - 1), q = l & 7;
      m = *reinterpret_cast<const uint4 *>(Vm + t * kv_tok + 8 * q);
      e = Ve[t * (kv_tok / 16) + (q >> 1)];
    };
#pragma unroll
    for (int d = 0; d < ROWS_DEPTH; ++d) load_v(d, R.m[d], R.e[d]);
    for (int k0 = 0; k0 < nvb; k0 += ROWS_DEPTH) {   // uniform
#pragma unroll
      for (int d = 0; d < ROWS_DEPTH; ++d) {
        const int k = k0 + d;
        if (k < nvb) {
          const uint4 u = R.m[d];
          const double s = ldexp(1.0, R.e[d] - 15);
          const unsigned wd[4] = {u.x, u.y, u.z, u.w};
          double2 *o = reinterpret_cast<double2 *>(work + (k & 1) * (ROWS_VB * 64) + (8 * (w - 4) + (l >> 3)) * 64 + 8 * (l & 7));
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
  // wave w < 4 holds pairs w, w + 4, w + 8
  double acc[3] = {0.0, 0.0, 0.0};
  const double *pp[3];
  int pn[3];
  int nc = 0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int pi = w + 4 * i;
    const bool on = pi < npl;
    pp[i] = sc + (on ? pi : 0) * scl;
    pn[i] = on ? pos0 + pi / nh + 1 : 0;
    nc += on ? 1 : 0;
  }
  for (int k = 0; k < nvb; ++k) {
    lds_barrier();   // block k is in place
    const double *vb = work + (k & 1) * (ROWS_VB * 64);
    if (nc == 3) av_block<3>(vb, pp, pn, k * ROWS_VB, acc);
    else if (nc == 2) av_block<2>(vb, pp, pn, k * ROWS_VB, acc);
    else if (nc == 1) av_block<1>(vb, pp, pn, k * ROWS_VB, acc);
  }
  {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int pi = w + 4 * i;
      if (pi >= npl) break;   // uniform
      const int qi = pi / nh, hi = pi - qi * nh;
      int e;
      const int m = quantize16_lanes(acc[i], e, true);   // tile_quantize(fp_quantize_vec(attn))
      const long long o = (long long)(row0 + qi) * L.D + (g * grp + h0 + hi) * 64 + l;
      L.att_m[o] = (int16_t)m;
      if ((l & 15) == 0) L.att_e[o >> 4] = (int8_t)e;
    }
  }
}

// ----------------------------------------------------------------- history
// The layer's output rows in canonical form into the history (epi_dres').
__global__ __launch_bounds__(256) void k_pf_hist(PrefillArgs a) {
  const int r = blockIdx.x, b = r / a.n, pos = a.p0 + (r - b * a.n), D = a.L.D;
  const long long o = (((long long)b * a.hist_steps + pos) * a.L.NL + a.L.layer) * D;
  for (int base = 0; base < D; base += blockDim.x) {
    const int i = base + threadIdx.x, ic = i < D ? i : 0;
    int m = a.L.h_m[(long long)r * D + ic], e = a.L.h_e[(long long)r * (D / 16) + (ic >> 4)];
    canon16_lanes(m, e);
    if (i < D) {
      a.hist_m[o + i] = (int16_t)m;
      if ((i & 15) == 0) a.hist_e[(o + i) >> 4] = (int8_t)e;
    }
  }
}

// --------------------------------------------------------------- launchers
int prepare_prefill_kernels() {
  return raise_lds_limit(reinterpret_cast<const void *>(k_pf_attn), PF_SC_BYTES + PF_WORK + 8 * PW_MAX_LEAVES * 8);
}

int launch_prefill_embed(const PrefillArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(k_pf_embed, dim3(a.batch * a.n), dim3(256), 0, s, a);
  return launch_status("prefill embed");
}

int launch_prefill_layer(const PrefillArgs &a, hipStream_t s) {
  const LayerArgs &L = a.L;
  const int rows = a.batch * a.n, nh = L.H_Q + 2 * L.H_KV;
  if (L.batch != rows || rows < 1 || rows > PF_ROWS || a.p0 + a.n > L.max_ctx)
    return set_err(BFP_EINVAL, "prefill: %d rows, positions [%d, %d)", rows, a.p0, a.p0 + a.n);
  BFP_TRY(launch_rows_qkv(L, s));
  hipLaunchKernelGGL(k_pf_rope, dim3((rows * nh + PF_ROPE_WAVES - 1) / PF_ROPE_WAVES), dim3(64 * PF_ROPE_WAVES), 0, s, a);
  const PfAttnShape sh = pf_attn_shape(L.H_Q, L.H_KV, a.n, a.p0 + a.n);
  if (sh.qt * sh.gh > PF_NP) return set_err(BFP_EINVAL, "prefill: %d x %d pairs", sh.qt, sh.gh);
  hipLaunchKernelGGL(k_pf_attn, dim3(L.H_KV * sh.ngh, (a.n + sh.qt - 1) / sh.qt, a.batch), dim3(PF_T), sh.lds, s, a,
                     sh.gh, sh.ngh, sh.qt, sh.scl);
  BFP_TRY(launch_rows_post(L, s));
  if (a.hist_m) hipLaunchKernelGGL(k_pf_hist, dim3(rows), dim3(256), 0, s, a);
  return launch_status("prefill layer");
}

}  // namespace bfp
