// RTL-exact BFP leaf ops (the hardware engines of rtl/vc707/src/smollm/), as
// batched HIP kernels.  Each kernel follows the reference's bit-exact Python
// golden of that engine (rtl/vc707/host/gen_*_bfp_golden.py): truncating
// arithmetic shifts, per-lane / per-element exponents, the engines' own
// sequential fold orders, LUT exp / SiLU and Newton-Raphson reciprocals.
// These ops are not on the model-level simulator's token path; they are the
// per-op semantics of the FPGA datapath.
#include <math.h>
#include <stdint.h>

#include <mutex>

#include "bfp.h"
#include "bfp_device.h"
#include "bfp_internal.h"
#include "bfp_f64.h"
#include "bfp_layer.h"
#include "bfp_mv.h"

namespace bfp {
namespace rtl {

constexpr int ACC_W = 48;

__device__ __forceinline__ int lead64(long long v) {
  if (v == 0) return 0;
  unsigned long long a = v < 0 ? (unsigned long long)(-v) : (unsigned long long)v;
  return 63 - __clzll(a);
}

// shift = lead - 14; mantissa = low 16 bits of v >> shift (or << -shift)
__device__ __forceinline__ int norm16(long long v, int lead, int &shift) {
  shift = lead - 14;
  long long s = shift >= 0 ? (v >> shift) : v * (1LL << (-shift));
  return (int)(short)(s & 0xFFFF);
}

__device__ __forceinline__ int clamp8(int e) { return e < -128 ? -128 : (e > 127 ? 127 : e); }

__device__ __forceinline__ int max16_lanes(int v) {
  v = pmax<8>(v);
  v = pmax<4>(v);
  v = pmax<2>(v);
  return pmax<1>(v);
}

// ------------------------------------------------------------------ matvec
// gen_matvec_bfp_golden.py:53-108: one thread per output row.
__global__ void k_rtl_matvec(const int16_t *__restrict__ xm, const int8_t *__restrict__ xe,
                             const int16_t *__restrict__ Wm, const int8_t *__restrict__ We,
                             int n_out, int nt, int16_t *ym, int8_t *ye) {
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= n_out) return;
  const long long HI = (1LL << (ACC_W - 1)) - 1, LO = -(1LL << (ACC_W - 1));
  long long acc = 0;
  int acc_e = 0;
  for (int t = 0; t < nt; ++t) {
    long long s = 0;
    const int16_t *w = Wm + ((long long)row * nt + t) * 16;
    for (int k = 0; k < 16; ++k) s += (long long)xm[t * 16 + k] * w[k];
    const int te = (int)xe[t] + (int)We[(long long)row * nt + t];
    if (t == 0) {
      acc = s;
      acc_e = te;
      continue;
    }
    const int d = te - acc_e;
    if (d > 0) {
      acc = d > ACC_W - 1 ? 0 : (acc >> d);
      acc_e = te;
    } else if (d < 0) {
      s = -d > ACC_W - 1 ? 0 : (s >> (-d));
    }
    acc += s;
    acc = acc > HI ? HI : (acc < LO ? LO : acc);
  }
  int sh;
  ym[row] = (int16_t)norm16(acc, lead64(acc), sh);
  ye[row] = (int8_t)clamp8(acc_e + sh - 15);
}

// requant_mant (smollm_layer_bfp.sv:1387-1396): the shift e_to - e_from is
// held in `logic signed [7:0]` and wraps; >= 16 gives 0, a negative shift
// leaves m unchanged.  The AV pre-shift of V (:2149-2166) has the same form.
__device__ __forceinline__ int shr8(int m, int e_to, int e_from) {
  const int sh = (int)(signed char)(e_to - e_from);
  return sh >= 16 ? 0 : (sh >= 0 ? (m >> sh) : m);
}

// ----------------------------------------------------------------- requant
// smollm_layer_bfp.sv:1387-1396 (requant_mant) with the chunk emax of
// :1672-1693: 16 lanes per chunk, one thread per lane.
__global__ void k_rtl_requant(const int16_t *__restrict__ m, const int8_t *__restrict__ e, int n,
                              int16_t *om, int8_t *oe) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool ok = i < n;
  const int ei = ok ? (int)e[i] : -128;
  const int emax = max16_lanes(ei);
  if (!ok) return;
  om[i] = (int16_t)shr8(m[i], emax, ei);
  if ((i & 15) == 0) oe[i >> 4] = (int8_t)emax;
}

// ----------------------------------------------------------------- rmsnorm
__constant__ int c_rms_seed[32] = {
    16777215, 16777215, 16777215, 16777215, 16777215, 16777215, 13698540, 9686330,
    6849270, 4843165, 3424635, 2421583, 1712317, 1210791, 856159, 605396,
    428079, 302698, 214040, 151349, 107020, 75674, 53510, 37837,
    26755, 18919, 13377, 9459, 6689, 4730, 3344, 2365};

// One step of the engine's ordered fold over tiles (gen_matvec_bfp_golden.py
// :53-108): the side with the smaller exponent is shifted right (zeroed past
// 47), then added.  The engine's 48-bit saturation cannot be reached: a tile
// sum is at most 2^34, so fewer than 2^13 of them stay below 2^47 (the
// callers have at most 4096 tiles).  acc_e is the running maximum of the
// exponents whatever the sums are, so the shift amounts do not wait for acc
// and only a shift and an add chain from step to step.
__device__ __forceinline__ void tile_fold(long long &acc, int &acc_e, long long s, int te) {
  const int d = te - acc_e;
  const int up = d > 0 ? d : 0, dn = d < 0 ? -d : 0;
  const long long s2 = dn > ACC_W - 1 ? 0 : (s >> dn);
  acc = (up > ACC_W - 1 ? 0 : (acc >> up)) + s2;
  acc_e = d > 0 ? te : acc_e;
}

// The same fold over nt <= 64 tiles (LDS) by a wave, tile t in lane t: the
// running maximum of the exponents is a scan, each sum's shift follows from
// it, and the sums between two rises of the maximum add in any order; acc is
// shifted once a rise (a few for 36 tiles).  Every lane returns the result.
__device__ __forceinline__ void fold_wave(const long long *S, const int *E, int nt, long long &acc, int &acc_e) {
  const int l = threadIdx.x & 63, lc = l < nt ? l : nt - 1;
  constexpr int NONE = -100000;
  const int e = l < nt ? E[lc] : NONE;
  const long long sv = S[lc];
  int p = e;
  auto scan = [&](int o) { p = o > p ? o : p; };
  scan(__builtin_amdgcn_update_dpp(NONE, p, 0x111, 0xf, 0xf, false));   // row_shr 1, 2, 4, 8
  scan(__builtin_amdgcn_update_dpp(NONE, p, 0x112, 0xf, 0xf, false));
  scan(__builtin_amdgcn_update_dpp(NONE, p, 0x114, 0xf, 0xf, false));
  scan(__builtin_amdgcn_update_dpp(NONE, p, 0x118, 0xf, 0xf, false));
  // the rows' maxima into the rows after them
  const int r0 = __builtin_amdgcn_readlane(p, 15), r1 = __builtin_amdgcn_readlane(p, 31);
  const int r2 = __builtin_amdgcn_readlane(p, 47);
  const int r01 = r0 > r1 ? r0 : r1, r012 = r01 > r2 ? r01 : r2;
  scan(l < 16 ? NONE : (l < 32 ? r0 : (l < 48 ? r01 : r012)));
  int before = __shfl_up(p, 1, 64);
  before = l == 0 ? e : before;
  const int dn = p - e;
  const long long s = l >= nt || dn > ACC_W - 1 ? 0 : (sv >> dn);
  unsigned long long rises = __ballot(l < nt && e > before);
  acc = 0;
  for (int from = 0;;) {   // uniform
    const int to = rises ? __builtin_ctzll(rises) : 64;
    long long seg = l >= from && l < to ? s : 0;
    seg = psum<8>(seg);
    seg = psum<4>(seg);
    seg = psum<2>(seg);
    seg = psum<1>(seg);
    seg = psum<16>(seg);
    seg = psum<32>(seg);
    acc += seg;
    if (to == 64) break;
    const int up = __builtin_amdgcn_readlane(e, to) - __builtin_amdgcn_readlane(before, to);
    acc = up > ACC_W - 1 ? 0 : (acc >> up);
    rises &= rises - 1;
    from = to;
  }
  acc_e = __builtin_amdgcn_readlane(p, 63);
}

// The RMSNorm engine on the D-vector (x, xex) by a whole workgroup (any
// multiple of 64 threads): gamma(i, m, e) gives gamma element i (called by
// whole waves, 16-lane groups on one tile), out(i, m, e) takes the result
// (i < D; lanes of a tile together).  sums: D/16 int64 of LDS, sexp: D/16
// ints.  Thread tid keeps its first RMS_KE elements in registers from one
// batch of loads.  Every thread folds the tile sums and runs the
// Newton-Raphson steps itself (the same values in every lane), so one
// barrier is enough.  (As one wave's chain of loads the norm of 576 elements
// was a launch of 17 us; the head's, in this form, takes 6.)
constexpr int RMS_KE = 3;
template <class Gamma, class Out>
__device__ __forceinline__ void rms_block(const int16_t *__restrict__ x, const int8_t *__restrict__ xex, Gamma gamma,
                                          int D, long long *sums, int *sexp, Out out) {
  const int tid = threadIdx.x, bs = blockDim.x, nt = D / 16;
  int xv[RMS_KE], xe[RMS_KE], gm[RMS_KE], ge[RMS_KE];
  auto load = [&](int base) {
#pragma unroll
    for (int k = 0; k < RMS_KE; ++k) {
      const int i = base + tid + k * bs, ic = i < D ? i : D - 1;
      xv[k] = x[ic];
      xe[k] = xex[ic >> 4];
    }
#pragma unroll
    for (int k = 0; k < RMS_KE; ++k) {
      const int i = base + tid + k * bs;
      gamma(i < D ? i : (D - 16) + (i & 15), gm[k], ge[k]);
    }
  };
  for (int base = 0; base < D; base += RMS_KE * bs) {   // uniform
    load(base);
#pragma unroll
    for (int k = 0; k < RMS_KE; ++k) {
      const int i = base + tid + k * bs;
      long long s = (long long)(xv[k] * xv[k]);   // at most 2^30
      s = psum<1>(s);
      s = psum<2>(s);
      s = psum<4>(s);
      s = psum<8>(s);
      if (i < D && (i & 15) == 0) {
        sums[i >> 4] = s;
        sexp[i >> 4] = 2 * xe[k];
      }
    }
  }
  lds_barrier();
  long long acc;
  int acc_e;
  if (nt <= 64) {   // uniform
    fold_wave(sums, sexp, nt, acc, acc_e);
  } else {
    acc = sums[0];
    acc_e = sexp[0];
#pragma unroll 4
    for (int t = 1; t < nt; ++t) tile_fold(acc, acc_e, sums[t], sexp[t]);
  }
  const unsigned long long inv_d = (1ULL << 32) / (unsigned)D;
  // mean = (acc * inv_d) >> 32, acc >= 0
  const unsigned __int128 prod = (unsigned __int128)(unsigned long long)acc * inv_d;
  const unsigned long long mean = (unsigned long long)(prod >> 32);
  int lead = mean ? 63 - __clzll(mean) : 0;
  if ((acc_e + lead) & 1) lead -= 1;
  long long v = lead >= 30 ? (long long)(mean >> (lead - 30)) : (long long)(mean << (30 - lead));
  v += 10737;                                       // EPS_Q30
  const int vmsb = v ? 63 - __clzll((unsigned long long)v) : 0;
  long long inv = vmsb < 32 ? c_rms_seed[vmsb] : 16777215;
  const long long C = (3LL << 30) / 2;
  for (int it = 0; it < 3; ++it) {
    const __int128 vy2 = ((__int128)v * inv * inv) >> 24;
    long long corr;
    if (vy2 >= ((__int128)1 << 32)) {
      corr = 0;
    } else {
      corr = C - ((long long)vy2 >> 1);
      corr = corr < 0 ? 0 : corr;
    }
    const long long ni = (inv * corr + (1LL << 29)) >> 30;
    inv = ni < 16777215 ? ni : 16777215;
  }
  const int einv = (30 - acc_e - lead) >> 1;
  for (int base = 0; base < D; base += RMS_KE * bs) {   // uniform
    if (D > RMS_KE * bs) load(base);
#pragma unroll
    for (int k = 0; k < RMS_KE; ++k) {
      const int i = base + tid + k * bs;
      const long long p = i < D ? (long long)xv[k] * gm[k] * inv : 0;
      const int ml = max16_lanes(p ? lead64(p) : 0);
      int sh;
      const int m = norm16(p, ml, sh);
      out(i, m, clamp8(xe[k] + ge[k] + einv + sh - 27));
    }
  }
}

// gen_rmsnorm_bfp_golden.py:42-142: one workgroup per vector, of just the
// waves its elements fill (up to RMS_T threads): the waves past them would
// only repeat the fold and the Newton-Raphson steps.  20000 vectors of 16 take
// 20 us so, 66 with RMS_T threads for each; 5000 of 64 7.6 against 20, 5000 of
// 576 19.5 against 23.
constexpr int RMS_T = 256;
inline int rms_threads(int D) {
  const int waves = (D + 64 * RMS_KE - 1) / (64 * RMS_KE);
  return waves < RMS_T / 64 ? 64 * waves : RMS_T;
}
__global__ __launch_bounds__(RMS_T) void k_rtl_rmsnorm(const int16_t *__restrict__ xm, const int8_t *__restrict__ xe,
                                                       const int16_t *__restrict__ gm, const int8_t *__restrict__ ge,
                                                       int D, int16_t *__restrict__ ym, int8_t *__restrict__ ye) {
  extern __shared__ long long sums[];   // nt tile sums, nt exponents
  const int b = blockIdx.x, nt = D / 16;
  ym += (long long)b * D;
  ye += (long long)b * nt;
  rms_block(
      xm + (long long)b * D, xe + (long long)b * nt,
      [&](int i, int &m, int &e) {
        m = gm[i];
        e = ge[i >> 4];
      },
      D, sums, reinterpret_cast<int *>(sums + nt),
      [&](int i, int m, int e) {
        if (i >= D) return;
        ym[i] = (int16_t)m;
        if ((i & 15) == 0) ye[i >> 4] = (int8_t)e;
      });
}

// -------------------------------------------------------------------- rope
constexpr long long PI_HALF_Q27 = 210828714, PI_Q27 = 421657428, PI_OVER_8_Q29 = 210828714,
                    K_Q3_27 = 81504109;
__constant__ long long c_atan[16] = {105414357, 62229729, 32880480, 16690645, 8377711, 4192939,
                                     2096981, 1048555, 524285, 262144, 131072, 65536,
                                     32768, 16384, 8192, 4096};

__device__ __forceinline__ long long wrap31(long long v) {
  v &= (1LL << 31) - 1;
  return (v & (1LL << 30)) ? v - (1LL << 31) : v;
}

// 16-iteration Q3.27 CORDIC of cordic_sincos.sv (gen_rope_bfp_golden.py:37-60).
__device__ void cordic(long long a, int &c, int &s) {
  long long z;
  bool neg;
  if (a > PI_HALF_Q27) {
    z = PI_Q27 - a;
    neg = true;
  } else if (a < -PI_HALF_Q27) {
    z = -PI_Q27 - a;
    neg = true;
  } else {
    z = a;
    neg = false;
  }
  long long x = K_Q3_27, y = 0;
  for (int i = 0; i < 16; ++i) {
    const long long xs = x >> i, ys = y >> i;
    if (z >= 0) {
      x -= ys;
      y += xs;
      z -= c_atan[i];
    } else {
      x += ys;
      y -= xs;
      z += c_atan[i];
    }
  }
  const long long xr = (x + 2048) >> 12, yr = (y + 2048) >> 12;
  if (xr > 32767)
    c = neg ? -32767 : 32767;
  else if (xr < -32768)
    c = neg ? 32767 : -32768;
  else
    c = (int)(neg ? -xr : xr);
  s = (int)(yr > 32767 ? 32767 : (yr < -32768 ? -32768 : yr));
}

// rope_bfp.sv golden (gen_rope_bfp_golden.py:72-121): one 64-thread
// workgroup per head, thread j < 32 rotates pair (j, j+32).
__global__ __launch_bounds__(64) void k_rtl_rope(const int16_t *__restrict__ xm,
                                                 const int8_t *__restrict__ xe, int pos,
                                                 const unsigned *__restrict__ freq, int16_t *ym,
                                                 int8_t *ye) {
  const int h = blockIdx.x, j = threadIdx.x;
  if (j >= 32) return;
  const int16_t *x = xm + h * 64;
  const int8_t *e = xe + h * 4;
  const long long ang = wrap31((wrap31((long long)pos * freq[j]) * PI_OVER_8_Q29) >> 29);
  int c, s;
  cordic(ang, c, s);
  const int a = x[j], bb = x[j + 32];
  const int ea = e[j >> 4], eb = e[(j + 32) >> 4];
  const int em = ea > eb ? ea : eb;
  const long long aa = em - ea < 16 ? (a >> (em - ea)) : 0;
  const long long ba = em - eb < 16 ? (bb >> (em - eb)) : 0;
  const long long lo = aa * c - ba * s, hi = ba * c + aa * s;
  int sh;
  ym[h * 64 + j] = (int16_t)norm16(lo, lead64(lo), sh);
  ye[h * 64 + j] = (int8_t)clamp8(em + sh - 15);
  ym[h * 64 + j + 32] = (int16_t)norm16(hi, lead64(hi), sh);
  ye[h * 64 + j + 32] = (int8_t)clamp8(em + sh - 15);
}

// ----------------------------------------------------------------- softmax
// softmax_bfp.sv golden (gen_softmax_bfp_golden.py:33-78): one 64-thread
// workgroup per problem of n <= 4096 scores sharing one exponent.
__global__ __launch_bounds__(64) void k_rtl_softmax(const int16_t *__restrict__ xm,
                                                    const int8_t *__restrict__ xe, int n,
                                                    int stride,
                                                    const uint16_t *__restrict__ lut,
                                                    int16_t *ym, int8_t *ye) {
  extern __shared__ long long vals[];   // n LUT values
  __shared__ long long s_inv;
  __shared__ int s_red[2];
  const int b = blockIdx.x, tid = threadIdx.x;
  const int16_t *x = xm + (long long)b * stride;
  int mx = -32768;
  for (int i = tid; i < n; i += 64) mx = x[i] > mx ? x[i] : mx;
  for (int o = 1; o < 64; o <<= 1) {
    int w = __shfl_xor(mx, o, 64);
    mx = w > mx ? w : mx;
  }
  const int sh = (int)xe[b] - 8;
  long long part = 0;
  for (int i = tid; i < n; i += 64) {
    const long long d = (long long)x[i] - mx;
    const long long ds = sh >= 0 ? d * (1LL << (sh > 40 ? 40 : sh)) : (d >> (-sh > 62 ? 62 : -sh));
    const int idx = ds >= 0 ? 1023 : (ds <= -1023 ? 0 : (int)(ds + 1023));
    vals[i] = lut[idx];
    part += lut[idx];
  }
  for (int o = 1; o < 64; o <<= 1) part += __shfl_xor(part, o, 64);
  if (tid == 0) {
    const long long tot = part;
    const int msb = tot ? 63 - __clzll((unsigned long long)tot) : 0;
    __int128 y = (__int128)1 << (31 - msb);
    for (int it = 0; it < 4; ++it) y = (y * (((__int128)1 << 33) - (__int128)tot * y)) >> 32;
    s_inv = (long long)y;
  }
  __syncthreads();
  const long long inv = s_inv;
  int ml = 0;
  for (int i = tid; i < n; i += 64) {
    const long long p = vals[i] * inv;
    const int l = p ? lead64(p) : 0;
    ml = l > ml ? l : ml;
  }
  for (int o = 1; o < 64; o <<= 1) {
    int w = __shfl_xor(ml, o, 64);
    ml = w > ml ? w : ml;
  }
  for (int i = tid; i < n; i += 64) {
    int s2;
    ym[(long long)b * stride + i] = (int16_t)norm16(vals[i] * inv, ml, s2);
  }
  if (tid == 0) ye[b] = (int8_t)clamp8(ml - 14 - 17);
  (void)s_red;
}

// ------------------------------------------------------------------ swiglu
// swiglu_bfp.sv golden (gen_swiglu_bfp_golden.py:43-78): one element per
// thread, 16-lane tiles.
__global__ void k_rtl_swiglu(const int16_t *__restrict__ gm, const int8_t *__restrict__ ge,
                             const int16_t *__restrict__ um, const int8_t *__restrict__ ue, int n,
                             const int16_t *__restrict__ lut, int16_t *ym, int8_t *ye) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool ok = i < n;
  long long p = 0;
  if (ok) {
    const int sh = (int)ge[i >> 4] - 5;
    const long long mg = gm[i];
    long long idx;
    if (sh >= 0)
      idx = sh >= 16 ? (mg > 0 ? 32767 : (mg < 0 ? -32768 : 0)) : mg * (1LL << sh);
    else
      idx = -sh >= 16 ? (mg < 0 ? -1 : 0) : (mg >> (-sh));
    idx = idx < -32768 ? -32768 : (idx > 32767 ? 32767 : idx);
    p = (long long)lut[idx & 0xFFFF] * um[i];
  }
  const int ml = max16_lanes(p ? lead64(p) : 0);
  if (!ok) return;
  int s;
  ym[i] = (int16_t)norm16(p, ml, s);
  if ((i & 15) == 0) ye[i >> 4] = (int8_t)clamp8((int)ue[i >> 4] + s - 10);
}

// ---------------------------------------------------------------- residual
// residual_bfp.sv golden (gen_residual_bfp_golden.py:23-48).
__global__ void k_rtl_residual(const int16_t *__restrict__ am, const int8_t *__restrict__ ae,
                               const int16_t *__restrict__ bm, const int8_t *__restrict__ be,
                               int n, int16_t *ym, int8_t *ye) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool ok = i < n;
  long long sum = 0;
  int em = 0;
  if (ok) {
    const int ea = ae[i >> 4], eb = be[i >> 4];
    em = ea > eb ? ea : eb;
    const long long a = em - ea < 16 ? (am[i] >> (em - ea)) : 0;
    const long long bv = em - eb < 16 ? (bm[i] >> (em - eb)) : 0;
    sum = a + bv;
  }
  const int ml = max16_lanes(sum ? lead64(sum) : 0);
  if (!ok) return;
  int s;
  ym[i] = (int16_t)norm16(sum, ml, s);
  if ((i & 15) == 0) ye[i >> 4] = (int8_t)clamp8(em + s);
}

// ------------------------------------------------------------------ argmax
__device__ __forceinline__ bool bfp_gt(int ma, int ea, int mb, int eb) {
  const int de = ea - eb;
  if (de == 0) return ma > mb;
  if (de > 0) return ma > (de >= 16 ? 0 : (mb >> de));
  return (-de >= 16 ? 0 : (ma >> (-de))) > mb;
}

// A chunk's best as one word: mantissa, exponent byte, lane.
__device__ __forceinline__ int arg_word(int m, int e, int k) {
  return (int)((unsigned)m << 16 | ((unsigned)e & 0xffu) << 8 | (unsigned)k);
}
__device__ __forceinline__ int arg_m(int w) { return w >> 16; }
__device__ __forceinline__ int arg_e(int w) { return (int)(signed char)((w >> 8) & 0xff); }

// The running argmax over chunk words w[0 .. nc) by one wave, in order
// (bfp_gt is not transitive under truncation, so the order counts): every
// lane compares one of 64 chunks with the best so far; the first lane whose
// chunk is greater is the next replacement -- the chunks before it were
// compared with the very best they would have met -- and the lanes after it
// compare again.  A block without a replacement costs one comparison, and a
// sequence's best is replaced about ln(nc) times: 3072 chunks take 11 us,
// against 485 as one lane's fold.  Returns the best's index (16 chunk + lane) in every lane.
__device__ __forceinline__ int argmax_fold(const int *__restrict__ w, int nc) {
  const int l = threadIdx.x & 63;
  constexpr int U = 16;   // blocks of 64 chunks loaded together
  int bm = -32768, be = -128, bi = 0;
  for (int c0 = 0; c0 < nc; c0 += 64 * U) {   // uniform
    int v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = c0 + 64 * u + l;
      v[u] = w[c < nc ? c : nc - 1];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int cb = c0 + 64 * u;
      const int m = arg_m(v[u]), e = arg_e(v[u]);
      unsigned long long rest = cb + 64 <= nc ? ~0ull : (cb < nc ? (1ull << (nc - cb)) - 1 : 0ull);
      for (;;) {
        const unsigned long long gt = __ballot(bfp_gt(m, e, bm, be)) & rest;
        if (!gt) break;
        const int j = __builtin_ctzll(gt);
        const int wj = __builtin_amdgcn_readlane(v[u], j);
        bm = arg_m(wj);
        be = arg_e(wj);
        bi = (cb + j) * 16 + (wj & 15);
        rest &= j == 63 ? 0ull : ~0ull << (j + 1);
      }
    }
  }
  return bi;
}

// The decode head's running argmax (smollm_decode_head_bfp.sv:322-324,
// 399-430): chunk-local bests in parallel (lane 0 of a chunk seeds, the
// others replace only when greater), then the ordered fold over chunks.
// work: one word per chunk.  A row's workgroup has a thread for each of its
// chunks, up to ARGMAX_T: 5000 rows of 64 take 10 us, 27 with ARGMAX_T threads
// for each, 2000 of 1024 7.6 against 13.
constexpr int ARGMAX_T = 1024;
inline int argmax_threads(int n) { return n / 16 < ARGMAX_T ? (n / 16 + 63) / 64 * 64 : ARGMAX_T; }
__global__ __launch_bounds__(ARGMAX_T) void k_rtl_argmax(const int16_t *__restrict__ m, const int8_t *__restrict__ e,
                                                         int n, int *work, int *out) {
  const int b = blockIdx.x, tid = threadIdx.x, nc = n / 16;
  const int16_t *mb = m + (long long)b * n;
  const int8_t *eb = e + (long long)b * n;
  int *W = work + (long long)b * nc;
  for (int c = tid; c < nc; c += blockDim.x) {
    int mm[16], ee[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      mm[k] = mb[c * 16 + k];
      ee[k] = eb[c * 16 + k];
    }
    int bm = mm[0], be = ee[0], bi = 0;
#pragma unroll
    for (int k = 1; k < 16; ++k) {
      const bool g = bfp_gt(mm[k], ee[k], bm, be);
      bm = g ? mm[k] : bm;
      be = g ? ee[k] : be;
      bi = g ? k : bi;
    }
    W[c] = arg_word(bm, be, bi);
  }
  __syncthreads();
  if (tid < 64) {
    const int bi = argmax_fold(W, nc);
    if (tid == 0) out[b] = bi;
  }
}

// The fold alone, over words that the head's matvec wrote.
__global__ __launch_bounds__(64) void k_rl_argmax_fold(const int *__restrict__ w, int nc, int *out) {
  const int bi = argmax_fold(w, nc);
  if (threadIdx.x == 0) *out = bi;
}

// ===================================================== composed RTL layer
// smollm_layer_bfp.sv:1603-2600 on one sequence: the engines above wired in
// the FSM's order, with the matvec engine's sequential tile fold over the
// device-layout weights.  Five launches: NORM1 + Q/K/V, RoPE + KV write +
// attention, O + residual 1, NORM2 + G/U + SwiGLU, D + residual 2.  Each launch
// is a chain of a few microseconds whatever its size, so the norm is
// recomputed by every chunk's workgroup, and RoPE by every head's: the layer
// of 576/1536 takes 37 us in a replayed step (7.8, 8.2, 5.2, 9.7 and 6.5),
// against 92 as eight launches with one-wave norms and in-order folds.

__device__ __forceinline__ void st_put(const StageDump *sd, int s, int i, int m) {
  if (sd && sd->m[s]) sd->m[s][i] = (int16_t)m;
}
__device__ __forceinline__ void st_pute(const StageDump *sd, int s, int t, int e) {
  if (sd && sd->e[s]) sd->e[s][t] = (int8_t)e;
}

// residual_bfp.sv on one tile held by 16 lanes (gen_residual_bfp_golden.py:23-48).
__device__ __forceinline__ void residual16(int am, int ea, int bm, int eb, int &ym, int &ye) {
  const int em = ea > eb ? ea : eb;
  const long long av = em - ea < 16 ? (am >> (em - ea)) : 0;
  const long long bv = em - eb < 16 ? (bm >> (em - eb)) : 0;
  const long long sum = av + bv;
  const int ml = max16_lanes(sum ? lead64(sum) : 0);
  int s;
  ym = norm16(sum, ml, s);
  ye = clamp8(em + s);
}

// swiglu_bfp.sv on one tile held by 16 lanes (gen_swiglu_bfp_golden.py:43-78).
__device__ __forceinline__ void swiglu16(int gm, int ge, int um, int ue,
                                         const int16_t *__restrict__ lut, int &ym, int &ye) {
  const int sh = ge - 5;
  long long idx;
  if (sh >= 0)
    idx = sh >= 16 ? (gm > 0 ? 32767 : (gm < 0 ? -32768 : 0)) : (long long)gm * (1LL << sh);
  else
    idx = -sh >= 16 ? (gm < 0 ? -1 : 0) : (gm >> (-sh));
  idx = idx < -32768 ? -32768 : (idx > 32767 ? 32767 : idx);
  const long long p = (long long)lut[idx & 0xFFFF] * um;
  const int ml = max16_lanes(p ? lead64(p) : 0);
  int s;
  ym = norm16(p, ml, s);
  ye = clamp8(ue + s - 10);
}

// Exact tile sums S = sum_k x[t,k] W[r,t,k] and exponents E = x_e[t] + W_e[r,t]
// of the tiles this lane owns (the layout of load_chunk), into LDS at
// [t*16 + r].
template <int NW, int TPT>
__device__ __forceinline__ void tile_sums_to_lds(const ChunkRegs<TPT> &R, const int *xs,
                                                 const int *xes, int nT, long long *Sl, int *El) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = lane & 15, tq = lane >> 4;
  typedef short s2 __attribute__((ext_vector_type(2)));
#define RL_DOT2(a, b, acc) \
  __builtin_amdgcn_sdot2(__builtin_bit_cast(s2, (a)), __builtin_bit_cast(s2, (b)), (acc), false)
#pragma unroll
  for (int j = 0; j < TPT; ++j) {
    const int t = tq + 4 * (w + NW * j);
    if (t < nT) {
      const int4 *xp = reinterpret_cast<const int4 *>(xs + t * 16);
      const int4 h0 = xp[0], h1 = xp[1], l0 = xp[2], l1 = xp[3];
      int ah = 0, al = 0;
      ah = RL_DOT2(R.a[j].x, h0.x, ah);
      al = RL_DOT2(R.a[j].x, l0.x, al);
      ah = RL_DOT2(R.a[j].y, h0.y, ah);
      al = RL_DOT2(R.a[j].y, l0.y, al);
      ah = RL_DOT2(R.a[j].z, h0.z, ah);
      al = RL_DOT2(R.a[j].z, l0.z, al);
      ah = RL_DOT2(R.a[j].w, h0.w, ah);
      al = RL_DOT2(R.a[j].w, l0.w, al);
      ah = RL_DOT2(R.b[j].x, h1.x, ah);
      al = RL_DOT2(R.b[j].x, l1.x, al);
      ah = RL_DOT2(R.b[j].y, h1.y, ah);
      al = RL_DOT2(R.b[j].y, l1.y, al);
      ah = RL_DOT2(R.b[j].z, h1.z, ah);
      al = RL_DOT2(R.b[j].z, l1.z, al);
      ah = RL_DOT2(R.b[j].w, h1.w, ah);
      al = RL_DOT2(R.b[j].w, l1.w, al);
      Sl[t * 16 + r] = (long long)ah * 256 + al;
      El[t * 16 + r] = xes[t] + R.e[j];
    }
  }
#undef RL_DOT2
}

// NC <= 2 16-row chunks (weights in R) on the engine: sets, in lane 16 c + r
// of wave 0 (c < NC), row r of chunk c's per-lane output (m, e) (the engine's
// out_mant / out_exp).  All threads call it; it synchronises.
template <int NW, int TPT, int NC>
__device__ __forceinline__ void rl_chunk_me(const ChunkRegs<TPT> (&R)[NC], int nT, const int *xs, const int *xes,
                                            long long *Sl, int *El, int &m, int &e) {
#pragma unroll
  for (int c = 0; c < NC; ++c) tile_sums_to_lds<NW, TPT>(R[c], xs, xes, nT, Sl + c * nT * 16, El + c * nT * 16);
  lds_barrier();
  m = 0;
  e = 0;
  if (threadIdx.x < 64) {
    // PQ lanes a row, each a run of tiles.  A run maps acc to (acc + B) >> T
    // with T the rise of the exponent's maximum over it and B its aligned
    // sums shifted up by the rise so far (floors of floors), so the runs
    // fold side by side and combine in order.  Rises past 20 in a run (B
    // might leave 64 bits, or a step drop acc) take the sequential form.
    constexpr int PQ = 4 / NC, NONE = -100000;
    const int grp = threadIdx.x >> 4, lc = NC == 2 ? grp & 1 : 0, q = NC == 2 ? grp >> 1 : grp;
    const long long *S = Sl + lc * nT * 16 + (threadIdx.x & 15);
    const int *E = El + lc * nT * 16 + (threadIdx.x & 15);
    const int run = (nT + PQ - 1) / PQ, t0 = q * run, t1 = t0 + run < nT ? t0 + run : nT;
    int mxq = NONE;
#pragma unroll 8
    for (int t = t0; t < t1; ++t) mxq = E[t * 16] > mxq ? E[t * 16] : mxq;
    // the maximum before this run (its own first exponent for the first)
    int p0 = E[0];
    if constexpr (NC == 1) {
      const int a = peer<16>(mxq), b = peer<32>(mxq), c = peer<32>(a);
      // rows of 16: q 1 has a = run 0; q 2 has b, c = runs 0, 1; q 3 a, b, c = runs 2, 1, 0
      const int bc = b > c ? b : c, abc = a > bc ? a : bc;
      p0 = q == 0 ? p0 : (q == 1 ? a : (q == 2 ? bc : abc));
    } else {
      const int b = peer<32>(mxq);
      p0 = q == 0 ? p0 : b;
    }
    int p = p0;
    long long B = 0;
#pragma unroll 4
    for (int t = t0; t < t1; ++t) {
      const int te = E[t * 16];
      p = te > p ? te : p;
      const int dn = p - te, up = p - p0;
      B += (dn > ACC_W - 1 ? 0 : (S[t * 16] >> dn)) << (up < 20 ? up : 20);
    }
    const int T = p - p0;
    long long acc;
    int acc_e;
    if (!__any(T > 20)) {
      acc = (B >> T);
      acc_e = p;
      if constexpr (NC == 1) {
        const long long B1 = peer<16>(B), B2 = peer<32>(B), B3 = peer<32>(B1);
        const int T1 = peer<16>(T), T2 = peer<32>(T), T3 = peer<32>(T1), e3 = peer<32>(peer<16>(p));
        acc = (((acc + B1) >> T1) + B2) >> T2;
        acc = (acc + B3) >> T3;
        acc_e = e3;
      } else {
        const long long B1 = peer<32>(B);
        const int T1 = peer<32>(T);
        acc = (acc + B1) >> T1;
        acc_e = peer<32>(p);
      }
    } else {
      acc = S[0];
      acc_e = E[0];
#pragma unroll 4
      for (int t = 1; t < nT; ++t) tile_fold(acc, acc_e, S[t * 16], E[t * 16]);
    }
    int sh;
    m = norm16(acc, lead64(acc), sh);
    e = clamp8(acc_e + sh - 15);
  }
}

// Gamma element i as the gamma ROM holds it: tile_quantize of the float
// gamma (whole waves, 16-lane groups on one tile).
struct RomGamma {
  const double *g;
  __device__ __forceinline__ void operator()(int i, int &m, int &e) const { m = quantize16_lanes(g[i], e); }
};

// LDS of a k_rl_mv workgroup of NC chunks over nT input tiles, in bytes from
// the start: the tile sums (at 0), their exponents, the input in the matvec's
// form, and where the input is a norm's output (NORM) that norm's tile sums;
// the exponents of both.  The input is read 16 bytes at a time and nT may be
// odd (FFN is any multiple of 16), so the parts stand in the order of their
// alignment.
struct RlMvLds {
  int El, xs, sums, xes, sexp, bytes;
};
template <int NC, bool NORM>
__host__ __device__ constexpr RlMvLds rl_mv_lds(int nT) {
  const int El = NC * nT * 128, xs = El + NC * nT * 64, sums = xs + nT * 64, xes = sums + (NORM ? nT * 8 : 0),
            sexp = xes + nT * 4;
  return {El, xs, sums, xes, sexp, sexp + (NORM ? nT * 4 : 0)};
}
template <int NC, bool NORM>
constexpr bool rl_mv_lds_aligned() {
  for (int nT = 1; nT <= 108; ++nT) {
    const RlMvLds o = rl_mv_lds<NC, NORM>(nT);
    if (o.xs % 16 || o.sums % 8 || o.El % 4 || o.xes % 4 || o.sexp % 4 || o.bytes > 65536) return false;
  }
  return true;
}
static_assert(rl_mv_lds_aligned<1, true>() && rl_mv_lds_aligned<1, false>() && rl_mv_lds_aligned<2, true>(),
              "the parts of k_rl_mv's LDS are aligned and fit a workgroup's default limit");

// The layer's matvecs, one 16-row output chunk per workgroup, every weight
// load issued before the input is staged.
//   OP 0: Q|K|V from NORM1(h, G1)  (chunks of qkv, re-tiled per chunk)
//   OP 1: O from att, then residual 1 with h -> h1
//   OP 2: G chunk c and U chunk c from NORM2(h1, G2), then SwiGLU -> mlp
//   OP 3: D from mlp, then residual 2 with h1 -> h
template <int NW, int op>
__global__ __launch_bounds__(64 * NW) void k_rl_mv(RtlArgs a) {
  constexpr int TPT = 3, NC = op == 2 ? 2 : 1;
  constexpr bool NORM = op == 0 || op == 2;
  extern __shared__ __align__(16) long long rl_lds[];
  const LayerArgs &L = a.L;
  const int c = blockIdx.x;
  const int nT = (op == 3 ? L.FFN : L.D) / 16;
  const RlMvLds o = rl_mv_lds<NC, NORM>(nT);
  char *lds = reinterpret_cast<char *>(rl_lds);
  long long *Sl = rl_lds;                                       // NC x nT x 16
  long long *sums = reinterpret_cast<long long *>(lds + o.sums);   // nT
  int *El = reinterpret_cast<int *>(lds + o.El);                // NC x nT x 16
  int *xs = reinterpret_cast<int *>(lds + o.xs);                // nT x 16
  int *xes = reinterpret_cast<int *>(lds + o.xes);              // nT
  int *sexp = reinterpret_cast<int *>(lds + o.sexp);            // nT
  const uint4 *wm = op == 0 ? L.w_qkv_m : (op == 1 ? L.w_o_m : (op == 2 ? L.w_gu_m : L.w_d_m));
  const int8_t *we = op == 0 ? L.w_qkv_e : (op == 1 ? L.w_o_e : (op == 2 ? L.w_gu_e : L.w_d_e));
  ChunkRegs<TPT> R[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k)
    load_chunk_nb<NW, TPT>(R[k], wm + (size_t)(NC * c + k) * nT * 32, we + (size_t)(NC * c + k) * nT * 16, nT);
  if constexpr (NORM) {
    const StageDump *sd = c == 0 ? L.dump : nullptr;
    constexpr int st = op == 0 ? ST_N1 : ST_N2;
    rms_block(op == 0 ? L.h_m : L.h1_m, op == 0 ? L.h_e : L.h1_e, RomGamma{op == 0 ? L.g1 : L.g2}, L.D, sums, sexp,
              [&](int i, int m, int e) {
                // the even lane writes the pair into the matvec's input form
                const int odd = __builtin_amdgcn_mov_dpp(m, 0xB1, 0xf, 0xf, false);   // quad_perm 1,0,3,2
                if (i >= L.D) return;
                if ((i & 1) == 0) put_x_pair(xs, i >> 4, (i >> 1) & 7, m, odd);
                if ((i & 15) == 0) xes[i >> 4] = e;
                st_put(sd, st, i, m);
                if ((i & 15) == 0) st_pute(sd, st, i >> 4, e);
              });
  } else {
    stage_x_bfp(xs, xes, op == 1 ? L.att_m : L.mlp_m, op == 1 ? L.att_e : L.mlp_e, nT);
  }
  lds_barrier();
  int m, e;
  rl_chunk_me<NW, TPT, NC>(R, nT, xs, xes, Sl, El, m, e);
  if (threadIdx.x >= 64) return;
  // the chunk re-tile (S_xMV_DRAIN/REQ): lanes 0-15 chunk 0, 16-31 chunk 1
  const int em = max16_lanes(e), mt = shr8(m, em, e);
  const int mq = mt, emax = em;
  const int mu = __shfl(mt, (threadIdx.x & 15) + 16, 64), eu = __shfl(em, (threadIdx.x & 15) + 16, 64);
  const int r = threadIdx.x & 15, i = c * 16 + r;
  const bool w = threadIdx.x < 16;
  const StageDump *sd = L.dump;
  if (op == 0) {
    if (w) {
      L.qkv_m[i] = (int16_t)mq;
      if (r == 0) L.qkv_e[c] = (int8_t)emax;
    }
    return;
  }
  int ym, ye;
  if (op == 1 || op == 3) {
    const int16_t *bm = op == 1 ? L.h_m : L.h1_m;
    const int8_t *be = op == 1 ? L.h_e : L.h1_e;
    residual16(bm[i], be[c], mq, emax, ym, ye);
    int16_t *om = op == 1 ? L.h1_m : L.h_m;
    int8_t *oe = op == 1 ? L.h1_e : L.h_e;
    const int so = op == 1 ? ST_O : ST_D, sr = op == 1 ? ST_H1 : ST_HOUT;
    if (w) {
      om[i] = (int16_t)ym;
      if (r == 0) oe[c] = (int8_t)ye;
      st_put(sd, so, i, mq);
      st_put(sd, sr, i, ym);
      if (r == 0) {
        st_pute(sd, so, c, emax);
        st_pute(sd, sr, c, ye);
      }
    }
    return;
  }
  swiglu16(mq, emax, mu, eu, a.silu_lut, ym, ye);
  if (w) {
    L.mlp_m[i] = (int16_t)ym;
    if (r == 0) L.mlp_e[c] = (int8_t)ye;
    st_put(sd, ST_G, i, mq);
    st_put(sd, ST_U, i, mu);
    st_put(sd, ST_MLP, i, ym);
    if (r == 0) {
      st_pute(sd, ST_G, c, emax);
      st_pute(sd, ST_U, c, eu);
      st_pute(sd, ST_MLP, c, ye);
    }
  }
}

// The step of the RTL layer: a.pos / a.kv_pos, or the device step counter.
__device__ __forceinline__ int rl_pos(const RtlArgs &a) { return a.pos_ptr ? *a.pos_ptr : a.pos; }
__device__ __forceinline__ int rl_kv_pos(const RtlArgs &a) { return a.pos_ptr ? *a.pos_ptr : a.kv_pos; }

// RoPE of one head (x: 64 mantissas, e: 4 exponents) by the first 32 lanes
// of a wave (lanes 32-63 repeat them), then the re-tile of its four tiles
// (S_ROPEx_RQ_A/B): elements j and j + 32 in (qlo, elo), (qhi, ehi).
__device__ __forceinline__ void rl_rope(const int16_t *x, const int8_t *e, int pos, const unsigned *freq, int &qlo,
                                        int &elo, int &qhi, int &ehi) {
  const int j = threadIdx.x & 31;
  const long long ang = wrap31((wrap31((long long)pos * freq[j]) * PI_OVER_8_Q29) >> 29);
  const int xa = x[j], xb = x[j + 32];
  const int ea = e[j >> 4], eb = e[(j + 32) >> 4];
  int cs, sn;
  cordic(ang, cs, sn);
  const int em = ea > eb ? ea : eb;
  const long long aa = em - ea < 16 ? (xa >> (em - ea)) : 0;
  const long long ba = em - eb < 16 ? (xb >> (em - eb)) : 0;
  const long long lo = aa * cs - ba * sn, hi = ba * cs + aa * sn;
  int sh;
  const int mlo = norm16(lo, lead64(lo), sh);
  const int e0 = clamp8(em + sh - 15);
  const int mhi = norm16(hi, lead64(hi), sh);
  const int e1 = clamp8(em + sh - 15);
  // lanes 0-15 hold tiles 0 (lo) and 2 (hi), lanes 16-31 tiles 1 and 3
  elo = max16_lanes(e0);
  ehi = max16_lanes(e1);
  qlo = shr8(mlo, elo, e0);
  qhi = shr8(mhi, ehi, e1);
}

constexpr int RL_ATT_T = 256;

__device__ __forceinline__ int wave_max_i(int v) {
  v = max16_lanes(v);
  v = pmax<16>(v);
  return pmax<32>(v);
}

// RoPE and attention of query head h (S_ROPE*, S_KVWR_*, S_QK_* .. S_AV_*):
// wave 0 rotates the head's Q, wave 1 its K head, wave 2 takes its V; the
// first head of a KV group writes the slot kv_pos (rotated K, V), and row
// kv_pos is used from LDS.  Then scores of t = 0..kv_pos on the engine's lane
// 0 (Q head as x, K[t] as the weight row), pre-align to the shared max
// exponent, softmax with exponent - 3 (1/sqrt(64)), then per 16-dim chunk the
// engine over one 16-input tile of probabilities (t <= 15) with V pre-shifted
// to its largest exponent over t <= kv_pos.
__global__ __launch_bounds__(RL_ATT_T) void k_rl_attn(RtlArgs a) {
  extern __shared__ long long rl_lds[];
  constexpr int NW = RL_ATT_T / 64;
  __shared__ int qs[64], qe[4], red_e[NW], red_x[NW], red_s[NW], red_v[4 * NW];
  __shared__ __align__(16) int16_t kc[64], vc[64];
  __shared__ int kce[4], vce[4];
  __shared__ int pm[16];
  const LayerArgs &L = a.L;
  const int h = blockIdx.x, tid = threadIdx.x, HD = 64, wv = tid >> 6, ln = tid & 63;
  const int g = (h * L.H_KV) / L.H_Q;
  const bool writer = h == 0 || ((h - 1) * L.H_KV) / L.H_Q != g;
  const int kv = rl_kv_pos(a), n = kv + 1;
  int *xs = reinterpret_cast<int *>(rl_lds);   // n aligned scores, then LUT values
  int *se = xs + n;                             // n score exponents
  const size_t slot0 = (size_t)kv * L.H_KV + g;   // sequence 0
  const StageDump *sd = L.dump;
  if (wv < 2) {
    const int off = wv == 0 ? h * HD : L.D + g * HD, j = ln & 31;
    int qlo, elo, qhi, ehi;
    rl_rope(L.qkv_m + off, L.qkv_e + off / 16, rl_pos(a), a.freq, qlo, elo, qhi, ehi);
    if (ln < 32) {
      if (wv == 0) {
        qs[j] = qlo;
        qs[j + 32] = qhi;
        if ((j & 15) == 0) {
          qe[j >> 4] = elo;
          qe[(j + 32) >> 4] = ehi;
        }
      } else {
        kc[j] = (int16_t)qlo;
        kc[j + 32] = (int16_t)qhi;
        if ((j & 15) == 0) {
          kce[j >> 4] = elo;
          kce[(j + 32) >> 4] = ehi;
        }
        if (writer) {
          int16_t *km = L.k_m + slot0 * HD;
          int8_t *ke = L.k_e + slot0 * (HD / 16);
          km[j] = (int16_t)qlo;
          km[j + 32] = (int16_t)qhi;
          if ((j & 15) == 0) {
            ke[j >> 4] = (int8_t)elo;
            ke[(j + 32) >> 4] = (int8_t)ehi;
          }
        }
      }
      const int st = wv == 0 ? ST_Q : ST_K, so = wv == 0 ? h * HD : g * HD;
      if (wv == 0 || writer) {
        st_put(sd, st, so + j, qlo);
        st_put(sd, st, so + j + 32, qhi);
        if ((j & 15) == 0) {
          st_pute(sd, st, so / 16 + (j >> 4), elo);
          st_pute(sd, st, so / 16 + ((j + 32) >> 4), ehi);
        }
      }
    }
  } else if (wv == 2) {
    const int off = L.D + L.KV + g * HD;
    const int v = L.qkv_m[off + ln], vt = L.qkv_e[off / 16 + (ln & 3)];
    vc[ln] = (int16_t)v;
    if (ln < 4) vce[ln] = vt;
    if (writer) {
      L.v_m[slot0 * HD + ln] = (int16_t)v;
      st_put(sd, ST_V, g * HD + ln, v);
      if (ln < 4) {
        L.v_e[slot0 * (HD / 16) + ln] = (int8_t)vt;
        st_pute(sd, ST_V, g * 4 + ln, vt);
      }
    }
  }
  lds_barrier();
  for (int t = tid; t < n; t += RL_ATT_T) {
    const size_t slot = (size_t)(t < kv ? t : 0) * L.H_KV + g;
    const uint4 *kp = reinterpret_cast<const uint4 *>(t < kv ? L.k_m + slot * HD : kc);
    const int ke4 = *reinterpret_cast<const int *>(L.k_e + slot * 4);
    uint4 kr[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) kr[q] = kp[q];
    long long acc = 0;
    int acc_e = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      long long s = 0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const unsigned wd[4] = {kr[2 * c + q].x, kr[2 * c + q].y, kr[2 * c + q].z, kr[2 * c + q].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int *x = qs + c * 16 + 8 * q + 2 * k;
          s += (long long)(x[0] * (int)(short)(wd[k] & 0xffff)) + (long long)(x[1] * ((int)wd[k] >> 16));
        }
      }
      const int te = qe[c] + (t < kv ? (int)(signed char)((ke4 >> (8 * c)) & 0xff) : kce[c]);
      if (c == 0) {
        acc = s;
        acc_e = te;
      } else {
        tile_fold(acc, acc_e, s, te);
      }
    }
    int sh;
    xs[t] = norm16(acc, lead64(acc), sh);
    se[t] = clamp8(acc_e + sh - 15);
  }
  // (each thread reads back only the scores it wrote until the last barrier)
  // the largest score exponent, and V's per 16-dim chunk over t <= kv_pos
  int lmax = -128, vm4[4] = {-128, -128, -128, -128};
  for (int t = tid; t < n; t += RL_ATT_T) {
    lmax = se[t] > lmax ? se[t] : lmax;
    const int ve4 = *reinterpret_cast<const int *>(L.v_e + ((size_t)(t < kv ? t : 0) * L.H_KV + g) * 4);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int ve = t < kv ? (int)(signed char)((ve4 >> (8 * c)) & 0xff) : vce[c];
      vm4[c] = ve > vm4[c] ? ve : vm4[c];
    }
  }
  lmax = wave_max_i(lmax);
#pragma unroll
  for (int c = 0; c < 4; ++c) vm4[c] = wave_max_i(vm4[c]);
  if (ln == 0) {
    red_e[wv] = lmax;
#pragma unroll
    for (int c = 0; c < 4; ++c) red_v[4 * wv + c] = vm4[c];
  }
  lds_barrier();
  int es = red_e[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) es = red_e[i] > es ? red_e[i] : es;
  int xmax = -32768;
  for (int t = tid; t < n; t += RL_ATT_T) {
    const int d = es - se[t];               // 9-bit in the FSM: no wrap
    const int v = d >= 16 ? 0 : (xs[t] >> d);
    xs[t] = v;
    xmax = v > xmax ? v : xmax;
  }
  xmax = wave_max_i(xmax);
  if (ln == 0) red_x[wv] = xmax;
  lds_barrier();
  int mx = red_x[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) mx = red_x[i] > mx ? red_x[i] : mx;
  const int xe = (int)(signed char)(es - 3);
  const int sh = xe - 8;
  int part = 0;                              // at most 4096 * 65535
  for (int t = tid; t < n; t += RL_ATT_T) {
    const long long d = (long long)xs[t] - mx;
    const long long ds = sh >= 0 ? d * (1LL << (sh > 40 ? 40 : sh)) : (d >> (-sh > 62 ? 62 : -sh));
    const int idx = ds >= 0 ? 1023 : (ds <= -1023 ? 0 : (int)(ds + 1023));
    const int v = a.exp_lut[idx];
    xs[t] = v;
    part += v;
  }
  part = psum<8>(part);
  part = psum<4>(part);
  part = psum<2>(part);
  part = psum<1>(part);
  part = psum<16>(part);
  part = psum<32>(part);
  if (ln == 0) red_s[wv] = part;
  lds_barrier();
  if (tid >= 64) return;
  const int c = tid >> 4, l = tid & 15;
  // 16 rows, every load issued before the first is used; p is 0 past kv_pos
  int vr[16], vt[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const size_t slot = (size_t)(t < kv ? t : 0) * L.H_KV + g;
    vr[t] = L.v_m[slot * HD + c * 16 + l];
    vt[t] = L.v_e[slot * 4 + c];
  }
  long long tot = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) tot += red_s[i];
  const int msb = tot ? 63 - __clzll((unsigned long long)tot) : 0;
  __int128 y = (__int128)1 << (31 - msb);
  for (int it = 0; it < 4; ++it) y = (y * (((__int128)1 << 33) - (__int128)tot * y)) >> 32;
  const long long inv = (long long)y;
  // the largest product's leading bit: the table rises, and the largest score
  // (difference 0) takes its last entry
  const long long pmax_ = (long long)a.exp_lut[1023] * inv;
  const int ml = pmax_ ? lead64(pmax_) : 0;
  if (tid < 16) {
    int s2;
    pm[tid] = tid < n ? norm16((long long)xs[tid] * inv, ml, s2) : 0;
  }
  const int s_pe = clamp8(ml - 14 - 17);
  int vmax = red_v[c];
#pragma unroll
  for (int i = 1; i < NW; ++i) vmax = red_v[4 * i + c] > vmax ? red_v[4 * i + c] : vmax;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  long long s = 0;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int v = t < kv ? vr[t] : vc[c * 16 + l], ve = t < kv ? vt[t] : vce[c];
    s += (long long)(pm[t] * shr8(v, vmax, ve));
  }
  int sh2;
  const int m = norm16(s, lead64(s), sh2);
  const int e = clamp8(s_pe + vmax + sh2 - 15);
  const int emax = max16_lanes(e);
  const int mq = shr8(m, emax, e);
  const int i = h * HD + c * 16 + l;
  L.att_m[i] = (int16_t)mq;
  if (l == 0) L.att_e[h * 4 + c] = (int8_t)emax;
  st_put(L.dump, ST_ATTN, i, mq);
  if (l == 0) st_pute(L.dump, ST_ATTN, h * 4 + c, emax);
}

// ------------------------------------------------------------- decode head
// smollm_decode_head_bfp.sv: S_NORM (the RMSNorm engine with the final norm
// gamma from its ROM, i.e. tile_quantize'd), then per 16-row chunk of the
// tied embedding the matvec engine (S_MV_*), whose per-lane (m, e) feed the
// bfp_gt running argmax (S_MV_LANE_CMP / S_MV_MERGE, k_rtl_argmax).
__global__ __launch_bounds__(RMS_T) void k_rl_head_norm(RtlHeadArgs a) {
  extern __shared__ long long rl_lds[];
  const int nt = a.D / 16;
  rms_block(a.h_m, a.h_e, RomGamma{a.norm_w}, a.D, rl_lds, reinterpret_cast<int *>(rl_lds + nt),
            [&](int i, int m, int e) {
              if (i >= a.D) return;
              a.xn_m[i] = (int16_t)m;
              if ((i & 15) == 0) a.xn_e[i >> 4] = (int8_t)e;
            });
}

// One 16-row chunk of the embedding per workgroup: the engine's per-row
// (m, e) into lg_m / lg_e, and the chunk's best (lane 0 seeds, the next
// lane that is greater replaces) into work[chunk].
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_rl_head_mv(RtlHeadArgs a) {
  constexpr int TPT = 3;
  extern __shared__ long long rl_lds[];
  const int c = blockIdx.x, nT = a.D / 16;
  long long *Sl = rl_lds;
  int *El = reinterpret_cast<int *>(Sl + nT * 16);
  int *xs = El + nT * 16;
  int *xes = xs + nT * 16;
  ChunkRegs<TPT> R[1];
  load_chunk_nb<NW, TPT>(R[0], a.emb_m + (size_t)c * nT * 32, a.emb_e + (size_t)c * nT * 16, nT);
  stage_x_bfp(xs, xes, a.xn_m, a.xn_e, nT);
  lds_barrier();
  int m, e;
  rl_chunk_me<NW, TPT, 1>(R, nT, xs, xes, Sl, El, m, e);
  if (threadIdx.x >= 64) return;
  if (threadIdx.x < 16) {
    a.lg_m[c * 16 + threadIdx.x] = (int16_t)m;
    a.lg_e[c * 16 + threadIdx.x] = (int8_t)e;
  }
  int bm = __builtin_amdgcn_readlane(m, 0), be = __builtin_amdgcn_readlane(e, 0), bk = 0;
  unsigned rest = 0xfffeu;
  for (;;) {
    const unsigned gt = (unsigned)__ballot(bfp_gt(m, e, bm, be)) & rest;
    if (!gt) break;
    bk = __builtin_ctz(gt);
    bm = __builtin_amdgcn_readlane(m, bk);
    be = __builtin_amdgcn_readlane(e, bk);
    rest &= ~0u << (bk + 1);
  }
  if (threadIdx.x == 0) a.work[c] = arg_word(bm, be, bk);
}

// One step of the FPGA driver's token loop on the device
// (autoregress_bfp_top.sv:357-386): record the head's token as this step's
// prediction (and the last layer's output when a history is kept), then the
// next step's input -- prompt[step + 1] while the prompt lasts, else this
// prediction -- and advance the step.  One 64-thread workgroup.
__global__ __launch_bounds__(64) void k_rtl_ctl(RtlCtlArgs a) {
  const int tid = threadIdx.x;
  const int step = a.state[0], tok = *a.tok;
  if (a.hist_m) {
    for (int i = tid; i < a.D; i += 64) a.hist_m[(size_t)step * a.D + i] = a.h_m[i];
    for (int i = tid; i < a.D / 16; i += 64) a.hist_e[(size_t)step * (a.D / 16) + i] = a.h_e[i];
  }
  __syncthreads();   // every thread has read the step before it changes
  if (tid == 0) {
    a.preds[step] = tok;
    a.state[1] = step + 1 < a.n_prompt ? a.prompt[step + 1] : tok;
    a.state[0] = step + 1;
  }
}

}  // namespace rtl
}  // namespace bfp

// ---------------------------------------------- allocation-free argmax
// Scratch of bfp_rtl_argmax_static_d: the per-chunk bests (a word of
// mantissa, exponent and lane each) of at most ARGMAX_STATIC_CHUNKS chunks
// (batch * n/16), in one device-global array per GPU: 1 MiB, held until the
// process ends.
// Host code never passes the array's name to a kernel (on the host it is a
// stand-in, not a device address): argmax_scratch() looks its address up
// once per device with hipGetSymbolAddress and hands that out.
namespace bfp {
namespace {
constexpr long long ARGMAX_STATIC_CHUNKS = 262144;
static __device__ __align__(256) int scratch[ARGMAX_STATIC_CHUNKS];
constexpr int SCRATCH_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
int *g_scratch[SCRATCH_MAX_DEVICES] = {};

int argmax_scratch(int **out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= SCRATCH_MAX_DEVICES)
    return set_err(BFP_EINVAL, "rtl_argmax_static: device %d beyond the %d supported", dev,
                   SCRATCH_MAX_DEVICES);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p)
      return set_err(BFP_EIO, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                     hipGetErrorString(err));
    g_scratch[dev] = static_cast<int *>(p);
  }
  *out = g_scratch[dev];
  return BFP_OK;
}
}  // namespace
}  // namespace bfp

using namespace bfp;

static inline unsigned nb(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

extern "C" {

// LUTs and tables of the RTL ops, built on the host from their defining
// formulas with the host libm: EXP_LUT (sim/gen_exp_lut.py:36-42),
// SILU_LUT (sim/gen_swiglu_lut.py:27-44, indexed by the int16 code & 0xFFFF),
// FREQ_TURNS_Q31 (sim/gen_rope_freq_table.py:31-37).  Any pointer may be NULL.
int bfp_rtl_tables(uint16_t *exp_lut, int16_t *silu_lut, uint32_t *freq_q31, int head_dim,
                   double base) {
  if (exp_lut)
    for (int i = 0; i < 1024; ++i) {
      double v = nearbyint(exp((i - 1023) / 128.0) * 32768.0);
      exp_lut[i] = (uint16_t)(v > 65535 ? 65535 : (v < 0 ? 0 : v));
    }
  if (silu_lut)
    for (int c = 0; c < 65536; ++c) {
      const double code = (double)(int16_t)(uint16_t)c;
      const double g = code / 32768.0 * 32.0;
      const double s = g * (1.0 / (1.0 + exp(-g)));
      double q = nearbyint(s * 32768.0 / 32.0);
      q = q > 32767 ? 32767 : (q < -32768 ? -32768 : q);
      silu_lut[c] = (int16_t)q;
    }
  if (freq_q31) {
    if (head_dim <= 0 || head_dim % 2) return set_err(BFP_EINVAL, "head_dim %d", head_dim);
    for (int j = 0; j < head_dim / 2; ++j) {
      const double f = 1.0 / pow(base, 2.0 * j / head_dim);
      freq_q31[j] = (uint32_t)nearbyint(f / (2.0 * M_PI) * (double)(1LL << 31));
    }
  }
  return BFP_OK;
}

int bfp_rtl_matvec_d(const int16_t *x_m, const int8_t *x_e, const int16_t *W_m, const int8_t *W_e,
                     int n_out, int n_in, int16_t *y_m, int8_t *y_e, void *stream) {
  if (n_out <= 0 || n_in <= 0 || n_in % 16) return set_err(BFP_EINVAL, "rtl_matvec: shape");
  hipLaunchKernelGGL(rtl::k_rtl_matvec, dim3(nb(n_out, 64)), dim3(64), 0, (hipStream_t)stream,
                     x_m, x_e, W_m, W_e, n_out, n_in / 16, y_m, y_e);
  return launch_status("rtl_matvec");
}

int bfp_rtl_requant_d(const int16_t *m, const int8_t *e, int n, int16_t *out_m, int8_t *out_e,
                      void *stream) {
  if (n <= 0 || n % 16) return set_err(BFP_EINVAL, "rtl_requant: n=%d", n);
  hipLaunchKernelGGL(rtl::k_rtl_requant, dim3(nb(n, 64)), dim3(64), 0, (hipStream_t)stream, m, e,
                     n, out_m, out_e);
  return launch_status("rtl_requant");
}

int bfp_rtl_rmsnorm_d(const int16_t *x_m, const int8_t *x_e, const int16_t *g_m, const int8_t *g_e,
                      int D, int batch, int16_t *y_m, int8_t *y_e, void *stream) {
  if (D <= 0 || D % 16 || D > 65536 || batch <= 0)
    return set_err(BFP_EINVAL, "rtl_rmsnorm: D=%d batch=%d", D, batch);
  hipLaunchKernelGGL(rtl::k_rtl_rmsnorm, dim3(batch), dim3(rtl::rms_threads(D)), (size_t)(D / 16) * 12,
                     (hipStream_t)stream, x_m, x_e, g_m, g_e, D, y_m, y_e);
  return launch_status("rtl_rmsnorm");
}

int bfp_rtl_rope_d(const int16_t *x_m, const int8_t *x_e, int pos, int n_heads,
                   const uint32_t *freq_q31, int16_t *y_m, int8_t *y_e, void *stream) {
  if (n_heads <= 0 || pos < 0) return set_err(BFP_EINVAL, "rtl_rope: heads=%d pos=%d", n_heads, pos);
  hipLaunchKernelGGL(rtl::k_rtl_rope, dim3(n_heads), dim3(64), 0, (hipStream_t)stream, x_m, x_e,
                     pos, freq_q31, y_m, y_e);
  return launch_status("rtl_rope");
}

int bfp_rtl_softmax_d(const int16_t *x_m, const int8_t *x_e, int n, int batch, int stride,
                      const uint16_t *exp_lut, int16_t *y_m, int8_t *y_e, void *stream) {
  if (n <= 0 || n > 4096 || batch <= 0 || stride < n)
    return set_err(BFP_EINVAL, "rtl_softmax: n=%d batch=%d stride=%d", n, batch, stride);
  hipLaunchKernelGGL(rtl::k_rtl_softmax, dim3(batch), dim3(64), (size_t)n * 8, (hipStream_t)stream,
                     x_m, x_e, n, stride, exp_lut, y_m, y_e);
  return launch_status("rtl_softmax");
}

int bfp_rtl_swiglu_d(const int16_t *g_m, const int8_t *g_e, const int16_t *u_m, const int8_t *u_e,
                     int n, const int16_t *silu_lut, int16_t *y_m, int8_t *y_e, void *stream) {
  if (n <= 0 || n % 16) return set_err(BFP_EINVAL, "rtl_swiglu: n=%d", n);
  hipLaunchKernelGGL(rtl::k_rtl_swiglu, dim3(nb(n, 64)), dim3(64), 0, (hipStream_t)stream, g_m, g_e,
                     u_m, u_e, n, silu_lut, y_m, y_e);
  return launch_status("rtl_swiglu");
}

int bfp_rtl_residual_d(const int16_t *a_m, const int8_t *a_e, const int16_t *b_m,
                       const int8_t *b_e, int n, int16_t *y_m, int8_t *y_e, void *stream) {
  if (n <= 0 || n % 16) return set_err(BFP_EINVAL, "rtl_residual: n=%d", n);
  hipLaunchKernelGGL(rtl::k_rtl_residual, dim3(nb(n, 64)), dim3(64), 0, (hipStream_t)stream, a_m,
                     a_e, b_m, b_e, n, y_m, y_e);
  return launch_status("rtl_residual");
}

// bfp_rtl_argmax_d with its workspace in the library's static device
// scratch (no allocation).  The kernel writes every chunk's entry before it
// reads it, so nothing needs clearing between calls; calls that overlap on
// one GPU share the scratch and race.
int bfp_rtl_argmax_static_d(const int16_t *m, const int8_t *e, int n, int batch, int32_t *idx,
                            void *stream) {
  if (n <= 0 || n % 16 || batch <= 0 || !m || !e || !idx)
    return set_err(BFP_EINVAL, "rtl_argmax_static: n=%d batch=%d", n, batch);
  const long long nc = (long long)batch * (n / 16);
  if (nc > bfp::ARGMAX_STATIC_CHUNKS)
    return set_err(BFP_EINVAL,
                   "rtl_argmax_static: batch * n/16 = %lld chunks exceeds the static scratch's "
                   "%lld (use bfp_rtl_argmax_d with a workspace)",
                   nc, bfp::ARGMAX_STATIC_CHUNKS);
  int *w = nullptr;
  BFP_TRY(bfp::argmax_scratch(&w));
  hipLaunchKernelGGL(rtl::k_rtl_argmax, dim3(batch), dim3(rtl::argmax_threads(n)), 0, (hipStream_t)stream, m, e, n, w, idx);
  return launch_status("rtl_argmax_static");
}

// work: batch * n/16 ints of device scratch supplied by the caller.
int bfp_rtl_argmax_d(const int16_t *m, const int8_t *e, int n, int batch, int32_t *work,
                     int32_t *idx, void *stream) {
  if (n <= 0 || n % 16 || batch <= 0 || !work) return set_err(BFP_EINVAL, "rtl_argmax: n=%d", n);
  hipLaunchKernelGGL(rtl::k_rtl_argmax, dim3(batch), dim3(rtl::argmax_threads(n)), 0, (hipStream_t)stream, m, e, n,
                     work, idx);
  return launch_status("rtl_argmax");
}

}  // extern "C"

namespace bfp {

namespace {
typedef void (*rl_mv_fn)(RtlArgs);
template <int OP>
rl_mv_fn rl_mv_kernel(int nw) {
  static const rl_mv_fn k[9] = {rtl::k_rl_mv<1, OP>, rtl::k_rl_mv<2, OP>, rtl::k_rl_mv<3, OP>,
                                rtl::k_rl_mv<4, OP>, rtl::k_rl_mv<5, OP>, rtl::k_rl_mv<6, OP>,
                                rtl::k_rl_mv<7, OP>, rtl::k_rl_mv<8, OP>, rtl::k_rl_mv<9, OP>};
  return nw >= 1 && nw <= 9 ? k[nw - 1] : nullptr;
}

// One matvec op of the layer: nT input tiles, n_wg output chunks.
template <int OP>
int rl_mv(const RtlArgs &a, int nT, int n_wg, hipStream_t s) {
  const int nw = (nT + 11) / 12;   // 3 tiles per lane, 4 tile lanes per wave
  rl_mv_fn f = rl_mv_kernel<OP>(nw);
  if (!f) return set_err(BFP_EINVAL, "rtl layer: %d input tiles unsupported", nT);
  const size_t lds = rtl::rl_mv_lds<OP == 2 ? 2 : 1, OP == 0 || OP == 2>(nT).bytes;
  hipLaunchKernelGGL(f, dim3(n_wg), dim3(64 * nw), lds, s, a);
  return launch_status("rtl layer matvec");
}
}  // namespace

int launch_rtl_layer(const RtlArgs &a, hipStream_t s) {
  const LayerArgs &L = a.L;
  const int ntD = L.D / 16, ntF = L.FFN / 16;
  // with pos_ptr the caller keeps the device step inside the capacity
  if (L.batch != 1 || L.HD != 64 ||
      (!a.pos_ptr && (a.kv_pos < 0 || a.kv_pos >= L.max_ctx || a.pos < 0)))
    return set_err(BFP_EINVAL, "rtl layer: batch %d, HD %d, pos %d, kv_pos %d (capacity %d)",
                   L.batch, L.HD, a.pos, a.kv_pos, L.max_ctx);
  const int n_att = a.pos_ptr ? L.max_ctx : a.kv_pos + 1;   // positions the attention's LDS holds
  BFP_TRY(rl_mv<0>(a, ntD, (L.D + 2 * L.KV) / 16, s));
  hipLaunchKernelGGL(rtl::k_rl_attn, dim3(L.H_Q), dim3(rtl::RL_ATT_T), (size_t)n_att * 8, s, a);
  BFP_TRY(launch_status("rtl layer attention"));
  BFP_TRY(rl_mv<1>(a, ntD, ntD, s));
  BFP_TRY(rl_mv<2>(a, ntD, ntF, s));
  return rl_mv<3>(a, ntF, ntD, s);
}

int launch_rtl_ctl(const RtlCtlArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(rtl::k_rtl_ctl, dim3(1), dim3(64), 0, s, a);
  return launch_status("rtl loop control");
}

int launch_rtl_head(const RtlHeadArgs &a, hipStream_t s) {
  const int nT = a.D / 16;
  if (a.D % 64 || a.VOCAB % 16 || a.VOCAB <= 0)
    return set_err(BFP_EINVAL, "rtl head: D %d (multiple of 64), VOCAB %d (multiple of 16)", a.D,
                   a.VOCAB);
  typedef void (*hm_fn)(RtlHeadArgs);
  static const hm_fn k[9] = {rtl::k_rl_head_mv<1>, rtl::k_rl_head_mv<2>, rtl::k_rl_head_mv<3>,
                             rtl::k_rl_head_mv<4>, rtl::k_rl_head_mv<5>, rtl::k_rl_head_mv<6>,
                             rtl::k_rl_head_mv<7>, rtl::k_rl_head_mv<8>, rtl::k_rl_head_mv<9>};
  const int nw = (nT + 11) / 12;   // 3 tiles per lane, 4 tile lanes per wave
  if (nw > 9) return set_err(BFP_EINVAL, "rtl head: %d input tiles unsupported", nT);
  hipLaunchKernelGGL(rtl::k_rl_head_norm, dim3(1), dim3(rtl::RMS_T), (size_t)nT * 12, s, a);
  BFP_TRY(launch_status("rtl head norm"));
  hipLaunchKernelGGL(k[nw - 1], dim3(a.VOCAB / 16), dim3(64 * nw), (size_t)nT * 260, s, a);
  BFP_TRY(launch_status("rtl head matvec"));
  hipLaunchKernelGGL(rtl::k_rl_argmax_fold, dim3(1), dim3(64), 0, s, a.work, a.VOCAB / 16, a.token);
  return launch_status("rtl head argmax");
}

}  // namespace bfp
