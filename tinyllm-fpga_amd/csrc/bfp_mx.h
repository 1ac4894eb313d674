// Exact BFP tile sums of many sequences on the matrix cores (int8 MFMA).
//
// Semantics are the engine's (rtl/vc707/host/gen_smollm_blockfp_full.py
// :217-233): per row o, sequence s and input tile t the exact
// S = sum_k W_m[o,t,k] x_m[s,t,k], E = W_e[o,t] + x_e[s,t], M = max_t E,
// A = sum_t floor(S / 2^(M-E)) for M-E <= 47.
//
// Both int16 operands are split into a signed high byte and an offset low
// byte: v = 256*vh + vl' + 128 with vh = v >> 8 and vl' = (v & 255) - 128,
// both in [-128, 127].  Over one 16-element tile
//   S = 65536*Phh + 256*(Phl + Plh + 128*sum Wh) + (Pll + 128*sum Wl')
//       + 128*sum x
// where Pab = sum_k Wa*xb.  Every product sum is one v_mfma_i32_16x16x32_i8,
// whose 32-deep k axis holds the tile twice (k-groups 0-1 and 2-3 of the
// operand layout).  The weight operand of all of them is A = [Wh, Wl'] (first
// copy high bytes, second low bytes); the input operand chooses the terms:
//   Phh            A . [xh, 0]
//   -(Phl + Plh + 128 sum Wh)   A . [~xl', ~xh] + A . [-127, 1]
//   -(Pll + 128 sum Wl')        A . [0, ~xl'] + A . [0, -127]
// with ~v = -v - 1, which stays in a signed byte: A . [~xl', ~xh] = -(Phl +
// Plh) - sum Wh - sum Wl', so the constant operand adds -127 sum Wh + sum
// Wl'; likewise for the low bytes.  The two constant products start the
// accumulators, the low one from -128 sum x (one value per sequence, from
// the vector unit).  |Phh| <= 2^18 and the rest fits in 29 bits.
//
// The aligned sum A is formed in float64 with the rounding mode toward minus
// infinity: an accumulator starting at C = 1.5 * 2^(52 + M) has 2^M as the
// unit of its last place, so fma(S, 2^E, acc) is acc + 2^M floor(S 2^(E - M))
// exactly -- one instruction for the shift, the floor and the 64-bit add --
// and A is the difference of the bit patterns of acc and C (|A| <= nT 2^34
// < 2^51, so acc keeps its binade).  S itself is exact in float64 (35 bits:
// fma(Phh, 65536, low part)), and 2^E is built from its exponent field: the
// weights' exponents lie in LDS as 16-bit pairs and the inputs' as a pair of
// one value, biased, so the largest and smallest E of pass 1 are formed two
// rows an instruction and 2^E is one shift-add.  A wave that has a tile with
// M - E > 47 (dropped by the engine) forms its sums with 2^E replaced by 0
// there; without one it skips the test.
//
// Against a 64-bit shift and add per output and operand sets selected per
// copy of the tile, the G/U launch of 64 sequences went from 13.4 to 12.2 us
// (its tile sums from 5.5 to 4.2), Q|K|V 12.6 to 12.4, O 10.3 to 10.1, D 13.5
// to 13.8.  (The input sums by three more products a tile instead of the
// vector unit: G/U 15.9 us, its registers no longer fitting one round.)
//
// A block is NC adjacent 16-row chunks of the device layout by 16
// sequences.  Lane l supplies row / sequence l % 16 and k-group l / 16
// (the tile's 8-element half (l/16) & 1), and owns outputs
// (row 4*(l/16) + v, sequence l % 16), v < 4, of every chunk.  The waves of
// a workgroup split the input tiles; M is reduced with LDS max and A with
// LDS 64-bit adds.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "bfp_device.h"

namespace bfp {

typedef int mx_v4 __attribute__((ext_vector_type(4)));

constexpr int MX_SEQ = 16;    // sequences per block
constexpr int MX_WAVES_MAX = 8;

// High bytes and offset low bytes of the 8 int16 in w (little-endian pairs).
__device__ __forceinline__ void mx_split(const uint4 w, long &hi, long &lo) {
  const unsigned h0 = __builtin_amdgcn_perm(w.y, w.x, 0x07050301u);
  const unsigned h1 = __builtin_amdgcn_perm(w.w, w.z, 0x07050301u);
  const unsigned l0 = __builtin_amdgcn_perm(w.y, w.x, 0x06040200u) ^ 0x80808080u;
  const unsigned l1 = __builtin_amdgcn_perm(w.w, w.z, 0x06040200u) ^ 0x80808080u;
  hi = (long)(((unsigned long)h1 << 32) | h0);
  lo = (long)(((unsigned long)l1 << 32) | l0);
}

__device__ __forceinline__ mx_v4 mx_mfma(long a, long b, mx_v4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0);
}

// The select-free form of one tile's sums (the pipelined batched step,
// bfp_pipe.hip, whose weights are split once per layer).  Every operand carries the tile
// in both k copies, so each 32-deep product is twice the tile's; only the
// per-lane constant k1 (ones in the first copy, zeros in the second) counts
// once.  With P the 32-deep sum and sum x = 256 sum xh + sum xl' + 2048,
//   2 S = 65536 (P(Wh, xh) + P(Wh, k1) + P(k1, xh) + 8)
//         + 256 (P(Wh, xl') + P(Wl', xh) + P(Wl', k1) + P(k1, xl'))
//         + P(Wl', xl')
// and floor(S / 2^d) = floor(2S / 2^(d+1)).  |hh| < 2^20 and the low part
// lo = 256 cr + ll fits 31 bits (tests/test_mx_split.py).  The two input
// sums P(k1, xh) + 8, P(k1, xl') are one pair per tile (mx_xsum), the
// initial accumulators of every chunk's hh and cr (8 is an inline operand
// of the product; 2^19 as the low sum's start would be a register copy per
// tile).
__device__ __forceinline__ long mx_k1() { return (threadIdx.x & 63) < 32 ? 0x0101010101010101L : 0L; }
__device__ __forceinline__ void mx_xsum(long xh, long xl, long k1, mx_v4 &sh, mx_v4 &sl) {
  const mx_v4 zero = {0, 0, 0, 0}, c8 = {8, 8, 8, 8};
  sh = mx_mfma(k1, xh, c8);
  sl = mx_mfma(k1, xl, zero);
}
__device__ __forceinline__ void mx_tile2(long wh, long wl, long xh, long xl, long k1, const mx_v4 &sh,
                                         const mx_v4 &sl, mx_v4 &hh, mx_v4 &lo) {
  const mx_v4 zero = {0, 0, 0, 0};
  hh = mx_mfma(wh, xh, sh);
  mx_v4 cr = mx_mfma(wh, xl, sl);
  const mx_v4 ll = mx_mfma(wl, xl, zero);
  hh = mx_mfma(wh, k1, hh);
  cr = mx_mfma(wl, xh, cr);
  cr = mx_mfma(wl, k1, cr);
#pragma unroll
  for (int v = 0; v < 4; ++v) lo[v] = (cr[v] << 8) + ll[v];
}
// floor(S / 2^d) of a tile from (hh, lo) of mx_tile2 with q = d + 1; WIN:
// 0 past the engine's 47-bit window (d > ALIGN_MAX), without a branch (a
// wave whose every (tile, output) lies inside the window skips the test).
template <bool WIN>
__device__ __forceinline__ long long mx_align2(int hh, int lo, int q) {
  const long long s2 = ((long long)hh << 16) + lo;
  if constexpr (!WIN) return s2 >> q;
  const long long t = s2 >> (q & 63);
  return q <= ALIGN_MAX + 1 ? t : 0;
}

// Phase stamps of a traced batched decode (100 MHz clock, thread 0 of each
// block): MX_TRACE_STAMPS per block -- 0 entry, 1 exponents staged, 2 M
// reduced, 3 tile sums formed, 4 A reduced, 5 epilogue done (stamped by the
// kernel) -- for at most MX_TRACE_BLOCKS blocks of each of the MX_TRACE_KERNELS
// matvec kernels (MX_K_*), the last launch of each kind overwriting the one
// before.
constexpr int MX_TRACE_STAMPS = 6, MX_TRACE_BLOCKS = 1024, MX_TRACE_KERNELS = 4;
constexpr int MX_K_QKV = 0, MX_K_O = 1, MX_K_GU = 2, MX_K_D = 3;
__device__ __forceinline__ void mx_mark(unsigned long long *tr, int k) {
  const unsigned b = blockIdx.x + blockIdx.y * gridDim.x;
  if (tr && threadIdx.x == 0 && b < (unsigned)MX_TRACE_BLOCKS)
    tr[b * MX_TRACE_STAMPS + k] = __builtin_amdgcn_s_memrealtime();
}

// LDS bytes mx_block<NC> needs beyond its caller's Ao / Mo: the block's
// weight exponents as 16-bit values, tile-major, and the input exponents as
// pairs of one 16-bit value.
__host__ __device__ constexpr int mx_lds_bytes(int nc, int nT) { return (nc * 32 + 64) * nT; }

typedef short mx_s2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ mx_s2 mx_pair(int v) { return __builtin_bit_cast(mx_s2, v); }
__device__ __forceinline__ int mx_bits(mx_s2 v) { return __builtin_bit_cast(int, v); }

// The float64 rounding mode of the wave: toward minus infinity, or nearest.
// Volatile statements keep their order among themselves, but nothing orders
// ordinary float64 operations against them: between the two only exact ones
// may stand (the conversions and S below).  tests/test_mx_rounding_code.py
// reads the built kernels for that.
__device__ __forceinline__ void mx_round_down() {
  asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 2\n\ts_nop 1");
}
__device__ __forceinline__ void mx_round_nearest() {
  asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0\n\ts_nop 1");
}
// acc = s * scale + acc under the mode set by mx_round_down (volatile: not
// moved across the mode changes).
__device__ __forceinline__ void mx_fma_down(double &acc, double s, double scale) {
  asm volatile("v_fma_f64 %0, %1, %2, %0" : "+v"(acc) : "v"(s), "v"(scale));
}

// (A, M) of the (row, sequence) pairs of a block: the NC adjacent 16-row
// chunks at pm / pe (device layout, nT tiles each; chunk c is rows
// 16c..16c+15) against sequences s < ns at x_m + s*nT*16, x_e + s*nT.
// Every thread of the workgroup calls it; on return (after a barrier)
// Ao[row*16 + s] and Mo[row*16 + s] (LDS) hold the pair of (row, s).
// ex: mx_lds_bytes(NC, nT) bytes of LDS.
template <int NC>
__device__ __forceinline__ void mx_block(const uint4 *__restrict__ pm, const int8_t *__restrict__ pe, int nT,
                         const int16_t *__restrict__ xm, const int8_t *__restrict__ xe, int ns,
                         long long *Ao, int *Mo, int8_t *ex, unsigned long long *tr = nullptr) {
  mx_mark(tr, 0);
  constexpr int G = 4;           // tiles whose loads are in flight together
  constexpr int RW = NC * 16;    // rows of the block
  constexpr int EB = 128;        // bias of a stored exponent
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int i = lane & 15, kg = lane >> 4, h = kg & 1;
  const bool first = kg < 2;     // first copy of the tile on the k axis
  const int sc = i < ns ? i : ns - 1;
  const uint4 *xr = reinterpret_cast<const uint4 *>(xm);
  const int wo = h * 16 + i, xo = sc * nT * 2 + h;   // + t*32 (+ c*nT*32), + t*2
  int16_t *wex = reinterpret_cast<int16_t *>(ex);    // [t*RW + row]
  int *xex = reinterpret_cast<int *>(wex + RW * nT); // [t*16 + sequence]
  const int tpw = (nT + nw - 1) / nw;
  const int t0 = w * tpw, t1 = t0 + tpw < nT ? t0 + tpw : nT;
  // operand registers of G tiles, loaded together (the last valid tile
  // stands in for those past t1: in range, never used).  Issuing the first
  // group's loads with the exponent loads measured slower for every kernel
  // (G/U 14.4 -> 15.6 us, D 11.0 -> 13.0 at batch 64).
  uint4 xv[G], wv[G][NC];
  auto load_group = [&](int tb) {
#pragma unroll
    for (int k = 0; k < G; ++k) {
      const int t = tb + k < t1 ? tb + k : t1 - 1;
      xv[k] = xr[xo + t * 2];
#pragma unroll
      for (int c = 0; c < NC; ++c) wv[k][c] = pm[wo + c * nT * 32 + t * 32];
    }
  };
  // exponents of the whole block into LDS, biased: the weights' as 4-row
  // words of 16-bit values, the inputs' as pairs, every load of a thread
  // issued before its stores
  {
    const int nw4 = NC * nT * 4, nx = MX_SEQ * nT, bs = blockDim.x;
    const int *pe4 = reinterpret_cast<const int *>(pe);
    for (int q0 = threadIdx.x; q0 < nw4 + nx; q0 += 4 * bs) {
      int v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int q = q0 + k * bs;
        if (q < nw4) {
          v[k] = pe4[q];
        } else {
          int qx = q - nw4;
          qx = qx < nx ? qx : nx - 1;
          const int t = qx >> 4, ss = qx & 15;
          v[k] = xe[(ss < ns ? ss : ns - 1) * nT + t];
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int q = q0 + k * bs;
        if (q < nw4) {
          // word q: chunk q / (4nT), tile (q / 4) % nT, rows 4*(q%4) .. +3;
          // a signed byte plus 128 is the byte with its sign bit flipped
          const int c = q / (4 * nT), t = (q >> 2) - c * nT;
          const unsigned u = (unsigned)v[k] ^ 0x80808080u;
          *reinterpret_cast<int2 *>(wex + t * RW + c * 16 + 4 * (q & 3)) =
              make_int2((int)__builtin_amdgcn_perm(0, u, 0x0c010c00u), (int)__builtin_amdgcn_perm(0, u, 0x0c030c02u));
        } else if (q < nw4 + nx) {
          xex[q - nw4] = (v[k] + EB) * 0x10001;
        }
      }
    }
  }
  for (int q = threadIdx.x; q < RW * MX_SEQ; q += blockDim.x) {
    Ao[q] = 0;
    Mo[q] = -(1 << 29);
  }
  __syncthreads();
  mx_mark(tr, 1);
  // (W_e + x_e, biased by 2 EB) of chunk c, tile t for this lane's outputs
  // (rows 4 kg + v, sequence i), two rows a pair
  auto tile_E = [&](int c, int t, mx_s2 (&E)[2]) {
    const int2 ww = *reinterpret_cast<const int2 *>(wex + t * RW + c * 16 + 4 * kg);
    const mx_s2 xp = mx_pair(xex[t * 16 + i]);
    E[0] = mx_pair(ww.x) + xp;
    E[1] = mx_pair(ww.y) + xp;
  };
  // pass 1: M over all tiles, split across the waves, reduced in LDS; and
  // the smallest E of this wave's tiles
  int M[NC][4];
  mx_s2 Emin[NC][2];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    mx_s2 mx[2];
    mx[0] = mx[1] = mx_s2{0, 0};
    Emin[c][0] = Emin[c][1] = mx_s2{1024, 1024};
#pragma unroll 4
    for (int t = t0; t < t1; ++t) {
      mx_s2 E[2];
      tile_E(c, t, E);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        mx[p] = __builtin_elementwise_max(mx[p], E[p]);
        Emin[c][p] = __builtin_elementwise_min(Emin[c][p], E[p]);
      }
    }
    if (t0 < t1) {
#pragma unroll
      for (int v = 0; v < 4; ++v) atomicMax(&Mo[(c * 16 + 4 * kg + v) * MX_SEQ + i], (int)mx[v >> 1][v & 1] - 2 * EB);
    }
  }
  __syncthreads();
  mx_mark(tr, 2);
  // accumulators at C = 1.5 * 2^(52 + M)
  double A[NC][4];
  bool far = false;   // a tile past the engine's 47-bit window
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      M[c][v] = Mo[(c * 16 + 4 * kg + v) * MX_SEQ + i];
      A[c][v] = __hiloint2double(((1075 + M[c][v]) << 20) | 0x80000, 0);
      far = far || M[c][v] + 2 * EB - (int)Emin[c][v >> 1][v & 1] > ALIGN_MAX;
    }
  // pass 2: aligned tile sums.  Byte selectors of v_perm_b32 over (second
  // dword, first dword) of 4 int16: high bytes, low bytes, zeros
  const unsigned HI = 0x07050301u, LO = 0x06040200u, ZR = 0x0c0c0c0cu;
  const unsigned sA = first ? HI : LO, mA = first ? 0u : 0x80808080u;       // [Wh, Wl']
  const unsigned sH = first ? HI : ZR;                                      // [xh, 0]
  const unsigned sC = first ? LO : HI, mC = first ? 0x7f7f7f7fu : ~0u;      // [~xl', ~xh]
  const unsigned sL = first ? ZR : LO, mL = first ? 0u : 0x7f7f7f7fu;       // [0, ~xl']
  auto planes = [](const uint4 &v, unsigned sel, unsigned mask) {
    const unsigned lo = __builtin_amdgcn_perm(v.y, v.x, sel) ^ mask, hi = __builtin_amdgcn_perm(v.w, v.z, sel) ^ mask;
    return (long)(((unsigned long)hi << 32) | lo);
  };
  const long kC = first ? (long)0x8181818181818181ull : 0x0101010101010101L;   // [-127, 1]
  const long kL = first ? 0L : (long)0x8181818181818181ull;                    // [0, -127]
  const mx_v4 zero = {0, 0, 0, 0};
  auto tiles = [&](auto window) {
    constexpr bool WIN = decltype(window)::value;
    for (int tb = t0; tb < t1; tb += G) {
      load_group(tb);
#pragma unroll
      for (int k = 0; k < G; ++k) {
        if (tb + k >= t1) break;
        const long xh = planes(xv[k], sH, 0u), xc = planes(xv[k], sC, mC), xl = planes(xv[k], sL, mL);
        // -128 sum x: this half's, then the tile's other half (k-group kg ^ 1)
        int sx = 0;
        const mx_s2 m128 = {-128, -128};
        sx = __builtin_amdgcn_sdot2(mx_pair((int)xv[k].x), m128, sx, false);
        sx = __builtin_amdgcn_sdot2(mx_pair((int)xv[k].y), m128, sx, false);
        sx = __builtin_amdgcn_sdot2(mx_pair((int)xv[k].z), m128, sx, false);
        sx = __builtin_amdgcn_sdot2(mx_pair((int)xv[k].w), m128, sx, false);
        const auto sw = __builtin_amdgcn_permlane16_swap(sx, sx, false, false);
        const int cx = (int)(sw[0] + sw[1]);
        const mx_v4 cxv = {cx, cx, cx, cx};
        const int xp = xex[(tb + k) * 16 + i];
        // high word of 2^E is (1023 - 2 EB + W_e' + x_e') << 20 (a pair shifted
        // left by 20 keeps its low value)
        const int xs = (xp << 20) + ((1023 - 2 * EB) << 20);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const long wa = planes(wv[k][c], sA, mA);
          mx_v4 cr = mx_mfma(wa, kC, zero);
          mx_v4 ll = mx_mfma(wa, kL, cxv);
          const mx_v4 hh = mx_mfma(wa, xh, zero);
          cr = mx_mfma(wa, xc, cr);
          ll = mx_mfma(wa, xl, ll);
          const int2 ww = *reinterpret_cast<const int2 *>(wex + (tb + k) * RW + c * 16 + 4 * kg);
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int wp = v < 2 ? ww.x : ww.y;
            int se = (v & 1) ? (int)((unsigned)wp >> 16 << 20) + xs : (wp << 20) + xs;
            if constexpr (WIN) {
              const int E = (int)((unsigned)se >> 20) - 1023;
              se = M[c][v] - E > ALIGN_MAX ? 0 : se;
            }
            const int lo = (cr[v] << 8) + ll[v];   // - (low part of S)
            const double S = fma((double)hh[v], 65536.0, -(double)lo);
            mx_fma_down(A[c][v], S, __hiloint2double(se, 0));
          }
        }
      }
    }
  };
  mx_round_down();
  if (__builtin_expect(__any(far), 0)) tiles(std::true_type{});
  else tiles(std::false_type{});
  mx_round_nearest();
  mx_mark(tr, 3);
  if (t0 < t1) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long long a = __double_as_longlong(A[c][v]) -
                            ((long long)(((1075 + M[c][v]) << 20) | 0x80000) << 32);
        atomicAdd(reinterpret_cast<unsigned long long *>(&Ao[(c * 16 + 4 * kg + v) * MX_SEQ + i]),
                  (unsigned long long)a);
      }
  }
  __syncthreads();
  mx_mark(tr, 4);
}

// A read back for an epilogue, clipped as the engine clips.
__device__ __forceinline__ long long mx_A(const long long *Ao, int q) {
  const long long A = Ao[q];
  return A < SAT_LO ? SAT_LO : (A > SAT_HI ? SAT_HI : A);
}

}  // namespace bfp
