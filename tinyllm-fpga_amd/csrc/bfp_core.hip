// Core BFP kernels for gfx950: device weight layout, tile quantisation and
// the exact-integer BFP matvec, plus their C-ABI launchers (include/bfp.h).
//
// Device weight layout (this build's own; the reference's DDR3 image is the
// 16-lane "wide" layout of gen_smollm_blockfp_ddr.py:88-119).  A matrix of
// n_out rows is cut into 16-row chunks (full.py's LANES=16 chunks).  Within a
// chunk the 16 x nT tiles are stored tile-major, each tile as two 256-byte
// half-planes:
//     mantissas: byte ((c*nT + t)*2 + h)*256 + r*16 holds
//                W_m[c*16 + r][t][8h .. 8h+7]   (8 x int16)
//     exponents: byte (c*nT + t)*16 + r holds W_e[c*16 + r][t]
// so a wave whose lanes are (row r = lane%16, tile t0 + lane/16) reads four
// fully used 256-byte runs per 16-byte-per-lane load.
#include <stdarg.h>
#include <stdlib.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <climits>

#include "bfp.h"
#include "bfp_device.h"
#include "bfp_internal.h"
#include "bfp_mv.h"

namespace bfp {

// ------------------------------------------------------------------ errors
static thread_local char g_err[1024] = "";

int set_err(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

const char *last_error() { return g_err; }

// ------------------------------------------------------------------ layout
// Source chunk c goes to destination chunk c*cstride (cstride 2 interleaves
// two matrices chunk by chunk).
__global__ void pack_m_kernel(const int16_t *__restrict__ Wm, long long total, int nT,
                              int cstride, uint4 *__restrict__ Pm) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  int r = (int)(i & 15), h = (int)((i >> 4) & 1);
  long long ct = i >> 5;
  long long c = ct / nT;
  int t = (int)(ct % nT);
  Pm[((c * cstride) * nT + t) * 32 + h * 16 + r] =
      *reinterpret_cast<const uint4 *>(Wm + ((c * 16 + r) * nT + t) * 16 + h * 8);
}

__global__ void pack_e_kernel(const int8_t *__restrict__ We, long long total, int nT,
                              int cstride, int8_t *__restrict__ Pe) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  int r = (int)(i & 15);
  long long ct = i >> 4;
  long long c = ct / nT;
  int t = (int)(ct % nT);
  Pe[((c * cstride) * nT + t) * 16 + r] = We[(c * 16 + r) * nT + t];
}

__global__ void unpack_m_kernel(const uint4 *__restrict__ Pm, long long total, int nT,
                                int16_t *__restrict__ Wm) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  int r = (int)(i & 15), h = (int)((i >> 4) & 1);
  long long ct = i >> 5;
  long long c = ct / nT;
  int t = (int)(ct % nT);
  *reinterpret_cast<uint4 *>(Wm + ((c * 16 + r) * nT + t) * 16 + h * 8) = Pm[i];
}

__global__ void unpack_e_kernel(const int8_t *__restrict__ Pe, long long total, int nT,
                                int8_t *__restrict__ We) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  int r = (int)(i & 15);
  long long ct = i >> 4;
  long long c = ct / nT;
  int t = (int)(ct % nT);
  We[(c * 16 + r) * nT + t] = Pe[i];
}

// ------------------------------------------------------------ quantisation
// One thread per 16-element tile.  EXACT: the encoding of values that are
// already BFP (decoded tiles, as the reference's float64 arrays hold them):
// tile_quantize's (canonical) tile, unless it rounds a value, in which case
// the tile with exponent one lower is taken when it holds every value
// exactly -- the raw form of a tile whose largest magnitude is the mantissa
// -32768 (value -2^e), which tile_quantize maps to exponent e + 1 and
// rounds odd mantissas.  Values that are not BFP-exact either way get
// tile_quantize's tile.
template <typename T, bool EXACT = false>
__global__ void tile_quantize_kernel(const T *__restrict__ v, long long n_tiles,
                                     int16_t *__restrict__ m, int8_t *__restrict__ e,
                                     int *__restrict__ inexact = nullptr) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n_tiles) return;
  double x[TILE];
  double amax = 0.0;
#pragma unroll
  for (int k = 0; k < TILE; ++k) {
    x[k] = (double)v[i * TILE + k];
    amax = fmax(amax, fabs(x[k]));
  }
  int ex = tile_exp_of(amax);
  int mm[TILE];
#pragma unroll
  for (int k = 0; k < TILE; ++k) mm[k] = tile_mant_of(x[k], ex);
  if constexpr (EXACT) {
    bool same = true;
#pragma unroll
    for (int k = 0; k < TILE; ++k) same = same && ldexp((double)mm[k], ex - 15) == x[k];
    if (!same) {
      bool raw = ex > -127;
      int rm[TILE];
#pragma unroll
      for (int k = 0; k < TILE; ++k) {
        const double s = ldexp(x[k], 16 - ex);
        raw = raw && s == rint(s) && s >= -32768.0 && s <= 32767.0;
        rm[k] = raw ? (int)s : 0;
      }
      if (raw) {
        --ex;
#pragma unroll
        for (int k = 0; k < TILE; ++k) mm[k] = rm[k];
      } else if (inexact) {
        *inexact = 1;   // not BFP-exact: tile_quantize's tile stands
      }
    }
  }
  uint4 lo, hi;
  lo.x = (mm[0] & 0xffff) | (mm[1] << 16);
  lo.y = (mm[2] & 0xffff) | (mm[3] << 16);
  lo.z = (mm[4] & 0xffff) | (mm[5] << 16);
  lo.w = (mm[6] & 0xffff) | (mm[7] << 16);
  hi.x = (mm[8] & 0xffff) | (mm[9] << 16);
  hi.y = (mm[10] & 0xffff) | (mm[11] << 16);
  hi.z = (mm[12] & 0xffff) | (mm[13] << 16);
  hi.w = (mm[14] & 0xffff) | (mm[15] << 16);
  uint4 *dst = reinterpret_cast<uint4 *>(m + i * TILE);
  dst[0] = lo;
  dst[1] = hi;
  e[i] = (int8_t)ex;
}

// quantize_W straight into the device layout.  Bound by memory: 4 bytes in
// and 2 1/16 out an element.  A wave takes two tiles of 16 rows (a chunk), in
// the layout's order, with four elements a lane, so that each instruction
// covers whole lines on both sides: a load 8 rows of 128 bytes, a store four
// runs of 8 rows by 16 bytes (one tile's half of 8 columns).  With an odd
// number of tiles a row a pair runs on into the next chunk.  49152 x 576: 28.5
// us a call (6.0 TB/s); a thread a tile, with lanes 64 bytes apart on the way
// in and 512 on the way out, took 32.6.  Small tables want the waves: with
// four pairs a wave 49152 x 80 took 6.1 us and x 400 24.4, so 4.9 and 22.1
// (every call back to back has 4 us of launch in it).
// The arithmetic is tile_exp_of's and tile_mant_of's on float32 values, in
// float32 and bit for bit the same: scaling by a power of two is exact (a
// result below the normal range rounds to 0 either way), and no float32 amax
// lies within 709 * 2^-53 below a power of two, so the exponent is frexp's.
__device__ __forceinline__ float quad_max(float v) {
  const int i = __float_as_int(v);
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, i, 0xB1, 0xf, 0xf, false)));   // lane ^ 1
  const int j = __float_as_int(v);
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, j, 0x4E, 0xf, 0xf, false)));  // lane ^ 2
}

__global__ __launch_bounds__(256) void quantize_pack_f32_kernel(const float *__restrict__ W, unsigned tiles,
                                                                unsigned nT, int cstride, uint2 *__restrict__ Pm,
                                                                int8_t *__restrict__ Pe) {
  const int l = threadIdx.x & 63;
  // lane: row 8j + (l >> 3) of the chunk, elements 4 (l & 3) .. of the pair's tile (l >> 2) & 1
  const unsigned blk = blockIdx.y * gridDim.x + blockIdx.x;
  const unsigned q = 2 * __builtin_amdgcn_readfirstlane(blk * 4 + (threadIdx.x >> 6)), odd = (l >> 2) & 1;
  const unsigned c0 = q / nT, t0 = q - c0 * nT + odd;
  const unsigned c = t0 < nT ? c0 : c0 + 1, t = t0 < nT ? t0 : 0;
  const bool live = q + odd < tiles;
  float4 f[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    f[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (live)
      f[j] = ld_nt(reinterpret_cast<const float4 *>(W + (((long long)c * 16 + 8 * j + (l >> 3)) * nT + t) * TILE +
                                                    4 * (l & 3)));
  }
  const long long ct = (long long)c * cstride * nT + t;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float x[4] = {f[j].x, f[j].y, f[j].z, f[j].w};
    float amax = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) amax = fmaxf(amax, fabsf(x[k]));
    amax = quad_max(amax);
    int ex = -127;
    if (amax > 0.f) {
      frexp((double)amax, &ex);
      ex = ex < -127 ? -127 : (ex > 127 ? 127 : ex);
    }
    int mm[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) mm[k] = (int)fminf(fmaxf(rintf(ldexpf(x[k], 15 - ex)), -32768.f), 32767.f);
    const int r = 8 * j + (l >> 3), h = (l >> 1) & 1;
    if (live) {
      Pm[((ct * 2 + h) * 16 + r) * 2 + (l & 1)] =
          make_uint2((mm[0] & 0xffff) | (mm[1] << 16), (mm[2] & 0xffff) | (mm[3] << 16));
      if ((l & 3) == 0) Pe[ct * 16 + r] = (int8_t)ex;
    }
  }
}

// The reference's wide layout (gen_smollm_blockfp_ddr.py:88-119, the DDR3
// image and the *_m.hex/_e.hex sets of gen_smollm_blockfp_full.py:131-161):
// mantissa entry (chunk, col) = 16 lanes (rows chunk*16 .. +15) x int16 LE,
// exponent entry (chunk, tile) = 16 lanes x int8.  Repacked into this
// build's device layout; source chunk c goes to destination chunk c*cstride.
// The exponent entries are already in the device order (per chunk and tile,
// one byte per row).
__global__ void pack_wide_m_kernel(const int16_t *__restrict__ Wm, long long total, int nT,
                                   int cstride, uint4 *__restrict__ Pm) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int r = (int)(i & 15), h = (int)((i >> 4) & 1);
  const long long ct = i >> 5;
  const long long c = ct / nT;
  const int t = (int)(ct % nT);
  const int16_t *src = Wm + (c * nT * 16 + t * 16 + 8 * h) * 16 + r;   // col t*16 + 8h, lane r
  unsigned v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    v[k] = ((unsigned)(unsigned short)src[(2 * k) * 16]) |
           ((unsigned)(unsigned short)src[(2 * k + 1) * 16] << 16);
  Pm[((c * cstride) * nT + t) * 32 + h * 16 + r] = make_uint4(v[0], v[1], v[2], v[3]);
}

__global__ void pack_wide_e_kernel(const int8_t *__restrict__ We, long long total, int nT,
                                   int cstride, int8_t *__restrict__ Pe) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= total) return;
  const long long ct = i >> 4;
  const long long c = ct / nT;
  const int t = (int)(ct % nT);
  Pe[((c * cstride) * nT + t) * 16 + (i & 15)] = We[i];
}

__global__ void tile_decode_kernel(const int16_t *__restrict__ m, const int8_t *__restrict__ e,
                                   long long n, double *__restrict__ v) {
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  v[i] = ldexp((double)m[i], (int)e[i >> 4] - 15);
}

// ------------------------------------------------------------------ matvec
// Output stores of the standalone matvec.  A few scattered partial-line
// writes per workgroup cost the streaming read several percent (a 64-byte
// store per 36 KB one-shot workgroup read: 6.6-6.7 TB/s against 7.2 without
// it); as dwords with the non-temporal policy the cost mostly goes (7.0).
// 2-byte stores with that policy were slower than plain ones.
// Lanes 0-15 hold rows 0-15 (m); the 16 mantissas go out as 8 dwords of row
// pairs when yr is 4-byte aligned.
__device__ __forceinline__ void store_rows16(int16_t *yr, int m, int lane) {
  if ((reinterpret_cast<uintptr_t>(yr) & 3) == 0) {
    const int src = (lane & 7) * 2;
    const int a = __shfl(m, src, 64), b = __shfl(m, src + 1, 64);
    const unsigned w = ((unsigned)a & 0xffffu) | ((unsigned)b << 16);
    if (lane < 8) __builtin_nontemporal_store(w, reinterpret_cast<unsigned *>(yr) + lane);
  } else if (lane < 16) {
    yr[lane] = (int16_t)m;
  }
}

// Standalone matvec: one 16-row chunk of one problem per workgroup (the
// engine and its exactness argument are in bfp_mv.h).  Problem r reads
// matrix (r mod ring) when ring > 0.  BUF: the weights through buffer
// loads (load_chunk_buf).
template <int NW, int TPT, bool BUF = false>
__global__ __launch_bounds__(64 * NW) void matvec_kernel(
    const uint4 *__restrict__ Pm, const int8_t *__restrict__ Pe, long long smat_m,
    long long smat_e, int nT, int n_chunks, int ring, const int16_t *__restrict__ xm,
    const int8_t *__restrict__ xe, long long x_stride, int16_t *__restrict__ ym,
    int8_t *__restrict__ ye, long long y_stride, int cstride) {
  extern __shared__ int smem[];
  int *xs = smem;              // nT * 16
  int *xes = smem + nT * 16;   // nT
  __shared__ int redM[NW * 16];
  __shared__ long long redA[NW * 16];

  const int mat = blockIdx.x / n_chunks;
  const int c = blockIdx.x - mat * n_chunks;
  const int wmat = ring > 0 ? mat % ring : mat;

  ChunkRegs<TPT> R;
  const long long cc = (long long)c * cstride;   // chunk c of this matrix in the layout
  if constexpr (BUF)
    load_chunk_buf<NW, TPT>(R, Pm + wmat * smat_m + cc * nT * 32, Pe + wmat * smat_e + cc * nT * 16,
                            nT);
  else
    load_chunk<NW, TPT, true>(R, Pm + wmat * smat_m + cc * nT * 32, Pe + wmat * smat_e + cc * nT * 16,
                              nT);
  stage_x_bfp(xs, xes, xm + mat * x_stride, xe + mat * (x_stride / 16), nT);
  __syncthreads();
  long long A;
  int M;
  chunk_AM<NW, TPT>(R, xs, xes, nT, redM, redA, A, M);
  if (threadIdx.x < 64) {
    int m, e;
    chunk_quant(A, M, m, e);
    const int lane = threadIdx.x;
    store_rows16(ym + mat * y_stride + c * 16, m, lane);
    if (lane == 0) ye[mat * (y_stride / 16) + c] = (int8_t)e;
  }
}

// Two adjacent 16-row chunks of one problem per workgroup: both chunks'
// weight loads are issued before any arithmetic, and one pass (chunk_AM2)
// forms both chunks' rows, so a workgroup streams twice the bytes per
// barrier round.  n_chunks is even.  On 576-input chunks (three waves) this
// streamed 7.11 TB/s on the 49152 x 576 sweep against 6.80 for one chunk per
// workgroup; on the 1536-input chunk (eight waves) it was slower (6.42
// against 6.63), so that shape keeps one chunk per workgroup.
template <int NW, int TPT>
__global__ __launch_bounds__(64 * NW) void matvec2_kernel(
    const uint4 *__restrict__ Pm, const int8_t *__restrict__ Pe, long long smat_m,
    long long smat_e, int nT, int n_chunks, int ring, const int16_t *__restrict__ xm,
    const int8_t *__restrict__ xe, long long x_stride, int16_t *__restrict__ ym,
    int8_t *__restrict__ ye, long long y_stride, int cstride) {
  extern __shared__ int smem[];
  int *xs = smem;              // nT * 16
  int *xes = smem + nT * 16;   // nT
  __shared__ int redM[2 * NW * 16];
  __shared__ long long redA[2 * NW * 16];
  const int pairs = n_chunks / 2;
  const int mat = blockIdx.x / pairs;
  const int c = 2 * (blockIdx.x - mat * pairs);
  const int wmat = ring > 0 ? mat % ring : mat;
  ChunkRegs<TPT> R1, R2;
  const long long c1 = (long long)c * cstride, c2 = (long long)(c + 1) * cstride;
  load_chunk<NW, TPT, true>(R1, Pm + wmat * smat_m + c1 * nT * 32, Pe + wmat * smat_e + c1 * nT * 16, nT);
  load_chunk<NW, TPT, true>(R2, Pm + wmat * smat_m + c2 * nT * 32, Pe + wmat * smat_e + c2 * nT * 16, nT);
  stage_x_bfp(xs, xes, xm + mat * x_stride, xe + mat * (x_stride / 16), nT);
  __syncthreads();
  long long A1, A2;
  int M1, M2;
  chunk_AM2<NW, TPT>(R1, R2, xs, xes, nT, redM, redA, A1, M1, A2, M2);
  if (threadIdx.x < 64) {
    int m1, e1, m2, e2;
    chunk_quant(A1, M1, m1, e1);
    chunk_quant(A2, M2, m2, e2);
    const int lane = threadIdx.x;
    int16_t *yr = ym + mat * y_stride + c * 16;   // 32 contiguous mantissas
    if ((reinterpret_cast<uintptr_t>(yr) & 3) == 0) {
      // as 16 dwords of row pairs with non-temporal stores (store_rows16):
      // lane L writes rows 2L, 2L + 1 of the pair (chunk c for L < 8, chunk
      // c + 1 above)
      const int src = (lane & 7) * 2;
      const int a1 = __shfl(m1, src, 64), b1 = __shfl(m1, src + 1, 64);
      const int a2 = __shfl(m2, src, 64), b2 = __shfl(m2, src + 1, 64);
      const int lo = lane < 8 ? a1 : a2, hi = lane < 8 ? b1 : b2;
      const unsigned w = ((unsigned)lo & 0xffffu) | ((unsigned)hi << 16);
      if (lane < 16) __builtin_nontemporal_store(w, reinterpret_cast<unsigned *>(yr) + lane);
    } else if (lane < 16) {
      yr[lane] = (int16_t)m1;
      yr[16 + lane] = (int16_t)m2;
    }
    if (lane == 0) {
      ye[mat * (y_stride / 16) + c] = (int8_t)e1;
      ye[mat * (y_stride / 16) + c + 1] = (int8_t)e2;
    }
  }
}

// Read-only streaming probe: workgroup w reads the contiguous range
// [w*per, (w+1)*per) of 16-byte words through a buffer resource over that
// range (four loads in flight per thread; loads past its end read 0, so
// there is no branch around a load), folded into one word per workgroup that
// is stored only when it equals a fixed sentinel, so the loads cannot be
// dropped.  NT: the loads carry the non-temporal cache
// policy (bit 1 of the policy operand), as the matvec's weight stream does.
// Measures the practical HBM read ceiling the matvec is compared with; with
// per = 1024 (16 KB per workgroup, every workgroup resident at once on a
// 4 GiB read) this measured 7.3-7.4 TB/s, against 7.1-7.2 for a few
// workgroups per CU each streaming a long range.
template <bool NT>
__global__ __launch_bounds__(256) void probe_read_kernel(const uint4 *__restrict__ p,
                                                         long long n16, long long per,
                                                         unsigned *__restrict__ out) {
  typedef unsigned v4u __attribute__((ext_vector_type(4)));
  constexpr int POL = NT ? 2 : 0;
  const long long i0 = blockIdx.x * per;
  const int n = (int)(i0 + per < n16 ? per : n16 - i0);
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint4 *>(p + i0), (short)0, n * 16, 0x00020000);
  unsigned acc = 0;
  for (int b = 0; b < n; b += 4 * 256) {
    v4u v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = __builtin_amdgcn_raw_buffer_load_b128(r, (b + k * 256 + (int)threadIdx.x) * 16, 0, POL);
#pragma unroll
    for (int k = 0; k < 4; ++k) acc ^= v[k].x ^ v[k].y ^ v[k].z ^ v[k].w;
  }
  // The compare keeps the loads live without a store per workgroup: one
  // 4-byte store per 16 KB workgroup cost 4% of the read rate (the lines
  // written are shared by workgroups on different XCDs).
  if (acc == 0x9E3779B9u) out[blockIdx.x] = acc;
}

// Narrow embedding rows of n token ids, one workgroup per id: the mantissa
// row as 16-byte words, the exponent bytes from a row of e_row bytes.
__global__ __launch_bounds__(128) void embed_gather_kernel(const uint4 *__restrict__ lu_m,
                                                           const int8_t *__restrict__ lu_e,
                                                           int vocab, int D, int e_row,
                                                           const int32_t *__restrict__ ids,
                                                           uint4 *__restrict__ out_m,
                                                           int8_t *__restrict__ out_e) {
  const int r = blockIdx.x;
  const int id = ids[r];
  const bool ok = id >= 0 && id < vocab;
  const int w = D / 8;  // 16-byte words per mantissa row
  for (int i = threadIdx.x; i < w; i += blockDim.x)
    out_m[(long long)r * w + i] = ok ? lu_m[(long long)id * w + i] : make_uint4(0, 0, 0, 0);
  for (int t = threadIdx.x; t < D / 16; t += blockDim.x)
    out_e[(long long)r * (D / 16) + t] = ok ? lu_e[(long long)id * e_row + t] : (int8_t)-127;
}

typedef void (*matvec_fn)(const uint4 *, const int8_t *, long long, long long, int, int, int,
                          const int16_t *, const int8_t *, long long, int16_t *, int8_t *,
                          long long, int);

template <int NW>
static matvec_fn pick_tpt(int tpt) {
  if (tpt <= 1) return matvec_kernel<NW, 1>;
  if (tpt <= 2) return matvec_kernel<NW, 2>;
  if (tpt <= 3) return matvec_kernel<NW, 3>;
  if (tpt <= 4) return matvec_kernel<NW, 4>;
  if (tpt <= 6) return matvec_kernel<NW, 6>;
  if (tpt <= 8) return matvec_kernel<NW, 8>;
  if (tpt <= 12) return matvec_kernel<NW, 12>;
  if (tpt <= 16) return matvec_kernel<NW, 16>;
  if (tpt <= 24) return matvec_kernel<NW, 24>;
  return nullptr;
}

static matvec_fn pick_matvec(int nw, int tpt) {
  switch (nw) {
    case 1: return pick_tpt<1>(tpt);
    case 2: return pick_tpt<2>(tpt);
    case 3: return pick_tpt<3>(tpt);
    case 4: return pick_tpt<4>(tpt);
    case 6: return pick_tpt<6>(tpt);
    case 8: return pick_tpt<8>(tpt);
    case 9: return pick_tpt<9>(tpt);
    default: return nullptr;
  }
}

int default_waves(int nT) {
  // about three tiles per lane, at most 9 waves
  int nw = (nT + 11) / 12;
  static const int allowed[] = {1, 2, 3, 4, 6, 8, 9};
  for (int a : allowed)
    if (a >= nw) return a;
  return 9;
}


int launch_matvec(const void *P_m, const void *P_e, int n_out, int n_in, int n_mats, int ring,
                  long long smat_m, long long smat_e, const int16_t *x_m, const int8_t *x_e,
                  long long x_stride, int16_t *y_m, int8_t *y_e, long long y_stride, int waves,
                  hipStream_t stream, int cstride) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16 || n_mats <= 0 || ring < 0 ||
      cstride < 1)
    return set_err(BFP_EINVAL, "matvec: bad shape n_out=%d n_in=%d n_mats=%d ring=%d", n_out,
                   n_in, n_mats, ring);
  if (!P_m || !P_e || !x_m || !x_e || !y_m || !y_e)
    return set_err(BFP_EINVAL, "matvec: null pointer");
  if (smat_m % 16 || x_stride % 16 || y_stride % 16)
    return set_err(BFP_EINVAL, "matvec: strides must be multiples of 16");
  const int nT = n_in / 16;
  const int nw = waves > 0 ? waves : default_waves(nT);
  const int tpt = (nT + 4 * nw - 1) / (4 * nw);
  matvec_fn fn = pick_matvec(nw, tpt);
  if (!fn)
    return set_err(BFP_EINVAL, "matvec: no kernel for n_in=%d with %d waves (tiles/lane=%d)",
                   n_in, nw, tpt);
  const int n_chunks = n_out / 16;
  long long blocks = (long long)n_chunks * n_mats;
  if (nw == 3 && tpt == 3 && n_chunks % 2 == 0) {
    fn = matvec2_kernel<3, 3>;
    blocks /= 2;
  } else if (nw == 8 && tpt == 3) {
    fn = matvec_kernel<8, 3, true>;
  }
  if (blocks > INT_MAX) return set_err(BFP_EINVAL, "matvec: grid too large");
  size_t shm = (size_t)nT * 17 * sizeof(int);
  if (shm > 60 * 1024) return set_err(BFP_EINVAL, "matvec: n_in=%d too large", n_in);
  // One 16-row chunk (two on 576-input shapes) of one problem per
  // workgroup, for every batch length: the workgroups run in order, so a
  // batch walks its problems (and a ring of weight copies) in sequence.  (A fixed grid in which each workgroup
  // streamed a contiguous range of chunks measured 5.5 TB/s on HBM-resident
  // weights against this form's 6.8.)
  hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3(64 * nw), shm, stream,
                     reinterpret_cast<const uint4 *>(P_m), reinterpret_cast<const int8_t *>(P_e),
                     smat_m / 16, smat_e, nT, n_chunks, ring, x_m, x_e, x_stride, y_m, y_e,
                     y_stride, cstride);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return set_err(BFP_EIO, "matvec launch: %s", hipGetErrorString(err));
  return BFP_OK;
}

static inline unsigned nblk(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

int launch_status(const char *what) {
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return set_err(BFP_EIO, "%s launch: %s", what, hipGetErrorString(err));
  return BFP_OK;
}

int pack(const int16_t *W_m, const int8_t *W_e, int n_out, int n_in, void *P_m, void *P_e,
         hipStream_t s, int cstride) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16 || !W_m || !W_e || !P_m || !P_e)
    return set_err(BFP_EINVAL, "pack: bad arguments (n_out=%d n_in=%d)", n_out, n_in);
  int nT = n_in / 16;
  long long tm = (long long)(n_out / 16) * nT * 32, te = (long long)(n_out / 16) * nT * 16;
  hipLaunchKernelGGL(pack_m_kernel, dim3(nblk(tm, 256)), dim3(256), 0, s, W_m, tm, nT, cstride,
                     reinterpret_cast<uint4 *>(P_m));
  hipLaunchKernelGGL(pack_e_kernel, dim3(nblk(te, 256)), dim3(256), 0, s, W_e, te, nT, cstride,
                     reinterpret_cast<int8_t *>(P_e));
  return launch_status("pack");
}

int pack_wide(const void *wide_m, const void *wide_e, int n_out, int n_in, void *P_m, void *P_e,
              hipStream_t s, int cstride) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16 || !wide_m || !wide_e || !P_m || !P_e)
    return set_err(BFP_EINVAL, "pack_wide: bad arguments (n_out=%d n_in=%d)", n_out, n_in);
  int nT = n_in / 16;
  long long tm = (long long)(n_out / 16) * nT * 32, te = (long long)(n_out / 16) * nT * 16;
  hipLaunchKernelGGL(pack_wide_m_kernel, dim3(nblk(tm, 256)), dim3(256), 0, s,
                     reinterpret_cast<const int16_t *>(wide_m), tm, nT, cstride,
                     reinterpret_cast<uint4 *>(P_m));
  hipLaunchKernelGGL(pack_wide_e_kernel, dim3(nblk(te, 256)), dim3(256), 0, s,
                     reinterpret_cast<const int8_t *>(wide_e), te, nT, cstride,
                     reinterpret_cast<int8_t *>(P_e));
  return launch_status("pack_wide");
}

int quantize_pack_f32(const float *W, int n_out, int n_in, void *P_m, void *P_e, hipStream_t s,
                      int cstride) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16 || !W || !P_m || !P_e)
    return set_err(BFP_EINVAL, "quantize_pack: bad arguments (n_out=%d n_in=%d)", n_out, n_in);
  int nT = n_in / 16;
  const long long tiles = (long long)(n_out / 16) * nT;   // of 16 rows
  if (tiles > (1LL << 31)) return set_err(BFP_EINVAL, "quantize_pack: n_out=%d n_in=%d", n_out, n_in);
  // a grid row stays below 2^32 threads
  const unsigned blocks = nblk((tiles + 1) / 2, 4), gx = std::min(blocks, 1u << 22);
  hipLaunchKernelGGL(quantize_pack_f32_kernel, dim3(gx, (blocks + gx - 1) / gx), dim3(256), 0, s, W,
                     (unsigned)tiles, (unsigned)nT, cstride, reinterpret_cast<uint2 *>(P_m),
                     reinterpret_cast<int8_t *>(P_e));
  return launch_status("quantize_pack");
}

int tile_encode_f64(const double *v, size_t n, int16_t *m, int8_t *e, int *inexact,
                    hipStream_t s) {
  if (n % 16 || !v || !m || !e) return set_err(BFP_EINVAL, "tile_encode: n=%zu", n);
  if (n == 0) return BFP_OK;
  long long nt = (long long)(n / 16);
  hipLaunchKernelGGL((tile_quantize_kernel<double, true>), dim3(nblk(nt, 256)), dim3(256), 0, s, v,
                     nt, m, e, inexact);
  return launch_status("tile_encode");
}

int tile_quantize_f64(const double *v, size_t n, int16_t *m, int8_t *e, hipStream_t s) {
  if (n % 16 || !v || !m || !e) return set_err(BFP_EINVAL, "tile_quantize: n=%zu", n);
  if (n == 0) return BFP_OK;
  long long nt = (long long)(n / 16);
  hipLaunchKernelGGL(tile_quantize_kernel<double>, dim3(nblk(nt, 256)), dim3(256), 0, s, v, nt, m,
                     e);
  return launch_status("tile_quantize");
}

}  // namespace bfp

using namespace bfp;

// ------------------------------------------------------------------- C ABI
extern "C" {

const char *bfp_last_error(void) { return bfp::last_error(); }
const char *bfp_version(void) { return "libbfp 0.1 (gfx950)"; }

size_t bfp_packed_bytes_m(int n_out, int n_in) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16) return 0;
  return (size_t)n_out * n_in * 2;
}
size_t bfp_packed_bytes_e(int n_out, int n_in) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16) return 0;
  return (size_t)n_out * (n_in / 16);
}

int bfp_pack_d(const int16_t *W_m, const int8_t *W_e, int n_out, int n_in, void *P_m, void *P_e,
               void *stream) {
  return bfp::pack(W_m, W_e, n_out, n_in, P_m, P_e, (hipStream_t)stream);
}

int bfp_unpack_d(const void *P_m, const void *P_e, int n_out, int n_in, int16_t *W_m,
                 int8_t *W_e, void *stream) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16 || !W_m || !W_e || !P_m || !P_e)
    return set_err(BFP_EINVAL, "unpack: bad arguments (n_out=%d n_in=%d)", n_out, n_in);
  hipStream_t s = (hipStream_t)stream;
  int nT = n_in / 16;
  long long tm = (long long)(n_out / 16) * nT * 32, te = (long long)(n_out / 16) * nT * 16;
  hipLaunchKernelGGL(unpack_m_kernel, dim3(nblk(tm, 256)), dim3(256), 0, s,
                     reinterpret_cast<const uint4 *>(P_m), tm, nT, W_m);
  hipLaunchKernelGGL(unpack_e_kernel, dim3(nblk(te, 256)), dim3(256), 0, s,
                     reinterpret_cast<const int8_t *>(P_e), te, nT, W_e);
  return launch_status("unpack");
}

int bfp_tile_quantize_f64_d(const double *v, size_t n, int16_t *m, int8_t *e, void *stream) {
  return bfp::tile_quantize_f64(v, n, m, e, (hipStream_t)stream);
}

int bfp_tile_encode_f64_d(const double *v, size_t n, int16_t *m, int8_t *e, int *inexact,
                          void *stream) {
  return bfp::tile_encode_f64(v, n, m, e, inexact, (hipStream_t)stream);
}

int bfp_tile_quantize_f32_d(const float *v, size_t n, int16_t *m, int8_t *e, void *stream) {
  if (n % 16 || !v || !m || !e) return set_err(BFP_EINVAL, "tile_quantize: n=%zu", n);
  if (n == 0) return BFP_OK;
  long long nt = (long long)(n / 16);
  hipLaunchKernelGGL(tile_quantize_kernel<float>, dim3(nblk(nt, 256)), dim3(256), 0,
                     (hipStream_t)stream, v, nt, m, e);
  return launch_status("tile_quantize");
}

int bfp_quantize_pack_f32_d(const float *W, int n_out, int n_in, void *P_m, void *P_e,
                            void *stream) {
  return bfp::quantize_pack_f32(W, n_out, n_in, P_m, P_e, (hipStream_t)stream);
}

int bfp_tile_decode_d(const int16_t *m, const int8_t *e, size_t n, double *v, void *stream) {
  if (n % 16 || !m || !e || !v) return set_err(BFP_EINVAL, "tile_decode: n=%zu", n);
  if (n == 0) return BFP_OK;
  hipLaunchKernelGGL(tile_decode_kernel, dim3(nblk((long long)n, 256)), dim3(256), 0,
                     (hipStream_t)stream, m, e, (long long)n, v);
  return launch_status("tile_decode");
}

int bfp_matvec_d(const void *P_m, const void *P_e, int n_out, int n_in, int n_mats,
                 long long mat_stride_m, long long mat_stride_e, const int16_t *x_m,
                 const int8_t *x_e, long long x_stride, int16_t *y_m, int8_t *y_e,
                 long long y_stride, int waves, void *stream) {
  return bfp::launch_matvec(P_m, P_e, n_out, n_in, n_mats, 0, mat_stride_m, mat_stride_e, x_m,
                            x_e, x_stride, y_m, y_e, y_stride, waves, (hipStream_t)stream);
}

int bfp_matvec_ring_d(const void *P_m, const void *P_e, int n_out, int n_in, int n_mats,
                      int ring, long long mat_stride_m, long long mat_stride_e,
                      const int16_t *x_m, const int8_t *x_e, long long x_stride, int16_t *y_m,
                      int8_t *y_e, long long y_stride, int waves, void *stream) {
  return bfp::launch_matvec(P_m, P_e, n_out, n_in, n_mats, ring, mat_stride_m, mat_stride_e, x_m,
                            x_e, x_stride, y_m, y_e, y_stride, waves, (hipStream_t)stream);
}

int bfp_pack_wide_d(const void *wide_m, const void *wide_e, int n_out, int n_in, void *P_m,
                    void *P_e, void *stream) {
  return bfp::pack_wide(wide_m, wide_e, n_out, n_in, P_m, P_e, (hipStream_t)stream);
}

int bfp_probe_read_d(const void *p, size_t bytes, uint32_t *out, int n_wg, int nt,
                     void *stream) {
  if (!p || !out || n_wg <= 0 || bytes % 16 || bytes == 0)
    return set_err(BFP_EINVAL, "probe_read: bad arguments (bytes=%zu n_wg=%d)", bytes, n_wg);
  const long long n16 = (long long)(bytes / 16);
  const long long per = (n16 + n_wg - 1) / n_wg;
  if ((long long)(n_wg - 1) * per >= n16)
    return set_err(BFP_EINVAL, "probe_read: %d workgroups leave some without words", n_wg);
  if (per > (1LL << 26))
    return set_err(BFP_EINVAL, "probe_read: more than 1 GiB per workgroup (n_wg=%d)", n_wg);
  hipLaunchKernelGGL(nt ? probe_read_kernel<true> : probe_read_kernel<false>, dim3(n_wg),
                     dim3(256), 0, (hipStream_t)stream, reinterpret_cast<const uint4 *>(p), n16,
                     per, reinterpret_cast<unsigned *>(out));
  return launch_status("probe_read");
}

int bfp_embed_gather_d(const void *lu_m, const void *lu_e, int vocab, int D, int e_row_bytes,
                       const int32_t *ids, int n, int16_t *out_m, int8_t *out_e, void *stream) {
  if (vocab <= 0 || D <= 0 || D % 16 || e_row_bytes < D / 16 || n < 0)
    return set_err(BFP_EINVAL, "embed_gather: bad arguments (vocab=%d D=%d e_row=%d n=%d)", vocab,
                   D, e_row_bytes, n);
  if (n == 0) return BFP_OK;
  if (!lu_m || !lu_e || !ids || !out_m || !out_e)
    return set_err(BFP_EINVAL, "embed_gather: null pointer");
  if ((reinterpret_cast<uintptr_t>(lu_m) | reinterpret_cast<uintptr_t>(out_m)) & 15)
    return set_err(BFP_EINVAL, "embed_gather: mantissa tables must be 16-byte aligned");
  hipLaunchKernelGGL(embed_gather_kernel, dim3(n), dim3(128), 0, (hipStream_t)stream,
                     reinterpret_cast<const uint4 *>(lu_m), reinterpret_cast<const int8_t *>(lu_e),
                     vocab, D, e_row_bytes, ids, reinterpret_cast<uint4 *>(out_m), out_e);
  return launch_status("embed_gather");
}

int bfp_matvec_h(const int16_t *W_m, const int8_t *W_e, int n_out, int n_in,
                 const int16_t *x_m, const int8_t *x_e, int16_t *y_m, int8_t *y_e) {
  if (n_out <= 0 || n_in <= 0 || n_out % 16 || n_in % 16 || !W_m || !W_e || !x_m || !x_e ||
      !y_m || !y_e)
    return set_err(BFP_EINVAL, "matvec_h: bad arguments (n_out=%d n_in=%d)", n_out, n_in);
  DevBuf buf;
  size_t bm = (size_t)n_out * n_in * 2, be = (size_t)n_out * n_in / 16;
  int16_t *dWm, *dxm, *dym;
  int8_t *dWe, *dxe, *dye;
  void *dPm, *dPe;
  int rc;
  if ((rc = buf.alloc((void **)&dWm, bm)) || (rc = buf.alloc((void **)&dWe, be)) ||
      (rc = buf.alloc(&dPm, bm)) || (rc = buf.alloc(&dPe, be)) ||
      (rc = buf.alloc((void **)&dxm, (size_t)n_in * 2)) ||
      (rc = buf.alloc((void **)&dxe, (size_t)n_in / 16)) ||
      (rc = buf.alloc((void **)&dym, (size_t)n_out * 2)) ||
      (rc = buf.alloc((void **)&dye, (size_t)n_out / 16)))
    return rc;
  HIP_TRY(hipMemcpy(dWm, W_m, bm, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(dWe, W_e, be, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(dxm, x_m, (size_t)n_in * 2, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(dxe, x_e, (size_t)n_in / 16, hipMemcpyHostToDevice));
  if ((rc = bfp::pack(dWm, dWe, n_out, n_in, dPm, dPe, 0))) return rc;
  if ((rc = bfp::launch_matvec(dPm, dPe, n_out, n_in, 1, 0, 0, 0, dxm, dxe, 0, dym, dye, 0, 0, 0)))
    return rc;
  HIP_TRY(hipMemcpy(y_m, dym, (size_t)n_out * 2, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(y_e, dye, (size_t)n_out / 16, hipMemcpyDeviceToHost));
  return BFP_OK;
}

}  // extern "C"
