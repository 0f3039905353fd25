// f32 linears of the layer entries and the model forward on the fp16 matrix
// cores of gfx950, without giving up f32 accuracy.
//
// An f32 row is scaled by a power of two so that its largest magnitude lies
// in [2^14, 2^15), and every scaled element v is stored as two fp16 values,
// hi = fp16(v) and lo = fp16(v - hi): 22 significant bits, elements down to
// 2^-29 of the row's largest still exact to 2^-40 of it. A product of two such
// rows is hi*hi + hi*lo + lo*hi on v_mfma_f32_16x16x32_f16 with f32
// accumulation (the dropped lo*lo is 2^-22 of a product), three fp16 products
// instead of one f32 product: 3/16 of the f32 matrix-core time.
//
// The planes are stored in the order the matrix cores read them: 16 rows x 32
// k as two 1 KB blocks (hi, lo), lane l of a wavefront holding row l % 16,
// k = 8 (l / 16) .. + 7 as 16 bytes at 16 l. So every LDS-DMA load moves 1 KB
// that is contiguous in memory and in LDS, and every operand read is one
// conflict-free 16-byte read per lane.
//
// Rows with an inf or NaN are marked in their exponent (their planes keep the
// inf or NaN in hi): every output of such a row is inf or NaN, and the GEMM's
// epilogue forms it by itself (NaN at once when the row holds one, else by a
// plain dot product), because inf * lo would turn inf into NaN.
#include <math.h>

#include "tfd_device.hpp"
#include "tfd_internal.hpp"

namespace tfd {
namespace {

// exps[row]: e with scaled value x * 2^-e, plus a mark on rows that are not finite.
constexpr int kRowInf = 1 << 14, kRowNan = 1 << 15;
__device__ __forceinline__ int row_exp(int e) {  // the exponent without the marks
  return e >= kRowNan - 512 ? e - kRowNan : (e >= kRowInf - 512 ? e - kRowInf : e);
}
__device__ __forceinline__ bool row_bad(int e) { return e >= kRowInf - 512; }
__device__ __forceinline__ bool row_nan(int e) { return e >= kRowNan - 512; }

// e for a row whose largest finite magnitude has these bits: x * 2^-e < 2^15.
__device__ __forceinline__ int split_exp(uint32_t max_bits) {
  if (max_bits == 0u) return 0;
  const int top = max_bits >= 0x800000u ? (int)(max_bits >> 23) - 126
                                        : 32 - (int)__builtin_clz(max_bits) - 149;
  return top - 15;
}

// Eight scaled elements as hi and lo fp16. A non-zero element never becomes
// zero (it keeps the sign that a product with inf needs).
__device__ __forceinline__ void split8(const float (&x)[8], int e, f16x8 &hi, f16x8 &lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float v = __builtin_amdgcn_ldexpf(x[i], -e);
    const _Float16 h = (_Float16)v;
    const float t = v - (float)h;  // NaN when x is not finite
    // |v| <= 2^-25 (v itself may have become 0) rounds to hi = 0: lo is then
    // fp16's smallest, 2^-24, unless x is 0.
    const float tiny = x[i] == 0.0f ? 0.0f : __builtin_copysignf(0x1p-24f, x[i]);
    const float w = fabsf(v) <= 0x1p-25f ? tiny : t;
    hi[i] = h;
    lo[i] = (_Float16)(w == w ? w : 0.0f);
  }
}

// One workgroup = 16 rows of one operand; its 8 waves take the 32-k blocks in
// turn (NIT each, held in registers between the max and the split, so the
// source is read once). Bound by HBM: 4 bytes read and 4 written per element.
// Source rows: contiguous in k (one lane reads 32 bytes of a row, a wave whole
// 128-byte lines), or transposed (SplitSeg::trans: 16 consecutive tokens per
// k). Anything unaligned or ragged goes element by element.
template <int NIT>
__global__ __launch_bounds__(512) void split_rows_kernel(SplitSegs segs) {
  __shared__ uint32_t s_max[8][16], s_flag[8][16];
  int blk = blockIdx.x, si = 0;
  while (si + 1 < segs.n && blk >= segs.seg[si].blocks) blk -= segs.seg[si++].blocks;
  const SplitSeg &g = segs.seg[si];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row16 = lane & 15, oct = lane >> 4;
  const int K = g.k, nkb = (K + 31) / 32;
  // Plane row -> source row: the GeGLU weights alternate 16-row blocks of
  // their two halves.
  int row;
  bool in;
  if (g.half > 0) {
    const int f = (blk >> 1) * 16 + row16;
    in = f < g.half;
    row = f + (blk & 1) * g.half;
  } else {
    row = blk * 16 + row16;
    in = row < g.rows;
  }
  if (!in) row = 0;
  if (g.map) row = g.map[row];
  const float *src;
  size_t ks = 1;
  if (g.trans) {
    const int r = row / g.length, t = row - r * g.length;
    src = g.src + (size_t)r * K * g.length + t;
    ks = (size_t)g.length;
  } else {
    src = g.src + (size_t)row * K;
  }
  float x[NIT][8];
  uint32_t mx = 0, fl = 0;
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int kb = wave + 8 * it, k = 32 * kb + 8 * oct;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[it][e] = 0.0f;
    if (in && kb < nkb) {
      if (g.vec && k + 8 <= K) {
        *reinterpret_cast<f32x4 *>(&x[it][0]) = *reinterpret_cast<const f32x4 *>(src + k);
        *reinterpret_cast<f32x4 *>(&x[it][4]) = *reinterpret_cast<const f32x4 *>(src + k + 4);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k + e < K) x[it][e] = src[(size_t)(k + e) * ks];
      }
    }
  }
#pragma unroll
  for (int it = 0; it < NIT; ++it)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t b = __float_as_uint(x[it][e]) & 0x7fffffffu;
      const bool fin = b < 0x7f800000u;
      mx = max(mx, fin ? b : 0u);
      fl |= fin ? 0u : (b == 0x7f800000u ? 1u : 2u);
    }
  mx = max(mx, (uint32_t)__shfl_xor((int)mx, 16));
  mx = max(mx, (uint32_t)__shfl_xor((int)mx, 32));
  fl |= (uint32_t)__shfl_xor((int)fl, 16);
  fl |= (uint32_t)__shfl_xor((int)fl, 32);
  if (lane < 16) {
    s_max[wave][lane] = mx;
    s_flag[wave][lane] = fl;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    mx = max(mx, s_max[w][row16]);
    fl |= s_flag[w][row16];
  }
  const int e = split_exp(mx);
  if (threadIdx.x < 16) g.exps[blk * 16 + lane] = e + (fl & 2u ? kRowNan : (fl & 1u ? kRowInf : 0));
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int kb = wave + 8 * it;
    if (kb < nkb) {
      f16x8 hi, lo;
      split8(x[it], e, hi, lo);
      unsigned char *p = g.dst + ((size_t)blk * nkb + kb) * kSplitBlock + 16 * lane;
      *reinterpret_cast<f16x8 *>(p) = hi;
      *reinterpret_cast<f16x8 *>(p + 1024) = lo;
    }
  }
}

// Any k: the rows are read twice (the second time from L2).
__global__ __launch_bounds__(512) void split_rows_long_kernel(SplitSegs segs) {
  __shared__ uint32_t s_max[8][16], s_flag[8][16];
  int blk = blockIdx.x, si = 0;
  while (si + 1 < segs.n && blk >= segs.seg[si].blocks) blk -= segs.seg[si++].blocks;
  const SplitSeg &g = segs.seg[si];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row16 = lane & 15, oct = lane >> 4;
  const int K = g.k, nkb = (K + 31) / 32;
  int row;
  bool in;
  if (g.half > 0) {
    const int f = (blk >> 1) * 16 + row16;
    in = f < g.half;
    row = f + (blk & 1) * g.half;
  } else {
    row = blk * 16 + row16;
    in = row < g.rows;
  }
  if (!in) row = 0;
  if (g.map) row = g.map[row];
  const float *src;
  size_t ks = 1;
  if (g.trans) {
    const int r = row / g.length, t = row - r * g.length;
    src = g.src + (size_t)r * K * g.length + t;
    ks = (size_t)g.length;
  } else {
    src = g.src + (size_t)row * K;
  }
  auto load = [&](int kb, float (&x)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 32 * kb + 8 * oct + e;
      x[e] = in && k < K ? src[(size_t)k * ks] : 0.0f;
    }
  };
  uint32_t mx = 0, fl = 0;
  for (int kb = wave; kb < nkb; kb += 8) {
    float x[8];
    load(kb, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t b = __float_as_uint(x[e]) & 0x7fffffffu;
      if (b < 0x7f800000u)
        mx = max(mx, b);
      else
        fl |= b == 0x7f800000u ? 1u : 2u;
    }
  }
  mx = max(mx, (uint32_t)__shfl_xor((int)mx, 16));
  mx = max(mx, (uint32_t)__shfl_xor((int)mx, 32));
  fl |= (uint32_t)__shfl_xor((int)fl, 16);
  fl |= (uint32_t)__shfl_xor((int)fl, 32);
  if (lane < 16) {
    s_max[wave][lane] = mx;
    s_flag[wave][lane] = fl;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    mx = max(mx, s_max[w][row16]);
    fl |= s_flag[w][row16];
  }
  const int e = split_exp(mx);
  if (threadIdx.x < 16) g.exps[blk * 16 + lane] = e + (fl & 2u ? kRowNan : (fl & 1u ? kRowInf : 0));
  for (int kb = wave; kb < nkb; kb += 8) {
    float x[8];
    load(kb, x);
    f16x8 hi, lo;
    split8(x, e, hi, lo);
    unsigned char *p = g.dst + ((size_t)blk * nkb + kb) * kSplitBlock + 16 * lane;
    *reinterpret_cast<f16x8 *>(p) = hi;
    *reinterpret_cast<f16x8 *>(p + 1024) = lo;
  }
}

// LayerNorm of feature columns (NormArgs; the arithmetic of
// norm_columns_kernel) written straight as planes. 32 lanes per column, 16
// columns = one plane row block per workgroup; a lane holds NO octets of its
// column (d <= 256 * NO) in registers. Bound by latency (one round trip of
// loads, three reductions): 8 waves per workgroup and all loads issued first.
template <int NO>
__global__ __launch_bounds__(512) void norm_split_kernel(NormArgs a, unsigned char *dst, int *exps,
                                                         int nkb) {
  const int l32 = threadIdx.x & 31, c16 = threadIdx.x >> 5;
  const long c = (long)blockIdx.x * 16 + c16;
  const bool in = c < a.cols;
  const int d = a.d;
  const float *x = a.x + (in ? (a.map ? (long)a.map[c] : c) : 0) * (long)a.ldx;
  auto sum32 = [](float v) {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
  };
  const bool vec = (d & 7) == 0 && ((reinterpret_cast<uintptr_t>(a.x) |
                                     reinterpret_cast<uintptr_t>(a.w) |
                                     reinterpret_cast<uintptr_t>(a.b)) & 15) == 0;
  auto load8 = [&](const float *p, int k, float (&r)[8]) {
    if (vec) {
      const bool here = k < d;
      const float *q = p + (here ? k : 0);
      const f32x4 u = *reinterpret_cast<const f32x4 *>(q), v = *reinterpret_cast<const f32x4 *>(q + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r[e] = here ? u[e] : 0.0f;
        r[4 + e] = here ? v[e] : 0.0f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = k + e < d ? p[k + e] : 0.0f;
    }
  };
  float r[NO][8], w[NO][8], b[NO][8];
#pragma unroll
  for (int j = 0; j < NO; ++j) load8(x, 8 * (l32 + 32 * j), r[j]);
#pragma unroll
  for (int j = 0; j < NO; ++j) load8(a.w, 8 * (l32 + 32 * j), w[j]);
  if (a.b) {
#pragma unroll
    for (int j = 0; j < NO; ++j) load8(a.b, 8 * (l32 + 32 * j), b[j]);
  }
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < NO; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += r[j][e];
  const float mean = sum32(s) / (float)d;
  float v = 0.0f;
#pragma unroll
  for (int j = 0; j < NO; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t = r[j][e] - mean;
      v += 8 * (l32 + 32 * j) + e < d ? t * t : 0.0f;
    }
  const float inv = 1.0f / sqrtf(sum32(v) / (float)d + a.eps);
  uint32_t mx = 0, fl = 0;
#pragma unroll
  for (int j = 0; j < NO; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float y = (r[j][e] - mean) * inv * w[j][e];
      if (a.b) y = y + b[j][e];
      y = in && 8 * (l32 + 32 * j) + e < d ? y : 0.0f;
      r[j][e] = y;
      const uint32_t u = __float_as_uint(y) & 0x7fffffffu;
      const bool fin = u < 0x7f800000u;
      mx = max(mx, fin ? u : 0u);
      fl |= fin ? 0u : (u == 0x7f800000u ? 1u : 2u);
    }
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) {
    mx = max(mx, (uint32_t)__shfl_xor((int)mx, o));
    fl |= (uint32_t)__shfl_xor((int)fl, o);
  }
  const int e = split_exp(mx);
  if (l32 == 0) exps[c] = e + (fl & 2u ? kRowNan : (fl & 1u ? kRowInf : 0));
#pragma unroll
  for (int j = 0; j < NO; ++j) {
    const int o = l32 + 32 * j;
    if (o < 4 * nkb) {
      f16x8 hi, lo;
      split8(r[j], e, hi, lo);
      unsigned char *p = dst + ((size_t)blockIdx.x * nkb + (o >> 2)) * kSplitBlock +
                         256 * (o & 3) + 16 * c16;
      *reinterpret_cast<f16x8 *>(p) = hi;
      *reinterpret_cast<f16x8 *>(p + 1024) = lo;
    }
  }
}

// ------------------------------------------------------------------- GEMM

// Unscaled dot product of plane rows m and n, element by element (rows with
// an inf only).
__device__ __noinline__ float plane_dot(const unsigned char *a, const unsigned char *b, int m,
                                        int n, int nkb) {
  const unsigned char *pa = a + (size_t)(m >> 4) * nkb * kSplitBlock + 16 * (m & 15);
  const unsigned char *pb = b + (size_t)(n >> 4) * nkb * kSplitBlock + 16 * (n & 15);
  float s = 0.0f;
  for (int kb = 0; kb < nkb; ++kb)
    for (int o = 0; o < 4; ++o) {
      const size_t off = (size_t)kb * kSplitBlock + 256 * o;
      const f16x8 ah = *reinterpret_cast<const f16x8 *>(pa + off);
      const f16x8 al = *reinterpret_cast<const f16x8 *>(pa + off + 1024);
      const f16x8 bh = *reinterpret_cast<const f16x8 *>(pb + off);
      const f16x8 bl = *reinterpret_cast<const f16x8 *>(pb + off + 1024);
      for (int i = 0; i < 8; ++i)
        s = fmaf((float)ah[i] + (float)al[i], (float)bh[i] + (float)bl[i], s);
    }
  return s;
}

// One workgroup = 4 waves (2 x 2) computes a BM x BN tile of A * B^T; a wave
// BM/2 x BN/2 as 16 x 16 blocks. Per 32-k step the tile's planes ((BM + BN) *
// 128 bytes) come by LDS-DMA, S - 1 steps ahead, into S buffers; one barrier
// per step. Bound by each wave's chain of operand reads, products and barrier
// (counters at 64 x 128: matrix cores busy 46 %, LDS 23 %, no conflicts), so
// what counts is that two or three workgroups share a CU, each SIMD having
// another wave to run during one's operand reads and barrier; deeper buffers
// with fewer workgroups were slower (64 x 128: 2 steps 51 us, 3 63 us, 6 93 us
// at 2304 x 4096 x 768). Measured there: 52 us, 810-850 TFLOP/s of fp16 work, against
// 112-136 us for an f32 matrix product, and 2.0e-7 relative error against 4.9e-7;
// 5120 x 4096 x 1024 150-160 us (353), 768 x 2309 x 1152 21 us (40).
template <int BM, int BN, int S, int EPI>
__global__ __launch_bounds__(256, 2) void split_gemm_kernel(SplitGemmArgs g) {
  constexpr int TM = BM / 32, TN = BN / 32;          // 16 x 16 blocks per wave
  constexpr int RA = BM / 16, RB = BN / 16;          // row blocks per tile
  constexpr int PIECES = 2 * (RA + RB);              // 1 KB pieces per step
  constexpr int PW = PIECES / 4;                     // per wave
  static_assert(PIECES % 4 == 0 && (S - 2) * PW < 64, "pieces per wave, vmcnt range");
  constexpr int STAGE = PIECES * 1024;
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int nkb = g.nkb;
  // Workgroup p runs on XCD p % 8: give each XCD a contiguous range of tiles,
  // the tiles of a range sharing B columns, so its L2 serves the re-reads.
  const int tiles = g.mt * g.nt;
  const int per = (tiles + 7) / 8;
  const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tile >= tiles || (int)(blockIdx.x >> 3) >= per) return;
  const int tn = tile / g.mt, tm = tile - tn * g.mt;
  const int mb0 = tm * RA, nb0 = tn * RB;            // first row blocks
  const int mblocks = (g.mrows + 15) / 16, nblocks = (g.n + 15) / 16;
  const size_t rowb = (size_t)nkb * kSplitBlock;     // bytes of a row block
  const int va = min(RA, mblocks - mb0), vb = min(RB, nblocks - nb0);
  const u32x4r ra = rsrc_words(g.a + (size_t)mb0 * rowb, (uint32_t)(va * rowb));
  const u32x4r rb = rsrc_words(g.b + (size_t)nb0 * rowb, (uint32_t)(vb * rowb));
  const uint32_t voff = 16 * lane;
  auto stage = [&](int kb, unsigned char *buf) {
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int p = wave * PW + i;
      {
        const int blk = p >> 1, plane = p & 1;
        // Row blocks past the matrix re-read its last one; their outputs are
        // never stored.
        if (blk < RA)
          load_lds16(ra, voff, (uint32_t)(min(blk, va - 1) * rowb + (size_t)kb * kSplitBlock + 1024 * plane),
                     buf + 1024 * p);
        else
          load_lds16(rb, voff, (uint32_t)(min(blk - RA, vb - 1) * rowb + (size_t)kb * kSplitBlock + 1024 * plane),
                     buf + 1024 * p);
      }
    }
  };
  // The cross products (2^-11 of the sum) have an accumulator of their own:
  // the matrix core rounds the sum once per instruction, and this leaves one
  // rounding of the full sum per 32 k instead of three.
  f32x4 acc[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = low[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < S - 1; ++i)
    if (i < nkb) stage(i, smem + i * STAGE);
  unsigned char *cur = smem, *next = smem + (S - 1) * STAGE;
  for (int kb = 0; kb < nkb; ++kb) {
    // This wave's loads of step kb have landed (those of the S - 2 steps
    // after it may be in flight) and its reads of the buffer about to be
    // refilled, step kb - 1's, are done.
    if (kb + S - 1 <= nkb)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * PW) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kb + S - 1 < nkb) stage(kb + S - 1, next);
    const unsigned char *pa = cur + wm * TM * 2048 + 16 * lane;
    const unsigned char *pb = cur + (RA + wn * TN) * 2048 + 16 * lane;
    f16x8 bh[TN], bl[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      bh[j] = *reinterpret_cast<const f16x8 *>(pb + 2048 * j);
      bl[j] = *reinterpret_cast<const f16x8 *>(pb + 2048 * j + 1024);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const f16x8 ah = *reinterpret_cast<const f16x8 *>(pa + 2048 * i);
      const f16x8 al = *reinterpret_cast<const f16x8 *>(pa + 2048 * i + 1024);
#pragma unroll
      for (int j = 0; j < TN; ++j) low[i][j] = mfma_16x16x32_f16(ah, bl[j], low[i][j]);
#pragma unroll
      for (int j = 0; j < TN; ++j) low[i][j] = mfma_16x16x32_f16(al, bh[j], low[i][j]);
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma_16x16x32_f16(ah, bh[j], acc[i][j]);
    }
    next = cur;
    cur = cur + STAGE == smem + S * STAGE ? smem : cur + STAGE;
  }
  // Epilogue. Lane l holds rows 4 (l / 16) .. + 3 of column l % 16 of a block.
  const int col = lane & 15, grp = lane >> 4;
  int ea[TM][4];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = 16 * (mb0 + wm * TM + i) + 4 * grp;
#pragma unroll
    for (int r = 0; r < 4; ++r) ea[i][r] = g.ea[min(m + r, 16 * mblocks - 1)];
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = 16 * (nb0 + wn * TN + j) + col;
    const bool nin = n < g.n;
    const int eb = g.eb[min(n, 16 * nblocks - 1)];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = 16 * (mb0 + wm * TM + i) + 4 * grp;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int e = ea[i][r];
        float s = acc[i][j][r] + low[i][j][r];
        if (row_bad(e) || row_bad(eb))
          s = row_nan(e) || row_nan(eb) || !nin || m + r >= 16 * mblocks
                  ? __builtin_nanf("")
                  : plane_dot(g.a, g.b, m + r, n, nkb);
        acc[i][j][r] = ldexpf(s, row_exp(e) + row_exp(eb));
      }
    }
    if (!nin) continue;
    if constexpr (EPI == kEpiCols) {
      float *out = g.out + (size_t)(g.map ? g.map[n] : n) * g.ldc;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = 16 * (mb0 + wm * TM + i) + 4 * grp;
        if (m >= g.m) continue;
        f32x4 v = acc[i][j];
        if (m + 4 <= g.m && (g.vec & 1)) {
          if (g.accumulate) v = v + *reinterpret_cast<const f32x4 *>(out + m);
          if (g.bias) v = v + *reinterpret_cast<const f32x4 *>(g.bias + m);
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = activate(v[r], g.act);
          *reinterpret_cast<f32x4 *>(out + m) = v;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (m + r < g.m) {
              float y = v[r];
              if (g.accumulate) y += out[m + r];
              if (g.bias) y += g.bias[m + r];
              out[m + r] = activate(y, g.act);
            }
        }
      }
    } else if constexpr (EPI == kEpiGeglu) {
      // Row blocks 2f and 2f + 1 of A are features 16 f .. of the two halves.
      float *out = g.out + (size_t)n * g.ldc;
#pragma unroll
      for (int i = 0; i < TM; i += 2) {
        const int f = 8 * (mb0 + wm * TM + i) + 4 * grp;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (f + r < g.m) {
            float x = acc[i][j][r], y = acc[i + 1][j][r];
            if (g.bias) {
              x += g.bias[f + r];
              y += g.bias[g.m + f + r];
            }
            acc[i][j][r] = gelu_erf(x) * y;
          }
        if (f + 4 <= g.m && (g.vec & 1))
          *reinterpret_cast<f32x4 *>(out + f) = acc[i][j];
        else
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (f + r < g.m) out[f + r] = acc[i][j][r];
      }
    } else {
      // Rows of A are tokens t of question rows, columns are features of up
      // to four outputs (rows x (L, width)).
      int s = 0;
      while (s + 1 < g.nouts && n >= g.outs[s + 1].begin) ++s;
      const int f = n - g.outs[s].begin, w = g.outs[s].width;
      if (f >= w) continue;  // padding between two weights' row blocks
      float *out = g.outs[s].ptr + (size_t)f * g.length;
      const size_t rs = (size_t)w * g.length;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = 16 * (mb0 + wm * TM + i) + 4 * grp;
        if (m >= g.m) continue;
        if (g.vec & 1) {  // length % 4 == 0: four tokens of one row
          const int row = m / g.length;
          *reinterpret_cast<f32x4 *>(out + row * rs + (m - row * g.length)) = acc[i][j];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (m + r < g.m) {
              const int row = (m + r) / g.length;
              out[row * rs + (m + r - row * g.length)] = acc[i][j][r];
            }
        }
      }
    }
  }
}

template <int BM, int BN, int S, int EPI>
hipError_t launch_tile(SplitGemmArgs g, hipStream_t stream) {
  constexpr int kLds = S * (BM + BN) * 128;
  g.mt = (g.mrows + BM - 1) / BM;
  g.nt = (g.n + BN - 1) / BN;
  const long tiles = (long)g.mt * g.nt;
  const unsigned grid = (unsigned)(8 * ((tiles + 7) / 8));
  static_assert(kLds <= 65536, "dynamic LDS without an opt-in");
  hipLaunchKernelGGL((split_gemm_kernel<BM, BN, S, EPI>), dim3(grid), dim3(256), kLds, stream, g);
  return hipGetLastError();
}

}  // namespace

bool norm_split_fits(int d) { return d <= 1024; }

hipError_t launch_norm_split(const NormArgs &a, unsigned char *dst, int *exps,
                             hipStream_t stream) {
  if (a.cols <= 0) return hipSuccess;
  const dim3 grid((unsigned)((a.cols + 15) / 16));
  const int nkb = (a.d + 31) / 32;
  if (a.d <= 256)
    hipLaunchKernelGGL(norm_split_kernel<1>, grid, dim3(512), 0, stream, a, dst, exps, nkb);
  else if (a.d <= 768)
    hipLaunchKernelGGL(norm_split_kernel<3>, grid, dim3(512), 0, stream, a, dst, exps, nkb);
  else
    hipLaunchKernelGGL(norm_split_kernel<4>, grid, dim3(512), 0, stream, a, dst, exps, nkb);
  return hipGetLastError();
}

hipError_t launch_split_rows(const SplitSegs &segs, hipStream_t stream) {
  long blocks = 0;
  int kmax = 0;
  for (int i = 0; i < segs.n; ++i) {
    blocks += segs.seg[i].blocks;
    kmax = segs.seg[i].k > kmax ? segs.seg[i].k : kmax;
  }
  if (blocks == 0) return hipSuccess;
  const dim3 grid((unsigned)blocks), block(512);
  if (kmax <= 1024)
    hipLaunchKernelGGL(split_rows_kernel<4>, grid, block, 0, stream, segs);
  else if (kmax <= 2048)
    hipLaunchKernelGGL(split_rows_kernel<8>, grid, block, 0, stream, segs);
  else if (kmax <= 3072)
    hipLaunchKernelGGL(split_rows_kernel<12>, grid, block, 0, stream, segs);
  else
    hipLaunchKernelGGL(split_rows_long_kernel, grid, block, 0, stream, segs);
  return hipGetLastError();
}

// The tile: the one that should finish first on this device. A CU's time per
// 32-k step is what its resident workgroups' matrix and LDS work takes, but
// at least one workgroup's latency (LDS reads, barrier); measured per step:
// 128 x 128 0.95 us alone and 0.60 us each with the second one a CU holds,
// 64 x 128 0.65 and 0.32 us (three), 64 x 64 0.45 and 0.19 us (three). The sum over the
// rounds of the busiest CU predicted the fastest of the three at all sizes
// tried (768 .. 5120 x 200 .. 4096, k 768 .. 3072).
hipError_t launch_split_gemm(const SplitGemmArgs &g, int epi, int cus, hipStream_t stream) {
  if (g.m <= 0 || g.n <= 0) return hipSuccess;
  struct Tile {
    int bm, bn, resident;
    float alone, each;
  };
  constexpr Tile kTiles[] = {{128, 128, 2, 0.95f, 0.60f}, {64, 128, 3, 0.65f, 0.32f},
                             {64, 64, 3, 0.45f, 0.19f}};
  int bm = 0, bn = 0;
  float best = 0.0f;
  for (const Tile &t : kTiles) {
    const long tiles = (long)((g.mrows + t.bm - 1) / t.bm) * ((g.n + t.bn - 1) / t.bn);
    const long each = (tiles + cus - 1) / cus, full = each / t.resident, rest = each % t.resident;
    const float cost = full * fmaxf(t.alone, t.resident * t.each) +
                       (rest ? fmaxf(t.alone, rest * t.each) : 0.0f);
    if (bm == 0 || cost < best) {
      best = cost;
      bm = t.bm;
      bn = t.bn;
    }
  }
#define TFD_TILE(BM, BN, S)                                                          \
  if (bm == BM && bn == BN) {                                                        \
    if (epi == kEpiCols) return launch_tile<BM, BN, S, kEpiCols>(g, stream);         \
    if (epi == kEpiRows) return launch_tile<BM, BN, S, kEpiRows>(g, stream);         \
    return launch_tile<BM, BN, S, kEpiGeglu>(g, stream);                             \
  }
  TFD_TILE(128, 128, 2)
  TFD_TILE(64, 128, 2)
  TFD_TILE(64, 64, 3)
#undef TFD_TILE
  return hipErrorInvalidValue;
}

}  // namespace tfd
