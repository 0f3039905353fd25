// f32 linears of the layer entries and the model forward on the bf16 matrix
// cores of gfx950, without giving up f32 accuracy.
//
// Every element is stored as three bf16 h + m + l (split_bf16x3: its 24
// significant bits over f32's whole exponent range, whatever the other elements
// of its row are). A product of two rows is hh' + (hm' + mh') + (hl' + lh' + mm')
// on v_mfma_f32_16x16x32_bf16 with f32 accumulation (what is dropped is below
// 2^-24 of each element's product, f32's own rounding), six bf16 products instead of
// one f32 product: 3/8 of the f32 matrix-core time. Splitting operands for
// lower-precision matrix units: Henry, Tang and Heinecke, "Leveraging the bfloat16
// artificial intelligence datatype for higher-precision computations", 2019.
//
// The planes are stored in the order the matrix cores read them: 16 rows x 32
// k as three 1 KB blocks (h, m, l), lane l of a wavefront holding row l % 16,
// k = 8 (l / 16) .. + 7 as 16 bytes at 16 l. So every LDS-DMA load moves 1 KB
// that is contiguous in memory and in LDS, and every operand read is one
// conflict-free 16-byte read per lane.
//
// Rows with an inf or NaN are marked (their planes keep it in h): the pieces of
// an inf make NaN of products that are inf, so the GEMM's epilogue forms the
// outputs of such rows by itself (NaN at once when the row holds one, else by a
// plain dot product), as it does an output that is not finite.
#include <math.h>

#include "tfd_device.hpp"
#include "tfd_internal.hpp"

namespace tfd {
namespace {

// marks[row]: whether the row holds an inf, a NaN.
constexpr int kRowInf = 1, kRowNan = 2;
__device__ __forceinline__ int mark_of(float x) {
  return __builtin_isfinite(x) ? 0 : (x == x ? kRowInf : kRowNan);
}

// Eight elements as their planes' 16 bytes at p. Finite elements above bf16's
// largest keep a finite h (m holds the rest).
__device__ __forceinline__ void write_split8(unsigned char *p, const float (&x)[8]) {
  constexpr float kMaxBf16 = 3.38953138925e38f;
  bf16x8 out[3];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bool fin = __builtin_isfinite(x[e]);
    const __bf16 h = (__bf16)(fin ? __builtin_amdgcn_fmed3f(x[e], -kMaxBf16, kMaxBf16) : x[e]);
    const float r = fin ? x[e] - (float)h : 0.0f;
    const __bf16 m = (__bf16)r;
    out[0][e] = h;
    out[1][e] = m;
    out[2][e] = (__bf16)(r - (float)m);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8 *>(p + 1024 * i) = out[i];
}

// One workgroup = 16 rows of one operand; its 8 waves take the 32-k blocks in
// turn, U of them in flight (4: 32 us for 4096 x 1024 token-contiguous with 7.3 M weights,
// 26 for 4096 x 2048; 8: 34 and 28, 2: 38 and 24). Bound by HBM: 4 bytes read and 6
// written per element. Source rows: contiguous in k (one lane reads 32 bytes of a row, a wave
// whole 128-byte lines), or transposed (SplitSeg::trans: 16 consecutive tokens per
// k). Anything unaligned or ragged goes element by element.
template <int U>
__global__ __launch_bounds__(512) void split_rows_kernel(SplitSegs segs) {
  __shared__ int s_mark[8][16];
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
  int mark = 0;
  for (int kb0 = wave; kb0 < nkb; kb0 += 8 * U) {
    float x[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kb = kb0 + 8 * u, k = 32 * kb + 8 * oct;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[u][e] = 0.0f;
      if (in && kb < nkb) {
        if (g.vec && k + 8 <= K) {
          *reinterpret_cast<f32x4 *>(&x[u][0]) = *reinterpret_cast<const f32x4 *>(src + k);
          *reinterpret_cast<f32x4 *>(&x[u][4]) = *reinterpret_cast<const f32x4 *>(src + k + 4);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (k + e < K) x[u][e] = src[(size_t)(k + e) * ks];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kb = kb0 + 8 * u;
      if (kb < nkb) {
#pragma unroll
        for (int e = 0; e < 8; ++e) mark |= mark_of(x[u][e]);
        write_split8(g.dst + ((size_t)blk * nkb + kb) * kSplitBlock + 16 * lane, x[u]);
      }
    }
  }
  mark |= __shfl_xor(mark, 16);
  mark |= __shfl_xor(mark, 32);
  if (lane < 16) s_mark[wave][lane] = mark;
  __syncthreads();
  if (threadIdx.x < 16) {
#pragma unroll
    for (int w = 0; w < 8; ++w) mark |= s_mark[w][lane];
    g.marks[blk * 16 + lane] = mark;
  }
}

// LayerNorm of feature columns (NormArgs; the arithmetic of
// norm_columns_kernel) written straight as planes. 32 lanes per column, 16
// columns = one plane row block per workgroup; a lane holds NO octets of its
// column (d <= 256 * NO) in registers. Bound by latency (one round trip of
// loads, three reductions): 8 waves per workgroup and all loads issued first.
template <int NO>
__global__ __launch_bounds__(512) void norm_split_kernel(NormArgs a, unsigned char *dst, int *marks,
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
  int mark = 0;
#pragma unroll
  for (int j = 0; j < NO; ++j) {
    const int o = l32 + 32 * j;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float y = (r[j][e] - mean) * inv * w[j][e];
      if (a.b) y = y + b[j][e];
      y = in && 8 * o + e < d ? y : 0.0f;
      r[j][e] = y;
      mark |= mark_of(y);
    }
    if (o < 4 * nkb)
      write_split8(dst + ((size_t)blockIdx.x * nkb + (o >> 2)) * kSplitBlock + 256 * (o & 3) + 16 * c16, r[j]);
  }
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) mark |= __shfl_xor(mark, o);
  if (l32 == 0) marks[c] = mark;
}

// ------------------------------------------------------------------- GEMM

// Dot product of plane rows m and n, element by element (outputs that are not
// finite, or may be). h alone is an inf or NaN element.
__device__ __noinline__ float plane_dot(const unsigned char *a, const unsigned char *b, int m,
                                        int n, int nkb) {
  const unsigned char *pa = a + (size_t)(m >> 4) * nkb * kSplitBlock + 16 * (m & 15);
  const unsigned char *pb = b + (size_t)(n >> 4) * nkb * kSplitBlock + 16 * (n & 15);
  auto load = [](const unsigned char *p, float (&x)[8]) {
    const bf16x8 h = *reinterpret_cast<const bf16x8 *>(p), i = *reinterpret_cast<const bf16x8 *>(p + 1024),
                 j = *reinterpret_cast<const bf16x8 *>(p + 2048);
    for (int e = 0; e < 8; ++e) x[e] = (float)h[e] + ((float)i[e] + (float)j[e]);
  };
  float s = 0.0f;
  for (int kb = 0; kb < nkb; ++kb)
    for (int o = 0; o < 4; ++o) {
      const size_t off = (size_t)kb * kSplitBlock + 256 * o;
      float x[8], y[8];
      load(pa + off, x);
      load(pb + off, y);
      for (int i = 0; i < 8; ++i) s = fmaf(x[i], y[i], s);
    }
  return s;
}

constexpr int kGroup = 8;  // A tiles per group of the tile order

// One workgroup = 4 waves (2 x 2) computes a BM x BN tile of A * B^T; a wave
// BM/2 x BN/2 as 16 x 16 blocks. Per 32-k step the tile's planes ((BM + BN) *
// 192 bytes) come by LDS-DMA into one of two buffers, and a step's operands are in
// registers while the next one's are read: one barrier per step and no wait inside
// a step's products. Large products are bound by the matrix cores' rate on this
// card (5120 x 4096 x 1024: 212-220 us, 1,170-1,215 TFLOP/s of bf16 work, where a large
// bf16 library product reaches 1,197), ones of few tiles per CU by the loads' latency
// (64 x 64 alone on a CU 0.45 us per step, 0.33 us each with three). Measured
// against f32 matrix products, alone, without the splits: 2304 x 4096 x 768 112-136 ->
// 90 us back to back (72 within a layer, whose other kernels leave the clocks higher),
// 768 x 2309 x 1152 40 -> 26, 5120 x 4096 x 1024 353 -> 220 (197 within a layer). As fp16
// pairs (half the products) the first took 52 us, but their rows lose the bits of
// elements far below the largest.
template <int BM, int BN, int EPI>
__global__ __launch_bounds__(256, 2) void split_gemm_kernel(SplitGemmArgs g) {
  constexpr int TM = BM / 32, TN = BN / 32;          // 16 x 16 blocks per wave
  constexpr int RA = BM / 16, RB = BN / 16;          // row blocks per tile
  constexpr int WA = RA / 4, WB = RB / 4;            // of them loaded per wave
  static_assert(RA % 4 == 0 && RB % 4 == 0, "row blocks per wave");
  constexpr int STAGE = (RA + RB) * kSplitBlock;
  __shared__ __align__(16) unsigned char smem[2 * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int nkb = g.nkb;
  // Workgroup p runs on XCD p % 8: give each XCD a contiguous range of tiles, in
  // groups of kGroup A tiles by all B tiles (64 x 64 at 5120 x 4096 x 1024 278 -> 212
  // us against whole columns of A tiles), so that its L2 serves the re-reads.
  const int tiles = g.mt * g.nt;
  const int per = (tiles + 7) / 8;
  const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tile >= tiles || (int)(blockIdx.x >> 3) >= per) return;
  const int grp0 = tile / (kGroup * g.nt), in0 = tile - grp0 * kGroup * g.nt;
  const int gm = min(kGroup, g.mt - grp0 * kGroup);
  const int tn = in0 / gm, tm = grp0 * kGroup + in0 - tn * gm;
  const int mb0 = tm * RA, nb0 = tn * RB;            // first row blocks
  const int mblocks = (g.mrows + 15) / 16, nblocks = (g.n + 15) / 16;
  const size_t rowb = (size_t)nkb * kSplitBlock;     // bytes of a row block
  const int va = min(RA, mblocks - mb0), vb = min(RB, nblocks - nb0);
  const u32x4r ra = rsrc_words(g.a + (size_t)mb0 * rowb, (uint32_t)(va * rowb));
  const u32x4r rb = rsrc_words(g.b + (size_t)nb0 * rowb, (uint32_t)(vb * rowb));
  const uint32_t voff = 16 * lane;
  // Row blocks past the matrix re-read its last one; their outputs are never
  // stored.
  uint32_t oa[WA], ob[WB];
#pragma unroll
  for (int i = 0; i < WA; ++i) oa[i] = (uint32_t)(min(WA * wave + i, va - 1) * rowb);
#pragma unroll
  for (int i = 0; i < WB; ++i) ob[i] = (uint32_t)(min(WB * wave + i, vb - 1) * rowb);
  auto stage = [&](int kb, unsigned char *buf) {
    const uint32_t k0 = (uint32_t)kb * kSplitBlock;
    unsigned char *const da = buf + WA * wave * kSplitBlock, *const db = buf + (RA + WB * wave) * kSplitBlock;
#pragma unroll
    for (int i = 0; i < WA; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        load_lds16(ra, voff, oa[i] + k0 + 1024 * p, da + kSplitBlock * i + 1024 * p);
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        load_lds16(rb, voff, ob[i] + k0 + 1024 * p, db + kSplitBlock * i + 1024 * p);
  };
  // The products but h*h (2^-8 of the sum) have an accumulator of their own:
  // the matrix core rounds the sum once per instruction, and this leaves one
  // rounding of the full sum per 32 k instead of six.
  f32x4 acc[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = low[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // A wave's operands of a step. Those of the next step are read while the current
  // one's products run, so a step's buffer is free for the step after next as
  // soon as every wave has read it.
  struct Operands {
    bf16x8 a[TM][3], b[TN][3];
  };
  Operands even, odd;
  auto read = [&](const unsigned char *buf, Operands &x) {
    const unsigned char *pa = buf + wm * TM * kSplitBlock + 16 * lane;
    const unsigned char *pb = buf + (RA + wn * TN) * kSplitBlock + 16 * lane;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) x.a[i][p] = *reinterpret_cast<const bf16x8 *>(pa + kSplitBlock * i + 1024 * p);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p) x.b[j][p] = *reinterpret_cast<const bf16x8 *>(pb + kSplitBlock * j + 1024 * p);
  };
  // This wave's loads have landed and its reads are done, and so for every wave.
  auto arrive = [] {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    // Said once more where the compiler sees it: else it waits for the next step's
    // reads before this step's products.
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Step kb, its operands in x and its buffer `mine`, step kb + 1 in `other`.
  auto step = [&](int kb, const Operands &x, Operands &next, unsigned char *mine, unsigned char *other) {
    arrive();
    if (kb + 2 < nkb) stage(kb + 2, mine);
    if (kb + 1 < nkb) read(other, next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int r = 2 - p; r >= 0; --r)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            f32x4 &c = p + r ? low[i][j] : acc[i][j];
            c = mfma_16x16x32_bf16(x.a[i][p], x.b[j][r], c);
          }
    __builtin_amdgcn_sched_barrier(0);
  };
  stage(0, smem);
  arrive();
  if (nkb > 1) stage(1, smem + STAGE);
  read(smem, even);
  for (int kb = 0; kb < nkb; kb += 2) {
    step(kb, even, odd, smem, smem + STAGE);
    if (kb + 1 < nkb) step(kb + 1, odd, even, smem + STAGE, smem);
  }
  // Epilogue. Lane l holds rows 4 (l / 16) .. + 3 of column l % 16 of a block.
  const int col = lane & 15, grp = lane >> 4;
  int ma[TM][4];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = 16 * (mb0 + wm * TM + i) + 4 * grp;
#pragma unroll
    for (int r = 0; r < 4; ++r) ma[i][r] = g.ma[min(m + r, 16 * mblocks - 1)];
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = 16 * (nb0 + wn * TN + j) + col;
    const bool nin = n < g.n;
    const int mb = g.mb[min(n, 16 * nblocks - 1)];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = 16 * (mb0 + wm * TM + i) + 4 * grp;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int mark = ma[i][r] | mb;
        float s = acc[i][j][r] + low[i][j][r];
        if (mark != 0 || !__builtin_isfinite(s))
          s = (mark & kRowNan) || !nin || m + r >= 16 * mblocks ? __builtin_nanf("")
                                                               : plane_dot(g.a, g.b, m + r, n, nkb);
        acc[i][j][r] = s;
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

template <int BM, int BN, int EPI>
hipError_t launch_tile(SplitGemmArgs g, hipStream_t stream) {
  g.mt = (g.mrows + BM - 1) / BM;
  g.nt = (g.n + BN - 1) / BN;
  const long tiles = (long)g.mt * g.nt;
  const unsigned grid = (unsigned)(8 * ((tiles + 7) / 8));
  hipLaunchKernelGGL((split_gemm_kernel<BM, BN, EPI>), dim3(grid), dim3(256), 0, stream, g);
  return hipGetLastError();
}

}  // namespace

bool norm_split_fits(int d) { return d <= 1024; }

hipError_t launch_norm_split(const NormArgs &a, unsigned char *dst, int *marks,
                             hipStream_t stream) {
  if (a.cols <= 0) return hipSuccess;
  const dim3 grid((unsigned)((a.cols + 15) / 16));
  const int nkb = (a.d + 31) / 32;
  if (a.d <= 768)
    hipLaunchKernelGGL(norm_split_kernel<3>, grid, dim3(512), 0, stream, a, dst, marks, nkb);
  else
    hipLaunchKernelGGL(norm_split_kernel<4>, grid, dim3(512), 0, stream, a, dst, marks, nkb);
  return hipGetLastError();
}

hipError_t launch_split_rows(const SplitSegs &segs, hipStream_t stream) {
  long blocks = 0;
  for (int i = 0; i < segs.n; ++i) blocks += segs.seg[i].blocks;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(split_rows_kernel<4>, dim3((unsigned)blocks), dim3(512), 0, stream, segs);
  return hipGetLastError();
}

// The tile: the one that should finish first on this device. A CU's time per
// 32-k step is what its resident workgroups' products and loads take, but
// at least one workgroup's latency; measured per step: 64 x 128 0.85 us alone and
// 0.63 us each with the second one a CU holds, 64 x 64 0.45 and 0.33 us (three). The
// sum over the rounds of the busiest CU predicts the faster of the two, or one within
// 4 % of it, at all sizes tried (512 .. 5120 x 640 .. 4096, k 512 .. 2048; 128 x 128
// and 256 x 128 were slower or equal at all of them).
hipError_t launch_split_gemm(const SplitGemmArgs &g, int epi, int cus, hipStream_t stream) {
  if (g.m <= 0 || g.n <= 0) return hipSuccess;
  struct Tile {
    int bm, bn, resident;
    float alone, each;
  };
  constexpr Tile kTiles[] = {{64, 128, 2, 0.85f, 0.63f}, {64, 64, 3, 0.45f, 0.33f}};
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
#define TFD_TILE(BM, BN)                                                             \
  if (bm == BM && bn == BN) {                                                        \
    if (epi == kEpiCols) return launch_tile<BM, BN, kEpiCols>(g, stream);            \
    if (epi == kEpiRows) return launch_tile<BM, BN, kEpiRows>(g, stream);            \
    return launch_tile<BM, BN, kEpiGeglu>(g, stream);                                \
  }
  TFD_TILE(64, 128)
  TFD_TILE(64, 64)
#undef TFD_TILE
  return hipErrorInvalidValue;
}

}  // namespace tfd
