// f32 linears over few columns (a short prompt's tokens, markers, one column
// per prompt): out (+)= W^T x with everything around it in one launch.
//
// At up to 160 columns a linear is bound by latency and by reading its weights
// once (7 MB take 1.5 us), not by the matrix cores, so the kernel does one
// memory round trip: a workgroup of 8 waves owns 16 weight rows (GeGLU: 16 of
// each half) x 16 or 32 columns, its waves take the 16-k chunks in turn, issue
// all their loads at once (16 bytes per lane, operands straight in the f32
// matrix cores' layout), and the eight partial sums meet once in LDS. LayerNorm
// of the columns (their elements are in the waves' registers anyway), the
// gather of the columns, bias, activation, GeGLU, residual add and the scatter
// of the result are part of it. Linears of more than 768 inputs come here up to 64
// columns only (f32 GEMMs beyond). Measured at 96 columns (768 -> 2304): 14.8 us
// with LayerNorm and scatter, against 16 us for the f32 GEMM plus 7 us for the
// LayerNorm and 4 us for the column move; 768 -> 768 12.7 us against 11 + 4. What
// remains is the chain of dependent round trips: arguments, column map,
// operands, LDS, store.
#include "tfd_device.hpp"
#include "tfd_internal.hpp"

namespace tfd {
namespace {

// CB: chunks per wave in flight. LN needs the whole column at once: K <= 128 * CB.
template <int RM, int NB, int CB, bool LN, bool GEGLU>
__global__ __launch_bounds__(512, LN ? 2 : 4) void skinny_kernel(SkinnyArgs g) {
  __shared__ __attribute__((aligned(16))) f32x4 s_acc[8 * RM * NB * 64];
  __shared__ float s_stat[LN ? 8 * NB * 16 : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int K = g.k, nchunk = (K + 15) / 16;
  constexpr int MB = GEGLU ? 1 : RM;  // 16-row blocks of outputs
  const int m0 = blockIdx.x * 16 * MB, n0 = blockIdx.y * 16 * NB;
  const float *wrow[RM], *xcol[NB];
#pragma unroll
  for (int r = 0; r < RM; ++r)
    wrow[r] = g.w + (size_t)(GEGLU ? min(m0 + col, g.m - 1) + r * g.half
                                   : min(m0 + 16 * r + col, g.m - 1)) * K;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int n = min(n0 + 16 * b + col, g.n - 1);
    xcol[b] = g.x + (size_t)(g.xmap ? g.xmap[n] : n) * g.ldx;
  }
  // What the epilogue adds, loaded now: at the end it would be one more round
  // trip. Thread u < 64 MB NB: rows 4 grp .. + 3 of one column of block u / 64.
  const int eb = wave % NB, er = wave / NB, en = n0 + 16 * eb + col, em = m0 + 16 * er + 4 * grp;
  const bool mine = wave < MB * NB && en < g.n;
  float *const out = g.out + (mine ? (size_t)(g.map ? g.map[en] : en) * g.ldc : 0);
  f32x4 add0 = {0.0f, 0.0f, 0.0f, 0.0f}, add1 = add0;
  if (mine) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (em + i < g.m) {
        if (g.accumulate) add0[i] = out[em + i];
        if (g.bias) add0[i] += g.bias[em + i];
        if (GEGLU && g.bias) add1[i] = g.bias[g.half + em + i];
      }
  }
  f32x4 acc[RM][NB];
#pragma unroll
  for (int r = 0; r < RM; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[r][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int base = 0; base < nchunk; base += 8 * CB) {
    // This lane's four k of chunk i: a wave takes chunks in pairs, whole
    // 128-byte lines of every row.
    auto kidx = [&](int i) { return 16 * (base + 16 * (i >> 1) + 2 * wave + (i & 1)) + 4 * grp; };
    f32x4 a[RM][CB], x[NB][CB], lw[LN ? CB : 1], lb[LN ? CB : 1];
#pragma unroll
    for (int i = 0; i < CB; ++i) {  // K % 4 == 0: a lane's four are all in or all out
      const int k = kidx(i), kc = k < K ? k : 0;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(xcol[b] + kc);
        x[b][i] = k < K ? v : zero;
      }
#pragma unroll
      for (int r = 0; r < RM; ++r) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(wrow[r] + kc);
        a[r][i] = k < K ? v : zero;
      }
      if constexpr (LN) {
        lw[i] = *reinterpret_cast<const f32x4 *>(g.ln_w + kc);
        lb[i] = g.ln_b ? *reinterpret_cast<const f32x4 *>(g.ln_b + kc) : zero;
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load is out before the first product
    if constexpr (LN) {
      // layer_norm_host (laya-infer model.rs:387-422): mean, then the mean of
      // squared deviations; a column's elements sit in four lane groups of
      // eight waves.
      auto total = [&](float (&p)[NB]) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          p[b] = pair_sum(pair16_sum(p[b]));
          if (grp == 0) s_stat[(wave * NB + b) * 16 + col] = p[b];
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          p[b] = 0.0f;
#pragma unroll
          for (int w = 0; w < 8; ++w) p[b] += s_stat[(w * NB + b) * 16 + col];
          p[b] /= (float)K;
        }
        __syncthreads();
      };
      float mean[NB], var[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        mean[b] = 0.0f;
#pragma unroll
        for (int i = 0; i < CB; ++i) mean[b] += (x[b][i][0] + x[b][i][1]) + (x[b][i][2] + x[b][i][3]);
      }
      total(mean);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        var[b] = 0.0f;
#pragma unroll
        for (int i = 0; i < CB; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float t = x[b][i][e] - mean[b];
            var[b] += kidx(i) < K ? t * t : 0.0f;
          }
      }
      total(var);
#pragma unroll
      for (int b = 0; b < NB; ++b) var[b] = 1.0f / sqrtf(var[b] + g.eps);
#pragma unroll
      for (int i = 0; i < CB; ++i)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float y = (x[b][i][e] - mean[b]) * var[b] * lw[i][e] + lb[i][e];
            x[b][i][e] = kidx(i) < K ? y : 0.0f;
          }
    }
#pragma unroll
    for (int i = 0; i < CB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int r = 0; r < RM; ++r)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[r][b] = mfma_16x16x4(a[r][i][e], x[b][i][e], acc[r][b]);
  }
#pragma unroll
  for (int r = 0; r < RM; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) s_acc[((wave * RM + r) * NB + b) * 64 + lane] = acc[r][b];
  __syncthreads();
  if (!mine) return;
  auto sum = [&](int r) {
    f32x4 v = s_acc[(r * NB + eb) * 64 + lane];
#pragma unroll
    for (int w = 1; w < 8; ++w) v += s_acc[((w * RM + r) * NB + eb) * 64 + lane];
    return v;
  };
  const f32x4 v0 = sum(GEGLU ? 0 : er) + add0;
  f32x4 y;
  if constexpr (GEGLU) {
    const f32x4 v1 = sum(RM - 1) + add1;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = gelu_erf(v0[i]) * v1[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = activate(v0[i], g.act);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (em + i < g.m) out[em + i] = y[i];
}

template <int RM, int NB, bool GEGLU>
hipError_t launch_nb(const SkinnyArgs &g, hipStream_t stream) {
  constexpr int MB = GEGLU ? 1 : RM;
  const dim3 grid((unsigned)((g.m + 16 * MB - 1) / (16 * MB)), (unsigned)((g.n + 16 * NB - 1) / (16 * NB)));
  const dim3 block(512);
  if (!g.ln_w)
    hipLaunchKernelGGL((skinny_kernel<RM, NB, 6, false, GEGLU>), grid, block, 0, stream, g);
  else if (g.k <= 768)
    hipLaunchKernelGGL((skinny_kernel<RM, NB, 6, true, GEGLU>), grid, block, 0, stream, g);
  else
    hipLaunchKernelGGL((skinny_kernel<RM, NB, 8, true, GEGLU>), grid, block, 0, stream, g);
  return hipGetLastError();
}

}  // namespace

// 32 columns per workgroup where that still gives half the CUs one, 32 weight
// rows as well where the grid would take more than one round (one workgroup
// with a LayerNorm per CU, two without).
hipError_t launch_skinny(const SkinnyArgs &g, int cus, hipStream_t stream) {
  if (g.m <= 0 || g.n <= 0) return hipSuccess;
  const long mb = (g.m + 15) / 16, nb2 = (g.n + 31) / 32;
  const bool two = g.n > 16 && mb * nb2 >= cus / 2;
  if (g.half > 0) return two ? launch_nb<2, 2, true>(g, stream) : launch_nb<2, 1, true>(g, stream);
  if (!two) return launch_nb<1, 1, false>(g, stream);
  return mb * nb2 > (g.ln_w ? cus : 2 * cus) ? launch_nb<2, 2, false>(g, stream)
                                            : launch_nb<1, 2, false>(g, stream);
}

}  // namespace tfd
