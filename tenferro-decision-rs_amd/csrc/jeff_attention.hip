// Jeff (Qwen3.5) full attention on gfx950 matrix cores.
//
// Arithmetic follows cpu-kernels jeff_full_attention_into
// (crates/cpu-kernels/src/lib.rs:609-763): per head, centered RMSNorm of q and
// k with x * (scale * (1 + w)) (676-691), partial RoPE on channel pairs
// (i, i + rot/2) with angle t * theta^(-2i/rot) (692-709, table built on the
// host with the same f32 libm calls), keys with key > query or mask == 0 are
// dropped (716), s = (q.k)/sqrt(hd), softmax, o = sum p*v skipping p == 0 and
// o = 0 when nothing is kept (731-754), out = o * 1/(1 + exp(-gate)) (755-758).
//
// Layout: every (L, W) tensor is token-contiguous (element t + L*f), so a
// wavefront's 32 queries or a tile's 32 keys are one 128-byte run per
// feature.
//
// One workgroup = 4 wavefronts sharing one kv head. With G = heads/kv_heads
// query heads per kv head, a workgroup holds hg = gcd(G, 4) heads x (4/hg)
// query sub-tiles of 16, so each K/V tile staged in LDS is used by every
// query head of the group (native GQA). K is RMS-normalized and rotated while
// it is staged; Q is normalized and rotated once per wave into registers.
// Key tiles outside [first active key, last query] are never visited.
//
// Each wavefront owns 16 queries and walks 32-key tiles on the 16x16x4 f32
// MFMA: S^T = K Q^T as two 16-key blocks, then O^T += V^T P^T. At hd = 256
// this keeps Q (hd/4 registers) and O^T (hd/4) within one wave's registers.
#include <type_traits>

#include "jeff_common.hpp"
#include "tfd_device.hpp"
#include "tfd_internal.hpp"

namespace tfd {

// Scans one row's key mask: first and last active key (mask != 0).
__device__ __forceinline__ void scan_active(const float *maskr, int L, int tid, int lane,
                                            int *s_span) {
  int lo = 0x7fffffff, hi = -1;
  for (int k0 = 0; k0 < L; k0 += 256 * 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {  // 8 loads in flight per thread
      const int k = k0 + tid + 256 * u;
      const float x = maskr[min(k, L - 1)];
      v[u] = k < L ? x : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = k0 + tid + 256 * u;
      if (v[u] != 0.0f) {
        lo = min(lo, k);
        hi = max(hi, k);
      }
    }
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  if (lane == 0) {
    atomicMin(&s_span[0], lo);
    atomicMax(&s_span[1], hi);
  }
}

// First active key of a row (rows with no active key: 0), for TFD_TRIM_LEADING.
__device__ __forceinline__ int row_start(const JeffArgs &a, const float *maskr, int tid, int lane,
                                         int *s_span) {
  if (!a.trim) return 0;
  if (tid == 0) {
    s_span[0] = 0x7fffffff;
    s_span[1] = -1;
  }
  __syncthreads();
  scan_active(maskr, a.L, tid, lane, s_span);
  __syncthreads();
  return s_span[1] >= 0 ? s_span[0] : 0;
}

// ---------------------------------------------------------------- K prep

// First active key of a row (mask != 0; 0 for a row with none), computed by
// one wave on its own.
__device__ __forceinline__ int wave_first_active(const float *maskr, int L, int lane) {
  int lo = 0x7fffffff;
  for (int k0 = 0; k0 < L; k0 += 64 * 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = maskr[min(k0 + lane + 64 * u, L - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k0 + lane + 64 * u < L && v[u] != 0.0f) lo = min(lo, k0 + lane + 64 * u);
  }
  lo = wave_min(lo);
  return __builtin_amdgcn_readfirstlane(lo == 0x7fffffff ? 0 : lo);
}

// Row span of the mask, computed by one wave on its own (no barrier): first
// and last active key (mask != 0), or (0, -1) for a row with none.
__device__ __forceinline__ void wave_active_span(const float *maskr, int L, int lane, int &first,
                                                 int &last) {
  int lo = 0x7fffffff, hi = -1;
  for (int k0 = 0; k0 < L; k0 += 64 * 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = maskr[min(k0 + lane + 64 * u, L - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = k0 + lane + 64 * u;
      if (k < L && v[u] != 0.0f) {
        lo = min(lo, k);
        hi = max(hi, k);
      }
    }
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  first = __builtin_amdgcn_readfirstlane(hi >= 0 ? lo : 0);
  last = __builtin_amdgcn_readfirstlane(hi);
}

// One wavefront: the row's active keys (mask != 0) as one bit per key (zero
// past L, 32 keys per word) and its (first, last) span, (0, -1) for a row
// with none, for the attention kernels' scalar loads.
__device__ void write_row_bits_span(const float *__restrict__ maskr, int L, int lane, int row,
                                    int *__restrict__ spans, uint32_t *__restrict__ kbits) {
  uint32_t *bits = kbits + (size_t)row * ((L + 31) / 32);
  int lo = 0x7fffffff, hi = -1;
  for (int b0 = 0; b0 < L; b0 += 64 * 8) {
    float mv[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) mv[v] = maskr[min(b0 + 64 * v + lane, L - 1)];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int kb = b0 + 64 * v;
      const uint64_t bm = __ballot(kb + lane < L && mv[v] != 0.0f);
      if (lane == 0 && kb < L) {
        bits[kb / 32] = (uint32_t)bm;
        if (kb + 32 < L) bits[kb / 32 + 1] = (uint32_t)(bm >> 32);
      }
      if (bm != 0) {
        lo = min(lo, kb + (int)__builtin_ctzll(bm));
        hi = max(hi, kb + 63 - (int)__builtin_clzll(bm));
      }
    }
  }
  if (lane == 0) {
    spans[2 * row] = hi >= 0 ? lo : 0;
    spans[2 * row + 1] = hi;
  }
}

// RMSNorm (lib.rs:676-691) and partial RoPE (692-709) of every key of one
// (row, kv head) once per call, so attention workgroups stage finished keys.
// One workgroup = 32 keys; output kp[row][kvh][key][HDP] (zero-padded past
// hd), written in whole 16-byte chunks. Out: f32, or for the bf16 attention
// kernels fp16 (RNE) of the key times 2^-e, e = norm_weight_exp(k_norm): the
// Q.K^T product of those kernels takes fp16 operands. Every global load
// (keys, norm weights, RoPE table)
// is issued before the first is used. With kbits set, the workgroups of kv
// head 0 also write their 32 keys' active bits (mask != 0), one word each.

template <int HDP, typename OutT>
__global__ __launch_bounds__(256) void jeff_k_prep_kernel(const JeffArgs a, OutT *__restrict__ kp,
                                                          uint32_t *__restrict__ kbits) {
  constexpr int DP = HDP / 8;  // dims per thread: 8 threads per key
  // LDS rows of the tile: feature d of key k at kx(k, d), one pad word after
  // every 32 features, so that the output loop's lanes (8 consecutive
  // features each, 32 lanes along one key) hit 32 different banks (with
  // rows of HDP + 1 they shared 4 of them).
  constexpr int KS = HDP + HDP / 32 + 1;
  auto kx = [](int k, int d) { return k * KS + d + (d >> 5); };
  constexpr int RT = (HDP / 2 + 7) / 8;  // RoPE pairs per thread, at most
  __shared__ float Kt[kKeyTile * KS];
  __shared__ float s_red[8 * kKeyTile];
  const int tid = threadIdx.x, lane = tid & 63;
  const int row = blockIdx.z, kvh = blockIdx.y;
  const int L = a.L, hd = a.hd, rh = a.rot_half;
  // Key blocks 2m and 2m + 1 go to workgroups i and i + 8 of each 16, which
  // the dispatcher sends to one XCD: in bf16 the two blocks are the two
  // halves of every 128-byte run of a feature's keys, so the second half's
  // loads find the run in that XCD's L2 (C5 prep 16.1 -> 15.1 us).
  int kb = (int)blockIdx.x;
  if ((gridDim.x & 15) == 0) {
    const int g = kb >> 4, r = kb & 15;
    kb = 16 * g + 2 * (r & 7) + (r >> 3);
  }
  const int k0 = kb * kKeyTile;
  const bool bf = sizeof(OutT) == 2;
  const size_t kv_off = row * a.kv_row + (size_t)kvh * a.kv_head;
  const int kk = tid & 31, part = tid >> 5;
  const int key = k0 + kk;
  const bool kin = key < L;
  const bool rope = a.cos_t != nullptr && rh > 0;
  const int start = a.trim ? wave_first_active(a.mask + (size_t)row * L, L, lane) : 0;
  if (kbits != nullptr && kvh == 0 && tid < 64) {
    const float mv = a.mask[(size_t)row * L + min(k0 + lane, L - 1)];
    const uint64_t bm = __ballot(lane < kKeyTile && k0 + lane < L && mv != 0.0f);
    if (lane == 0) kbits[(size_t)row * ((L + 31) / 32) + kb] = (uint32_t)bm;
  }
  float xs[DP], wn[DP], c[RT], sn[RT];
#pragma unroll
  for (int i = 0; i < DP; ++i) {
    const int d = part * DP + i;
    const int dc = d < hd ? d : hd - 1;
    const size_t at = kv_off + (kin ? key : 0) + (size_t)L * dc;
    xs[i] = bf ? __uint_as_float((uint32_t)static_cast<const uint16_t *>(a.k)[at] << 16)
               : static_cast<const float *>(a.k)[at];
  }
  // Norm weights: 16 bytes per load when the thread's run is whole and aligned.
  if (DP % 4 == 0 && part * DP + DP <= hd && (reinterpret_cast<uintptr_t>(a.k_norm) & 15) == 0) {
#pragma unroll
    for (int i = 0; i < DP; i += 4) {
      const f32x4 w4 = *reinterpret_cast<const f32x4 *>(a.k_norm + part * DP + i);
#pragma unroll
      for (int t = 0; t < 4; ++t) wn[i + t] = w4[t];
    }
  } else {
#pragma unroll
    for (int i = 0; i < DP; ++i) wn[i] = a.k_norm[min(part * DP + i, hd - 1)];
  }
  // Thread (kk, part) rotates pairs i = part, part + 8, ... of key k0 + kk.
  const size_t pos = (size_t)min(max(key - start, 0), L - 1) * rh;
  if (rope) {
#pragma unroll
    for (int u = 0; u < RT; ++u) {
      // Only the pairs below rot/2 are rotated (8u < rh: uniform).
      if (8 * u < rh) {
        const int i = min(part + 8 * u, rh - 1);
        c[u] = a.cos_t[pos + i];
        sn[u] = a.sin_t[pos + i];
      }
    }
  }
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < DP; ++i) {
    const int d = part * DP + i;
    xs[i] = (kin && d < hd) ? xs[i] : 0.0f;
    ss += xs[i] * xs[i];
  }
  s_red[part * kKeyTile + kk] = ss;
  __syncthreads();
  {
    float tot = 0.0f;
#pragma unroll
    for (int p = 0; p < 8; ++p) tot += s_red[p * kKeyTile + kk];
    const float scale = rms_scale(tot, hd, a.eps);
#pragma unroll
    for (int i = 0; i < DP; ++i) {
      const int d = part * DP + i;
      Kt[kx(kk, d)] = (kin && d < hd) ? rms_apply(xs[i], scale, wn[i]) : 0.0f;
    }
  }
  if (rope) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < RT; ++u) {
      const int i = part + 8 * u;
      if (i < rh && kin) {
        const float x = Kt[kx(kk, i)], y = Kt[kx(kk, i + rh)];
        Kt[kx(kk, i)] = rope_lo(x, y, c[u], sn[u]);
        Kt[kx(kk, i + rh)] = rope_hi(x, y, c[u], sn[u]);
      }
    }
  }
  __syncthreads();
  OutT *dst = kp + (((size_t)row * a.kv_heads + kvh) * L + k0) * HDP;
  const int nkeys = min(kKeyTile, L - k0);
  const float ksig = bf ? ldexpf(1.0f, -norm_weight_exp(a.k_norm, hd, lane)) : 1.0f;
  constexpr int CH = 16 / (int)sizeof(OutT);  // elements per 16-byte chunk
  for (int e = tid; e < nkeys * (HDP / CH); e += 256) {
    const int k2 = e / (HDP / CH), d0 = (e % (HDP / CH)) * CH;
    const float *src = &Kt[kx(k2, d0)];  // d0 .. d0 + CH - 1 share one 32-feature run
    if constexpr (sizeof(OutT) == 2) {
      u16x8 o;
#pragma unroll
      for (int t = 0; t < 8; ++t) o[t] = f32_to_f16_bits(src[t] * ksig);
      *reinterpret_cast<u16x8 *>(dst + (size_t)k2 * HDP + d0) = o;
    } else {
      const f32x4 o = {src[0], src[1], src[2], src[3]};
      *reinterpret_cast<f32x4 *>(dst + (size_t)k2 * HDP + d0) = o;
    }
  }
}

// Planes of the f32 kernel at hd 256: per (row, kv head) and 32-key tile 96
// KB in the order the 16x16x32 bf16 matrix cores read them, every f32 as three
// bf16 (split_bf16x3; blocks of three 1 KB planes, 16 bytes per lane). K: blocks
// (16-key half b, step s), lane (key, g) holding features 32 s + 8 g .. + 7. V:
// blocks of 16 features, lane (feature, g) holding keys 4 g .. + 3 and 16 + 4 g
// .. + 3, the keys whose probabilities lane group g of S^T holds. The attention
// kernel walks a tile as four pieces: the K halves, then V's feature halves.
constexpr int kJeffBlock = 3072, kJeffPieceBytes = 8 * kJeffBlock;
constexpr int kJeffTileBytes = 4 * kJeffPieceBytes, kJeffTileV = 2 * kJeffPieceBytes;

// Writes eight elements' planes (a lane's 16 bytes in each).
__device__ __forceinline__ void write_planes(unsigned char *p, f32x4 lo, f32x4 hi) {
  const Bf16x3 a = split_bf16x3(lo), b = split_bf16x3(hi);
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8 *>(p + 1024 * i) = join_bf16(a, b, i);
}

// One workgroup = the K (blockIdx.y even) or V planes of one (row, kv head,
// 32-key tile): the split done once per call instead of once per query tile
// that reads the tile (16 or more at L 256). K: thread (key tid & 31, part
// tid >> 5) owns features 32 part .. + 31 of its key, loaded with one 128-byte
// run per feature; RMSNorm (lib.rs:676-691) with the sum of squares reduced
// over the eight parts (lane swap, then LDS), partial RoPE (692-709) in
// registers when the partner feature i + rot/2 sits in the same wave (rot/2 =
// 32: part p pairs with part p + 1, lane + 32), else through LDS. V: thread =
// feature, its 32 keys as eight 16-byte loads (dword alignment suffices).
// Workgroups with blockIdx.x == 0 of kv head 0 also write the row's active-key
// bits and key span. Bound by HBM and one memory round trip.
__global__ __launch_bounds__(256) void jeff_k_prep_split_kernel(
    const JeffArgs a, unsigned char *__restrict__ planes, int *__restrict__ spans,
    uint32_t *__restrict__ kbits) {
  constexpr int HDP = 256, KB = 32, KS = HDP + 4;
  __shared__ __attribute__((aligned(16))) float Kt[KB * KS];
  __shared__ float s_red[4 * KB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row = blockIdx.z, kvh = blockIdx.y >> 1;
  const bool is_v = (blockIdx.y & 1) != 0;
  const int L = a.L, hd = a.hd, rh = a.rot_half;
  const int k0 = blockIdx.x * KB;
  const float *maskr = a.mask + (size_t)row * L;

  // A tile with no active key is never read by a wave that computes with it.
  // Such blocks leave their workspace untouched, except the one that also
  // writes the row's bits.
  if (!(blockIdx.x == 0 && blockIdx.y == 0)) {
    const int kl = min(k0 + (lane & 31), L - 1);
    const bool act = k0 + (lane & 31) < L && maskr[kl] != 0.0f;
    if (__ballot(act) == 0) return;  // the same in every wave
  }
  const size_t unit = ((size_t)row * a.kv_heads + kvh) * gridDim.x + blockIdx.x;
  unsigned char *tile = planes + unit * kJeffTileBytes;

  if (is_v) {
    const float *V = static_cast<const float *>(a.v) + row * a.kv_row + (size_t)kvh * a.kv_head;
    const __amdgpu_buffer_rsrc_t rv = buffer_rsrc(V, (uint32_t)((size_t)hd * L * 4));
    f32x4 x[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) x[c] = buffer_load4(rv, (tid * L + 4 * c) * 4, k0 * 4);
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)  // past L lies the next feature; past hd the loads read 0
        x[c][e] = k0 + 4 * c + e < L ? x[c][e] : 0.0f;
    unsigned char *p = tile + kJeffTileV + (tid >> 4) * kJeffBlock + (tid & 15) * 16;
#pragma unroll
    for (int g = 0; g < 4; ++g) write_planes(p + 256 * g, x[g], x[4 + g]);
    return;
  }

  const float *K = static_cast<const float *>(a.k) + row * a.kv_row + (size_t)kvh * a.kv_head;
  const __amdgpu_buffer_rsrc_t rk = buffer_rsrc(K, (uint32_t)((size_t)hd * L * 4));
  const int kk = tid & 31, part = tid >> 5;  // this thread's key and 32-feature part
  const int key = k0 + kk;
  const bool kin = key < L;
  float kv[32];
  {
    const int off = (32 * part * L + key) * 4;  // features past hd read as 0
#pragma unroll
    for (int i = 0; i < 32; ++i) kv[i] = buffer_load1(rk, off, i * L * 4);
  }
  const __amdgpu_buffer_rsrc_t rn = buffer_rsrc(a.k_norm, (uint32_t)(hd * 4));
  f32x4 wn[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) wn[c] = buffer_load4(rn, (32 * part + 4 * c) * 4, 0);
  const bool rope = a.cos_t != nullptr && rh > 0;
  const int start = a.trim ? wave_first_active(maskr, L, lane) : 0;
  const size_t pos = (size_t)min(max(key - start, 0), L - 1) * rh;
  f32x4 tc[8], ts[8];  // rot/2 == 32, parts 0 and 1 (wave 0): pairs i = 4c + e of its key
  if (rope && rh == 32 && part < 2) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      tc[c] = *reinterpret_cast<const f32x4 *>(a.cos_t + pos + 4 * c);
      ts[c] = *reinterpret_cast<const f32x4 *>(a.sin_t + pos + 4 * c);
    }
  }
  if (blockIdx.x == 0 && kvh == 0 && wave == 0) write_row_bits_span(maskr, L, lane, row, spans, kbits);

  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    kv[i] = kin ? kv[i] : 0.0f;  // past L lies the next feature
    ss += kv[i] * kv[i];
  }
  ss = pair_sum(ss);  // the wave's two parts of this key
  if (lane < 32) s_red[wave * KB + lane] = ss;
  __syncthreads();
  const float tot = s_red[kk] + s_red[KB + kk] + s_red[2 * KB + kk] + s_red[3 * KB + kk];
  const float scale = rms_scale(tot, hd, a.eps);
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = 32 * part + 4 * c + e;
      kv[4 * c + e] = (kin && d < hd) ? rms_apply(kv[4 * c + e], scale, wn[c][e]) : 0.0f;
    }
  if (rope && rh == 32) {
    // Part 0 (lanes 0..31 of wave 0) holds pairs i = j, part 1 (lanes
    // 32..63 of the same wave) their partners i + 32.
    if (wave == 0) {
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(kv[j]),
                                                        __float_as_uint(kv[j]), false, false);
        const float other = __uint_as_float(lane < 32 ? r[1] : r[0]);
        const float xl = part == 0 ? kv[j] : other, yh = part == 0 ? other : kv[j];
        const float cc = tc[j >> 2][j & 3], sn = ts[j >> 2][j & 3];
        if (kin) kv[j] = part == 0 ? rope_lo(xl, yh, cc, sn) : rope_hi(xl, yh, cc, sn);
      }
    }
  } else if (rope) {
#pragma unroll
    for (int j = 0; j < 32; ++j) Kt[kk * KS + 32 * part + j] = kv[j];
    __syncthreads();
    if (kin) {
      for (int i = part; i < rh; i += 8) {
        const float xl = Kt[kk * KS + i], yh = Kt[kk * KS + i + rh];
        const float cc = a.cos_t[pos + i], sn = a.sin_t[pos + i];
        Kt[kk * KS + i] = rope_lo(xl, yh, cc, sn);
        Kt[kk * KS + i + rh] = rope_hi(xl, yh, cc, sn);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 32; ++j) kv[j] = Kt[kk * KS + 32 * part + j];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)  // step part, lane group c
    write_planes(tile + ((kk >> 4) * 8 + part) * kJeffBlock + (c * 16 + (kk & 15)) * 16,
                 f32x4{kv[8 * c], kv[8 * c + 1], kv[8 * c + 2], kv[8 * c + 3]},
                 f32x4{kv[8 * c + 4], kv[8 * c + 5], kv[8 * c + 6], kv[8 * c + 7]});
}

// ----------------------------------------------------------- f32 attention

// RMSNorm + partial RoPE of one wave's 16 queries of one head into the
// B-operand registers of S^T = K Q^T: lane (col, grp) ends with
// Qn[q0 + col][grp*QS + s]. Goes through the wave's own LDS rows qw
// (16 x (HDP + 4) floats): raw rows (16-byte loads along tokens when VEC),
// normalized in registers, rotated pairs in LDS, read back. Queries that are
// past L or dropped (q < start) get zeros.
template <int HDP, bool VEC>
__device__ __forceinline__ void jeff_q_prep(const JeffArgs &a, const float *Q, int q0, int start,
                                            float *qw, float (&qreg)[HDP / 4]) {
  constexpr int QS = HDP / 4, QP = HDP + 4;
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int L = a.L, hd = a.hd, rh = a.rot_half;
  const int q = q0 + col;
  const bool q_live = q < L && q >= start;
  // Issued first, so that they share the Q loads' round trip: this lane's
  // norm weights (past hd they read 0 or anything; those dims are zeroed
  // below) and the table entries of its first 8 RoPE pairs i = grp + 4u.
  const __amdgpu_buffer_rsrc_t rn = buffer_rsrc(a.q_norm, (uint32_t)(hd * 4));
  f32x4 wv[QS / 4];
#pragma unroll
  for (int c = 0; c < QS / 4; ++c) wv[c] = buffer_load4(rn, (grp * QS + 4 * c) * 4, 0);
  const bool rope = a.cos_t != nullptr && rh > 0;
  const size_t pos = (size_t)min(max(q - start, 0), L - 1) * rh;
  float c8[8], s8[8];
  if (rope) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = min(grp + 4 * u, rh - 1);
      c8[u] = a.cos_t[pos + i];
      s8[u] = a.sin_t[pos + i];
    }
  }
  if constexpr (VEC) {
    // Task (d, g): queries q0 + 4g .. +3 of feature d, one 16-byte load;
    // features past hd read as 0.
    const __amdgpu_buffer_rsrc_t rq = buffer_rsrc(Q, (uint32_t)((size_t)hd * L * 4));
#pragma unroll
    for (int i0 = 0; i0 < HDP * 4; i0 += 64 * 4) {
      f32x4 x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // HDP * 4 < 256 only at HDP = 32: clamp, skip below
        const int e = min(i0 + lane + 64 * u, HDP * 4 - 1), d = e >> 2, g = e & 3;
        x[u] = buffer_load4(rq, (int)(((size_t)d * L + 4 * g) * 4), q0 * 4);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = i0 + lane + 64 * u, d = e >> 2, g = e & 3;
        if (HDP * 4 % 256 == 0 || e < HDP * 4) {
#pragma unroll
          for (int t = 0; t < 4; ++t) qw[(4 * g + t) * QP + d] = x[u][t];
        }
      }
    }
  } else {
    for (int e0 = 0; e0 < 16 * HDP; e0 += 64 * 8) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = e0 + lane + 64 * u, d = e >> 4, t = e & 15;
        x[u] = Q[min(q0 + t, L - 1) + (size_t)L * min(d, hd - 1)];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = e0 + lane + 64 * u, d = e >> 4, t = e & 15;
        qw[t * QP + d] = d < hd ? x[u] : 0.0f;
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float *qs = qw + col * QP + grp * QS;
  f32x4 xv[QS / 4];
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < QS / 4; ++c) {
    xv[c] = *reinterpret_cast<const f32x4 *>(qs + 4 * c);
    ss += xv[c][0] * xv[c][0] + xv[c][1] * xv[c][1] + xv[c][2] * xv[c][2] + xv[c][3] * xv[c][3];
  }
  ss += __shfl_xor(ss, 16);
  ss += pair_sum(ss) - ss;  // lanes l and l ^ 32 hold the other two groups
  const float scale = rms_scale(ss, hd, a.eps);
#pragma unroll
  for (int c = 0; c < QS / 4; ++c) {
    f32x4 y;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int d = grp * QS + 4 * c + t;
      y[t] = (q_live && d < hd) ? rms_apply(xv[c][t], scale, wv[c][t]) : 0.0f;
    }
    *reinterpret_cast<f32x4 *>(qs + 4 * c) = y;
  }
  if (rope) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // Lane (col, grp) rotates pairs i = grp, grp + 4, ... of query q0 + col;
    // the first 8 with the entries loaded up front.
    if (q_live) {
      float *qr = qw + col * QP;
      for (int i0 = grp; i0 < rh; i0 += 4 * 8) {
        float c[8], sn[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = min(i0 + 4 * u, rh - 1);
          c[u] = i0 == grp ? c8[u] : a.cos_t[pos + i];
          sn[u] = i0 == grp ? s8[u] : a.sin_t[pos + i];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + 4 * u;
          if (i < rh) {
            const float x = qr[i], y = qr[i + rh];
            qr[i] = rope_lo(x, y, c[u], sn[u]);
            qr[i + rh] = rope_hi(x, y, c[u], sn[u]);
          }
        }
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int c = 0; c < QS / 4; ++c) {
    const f32x4 y = *reinterpret_cast<const f32x4 *>(qs + 4 * c);
#pragma unroll
    for (int t = 0; t < 4; ++t) qreg[4 * c + t] = y[t];
  }
}

// o = O^T * inv (0 when nothing was kept), times the sigmoid gate, stored
// feature-major: the wave writes its 16 x HDP block through its LDS rows ow
// (16 x (HDP + 4) floats) so that gate loads and output stores run along
// tokens, 16 bytes at a time, when VEC. Dropped queries (q < start) get 0.
// Only features d_lo <= d < d_hi are stored (a workgroup that owns part of
// the head's features).
template <int HDP, bool VEC>
__device__ __forceinline__ void jeff_store(const JeffArgs &a, const float *Gt, float *OUT, int q0,
                                           int start, float *ow, const f32x4 (&O)[HDP / 16],
                                           float inv, int d_lo = 0, int d_hi = 1 << 30) {
  constexpr int NB = HDP / 16, QP = HDP + 4;
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int L = a.L, hd = a.hd;
  if constexpr (VEC) {
    // The gate loads go out before O is written to LDS.
    const __amdgpu_buffer_rsrc_t rg = buffer_rsrc(Gt, (uint32_t)((size_t)hd * L * 4));
    const __amdgpu_buffer_rsrc_t ro = buffer_rsrc(OUT, (uint32_t)((size_t)hd * L * 4));
    constexpr int NG = (HDP * 4 + 63) / 64;
    f32x4 g[NG];
#pragma unroll
    for (int u = 0; u < NG; ++u) {  // clamped as in the Q prep
      const int e = min(lane + 64 * u, HDP * 4 - 1), d = e >> 2, gq = e & 3;
      g[u] = buffer_load4(rg, (int)(((size_t)d * L + 4 * gq) * 4), q0 * 4);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const f32x4 v = O[j] * inv;  // dims 16j + 4grp + 0..3 of query q0 + col
      *reinterpret_cast<f32x4 *>(ow + col * QP + 16 * j + 4 * grp) = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    {
      const int i0 = 0;
#pragma unroll
      for (int u = 0; u < NG; ++u) {
        const int e = min(i0 + lane + 64 * u, HDP * 4 - 1), d = e >> 2, gq = e & 3;
        const int qa = q0 + 4 * gq;
        f32x4 o;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float x = ow[(4 * gq + t) * QP + d] * fast_sigmoid(g[u][t]);
          o[t] = qa + t < start ? 0.0f : x;
        }
        if (d < hd && d >= d_lo && d < d_hi) {
          const int off = (int)(((size_t)d * L + 4 * gq) * 4);
          if (qa + 4 <= L) {
            buffer_store4_nt(o, ro, off, q0 * 4);
          } else {  // the row ends inside these four queries (L % 4 != 0) or before them
#pragma unroll
            for (int t = 0; t < 3; ++t)
              if (qa + t < L) buffer_store1_nt(o[t], ro, off + 4 * t, q0 * 4);
          }
        }
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const f32x4 v = O[j] * inv;  // dims 16j + 4grp + 0..3 of query q0 + col
      *reinterpret_cast<f32x4 *>(ow + col * QP + 16 * j + 4 * grp) = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int e0 = 0; e0 < 16 * HDP; e0 += 64 * 8) {
      float g[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = e0 + lane + 64 * u, d = e >> 4, t = e & 15;
        g[u] = Gt[min(q0 + t, L - 1) + (size_t)L * min(d, hd - 1)];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = e0 + lane + 64 * u, d = e >> 4, t = e & 15;
        const int qq = q0 + t;
        if (qq < L && d < hd && d >= d_lo && d < d_hi)
          __builtin_nontemporal_store(qq < start ? 0.0f : ow[t * QP + d] * fast_sigmoid(g[u]),
                                      &OUT[qq + (size_t)L * d]);
      }
    }
  }
}

// Tile data for one 16-key tile, prefetched into registers: finished K rows
// from the prep workspace and V columns, all 16-byte buffer loads with a
// fixed per-lane offset and a scalar tile offset (VEC), or element loads
// with clamped indices. Keys past L read as 0 (K) or are zeroed at commit
// (V). LDS holds K as [key][d] and V as [d][key], V's layout in memory.
template <int HDP, bool VEC, int NT>
struct JeffStage {
  static constexpr int KT = kJeffKeyTile;
  static constexpr int TASKS = KT * HDP / 4;       // 16-byte chunks of K (and of V)
  static constexpr int KN = (TASKS + NT - 1) / NT;  // chunks per thread (NT threads)
  f32x4 k[KN], v[KN];
  __amdgpu_buffer_rsrc_t rk, rv;
  int ok[KN], ov[KN];

  __device__ __forceinline__ void init(const float *KP, const float *V, int L, int hd, int tid) {
    rk = buffer_rsrc(KP, (uint32_t)((size_t)L * HDP * 4));
    rv = buffer_rsrc(V, (uint32_t)((size_t)hd * L * 4));
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const int e = min(tid + NT * i, TASKS - 1);
      ok[i] = e * 16;                                  // chunk e of the KT x HDP tile
      const int d = e / (KT / 4), g = e % (KT / 4);    // feature d, keys 4g .. 4g+3
      ov[i] = (int)(((size_t)d * L + 4 * g) * 4);
    }
  }

  __device__ __forceinline__ void fetch(const float *KP, const float *V, int L, int hd, int k0,
                                        int tid) {
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < KN; ++i) {
        k[i] = buffer_load4(rk, ok[i], k0 * HDP * 4);
        v[i] = buffer_load4(rv, ov[i], k0 * 4);
      }
    } else {
#pragma unroll
      for (int i = 0; i < KN; ++i) {
        const int e = min(tid + NT * i, TASKS - 1);
        const int kk = min((4 * e) / HDP, L - 1 - k0);
        k[i] = reinterpret_cast<const f32x4 *>(KP + (size_t)k0 * HDP)[kk * (HDP / 4) + e % (HDP / 4)];
        const int d = min(e / (KT / 4), hd - 1), g = e % (KT / 4);
        const float *src = V + (size_t)L * d;
#pragma unroll
        for (int t = 0; t < 4; ++t) v[i][t] = src[min(k0 + 4 * g + t, L - 1)];
      }
    }
  }

  __device__ __forceinline__ void commit(float *Ks, float *Vs, int tid, int k0, int L, int hd) {
    constexpr int KS = HDP + 4, VS = KT + 4;
    const bool tail = k0 + KT > L;  // uniform: the row's last, partial tile
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const int e = tid + NT * i;
      if (TASKS % NT == 0 || e < TASKS) {  // blockDim is NT
        const int kk = (4 * e) / HDP, dk = (4 * e) % HDP;
        f32x4 kv = k[i];
        const int d = e / (KT / 4), g = e % (KT / 4);
        f32x4 vv = v[i];
        if (!VEC || tail) {
#pragma unroll
          for (int t = 0; t < 4; ++t) vv[t] = (d < hd && k0 + 4 * g + t < L) ? vv[t] : 0.0f;
          if (k0 + kk >= L) kv = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        *reinterpret_cast<f32x4 *>(&Ks[kk * KS + dk]) = kv;
        *reinterpret_cast<f32x4 *>(&Vs[d * VS + 4 * g]) = vv;
      }
    }
  }
};

// TAG gives each calling kernel its own copy, compiled to that kernel's
// register budget; TAG 1 (the split kernel) and TAG 2 (the fused kernels)
// normalize and rotate each key tile from K itself into LDS.
template <int HDP, bool VEC, int TAG = 0>
__device__ __noinline__ void jeff_redo_wave(const JeffArgs *ap, const float *__restrict__ kp,
                                            int row, int head, int q0, int kt_begin, int kt_end,
                                            int start, float *ws, int d_lo = 0,
                                            int d_hi = 1 << 30);

// The calling kernel's JeffArgs (its first parameter, at offset 0 of the
// kernel argument segment), for the out-of-line redo: passing the struct by
// value would make every wave copy it to scratch on entry.
__device__ __forceinline__ const JeffArgs *kernel_jeff_args() {
  return (const JeffArgs *)__builtin_amdgcn_kernarg_segment_ptr();
}

// One workgroup = 8 wavefronts (one workgroup per CU) sharing one kv head:
// hg = heads_per_group query heads x (8 / hg) query tiles of 16. The query
// tiles come in causal pairs (p, n - 1 - p), n = ceil(L / 16), so every
// workgroup carries about the same number of key tiles; the walk covers the
// group's span and a wave skips the tiles its own queries do not reach.
template <int HDP, bool VEC>
__global__ __launch_bounds__(kJeffF32Waves * 64, 1) void jeff_attention_f32_kernel(
    const JeffArgs a, const float *__restrict__ kp) {
  constexpr int NT = kJeffF32Waves * 64;
  constexpr int KT = kJeffKeyTile;  // 16 keys per tile
  constexpr int QS = HDP / 4;       // Q registers per lane (4 lane groups split hd)
  constexpr int NB = HDP / 16;      // 16-row blocks of O^T
  constexpr int KS = HDP + 4;       // K stored [key][d]
  constexpr int VS = KT + 4;        // V stored [d][key]: conflict-free 16-byte reads
  constexpr int KBUF = KT * KS, VBUF = HDP * VS;
  constexpr int QP = HDP + 4;       // per-wave Q / output rows before and after the walk
  constexpr int WROWS = kJeffF32Waves * kJeffWaveQueries * QP;
  constexpr int SMEM = WROWS > 2 * (KBUF + VBUF) ? WROWS : 2 * (KBUF + VBUF);
  __shared__ __attribute__((aligned(16))) float smem[SMEM];
  auto Ks = [&](int i) { return smem + i * KBUF; };
  auto Vs = [&](int i) { return smem + 2 * KBUF + i * VBUF; };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform, in a scalar register
  const int col = lane & 15, grp = lane >> 4;
  const int hg = a.heads_per_group, S = kJeffF32Waves / hg;  // query tiles per workgroup
  // XCD-aware order: the dispatcher hands workgroup p to XCD p % 8, each XCD
  // with its own L2. Workgroups sharing one (row, kv head) -- its K/V -- are
  // given ids p = 8*i + c for one c, so they land on one XCD; consecutive
  // groups go to consecutive XCDs.
  int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  {
    const int nx = gridDim.x, ngroups = gridDim.y * gridDim.z;
    const int p = blockIdx.x + nx * (blockIdx.y + gridDim.y * blockIdx.z);
    if (ngroups % 8 == 0) {
      const int c = p % 8, i = p / 8;  // i-th workgroup of XCD c
      const int g = 8 * (i / nx) + c;  // (row, kv group) index
      bx = i % nx;
      by = g % gridDim.y;
      bz = g / gridDim.y;
    }
  }
  const int row = bz;
  const int head = by * hg + wave % hg;
  const int kvh = min(head / a.groups, a.kv_heads - 1);
  const int L = a.L, hd = a.hd;
  const int nq = (L + kJeffWaveQueries - 1) / kJeffWaveQueries;
  const int npairs = (nq + 1) / 2;
  const int s_idx = wave / hg, pair = bx * (S / 2) + s_idx / 2;
  const bool hi_member = s_idx & 1;
  const int qtile = hi_member ? nq - 1 - pair : pair;
  // a wave with no query tile (past the pairs, or the middle tile's twin)
  const bool wave_live = pair < npairs && (!hi_member || nq - 1 - pair != pair);
  const int q0 = qtile * kJeffWaveQueries;
  const int q = q0 + col;
  // the group's last query: the upper member of its lowest pair
  const int q_last = min((nq - bx * (S / 2)) * kJeffWaveQueries, L) - 1;
  const float *maskr = a.mask + (size_t)row * L;
  const float *Q = static_cast<const float *>(a.q) + row * a.q_row + (size_t)head * hd * L;
  const float *Gt = static_cast<const float *>(a.gate) + row * a.q_row + (size_t)head * hd * L;
  const float *V = static_cast<const float *>(a.v) + row * a.kv_row + (size_t)kvh * a.kv_head;
  const float *KP = kp + ((size_t)row * a.kv_heads + kvh) * L * HDP;
  float *OUT = a.out + row * a.q_row + (size_t)head * hd * L;
  float *qw = smem + wave * (kJeffWaveQueries * QP);

  // -------- active-key span (each wave on its own); RoPE positions restart
  // at `start` when trimming. Tiles past the group's last query are causal-
  // ly dead.
  int first, last;
  wave_active_span(maskr, L, lane, first, last);
  const int start = (a.trim && last >= 0) ? first : 0;
  int kt_begin = 0, kt_end = 0;
  {
    const int kl = min(last, q_last);
    if (last >= 0 && first <= kl) {
      kt_begin = first / KT;
      kt_end = kl / KT + 1;
    }
  }
  const bool q_live = wave_live && q < L && q >= start;

  // The first tile's loads go out before the Q prep and land during it.
  JeffStage<HDP, VEC, NT> st;
  st.init(KP, V, L, hd, tid);
  float m0 = 0.0f;
  if (kt_begin < kt_end) {
    m0 = maskr[min(kt_begin * KT + col, L - 1)];
    st.fetch(KP, V, L, hd, kt_begin * KT, tid);
  }
  float qreg[QS];
  jeff_q_prep<HDP, VEC>(a, Q, wave_live ? q0 : 0, start, qw, qreg);
  __syncthreads();  // the wave rows become the K/V buffers

  // Keep word for a 16-key tile: active key, key >= start, causal key <= query.
  // The mask value is fetched one tile ahead (mask_of) and turned into the
  // word (keep_word) only after that tile's barrier.
  auto mask_of = [&](int kt) -> float { return maskr[min(kt * KT + col, L - 1)]; };
  auto keep_word = [&](int kt, float mv) -> uint32_t {
    const int k0 = kt * KT;
    const int kc = k0 + col;
    const bool act = kc < L && kc >= start && mv != 0.0f;
    const uint32_t abits = (uint32_t)__ballot(act) & 0xffffu;
    return q_live ? (abits & range_bits(0, q - k0)) : 0u;
  };

  f32x4 O[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) O[j][r] = 0.0f;
  float m = kNoMax, l = 0.0f;
  const float c1 = a.c1;

  // -------- the walk (see the Laya kernel for the scheme): tile kt+1 is
  // fetched before the products of tile kt and committed after them; one
  // barrier per tile; lazily moved exponent reference; a wave whose kept
  // scores sum to NaN or inf stops computing, and it or a wave whose O took
  // a NaN or inf redoes its queries with the reference's exact semantics.
  uint32_t w = 0u;
  float m_next = 0.0f;
  if (kt_begin < kt_end) {
    st.commit(Ks(0), Vs(0), tid, kt_begin * KT, L, hd);
    w = keep_word(kt_begin, m0);
  }
  __syncthreads();
  bool tainted = false;  // wave-uniform
  int cur = 0;
  for (int kt = kt_begin; kt < kt_end; ++kt) {
    const bool more = kt + 1 < kt_end;
    if (more) {
      m_next = mask_of(kt + 1);
      st.fetch(KP, V, L, hd, (kt + 1) * KT, tid);
    }
    if (!tainted && __ballot(w != 0u) != 0) {
      const float *Kc = Ks(cur);
      f32x4 s0, s1;  // two partial sums over alternate chunks of hd
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s0[r] = 0.0f;
        s1[r] = 0.0f;
      }
      const f32x4 *krow = reinterpret_cast<const f32x4 *>(&Kc[col * KS + grp * QS]);
#pragma unroll
      for (int c = 0; c < QS / 4; ++c) {
        const f32x4 ka = krow[c];
        if (c & 1) {
#pragma unroll
          for (int e = 0; e < 4; ++e) s1 = mfma_16x16x4(ka[e], qreg[4 * c + e], s1);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) s0 = mfma_16x16x4(ka[e], qreg[4 * c + e], s0);
        }
      }
      s0 += s1;
      // lane group g holds keys 4g + r of its query
      if (__ballot(q_live && w != 0xffffu) != 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s0[r] = ((w >> (4 * grp + r)) & 1u) ? s0[r] : -INFINITY;
      }
      float mx = fmaxf(fmaxf(s0[0], s0[1]), fmaxf(s0[2], s0[3]));
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = pair_max(mx);
      const float mxs = mx * c1;
      const bool need = mxs > m + kRescaleSlack;
      const float mn = need ? mxs : m;
      float rs = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s0[r] = fast_exp2(__builtin_fmaf(s0[r], c1, -mn));
        rs += s0[r];
      }
      if (__ballot(q_live && !(__builtin_isfinite(rs) && reference_usable(mn))) != 0) {
        tainted = true;
      } else {
        if (__ballot(need) != 0) {
          const float alpha = fast_exp2(m - mn);  // exactly 1 where the reference stays
#pragma unroll
          for (int j = 0; j < NB; ++j) O[j] *= alpha;
          l *= alpha;
        }
        l += rs;
        m = mn;
        // A operand of block j: V[key 4*grp + r][d = 16*j + col], one 16-byte read.
        const float *v0 = &Vs(cur)[col * VS + 4 * grp];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const f32x4 vv = *reinterpret_cast<const f32x4 *>(v0 + j * 16 * VS);
#pragma unroll
          for (int r = 0; r < 4; ++r) O[j] = mfma_16x16x4(vv[r], s0[r], O[j]);
        }
      }
    }
    if (more) st.commit(Ks(cur ^ 1), Vs(cur ^ 1), tid, (kt + 1) * KT, L, hd);
    __syncthreads();
    if (more) w = keep_word(kt + 1, m_next);
    cur ^= 1;
  }

  // -------- careful redo (rare), out of line; every wave's LDS reads of the
  // walk precede its last barrier, so each wave may now use its own rows.
  bool bad = false;
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) bad |= !__builtin_isfinite(O[j][r]);
  if (!wave_live) return;
  if (tainted || __ballot(q_live && bad) != 0) {
    jeff_redo_wave<HDP, VEC>(kernel_jeff_args(), kp, row, head, q0, kt_begin, kt_end, start, qw);
    return;
  }

  // -------- o / sum (0 when nothing was kept), sigmoid gate, store
  float lt = l + __shfl_xor(l, 16);
  lt = pair_sum(lt);
  const float inv = lt > 0.0f ? fast_rcp(lt) : 0.0f;
  jeff_store<HDP, VEC>(a, Gt, OUT, q0, start, qw, O, inv);
}

// The careful path for one wave's 16 queries of one head (rare: NaN or inf
// among its kept scores or values), from global memory without barriers:
// the reference's masked softmax with an exact running max (non-finite
// scores weigh 0, a +inf score empties the row) and o = sum p*v over
// p != 0 in key order (lib.rs:716-754), then the gate. Kept out of line so
// that its registers never weigh on the walk. ws: the wave's LDS rows.
template <int HDP, bool VEC, int TAG>
__device__ __noinline__ void jeff_redo_wave(const JeffArgs *ap, const float *__restrict__ kp,
                                            int row, int head, int q0, int kt_begin, int kt_end,
                                            int start, float *ws, int d_lo, int d_hi) {
  const JeffArgs &a = *ap;
  constexpr int KT = kJeffKeyTile, QS = HDP / 4, NB = HDP / 16, PS = KT + 1;
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int L = a.L, hd = a.hd;
  const int kvh = min(head / a.groups, a.kv_heads - 1);
  const int q = q0 + col;
  const bool q_live = q < L && q >= start;
  const float *maskr = a.mask + (size_t)row * L;
  const float *Q = static_cast<const float *>(a.q) + row * a.q_row + (size_t)head * hd * L;
  const float *Gt = static_cast<const float *>(a.gate) + row * a.q_row + (size_t)head * hd * L;
  const float *V = static_cast<const float *>(a.v) + row * a.kv_row + (size_t)kvh * a.kv_head;
  constexpr bool RAW = TAG != 0;  // keys straight from K, normalized per tile into LDS
  const float *KP = RAW ? nullptr : kp + ((size_t)row * a.kv_heads + kvh) * (size_t)L * HDP;
  const float *Kraw = static_cast<const float *>(a.k) + row * a.kv_row + (size_t)kvh * a.kv_head;
  constexpr int QP = HDP + 4;
  float *Kw = ws + 512;  // RAW: 16 keys x QP floats, after Pw
  float *OUT = a.out + row * a.q_row + (size_t)head * hd * L;
  float qreg[QS];
  jeff_q_prep<HDP, VEC>(a, Q, q0, start, ws, qreg);
  f32x4 O[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) O[j][r] = 0.0f;
  float m = kNoMax, l = 0.0f;
  float *Pw = ws;  // 16 keys x 17 floats, after the Q rows are consumed
#pragma unroll 1
  for (int kt = kt_begin; kt < kt_end; ++kt) {
    const int k0 = kt * KT;
    const int kc = k0 + col;
    const bool act = kc < L && kc >= start && maskr[min(kc, L - 1)] != 0.0f;
    const uint32_t abits = (uint32_t)__ballot(act) & 0xffffu;
    const uint32_t w = q_live ? (abits & range_bits(0, q - k0)) : 0u;
    if (__ballot(w != 0u) == 0) continue;
    const int kcl = min(kc, L - 1);
    if constexpr (RAW) {
      // The reference's key arithmetic (lib.rs:676-709) for keys k0 .. k0 +
      // 15: lane (col, grp) normalizes features grp*QS .. + QS - 1 of key
      // kcl, then rotates pairs i = grp, grp + 4, ... of it.
      float xk[QS];
      float ss = 0.0f;
#pragma unroll
      for (int x = 0; x < QS; ++x) {
        const int d = grp * QS + x;
        xk[x] = d < hd ? Kraw[kcl + (size_t)L * d] : 0.0f;
        ss += xk[x] * xk[x];
      }
      ss += __shfl_xor(ss, 16);
      ss += __shfl_xor(ss, 32);
      const float scale = rms_scale(ss, hd, a.eps);
#pragma unroll
      for (int x = 0; x < QS; ++x) {
        const int d = grp * QS + x;
        Kw[col * QP + d] = d < hd ? rms_apply(xk[x], scale, a.k_norm[d]) : 0.0f;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (a.cos_t != nullptr && a.rot_half > 0) {
        const int rh = a.rot_half;
        const size_t pos = (size_t)min(max(kcl - start, 0), L - 1) * rh;
        for (int i = grp; i < rh; i += 4) {
          const float x = Kw[col * QP + i], y = Kw[col * QP + i + rh];
          Kw[col * QP + i] = rope_lo(x, y, a.cos_t[pos + i], a.sin_t[pos + i]);
          Kw[col * QP + i + rh] = rope_hi(x, y, a.cos_t[pos + i], a.sin_t[pos + i]);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    const float *krow = RAW ? Kw + col * QP + grp * QS : KP + (size_t)kcl * HDP + grp * QS;
    f32x4 s;
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] = 0.0f;
#pragma unroll
    for (int x = 0; x < QS; ++x) {
      s = mfma_16x16x4(kc < L ? krow[x] : 0.0f, qreg[x], s);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float x = ((w >> (4 * grp + r)) & 1u) ? s[r] * a.c1 : -INFINITY;
      s[r] = x;
      mx = fmaxf(mx, x);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = pair_max(mx);
    const float mn = fmaxf(m, mx);
    const float alpha = (m == mn) ? 1.0f : fast_exp2(m - mn);
    float rs = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float e = __builtin_isfinite(s[r]) ? fast_exp2(s[r] - mn) : 0.0f;
      s[r] = e;
      rs += e;
    }
    l = l * alpha + rs;
    m = mn;
    // alpha == 0: earlier probabilities are 0 against the new max, so their
    // (possibly infinite) values drop out as in the reference.
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) O[j][r] = alpha == 0.0f ? 0.0f : O[j][r] * alpha;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) Pw[(4 * grp + r) * PS + col] = s[r];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
    for (int kk = 0; kk < KT; ++kk) {
      const float pk = Pw[kk * PS + col];
      if (pk == 0.0f) continue;  // only kept keys inside the row get here
      const float *vcol = V + (k0 + kk);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = 16 * j + 4 * grp + r;
          if (d < hd) O[j][r] += pk * vcol[(size_t)L * d];
        }
    }
    __builtin_amdgcn_wave_barrier();
  }
  float lt = l + __shfl_xor(l, 16);
  lt = pair_sum(lt);
  const float inv = lt > 0.0f ? fast_rcp(lt) : 0.0f;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  jeff_store<HDP, VEC>(a, Gt, OUT, q0, start, ws, O, inv, d_lo, d_hi);
}

// ------------------------------------------------- f32 attention, split head

// (row, head) of work unit u < rows * heads of the fused
// kernels, whose grids are (units, query tiles) and dispatch in the linear
// order u + units * y, workgroup id % 8 being the XCD: when the counts allow
// it, the 8 * G consecutive units of one XCD round are the G query heads of
// eight (row, kv head) pairs, so a pair's K/V tiles are read through one L2.
// The divisions go through FastDiv (operands below rows * heads, divisors
// at most heads; the launchers check rows * heads^2 <= 2^32).
__device__ __forceinline__ void jeff_unit_of(const JeffArgs &a, int rows, int u, int &row,
                                             int &head) {
  const int units = rows * a.heads, G = a.groups;
  if (units % 8 == 0 && (rows * a.kv_heads) % 8 == 0) {
    const int x = u % 8, i = u / 8;
    const int ig = (int)a.gdiv.div((uint32_t)i);
    const int kvu = x + 8 * ig;  // (row, kv head) unit of XCD x
    row = (int)a.kvdiv.div((uint32_t)kvu);
    head = (kvu - row * a.kv_heads) * G + (i - ig * G);
  } else {
    row = (int)a.hdiv.div((uint32_t)u);
    head = u - row * a.heads;
  }
}

// One workgroup = 4 wavefronts = hg query heads of a GQA group (hg = 4, 2 or
// 1) x 4 / hg query tiles of 16; a wave owns one head's 16 queries and walks
// the group's 32-key tiles with every f32 product as six bf16 ones
// (split_bf16x3, f32 accumulation):
//   S^T (2 x 16 keys x 16 queries) = K_tile Q^T     (96 MFMA 16x16x32)
//   O^T (256 x 16)                += V_tile^T P^T   (96 MFMA 16x16x32)
// 3,072 matrix-core cycles per wave and tile instead of 8,192 in f32, with
// the vector work beside them (f32 MFMAs exclude it); the operands of eight waves
// take 6,144 cycles of a CU's LDS reads, as long as its matrix cores need. The
// pieces hold all 24 bits over f32's exponent range, and a key's depend on
// that key alone: masked, future and improbable keys of any magnitude stay out of
// the others' way (fp16 pairs with a scale per tile need half the products, but do
// not have that property). Q is normalized and rotated once into registers (96 of
// them) and O^T stays there (64). The tile's planes (jeff_k_prep_split_kernel) come
// by LDS-DMA in four pieces of 24 KB through a ring of three, two pieces ahead of
// their use, so 75 KB serve a workgroup and two of them share a CU: one's loads of Q
// (a burst of the whole tensor over all CUs: 4-5 us), waits and output stores run
// beside the other's products. Cycles of a wave: Q 9,000-14,000, its norm and split
// 4,200-5,000, the first tile's arrival 2,500, a tile 6,900 alone on its SIMD and 7,800
// with another wave (3,260 of matrix-core time each), the gate and output 10,000-11,000.
// Measured with the prep (f32 MFMA -> fp16 pairs -> this): 16 rows x 256 left-padded
// 48-51 -> 39 -> 48 us, 5 rows x 333 108 -> 46 -> 57 us; relative error against 64
// bits 2.0e-7 -> 2.0e-7 -> 1.5e-7 and 2.9e-7 -> 2.1e-7 -> 1.6e-7. A ring of six with one
// workgroup per CU: 65 and 62 us.
//
// Workgroups are numbered from the last query tile down, so the longest
// causal walks start first; the workgroups of one (row, kv head) share an id
// residue mod 8 (one XCD, one L2) when rows x kv heads is a multiple of 8.
template <int HDP>
__global__ __launch_bounds__(256, 2) void jeff_split_f32_kernel(
    const JeffArgs a, const unsigned char *__restrict__ planes, const int *__restrict__ spans,
    const uint32_t *__restrict__ kbits, int rows) {
  static_assert(HDP == 256, "plane layout of 96 KB tiles");
  constexpr int NB = HDP / 16, ST = HDP / 32;
  // Per wave: the redo's rows (512 + 16 * (HDP + 4) floats), of which the Q
  // prep and the output use 16 * (HDP + 4). The ring of pieces aliases them.
  constexpr int WROWS = 512 + 16 * (HDP + 4);
  constexpr int RING = 3, PW = kJeffPieceBytes / 4096;  // 1 KB loads of a piece per wave
  static_assert(4 * WROWS * 4 >= RING * kJeffPieceBytes, "the ring aliases the wave rows");
  __shared__ __attribute__((aligned(16))) float smem[4 * WROWS];
  unsigned char *const lds = reinterpret_cast<unsigned char *>(smem);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int L = a.L, hd = a.hd, hg = a.heads_per_group;
  float *const ws = smem + wave * WROWS;

  const int kvunits = rows * a.kv_heads;
  const int sub = (int)blockIdx.x / kvunits, kvu = (int)blockIdx.x - sub * kvunits;
  const int row = (int)a.kvdiv.div((uint32_t)kvu), kvh = kvu - row * a.kv_heads;
  const int tiles = 4 / hg;  // query tiles per workgroup
  const int yg = (int)gridDim.y - 1 - (int)blockIdx.y;
  const int head = kvh * a.groups + sub * hg + wave % hg;
  const int q0 = 16 * (yg * tiles + wave / hg), q = q0 + col;
  const float *Q = static_cast<const float *>(a.q) + row * a.q_row + (size_t)head * hd * L;
  const float *Gt = static_cast<const float *>(a.gate) + row * a.q_row + (size_t)head * hd * L;
  float *OUT = a.out + row * a.q_row + (size_t)head * hd * L;
  const int nt = (L + 31) / 32;
  const unsigned char *unit = planes + (size_t)kvu * nt * kJeffTileBytes;
  const uint32_t *rbits = kbits + (size_t)row * nt;

  // The Q tile and its norm weights: issued first (wasted only for a tile
  // with no key). Task e = lane + 64 u: feature e / 4, queries q0 + 4 (e % 4) ..
  // + 3, features past hd read 0; weights of features 32 s + 8 grp .. + 7.
  const __amdgpu_buffer_rsrc_t rq = buffer_rsrc(Q, (uint32_t)((size_t)hd * L * 4));
  const __amdgpu_buffer_rsrc_t rn = buffer_rsrc(a.q_norm, (uint32_t)(hd * 4));
  f32x4 qx[HDP / 16], wv[HDP / 16];
#pragma unroll
  for (int u = 0; u < HDP / 16; ++u)
    qx[u] = buffer_load4(rq, ((lane >> 2) * L + 4 * (lane & 3)) * 4, u * 16 * L * 4 + q0 * 4);
#pragma unroll
  for (int c = 0; c < HDP / 16; ++c)
    wv[c] = buffer_load4(rn, (8 * grp + 4 * (c & 1)) * 4, 128 * (c / 2));

  const int first = spans[2 * row], last = spans[2 * row + 1];
  const int start = (a.trim && last >= 0) ? first : 0;
  const bool q_live = q < L && q >= start;
  // The workgroup's 32-key tiles: first active key .. last query.
  int t_begin = 0, t_end = 0;
  {
    const int q_hi = min(16 * (yg + 1) * tiles - 1, L - 1), kl = min(last, q_hi);
    if (last >= 0 && first <= kl && q_hi >= start) {
      t_begin = first / 32;
      t_end = kl / 32 + 1;
    }
  }
  t_begin = __builtin_amdgcn_readfirstlane(t_begin);
  t_end = __builtin_amdgcn_readfirstlane(t_end);

  f32x4 O[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) O[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m = kNoMax, l = 0.0f;  // l: this lane's share of the row sum
  bool tainted = false;        // wave-uniform
  if (t_begin < t_end) {
    bf16x8 qp[3][ST];
    const float c1 = a.c1;
    {
      // RMSNorm (lib.rs:676-691) and partial RoPE (692-709): the queries
      // transposed through the wave's LDS rows into the B operands' order,
      // lane (col, grp) holding features 32 s + 8 grp .. + 7 of query col.
      constexpr int QP = HDP + 4;
      const int rh = a.rot_half;
      const bool rope = a.cos_t != nullptr && rh > 0;
      const size_t pos = (size_t)min(max(q - start, 0), L - 1) * rh;
      f32x4 tc[2], ts[2];
      if (rope && rh == 32) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          tc[h] = *reinterpret_cast<const f32x4 *>(a.cos_t + pos + 8 * grp + 4 * h);
          ts[h] = *reinterpret_cast<const f32x4 *>(a.sin_t + pos + 8 * grp + 4 * h);
        }
      }
      auto settle = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      };
#pragma unroll
      for (int u = 0; u < HDP / 16; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          ws[(4 * (lane & 3) + i) * QP + (lane >> 2) + 16 * u] = qx[u][i];
      settle();
      float *const qr = ws + col * QP;
      float ss = 0.0f;
#pragma unroll
      for (int c = 0; c < 2 * ST; ++c) {
        qx[c] = *reinterpret_cast<const f32x4 *>(qr + 32 * (c / 2) + 8 * grp + 4 * (c & 1));
        ss += qx[c][0] * qx[c][0] + qx[c][1] * qx[c][1] + qx[c][2] * qx[c][2] + qx[c][3] * qx[c][3];
      }
      const float scale = rms_scale(pair_sum(pair16_sum(ss)), hd, a.eps);
#pragma unroll
      for (int c = 0; c < 2 * ST; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          qx[c][e] = q_live && 32 * (c / 2) + 8 * grp + 4 * (c & 1) + e < hd
                         ? rms_apply(qx[c][e], scale, wv[c][e])
                         : 0.0f;
      if (rope && rh == 32) {
        if (q_live) {  // pairs (i, i + 32): the same element of steps 0 and 1
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float x = qx[h][e], y = qx[2 + h][e];
              qx[h][e] = rope_lo(x, y, tc[h][e], ts[h][e]);
              qx[2 + h][e] = rope_hi(x, y, tc[h][e], ts[h][e]);
            }
        }
      } else if (rope) {
#pragma unroll
        for (int c = 0; c < 2 * ST; ++c)
          *reinterpret_cast<f32x4 *>(qr + 32 * (c / 2) + 8 * grp + 4 * (c & 1)) = qx[c];
        settle();
        if (q_live)
          for (int i = grp; i < rh; i += 4) {
            const float x = qr[i], y = qr[i + rh], cc = a.cos_t[pos + i], sn = a.sin_t[pos + i];
            qr[i] = rope_lo(x, y, cc, sn);
            qr[i + rh] = rope_hi(x, y, cc, sn);
          }
        settle();
#pragma unroll
        for (int c = 0; c < 2 * ST; ++c)
          qx[c] = *reinterpret_cast<const f32x4 *>(qr + 32 * (c / 2) + 8 * grp + 4 * (c & 1));
      }
#pragma unroll
      for (int x = 0; x < ST; ++x) {
        const Bf16x3 lo = split_bf16x3(qx[2 * x]), hi = split_bf16x3(qx[2 * x + 1]);
#pragma unroll
        for (int i = 0; i < 3; ++i) qp[i][x] = join_bf16(lo, hi, i);
      }
    }
    __syncthreads();  // the wave rows become the ring

    // Piece p of the walk (piece p % 4 of tile t_begin + p / 4) goes to ring slot
    // p % RING: this wave's share of its 1 KB loads.
    const int pieces = 4 * (t_end - t_begin);
    const unsigned char *const first_piece = unit + (size_t)t_begin * kJeffTileBytes;
    const uint32_t voff = 16 * lane + 1024 * PW * wave;
    int ahead = 0;                // the next piece to load
    unsigned char *fill = lds;    // its slot
    auto load_piece = [&] {
      const u32x4r r = rsrc_words(first_piece + (size_t)ahead * kJeffPieceBytes, kJeffPieceBytes);
#pragma unroll
      for (int i = 0; i < PW; ++i)
        load_lds16(r, voff, (uint32_t)(1024 * i), fill + 1024 * (PW * wave + i));
      ++ahead;
      fill = fill == lds + (RING - 1) * kJeffPieceBytes ? lds : fill + kJeffPieceBytes;
    };
    // The next piece has landed for every wave (one more may be in flight) and every
    // wave's reads of the piece before it are done, whose slot is refilled. Called
    // four times per tile by every wave.
    const unsigned char *at = lds + (RING - 1) * kJeffPieceBytes;  // the piece in use
    auto next_piece = [&](bool last) {
      if (last)
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PW) : "memory");
      // Said once more where the compiler sees it: with a scalar load possibly in
      // flight it would wait for every LDS read before the first product.
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (ahead < pieces) load_piece();
      at = at == lds + (RING - 1) * kJeffPieceBytes ? lds : at + kJeffPieceBytes;
    };
    load_piece();
    load_piece();  // a tile has four
    uint32_t word_next = rbits[t_begin];  // scalar loads, one tile ahead of their use
    for (int t = t_begin; t < t_end; ++t) {
      const uint32_t word = word_next;
      word_next = rbits[min(t + 1, nt - 1)];
      const uint32_t w = q_live ? (word & range_bits(0, q - 32 * t)) : 0u;
      const bool mine = !tainted && __ballot(w != 0u) != 0;
      // A 16-key half's scores: accumulators for h*h of even and odd steps and for
      // the smaller products, fewer roundings of the whole sum than one, and no
      // product right behind one into the same accumulator (it would wait for that
      // one's eight passes). Operands two steps ahead of their products (an LDS
      // read takes about as long as two steps' products when all waves read).
      auto scores = [&](f32x4 &s) {
        const unsigned char *const kl = at + 16 * lane;
        f32x4 u = s, r[3] = {s, s, s};
        bf16x8 kx[3][3];
        auto take = [&](int x) {
#pragma unroll
          for (int i = 0; i < 3; ++i)
            kx[x % 3][i] = *reinterpret_cast<const bf16x8 *>(kl + kJeffBlock * x + 1024 * i);
        };
        take(0);
        take(1);
#pragma unroll
        for (int x = 0; x < ST; ++x) {
          if (x + 2 < ST) take(x + 2);
          const bf16x8 (&k)[3] = kx[x % 3];
          f32x4 &a0 = r[2 * x % 3], &a1 = r[(2 * x + 1) % 3], &a2 = r[(2 * x + 2) % 3];
          a0 = mfma_16x16x32_bf16(k[2], qp[0][x], a0);
          a1 = mfma_16x16x32_bf16(k[1], qp[1][x], a1);
          if (x & 1)
            u = mfma_16x16x32_bf16(k[0], qp[0][x], u);
          else
            s = mfma_16x16x32_bf16(k[0], qp[0][x], s);
          a2 = mfma_16x16x32_bf16(k[0], qp[2][x], a2);
          a0 = mfma_16x16x32_bf16(k[1], qp[0][x], a0);
          a1 = mfma_16x16x32_bf16(k[0], qp[1][x], a1);
          __builtin_amdgcn_sched_barrier(0);
        }
        s += u + (r[0] + (r[1] + r[2]));
      };
      f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;
      next_piece(false);
      if (mine) scores(s0);
      next_piece(false);
      if (mine) scores(s1);
      next_piece(false);
      bool ok = mine;
      bf16x8 pp[3];
      if (mine) {
        if (__ballot(q_live && w != 0xffffffffu) != 0) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            s0[r] = ((w >> (4 * grp + r)) & 1u) ? s0[r] : -INFINITY;
            s1[r] = ((w >> (16 + 4 * grp + r)) & 1u) ? s1[r] : -INFINITY;
          }
        }
        f32x4 e0, e1;
        float rs = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          e0[r] = fast_exp2(__builtin_fmaf(s0[r], c1, -m));
          e1[r] = fast_exp2(__builtin_fmaf(s1[r], c1, -m));
          rs += e0[r] + e1[r];
        }
        if (__ballot(q_live && !(rs <= kLazyLimit)) != 0) {
          // Move the reference where the tile max exceeds it by more than the slack.
          const float mx = fmaxf(fmaxf(fmaxf(s0[0], s0[1]), fmaxf(s0[2], s0[3])),
                                 fmaxf(fmaxf(s1[0], s1[1]), fmaxf(s1[2], s1[3])));
          const float mxs = pair_max(pair16_max(mx)) * c1;
          const bool need = mxs > m + kRescaleSlack;
          const float mn = need ? mxs : m;
          rs = 0.0f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            e0[r] = fast_exp2(__builtin_fmaf(s0[r], c1, -mn));
            e1[r] = fast_exp2(__builtin_fmaf(s1[r], c1, -mn));
            rs += e0[r] + e1[r];
          }
          if (__ballot(q_live && !(__builtin_isfinite(rs) && reference_usable(mn))) != 0) {
            tainted = true;
            ok = false;
          } else {
            const float alpha = fast_exp2(m - mn);  // exactly 1 where the reference stays
#pragma unroll
            for (int j = 0; j < NB; ++j) O[j] *= alpha;
            l *= alpha;
            m = mn;
          }
        }
        if (ok) {
          l += rs;
          const Bf16x3 p0 = split_bf16x3(e0), p1 = split_bf16x3(e1);
#pragma unroll
          for (int i = 0; i < 3; ++i) pp[i] = join_bf16(p0, p1, i);
        }
      }
      // O^T of features 128 half ..: two 16-feature blocks per step, their
      // operands a step ahead; the products but h*h are summed by themselves.
      auto values = [&](auto hv) {
        constexpr int half = decltype(hv)::value;
        const unsigned char *const vl = at + 16 * lane;
        bf16x8 vx[2][6];
        auto take = [&](int g) {
#pragma unroll
          for (int i = 0; i < 6; ++i)
            vx[g & 1][i] = *reinterpret_cast<const bf16x8 *>(vl + kJeffBlock * (2 * g + i / 3) + 1024 * (i % 3));
        };
        take(0);
#pragma unroll
        for (int g = 0; g < NB / 4; ++g) {
          if (g + 1 < NB / 4) take(g + 1);
          const bf16x8 (&v)[6] = vx[g & 1];
          f32x4 &o0 = O[NB / 2 * half + 2 * g], &o1 = O[NB / 2 * half + 2 * g + 1];
          f32x4 r0 = {0.0f, 0.0f, 0.0f, 0.0f}, r1 = r0;
#pragma unroll
          for (int i = 2; i >= 0; --i)
#pragma unroll
            for (int j = 0; i + j < 3; ++j) {
              f32x4 &x0 = i + j ? r0 : o0, &x1 = i + j ? r1 : o1;
              x0 = mfma_16x16x32_bf16(v[i], pp[j], x0);
              x1 = mfma_16x16x32_bf16(v[3 + i], pp[j], x1);
            }
          o0 += r0;
          o1 += r1;
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (ok) values(std::integral_constant<int, 0>{});
      next_piece(t + 1 == t_end);
      if (ok) values(std::integral_constant<int, 1>{});
    }
    __syncthreads();  // the ring becomes wave rows again
  }
  if (q0 >= L) return;  // no barrier follows

  // -------- careful redo (rare), out of line: NaN / inf among this wave's
  // kept scores or values.
  bool bad = false;
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) bad |= !__builtin_isfinite(O[j][r]);
  if (tainted || __ballot(q_live && bad) != 0) {
    jeff_redo_wave<HDP, true, 1>(kernel_jeff_args(), nullptr, row, head, q0, 2 * t_begin, 2 * t_end,
                                 start, ws);
    return;
  }
  // -------- o / sum (0 when nothing was kept), sigmoid gate, store
  const float lt = pair_sum(pair16_sum(l));
  const float inv = lt > 0.0f ? fast_rcp(lt) : 0.0f;
  jeff_store<HDP, true>(a, Gt, OUT, q0, start, ws, O, inv);
}

// ------------------------------------------- f32 attention, fused, hd 256

constexpr int kJeffFusedWaves = 8;  // waves per fused workgroup (the key range's parts)
constexpr int kJeffHalfMaxL = 4096;  // longest row of the two-workgroup fused kernel

// One kernel for the whole op at hd 256 (no K prep): one workgroup = NW
// wavefronts = one (row, head, 16-query tile). The RMSNorm scales are
// folded into the scores: with q' = R_q(x_q (1 + w_q)) and, per key,
// k' = R_k(x_k (1 + w_k)) on the rotated features and x_k elsewhere,
//   s(q, k) = scale_q scale_k (q'' . k') / sqrt(hd),
// where q'' is q' times (1 + w_k) on the features past rot_dim (the same
// product as the reference's q^.k^ of lib.rs:676-716, up to rounding). So
// wave w prepares Q's features 64 w .. 64 w + 63 elementwise (its RoPE pairs
// stay inside slice 0) into LDS, where every wave reads its B operands, and
// scale_q waits in the exponent's factor; a key tile needs only its sum of
// squares, (1 + w_k) and RoPE on its first rot_dim features, all in the
// lanes that feed them to the matrix cores.
//
// Layout (lane = 16 grp + col): B operand Q^T and A operand K carry feature
// f = 64 s + 16 c + 4 grp + e at step (s, c, e) of the S^T chain, for query
// (K: key) col; S^T holds keys 4 grp + r of query col; O^T block J holds
// features 16 J + 4 grp + r. RoPE partners (i, i + rot/2) sit in one lane,
// rot/32 blocks of 16 apart (rot/2 = 16 or 32).
//
// The tile's key range (first active key .. last query) is cut into NW
// contiguous parts walked by the NW waves with no barrier; the partial
// states merge once through LDS. K arrives with 4-byte loads (a lane needs
// one key's features), V with 16-byte loads along tokens; both stream
// through a ring of four 16-register pieces, three ahead: K slices 1, 2, 3,
// then slice 0 (the rotated features, whose table entries load a tile
// ahead), then V groups 0 .. 3. (Eight slots, each piece a whole tile ahead,
// measured slower: 21.7 against 19.3 us per C4 row.)
template <int NW, int RB>  // RB: rotated blocks of 16 in the lower half (rot_dim / 32: 0, 1, 2)
__global__ __launch_bounds__(NW * 64, 8 / NW) void jeff_fused_f32_kernel(const JeffArgs a,
                                                                         int rows) {
  static_assert(RB >= 0 && RB <= 2, "rot_dim 0, 32 or 64");
  constexpr int HDP = 256, NB = 16, KT = 16;
  constexpr int BPW = NB / NW;  // O^T blocks each wave finishes
  static_assert(NW == 4 || NW == 8, "four Q-prep slices; 16 O^T blocks over the waves");
  constexpr int OMF = NW * NB * 64 * 4;  // partial O^T of every wave (the redo's rows too)
  // Q operands [slice][run c][lane] as f32x4 (feature 64 s + 16 c + 4 grp + e
  // of query col), 16 KB at the front of smem until the merge.
  __shared__ __attribute__((aligned(16))) float smem[OMF];
  __shared__ __attribute__((aligned(16))) float s_wkr[4 * 4 * 4];  // (1 + w_k), rotated blocks
  __shared__ float s_ssq[4 * 16];
  __shared__ float s_m[NW * 16], s_l[NW * 16];
  __shared__ int s_bad;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int L = a.L;
  const int L4 = 4 * L;

  // -------- work item: query tiles from the last one down; the heads of a
  // (row, kv head) on one XCD.
  const int qt = (int)gridDim.y - 1 - (int)blockIdx.y;
  int row, head;
  jeff_unit_of(a, rows, blockIdx.x, row, head);
  const int kvh = min((int)a.gdiv.div((uint32_t)head), a.kv_heads - 1);
  const int q0 = qt * 16, q = q0 + col;
  const uint32_t bytes = (uint32_t)((size_t)HDP * L * 4);
  const __amdgpu_buffer_rsrc_t rq = buffer_rsrc(
      static_cast<const float *>(a.q) + row * a.q_row + (size_t)head * HDP * L, bytes);
  const __amdgpu_buffer_rsrc_t rg = buffer_rsrc(
      static_cast<const float *>(a.gate) + row * a.q_row + (size_t)head * HDP * L, bytes);
  const __amdgpu_buffer_rsrc_t ro =
      buffer_rsrc(a.out + row * a.q_row + (size_t)head * HDP * L, bytes);
  const float *Kb = static_cast<const float *>(a.k) + row * a.kv_row + (size_t)kvh * a.kv_head;
  const __amdgpu_buffer_rsrc_t rk = buffer_rsrc(Kb, bytes);
  const __amdgpu_buffer_rsrc_t rv = buffer_rsrc(
      static_cast<const float *>(a.v) + row * a.kv_row + (size_t)kvh * a.kv_head, bytes);
  const __amdgpu_buffer_rsrc_t rm = buffer_rsrc(a.mask + (size_t)row * L, (uint32_t)L4);
  // Per-lane byte offsets: feature 4 grp (+ the step's 64s + 16c + e, a
  // scalar offset) of token col (+ the tile's first token, scalar). A lane
  // with nothing to load takes an offset past the buffer's end, which the
  // hardware range check reads as 0 (whether or not it adds the scalar part).
  const int ofs_t = (4 * grp * L + col) * 4;
  const int koob = (int)bytes;
  const int ofs_q = q < L ? ofs_t : koob;

  // -------- loads that need nothing: Q slice `wave` (waves 0 .. 3) in
  // B-operand order (feature 64 wave + 16 c + 4 grp + e), its norm weights.
  const bool prep = wave < 4;
  const int sw = wave & 3;
  float xq[16];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      xq[4 * c + e] = prep ? buffer_load1(rq, ofs_q, q0 * 4 + (64 * sw + 16 * c + e) * L4) : 0.0f;
  const __amdgpu_buffer_rsrc_t rwq = buffer_rsrc(a.q_norm, HDP * 4);
  const __amdgpu_buffer_rsrc_t rwk = buffer_rsrc(a.k_norm, HDP * 4);
  f32x4 wq[4], wk[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    wq[c] = buffer_load4(rwq, (64 * sw + 16 * c + 4 * grp) * 4, 0);
    wk[c] = buffer_load4(rwk, (64 * sw + 16 * c + 4 * grp) * 4, 0);
  }

  // -------- the row's active span (mask != 0), every wave on its own.
  int first, last;
  {
    int lo = 0x7fffffff, hi = -1;
    for (int k0 = 0; k0 < L; k0 += 256) {
      const f32x4 mv = buffer_load4(rm, (k0 + 4 * lane) * 4, 0);  // past L: 0
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (mv[t] != 0.0f) {
          lo = min(lo, k0 + 4 * lane + t);
          hi = max(hi, k0 + 4 * lane + t);
        }
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    first = __builtin_amdgcn_readfirstlane(hi >= 0 ? lo : 0);
    last = __builtin_amdgcn_readfirstlane(hi);
  }
  const int start = (a.trim && last >= 0) ? first : 0;
  const bool q_live = q < L && q >= start;
  const int q_last = min(q0 + 15, L - 1);
  int kt_begin = 0, kt_end = 0;
  {
    const int kl = min(last, q_last);
    if (last >= 0 && first <= kl && q_last >= start) {
      kt_begin = first / KT;
      kt_end = kl / KT + 1;
    }
  }
  // o * sigmoid(gate) (lib.rs:755-758) for the wave's features 16 (BPW wave
  // + j) + 4 grp + r of query col; 0 for a dropped query (q < start).
  auto finish = [&](const f32x4 (&o)[BPW]) {
    float g[4 * BPW];
#pragma unroll
    for (int j = 0; j < BPW; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        g[4 * j + r] = buffer_load1(rg, ofs_q, q0 * 4 + (16 * (BPW * wave + j) + r) * L4);
    if (q < L) {
#pragma unroll
      for (int j = 0; j < BPW; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = q < start ? 0.0f : o[j][r] * fast_sigmoid(g[4 * j + r]);
          buffer_store1_nt(x, ro, ofs_t, q0 * 4 + (16 * (BPW * wave + j) + r) * L4);
        }
    }
  };
  if (kt_begin >= kt_end) {  // no key at or before these queries: o = 0 (lib.rs:739-743)
    const f32x4 z[BPW] = {};
    finish(z);
    return;
  }

  // -------- Q: x (1 + w_q), RoPE, (1 + w_k) past rot_dim, into LDS; the sum
  // of squares over the four slices gives scale_q.
  constexpr int rb = RB, rh = 16 * RB;
  float ssq = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) ssq += xq[i] * xq[i];
  ssq += __shfl_xor(ssq, 16);
  ssq += __shfl_xor(ssq, 32);
  if (prep && grp == 0) s_ssq[sw * 16 + col] = ssq;
  float qs[16];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) qs[4 * c + e] = xq[4 * c + e] * (1.0f + wq[c][e]);
  if (rb > 0 && wave == 0) {  // slice 0 holds the rotated features
    const int pos = min(max(q - start, 0), L - 1);
#pragma unroll
    for (int b = 0; b < rb; ++b) {
      const f32x4 cs = *reinterpret_cast<const f32x4 *>(a.cos_t + (size_t)pos * rh + 16 * b + 4 * grp);
      const f32x4 sn = *reinterpret_cast<const f32x4 *>(a.sin_t + (size_t)pos * rh + 16 * b + 4 * grp);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = qs[4 * b + e], y = qs[4 * (b + rb) + e];
        qs[4 * b + e] = rope_lo(x, y, cs[e], sn[e]);
        qs[4 * (b + rb) + e] = rope_hi(x, y, cs[e], sn[e]);
      }
    }
  }
  f32x4 *QL = reinterpret_cast<f32x4 *>(smem);
  if (prep) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const bool rotated = wave == 0 && c < 2 * rb;
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = q_live ? qs[4 * c + e] * (rotated ? 1.0f : 1.0f + wk[c][e]) : 0.0f;
      QL[(sw * 4 + c) * 64 + lane] = y;
    }
  }
  if (wave == 0 && col == 0) {
#pragma unroll
    for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4 *>(s_wkr + (c * 4 + grp) * 4) = wk[c] + 1.0f;
  }
  __syncthreads();
  const float c1q =
      a.c1 * rms_scale(s_ssq[col] + s_ssq[16 + col] + s_ssq[32 + col] + s_ssq[48 + col], HDP, a.eps);

  // -------- this wave's part of the key range.
  const int T = kt_end - kt_begin;
  const int w_begin = kt_begin + (T * wave) / NW, w_end = kt_begin + (T * (wave + 1)) / NW;
  // Ring slot i % 4: piece i of a tile, i = 0, 1, 2: K slice i + 1; 3: K
  // slice 0; 4 .. 7: V group i - 4 (O^T blocks 4 (i - 4) .. + 3). Loads are
  // unconditional (at the last tile the "next" K pieces re-read the current
  // tile), so no ring slot ever holds one of two values.
  f32x4 ring[4][4];
  f32x4 tcs[2], tsn[2];  // the tile's table entries (rotated pairs of key col)
  auto k_off = [&](int kt) -> int { return kt * KT + col < L ? ofs_t : koob; };
  auto load_k = [&](int slot, int sl, int kt) {
    const int vo = k_off(kt);
    kt = __builtin_amdgcn_readfirstlane(kt);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        ring[slot][c][e] = buffer_load1(rk, vo, kt * KT * 4 + (64 * sl + 16 * c + e) * L4);
  };
  auto load_tab = [&](int kt) {
    if (rb > 0) {
      const int pos = min(max(kt * KT + col - start, 0), L - 1);
#pragma unroll
      for (int b = 0; b < rb; ++b) {
        tcs[b] = *reinterpret_cast<const f32x4 *>(a.cos_t + (size_t)pos * rh + 16 * b + 4 * grp);
        tsn[b] = *reinterpret_cast<const f32x4 *>(a.sin_t + (size_t)pos * rh + 16 * b + 4 * grp);
      }
    }
  };
  // V: features 16 J + col, keys k0 + 4 grp .. + 3 (L % 4 == 0: all in or out).
  const int ofs_v = (col * L + 4 * grp) * 4;
  auto load_v = [&](int slot, int g, int kt) {
    const int k = kt * KT + 4 * grp;
    const int vo = k < L ? ofs_v + kt * KT * 4 : koob;
#pragma unroll
    for (int j = 0; j < 4; ++j) ring[slot][j] = buffer_load4(rv, vo, (4 * g + j) * 16 * L4);
  };

  f32x4 O[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) O[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m = kNoMax, l = 0.0f;  // l: this lane's share of the row sum
  bool tainted = false;        // wave-uniform

  if (w_begin < w_end) {
    load_tab(w_begin);
    load_k(0, 1, w_begin);
    load_k(1, 2, w_begin);
    load_k(2, 3, w_begin);
  }
  for (int kt = w_begin; kt < w_end; ++kt) {
    const int kn = kt + 1 < w_end ? kt + 1 : kt;
    const int k0 = kt * KT;
    const float mv = buffer_load1(rm, (k0 + col) * 4, 0);  // past L: 0
    f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = {0.0f, 0.0f, 0.0f, 0.0f};
    float ssk = 0.0f;
    // S^T over K slices 1, 2, 3 (features past the rotated ones)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (i == 0)
        load_k(3, 0, kt);
      else
        load_v(i - 1, i - 1, kt);  // V groups 0, 1
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = ring[i][c][e];
          ssk += x * x;
          const float y = QL[((i + 1) * 4 + c) * 64 + lane][e];
          if (c & 1)
            s1 = mfma_16x16x4(x, y, s1);
          else
            s0 = mfma_16x16x4(x, y, s0);
        }
    }
    // slice 0: sum of squares of the raw key, then x (1 + w_k) and RoPE on
    // the rotated blocks (0 .. 2 rb - 1)
    load_v(2, 2, kt);  // V group 2
    {
      f32x4(&k)[4] = ring[3];
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) ssk += k[c][e] * k[c][e];
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < 2 * rb) k[c] *= *reinterpret_cast<const f32x4 *>(s_wkr + (c * 4 + grp) * 4);
#pragma unroll
      for (int b = 0; b < rb; ++b) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = k[b][e], y = k[b + rb][e];
          k[b][e] = rope_lo(x, y, tcs[b][e], tsn[b][e]);
          k[b + rb][e] = rope_hi(x, y, tcs[b][e], tsn[b][e]);
        }
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = QL[c * 64 + lane][e];
          if (c & 1)
            s1 = mfma_16x16x4(k[c][e], y, s1);
          else
            s0 = mfma_16x16x4(k[c][e], y, s0);
        }
    }
    // the key's scale (lanes col hold key col), to the S^T rows 4 grp + r
    ssk += __shfl_xor(ssk, 16);
    ssk += __shfl_xor(ssk, 32);
    const float sck = rms_scale(ssk, HDP, a.eps);
    const uint32_t abits = (uint32_t)__ballot(mv != 0.0f && k0 + col >= start) & 0xffffu;
    const uint32_t w = q_live ? (abits & range_bits(0, q - k0)) : 0u;
    f32x4 s = s0 + s1;
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] *= c1q * __shfl(sck, 4 * grp + r);
    if (__ballot(q_live && w != 0xffffu) != 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = ((w >> (4 * grp + r)) & 1u) ? s[r] : -INFINITY;
    }
    load_tab(kn);  // the next tile's table entries
    f32x4 ex;
    float rs = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ex[r] = fast_exp2(s[r] - m);
      rs += ex[r];
    }
    if (__builtin_expect(__ballot(q_live && !(rs <= kLazyLimit)) != 0, 0)) {
      const float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      const float mxs = pair_max(pair16_max(mx));
      const float mn = mxs > m + kRescaleSlack ? mxs : m;
      rs = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ex[r] = fast_exp2(s[r] - mn);
        rs += ex[r];
      }
      if (__ballot(q_live && !(__builtin_isfinite(rs) && reference_usable(mn))) != 0) {
        tainted = true;
      } else {
        const float alpha = fast_exp2(m - mn);  // exactly 1 where the reference stays
#pragma unroll
        for (int j = 0; j < NB; ++j) O[j] *= alpha;
        l *= alpha;
        m = mn;
      }
    }
    l += rs;
    // P.V: V groups 0 .. 3 in slots 0, 1, 2 and (loaded now) 3; the next
    // tile's K slices 1 .. 3 into slots 0 .. 2 as they free up.
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (g == 0)
        load_v(3, 3, kt);
      else
        load_k(g - 1, g, kn);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          O[4 * g + j] = mfma_16x16x4(ring[g][j][r], ex[r], O[4 * g + j]);
    }
    if (tainted) break;  // wave-uniform; the whole tile is redone below
  }

  // -------- careful redo (rare): some wave's scores or O went non-finite;
  // one wave redoes the whole tile with the reference's exact semantics.
  if (tid == 0) s_bad = 0;
  __syncthreads();
  bool bad = tainted;
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) bad |= q_live && !__builtin_isfinite(O[j][r]);
  if (__ballot(bad) != 0 && lane == 0) s_bad = 1;
  __syncthreads();
  if (s_bad != 0) {
    if (wave == 0)
      jeff_redo_wave<HDP, true, 2>(kernel_jeff_args(), nullptr, row, head, q0, kt_begin, kt_end,
                                   start, smem);
    return;
  }

  // -------- merge: O = sum_w 2^(m_w - M) O_w / sum_w 2^(m_w - M) l_w; wave w
  // finishes O^T blocks BPW w .. BPW w + BPW - 1. Every
  // wave is past its walk (the barrier above), so OM may cover the Q rows.
  f32x4 *OM = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
  for (int j = 0; j < NB; ++j) OM[(wave * NB + j) * 64 + lane] = O[j];
  const float lt = pair_sum(pair16_sum(l));
  if (grp == 0) {
    s_m[wave * 16 + col] = m;
    s_l[wave * 16 + col] = lt;
  }
  __syncthreads();
  float M = s_m[col];
#pragma unroll
  for (int v = 1; v < NW; ++v) M = fmaxf(M, s_m[v * 16 + col]);
  float fac[NW], lsum = 0.0f;
#pragma unroll
  for (int v = 0; v < NW; ++v) {
    fac[v] = fast_exp2(s_m[v * 16 + col] - M);  // 0 for a wave without keys (m = kNoMax)
    lsum += fac[v] * s_l[v * 16 + col];
  }
  const float inv = lsum > 0.0f ? fast_rcp(lsum) : 0.0f;
  f32x4 Of[BPW];
#pragma unroll
  for (int j = 0; j < BPW; ++j) {
    Of[j] = OM[(BPW * wave + j) * 64 + lane] * fac[0];
#pragma unroll
    for (int v = 1; v < NW; ++v) Of[j] += OM[(v * NB + BPW * wave + j) * 64 + lane] * fac[v];
    Of[j] *= inv;
  }
  finish(Of);
}

// ------------------------------------ f32 attention, fused, hd 256, halves

// Grids that fill at most half the CUs (a per-row call is 128 work items):
// each (row, head, 16-query tile) item runs as two workgroups, blockIdx.z =
// h, that each compute the item's whole S^T (all 256 features) and its
// softmax, and P.V and the output for features 128 h .. 128 h + 127 only.
// The scores are computed twice, but the grid fills twice as many CUs, an
// item's longest walk on one CU carries 96 instead of 128 MFMAs per key
// tile, and the two workgroups exchange nothing: each writes its own
// features, and decides on its own whether its half needs the careful redo.
// The ring holds one whole tile (six 16-register pieces: K slices 1, 2, 3,
// 0 and V groups 2h, 2h + 1), and every piece is reloaded with the next
// tile's as soon as its MFMAs have read it, so each load has a whole tile
// of the wave's work to land. The eight waves take the key tiles in turn
// from the diagonal down (wave w: the w-th, (w + 8)-th, ... below it), so a
// wave's first tile is known from the query tile alone in rows without
// right padding, and its loads go out with Q's. Layouts, the folded RMSNorm
// scales, the walk's softmax and the merge are those of
// jeff_fused_f32_kernel.
template <int RB, bool TRIM>  // RB: rotated blocks of 16 in the lower half (rot_dim / 32: 0, 1, 2);
                               // TRIM: a.trim (positions count from the row's first active key)
__global__ __launch_bounds__(512, 1) void jeff_fused_half_f32_kernel(const JeffArgs a, int rows) {
  static_assert(RB >= 0 && RB <= 2, "rot_dim 0, 32 or 64");
  constexpr int NW = 8, HDP = 256, NBH = 8, KT = 16;  // NBH: O^T blocks of the half, one per wave
  constexpr int OMF = NW * NBH * 64 * 4;  // partial O^T of every wave (the redo's rows too)
  static_assert(OMF >= 16 * 64 * 4, "the Q operands fit in front of the merge rows");
  __shared__ __attribute__((aligned(16))) float smem[OMF];
  __shared__ __attribute__((aligned(16))) float s_wkr[4 * 4 * 4];  // (1 + w_k), rotated blocks
  __shared__ float s_ssq[4 * 16];
  __shared__ float s_m[NW * 16], s_l[NW * 16];
  __shared__ int s_bad;
  __shared__ uint8_t s_act[kJeffHalfMaxL];  // mask != 0 per key of the row (launcher: L <= this)

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int L = a.L;
  const int L4 = 4 * L;
  const int h = (int)blockIdx.z;  // feature half

  const int qt = (int)gridDim.y - 1 - (int)blockIdx.y;
  int row, head;
  jeff_unit_of(a, rows, blockIdx.x, row, head);
  const int kvh = min((int)a.gdiv.div((uint32_t)head), a.kv_heads - 1);
  const int q0 = qt * 16, q = q0 + col;
  const uint32_t bytes = (uint32_t)((size_t)HDP * L * 4);
  const __amdgpu_buffer_rsrc_t rq = buffer_rsrc(
      static_cast<const float *>(a.q) + row * a.q_row + (size_t)head * HDP * L, bytes);
  const __amdgpu_buffer_rsrc_t rg = buffer_rsrc(
      static_cast<const float *>(a.gate) + row * a.q_row + (size_t)head * HDP * L, bytes);
  const __amdgpu_buffer_rsrc_t ro =
      buffer_rsrc(a.out + row * a.q_row + (size_t)head * HDP * L, bytes);
  const float *Kb = static_cast<const float *>(a.k) + row * a.kv_row + (size_t)kvh * a.kv_head;
  const __amdgpu_buffer_rsrc_t rk = buffer_rsrc(Kb, bytes);
  const __amdgpu_buffer_rsrc_t rv = buffer_rsrc(
      static_cast<const float *>(a.v) + row * a.kv_row + (size_t)kvh * a.kv_head, bytes);
  const __amdgpu_buffer_rsrc_t rm = buffer_rsrc(a.mask + (size_t)row * L, (uint32_t)L4);
  // Per-lane byte offsets: feature 4 grp (+ the step's 64s + 16c + e, a
  // scalar offset) of token col (+ the tile's first token, scalar); past the
  // buffer's end (read as 0) for a lane with nothing to load.
  const int ofs_t = (4 * grp * L + col) * 4;
  const int koob = (int)bytes;
  const int ofs_q = q < L ? ofs_t : koob;

  // -------- Q slice `wave` (waves 0 .. 3) and its norm weights.
  const bool prep = wave < 4;
  const int sw = wave & 3;
  float xq[16];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      xq[4 * c + e] = buffer_load1(rq, ofs_q, q0 * 4 + (64 * sw + 16 * c + e) * L4);  // waves 4-7: unused
  const __amdgpu_buffer_rsrc_t rwq = buffer_rsrc(a.q_norm, HDP * 4);
  const __amdgpu_buffer_rsrc_t rwk = buffer_rsrc(a.k_norm, HDP * 4);
  f32x4 wq[4], wk[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    wq[c] = buffer_load4(rwq, (64 * sw + 16 * c + 4 * grp) * 4, 0);
    wk[c] = buffer_load4(rwk, (64 * sw + 16 * c + 4 * grp) * 4, 0);
  }

  // -------- the ring, the gate, and a first key tile on a guess. Wave w
  // walks key tiles kt_end - 1 - w, kt_end - 1 - w - NW, ... down to
  // kt_begin; the span (below) gives kt_end = qt + 1 whenever the row's last
  // active key is at or past the tile's last query (no right padding), so
  // the wave's first tile qt - w is loaded with Q, before the span is known,
  // and loaded again only if the guess was wrong.
  constexpr int rb = RB, rh = 16 * RB;
  f32x4 ring[6][4];
  f32x4 tcs[2], tsn[2];  // the tile's table entries (rotated pairs of key col)
  auto k_off = [&](int kt) -> int { return kt * KT + col < L ? ofs_t : koob; };
  auto load_k = [&](int slot, int sl, int kt) {
    const int vo = k_off(kt);
    kt = __builtin_amdgcn_readfirstlane(kt);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        ring[slot][c][e] = buffer_load1(rk, vo, kt * KT * 4 + (64 * sl + 16 * c + e) * L4);
  };
  // V: features 16 J + col, keys k0 + 4 grp .. + 3 (L % 4 == 0: all in or out).
  const int ofs_v = (col * L + 4 * grp) * 4;
  auto load_v = [&](int slot, int g, int kt) {
    const int k = kt * KT + 4 * grp;
    const int vo = k < L ? ofs_v + kt * KT * 4 : koob;
#pragma unroll
    for (int j = 0; j < 4; ++j) ring[slot][j] = buffer_load4(rv, vo, (4 * g + j) * 16 * L4);
  };
  auto load_tile = [&](int kt) {
    load_k(0, 1, kt);
    load_k(1, 2, kt);
    load_k(2, 3, kt);
    load_k(3, 0, kt);
    load_v(4, 2 * h, kt);
    load_v(5, 2 * h + 1, kt);
  };
  // o * sigmoid(gate) (lib.rs:755-758) for features 16 (8 h + wave) + 4 grp
  // + r of query col; 0 for a dropped query (q < start).
  const int fb = 16 * (NBH * h + wave);
  float gt[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) gt[r] = buffer_load1(rg, ofs_q, q0 * 4 + (fb + r) * L4);
  // Q's table entries: at position q, loaded with Q, when nothing is
  // trimmed; after the span (position q - start) when rows are trimmed.
  f32x4 qcs[2], qsn[2];
  auto load_qtab = [&](int pos) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      qcs[b] = *reinterpret_cast<const f32x4 *>(a.cos_t + (size_t)pos * rh + 16 * b + 4 * grp);
      qsn[b] = *reinterpret_cast<const f32x4 *>(a.sin_t + (size_t)pos * rh + 16 * b + 4 * grp);
    }
  };
  if constexpr (!TRIM) load_qtab(min(q, L - 1));
  // The mask's first 256 keys are loaded before the guessed tile, so that
  // waiting for them (loads complete in order) does not wait for the tile.
  const f32x4 mv0 = buffer_load4(rm, 4 * lane * 4, 0);  // past L: 0
  // Unconditional (tile 0 for a wave past the diagonal), so that the
  // compiler's waits after it count the same loads on every path.
  const int guess = max(qt - wave, 0);
  asm volatile("" ::: "memory");  // keeps the loads above ahead of the tile's
  load_tile(guess);

  // -------- the row's active span (mask != 0), every wave on its own; wave
  // 0 also keeps each key's flag in LDS for the walk (read after the Q-prep
  // barrier), so no load of the walk is waited for out of its order.
  int first, last;
  {
    int lo = 0x7fffffff, hi = -1;
    for (int k0 = 0; k0 < L; k0 += 256) {
      const f32x4 mv = k0 == 0 ? mv0 : buffer_load4(rm, (k0 + 4 * lane) * 4, 0);  // past L: 0
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (mv[t] != 0.0f) {
          lo = min(lo, k0 + 4 * lane + t);
          hi = max(hi, k0 + 4 * lane + t);
        }
        if (wave == 0 && k0 + 4 * lane + t < L) s_act[k0 + 4 * lane + t] = mv[t] != 0.0f;
      }
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    first = __builtin_amdgcn_readfirstlane(hi >= 0 ? lo : 0);
    last = __builtin_amdgcn_readfirstlane(hi);
  }
  const int start = (TRIM && last >= 0) ? first : 0;
  const bool q_live = q < L && q >= start;
  const int q_last = min(q0 + 15, L - 1);
  int kt_begin = 0, kt_end = 0;
  {
    const int kl = min(last, q_last);
    if (last >= 0 && first <= kl && q_last >= start) {
      kt_begin = first / KT;
      kt_end = kl / KT + 1;
    }
  }
  auto finish = [&](const f32x4 o) {
    if (q < L) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = q < start ? 0.0f : o[r] * fast_sigmoid(gt[r]);
        buffer_store1_nt(x, ro, ofs_t, q0 * 4 + (fb + r) * L4);
      }
    }
  };
  if (kt_begin >= kt_end) {  // no key at or before these queries: o = 0 (lib.rs:739-743)
    finish(f32x4{0.0f, 0.0f, 0.0f, 0.0f});
    return;
  }
  const int kt_first = kt_end - 1 - wave;  // this wave's first tile (none below kt_begin)
  auto load_tab = [&](int kt) {
    if (rb > 0) {
      const int pos = min(max(kt * KT + col - start, 0), L - 1);
#pragma unroll
      for (int b = 0; b < rb; ++b) {
        tcs[b] = *reinterpret_cast<const f32x4 *>(a.cos_t + (size_t)pos * rh + 16 * b + 4 * grp);
        tsn[b] = *reinterpret_cast<const f32x4 *>(a.sin_t + (size_t)pos * rh + 16 * b + 4 * grp);
      }
    }
  };
  if (kt_first >= kt_begin) {
    if (kt_first != guess) load_tile(kt_first);
    load_tab(kt_first);
  }

  // -------- Q: x (1 + w_q), RoPE, (1 + w_k) past rot_dim, into LDS; the sum
  // of squares over the four slices gives scale_q.
  float ssq = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) ssq += xq[i] * xq[i];
  ssq += __shfl_xor(ssq, 16);
  ssq += __shfl_xor(ssq, 32);
  if (prep && grp == 0) s_ssq[sw * 16 + col] = ssq;
  float qs[16];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) qs[4 * c + e] = xq[4 * c + e] * (1.0f + wq[c][e]);
  if constexpr (TRIM) load_qtab(min(max(q - start, 0), L - 1));
  if (rb > 0 && wave == 0) {  // slice 0 holds the rotated features
#pragma unroll
    for (int b = 0; b < rb; ++b) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = qs[4 * b + e], y = qs[4 * (b + rb) + e];
        qs[4 * b + e] = rope_lo(x, y, qcs[b][e], qsn[b][e]);
        qs[4 * (b + rb) + e] = rope_hi(x, y, qcs[b][e], qsn[b][e]);
      }
    }
  }
  f32x4 *QL = reinterpret_cast<f32x4 *>(smem);
  if (prep) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const bool rotated = wave == 0 && c < 2 * rb;
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = q_live ? qs[4 * c + e] * (rotated ? 1.0f : 1.0f + wk[c][e]) : 0.0f;
      QL[(sw * 4 + c) * 64 + lane] = y;
    }
  }
  if (wave == 0 && col == 0) {
#pragma unroll
    for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4 *>(s_wkr + (c * 4 + grp) * 4) = wk[c] + 1.0f;
  }
  __syncthreads();
  const float c1q =
      a.c1 * rms_scale(s_ssq[col] + s_ssq[16 + col] + s_ssq[32 + col] + s_ssq[48 + col], HDP, a.eps);

  f32x4 O[4 * 2];  // O^T blocks 8 h .. 8 h + 7 (groups 2h, 2h + 1)
#pragma unroll
  for (int j = 0; j < 8; ++j) O[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m = kNoMax, l = 0.0f;  // l: this lane's share of the row sum
  bool tainted = false;        // wave-uniform

  // Each piece is reloaded with the next tile's right after its MFMAs; at
  // the wave's last tile the "next" pieces re-read it (unconditional, so no
  // ring slot ever holds one of two values).
  for (int kt = kt_first; kt >= kt_begin; kt -= NW) {
    const int kn = kt - NW >= kt_begin ? kt - NW : kt;
    const int k0 = kt * KT;
    const bool act = k0 + col < L && s_act[k0 + col] != 0;
    f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = {0.0f, 0.0f, 0.0f, 0.0f};
    float ssk = 0.0f;
    // S^T over K slices 1, 2, 3 (features past the rotated ones)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = ring[i][c][e];
          ssk += x * x;
          const float y = QL[((i + 1) * 4 + c) * 64 + lane][e];
          if (c & 1)
            s1 = mfma_16x16x4(x, y, s1);
          else
            s0 = mfma_16x16x4(x, y, s0);
        }
      load_k(i, i + 1, kn);
    }
    // slice 0: sum of squares of the raw key, then x (1 + w_k) and RoPE on
    // the rotated blocks (0 .. 2 rb - 1)
    {
      f32x4(&k)[4] = ring[3];
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) ssk += k[c][e] * k[c][e];
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < 2 * rb) k[c] *= *reinterpret_cast<const f32x4 *>(s_wkr + (c * 4 + grp) * 4);
#pragma unroll
      for (int b = 0; b < rb; ++b) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = k[b][e], y = k[b + rb][e];
          k[b][e] = rope_lo(x, y, tcs[b][e], tsn[b][e]);
          k[b + rb][e] = rope_hi(x, y, tcs[b][e], tsn[b][e]);
        }
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = QL[c * 64 + lane][e];
          if (c & 1)
            s1 = mfma_16x16x4(k[c][e], y, s1);
          else
            s0 = mfma_16x16x4(k[c][e], y, s0);
        }
    }
    load_k(3, 0, kn);
    load_tab(kn);
    // the key's scale (lanes col hold key col), to the S^T rows 4 grp + r
    ssk += __shfl_xor(ssk, 16);
    ssk += __shfl_xor(ssk, 32);
    const float sck = rms_scale(ssk, HDP, a.eps);
    const uint32_t abits = (uint32_t)__ballot(act && k0 + col >= start) & 0xffffu;
    const uint32_t w = q_live ? (abits & range_bits(0, q - k0)) : 0u;
    f32x4 s = s0 + s1;
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] *= c1q * __shfl(sck, 4 * grp + r);
    if (__ballot(q_live && w != 0xffffu) != 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] = ((w >> (4 * grp + r)) & 1u) ? s[r] : -INFINITY;
    }
    f32x4 ex;
    float rs = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ex[r] = fast_exp2(s[r] - m);
      rs += ex[r];
    }
    if (__builtin_expect(__ballot(q_live && !(rs <= kLazyLimit)) != 0, 0)) {
      const float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      const float mxs = pair_max(pair16_max(mx));
      const float mn = mxs > m + kRescaleSlack ? mxs : m;
      rs = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ex[r] = fast_exp2(s[r] - mn);
        rs += ex[r];
      }
      if (__ballot(q_live && !(__builtin_isfinite(rs) && reference_usable(mn))) != 0) {
        tainted = true;
      } else {
        const float alpha = fast_exp2(m - mn);  // exactly 1 where the reference stays
#pragma unroll
        for (int j = 0; j < 8; ++j) O[j] *= alpha;
        l *= alpha;
        m = mn;
      }
    }
    l += rs;
    // P.V: the half's V groups in slots 4, 5, each reloaded after its MFMAs.
#pragma unroll
    for (int g = 0; g < 2; ++g) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          O[4 * g + j] = mfma_16x16x4(ring[4 + g][j][r], ex[r], O[4 * g + j]);
      load_v(4 + g, 2 * h + g, kn);
    }
    if (tainted) break;  // wave-uniform; the half is redone below
  }

  // -------- careful redo (rare): a wave's scores, or this half's O, went
  // non-finite; one wave redoes the tile with the reference's exact
  // semantics and stores this half's features.
  if (tid == 0) s_bad = 0;
  __syncthreads();
  bool bad = tainted;
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) bad |= q_live && !__builtin_isfinite(O[j][r]);
  if (__ballot(bad) != 0 && lane == 0) s_bad = 1;
  __syncthreads();
  if (s_bad != 0) {
    if (wave == 0)
      jeff_redo_wave<HDP, true, 2>(kernel_jeff_args(), nullptr, row, head, q0, kt_begin, kt_end,
                                   start, smem, 128 * h, 128 * h + 128);
    return;
  }

  // -------- merge: O = sum_w 2^(m_w - M) O_w / sum_w 2^(m_w - M) l_w; wave w
  // finishes O^T block 8 h + w. Every wave is past its walk (the barrier
  // above), so OM may cover the Q rows.
  f32x4 *OM = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
  for (int j = 0; j < NBH; ++j) OM[(wave * NBH + j) * 64 + lane] = O[j];
  const float lt = pair_sum(pair16_sum(l));
  if (grp == 0) {
    s_m[wave * 16 + col] = m;
    s_l[wave * 16 + col] = lt;
  }
  __syncthreads();
  float M = s_m[col];
#pragma unroll
  for (int v = 1; v < NW; ++v) M = fmaxf(M, s_m[v * 16 + col]);
  float fac[NW], lsum = 0.0f;
#pragma unroll
  for (int v = 0; v < NW; ++v) {
    fac[v] = fast_exp2(s_m[v * 16 + col] - M);  // 0 for a wave without keys (m = kNoMax)
    lsum += fac[v] * s_l[v * 16 + col];
  }
  const float inv = lsum > 0.0f ? fast_rcp(lsum) : 0.0f;
  f32x4 Of = OM[wave * 64 + lane] * fac[0];
#pragma unroll
  for (int v = 1; v < NW; ++v) Of += OM[(v * NBH + wave) * 64 + lane] * fac[v];
  Of *= inv;
  finish(Of);
}

// ---------------------------------------------------------- bf16 attention

// Tile data for one 32-key bf16 tile: finished K rows from the prep workspace
// and the V columns, all as 16-byte loads with clamped indices. LDS holds K
// as [key][d] and V as [d][key] (bf16).
template <int HDP, bool VEC>
struct JeffStageBf16 {
  static constexpr int KT = 32;
  static constexpr int KTASKS = KT * HDP / 8;  // 16-byte chunks of K
  static constexpr int VTASKS = HDP * KT / 8;  // 16-byte chunks of V
  static constexpr int KN = (KTASKS + 255) / 256;
  static constexpr int VN = (VTASKS + 255) / 256;
  u16x8 k[KN], v[VN];

  __device__ __forceinline__ void fetch(const uint16_t *kp_tile, const uint16_t *V, int L, int hd,
                                        int k0, int tid) {
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const int e = min(tid + 256 * i, KTASKS - 1);
      const int kk = min(e / (HDP / 8), L - 1 - k0);
      k[i] = reinterpret_cast<const u16x8 *>(kp_tile)[kk * (HDP / 8) + e % (HDP / 8)];
    }
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const int e = min(tid + 256 * i, VTASKS - 1);
      const int d = min(e / (KT / 8), hd - 1), g = e % (KT / 8);
      const uint16_t *src = V + (size_t)L * d;
      const int key = k0 + 8 * g;
      if (VEC) {
        v[i] = *reinterpret_cast<const u16x8 *>(src + min(key, L - 8));
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) v[i][t] = src[min(key + t, L - 1)];
      }
    }
  }

  __device__ __forceinline__ int commit(uint16_t *Ks, uint16_t *Vs, int tid, int k0, int L, int hd) {
    constexpr int KSB = HDP + 8, VSB = KT + 8;
    const u16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    int nonfinite = 0;
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const int e = tid + 256 * i;
      const int kk = e / (HDP / 8), c = e % (HDP / 8);
      if (e < KTASKS) *reinterpret_cast<u16x8 *>(&Ks[kk * KSB + 8 * c]) = k0 + kk < L ? k[i] : z;
    }
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const int e = tid + 256 * i;
      const int d = e / (KT / 8), g = e % (KT / 8);
      if (e >= VTASKS) continue;
      u16x8 x = v[i];
      const int key = k0 + 8 * g;
      if (VEC && key + 8 > L) {  // the clamped load was shifted back: realign
        const int sh = key - (L - 8);
        u16x8 y = z;
#pragma unroll
        for (int t = 0; t < 8; ++t)
          if (t + sh < 8) y[t] = x[t + sh];
        x = y;
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const bool live = d < hd && key + t < L;
        const bool fin = bf16_finite(x[t]);
        nonfinite |= live && !fin;
        x[t] = (live && fin) ? x[t] : (unsigned short)0;
      }
      *reinterpret_cast<u16x8 *>(&Vs[d * VSB + 8 * g]) = x;
    }
    return nonfinite;
  }
};

// LDS bytes of the bf16 kernel's workgroup (two K/V tiles or the Q scratch).
template <int HDP>
__host__ __device__ constexpr int jeff_bf16_smem_bytes() {
  constexpr int KT = 32, KSB = HDP + 8, VSB = KT + 8;
  constexpr int TILE_BYTES = 2 * (KT * KSB + HDP * VSB) * 2;
  constexpr int QSCR_BYTES = kWavesPerGroup * kJeffWaveQueries * (HDP + 1) * 4;
  return TILE_BYTES > QSCR_BYTES ? TILE_BYTES : QSCR_BYTES;
}

// Same arithmetic as jeff_attention_f32_kernel with q, k, v and gate in bf16:
// normalized/rotated q and k, scaled by powers of two (norm_weight_exp), are
// rounded to fp16 for S^T on v_mfma_f32_16x16x32_f16, and the probabilities
// to bf16 for P.V on v_mfma_f32_16x16x32_bf16 (V stays bf16); the row sum l
// adds the rounded probabilities; softmax, accumulation and output stay f32.
// A 32-key tile is two 16-key S^T blocks (lane group g holds keys 4g + r and
// 16 + 4g + r of its query), which together are exactly the B operand of one
// P.V MFMA per 16-row block of O^T.
// Whether jeff_bf16_wide_kernel flagged (non-finite values) a query tile of
// redo_qt queries that unit (bx, by, bz) of the bf16 grid covers, for any
// head of its group.
__device__ __forceinline__ bool jeff_bf16_unit_flagged(const JeffArgs &a, const int *redo,
                                                       int redo_qt, int bx, int by, int bz) {
  const int hg = a.heads_per_group, QT = kJeffWaveQueries * (kWavesPerGroup / hg);
  const int L = a.L, qa = bx * QT;
  const int nqt = (L + redo_qt - 1) / redo_qt;
  const int t_lo = qa / redo_qt, t_hi = (min(qa + QT, L) - 1) / redo_qt;
  int any = 0;
  for (int h = by * hg; h < by * hg + hg; ++h)
    for (int t = t_lo; t <= t_hi; ++t) any |= redo[((size_t)bz * a.heads + h) * nqt + t];
  return any != 0;
}

// One workgroup's unit (bx, by, bz) of the grid (query tile, head group,
// row); smem_raw: jeff_bf16_smem_bytes() of LDS, s_span: two ints.
template <int HDP, bool VEC>
__device__ __forceinline__ void jeff_bf16_unit(const JeffArgs &a, const uint16_t *__restrict__ kp,
                                               const int bx, const int by, const int bz,
                                               unsigned char *smem_raw, int *s_span) {
  constexpr int KT = 32;
  constexpr int QS8 = HDP / 32;  // bf16x8 B operands of Q per lane
  constexpr int NB = HDP / 16;   // 16-row blocks of O^T
  constexpr int KSB = HDP + 8, VSB = KT + 8;
  constexpr int KBUF = KT * KSB, VBUF = HDP * VSB;  // uint16 elements
  constexpr int QP = HDP + 1;
  uint16_t *const lds16 = reinterpret_cast<uint16_t *>(smem_raw);
  float *const qscr = reinterpret_cast<float *>(smem_raw);

  // The thread index goes through an opaque move: the exact pass runs units
  // in a loop, and what is derived from the index stays inside the unit
  // instead of being hoisted (and held live) across the whole loop.
  int tid;
  asm volatile("v_mov_b32 %0, %1" : "=v"(tid) : "v"((int)threadIdx.x));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform, in a scalar register
  const int col = lane & 15, grp = lane >> 4;
  const int hg = a.heads_per_group, qsubs = kWavesPerGroup / hg;
  const int row = bz;
  const int head = by * hg + wave % hg;
  const int kvh = min(head / a.groups, a.kv_heads - 1);
  const int L = a.L, hd = a.hd, rh = a.rot_half;
  const int QT = kJeffWaveQueries * qsubs;
  const int qa = bx * QT;
  const int q = qa + (wave / hg) * kJeffWaveQueries + col;
  const bool qin = q < L;
  const float *maskr = a.mask + (size_t)row * L;
  const uint16_t *Q = static_cast<const uint16_t *>(a.q) + row * a.q_row + (size_t)head * hd * L;
  const uint16_t *Gt = static_cast<const uint16_t *>(a.gate) + row * a.q_row + (size_t)head * hd * L;
  const uint16_t *V = static_cast<const uint16_t *>(a.v) + row * a.kv_row + (size_t)kvh * a.kv_head;
  const uint16_t *KP = kp + ((size_t)row * a.kv_heads + kvh) * L * HDP;
  float *OUT = a.out + row * a.q_row + (size_t)head * hd * L;
  const bool rope = a.cos_t != nullptr && rh > 0;

  if (tid == 0) {
    s_span[0] = 0x7fffffff;
    s_span[1] = -1;
  }
  __syncthreads();
  scan_active(maskr, L, tid, lane, s_span);
  __syncthreads();
  const int first = s_span[0], last = s_span[1];
  const int start = (a.trim && last >= 0) ? first : 0;
  int kt_begin = 0, kt_end = 0;
  {
    const int kl = min(last, min(qa + QT, L) - 1);
    if (last >= 0 && first <= kl) {
      kt_begin = first / KT;
      kt_end = kl / KT + 1;
    }
  }

  // -------- Q: RMSNorm + partial RoPE in f32 (wave-local LDS phases), then
  // scaled by 2^-e_q and rounded to fp16 (the prepared keys are fp16 with
  // 2^-e_k): lane (col, grp) holds Q[q][32*s + 8*grp + e] in qb[s].
  const int eq = norm_weight_exp(a.q_norm, hd, lane);
  const float qsig = ldexpf(1.0f, -eq);
  const float c1 = ldexpf(a.c1, eq + norm_weight_exp(a.k_norm, hd, lane));
  f16x8 qb[QS8];
  const bool q_live = qin && q >= start;
  {
    float *qw = qscr + wave * (kJeffWaveQueries * QP);
    float *qs = qw + col * QP;
    constexpr int QQ = HDP / 4;
    float ss = 0.0f;
    const int qc = q_live ? q : 0;
#pragma unroll
    for (int s = 0; s < QQ; ++s) {
      const int d = grp * QQ + s;
      const float x = bf16_to_f32(Q[qc + (size_t)L * (d < hd ? d : hd - 1)]);
      const float y = (q_live && d < hd) ? x : 0.0f;
      qs[d] = y;
      ss += y * y;
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    const float scale = rms_scale(ss, hd, a.eps);
#pragma unroll 16
    for (int s = 0; s < QQ; ++s) {
      const int d = grp * QQ + s;
      const float wq = a.q_norm[min(d, hd - 1)];
      const float y = rms_apply(qs[d], scale, wq);
      qs[d] = d < hd ? y : 0.0f;
    }
    if (rope) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int q0 = qa + (wave / hg) * kJeffWaveQueries;
      for (int e0 = 0; e0 < kJeffWaveQueries * rh; e0 += 64 * 8) {
        float c[8], sn[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int e = min(e0 + lane + 64 * u, kJeffWaveQueries * rh - 1);
          const int qi = e / rh, i = e - qi * rh;
          const int pos = min(max(q0 + qi - start, 0), L - 1);
          c[u] = a.cos_t[(size_t)pos * rh + i];
          sn[u] = a.sin_t[(size_t)pos * rh + i];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int e = e0 + lane + 64 * u;
          const int qi = e / rh, i = e - qi * rh;
          const int qq = q0 + qi;
          if (e < kJeffWaveQueries * rh && qq < L && qq >= start) {
            const float x = qw[qi * QP + i], y = qw[qi * QP + i + rh];
            qw[qi * QP + i] = rope_lo(x, y, c[u], sn[u]);
            qw[qi * QP + i + rh] = rope_hi(x, y, c[u], sn[u]);
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int s = 0; s < QS8; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) qb[s][e] = (_Float16)(qs[32 * s + 8 * grp + e] * qsig);
  }
  __syncthreads();  // the Q scratch becomes the K/V buffers

  auto mask_of = [&](int kt) -> float { return maskr[min(kt * KT + (lane & 31), L - 1)]; };
  auto keep_word = [&](int kt, float mv) -> uint32_t {
    const int k0 = kt * KT;
    const int kc = k0 + (lane & 31);
    const bool act = kc < L && kc >= start && mv != 0.0f;
    const uint32_t abits = (uint32_t)__ballot(act);  // lanes 0..31 = keys of the tile
    return q_live ? (abits & range_bits(0, q - k0)) : 0u;
  };

  f32x4 O[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) O[j][r] = 0.0f;
  float m = -INFINITY, l = 0.0f;

  JeffStageBf16<HDP, VEC> st;
  int nonfinite = 0;
  uint32_t w = 0u;
  float m_next = 0.0f;
  if (kt_begin < kt_end) {
    const float m0 = mask_of(kt_begin);
    st.fetch(KP + (size_t)kt_begin * KT * HDP, V, L, hd, kt_begin * KT, tid);
    nonfinite = st.commit(lds16, lds16 + 2 * KBUF, tid, kt_begin * KT, L, hd);
    w = keep_word(kt_begin, m0);
  }
  int nf = __syncthreads_or(nonfinite);
  int any_nf = 0;

  for (int kt = kt_begin; kt < kt_end; ++kt) {
    const int cur = (kt - kt_begin) & 1;
    const bool more = kt + 1 < kt_end;
    if (more) {
      m_next = mask_of(kt + 1);
      st.fetch(KP + (size_t)(kt + 1) * KT * HDP, V, L, hd, (kt + 1) * KT, tid);
    }
    const uint16_t *Kc = lds16 + cur * KBUF;
    const uint16_t *Vc = lds16 + 2 * KBUF + cur * VBUF;

    if (__ballot(w != 0u) != 0) {
      f32x4 s0, s1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s0[r] = 0.0f;
        s1[r] = 0.0f;
      }
      const uint16_t *k0row = Kc + col * KSB + 8 * grp;
      const uint16_t *k1row = Kc + (16 + col) * KSB + 8 * grp;
#pragma unroll
      for (int st8 = 0; st8 < QS8; ++st8) {
        const f16x8 ka = *reinterpret_cast<const f16x8 *>(k0row + 32 * st8);
        const f16x8 kb = *reinterpret_cast<const f16x8 *>(k1row + 32 * st8);
        s0 = mfma_16x16x32_f16(ka, qb[st8], s0);
        s1 = mfma_16x16x32_f16(kb, qb[st8], s1);
      }
      // The probabilities are summed as the bf16 values P.V consumes.
      const float alpha = softmax_tile16<true>(s0, s1, w, grp, c1, m, l);
      if (alpha != 1.0f) {
#pragma unroll
        for (int j = 0; j < NB; ++j) O[j] *= alpha;
      }
      bf16x8 pb;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pb[r] = (__bf16)s0[r];
        pb[4 + r] = (__bf16)s1[r];
      }
      // A operand of block j: V[keys 4g+0..3 and 16+4g+0..3][d = 16*j + col].
      const uint16_t *v0 = Vc + col * VSB + 4 * grp;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const u16x4 lo = *reinterpret_cast<const u16x4 *>(v0 + j * 16 * VSB);
        const u16x4 hi = *reinterpret_cast<const u16x4 *>(v0 + j * 16 * VSB + 16);
        u16x8 vv;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vv[e] = lo[e];
          vv[4 + e] = hi[e];
        }
        O[j] = mfma_16x16x32_bf16(__builtin_bit_cast(bf16x8, vv), pb, O[j]);
        if ((j & 7) == 7) __builtin_amdgcn_sched_barrier(0);
      }
    }
    any_nf |= nf;
    nonfinite = 0;
    if (more)
      nonfinite = st.commit(lds16 + (cur ^ 1) * KBUF, lds16 + 2 * KBUF + (cur ^ 1) * VBUF, tid,
                            (kt + 1) * KT, L, hd);
    nf = __syncthreads_or(nonfinite);
    if (more) w = keep_word(kt + 1, m_next);
  }

  // -------- non-finite values of kept keys (rare), as in the f32 kernel
  uint32_t special[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) special[j] = 0u;
  if (any_nf) {
    const int k_lo = kt_begin * KT, k_hi = min(kt_end * KT, L);
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = j * 16 + 4 * grp + r;
        uint32_t f = 0u;
        if (q_live && d < hd) {
#pragma nounroll
          for (int k = k_lo; k < k_hi && k <= q; ++k) {
            if (k < start || maskr[k] == 0.0f) continue;
            const float v = bf16_to_f32(V[k + (size_t)L * d]);
            if (!__builtin_isfinite(v)) f |= __builtin_isnan(v) ? 1u : (v > 0.0f ? 2u : 4u);
          }
        }
        special[j] |= f << (8 * r);
      }
  }

  float lt = l + __shfl_xor(l, 16);
  lt += __shfl_xor(lt, 32);
  const float inv = lt > 0.0f ? fast_rcp(lt) : 0.0f;
  if (qin) {
    const bool dropped = a.trim && q < start;
    f32x4 gv[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = j * 16 + 4 * grp + r;
        gv[j][r] = bf16_to_f32(Gt[q + (size_t)L * (d < hd ? d : hd - 1)]);
      }
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = j * 16 + 4 * grp + r;
        float o = O[j][r] * inv;
        const uint32_t f = (special[j] >> (8 * r)) & 7u;
        if (f) o = ((f & 1u) || f == 6u) ? __builtin_nanf("") : (f == 2u ? INFINITY : -INFINITY);
        if (d < hd)
          __builtin_nontemporal_store(dropped ? 0.0f : o * fast_sigmoid(gv[j][r]), &OUT[q + (size_t)L * d]);
      }
  }
}

template <int HDP, bool VEC>
__global__ __launch_bounds__(256, 2) void jeff_attention_bf16_kernel(const JeffArgs a,
                                                                     const uint16_t *__restrict__ kp) {
  __shared__ __attribute__((aligned(16))) unsigned char smem_raw[jeff_bf16_smem_bytes<HDP>()];
  __shared__ int s_span[2];
  jeff_bf16_unit<HDP, VEC>(a, kp, blockIdx.x, blockIdx.y, blockIdx.z, smem_raw, s_span);
}

// The exact pass after jeff_bf16_wide_kernel: the same units over a grid of
// gx x gy x gz, each run only where the wide kernel flagged one of its
// query tiles. A resident grid of workgroups walks the units (workgroup p
// takes p, p + gridDim.x, ...; the flags of up to 64 of them read in one
// round trip), so a call with nothing flagged costs one dispatch round of
// flag reads rather than a full grid of workgroups.
template <int HDP, bool VEC>
__global__ __launch_bounds__(256, 2) void jeff_bf16_exact_kernel(const JeffArgs a,
                                                                 const uint16_t *__restrict__ kp,
                                                                 const int *__restrict__ redo,
                                                                 int redo_qt, int gx, int gy,
                                                                 int gz) {
  __shared__ __attribute__((aligned(16))) unsigned char smem_raw[jeff_bf16_smem_bytes<HDP>()];
  __shared__ int s_span[2];
  const int n = gx * gy * gz, lane = threadIdx.x & 63, stride = gridDim.x;
  for (int v0 = blockIdx.x; v0 < n; v0 += 64 * stride) {
    // Lane k reads the flags of unit v0 + k*stride, all at once; every wave
    // gets the same ballot, so the loop below is uniform over the workgroup.
    const int v = v0 + lane * stride;
    const bool f = v < n && jeff_bf16_unit_flagged(a, redo, redo_qt, v % gx, (v / gx) % gy,
                                                   v / (gx * gy));
    uint64_t m = __ballot(f);
    while (m != 0) {
      const int u = v0 + (int)__builtin_ctzll(m) * stride;
      m &= m - 1;
      __syncthreads();  // the previous unit is done with the LDS
      jeff_bf16_unit<HDP, VEC>(a, kp, u % gx, (u / gx) % gy, u / (gx * gy), smem_raw, s_span);
    }
  }
}

// ----------------------------------------------------------------- launchers

// Workspace: the prepared keys (per row and kv head, keys rounded up to 16
// for whole 16-key blocks) or the split kernel's planes, then one (first, last)
// key span per row and the rows' active-key bits (32 keys per word).
static size_t jeff_kp_main_bytes(const JeffArgs &a, int rows, int hd_pad, bool bf16) {
  const size_t Lp = ((size_t)a.L + 15) & ~(size_t)15;
  const size_t b = (size_t)rows * a.kv_heads * Lp * hd_pad * (bf16 ? 2 : 4);
  return (b + 255) & ~(size_t)255;
}

// Which f32 kernel takes a call (also sizes its workspace).
enum class JeffF32Path { kHalf, kFused, kSplit, kGeneral };

// 16-byte accesses along tokens need L % 4 == 0 and aligned bases; buffer
// offsets need one head's (hd, L) block and one kv head's K rows within
// 2 GiB.
static bool jeff_f32_vec(const JeffArgs &a, int hd_pad) {
  const uintptr_t bases = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.v) |
                          reinterpret_cast<uintptr_t>(a.gate) | reinterpret_cast<uintptr_t>(a.out);
  return a.L % 4 == 0 && (bases & 15) == 0 && ((size_t)a.L + 15) * (size_t)hd_pad * 4 < ((size_t)1 << 31);
}

// Grids of at most two workgroups per CU (one row of C4 is 128) take
// the fused kernel: one launch, no K prep, every query tile's key range
// on eight wavefronts; of at most half the CUs (one C4 row per call) with each
// item as two workgroups, one per half of the output features. Larger grids
// take the prep and the split kernel, whose tiles are normalized and split once
// instead of for every query tile. It takes every length and alignment (its
// 16-byte accesses along tokens need dword alignment only); its buffer offsets
// need one head's (hd, L) block within 2 GiB.
static JeffF32Path jeff_f32_path(const JeffArgs &a, int rows, int hd_pad) {
  const bool div_ok = (uint64_t)rows * a.heads * a.heads <= ((uint64_t)1 << 32);
  if (hd_pad != 256 || !div_ok) return JeffF32Path::kGeneral;
  const int rb = a.cos_t == nullptr ? 0 : (a.rot_half % 16 == 0 ? a.rot_half / 16 : -1);
  const long items = (long)((a.L + kJeffWaveQueries - 1) / kJeffWaveQueries) * rows * a.heads;
  const long cus = a.cus > 0 ? a.cus : 1;
  if (jeff_f32_vec(a, hd_pad) && a.hd == 256 && rb >= 0 && rb <= 2) {
    if (a.L <= kJeffHalfMaxL && 2 * items <= cus) return JeffF32Path::kHalf;
    if (items <= 2 * cus) return JeffF32Path::kFused;
  }
  return ((size_t)a.L + 15) * (size_t)hd_pad * 4 < ((size_t)1 << 31) && a.kv_heads <= 32767
             ? JeffF32Path::kSplit
             : JeffF32Path::kGeneral;
}

template <int HDP>
static hipError_t launch_jeff_f32_hd(const JeffArgs &a, int rows, float *kp, hipStream_t stream,
                                     const KernelEvents &ev) {
  dim3 pgrid((a.L + kKeyTile - 1) / kKeyTile, a.kv_heads, rows);
  // Query tiles of 16 in causal pairs, kJeffF32Waves / heads_per_group tiles
  // (half as many pairs) per workgroup.
  const int nq = (a.L + kJeffWaveQueries - 1) / kJeffWaveQueries;
  const int pairs_per_group = kJeffF32Waves / a.heads_per_group / 2;
  const int npairs = (nq + 1) / 2;
  dim3 grid((npairs + pairs_per_group - 1) / pairs_per_group, a.heads / a.heads_per_group, rows);
  if constexpr (HDP == 256) {
    const JeffF32Path path = jeff_f32_path(a, rows, HDP);
    const int rb = a.cos_t == nullptr ? 0 : a.rot_half / 16;
    if (path == JeffF32Path::kHalf) {
      const dim3 hgrid((unsigned)(rows * a.heads), (unsigned)nq, 2u);
      void (*const kern[3][2])(JeffArgs, int) = {
          {jeff_fused_half_f32_kernel<0, false>, jeff_fused_half_f32_kernel<0, true>},
          {jeff_fused_half_f32_kernel<1, false>, jeff_fused_half_f32_kernel<1, true>},
          {jeff_fused_half_f32_kernel<2, false>, jeff_fused_half_f32_kernel<2, true>}};
      hipExtLaunchKernelGGL(kern[rb][a.trim ? 1 : 0], hgrid, dim3(512), 0, stream, ev.start,
                            ev.stop, 0, a, rows);
      return hipGetLastError();
    }
    if (path == JeffF32Path::kFused) {
      constexpr int NW = kJeffFusedWaves;
      const dim3 fgrid((unsigned)(rows * a.heads), (unsigned)nq);
      if (rb == 0)
        hipExtLaunchKernelGGL((jeff_fused_f32_kernel<NW, 0>), fgrid, dim3(NW * 64), 0, stream,
                              ev.start, ev.stop, 0, a, rows);
      else if (rb == 1)
        hipExtLaunchKernelGGL((jeff_fused_f32_kernel<NW, 1>), fgrid, dim3(NW * 64), 0, stream,
                              ev.start, ev.stop, 0, a, rows);
      else
        hipExtLaunchKernelGGL((jeff_fused_f32_kernel<NW, 2>), fgrid, dim3(NW * 64), 0, stream,
                              ev.start, ev.stop, 0, a, rows);
      return hipGetLastError();
    }
    if (path == JeffF32Path::kSplit) {
      const int nt = (a.L + 31) / 32;
      const size_t tiles = (size_t)rows * a.kv_heads * nt;
      unsigned char *planes = reinterpret_cast<unsigned char *>(kp);
      int *spans = reinterpret_cast<int *>(planes + tiles * kJeffTileBytes);
      uint32_t *kbits = reinterpret_cast<uint32_t *>(spans + 2 * rows);
      hipExtLaunchKernelGGL(jeff_k_prep_split_kernel, dim3(nt, 2 * a.kv_heads, rows), dim3(256), 0,
                            stream, ev.start, nullptr, 0, a, planes, spans, kbits);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      const unsigned units = (unsigned)(rows * a.kv_heads * (a.groups / a.heads_per_group));
      const unsigned n4 = (unsigned)((nq * a.heads_per_group + 3) / 4);
      hipExtLaunchKernelGGL((jeff_split_f32_kernel<HDP>), dim3(units, n4), dim3(256), 0, stream,
                            nullptr, ev.stop, 0, a, planes, spans, kbits, rows);
      return hipGetLastError();
    }
  }
  hipExtLaunchKernelGGL((jeff_k_prep_kernel<HDP, float>), pgrid, dim3(256), 0, stream, ev.start,
                        nullptr, 0, a, kp, nullptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const dim3 block(kJeffF32Waves * 64);
  if (jeff_f32_vec(a, HDP))
    hipExtLaunchKernelGGL((jeff_attention_f32_kernel<HDP, true>), grid, block, 0, stream, nullptr,
                          ev.stop, 0, a, kp);
  else
    hipExtLaunchKernelGGL((jeff_attention_f32_kernel<HDP, false>), grid, block, 0, stream, nullptr,
                          ev.stop, 0, a, kp);
  return hipGetLastError();
}

hipError_t launch_jeff_attention_f32(const JeffArgs &a, int rows, int hd_pad, void *kp,
                                     hipStream_t stream, const KernelEvents &ev) {
  float *k = static_cast<float *>(kp);
  switch (hd_pad) {
    case 32: return launch_jeff_f32_hd<32>(a, rows, k, stream, ev);
    case 64: return launch_jeff_f32_hd<64>(a, rows, k, stream, ev);
    case 128: return launch_jeff_f32_hd<128>(a, rows, k, stream, ev);
    case 256: return launch_jeff_f32_hd<256>(a, rows, k, stream, ev);
    default: return hipErrorInvalidValue;
  }
}

// bf16 at head dim 256: the flags of jeff_bf16_wide_kernel follow.
size_t jeff_bf16_flags_offset(const JeffArgs &a, int rows) {
  const size_t b = jeff_kp_main_bytes(a, rows, 256, true) + (size_t)rows * 2 * sizeof(int) +
                   (size_t)rows * ((a.L + 31) / 32) * sizeof(uint32_t);
  return (b + 255) & ~(size_t)255;
}

size_t jeff_kp_bytes(const JeffArgs &a, int rows, int hd_pad, bool bf16) {
  if (bf16 && hd_pad == 256 && jeff_bf16_wide_fits(a))
    return jeff_bf16_flags_offset(a, rows) + jeff_bf16_wide_flag_count(a, rows) * sizeof(int);
  const size_t nt = ((size_t)a.L + 31) / 32;
  const size_t keys = !bf16 && jeff_f32_path(a, rows, hd_pad) == JeffF32Path::kSplit
                          ? (size_t)rows * a.kv_heads * nt * kJeffTileBytes
                          : jeff_kp_main_bytes(a, rows, hd_pad, bf16);
  return keys + (size_t)rows * 2 * sizeof(int) +
         (size_t)rows * nt * sizeof(uint32_t);
}

template <int HDP>
static hipError_t launch_jeff_bf16_hd(const JeffArgs &a, int rows, uint16_t *kp,
                                      hipStream_t stream, const KernelEvents &ev) {
  dim3 pgrid((a.L + kKeyTile - 1) / kKeyTile, a.kv_heads, rows);
  // The wide bf16 kernel takes the rows' active key bits from the prep.
  const bool wide = HDP == 256 && jeff_bf16_wide_fits(a);
  uint32_t *kbits =
      wide ? reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(kp) +
                                          jeff_kp_main_bytes(a, rows, HDP, true) +
                                          (size_t)rows * 2 * sizeof(int))
           : nullptr;
  hipExtLaunchKernelGGL((jeff_k_prep_kernel<HDP, uint16_t>), pgrid, dim3(256), 0, stream, ev.start,
                        nullptr, 0, a, kp, kbits);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int qsubs = kWavesPerGroup / a.heads_per_group;
  const int qt = kJeffWaveQueries * qsubs;
  dim3 grid((a.L + qt - 1) / qt, a.heads / a.heads_per_group, rows);
  // 16-byte V loads along tokens need L % 8 == 0 and an aligned base.
  const bool vec = a.L % 8 == 0 && (reinterpret_cast<uintptr_t>(a.v) & 15) == 0;
  if constexpr (HDP == 256) {
    // The 32x32x16 kernel, then the exact pass over the query tiles it
    // flagged (non-finite values) on a resident grid (two workgroups per CU).
    if (jeff_bf16_wide_fits(a)) {
      int *flags = reinterpret_cast<int *>(reinterpret_cast<char *>(kp) + jeff_bf16_flags_offset(a, rows));
      e = launch_jeff_bf16_wide(a, rows, kp, kbits, flags, stream);
      if (e != hipSuccess) return e;
      const int redo_qt = jeff_bf16_wide_query_tile(a);
      const long units = (long)grid.x * grid.y * grid.z;
      const long slots = 2L * (a.cus > 0 ? a.cus : 1);
      const dim3 egrid((unsigned)(units < slots ? units : slots));
      if (vec)
        hipExtLaunchKernelGGL((jeff_bf16_exact_kernel<HDP, true>), egrid, dim3(256), 0, stream,
                              nullptr, ev.stop, 0, a, kp, flags, redo_qt, (int)grid.x,
                              (int)grid.y, (int)grid.z);
      else
        hipExtLaunchKernelGGL((jeff_bf16_exact_kernel<HDP, false>), egrid, dim3(256), 0, stream,
                              nullptr, ev.stop, 0, a, kp, flags, redo_qt, (int)grid.x,
                              (int)grid.y, (int)grid.z);
      return hipGetLastError();
    }
  }
  if (vec)
    hipExtLaunchKernelGGL((jeff_attention_bf16_kernel<HDP, true>), grid, dim3(256), 0, stream,
                          nullptr, ev.stop, 0, a, kp);
  else
    hipExtLaunchKernelGGL((jeff_attention_bf16_kernel<HDP, false>), grid, dim3(256), 0, stream,
                          nullptr, ev.stop, 0, a, kp);
  return hipGetLastError();
}

hipError_t launch_jeff_attention_bf16(const JeffArgs &a, int rows, int hd_pad, void *kp,
                                      hipStream_t stream, const KernelEvents &ev) {
  uint16_t *k = static_cast<uint16_t *>(kp);
  switch (hd_pad) {
    case 32: return launch_jeff_bf16_hd<32>(a, rows, k, stream, ev);
    case 64: return launch_jeff_bf16_hd<64>(a, rows, k, stream, ev);
    case 128: return launch_jeff_bf16_hd<128>(a, rows, k, stream, ev);
    case 256: return launch_jeff_bf16_hd<256>(a, rows, k, stream, ev);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tfd

