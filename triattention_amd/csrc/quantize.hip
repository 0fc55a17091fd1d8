// Rotate + quantize kernels for gfx950: Q per-token INT8/INT4 codes, per-channel
// K/V statistics, centred+rotated K records with per-(tile, 16-key group) scales,
// and the normalised V records.  All arithmetic is IEEE fp32 with the
// reference's operation order, so codes and scales are bit-exact.
//
// Reference semantics: triattention/kernels/cuda/common_device.cuh:1-172.
#include "common.h"

namespace tri {

// n / d for n < 2^31 by a multiplication (a division of workgroup indexes costs a vector reciprocal and a dozen
// dependent instructions before a workgroup's first load).
struct Divisor {
  uint32_t d, m, s;
  __device__ __forceinline__ int quotient(int n) const { return (int)((__umulhi(m, (uint32_t)n) + (uint32_t)n) >> s); }
};
inline Divisor divisor(int64_t d) {
  uint32_t s = 0;
  while (((int64_t)1 << s) < d) ++s;
  return Divisor{(uint32_t)d, (uint32_t)(((uint64_t)(((uint64_t)1 << s) - d) << 32) / d + 1), s};
}

// Arguments of one prepare call.  Parts that a call leaves out have a null source: q (the Q codes), k (K
// statistics and records), v (V records; its statistics too unless v_identity), exact (KX / VX records).
struct PrepareArgs {
  const uint16_t *q, *k, *v;  // bf16 [B][H][T][128], strides in elements
  int64_t qsb, qsh, qst, ksb, ksh, kst, vsb, vsh, vst;
  int batch, hq, hk, t;
  int8_t* q8;
  float* qa;
  uint8_t* q4;  // (q4, qa4, k4, ka4 null together)
  float* qa4;
  uint8_t* k8;
  float* ka;
  uint8_t* k4;
  float* ka4;
  uint8_t* k4x;  // may be null
  float *kpart, *vpart;  // [B][Hk][64][3][128] block partials
  float *kstat, *vstat;  // [B][Hk][3][128] mean, scale, 1 / scale
  int v_identity;        // V' = V: no V8 or V4 records, statistics (0, 1, 1)
  uint8_t *v16, *v8, *v4;  // may be null
  int32_t* v8s;            // may be null
  const int32_t* exact;    // [hq]: 1 + record slot of the q-head's KV head, 0 if quantized
  int nx;
  uint8_t *kx, *vx;
  // workgroups per part, and the launch's first workgroup (set by the host)
  int kstat_wgs, vstat_wgs, krec_wgs, vrec_wgs, wg0;
  Divisor qblocks, qheads, kvheads, ktiles;  // 32-row blocks of Q, q-heads, KV heads, tiles
  int finalized;  // the statistics are complete (prepare_finalize_kernel): record workgroups read them
};

// Q codes: one 128-feature row per 8 lanes (16 features per lane, rotated with DPP lane moves by
// rotate128_x16), 32 rows per 256-thread workgroup.  common_device.cuh:1-28 (quantize_q_kernel).
__device__ __forceinline__ void quantize_q_rows(const PrepareArgs& a, int wg) {
  const int hw = a.qblocks.quotient(wg), b = a.qheads.quotient(hw), h = hw - b * a.hq;
  const int sub = threadIdx.x & 7, row = (wg - hw * (int)a.qblocks.d) * 32 + (threadIdx.x >> 3);
  if (row >= a.t) return;  // whole 8-lane groups leave together
  const uint16_t* src = a.q + b * a.qsb + h * a.qsh + (int64_t)row * a.qst + sub * 16;
  float x[16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint2 raw = *reinterpret_cast<const uint2*>(src + 4 * i);
    x[4 * i] = bf16f(raw.x & 0xffffu);
    x[4 * i + 1] = bf16f(raw.x >> 16);
    x[4 * i + 2] = bf16f(raw.y & 0xffffu);
    x[4 * i + 3] = bf16f(raw.y >> 16);
  }
  rotate128_x16(x, sub);
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) m = fmaxf(m, fabsf(x[i]));
  m = lanes8_max(m);
  const int64_t r = ((int64_t)b * a.hq + h) * a.t + row;
  const float inv = m > 0.f ? 127.f / m : 0.f;
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    w[k] = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[k] |= ((uint32_t)(int)__builtin_rintf(x[4 * k + i] * inv) & 0xffu) << (8 * i);
  }
  *reinterpret_cast<uint4*>(a.q8 + r * D + sub * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  if (sub == 0) a.qa[r] = m / 127.f;
  if (a.q4 != nullptr) {
    const float inv4 = m > 0.f ? 7.f / m : 0.f;
    uint32_t nib[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 16; ++i) nib[i >> 3] |= ((uint32_t)(int)__builtin_rintf(x[i] * inv4) & 0xfu) << (4 * (i & 7));
    uint32_t* dst = reinterpret_cast<uint32_t*>(a.q4 + r * (D / 2) + sub * 8);
    dst[0] = nib[0];
    dst[1] = nib[1];
    if (sub == 0) a.qa4[r] = m / 7.f;
  }
}

// Per channel: sequential sum/max/min over tokens t = blk, blk+64, ...
// common_device.cuh:32-42 (partial_kernel).  One wave per (blk, head): lane i takes channels 2i and
// 2i + 1 (one 4-byte load per token; rows are 8-byte aligned).  Each channel's sum is formed in the
// reference's token order, so the chain is serial; the loads are not: the next STAT_DEPTH tokens load
// while the current ones are added.
constexpr int STAT_DEPTH = 16;
__device__ __forceinline__ void stat_block(const uint16_t* __restrict__ src, int64_t st, int t, int blk,
                                           float* __restrict__ partial) {
  const int c = 2 * (threadIdx.x & 63);
  float sum0 = 0.f, sum1 = 0.f, hi0 = -3.402823466e38f, hi1 = hi0, lo0 = 3.402823466e38f, lo1 = lo0;
  uint32_t cur[STAT_DEPTH], nxt[STAT_DEPTH];
  auto load = [&](uint32_t (&w)[STAT_DEPTH], int tk) {
#pragma unroll
    for (int j = 0; j < STAT_DEPTH; ++j)
      if (tk + j * STAT_BLOCKS < t)
        w[j] = *reinterpret_cast<const uint32_t*>(src + (int64_t)(tk + j * STAT_BLOCKS) * st + c);
  };
  auto add = [&](const uint32_t (&w)[STAT_DEPTH], int tk) {
#pragma unroll
    for (int j = 0; j < STAT_DEPTH; ++j)
      if (tk + j * STAT_BLOCKS < t) {
        const float v0 = bf16f((uint16_t)(w[j] & 0xffffu)), v1 = bf16f((uint16_t)(w[j] >> 16));
        sum0 += v0;
        sum1 += v1;
        hi0 = fmaxf(hi0, v0);
        hi1 = fmaxf(hi1, v1);
        lo0 = fminf(lo0, v0);
        lo1 = fminf(lo1, v1);
      }
  };
  constexpr int STEP = STAT_DEPTH * STAT_BLOCKS;
  load(cur, blk);
  for (int tk = blk; tk < t; tk += 2 * STEP) {
    load(nxt, tk + STEP);
    add(cur, tk);
    load(cur, tk + 2 * STEP);
    add(nxt, tk + STEP);
  }
  float* o = partial + (int64_t)blk * 3 * D + c;
  *reinterpret_cast<float2*>(o) = make_float2(sum0, sum1);
  *reinterpret_cast<float2*>(o + D) = make_float2(hi0, hi1);
  *reinterpret_cast<float2*>(o + 2 * D) = make_float2(lo0, lo1);
}

// First launch of a prepare call: the K and V statistics' block partials and the Q codes, which depend on
// nothing but the inputs.  The statistics are latency-bound (64 serial sums per head and channel pair, one
// wave each) and come first in the grid; the Q codes are HBM-bound and fill the rest of the chip meanwhile
// (64 VGPRs at most, so that eight waves per SIMD keep their loads in flight).  Against a launch each
// (Q codes, K partials, V partials): 4 x 8192 tokens, Hq 28 / Hk 4, 108 -> 98 us (4.9 TB/s, as a plain copy;
// 108 with the indexes of a workgroup by division); 30,001 tokens, Hq 32 / Hk 8, 160 -> 108 us (117); 1,024 tokens,
// Hq 24 / Hk 8, 10.8 (and two launches) -> 7.2 us.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void prepare_stats_kernel(PrepareArgs a) {
  int wg = a.wg0 + blockIdx.x;
  if (wg < a.kstat_wgs + a.vstat_wgs) {
    const bool isv = wg >= a.kstat_wgs;
    if (isv) wg -= a.kstat_wgs;
    const int hb = wg / (STAT_BLOCKS / 4), blk = (wg % (STAT_BLOCKS / 4)) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int b = a.kvheads.quotient(hb), hd = hb - b * a.hk;
    const uint16_t* src = isv ? a.v + b * a.vsb + hd * a.vsh : a.k + b * a.ksb + hd * a.ksh;
    stat_block(src, isv ? a.vst : a.kst, a.t, blk, (isv ? a.vpart : a.kpart) + (int64_t)hb * STAT_BLOCKS * 3 * D);
    return;
  }
  quantize_q_rows(a, wg - a.kstat_wgs - a.vstat_wgs);
}

// Statistics of one head from its block partials: mean = (sum of block sums in block order) / T, scale =
// range/127 (1 if 0), inv = 1/scale.  common_device.cuh:44-56 (finalize_kernel).  In a call of few heads every record
// workgroup forms them again (L2-resident partials) instead of waiting for a launch that does nothing
// else.  256 threads: one half adds the channel's block sums, the other takes its extremes; mean and
// inv (LDS, 128 each) are complete after the call's barrier.  stat (when not null) receives all three.
// `range`: whether scale and inv are needed (a K record needs the mean alone).
__device__ __forceinline__ void head_stats(const float* __restrict__ partial, int t, bool range, float* mean_lds,
                                           float* inv_lds, float* hi_lds, float* lo_lds, float* __restrict__ stat) {
  const int c = threadIdx.x & (D - 1);
  const float* in = partial + c;
  float sum = 0.f;
  if (threadIdx.x < D) {
    // (unrolled: the 64 loads issue together, and the sum still runs in block order)
#pragma unroll
    for (int blk = 0; blk < STAT_BLOCKS; ++blk) sum += in[blk * 3 * D];
  } else if (range) {
    float hi = -3.402823466e38f, lo = 3.402823466e38f;
#pragma unroll 32
    for (int blk = 0; blk < STAT_BLOCKS; ++blk) {
      hi = fmaxf(hi, in[blk * 3 * D + D]);
      lo = fminf(lo, in[blk * 3 * D + 2 * D]);
    }
    hi_lds[c] = hi;
    lo_lds[c] = lo;
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const float mean = sum / (float)t;
    mean_lds[c] = mean;
    if (range) {
      const float r = fmaxf(hi_lds[c] - mean, mean - lo_lds[c]);
      const float scale = r > 0.f ? r / 127.f : 1.f;
      inv_lds[c] = 1.f / scale;
      if (stat != nullptr) {
        stat[c] = mean;
        stat[D + c] = scale;
        stat[2 * D + c] = 1.f / scale;
      }
    }
  }
  __syncthreads();
}

// A 64-key tile's bf16 rows src + r * st (r < rows), loaded ahead of their use: quantize_k_tile's key
// layout (wave w rows 16w..16w+15 in two passes of 8 keys, 16 features per lane) and pack_v_tile's (four
// channels per thread, 8 rows apart).
struct KRaw {
  uint2 w[2][4];
};
struct VRaw {
  uint2 w[8];
};
__device__ __forceinline__ void load_k_tile(KRaw& raw, const uint16_t* __restrict__ src, int64_t st, int rows) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int r = wave * 16 + it * 8 + (lane >> 3);
#pragma unroll
    for (int i = 0; i < 4; ++i) raw.w[it][i] = make_uint2(0u, 0u);
    if (r < rows) {
      const uint16_t* row = src + (int64_t)r * st + (lane & 7) * 16;
#pragma unroll
      for (int i = 0; i < 4; ++i) raw.w[it][i] = *reinterpret_cast<const uint2*>(row + 4 * i);
    }
  }
}
__device__ __forceinline__ void load_v_tile(VRaw& raw, const uint16_t* __restrict__ src, int64_t st, int rows) {
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int r = n * 8 + (threadIdx.x >> 5), c0 = (threadIdx.x & 31) * 4;
    raw.w[n] = make_uint2(0u, 0u);
    if (r < rows) raw.w[n] = *reinterpret_cast<const uint2*>(src + (int64_t)r * st + c0);
  }
}

// y = R(k - mean) of one 64-key tile: the rows of raw below `rows` (zeros past); the INT8 record rec8
// with its four group scales ka, and the INT4 record rec4 with ka4 (either pair may be null).  Wave w
// owns the 16-key group w, one key per 8 lanes (16 features per lane, DPP rotation), two passes of 8
// keys; c8 / c4 are the workgroup's LDS staging.  256 threads.
// common_device.cuh:58-131 (quantize_k_kernel).
// Extension: rec4x (with rec4; may be null) receives the INT4 codes once more, expanded to one byte of
// 16 * code each in the INT8 record's layout (8 KiB): the bytes the prefill kernel would otherwise expand
// from rec4 in every tile it reads.
__device__ __forceinline__ void quantize_k_tile(const KRaw& in, int rows,
                                                const float* __restrict__ mean, uint8_t* __restrict__ rec8,
                                                float* __restrict__ ka, uint8_t* __restrict__ rec4,
                                                float* __restrict__ ka4, uint8_t (*c8)[D], uint8_t (*c4)[D],
                                                uint8_t* __restrict__ rec4x = nullptr) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, sub = lane & 7;
  float mc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) mc[i] = mean[sub * 16 + i];
  float y[2][16];
  float cm = 0.f;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int r = wave * 16 + it * 8 + (lane >> 3);
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = 0.f;
    if (r < rows) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint2 raw = in.w[it][i];
        x[4 * i] = bf16f(raw.x & 0xffffu) - mc[4 * i];
        x[4 * i + 1] = bf16f(raw.x >> 16) - mc[4 * i + 1];
        x[4 * i + 2] = bf16f(raw.y & 0xffffu) - mc[4 * i + 2];
        x[4 * i + 3] = bf16f(raw.y >> 16) - mc[4 * i + 3];
      }
    }
    rotate128_x16(x, sub);  // every lane of the wave takes part (padded rows rotate zeros)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      y[it][i] = x[i];
      cm = fmaxf(cm, fabsf(x[i]));
    }
  }
  cm = wave_max(cm);
  const float inv = cm > 0.f ? 127.f / cm : 0.f, inv4 = cm > 0.f ? 7.f / cm : 0.f;
  if (lane == 0) {
    if (rec8 != nullptr) ka[wave] = cm > 0.f ? cm / 127.f : 1.f;
    if (rec4 != nullptr) ka4[wave] = cm > 0.f ? cm / 7.f : 1.f;
  }
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int r = wave * 16 + it * 8 + (lane >> 3);
    uint32_t w8[4], w4[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      w8[q] = 0u;
      w4[q] = 0u;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        w8[q] |= ((uint32_t)(int)__builtin_rintf(y[it][4 * q + i] * inv) & 0xffu) << (8 * i);
        w4[q] |= ((uint32_t)(int)__builtin_rintf(y[it][4 * q + i] * inv4) & 0xfu) << (8 * i);
      }
    }
    *reinterpret_cast<uint4*>(&c8[r][sub * 16]) = make_uint4(w8[0], w8[1], w8[2], w8[3]);
    *reinterpret_cast<uint4*>(&c4[r][sub * 16]) = make_uint4(w4[0], w4[1], w4[2], w4[3]);
  }
  __syncthreads();
  if (rec8 != nullptr) {
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int s = tid + it * 256, F = s >> 6, L = s & 63, kb = F >> 2, ks = F & 3;
      const int key = kb * 32 + (L & 31), f0 = ks * 32 + 16 * (L >> 5);
      *reinterpret_cast<uint4*>(rec8 + F * 1024 + L * 16) = *reinterpret_cast<const uint4*>(&c8[key][f0]);
    }
  }
  if (rec4 == nullptr) return;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int s = tid + it * 256, F = s >> 6, L = s & 63, kb = F >> 2, ks = F & 3;
    const int key = kb * 32 + (L & 31), f0 = ks * 32 + 16 * (L >> 5);
    const uint4 n = *reinterpret_cast<const uint4*>(&c4[key][f0]);  // one nibble value per byte
    const uint32_t w0 = n.x | (n.y << 4), w1 = n.z | (n.w << 4);
    *reinterpret_cast<uint2*>(rec4 + (F >> 1) * 1024 + L * 16 + (F & 1) * 8) = make_uint2(w0, w1);
    if (rec4x != nullptr)
      *reinterpret_cast<uint4*>(rec4x + F * 1024 + L * 16) =
          make_uint4((n.x << 4) & 0xf0f0f0f0u, (n.y << 4) & 0xf0f0f0f0u, (n.z << 4) & 0xf0f0f0f0u,
                     (n.w << 4) & 0xf0f0f0f0u);
  }
}

// v' = (v - mean) * inv of one 64-key tile (the rows of raw below `rows`, zeros past) into the V16
// (fp16), V8 and V4 records (any may be null); vn is the workgroup's LDS staging.  256 threads.
// common_device.cuh:132-172 (vnorm, pack_v_kernel).
// Extension: v8s (with v8; may be null) receives -127 times each channel's sum of the tile's 64 V8 codes
// (int32 [128], channel order), the value the prefill's P V product starts from (vsum: LDS of 128 ints).
__device__ __forceinline__ void pack_v_tile(const VRaw& in, int rows,
                                            const float* __restrict__ mean, const float* __restrict__ inv,
                                            uint8_t* __restrict__ v16, uint8_t* __restrict__ v8,
                                            uint8_t* __restrict__ v4, float (*vn)[D + 1],
                                            int32_t* __restrict__ v8s = nullptr, int* vsum = nullptr) {
  const int tid = threadIdx.x;
  if (v8s != nullptr && tid < D) vsum[tid] = 0;
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int r = n * 8 + (tid >> 5), c0 = (tid & 31) * 4;
    float x[4] = {0.f, 0.f, 0.f, 0.f};
    if (r < rows) {
      const uint2 raw = in.w[n];
      x[0] = (bf16f(raw.x & 0xffffu) - mean[c0]) * inv[c0];
      x[1] = (bf16f(raw.x >> 16) - mean[c0 + 1]) * inv[c0 + 1];
      x[2] = (bf16f(raw.y & 0xffffu) - mean[c0 + 2]) * inv[c0 + 2];
      x[3] = (bf16f(raw.y >> 16) - mean[c0 + 3]) * inv[c0 + 3];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) vn[r][c0 + j] = x[j];
  }
  __syncthreads();
  if (v16 != nullptr) {
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int s = tid + it * 256, F = s >> 6, L = s & 63, kh = F & 1, kb = (F >> 1) & 1, cb = F >> 2;
      const int ch = cb * 32 + (L & 31), g = L >> 5;
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const int k0 = kb * 32 + 8 * (2 * kh + e / 4) + 4 * g + e % 4;
        w[e / 2] = (uint32_t)f32_to_f16_bits(vn[k0][ch]) | ((uint32_t)f32_to_f16_bits(vn[k0 + 1][ch]) << 16);
      }
      *reinterpret_cast<uint4*>(v16 + F * 1024 + L * 16) = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  if (v8 == nullptr && v4 == nullptr) return;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int s = tid + it * 256, F = s >> 6, L = s & 63, kb = F & 1, cb = F >> 1;
    const int ch = cb * 32 + (L & 31), g = L >> 5;
    uint32_t b8[4] = {0, 0, 0, 0}, b4[4] = {0, 0, 0, 0};
    int sum8 = 0;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
      const float x = vn[kb * 32 + 8 * (p / 4) + 4 * g + p % 4][ch];
      const int q8 = max(-127, min(127, (int)__builtin_rintf(x)));
      const int q4 = max(-7, min(7, (int)__builtin_rintf(x * (7.f / 127.f))));
      b8[p / 4] |= ((uint32_t)q8 & 0xffu) << (8 * (p % 4));
      b4[p / 4] |= ((uint32_t)q4 & 0xfu) << (8 * (p % 4));
      sum8 += q8;
    }
    // four threads hold 16 keys each of channel ch: integer adds, so the sum is order-free
    if (v8s != nullptr) atomicAdd(&vsum[ch], sum8);
    if (v8 != nullptr) *reinterpret_cast<uint4*>(v8 + F * 1024 + L * 16) = make_uint4(b8[0], b8[1], b8[2], b8[3]);
    if (v4 != nullptr)
      *reinterpret_cast<uint2*>(v4 + (F >> 1) * 1024 + L * 16 + (F & 1) * 8) =
          make_uint2(b4[0] | (b4[1] << 4), b4[2] | (b4[3] << 4));
  }
  if (v8s != nullptr) {
    __syncthreads();
    if (tid < D) v8s[tid] = -127 * vsum[tid];
  }
}

// The KX / VX records of the exact KV heads.  Keys at or past t are zero.  Per 64-key tile, 16 KiB each, 32-key
// half kb at byte kb*8192:
//   KX fragment F = ks (16-feature step), lane L 16 bytes = bf16 K[key kb*32 + L%32]
//      [features ks*16 + 8*(L/32) .. +7]      (A operand of S^T = K Q^T)
//   VX fragment F = cb*2 + kh, lane L element e = bf16 V[key kb*32 + 16*kh + 8*(e/4)
//      + 4*(L/32) + e%4][channel cb*32 + L%32] (A operand of O^T = V^T P^T)
// One tile: keys r < rows of ksrc / vsrc (row strides kst / vst) into the KX and VX
// records kd / vd; vt is the workgroup's LDS staging of V.  256 threads.
constexpr int EXACT_VP = D + 8;  // padded LDS row of the V staging (bf16 elements)
__device__ __forceinline__ void pack_exact_tile(const uint16_t* ksrc, int64_t kst, const uint16_t* vsrc, int64_t vst,
                                                int rows, uint8_t* kd, uint8_t* vd, uint16_t* vt) {
  const int tid = threadIdx.x;
  // K: 1024 16-byte pieces in source order (key, 8-feature piece)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + 256 * i, key = c >> 4, f0 = (c & 15) * 8;
    uint4 w = make_uint4(0, 0, 0, 0), u = w;
    if (key < rows) {
      w = *reinterpret_cast<const uint4*>(ksrc + (int64_t)key * kst + f0);
      u = *reinterpret_cast<const uint4*>(vsrc + (int64_t)key * vst + f0);
    }
    const int kb = key >> 5, lk = key & 31, ks = f0 >> 4, h = (f0 >> 3) & 1;
    *reinterpret_cast<uint4*>(kd + kb * (KX_BYTES / 2) + ks * 1024 + (h * 32 + lk) * 16) = w;
    *reinterpret_cast<uint4*>(vt + key * EXACT_VP + f0) = u;
  }
  __syncthreads();
  // V: 1024 output pieces in destination order
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + 256 * i, F = c >> 6, L = c & 63;  // F = kb*8 + cb*2 + kh
    const int kb = F >> 3, cb = (F >> 1) & 3, khalf = F & 1, ch = cb * 32 + (L & 31), h = L >> 5;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e0 = 2 * j, e1 = 2 * j + 1;
      const int k0 = kb * 32 + 16 * khalf + 8 * (e0 >> 2) + 4 * h + (e0 & 3);
      const int k1 = kb * 32 + 16 * khalf + 8 * (e1 >> 2) + 4 * h + (e1 & 3);
      w[j] = (uint32_t)vt[k0 * EXACT_VP + ch] | ((uint32_t)vt[k1 * EXACT_VP + ch] << 16);
    }
    *reinterpret_cast<uint4*>(vd + c * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// The statistics of every (part, head), one workgroup each, for the calls whose record workgroups read them.
__global__ __launch_bounds__(256) void prepare_finalize_kernel(PrepareArgs a) {
  __shared__ float mean[D], inv[D], hi[D], lo[D];
  const int heads = a.hk * a.batch, hb = blockIdx.x % heads;
  const bool isv = a.kstat_wgs == 0 || (int)blockIdx.x >= heads;
  head_stats((isv ? a.vpart : a.kpart) + (int64_t)hb * STAT_BLOCKS * 3 * D, a.t, true, mean, inv, hi, lo,
             (isv ? a.vstat : a.kstat) + (int64_t)hb * 3 * D);
}

// Whether a finalize launch pays, for `heads` (sequence, KV head) pairs of `tiles` tiles and the parts (0 or 1 each)
// that have statistics.  It costs a launch (~1.5 us); without it every record workgroup reads its head's partials (32
// KiB of K's, 96 of V's), which is free while they are few, and not once many heads' partials pass through every
// XCD's 4 MiB L2.  Calls without / with it, K, V (K and V): 4 heads x 64 tiles 25.7 / 27.4 us, 8 x 64 29.7 / 30.1, 32 x 8
// 24.2 / 22.5, 80 x 8 45.2 / 39.3, 8 x 219 77.2 / 73.2, 32 x 469 680 / 609; K alone, 32 x 24 32.1 / 33.3, 80 x 8 33.5 /
// 32.0, 32 x 64 67.3 / 65.5; V alone, 16 x 16 13.4 / 13.4, 32 x 8 16.3 / 14.0, 80 x 2 17.5 / 16.7.
inline bool finalize_pays(int64_t tiles, int64_t heads, int kparts, int vparts) {
  const int64_t partials = heads * (32 * kparts + 96 * vparts), work = heads * tiles;
  return partials > 0 && tiles > 1 && ((partials >= 2560 && work >= (vparts ? 128 : 512)) || work >= 1280);
}

// Last launch of a prepare call: the K records, the V records and the exact heads' KX / VX records, one workgroup per
// tile.  A K or V workgroup takes its head's statistics from prepare_finalize_kernel or forms them from the block
// partials (finalize_pays); then the one of a head's first tile writes them out.  HBM-bound for long prompts,
// latency-bound for short ones: a tile's rows are loaded before the statistics.  Against launches of their own for
// each head's statistics (K, V) and the K and V records: 1,024 tokens, 8 KV heads, 14.5 (and three launches) -> 7.2 us;
// with the finalize launch, 30,001 tokens, 8 KV heads, 71 -> 60 us, 4 x 8192 tokens, 4 KV heads, 47 -> 40 us, 4 x 30,000
// tokens, 8 KV heads, 263 -> 219 us.  (With up to 1,088 workgroups of several tiles each, the next one's rows loaded
// ahead, and the statistics formed in each: 76, 41 and 276 us; two tiles per workgroup after the finalize launch are
// 4% slower than one.)
__global__ __launch_bounds__(256) void prepare_records_kernel(PrepareArgs a) {
  // one staging buffer for the three parts: V' of a tile (fp32), K codes (one byte each, INT8 and INT4), or
  // the exact heads' bf16 V
  __shared__ __align__(16) float stage[BN][D + 1];
  __shared__ float mean[D], inv[D], hi[D], lo[D];
  __shared__ int vsum[D];
  static_assert(sizeof(stage) >= 2 * BN * D && sizeof(stage) >= BN * EXACT_VP * 2, "staging");
  const int tiles = (a.t + BN - 1) / BN;
  int wg = a.wg0 + blockIdx.x;
  if (wg < a.krec_wgs + a.vrec_wgs) {
    const bool isv = wg >= a.krec_wgs;
    if (isv) wg -= a.krec_wgs;
    const int hb = a.ktiles.quotient(wg), j = wg - hb * tiles, b = a.kvheads.quotient(hb), hd = hb - b * a.hk;
    const int rows = a.t - j * BN;
    const int64_t rec = (int64_t)hb * tiles + j;
    // the head's statistics into LDS; where they come from the partials, the workgroup of tile 0 writes them out
    auto stats = [&](const float* part, float* stat, bool range) {
      part += (int64_t)hb * STAT_BLOCKS * 3 * D;
      stat += (int64_t)hb * 3 * D;
      if (a.finalized) {
        if (threadIdx.x < D) mean[threadIdx.x] = stat[threadIdx.x];
        else inv[threadIdx.x - D] = stat[D + threadIdx.x];  // (threads D to 2 D - 1: stat[2 D + channel])
        __syncthreads();
      } else {
        head_stats(part, a.t, range || j == 0, mean, inv, hi, lo, j == 0 ? stat : nullptr);
      }
    };
    if (!isv) {
      KRaw raw;
      load_k_tile(raw, a.k + b * a.ksb + hd * a.ksh + (int64_t)j * BN * a.kst, a.kst, rows);
      stats(a.kpart, a.kstat, false);
      auto* c8 = reinterpret_cast<uint8_t (*)[D]>(&stage[0][0]);
      quantize_k_tile(raw, rows, mean, a.k8 + rec * K8_BYTES, a.ka + rec * 4,
                      a.k4 != nullptr ? a.k4 + rec * K4_BYTES : nullptr, a.k4 != nullptr ? a.ka4 + rec * 4 : nullptr, c8,
                      c8 + BN, a.k4x != nullptr ? a.k4x + rec * K8_BYTES : nullptr);
      return;
    }
    VRaw raw;
    load_v_tile(raw, a.v + b * a.vsb + hd * a.vsh + (int64_t)j * BN * a.vst, a.vst, rows);
    if (!a.v_identity) {
      stats(a.vpart, a.vstat, true);
    } else {
      if (threadIdx.x < D) {
        mean[threadIdx.x] = 0.f;
        inv[threadIdx.x] = 1.f;
        if (j == 0) {
          float* stat = a.vstat + (int64_t)hb * 3 * D + threadIdx.x;
          stat[0] = 0.f;
          stat[D] = 1.f;
          stat[2 * D] = 1.f;
        }
      }
      __syncthreads();
    }
    pack_v_tile(raw, rows, mean, inv, a.v16 != nullptr ? a.v16 + rec * V16_BYTES : nullptr,
                a.v8 != nullptr ? a.v8 + rec * V8_BYTES : nullptr, a.v4 != nullptr ? a.v4 + rec * V4_BYTES : nullptr,
                stage, a.v8s != nullptr ? a.v8s + rec * D : nullptr, vsum);
    return;
  }
  wg -= a.krec_wgs;
  wg -= a.vrec_wgs;
  // exact heads: workgroup (KV head, tile) of sequence b; other heads leave
  const int hb = a.ktiles.quotient(wg), tile = wg - hb * tiles, b = a.kvheads.quotient(hb), kh = hb - b * a.hk;
  const int slot = a.exact[kh * (a.hq / a.hk)] - 1;
  if (slot < 0 || slot >= a.nx) return;
  const int64_t rec = ((int64_t)b * a.nx + slot) * tiles + tile;
  pack_exact_tile(a.k + b * a.ksb + kh * a.ksh + (int64_t)tile * BN * a.kst, a.kst,
                  a.v + b * a.vsb + kh * a.vsh + (int64_t)tile * BN * a.vst, a.vst, a.t - tile * BN,
                  a.kx + rec * KX_BYTES, a.vx + rec * KX_BYTES, reinterpret_cast<uint16_t*>(&stage[0][0]));
}

}  // namespace tri
