// gfx950 kernels of a SmolLM layer over several token rows besides its GEMMs (lb_ring.h): RMSNorm of rows, and
// causal grouped-query attention of new rows over a KV cache.
#pragma once
#include "lb_common.h"

namespace lb {

constexpr int kRowsMaxHidden = 4096;
constexpr int kAttendMaxKeys = 2016;  // score rows of a workgroup in 64 KB of LDS

// y[m] = fp16(fp16(x[m] * rsqrt(mean(x[m]^2) + eps)) * gamma), a wave per row: 16-byte loads, the row kept in
// registers.  Bound by its launch: 256 x 576 rows move 0.6 MB (2.1 us a launch; the staged torch operations it
// stands for took seven launches, 15 us of kernel time).
__global__ __launch_bounds__(256) void rms_rows_kernel(const f16 *x, const f16 *gamma, f16 *y, int M, int K, float eps) {
  const int lane = threadIdx.x & 63, m = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;
  const f16 *row = x + (size_t)m * K;
  constexpr int PER = kRowsMaxHidden / 512;
  h8 v[PER], w[PER];
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int k = 512 * i + 8 * lane;
    if (512 * i >= K) break;
    if (k < K) {
      v[i] = *reinterpret_cast<const h8 *>(row + k);
      w[i] = *reinterpret_cast<const h8 *>(gamma + k);
    } else {
      v[i] = w[i] = h8{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) sum += (float)v[i][e] * (float)v[i][e];
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
  const float inv = 1.0f / sqrtf(sum / (float)K + eps);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int k = 512 * i + 8 * lane;
    if (k >= K) break;
    h8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (f16)((float)(f16)((float)v[i][e] * inv) * (float)w[i][e]);
    *reinterpret_cast<h8 *>(y + (size_t)m * K + k) = o;
  }
}

struct AttendParams {
  const f16 *q;               // [batch * seq, heads * 64], rotated
  const f16 *keys, *values;   // [batch, kv_heads, capacity, 64]
  f16 *out;                   // [batch * seq, heads * 64]
  int seq, start, capacity, heads, kv_heads, pitch;  // pitch: halves of a score row in LDS
  float scale;
};

// Causal attention of 16 query rows of one head and sequence: row m (position start + m) over cache slots
// 0 .. start + m, with the staging of the reference (scores fp16(q.k), fp16(* scale), softmax in fp32 rounded to
// fp16, fp16(P.V)).  Four waves deal the key tiles of Q.K^T (v_mfma_f32_16x16x32_f16, K rows straight from the
// cache as B operands), all scores of the rows stay in LDS as fp16 (16 x 2016 take 64 KB), each wave normalises
// four rows there, sixteen lanes a row, and P.V is dealt by output columns: wave w owns 16 of the 64 dims, its
// first 256 keys of V requested with the first keys.  Rows past the last visible
// slot are out of the buffers' range and read zero, so what lies there does not matter.  A whole score row is
// kept, not folded online, because the reference rounds the normalised probabilities.  Bound by latency at these
// sizes: 9 heads x 256 rows are 144 workgroups of at most 16 key tiles.
__global__ __launch_bounds__(256) void attend_rows_kernel(AttendParams p) {
  extern __shared__ __align__(16) f16 scores[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int q0 = blockIdx.x * 16, head = blockIdx.y, b = blockIdx.z;
  const int rows = min(16, p.seq - q0), ld = p.heads * 64;
  const int keys = p.start + q0 + rows;           // slots the last row sees
  const int tiles = (keys + 31) / 32 * 2;         // key tiles of 16, in whole pairs
  const size_t cache = ((size_t)b * p.kv_heads + head / (p.heads / p.kv_heads)) * p.capacity * 64;
  const __amdgpu_buffer_rsrc_t kbuf = buffer_rsrc(p.keys + cache, (size_t)keys * 128);
  const __amdgpu_buffer_rsrc_t vbuf = buffer_rsrc(p.values + cache, (size_t)keys * 128);

  const f16 *qrow = p.q + ((size_t)b * p.seq + q0 + j) * ld + head * 64 + 8 * g;
  h8 fq[2] = {{0, 0, 0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 0, 0, 0, 0}};
  if (j < rows) {
    fq[0] = *reinterpret_cast<const h8 *>(qrow);
    fq[1] = *reinterpret_cast<const h8 *>(qrow + 32);
  }
  // V of 32 keys as a B operand: lane (j, g) holds dim 16 wave + j of keys 8 g .. 8 g + 7.
  constexpr int VT = 8;                           // chunks of 32 keys in flight, requested ahead of the scores
  auto load_v = [&](int c) {
    h8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] = __builtin_bit_cast(f16, __builtin_amdgcn_raw_buffer_load_b16(
          vbuf, (32 * c + 8 * g + e) * 128 + (16 * wave + j) * 2, 0, 0));
    return v;
  };
  const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int KT = 4;                           // key tiles of a wave in flight
  h8 fv[VT];
  for (int t0 = wave; t0 < tiles; t0 += 4 * KT) {
    h8 fk[KT][2];
#pragma unroll
    for (int i = 0; i < KT; ++i)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        fk[i][u] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(
            kbuf, (16 * (t0 + 4 * i) + j) * 128 + 64 * u + 16 * g, 0, 0));
    if (t0 == wave) {
#pragma unroll
      for (int i = 0; i < VT; ++i) fv[i] = load_v(i);
    }
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int t = t0 + 4 * i;
      if (t >= tiles) break;
      f4 s = __builtin_amdgcn_mfma_f32_16x16x32_f16(fq[0], fk[i][0], zero, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x32_f16(fq[1], fk[i][1], s, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {               // row 4 g + e, key 16 t + j
        const int r = 4 * g + e, key = 16 * t + j;
        const f16 v = (f16)((float)(f16)s[e] * p.scale);
        scores[r * p.pitch + key] = key <= p.start + q0 + r ? v : (f16)-INFINITY;
      }
    }
  }
  if (wave >= tiles) {                            // two key tiles: waves 2 and 3 had none
#pragma unroll
    for (int i = 0; i < VT; ++i) fv[i] = load_v(i);
  }
  __syncthreads();
  // Softmax: sixteen lanes per row, eight scores a lane at a time; the exponentials of the first 256 scores
  // stay in registers for the division.
  {
    const int r = 4 * wave + (lane >> 4), chunks = 2 * tiles;
    f16 *row = scores + r * p.pitch + 8 * (lane & 15);
    constexpr int HELD = 2;
    float e[HELD][8], top = -INFINITY, total = 0.0f;
    for (int c = lane & 15, at = 0; c < chunks; c += 16, at += 128) {
      const h8 v = *reinterpret_cast<const h8 *>(row + at);
#pragma unroll
      for (int q = 0; q < 8; ++q) top = fmaxf(top, (float)v[q]);
    }
#pragma unroll
    for (int d = 8; d > 0; d >>= 1) top = fmaxf(top, __shfl_xor(top, d));
#pragma unroll
    for (int i = 0; i < HELD; ++i)
      if ((lane & 15) + 16 * i < chunks) {
        const h8 v = *reinterpret_cast<const h8 *>(row + 128 * i);
#pragma unroll
        for (int q = 0; q < 8; ++q) total += e[i][q] = expf((float)v[q] - top);
      }
    for (int c = (lane & 15) + 16 * HELD, at = 128 * HELD; c < chunks; c += 16, at += 128) {
      const h8 v = *reinterpret_cast<const h8 *>(row + at);
#pragma unroll
      for (int q = 0; q < 8; ++q) total += expf((float)v[q] - top);
    }
#pragma unroll
    for (int d = 8; d > 0; d >>= 1) total += __shfl_xor(total, d);
#pragma unroll
    for (int i = 0; i < HELD; ++i)
      if ((lane & 15) + 16 * i < chunks) {
        h8 v;
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = (f16)(e[i][q] / total);
        *reinterpret_cast<h8 *>(row + 128 * i) = v;
      }
    for (int c = (lane & 15) + 16 * HELD, at = 128 * HELD; c < chunks; c += 16, at += 128) {
      h8 v = *reinterpret_cast<const h8 *>(row + at);
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = (f16)(expf((float)v[q] - top) / total);
      *reinterpret_cast<h8 *>(row + at) = v;
    }
  }
  __syncthreads();
  f4 acc = zero;
  for (int c0 = 0; c0 < tiles / 2; c0 += VT) {
    if (c0 > 0) {
#pragma unroll
      for (int i = 0; i < VT; ++i) fv[i] = load_v(c0 + i);
    }
#pragma unroll
    for (int i = 0; i < VT; ++i) {
      if (c0 + i >= tiles / 2) break;
      h8 fp = *reinterpret_cast<const h8 *>(scores + j * p.pitch + 32 * (c0 + i) + 8 * g);
      if (j >= rows) fp = h8{0, 0, 0, 0, 0, 0, 0, 0};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(fp, fv[i], acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 4 * g + e;
    if (r < rows) p.out[((size_t)b * p.seq + q0 + r) * ld + head * 64 + 16 * wave + j] = (f16)acc[e];
  }
}

}  // namespace lb
