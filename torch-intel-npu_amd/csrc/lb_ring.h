// gfx950 GEMM for grids of few tiles: y[M,N] = x[M,K] . dequant(W)[N,K]^T with the rank-r correction,
// the residual and the SmolLM layer's RoPE and SiLU-multiply in the same launch.
//
// A workgroup of eight waves owns 16 RT rows and 64 weight rows.  K advances in stages of 128 codes: the two
// K groups of four waves take a half of each stage, wave w of a group the weight rows 16 w .. 16 w + 15, and the
// groups' sums meet in LDS at the end.  Everything a stage needs (activations, packed weights, V) goes from
// memory straight to one of D LDS slots, D - 1 stages ahead of its use; the tile's scales are read once.
//
// What bounds it.  These grids leave most CUs with one workgroup, so a launch lasts as long as one workgroup's
// chain of stages.  Two things made the chain of the two-stage GEMM (lb_gemm.h, 64 x 64 tiles: 0.6 us per 64
// codes) long, and shape this kernel:
//   - a wave-wide load whose neighbouring lanes read different rows (the MFMA operand order: 16 rows) costs
//     27 ns of a CU's address unit whatever its width, a transfer of 1 KB in row order 10 ns (measured, four
//     waves, data in L2).  One weight load and one 2-byte scale load per wave and 64 codes took 0.22 us a step.
//     So weights are moved in row order and take their MFMA order from LDS, and scales are not loaded in the loop;
//   - a step that reads LDS, decodes and multiplies one after the other.  Here the reads of stage t + 2, the
//     decode of stage t + 1 and the products of stage t are independent of one another.
// Scales.  A wave's half stage of 64 codes lies in one group when groups are whole multiples of 64 (POST): codes
// enter the MFMA exact, from a zero accumulator, and the half's sums are scaled into the fp32 accumulator, so
// the product is the exact x.(q s).  Groups of 32 scale the weights (fp16(q s)) as they are decoded.
#pragma once
#include <type_traits>
#include <utility>

#include "lb_common.h"

namespace lb {

typedef uint32_t u2 __attribute__((ext_vector_type(2)));
constexpr int kRingMaxProblems = 3;
constexpr int kRingThreads = 512;
// RING_PLAIN: the problems' columns side by side.  RING_SILU: problems 0 and 1 are gate and up, the output is
// fp16(fp16(silu(gate)) up).  RING_ROPE: problems 0, 1, 2 are q (rotated), k (rotated, to the cache) and v (to
// the cache).  RING_SLICE: one problem, workgroup z sums codes z kslice .. of every row into fp32 partials
// [z, M, N], which splitk_reduce_kernel adds in slice order.
enum RingMode { RING_PLAIN = 0, RING_SILU = 1, RING_ROPE = 2, RING_SLICE = 3 };

struct RingProblem {
  const uint8_t *codes;   // packed codes (fp16 weights for FMT_FP16), rows [N, K]
  const f16 *scales;      // [N, G]
  const f16 *bias;        // [N] or null
  const f16 *residual;    // [M, ldr] or null: y = fp16(residual + y) last (may be y itself)
  const f16 *down;        // V [rank, K] or null
  const f16 *up;          // U [N, up_ld] or null
  f16 *y;                 // [M, ldy]
  int N, ldy, ldr, rank, up_ld;
  int tiles_end;          // exclusive prefix sum of column tiles over the problems
  int vec;                // y (and residual) rows are 16-byte aligned
};

struct RingParams {
  const f16 *x;           // [M, ldx]
  int M, K, ldx, G, group_shift, per_row;
  int row_bytes;          // bytes of a weight row
  int kslice;             // RING_SLICE: codes per slice, whole stages of 128
  float *partial;         // RING_SLICE: [slices, M, N]
  RingProblem prob[kRingMaxProblems];
  // RING_ROPE: row m is position start + m % seq of sequence m / seq.
  const f16 *cos, *sin;   // [capacity, 64]
  f16 *keys, *values;     // [batch, kv_heads, capacity, 64]
  int seq, start, capacity, kv_heads;
};

template <int N, class F, int... I>
__device__ __forceinline__ void ring_unroll_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void ring_unroll(F &&f) {
  ring_unroll_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// Layout of one stage: 128 codes of K.  Rows are staged without padding in 16-byte chunks, chunk c of row r
// at position c ^ swizzle(r), so that the 16 rows a fragment read serves together fall on distinct banks.
template <int FMT, int RT, int NV, int SCALE_KB>
struct RingTraits {
  static constexpr int BM = 16 * RT, BITS = FormatTraits<FMT>::BITS;
  static constexpr int B_ROW = 128 * BITS / 8;                     // bytes of a weight row per stage: 64, 128 or 256
  static constexpr int A_BYTES = BM * 256, B_BYTES = 64 * B_ROW, V_BYTES = 32 * 256;
  // Operands of four 1 KB blocks (the activations of RT = 1, 4-bit weights) are moved by one K group; the other
  // issues a transfer of no bytes into a spare 4 KB, so that every wave has the same transfers in flight.
  static constexpr bool A_SPARE = RT == 1, B_SPARE = BITS == 4;
  static constexpr int SPARE = A_BYTES + B_BYTES + NV * V_BYTES;
  static constexpr int STAGE = SPARE + (A_SPARE || B_SPARE ? 4096 : 0);
  static constexpr int FIT = (158 - SCALE_KB) * 1024 / STAGE;  // (160 KB less the NF4 table)
  static constexpr int DEPTH = FIT > 6 ? 6 : FIT;                  // slots in the ring
  // 1 KB transfers per wave: of the activations, of the weights, and of a whole stage.
  static constexpr int A_PER = A_SPARE ? 1 : RT / 2, B_PER = B_SPARE ? 1 : BITS / 8, OPS = A_PER + B_PER + NV;
};
// Swizzles of rows of 256 bytes (activations, V, fp16 weights), 128 (int8, the output tile) and 64 (4-bit codes).
template <int BYTES> __device__ __forceinline__ int ring_swz(int r) {
  return BYTES == 256 ? r & 15 : BYTES == 128 ? (r >> 1) & 7 : (r >> 2) & 3;
}

template <int FMT, int SCALE_KB, bool POST, bool RANKED, int RT, int MODE>
__global__ __launch_bounds__(kRingThreads) void ring_gemm_kernel(RingParams p) {
  constexpr bool PAIR = MODE == RING_SILU, SLICE = MODE == RING_SLICE, SCALED = SCALE_KB > 0;
  static_assert(!(SLICE && RANKED), "a correction's z takes the whole of K");
  static_assert(!POST || SCALED, "scales to apply");
  constexpr int NP = PAIR ? 2 : 1;                     // problems a tile's weight rows come from (32 of each)
  constexpr int NV = RANKED ? NP : 0;
  using T = RingTraits<FMT, RT, NV, SCALE_KB>;
  constexpr int D = T::DEPTH, BITS = FormatTraits<FMT>::BITS, BM = T::BM;
  constexpr int PART = 64 / NP;                        // output columns of a workgroup
  constexpr int kOutOfRange = (int)0x80000000u;
  // Correction activations z = x.V^T: RT x 2 NV tiles of 16 x 16, dealt to the four waves of a K group (a
  // wave's tiles share their rows).
  constexpr int ZCOLS = NV > 0 ? 2 * NV : 1, ZT = NV > 0 ? RT * ZCOLS : 0, ZPER = NV > 0 ? (ZT + 3) / 4 : 0;
  static_assert(ZPER <= 2 * NV && D >= 4 && (D - 2) * T::OPS < 63, "vmcnt range");

  // One array per slot: the compiler then sees that a transfer into one aliases no read of another.
  __shared__ __align__(1024) uint8_t S0[T::STAGE];
  __shared__ __align__(1024) uint8_t S1[T::STAGE];
  __shared__ __align__(1024) uint8_t S2[T::STAGE];
  __shared__ __align__(1024) uint8_t S3[T::STAGE];
  __shared__ __align__(1024) uint8_t S4[D > 4 ? T::STAGE : 16];
  __shared__ __align__(1024) uint8_t S5[D > 5 ? T::STAGE : 16];
  __shared__ uint32_t nf4_table[FMT == FMT_NF4 ? 256 : 1];
  __shared__ __align__(16) f16 scales_lds[SCALED ? SCALE_KB * 512 + 32 : 8];  // [64][G], the tile's scales (reads run two stages ahead)
  static_assert(RT * 4096 <= T::STAGE && ZPER * 4096 <= T::STAGE && NV * BM * 80 <= T::STAGE, "the epilogue reuses the slots");
  auto stage = [&](auto i) -> uint8_t * {
    constexpr int I = decltype(i)::value;
    if constexpr (I == 0) return S0;
    else if constexpr (I == 1) return S1;
    else if constexpr (I == 2) return S2;
    else if constexpr (I == 3) return S3;
    else if constexpr (I == 4) return S4;
    else return S5;
  };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;  // within its K group
  const int kg = __builtin_amdgcn_readfirstlane(tid >> 8);        // K group: half kg of every stage
  const int j = lane & 15, g = lane >> 4;
  if constexpr (FMT == FMT_NF4) build_nf4_pair_table(nf4_table);

  // The tile's problem and first column.
  int pi = 0, ct = blockIdx.x;
  if constexpr (!PAIR) {
    if (ct >= p.prob[0].tiles_end) pi = 1;
    if (ct >= p.prob[1].tiles_end) pi = 2;
    ct -= pi == 0 ? 0 : p.prob[pi - 1].tiles_end;
  }
  const RingProblem &pr = p.prob[pi];
  const int bn = ct * PART, bm = blockIdx.y * BM;
  const int rows_a = min(BM, p.M - bm);
  const int k0 = SLICE ? (int)blockIdx.z * p.kslice : 0, K = SLICE ? min(p.kslice, p.K - k0) : p.K;
  const int full = K / 128, rest = K % 128, stages = full + (rest ? 1 : 0);
  auto problem = [&](int e) -> const RingProblem & { return PAIR ? p.prob[e] : pr; };

  // Buffer views: (base, bytes).  A wave's transfer moves a block of 1 KB: 4 rows of 256 bytes, 8 of 128 or
  // 16 of 64; lane L fills position L % (row / 16) of its row, so it reads that position's chunk of the row.
  // Block i of a wave is block wave + 4 (kg + 2 i) of the operand.
  const f16 *xbase = p.x + (size_t)bm * p.ldx + k0;
  const int xbytes = ((rows_a - 1) * p.ldx + K) * 2;
  int a_off[T::A_PER];
#pragma unroll
  for (int i = 0; i < T::A_PER; ++i) {
    const int r = 4 * (wave + 4 * ((T::A_SPARE ? 0 : kg) + 2 * i)) + (lane >> 4);
    a_off[i] = r < rows_a && !(T::A_SPARE && kg > 0) ? r * p.ldx * 2 + 16 * ((lane & 15) ^ ring_swz<256>(r)) : kOutOfRange;
  }
  constexpr int CH = T::B_ROW / 16, BLOCK_ROWS = 64 / CH;
  const uint8_t *wbase[T::B_PER];
  int wbytes[T::B_PER], b_off[T::B_PER];
#pragma unroll
  for (int i = 0; i < T::B_PER; ++i) {
    const int first = BLOCK_ROWS * (wave + 4 * ((T::B_SPARE ? 0 : kg) + 2 * i)), r = first + lane / CH;
    const RingProblem &q = problem(first / PART);        // a block's rows belong to one problem
    const int rows_b = min(PART, q.N - bn), n = r % PART;
    wbase[i] = q.codes + (size_t)bn * p.row_bytes + k0 * BITS / 8;
    wbytes[i] = rows_b * p.row_bytes - k0 * BITS / 8;
    b_off[i] = n < rows_b && !(T::B_SPARE && kg == 0) ? n * p.row_bytes + 16 * ((lane % CH) ^ ring_swz<T::B_ROW>(r)) : kOutOfRange;
  }
  const int v_row = 4 * (wave + 4 * kg) + (lane >> 4);
  const int v_off = v_row * p.K * 2 + 16 * ((lane & 15) ^ ring_swz<256>(v_row));
  const int a_dst = wave * 1024 + (!T::A_SPARE ? kg * 4096 : kg > 0 ? T::SPARE : 0);
  const int b_dst = wave * 1024 + (!T::B_SPARE ? T::A_BYTES + kg * 4096 : kg == 0 ? T::SPARE : T::A_BYTES);
  // Transfers of stage t into ring slot I.  Stages past the last one move nothing and keep the count of
  // outstanding transfers the same in every stage.
  auto issue = [&](auto slot, int t) {
    const bool live = t < stages;
    // The waits count transfers, so those of one stage stay together: nothing moves across either end.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
#if defined(__HIP_DEVICE_COMPILE__)  // the LDS address space exists in the device pass only
    auto dma = [&](const void *base, int bytes, uint8_t *dst, int off) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer_rsrc(base, live ? bytes : 0),
                                               (__attribute__((address_space(3))) void *)dst, 16, off, 0, 0, 0);
    };
    uint8_t *dst = stage(slot);
#pragma unroll
    for (int i = 0; i < T::A_PER; ++i) dma(xbase, xbytes, dst + a_dst + i * 8192, a_off[i] + t * 256);
#pragma unroll
    for (int i = 0; i < T::B_PER; ++i) dma(wbase[i], wbytes[i], dst + b_dst + i * 8192, b_off[i] + t * T::B_ROW);
#pragma unroll
    for (int v = 0; v < NV; ++v)  // rows past the rank are out of range
      dma(problem(v).down, problem(v).rank * p.K * 2, dst + T::A_BYTES + T::B_BYTES + v * T::V_BYTES + kg * 4096 + wave * 1024,
          v_off + t * 256);
#endif
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  f4 acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  f4 zacc[ZPER > 0 ? ZPER : 1];
#pragma unroll
  for (int i = 0; i < ZPER; ++i) zacc[i] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  // What a wave reads of its half of a stage (64 codes): lane (j, g) holds k = 16 g .. 16 g + 15 of it, 8 per
  // MFMA, of activation row 16 r + j and weight row 16 wave + j.
  struct Raw {
    h8 a[2][RT], zv[2][ZPER > 0 ? ZPER : 1];
    uint32_t w[BITS / 2];
    f16 s;
  } raw[2];
  const int a_at[2] = {16 * ((8 * kg + 2 * g) ^ j) + j * 256, 16 * ((8 * kg + 2 * g + 1) ^ j) + j * 256};
  const int b_at = (16 * wave + j) * T::B_ROW +
                   (BITS == 4 ? 16 * ((2 * kg + (g >> 1)) ^ ring_swz<64>(j)) + 8 * (g & 1)
                    : BITS == 8 ? 16 * ((4 * kg + g) ^ ring_swz<128>(j)) : 16 * ((8 * kg + 2 * g) ^ j));
  auto read = [&](auto slot, int t, Raw &f) {
    const uint8_t *a = stage(slot), *b = a + T::A_BYTES;
    if constexpr (BITS == 4) {
      const u2 v = *reinterpret_cast<const u2 *>(b + b_at);
      f.w[0] = v[0];
      f.w[1] = v[1];
    } else {  // fp16: chunk 2 g + 1 is at the swizzled position of chunk 2 g with its lowest bit flipped
#pragma unroll
      for (int i = 0; i < BITS / 8; ++i) {
        const u4 v = *reinterpret_cast<const u4 *>(b + (b_at ^ (16 * i)));
#pragma unroll
        for (int e = 0; e < 4; ++e) f.w[4 * i + e] = v[e];
      }
    }
    if constexpr (SCALED) f.s = scales_lds[(16 * wave + j) * p.G + ((k0 + 128 * t + 64 * kg + 16 * g) >> p.group_shift)];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < RT; ++r) f.a[u][r] = *reinterpret_cast<const h8 *>(a + r * 4096 + a_at[u]);
#pragma unroll
      for (int i = 0; i < ZPER; ++i) {
        const int z = ZT % 4 != 0 ? min(wave * ZPER + i, ZT - 1) : wave * ZPER + i;
        f.zv[u][i] = *reinterpret_cast<const h8 *>(b + T::B_BYTES + (z % ZCOLS) * 4096 + a_at[u]);
      }
    }
  };
  struct Weights { h8 b[2]; float s; } wt[2];
  auto decode = [&](const Raw &f, Weights &o) {
    constexpr bool PRE = SCALED && !POST;
    const h2 s2 = PRE ? h2{f.s, f.s} : h2{(f16)1.0f, (f16)1.0f};
    if constexpr (POST) o.s = (float)f.s;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if constexpr (BITS == 4) o.b[u] = decode8_natural<FMT, PRE>(f.w[u], 0u, s2, nf4_table);
      else if constexpr (BITS == 8) o.b[u] = decode8_natural<FMT, PRE>(f.w[2 * u], f.w[2 * u + 1], s2, nf4_table);
      else o.b[u] = __builtin_bit_cast(h8, u4{f.w[4 * u], f.w[4 * u + 1], f.w[4 * u + 2], f.w[4 * u + 3]});
    }
  };
  static_assert(NV == 0 || RT <= 2, "a wave's z tiles take row tile 0 or RT - 1");
  const bool z_row = NV > 0 && ZT % 4 == 0 && wave * ZPER / ZCOLS > 0;  // (wave-uniform)
  auto multiply = [&](const Raw &f, const Weights &o) {
    f4 part[RT];  // D layout: a lane's sums are all of weight row 16 wave + j, whose scale it holds
#pragma unroll
    for (int r = 0; r < RT; ++r) part[r] = POST ? f4{0.0f, 0.0f, 0.0f, 0.0f} : acc[r];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < RT; ++r) part[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.a[u][r], o.b[u], part[r], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < ZPER; ++i)
        zacc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(RT > 1 && z_row ? f.a[u][RT - 1] : f.a[u][0], f.zv[u][i], zacc[i], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      if constexpr (POST) acc[r] += o.s * part[r];
      else acc[r] = part[r];
    }
  };

  // Ahead of the ring: the tile's scales (contiguous rows of G, through registers) and the correction's
  // rows of U (16-byte pieces of ranks 8 g ..).
  constexpr int S_PER = SCALED ? (SCALE_KB * 64 / NP + kRingThreads - 1) / kRingThreads : 1;
  u4 sreg[NP][S_PER];
  if constexpr (SCALED) {
#pragma unroll
    for (int e = 0; e < NP; ++e) {
      const int rows_b = min(PART, problem(e).N - bn);
      const int bytes = rows_b * p.G * 2;
      const __amdgpu_buffer_rsrc_t sbuf = buffer_rsrc(problem(e).scales + (size_t)bn * p.G, bytes);
#pragma unroll
      for (int i = 0; i < S_PER; ++i) {
        const int at = 16 * (tid + kRingThreads * i);
        sreg[e][i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(sbuf, at, 0, 0));
        if (at < bytes && at + 16 > bytes) {  // the end of the array inside a chunk (out-of-range dwords read zero)
          h8 v;
#pragma unroll
          for (int q = 0; q < 8; ++q)
            v[q] = __builtin_bit_cast(f16, __builtin_amdgcn_raw_buffer_load_b16(sbuf, at + 2 * q, 0, 0));
          sreg[e][i] = __builtin_bit_cast(u4, v);
        }
      }
    }
  }
  const int we = PAIR ? wave >> 1 : 0;                            // the wave's problem of the pair ...
  const int wn = bn + (PAIR ? 16 * (wave & 1) : 16 * wave) + j;   // ... and its lane's weight row
  h8 fu = {0, 0, 0, 0, 0, 0, 0, 0};
  if constexpr (RANKED) {
    const RingProblem &q = problem(we);
    const __amdgpu_buffer_rsrc_t ubuf = buffer_rsrc(q.up, q.rank > 0 ? ((size_t)(q.N - 1) * q.up_ld + q.rank) * 2 : 0);
    const int off = wn < q.N && 8 * g < q.rank ? (wn * q.up_ld + 8 * g) * 2 : kOutOfRange;
    fu = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(ubuf, off, 0, 0));
  }
  ring_unroll<D - 1>([&](auto i) { issue(i, decltype(i)::value); });
  if constexpr (SCALED) {
#pragma unroll
    for (int e = 0; e < NP; ++e)
#pragma unroll
      for (int i = 0; i < S_PER; ++i) {
        const int at = 8 * (tid + kRingThreads * i);
        if (at < PART * p.G) *reinterpret_cast<u4 *>(scales_lds + e * PART * p.G + at) = sreg[e][i];
      }
  }
  // All but the last `pending` stages' transfers of this wave are complete; past the barrier every wave's are.
  auto arrive = [&](auto pending) {
    constexpr int N = decltype(pending)::value;
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N * T::OPS) : "memory");
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the scales and the NF4 table are written
  arrive(std::integral_constant<int, D - 3>{});
  read(I0{}, 0, raw[0]);
  read(I1{}, 1, raw[1]);
  decode(raw[0], wt[0]);
  // Stage t: its products, the decode of stage t + 1, the reads of stage t + 2, and the transfers of stage
  // t + D - 1 into the slot of stage t - 1 (whose last reads fed products that every wave issued before the
  // barrier).
  constexpr int U = D % 2 ? 2 * D : D;
  auto advance = [&](auto i, int t) {
    constexpr int I = decltype(i)::value;
    __builtin_amdgcn_sched_barrier(0);
    arrive(std::integral_constant<int, D - 4>{});
    issue(std::integral_constant<int, (I + D - 1) % D>{}, t + D - 1);
    multiply(raw[I & 1], wt[I & 1]);
    read(std::integral_constant<int, (I + 2) % D>{}, t + 2, raw[I & 1]);
    decode(raw[(I & 1) ^ 1], wt[(I & 1) ^ 1]);
  };
  int t0 = 0;
  for (; t0 + U <= full; t0 += U) ring_unroll<U>([&](auto i) { advance(i, t0 + decltype(i)::value); });
  ring_unroll<U - 1>([&](auto i) {
    if (t0 + decltype(i)::value < full) advance(i, t0 + decltype(i)::value);
  });
  // A last stage of 32, 64 or 96 codes: whole halves as they are; of half a half, lanes past its end hold zeros.
  auto last = [&](Raw &f, Weights &o) {
    if (rest < 64 + 64 * kg) {
      const h8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        o.b[u] = g >= 2 ? zero : o.b[u];
#pragma unroll
        for (int r = 0; r < RT; ++r) f.a[u][r] = g >= 2 ? zero : f.a[u][r];
#pragma unroll
        for (int i = 0; i < ZPER; ++i) f.zv[u][i] = g >= 2 ? zero : f.zv[u][i];
      }
    }
    multiply(f, o);
  };
  if (rest > 64 * kg) {
    if (full & 1) last(raw[1], wt[1]);
    else last(raw[0], wt[0]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no transfer into LDS outlives the loop
  __syncthreads();

  // The second group's sums are added to the first's through S0 (S1: z).
  {
    auto slot = [&](uint8_t *base, int i) { return reinterpret_cast<f4 *>(base) + (i * 4 + wave) * 64 + lane; };
    if (kg == 1) {
#pragma unroll
      for (int r = 0; r < RT; ++r) *slot(S0, r) = acc[r];
#pragma unroll
      for (int i = 0; i < ZPER; ++i) *slot(S1, i) = zacc[i];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[r] += *slot(S0, r);
#pragma unroll
      for (int i = 0; i < ZPER; ++i) zacc[i] += *slot(S1, i);
    }
  }
  // D layout of the 16x16 MFMA: lane (j, g), register q -> row 4 g + q, column j.
  if constexpr (SLICE) {
    if (kg == 0 && wn < pr.N) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int m = bm + 16 * r + 4 * g + e;
          if (m < p.M) p.partial[((size_t)blockIdx.z * p.M + m) * pr.N + wn] = acc[r][e];
        }
    }
    return;
  }
  // S2: the fp16 z of the problems, rows of 32 at a pitch of 40.  S3: the output tile, 64 columns (gate's 32, then
  // up's) in rows of 128 bytes with swizzled chunks.
  f16 *zs = reinterpret_cast<f16 *>(S2);
  auto out_at = [&](int r, int col) -> f16 * {
    return reinterpret_cast<f16 *>(S3 + r * 128 + 16 * ((col >> 3) ^ ring_swz<128>(r))) + (col & 7);
  };
  f4 d[RANKED ? RT : 1];
  if constexpr (RANKED) {
#pragma unroll
    for (int i = 0; i < ZPER; ++i) {
      const int z = wave * ZPER + i;
      if (kg > 0 || (ZT % 4 != 0 && z >= ZT)) continue;
      const int v = z % ZCOLS / 2, col = 16 * (z & 1) + j;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        zs[(v * BM + 16 * (z / ZCOLS) + 4 * g + e) * 40 + col] = col < problem(v).rank ? (f16)zacc[i][e] : (f16)0.0f;
    }
    __syncthreads();
    const f4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const h8 fz = *reinterpret_cast<const h8 *>(zs + (we * BM + 16 * r + j) * 40 + 8 * g);
      d[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fz, fu, zero4, 0, 0, 0);
    }
  }
  if (kg == 0) {
    const RingProblem &q = problem(we);
    const float scale = p.per_row && wn < q.N ? (float)q.scales[wn] : 1.0f;
    const bool biased = q.bias != nullptr;
    const float bias = biased && wn < q.N ? (float)q.bias[wn] : 0.0f;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f16 h = (f16)(acc[r][e] * scale);
        if (biased) h = (f16)((float)h + bias);
        if constexpr (RANKED) h = (f16)((float)h + (float)(f16)d[r][e]);
        *out_at(16 * r + 4 * g + e, 16 * wave + j) = h;
      }
  }
  __syncthreads();
  // The tile leaves in rows of 16-byte chunks.
  constexpr int PER_ROW = PART / 8;
#pragma unroll
  for (int i = 0; i < (BM * PER_ROW + kRingThreads - 1) / kRingThreads; ++i) {
    const int at = tid + kRingThreads * i, r = at / PER_ROW, c = (at % PER_ROW) * 8;
    if (BM * PER_ROW % kRingThreads != 0 && r >= BM) continue;
    if (r >= rows_a || bn + c >= pr.N) continue;
    const int m = bm + r, n = bn + c;
    h8 v = *reinterpret_cast<const h8 *>(out_at(r, c));
    if constexpr (PAIR) {
      const h8 up = *reinterpret_cast<const h8 *>(out_at(r, 32 + c));
      // __expf: over all finite fp16 gates the rounded SiLU is off by rms 1.71271e-4 of its value, as with expf (3 and 1
      // of 63488 differ from the rounded 64-bit value); expf takes 0.6 us more a launch (256 rows, 1536 columns).
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float gate = (float)v[e];
        const f16 act = (f16)(gate / (1.0f + __expf(-gate)));
        v[e] = (f16)((float)act * (float)up[e]);
      }
    }
    if constexpr (MODE == RING_ROPE) {
      const int b = m / p.seq, pos = p.start + m % p.seq;
      if (pi < 2) {  // fp16(fp16(t cos) + fp16(rotate_half(t) sin))
        const h8 other = *reinterpret_cast<const h8 *>(out_at(r, c ^ 32));
        const h8 cs = *reinterpret_cast<const h8 *>(p.cos + (size_t)pos * 64 + c);
        const h8 sn = *reinterpret_cast<const h8 *>(p.sin + (size_t)pos * 64 + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const f16 o = c < 32 ? (f16)-other[e] : other[e];
          const f16 t0 = (f16)((float)v[e] * (float)cs[e]), t1 = (f16)((float)o * (float)sn[e]);
          v[e] = (f16)((float)t0 + (float)t1);
        }
      }
      f16 *dst = pi == 0 ? pr.y + (size_t)m * pr.ldy + n
                         : (pi == 1 ? p.keys : p.values) + (((size_t)b * p.kv_heads + ct) * p.capacity + pos) * 64 + c;
      *reinterpret_cast<h8 *>(dst) = v;
      continue;
    }
    f16 *dst = pr.y + (size_t)m * pr.ldy + n;
    const f16 *res = pr.residual ? pr.residual + (size_t)m * pr.ldr + n : nullptr;
    if (pr.vec && n + 8 <= pr.N) {
      if (res) {
        const h8 o = *reinterpret_cast<const h8 *>(res);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (f16)((float)o[e] + (float)v[e]);
      }
      *reinterpret_cast<h8 *>(dst) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < pr.N) dst[e] = res ? (f16)((float)res[e] + (float)v[e]) : v[e];
    }
  }
}

// LDS kept for the tile's scales: 8 KB, or 28 where they need more (0: the kernel does not take them).
constexpr int ring_scale_kb(long long G) { return 128 * G <= 8 * 1024 ? 8 : 128 * G <= 28 * 1024 ? 28 : 0; }

// Launches the kernel over `tiles` column tiles (all problems) and row tiles of 16 rt (ring_abi.hip).
void launch_ring(const RingParams &p, int format, bool scaled, bool ranked, int rt, int tiles, hipStream_t stream);
// The same over `slices` K slices of p.kslice codes: per-row int8, int4 / nf4 in groups of 64 and more, rt 1, 2 or 4.
void launch_ring_slices(const RingParams &p, int format, int rt, int tiles, int slices, hipStream_t stream);

}  // namespace lb
