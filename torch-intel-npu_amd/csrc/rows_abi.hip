// lb_rms_rows and lb_layer_rows: a SmolLM layer over several token rows in seven launches.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/lowbit_decode_hip.h"
#include "abi_util.h"
#include "fused_launch.h"
#include "lb_ring.h"
#include "lb_rows.h"

using namespace lb;
using namespace lb::abi;

namespace {

template <int FMT, int SCALE_KB, bool POST, bool RANKED, int MODE>
void launch_mode_t(const RingParams &p, int rt, int tiles, hipStream_t s) {
  const dim3 grid((unsigned)tiles, (unsigned)((p.M + 16 * rt - 1) / (16 * rt)));
  switch (rt) {
    case 1: hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, POST, RANKED, 1, MODE>), grid, dim3(kRingThreads), 0, s, p); break;
    case 2: hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, POST, RANKED, 2, MODE>), grid, dim3(kRingThreads), 0, s, p); break;
    default:
      if constexpr (!RANKED) hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, POST, RANKED, 4, MODE>), grid, dim3(kRingThreads), 0, s, p);
      break;
  }
}

template <int MODE>
void launch_mode(const RingParams &p, int format, bool ranked, int rt, int tiles, hipStream_t s) {
  switch (format) {
    case FMT_INT8:
      ranked ? launch_mode_t<FMT_INT8, 0, false, true, MODE>(p, rt, tiles, s) : launch_mode_t<FMT_INT8, 0, false, false, MODE>(p, rt, tiles, s);
      break;
    case FMT_INT4:
      p.group_shift == 5 ? launch_mode_t<FMT_INT4, 8, false, false, MODE>(p, rt, tiles, s) : launch_mode_t<FMT_INT4, 8, true, false, MODE>(p, rt, tiles, s);
      break;
    case FMT_NF4:
      p.group_shift == 5 ? launch_mode_t<FMT_NF4, 8, false, false, MODE>(p, rt, tiles, s) : launch_mode_t<FMT_NF4, 8, true, false, MODE>(p, rt, tiles, s);
      break;
    default: launch_mode_t<FMT_FP16, 0, false, false, MODE>(p, rt, tiles, s); break;
  }
}

// Rows per workgroup (in sixteens): the smallest tile that leaves one round of 256 workgroups, past one round the largest
// there is (RoPE, the cache's append, SiLU and the residual are part of the launch, which gemm4_kernel's larger tiles
// have no form of).  A layer of 8 x 256 rows takes 146 us with W8 and rank 32, 94 with INT4, 64 x 256 rows 905 and 506,
// one prompt of 2000 rows 208 and 156; lb_linear per projection between torch operations 538, 438, 1528, 1131, 847, 687.
int rows_rt(int64_t M, int64_t tiles, bool ranked) {
  if ((M + 15) / 16 * tiles <= 256) return 1;
  if ((M + 31) / 32 * tiles <= 256 || ranked) return 2;
  return 4;
}

RingParams ring_params(const lb_layer_projection *q, int count, const void *x, int64_t M, int64_t K, int64_t ldx) {
  RingParams p{};
  const int fmt = (int)q[0].format;
  const bool dense = fmt == FMT_FP16;
  const int64_t group = dense ? K : q[0].group_size;
  p.x = static_cast<const f16 *>(x);
  p.M = (int)M;
  p.K = (int)K;
  p.ldx = (int)ldx;
  p.G = (int)(K / group);
  p.group_shift = group == K ? 31 : __builtin_ctzll((unsigned long long)group);
  p.per_row = fmt == FMT_INT8;
  p.row_bytes = (int)(dense ? 2 * K : fmt == FMT_INT8 ? K : K / 2);
  for (int i = 0; i < count; ++i) {
    RingProblem &r = p.prob[i];
    r.codes = static_cast<const uint8_t *>(q[i].codes);
    r.scales = static_cast<const f16 *>(q[i].scales);
    r.N = (int)q[i].N;
    r.rank = (int)q[i].rank;
    r.down = static_cast<const f16 *>(q[i].down);
    r.up = static_cast<const f16 *>(q[i].up);
    r.up_ld = (int)q[i].up_ld;
    r.vec = 1;
  }
  return p;
}

bool any_rank(const lb_layer_projection *q, int count) {
  for (int i = 0; i < count; ++i)
    if (q[i].rank > 0) return true;
  return false;
}

lb_status check_projection(const lb_layer_projection &q, int index, int64_t N, int64_t K) {
  if (q.format > LB_FORMAT_FP16) return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: projection %d: unknown format %u", index, q.format);
  if (q.N != N || q.K != K)
    return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: projection %d is %lldx%lld, expected %lldx%lld", index, (long long)q.N,
                (long long)q.K, (long long)N, (long long)K);
  if (!q.codes || !aligned(q.codes, 16)) return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: projection %d: codes need 16-byte alignment", index);
  if (q.format != LB_FORMAT_FP16) {
    if (!q.scales || !aligned(q.scales, 16)) return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: projection %d: scales need 16-byte alignment", index);
    if (q.group_size < 1 || q.group_size > K || K % q.group_size != 0)
      return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: projection %d: group_size %lld must divide %lld", index,
                  (long long)q.group_size, (long long)K);
    const bool power = q.group_size >= 32 && (q.group_size & (q.group_size - 1)) == 0;
    if (q.format == LB_FORMAT_INT8 ? q.group_size != K : !(power || q.group_size == K))
      return fail(LB_UNSUPPORTED, "lb_layer_rows: projection %d: int8 per row, int4 / nf4 groups a power of two >= 32 or one per row", index);
    if (q.format != LB_FORMAT_INT8 && ring_scale_kb(K / q.group_size) != 8)
      return fail(LB_UNSUPPORTED, "lb_layer_rows: projection %d: at most 64 groups per row", index);
  }
  if (q.rank < 0 || q.rank > 32 || q.rank % 8 != 0 || (q.rank > 0 && q.format != LB_FORMAT_INT8))
    return fail(LB_UNSUPPORTED, "lb_layer_rows: projection %d: ranks 8, 16, 24 or 32 with int8 weights", index);
  if (q.rank > 0 && (!q.down || !q.up || !aligned(q.down, 16) || !aligned(q.up, 16) || q.up_ld < q.rank || q.up_ld % 8 != 0))
    return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: projection %d: down / up need 16-byte alignment, up_ld >= rank a multiple of 8", index);
  if (q.rank > 0 && q.up_ld > INT32_MAX / 2 / q.N)  // (byte offsets into U are 32-bit)
    return fail(LB_UNSUPPORTED, "lb_layer_rows: projection %d: up_ld %lld is past 32-bit offsets", index, (long long)q.up_ld);
  return LB_OK;
}

bool same_kind(const lb_layer_projection &a, const lb_layer_projection &b) {
  return a.format == b.format && (a.format == LB_FORMAT_FP16 || a.group_size == b.group_size);
}

// One row of a layer whose K the single-row kernels take: five launches of them (lb_fused_linear without a
// workspace, lb_decode_attention), which neither stage sixteen rows for one nor walk K in stages: a 135M layer's
// W8 + rank 32 token 40 -> 25 us.
bool one_row(const lb_layer_rows_args *a) {
  if (a->batch != 1 || a->seq != 1 || a->intermediate > kFusedMaxK || a->hidden > kFusedMaxK) return false;
  for (const lb_layer_projection &q : a->proj)
    if ((q.format == LB_FORMAT_INT4 || q.format == LB_FORMAT_NF4) && (q.group_size & (q.group_size - 1)) != 0) return false;
  return true;
}

void launch_one_row(const lb_layer_rows_args *a, hipStream_t s) {
  const int64_t H = a->hidden, I = a->intermediate, kv = 64 * a->kv_heads;
  f16 *q = static_cast<f16 *>(a->workspace), *k = q + H, *v = k + kv, *att = v + kv, *h1 = att + H, *gate = h1 + H, *up = gate + I;
  auto linear = [&](const lb_layer_projection *w, int count, int prologue, const void *x, const void *x2, const void *gamma,
                    const void *residual, f16 *const *ys) {
    const int fmt = (int)w[0].format;
    const bool dense = fmt == FMT_FP16;
    const int64_t K = w[0].K, group = dense ? K : w[0].group_size;
    FusedParams p{};
    p.x = static_cast<const f16 *>(x);
    p.x2 = static_cast<const f16 *>(x2);
    p.gamma = static_cast<const f16 *>(gamma);
    p.eps = a->eps;
    p.K = (int)K;
    p.G = (int)(K / group);
    p.group_shift = group == K ? 31 : __builtin_ctzll((unsigned long long)group);
    p.per_row = fmt == FMT_INT8;
    p.prologue = prologue;
    int tiles = 0;
    for (int i = 0; i < kFusedMaxProblems; ++i) {
      FusedProblem &r = p.prob[i];
      if (i < count) {
        r.codes = static_cast<const uint8_t *>(w[i].codes);
        r.scales = static_cast<const f16 *>(w[i].scales);
        r.y = ys[i];
        r.residual = static_cast<const f16 *>(residual);
        r.N = (int)w[i].N;
        r.rank = (int)w[i].rank;
        r.down = static_cast<const f16 *>(w[i].down);
        r.up = static_cast<const f16 *>(w[i].up);
        r.up_ld = (int)w[i].up_ld;
        tiles += (int)((w[i].N + 15) / 16);
      }
      r.tiles_end = tiles;
    }
    launch_fused(p, fmt, !dense && fmt != FMT_INT8, any_rank(w, count), tiles, s);
  };
  f16 *const qkv[] = {q, k, v}, *const o[] = {h1}, *const gu[] = {gate, up}, *const out[] = {static_cast<f16 *>(a->out)};
  linear(a->proj, 3, PRO_RMSNORM, a->x, nullptr, a->norm1, nullptr, qkv);
  AttnParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.cos = static_cast<const f16 *>(a->cos);
  p.sin = static_cast<const f16 *>(a->sin);
  p.slot = (int)a->start;
  p.keys = static_cast<f16 *>(a->keys);
  p.values = static_cast<f16 *>(a->values);
  p.out = att;
  p.heads = (int)a->heads;
  p.kv_heads = (int)a->kv_heads;
  p.capacity = (int)a->capacity;
  p.scale = a->scale;
  launch_decode_attention(p, s);
  linear(a->proj + 3, 1, PRO_NONE, att, nullptr, nullptr, a->x, o);
  linear(a->proj + 4, 2, PRO_RMSNORM, h1, nullptr, a->norm2, nullptr, gu);
  linear(a->proj + 6, 1, PRO_SILU_MUL, gate, up, nullptr, h1, out);
}

// Workspace: normalised rows, q, attention and h1 [M, hidden], act [M, intermediate]; of one row q, k, v, attention,
// h1, gate and up.
size_t rows_workspace(int64_t M, int64_t hidden, int64_t intermediate) {
  return ((size_t)M * (4 * hidden + intermediate) + 2 * hidden + intermediate) * 2;
}

}  // namespace

extern "C" {

lb_status lb_rms_rows(const void *x, const void *gamma, void *y, int64_t M, int64_t K, float eps, void *stream) {
  if (const lb_status bad = refuse_if_failed("lb_rms_rows"); bad != LB_OK) return bad;
  if (!x || !gamma || !y || M < 1 || M > INT32_MAX / 4 || K < 8 || K > kRowsMaxHidden || K % 8 != 0)
    return fail(LB_INVALID_ARGUMENT, "lb_rms_rows: M >= 1 rows of K = 8..%d values (a multiple of 8)", kRowsMaxHidden);
  if (!aligned(x, 16) || !aligned(gamma, 16) || !aligned(y, 16))
    return fail(LB_INVALID_ARGUMENT, "lb_rms_rows: x, gamma and y need 16-byte alignment");
  const Range out = range_of(y, (size_t)M * K * 2, "y");
  if (overlaps(out, range_of(x, (size_t)M * K * 2, "x")) || overlaps(out, range_of(gamma, (size_t)K * 2, "gamma")))
    return fail(LB_INVALID_ARGUMENT, "lb_rms_rows: y overlaps an input");
  hipLaunchKernelGGL(rms_rows_kernel, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const f16 *>(x), static_cast<const f16 *>(gamma), static_cast<f16 *>(y), (int)M, (int)K, eps);
  return launch_status("lb_rms_rows");
}

lb_status lb_layer_rows(const lb_layer_rows_args *a, void *stream) {
  if (const lb_status bad = refuse_if_failed("lb_layer_rows"); bad != LB_OK) return bad;
  if (!a) return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: args is NULL");
  if (a->struct_size < sizeof(lb_layer_rows_args))
    return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: struct_size %u < %zu", a->struct_size, sizeof(lb_layer_rows_args));
  // Comparisons that no 64-bit argument overflows; the products and sums below are of checked values.
  if (a->batch < 1 || a->batch > 65535 || a->seq < 1 || a->start < 0 || a->capacity < a->seq || a->capacity > INT32_MAX ||
      a->start > a->capacity - a->seq)
    return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: batch 1..65535, seq >= 1 and start + seq <= capacity <= 2^31 - 1 required");
  if (a->hidden < 64 || a->hidden > kRowsMaxHidden || a->heads < 1 || a->heads > kRowsMaxHidden / 64 || a->hidden != 64 * a->heads ||
      a->kv_heads < 1 || a->heads % a->kv_heads != 0 || a->intermediate < 32 || a->intermediate % 32 != 0 || a->intermediate > 65536)
    return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: hidden = 64 heads <= %d, heads a multiple of kv_heads, intermediate a "
                "multiple of 32 up to 65536", kRowsMaxHidden);
  const int64_t H = a->hidden, I = a->intermediate, M = a->batch * a->seq, kv = 64 * a->kv_heads;
  if (a->start + a->seq > kAttendMaxKeys || M > INT32_MAX / I / 4)
    return fail(LB_UNSUPPORTED, "lb_layer_rows: at most %d positions", kAttendMaxKeys);
  const struct { const void *p; const char *name; } pointers[] = {
      {a->x, "x"}, {a->out, "out"}, {a->norm1, "norm1"}, {a->norm2, "norm2"}, {a->cos, "cos"}, {a->sin, "sin"},
      {a->keys, "keys"}, {a->values, "values"}, {a->workspace, "workspace"}};
  for (const auto &q : pointers)
    if (!q.p || !aligned(q.p, 16)) return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: %s must be non-NULL with 16-byte alignment", q.name);
  const size_t need = rows_workspace(M, H, I);
  if (a->workspace_bytes < need)
    return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: workspace of %zu bytes required (got %zu)", need, a->workspace_bytes);
  const int64_t N[7] = {H, kv, kv, H, I, I, H}, K[7] = {H, H, H, H, H, H, I};
  for (int i = 0; i < 7; ++i)
    if (const lb_status st = check_projection(a->proj[i], i, N[i], K[i]); st != LB_OK) return st;
  if (!same_kind(a->proj[0], a->proj[1]) || !same_kind(a->proj[0], a->proj[2]) || !same_kind(a->proj[4], a->proj[5]))
    return fail(LB_UNSUPPORTED, "lb_layer_rows: q, k, v share one format and group, and gate, up another");
  const size_t cache = (size_t)a->batch * a->kv_heads * a->capacity * 128;
  const Range outs[] = {range_of(a->out, (size_t)M * H * 2, "out"), range_of(a->keys, cache, "keys"),
                        range_of(a->values, cache, "values"), range_of(a->workspace, need, "workspace")};
  const Range ins[] = {range_of(a->x, (size_t)M * H * 2, "x"), range_of(a->norm1, (size_t)H * 2, "norm1"),
                       range_of(a->norm2, (size_t)H * 2, "norm2"), range_of(a->cos, (size_t)a->capacity * 128, "cos"),
                       range_of(a->sin, (size_t)a->capacity * 128, "sin")};
  for (int i = 0; i < 4; ++i) {
    for (const Range &r : ins)
      if (overlaps(outs[i], r)) return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: %s overlaps %s", outs[i].name, r.name);
    for (int k = i + 1; k < 4; ++k)
      if (overlaps(outs[i], outs[k])) return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: %s overlaps %s", outs[i].name, outs[k].name);
  }
  for (int i = 0; i < 7; ++i) {
    const lb_layer_projection &q = a->proj[i];
    const bool dense = q.format == LB_FORMAT_FP16;
    const size_t codes = (size_t)q.N * q.K, ranked = q.rank > 0;
    const Range weights[] = {
        range_of(q.codes, dense ? 2 * codes : q.format == LB_FORMAT_INT8 ? codes : codes / 2, "codes"),
        range_of(q.scales, dense ? 0 : codes / q.group_size * 2, "scales"), range_of(q.down, (size_t)(q.rank * q.K * 2), "down"),
        range_of(q.up, ranked * (size_t)((q.N - 1) * q.up_ld + q.rank) * 2, "up")};
    for (const Range &out : outs)
      for (const Range &r : weights)
        if (overlaps(out, r))
          return fail(LB_INVALID_ARGUMENT, "lb_layer_rows: %s overlaps %s of projection %d", out.name, r.name, i);
  }

  hipStream_t s = static_cast<hipStream_t>(stream);
  if (one_row(a)) {
    launch_one_row(a, s);
    return launch_status("lb_layer_rows");
  }
  f16 *normed = static_cast<f16 *>(a->workspace), *q = normed + M * H, *att = q + M * H, *h1 = att + M * H, *act = h1 + M * H;
  auto norm = [&](const void *x, const void *gamma) {
    hipLaunchKernelGGL(rms_rows_kernel, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, s, static_cast<const f16 *>(x),
                       static_cast<const f16 *>(gamma), normed, (int)M, (int)H, a->eps);
  };
  auto residual = [&](const lb_layer_projection &w, const f16 *x, int64_t k, const void *res, void *y) {
    RingParams p = ring_params(&w, 1, x, M, k, k);
    const int tiles = (int)((H + 63) / 64);
    p.prob[0].y = static_cast<f16 *>(y);
    p.prob[0].residual = static_cast<const f16 *>(res);
    p.prob[0].ldy = p.prob[0].ldr = (int)H;
    for (RingProblem &r : p.prob) r.tiles_end = tiles;
    launch_ring(p, (int)w.format, w.format == LB_FORMAT_INT4 || w.format == LB_FORMAT_NF4, w.rank > 0, rows_rt(M, tiles, w.rank > 0),
                tiles, s);
  };
  norm(a->x, a->norm1);
  {
    RingParams p = ring_params(a->proj, 3, normed, M, H, H);
    const int tiles = (int)(a->heads + 2 * a->kv_heads);
    p.prob[0].y = q;
    p.prob[0].ldy = (int)H;
    p.prob[0].tiles_end = (int)a->heads;
    p.prob[1].tiles_end = (int)(a->heads + a->kv_heads);
    p.prob[2].tiles_end = tiles;
    p.cos = static_cast<const f16 *>(a->cos);
    p.sin = static_cast<const f16 *>(a->sin);
    p.keys = static_cast<f16 *>(a->keys);
    p.values = static_cast<f16 *>(a->values);
    p.seq = (int)a->seq;
    p.start = (int)a->start;
    p.capacity = (int)a->capacity;
    p.kv_heads = (int)a->kv_heads;
    const bool ranked = any_rank(a->proj, 3);
    launch_mode<RING_ROPE>(p, (int)a->proj[0].format, ranked, rows_rt(M, tiles, ranked), tiles, s);
  }
  {
    AttendParams p{};
    p.q = q;
    p.keys = static_cast<const f16 *>(a->keys);
    p.values = static_cast<const f16 *>(a->values);
    p.out = att;
    p.seq = (int)a->seq;
    p.start = (int)a->start;
    p.capacity = (int)a->capacity;
    p.heads = (int)a->heads;
    p.kv_heads = (int)a->kv_heads;
    p.pitch = (int)((a->start + a->seq + 31) / 32 * 32 + 8);
    p.scale = a->scale;
    hipLaunchKernelGGL(attend_rows_kernel, dim3((unsigned)((a->seq + 15) / 16), (unsigned)a->heads, (unsigned)a->batch), dim3(256),
                       (size_t)16 * p.pitch * 2, s, p);
  }
  residual(a->proj[3], att, H, a->x, h1);
  norm(h1, a->norm2);
  {
    RingParams p = ring_params(a->proj + 4, 2, normed, M, H, H);
    const int tiles = (int)(I / 32);
    p.prob[0].y = act;
    p.prob[0].ldy = (int)I;
    const bool ranked = any_rank(a->proj + 4, 2);
    launch_mode<RING_SILU>(p, (int)a->proj[4].format, ranked, rows_rt(M, tiles, ranked), tiles, s);
  }
  residual(a->proj[6], act, I, h1, a->out);
  return launch_status("lb_layer_rows");
}

}  // extern "C"
