// Paged causal softmax attention of the float32 path on the 32-bit matrix instruction, head sizes that are multiples of
// 16 up to 128: prompt portions and single tokens, no sink, cap, chunk or bias (attention.hip takes those).
//
// One order of arithmetic for both kernels, so that a token's result is bit-identical however its request is cut: the
// keys are taken in segments of 128 whose bounds are absolute positions.  A segment gives its maximum m, the sum l of
// exp(s - m) and the sum O of exp(s - m) v; segments join in order,
//     M' = max(M, m),  L' = L exp(M - M') + l exp(m - M'),  O' likewise,
// and the result is O / L.  A masked key adds an exact zero to l and O, a segment a query sees nothing of changes nothing.
//
// A wave owns 16 queries of one kv head: the heads of its group, for as many neighbouring tokens as fit (16 / heads a
// group).  S^T = K Q^T and O^T += V^T P^T by v_mfma_f32_16x16x4_f32: a lane of the scores' accumulator holds four keys
// of one query, which is what the second product takes as its B operand, key 4 g + i of lane group g in instruction i;
// K rows and the values (transposed within their page) are read from memory in exactly these 16-byte pieces, a page's
// 16 keys at a time.  The queries of a group share every load; nothing goes through the LDS but the query fragments.
//   portions: a wave walks its segments itself.     single tokens: a wave a segment, joined by merge_f32_kernel.
// What bounds it is the latency of a wave's own loads (a segment's K, then its V, all of one issued together) and, for
// portions, the reads out of the L2s.  The kernel of attention.hip, one wave a (token, head), reads every key once a head
// and token, a quarter of a cache line a load: 512 tokens of 32 / 4 heads of 64 642 -> 38 us, 4 single tokens of 300 to
// 900 keys 200 -> 11 + 5 (MI355X).
#include "common.hpp"

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int AF_SEG = 128;                   // keys a segment
constexpr int AF_TILES = AF_SEG / 16;

struct AttArgs {
  const float* q;
  long q_stride;
  const float *k_cache, *v_cache;
  const int* block_tables;
  int max_blocks, Hq, Hkv, page, window;
  float scale;
};

// What segment `seg` gives 16 queries of kv head kvh: fragments qf, each lane's query at position pos (-1: none) with
// keys from lo on; first / last: the smallest lo and the largest position among the 16.  Every query sees the keys from all_lo to
// all_pos; a value that is not finite at another key, one that only some of them see, sets `odd`: a query that does not see
// the key has weight 0 there, and 0 times that value is not 0, so m and l are right and o is not.
template <int DT>
__device__ __forceinline__ void segment_sums(const AttArgs& a, const int* bt, int kvh, int seg, const f32x4 (&qf)[DT], int pos, int lo,
                                             int first, int last, int all_lo, int all_pos, float& m, float& l, f32x4 (&o)[DT], bool& odd) {
  constexpr int D = DT * 16;
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  const int base = seg * AF_SEG;
  const int t0 = first > base ? (first - base) >> 4 : 0;
  const int t1 = last - base >= AF_SEG ? AF_TILES : ((last - base) >> 4) + 1;
  constexpr int AHEAD = 32 / DT < AF_TILES ? (32 / DT >= 4 ? 4 : 2) : AF_TILES;   // tiles of 16 keys whose loads are issued together
  f32x4 s[AF_TILES];
  size_t at[AF_TILES];                        // of the page stretch a tile of 16 keys lies in
#pragma unroll
  for (int t = 0; t < AF_TILES; ++t) {        // a tile nobody sees stands for its neighbour: every table entry read is one of the request's
    const int tt = t < t0 ? t0 : t >= t1 ? t1 - 1 : t;
    at[t] = ((size_t)bt[(base + tt * 16) / a.page] * a.Hkv + kvh) * a.page * D;
  }
#pragma unroll
  for (int u = 0; u < AF_TILES; u += AHEAD) {
    f32x4 kf[AHEAD][DT];
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) {
      const float* kp = a.k_cache + at[u + t] + (size_t)((base + (u + t) * 16) % a.page + r16) * D + 4 * g;
#pragma unroll
      for (int c = 0; c < DT; ++c) kf[t][c] = *reinterpret_cast<const f32x4*>(kp + 16 * c);
    }
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) s[u + t] = none;
#pragma unroll
    for (int c = 0; c < DT; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < AHEAD; ++t) s[u + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][c][j], qf[c][j], s[u + t], 0, 0, 0);
  }
  float top = -INFINITY;
#pragma unroll
  for (int t = 0; t < AF_TILES; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = base + t * 16 + 4 * g + i;
      s[t][i] = key <= pos && key >= lo ? __fmul_rn(s[t][i], a.scale) : -INFINITY;
      top = fmaxf(top, s[t][i]);
    }
  top = fmaxf(top, __shfl_xor(top, 16, 64));
  top = fmaxf(top, __shfl_xor(top, 32, 64));
  m = top;
  const float sub = top == -INFINITY ? 0.f : top;
  float sum = 0.f;
#pragma unroll
  for (int t = 0; t < AF_TILES; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[t][i] = expf(s[t][i] - sub);
      sum += s[t][i];
    }
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  l = sum;
#pragma unroll
  for (int c = 0; c < DT; ++c) o[c] = none;
  bool some = false;
#pragma unroll
  for (int u = 0; u < AF_TILES; u += AHEAD) {
    f32x4 vf[AHEAD][DT];
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) {
      const float* vp = a.v_cache + at[u + t] + (size_t)r16 * a.page + (base + (u + t) * 16) % a.page + 4 * g;
#pragma unroll
      for (int c = 0; c < DT; ++c) vf[t][c] = *reinterpret_cast<const f32x4*>(vp + (size_t)(16 * c) * a.page);
    }
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) {
      const int key = base + (u + t) * 16 + 4 * g;
      if (key - 4 * g < all_lo || key - 4 * g + 15 > all_pos) {
        // keys none of the queries sees: nobody wrote them, or their page went back; and keys some of them see
#pragma unroll
        for (int c = 0; c < DT; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            vf[t][c][i] = key + i >= first && key + i <= last ? vf[t][c][i] : 0.f;
            some |= !(fabsf(vf[t][c][i]) < INFINITY) && (key + i < all_lo || key + i > all_pos);
          }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < DT; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t][c][i], s[u + t][i], o[c], 0, 0, 0);
    }
  }
  odd = __builtin_amdgcn_ballot_w64(some) != 0;
}

// weights of what is there and of what joins
__device__ __forceinline__ void join_weights(float& M, float m, float& a, float& b) {
  const float n = fmaxf(M, m), sub = n == -INFINITY ? 0.f : n;
  a = expf(M - sub);
  b = expf(m - sub);
  M = n;
}
__device__ __forceinline__ float joined(float L, float a, float l, float b) { return fmaf(L, a, __fmul_rn(l, b)); }

// The 16 queries of a wave: lane column r16 is head h of token t (t < 0: none).
template <int DT>
__device__ __forceinline__ void load_queries(const AttArgs& a, int t, int h, f32x4 (&qf)[DT]) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int c = 0; c < DT; ++c) {
    qf[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (t >= 0) qf[c] = *reinterpret_cast<const f32x4*>(a.q + (size_t)t * a.q_stride + (size_t)h * DT * 16 + 16 * c + 4 * g);
  }
}

template <int DT>
__global__ void __launch_bounds__(64)
portion_f32_kernel(AttArgs a, float* __restrict__ out, const int* __restrict__ row_start, const int* __restrict__ row_position,
                   int row0, int per_tile) {
  constexpr int D = DT * 16;
  const int row = row0 + blockIdx.z, begin = row_start[row], n = row_start[row + 1] - begin;
  const int rep = a.Hq / a.Hkv, head_tiles = per_tile > 1 ? 1 : (rep + 15) / 16;
  const int kvh = blockIdx.y / head_tiles, h0 = (blockIdx.y - kvh * head_tiles) * 16;
  // the last tokens see the most keys: their waves start first
  const int tile = gridDim.x - 1 - blockIdx.x;
  const int t0 = tile * per_tile;
  if (t0 >= n) return;
  const int lane = threadIdx.x, r16 = lane & 15, g = lane >> 4;
  const int ti = per_tile > 1 ? r16 / rep : 0, hi = per_tile > 1 ? r16 - ti * rep : h0 + r16;
  const bool live = hi < rep && ti < per_tile && t0 + ti < n;
  const int t = live ? begin + t0 + ti : -1, h = kvh * rep + hi;
  const int p0 = row_position[row] + t0;
  const int last = p0 + (n - t0 < per_tile ? n - t0 : per_tile) - 1;
  const int first = a.window > 0 && p0 - a.window + 1 > 0 ? p0 - a.window + 1 : 0;
  const int pos = live ? p0 + ti : -1;
  const int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
  f32x4 qf[DT], O[DT];
  load_queries<DT>(a, t, h, qf);
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int c = 0; c < DT; ++c) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int* bt = a.block_tables + (size_t)row * a.max_blocks;
  const auto first_of = [&](int p) { return a.window > 0 && p - a.window + 1 > 0 ? p - a.window + 1 : 0; };
  bool odd = false;
  auto add = [&](int seg, int qpos, int f, int e, int all_lo, int all_pos, bool mine) {
    float m, l, wa, wb;
    f32x4 o[DT];
    segment_sums<DT>(a, bt, kvh, seg, qf, qpos, lo, f, e, all_lo, all_pos, m, l, o, odd);
    if (!mine) return;
    join_weights(M, m, wa, wb);
    L = joined(L, wa, l, wb);
#pragma unroll
    for (int c = 0; c < DT; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) O[c][i] = joined(O[c][i], wa, o[c][i], wb);
  };
  for (int seg = first / AF_SEG; seg * AF_SEG <= last && !odd; ++seg) add(seg, pos, first, last, first_of(last), p0, true);
  if (odd) {
    // (values of the row's later tokens, or, beside padding tokens, of slots of its last page that nobody wrote)  All over
    // again, one token after the other: the same bits for what is a number
    M = -INFINITY;
    L = 0.f;
#pragma unroll
    for (int c = 0; c < DT; ++c) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int p = p0; p <= last; ++p) {
      const bool mine = pos == p;
      const int f = first_of(p);
#pragma unroll 1
      for (int seg = f / AF_SEG; seg * AF_SEG <= p; ++seg) add(seg, mine ? pos : -1, f, p, f, p, mine);
    }
  }
  if (!live) return;
  const float inv = 1.0f / L;
  // O[c][i] of lane (r16, g): dim 16 c + 4 g + i of the lane's query
  float* op = out + ((size_t)t * a.Hq + h) * D + 4 * g;
#pragma unroll
  for (int c = 0; c < DT; ++c) *reinterpret_cast<f32x4*>(op + 16 * c) = O[c] * inv;
}

// Single tokens: wave (split, kv head and tile of 16 heads, token).  Segment first / 128 + split of the token's keys;
// one segment only: the result itself, else (m, l) to ml [tokens, Hq, splits, 2] and O to o_part [tokens, Hq, splits, D].
template <int DT>
__global__ void __launch_bounds__(64)
single_f32_kernel(AttArgs a, float* __restrict__ out, float* __restrict__ o_part, float* __restrict__ ml,
                  const int* __restrict__ token_row, const int* __restrict__ positions, int splits) {
  constexpr int D = DT * 16;
  const int t = blockIdx.z, rep = a.Hq / a.Hkv, head_tiles = (rep + 15) / 16;
  const int kvh = blockIdx.y / head_tiles, h0 = (blockIdx.y - kvh * head_tiles) * 16;
  const int p = positions[t];
  const int first = a.window > 0 && p - a.window + 1 > 0 ? p - a.window + 1 : 0;
  const int seg = first / AF_SEG + blockIdx.x;
  if (seg * AF_SEG > p) return;
  const int lane = threadIdx.x, r16 = lane & 15, g = lane >> 4;
  const bool live = h0 + r16 < rep;
  const int h = kvh * rep + h0 + r16;
  f32x4 qf[DT], o[DT];
  load_queries<DT>(a, live ? t : -1, h, qf);
  float m, l;
  bool odd;                                   // (of no account: all queries are one token's)
  segment_sums<DT>(a, a.block_tables + (size_t)token_row[t] * a.max_blocks, kvh, seg, qf, live ? p : -1, first, first, p, first, p, m, l, o, odd);
  if (!live) return;
  if (splits == 1) {                          // joined with nothing: O 0 + o 1, L 0 + l 1
    const float inv = 1.0f / l;
    float* op = out + ((size_t)t * a.Hq + h) * D + 4 * g;
#pragma unroll
    for (int c = 0; c < DT; ++c) *reinterpret_cast<f32x4*>(op + 16 * c) = o[c] * inv;
    return;
  }
  const size_t at = ((size_t)t * a.Hq + h) * splits + blockIdx.x;
#pragma unroll
  for (int c = 0; c < DT; ++c) *reinterpret_cast<f32x4*>(o_part + at * D + 16 * c + 4 * g) = o[c];
  if (g == 0) *reinterpret_cast<float2*>(ml + 2 * at) = make_float2(m, l);
}

// Joins a token's segments in order: one wave a (token, head), lane d and d + 64 of the head.
__global__ void __launch_bounds__(64)
merge_f32_kernel(const float* __restrict__ o_part, const float* __restrict__ ml, float* __restrict__ out, const int* __restrict__ positions,
                 int Hq, int D, int window, int splits) {
  constexpr int AHEAD = 8;                    // segments whose loads are issued together
  const int t = blockIdx.y, h = blockIdx.x, lane = threadIdx.x, p = positions[t];
  const int first = window > 0 && p - window + 1 > 0 ? p - window + 1 : 0;
  const int n = p / AF_SEG - first / AF_SEG + 1;
  const size_t at = ((size_t)t * Hq + h) * splits;
  const int d0 = lane < D ? lane : 0, d1 = lane + 64 < D ? lane + 64 : 0;
  float M = -INFINITY, L = 0.f, O0 = 0.f, O1 = 0.f;
  for (int s0 = 0; s0 < n; s0 += AHEAD) {
    float2 x[AHEAD];
    float v0[AHEAD], v1[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const size_t s = at + (s0 + i < n ? s0 + i : n - 1);
      x[i] = *reinterpret_cast<const float2*>(ml + 2 * s);
      v0[i] = o_part[s * D + d0];
      v1[i] = o_part[s * D + d1];
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (s0 + i >= n) break;
      float wa, wb;
      join_weights(M, x[i].x, wa, wb);
      L = joined(L, wa, x[i].y, wb);
      O0 = joined(O0, wa, v0[i], wb);
      O1 = joined(O1, wa, v1[i], wb);
    }
  }
  const float inv = 1.0f / L;
  float* op = out + ((size_t)t * Hq + h) * D;
  if (lane < D) op[lane] = O0 * inv;
  if (lane + 64 < D) op[lane + 64] = O1 * inv;
}

MIE_EXPORT const char* attention_f32_last_error() { return g_mie_error; }
MIE_EXPORT int mie_attention_f32_segment() { return AF_SEG; }

#define AF_BY_HEAD(D_, CALL)                                                                                             \
  switch (D_) {                                                                                                          \
    case 16: CALL(1); break;                                                                                             \
    case 32: CALL(2); break;                                                                                             \
    case 48: CALL(3); break;                                                                                             \
    case 64: CALL(4); break;                                                                                             \
    case 80: CALL(5); break;                                                                                             \
    case 96: CALL(6); break;                                                                                             \
    case 112: CALL(7); break;                                                                                            \
    case 128: CALL(8); break;                                                                                            \
    default: MIE_FAIL("attention_f32: head_dim %d (multiples of 16 up to 128)", D_);                                     \
  }

static int check(const AttArgs& a, const void* out, int D) {
  if (a.Hkv <= 0 || a.Hq % a.Hkv) MIE_FAIL("attention_f32: %d query heads on %d kv heads", a.Hq, a.Hkv);
  if (a.page <= 0 || (a.page & 15) || a.max_blocks <= 0) MIE_FAIL("attention_f32: page %d (a multiple of 16), max_blocks %d", a.page, a.max_blocks);
  if (a.q_stride < (long)a.Hq * D || (a.q_stride & 3)) MIE_FAIL("attention_f32: q row stride %ld for %d columns", a.q_stride, a.Hq * D);
  if (((uintptr_t)a.q | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache | (uintptr_t)out) & 15) MIE_FAIL("attention_f32: operands must be 16-byte aligned");
  return 0;
}

// Tokens [0, tokens) of the step, each by itself (row token_row[t], position positions[t]); splits: at least the number of
// 128-key segments any of them sees; o_part and ml as above (not read or written for one split).
MIE_EXPORT int mie_attention_f32_single(const float* q, long q_stride, const float* k_cache, const float* v_cache, float* out,
                                        const int* block_tables, int max_blocks, const int* token_row, const int* positions,
                                        int tokens, int Hq, int Hkv, int D, int page, float scale, int window, int splits,
                                        float* o_part, float* ml, hipStream_t s) {
  if (tokens <= 0) return 0;
  AttArgs a = {q, q_stride, k_cache, v_cache, block_tables, max_blocks, Hq, Hkv, page, window, scale};
  if (check(a, out, D)) return -1;
  if (splits < 1 || tokens > 65535) MIE_FAIL("attention_f32: %d splits, %d tokens", splits, tokens);
  if (splits > 1 && (!o_part || !ml || (((uintptr_t)o_part | (uintptr_t)ml) & 15))) MIE_FAIL("attention_f32: memory for %d splits", splits);
  const int rep = Hq / Hkv, head_tiles = (rep + 15) / 16;
  if (Hkv * head_tiles > 65535) MIE_FAIL("attention_f32: %d kv heads are beyond the grid", Hkv);
  const dim3 grid(splits, Hkv * head_tiles, tokens);
#define AF_SINGLE(DT) hipLaunchKernelGGL(single_f32_kernel<DT>, grid, dim3(64), 0, s, a, out, o_part, ml, token_row, positions, splits)
  AF_BY_HEAD(D, AF_SINGLE)
  MIE_CHECK_LAUNCH("attention_f32 single");
  if (splits > 1) {
    hipLaunchKernelGGL(merge_f32_kernel, dim3(Hq, tokens), dim3(64), 0, s, o_part, ml, out, positions, Hq, D, window, splits);
    MIE_CHECK_LAUNCH("attention_f32 merge");
  }
  return 0;
}

// Rows [row0, rows) of the step: row r's tokens are [row_start[r], row_start[r + 1]) at positions from row_position[r] on,
// at most max_row_tokens of them; q and out start at the step's token 0.
MIE_EXPORT int mie_attention_f32_portions(const float* q, long q_stride, const float* k_cache, const float* v_cache, float* out,
                                          const int* block_tables, int max_blocks, const int* row_start, const int* row_position,
                                          int row0, int rows, int max_row_tokens, int Hq, int Hkv, int D, int page, float scale,
                                          int window, hipStream_t s) {
  if (rows <= row0 || max_row_tokens <= 0) return 0;
  AttArgs a = {q, q_stride, k_cache, v_cache, block_tables, max_blocks, Hq, Hkv, page, window, scale};
  if (check(a, out, D)) return -1;
  const int rep = Hq / Hkv, per_tile = rep <= 16 ? 16 / rep : 1, head_tiles = per_tile > 1 ? 1 : (rep + 15) / 16;
  if (Hkv * head_tiles > 65535 || rows - row0 > 65535) MIE_FAIL("attention_f32: %d kv heads, %d rows are beyond the grid", Hkv, rows - row0);
  const dim3 grid((max_row_tokens + per_tile - 1) / per_tile, Hkv * head_tiles, rows - row0);
#define AF_PORTIONS(DT) hipLaunchKernelGGL(portion_f32_kernel<DT>, grid, dim3(64), 0, s, a, out, row_start, row_position, row0, per_tile)
  AF_BY_HEAD(D, AF_PORTIONS)
  MIE_CHECK_LAUNCH("attention_f32 portions");
  return 0;
}
