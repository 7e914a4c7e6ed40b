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
// K rows and the values (transposed within their page) are used in exactly these 16-byte pieces, a page's
// 16 keys at a time.
//   portions: a wave by itself where there is little to share (alone()), else four waves side by side (neighbouring tiles of 16
//     queries) that walk their segments together.  A segment's K, then its V, come into a ring in the LDS by loads that write it directly, whole cache lines, each read once for all four waves and one to three
//     of them on their way while one is used; the 16-byte blocks of a K row are turned by the row, those of a V row by a quarter of it,
//     so that the fragment reads spread over all banks.  What bounds it: the longest workgroup's chain of segments, 3.4 us of matrix
//     instructions and 1.5 of exponentials each.  Read by every wave for itself (16 cache lines a quarter wave and load) it
//     took 41 us for 512 tokens of 32 / 4 heads of 64, now 30; 1,024 tokens 113 and 64, of 32 / 8 heads of 128 197 and 114.
//   single tokens: a wave, or four, a segment, joined by merge_f32_kernel.  What bounds it is latency: the page table, K and V, matrix
//     instructions, exponentials, one after the other.
// The kernel of attention.hip, one wave a (token, head), reads every key once a head and token, a quarter of a cache line a load: 512
// tokens of 32 / 4 heads of 64 642 us, 4 single tokens of 300 to 900 keys 200 for 11 + 5 here (MI355X).
#include "launch.hpp"

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

// The scores of a segment (lane column r16's query at position pos with keys from lo on) become exp(s - m); m and l.
__device__ __forceinline__ void segment_weights(f32x4 (&s)[AF_TILES], int base, int pos, int lo, float scale, float& m, float& l) {
  const int g = (threadIdx.x & 63) >> 4;
  float top = -INFINITY;
#pragma unroll
  for (int t = 0; t < AF_TILES; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = base + t * 16 + 4 * g + i;
      s[t][i] = key <= pos && key >= lo ? __fmul_rn(s[t][i], scale) : -INFINITY;
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
}

// A value tile's fragment c (keys key .. key + 3 of this lane): what none of the 16 queries sees becomes zero; true if what only some
// of them see is not finite.
__device__ __forceinline__ bool clean_values(f32x4& v, int key, int first, int last, int all_lo, int all_pos) {
  bool some = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = key + i >= first && key + i <= last ? v[i] : 0.f;
    some |= !(fabsf(v[i]) < INFINITY) && (key + i < all_lo || key + i > all_pos);
  }
  return some;
}

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
  segment_weights(s, base, pos, lo, a.scale, m, l);
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
        for (int c = 0; c < DT; ++c) some |= clean_values(vf[t][c], key, first, last, all_lo, all_pos);
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

// A segment's m, l and o join what the 16 queries have so far.
template <int DT>
__device__ __forceinline__ void join_segment(float& M, float& L, f32x4 (&O)[DT], float m, float l, const f32x4 (&o)[DT]) {
  float wa, wb;
  join_weights(M, m, wa, wb);
  L = joined(L, wa, l, wb);
#pragma unroll
  for (int c = 0; c < DT; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) O[c][i] = joined(O[c][i], wa, o[c][i], wb);
}

__device__ __forceinline__ int first_key(const AttArgs& a, int p) { return a.window > 0 && p - a.window + 1 > 0 ? p - a.window + 1 : 0; }

// All over again, one token after the other (values of the row's later tokens, or, beside padding tokens, of slots of its last page that
// nobody wrote, are not finite): the same bits for what is a number.  The tile's tokens are at positions p0 .. last.
template <int DT>
__device__ __forceinline__ void one_by_one(const AttArgs& a, const int* bt, int kvh, const f32x4 (&qf)[DT], int pos, int lo, int p0, int last,
                                           float& M, float& L, f32x4 (&O)[DT]) {
  M = -INFINITY;
  L = 0.f;
#pragma unroll
  for (int c = 0; c < DT; ++c) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int p = p0; p <= last; ++p) {
    const bool mine = pos == p;
    const int f = first_key(a, p);
#pragma unroll 1
    for (int seg = f / AF_SEG; seg * AF_SEG <= p; ++seg) {
      float m, l;
      f32x4 o[DT];
      bool again;                             // (of no account: all queries are one token's)
      segment_sums<DT>(a, bt, kvh, seg, qf, mine ? pos : -1, lo, f, p, f, p, m, l, o, again);
      if (mine) join_segment<DT>(M, L, O, m, l, o);
    }
  }
}

// O[c][i] of lane (r16, g): dim 16 c + 4 g + i of the lane's query, head h of token t
template <int DT>
__device__ __forceinline__ void store_result(const AttArgs& a, float* out, int t, int h, float L, const f32x4 (&O)[DT]) {
  const int g = (threadIdx.x & 63) >> 4;
  const float inv = 1.0f / L;
  float* op = out + ((size_t)t * a.Hq + h) * DT * 16 + 4 * g;
#pragma unroll
  for (int c = 0; c < DT; ++c) *reinterpret_cast<f32x4*>(op + 16 * c) = O[c] * inv;
}

// A portion by single waves: wave (tile of per_tile tokens, the last first: they see the most keys; kv head and tile of 16 heads; row) reads
// every segment for itself.  The same bits as portion_f32_kernel, for the steps that alone() names.
template <int DT>
__global__ void __launch_bounds__(64)
portion_alone_f32_kernel(AttArgs a, float* __restrict__ out, const int* __restrict__ row_start, const int* __restrict__ row_position,
                         int row0, int per_tile) {
  const int row = row0 + blockIdx.z, begin = row_start[row], n = row_start[row + 1] - begin;
  const int rep = a.Hq / a.Hkv, head_tiles = per_tile > 1 ? 1 : (rep + 15) / 16;
  const int kvh = blockIdx.y / head_tiles, h0 = (blockIdx.y - kvh * head_tiles) * 16;
  const int t0 = (gridDim.x - 1 - blockIdx.x) * per_tile;
  if (t0 >= n) return;
  const int r16 = threadIdx.x & 15;
  const int ti = per_tile > 1 ? r16 / rep : 0, hi = per_tile > 1 ? r16 - ti * rep : h0 + r16;
  const bool live = hi < rep && ti < per_tile && t0 + ti < n;
  const int t = live ? begin + t0 + ti : -1, h = kvh * rep + hi;
  const int p0 = row_position[row] + t0, last = p0 + (n - t0 < per_tile ? n - t0 : per_tile) - 1;
  const int first = first_key(a, p0), pos = live ? p0 + ti : -1, lo = first_key(a, pos);
  const int* bt = a.block_tables + (size_t)row * a.max_blocks;
  f32x4 qf[DT], O[DT];
  load_queries<DT>(a, t, h, qf);
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int c = 0; c < DT; ++c) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  bool odd = false;
  for (int seg = first / AF_SEG; seg * AF_SEG <= last && !odd; ++seg) {
    float m, l;
    f32x4 o[DT];
    segment_sums<DT>(a, bt, kvh, seg, qf, pos, lo, first, last, first_key(a, last), p0, m, l, o, odd);
    join_segment<DT>(M, L, O, m, l, o);
  }
  if (odd) one_by_one<DT>(a, bt, kvh, qf, pos, lo, p0, last, M, L, O);
  if (live) store_result<DT>(a, out, t, h, L, O);
}

// A portion's workgroup: AF_TILE_WAVES tiles of 16 queries side by side.  Up to head size 64 two waves a tile take the segments in turn, two
// at a time; the second hands m, l and O to the first, which joins all in order: 512 tokens of 32 / 4 heads of 64 35.0 us with one
// wave, 30.0 with two (33.1 with one of them at its scores while the other is at its values).  Beyond, the LDS holds no two segments
// twice.
constexpr int AF_TILE_WAVES = 4;
template <int DT> constexpr int AF_SIDES = DT <= 4 ? 2 : 1;
template <int DT> constexpr int AF_RING = DT <= 4 ? 2 : 160 / (8 * DT);      // steps: AF_SIDES segments' K or V
template <int DT> constexpr int AF_EXCHANGE = DT <= 4 ? AF_TILE_WAVES * (4 * DT + 3) * 256 : 0;
template <int DT> constexpr int AF_LDS = AF_RING<DT> * AF_SIDES<DT> * AF_SEG * DT * 64 + AF_EXCHANGE<DT>;

// Workgroup (tile of AF_TILE_WAVES * per_tile tokens, the last first; kv head and tile of 16 heads), row blockIdx.y.
template <int DT>
__global__ void __launch_bounds__(AF_TILE_WAVES * AF_SIDES<DT> * 64)
portion_f32_kernel(AttArgs a, float* __restrict__ out, const int* __restrict__ row_start, const int* __restrict__ row_position,
                   int row0, int per_tile, int tiles) {
  constexpr int D = DT * 16, BLOCKS = 4 * DT, RING = AF_RING<DT>, SIDES = AF_SIDES<DT>, BUFFER = AF_SEG * D * 4;
  constexpr int WAVES = AF_TILE_WAVES * SIDES, OWN = AF_TILES / AF_TILE_WAVES, L = OWN * DT;      // tiles of 16 keys a wave brings in a step
  static_assert((RING - 2) * L <= 63 && RING >= 2, "more loads in flight than the counter holds");
  extern __shared__ __align__(1024) char af_lds[];
  const int row = row0 + blockIdx.y, begin = row_start[row], n = row_start[row + 1] - begin;
  const int rep = a.Hq / a.Hkv, head_tiles = per_tile > 1 ? 1 : (rep + 15) / 16, heads = a.Hkv * head_tiles;
  const int tile = tiles - 1 - blockIdx.x / heads, hy = blockIdx.x % heads;
  const int kvh = hy / head_tiles, h0 = (hy - kvh * head_tiles) * 16;
  const int all_waves = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = all_waves % AF_TILE_WAVES, side = all_waves / AF_TILE_WAVES;
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int T0 = tile * AF_TILE_WAVES * per_tile;
  if (T0 >= n) return;
  const auto first_of = [&](int p) { return first_key(a, p); };
  // of the workgroup's queries, and of this wave's (none: last before first)
  const int all_last = row_position[row] + T0 + (n - T0 < AF_TILE_WAVES * per_tile ? n - T0 : AF_TILE_WAVES * per_tile) - 1;
  const int all_first = first_of(row_position[row] + T0);
  const int t0 = T0 + wave * per_tile;
  const int ti = per_tile > 1 ? r16 / rep : 0, hi = per_tile > 1 ? r16 - ti * rep : h0 + r16;
  const bool live = hi < rep && ti < per_tile && t0 + ti < n;
  const int t = live ? begin + t0 + ti : -1, h = kvh * rep + hi;
  const int p0 = row_position[row] + t0;
  const int last = t0 < n ? p0 + (n - t0 < per_tile ? n - t0 : per_tile) - 1 : -1;
  const int first = first_of(p0), pos = live ? p0 + ti : -1, lo = first_of(pos);
  f32x4 qf[DT], O[DT];
  load_queries<DT>(a, t, h, qf);
  float M = -INFINITY, L_sum = 0.f;
#pragma unroll
  for (int c = 0; c < DT; ++c) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int* bt = a.block_tables + (size_t)row * a.max_blocks;

  // The ring: step 2 i is K of the workgroup's segments SIDES i and on (a side takes one), step 2 i + 1 their V.  A wave brings in two
  // tiles of 16 keys a step.
  // K: 16-byte block b of key r at place (b + r) % BLOCKS of its row.  V: block g of dim d at (g + d / 4) % 4.
  const int seg0 = all_first / AF_SEG, segs = all_last / AF_SEG - seg0 + 1, steps = 2 * ((segs + SIDES - 1) / SIDES);
  uint32_t koff[DT];
#pragma unroll
  for (int j = 0; j < DT; ++j) {
    const int i = j * 64 + lane, r = i / BLOCKS, place = i - r * BLOCKS;
    koff[j] = r * D * 4 + ((place + BLOCKS - r % BLOCKS) % BLOCKS) * 16;
  }
  const uint32_t voff = (lane >> 2) * a.page * 4 + (((lane & 3) - (lane >> 4)) & 3) * 16;
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)af_lds;
  // pages are looked up through the scalar unit, a step ahead of their use: a vector load would come back after all that is on its way
  const auto* pages = (const __attribute__((address_space(4))) int*)(uintptr_t)bt;
  int own_page[OWN];
  auto key_of = [&](int p, int u) {           // first key of the wave's tile u in step p
    const int seg = (p >> 1) * SIDES + side, key = (seg0 + seg) * AF_SEG + (wave * OWN + u) * 16;
    // a tile nobody sees stands for a neighbour: every table entry read is one of the request's
    return key > all_last ? all_last & ~15 : key + 15 < all_first ? all_first & ~15 : key;
  };
  auto look_up = [&](int p) {
#pragma unroll
    for (int u = 0; u < OWN; ++u) own_page[u] = pages[key_of(p, u) / a.page];
  };
  auto issue = [&](int p) {
    const bool v = p & 1;
#pragma unroll
    for (int u = 0; u < OWN; ++u) {
      const int tt = wave * OWN + u, key = key_of(p, u);
      const size_t at = ((size_t)own_page[u] * a.Hkv + kvh) * a.page * D;
      const uint32_t to = lds0 + (p % RING * SIDES + side) * BUFFER + tt * 1024 * DT;
      if (v) {
        const float* vp = a.v_cache + at + key % a.page;
#pragma unroll
        for (int j = 0; j < DT; ++j) mie_load_to_lds(vp + (size_t)(16 * j) * a.page, voff, to + j * 1024);
      } else {
        const float* kp = a.k_cache + at + (size_t)(key % a.page) * D;
#pragma unroll
        for (int j = 0; j < DT; ++j) mie_load_to_lds(kp, koff[j], to + j * 1024);
      }
    }
  };
  look_up(0);
  issue(0);
#pragma unroll
  for (int c = 0; c < DT; ++c) asm volatile("" : "+v"(qf[c]));      // the queries are waited for here, with the first K alone on its way
#pragma unroll
  for (int p = 1; p < RING - 1; ++p)
    if (p < steps) {
      look_up(p);
      issue(p);
    }
  look_up(RING - 1);

  int kat[DT];                                // of this lane's fragments: K block 4 c + g of key r16, V block g of dim r16
#pragma unroll
  for (int c = 0; c < DT; ++c) kat[c] = r16 * D * 4 + ((4 * c + g + r16) % BLOCKS) * 16;
  const int vat = r16 * 64 + ((g + (r16 >> 2)) & 3) * 16;
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  f32x4 s[AF_TILES];
  float m = 0.f, l = 0.f;
  bool odd = false;
  // what the other side made of its segment, a barrier after it did: the next time it writes is two barriers on
  float* exchange = reinterpret_cast<float*>(af_lds + RING * SIDES * BUFFER) + wave * (4 * DT + 3) * 64 + lane;
  auto join_other = [&](int seg) {
    const int base = (seg0 + seg) * AF_SEG;
    if (base > last || base + AF_SEG <= first) return;
    f32x4 o[DT];
#pragma unroll
    for (int c = 0; c < DT; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[c][i] = exchange[(4 * c + i) * 64];
    odd |= exchange[(4 * DT + 2) * 64] != 0.f;
    join_segment<DT>(M, L_sum, O, exchange[4 * DT * 64], exchange[(4 * DT + 1) * 64], o);
  };
  for (int p = 0; p < steps; ++p) {
    if (p + RING - 1 <= steps) MIE_VMCNT((RING - 2) * L);
    else MIE_VMCNT(0);
    __builtin_amdgcn_s_barrier();             // step p is in the LDS; everybody is done with step p - 1
    asm volatile("" ::: "memory");
    if (p + RING - 1 < steps) {
      issue(p + RING - 1);
      look_up(p + RING);
    }
    const bool values = p & 1;
    const int seg = (p >> 1) * SIDES + side, base = (seg0 + seg) * AF_SEG;
    if (SIDES == 2 && !side && !values && p) join_other(seg - 1);
    const char* buf = af_lds + (p % RING * SIDES + side) * BUFFER;
    const bool sees = base <= last && base + AF_SEG > first;
    if (sees && !values) {
#pragma unroll
      for (int u = 0; u < AF_TILES; u += 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) s[u + k] = none;
#pragma unroll
        for (int c = 0; c < DT; ++c) {
          f32x4 kf[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) kf[k] = *reinterpret_cast<const f32x4*>(buf + (u + k) * 1024 * DT + kat[c]);
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) s[u + k] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[k][j], qf[c][j], s[u + k], 0, 0, 0);
        }
      }
      segment_weights(s, base, pos, lo, a.scale, m, l);
    }
    if (sees && values) {
      f32x4 o[DT];
      bool some = false;
#pragma unroll
      for (int c = 0; c < DT; ++c) o[c] = none;
#pragma unroll
      for (int u = 0; u < AF_TILES; ++u) {
        f32x4 vf[DT];
#pragma unroll
        for (int c = 0; c < DT; ++c) vf[c] = *reinterpret_cast<const f32x4*>(buf + u * 1024 * DT + c * 1024 + vat);
        const int key = base + u * 16;
        if (key < first_of(last) || key + 15 > p0) {
#pragma unroll
          for (int c = 0; c < DT; ++c) some |= clean_values(vf[c], key + 4 * g, first, last, first_of(last), p0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < DT; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[c][i], s[u][i], o[c], 0, 0, 0);
      }
      const bool bad = __builtin_amdgcn_ballot_w64(some) != 0;
      if (SIDES == 2 && side) {
#pragma unroll
        for (int c = 0; c < DT; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) exchange[(4 * c + i) * 64] = o[c][i];
        exchange[4 * DT * 64] = m;
        exchange[(4 * DT + 1) * 64] = l;
        exchange[(4 * DT + 2) * 64] = bad ? 1.f : 0.f;
      } else {
        odd |= bad;
        join_segment<DT>(M, L_sum, O, m, l, o);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // this wave has read the buffer before the next barrier
  }
  if (SIDES == 2) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (side) return;
    join_other(steps - 1);                    // (the pair's second segment; not there: seen by nobody)
  }
  if (odd) one_by_one<DT>(a, bt, kvh, qf, pos, lo, p0, last, M, L_sum, O);
  if (live) store_result<DT>(a, out, t, h, L_sum, O);
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

// The same by four waves, without another order of any sum: a wave makes the scores and exponentials of two of the eight tiles of 16
// keys, all of them meet in the LDS, every wave adds them up as one wave would, and a wave takes every fourth tile of 16 dims of the
// values.  4 tokens of 300 to 900 keys of 32 / 4 heads of 64 13.6 us with one wave and the kernel that joins, 10.0 with four; where the
// segments are many, one wave each has less to exchange (64 tokens of 2,000 keys of 4 / 2 heads of 16: 15.2 and 20.9; 16 of 900
// of 32 / 8 heads of 128: 34.6 and 37.4): four_waves() draws the line.
constexpr int AF_SINGLE_WAVES = 4;
template <int DT>
__global__ void __launch_bounds__(AF_SINGLE_WAVES * 64)
single_few_f32_kernel(AttArgs a, float* __restrict__ out, float* __restrict__ o_part, float* __restrict__ ml,
                  const int* __restrict__ token_row, const int* __restrict__ positions, int splits) {
  constexpr int D = DT * 16, OWN = AF_TILES / AF_SINGLE_WAVES, CT = (DT + AF_SINGLE_WAVES - 1) / AF_SINGLE_WAVES;
  __shared__ __align__(16) float weights[AF_TILES * 64 * 4];
  __shared__ float s_top[AF_SINGLE_WAVES][16];
  const int t = blockIdx.z, rep = a.Hq / a.Hkv, head_tiles = (rep + 15) / 16;
  const int kvh = blockIdx.y / head_tiles, h0 = (blockIdx.y - kvh * head_tiles) * 16;
  const int p = positions[t];
  const int first = a.window > 0 && p - a.window + 1 > 0 ? p - a.window + 1 : 0;
  const int seg = first / AF_SEG + blockIdx.x;
  if (seg * AF_SEG > p) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const bool live = h0 + r16 < rep;
  const int h = kvh * rep + h0 + r16, base = seg * AF_SEG;
  const int* bt = a.block_tables + (size_t)token_row[t] * a.max_blocks;
  f32x4 qf[DT];
  load_queries<DT>(a, live ? t : -1, h, qf);
  size_t at[AF_TILES];                        // of the page stretch a tile of 16 keys lies in; a tile nobody sees stands for its neighbour
  const int t0 = first > base ? (first - base) >> 4 : 0, t1 = p - base >= AF_SEG ? AF_TILES : ((p - base) >> 4) + 1;
#pragma unroll
  for (int u = 0; u < AF_TILES; ++u) {
    const int tt = u < t0 ? t0 : u >= t1 ? t1 - 1 : u;
    at[u] = ((size_t)bt[(base + tt * 16) / a.page] * a.Hkv + kvh) * a.page * D;
  }
  f32x4 kf[OWN][DT], vf[AF_TILES][CT], s[OWN];
#pragma unroll
  for (int u = 0; u < OWN; ++u) {
    const int tile = wave * OWN + u;
    size_t from = at[0];
#pragma unroll
    for (int k = 1; k < AF_TILES; ++k) from = tile == k ? at[k] : from;
    const float* kp = a.k_cache + from + (size_t)((base + tile * 16) % a.page + r16) * D + 4 * g;
#pragma unroll
    for (int c = 0; c < DT; ++c) kf[u][c] = *reinterpret_cast<const f32x4*>(kp + 16 * c);
  }
#pragma unroll
  for (int u = 0; u < AF_TILES; ++u) {
    const float* vp = a.v_cache + at[u] + (size_t)r16 * a.page + (base + u * 16) % a.page + 4 * g;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int c = wave + j * AF_SINGLE_WAVES;
      vf[u][j] = *reinterpret_cast<const f32x4*>(vp + (size_t)(16 * (c < DT ? c : 0)) * a.page);
    }
  }
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < OWN; ++u) s[u] = none;
#pragma unroll
  for (int c = 0; c < DT; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < OWN; ++u) s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u][c][j], qf[c][j], s[u], 0, 0, 0);
  const int pos = live ? p : -1;
  float top = -INFINITY;
#pragma unroll
  for (int u = 0; u < OWN; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = base + (wave * OWN + u) * 16 + 4 * g + i;
      s[u][i] = key <= pos && key >= first ? __fmul_rn(s[u][i], a.scale) : -INFINITY;
      top = fmaxf(top, s[u][i]);
    }
  top = fmaxf(top, __shfl_xor(top, 16, 64));
  top = fmaxf(top, __shfl_xor(top, 32, 64));
  if (g == 0) s_top[wave][r16] = top;
  __syncthreads();
  float m = s_top[0][r16];
#pragma unroll
  for (int w = 1; w < AF_SINGLE_WAVES; ++w) m = fmaxf(m, s_top[w][r16]);
  const float sub = m == -INFINITY ? 0.f : m;
#pragma unroll
  for (int u = 0; u < OWN; ++u) {
#pragma unroll
    for (int i = 0; i < 4; ++i) s[u][i] = expf(s[u][i] - sub);
    *reinterpret_cast<f32x4*>(weights + ((wave * OWN + u) * 64 + lane) * 4) = s[u];
  }
  __syncthreads();
  f32x4 o[CT], e[AF_TILES];
#pragma unroll
  for (int u = 0; u < AF_TILES; ++u) e[u] = *reinterpret_cast<const f32x4*>(weights + (u * 64 + lane) * 4);
  float l = 0.f;
#pragma unroll
  for (int u = 0; u < AF_TILES; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) l += e[u][i];
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
#pragma unroll
  for (int j = 0; j < CT; ++j) o[j] = none;
#pragma unroll
  for (int u = 0; u < AF_TILES; ++u) {
    const int key = base + u * 16;
    if (key < first || key + 15 > p) {
#pragma unroll
      for (int j = 0; j < CT; ++j) clean_values(vf[u][j], key + 4 * g, first, p, first, p);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[u][j][i], e[u][i], o[j], 0, 0, 0);
  }
  if (!live) return;
  const size_t part = ((size_t)t * a.Hq + h) * splits + blockIdx.x;
  const float inv = 1.0f / l;                 // one segment, joined with nothing: O 0 + o 1, L 0 + l 1
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    const int c = wave + j * AF_SINGLE_WAVES;
    if (c >= DT) break;
    if (splits == 1) *reinterpret_cast<f32x4*>(out + ((size_t)t * a.Hq + h) * D + 16 * c + 4 * g) = o[j] * inv;
    else *reinterpret_cast<f32x4*>(o_part + part * D + 16 * c + 4 * g) = o[j];
  }
  if (splits > 1 && wave == 0 && g == 0) *reinterpret_cast<float2*>(ml + 2 * part) = make_float2(m, l);
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

// Whether a segment of single tokens is four waves' work: while the segments are at most so many a compute unit.  The waves take tiles of
// 16 dims in fours, so the fewer a head has, and 80 and 96 that take eight for five or six, the sooner one wave each is the better; and
// the sooner where tokens have one segment, often a short one.  Four waves / one, at 1, 2, 3 and 4 segments a compute unit (MI355X, 80
// shapes a head size; in brackets of one segment): 16 0.86, 1.01, 1.15, 1.29; 32 0.80, 0.91, 1.02, 1.09; 48 0.74, 0.86, 0.95, 1.01 (1.05); 64
// 0.71, 0.82, 0.92, 0.97; 80 0.69, 0.86, 0.98 (1.01), 1.06; 96 0.67, 0.85, 0.99 (1.01), 1.05; 112 0.61, 0.78, 0.91, 0.98; 128 0.61, 0.80, 0.93, 0.99.
static bool four_waves(int tokens, int Hq, int Hkv, int D, int splits) {
  constexpr int most[2][8] = {{1, 2, 4, 4, 3, 3, 4, 4}, {1, 2, 3, 4, 2, 2, 4, 4}};      // of head size 16, 32, ...; the second: one segment
  if (D < 16 || D > 128) return false;
  return (long)splits * Hkv * ((Hq / Hkv + 15) / 16) * tokens <= (long)most[splits == 1][D / 16 - 1] * mie_compute_units();
}
MIE_EXPORT int mie_attention_f32_four_waves(int tokens, int Hq, int Hkv, int D, int splits) {
  return Hkv > 0 && Hq >= Hkv && four_waves(tokens, Hq, Hkv, D, splits);
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
  const bool few = four_waves(tokens, Hq, Hkv, D, splits);
#define AF_SINGLE(DT)                                                                                                                      \
  if (few) hipLaunchKernelGGL(single_few_f32_kernel<DT>, grid, dim3(AF_SINGLE_WAVES * 64), 0, s, a, out, o_part, ml, token_row, positions, splits); \
  else hipLaunchKernelGGL(single_f32_kernel<DT>, grid, dim3(64), 0, s, a, out, o_part, ml, token_row, positions, splits)
  AF_BY_HEAD(D, AF_SINGLE)
  MIE_CHECK_LAUNCH("attention_f32 single");
  if (splits > 1) {
    hipLaunchKernelGGL(merge_f32_kernel, dim3(Hq, tokens), dim3(64), 0, s, o_part, ml, out, positions, Hq, D, window, splits);
    MIE_CHECK_LAUNCH("attention_f32 merge");
  }
  return 0;
}

// Whether portions of up to max_row_tokens tokens go to single waves, not to workgroups of AF_TILE_WAVES tiles (max_context: of the longest
// row, 0: not known).  A page's offsets take more than 32 bits; or
//  - one segment at most, so that no sides take turns, and two waves a compute unit or small heads: a workgroup's start costs more than the
//    shared loads save.  Four / one wave, us: 64 tokens of 32 / 4 heads of 64 13.4 / 12.2, of 4 / 2 of 16 8.5 / 7.4, 100 of
//    32 / 8 of 128 19.4 / 18.8, but four rows of 100 of 32 / 4 of 64 (800 waves) 14.3 / 15.4;
//  - more workgroups than compute units, whose waves are not all of them needed (rows of few tiles): 64 rows of 8 tokens of 12 / 12
//    heads of 64 (one tile a workgroup) 34.5 / 14.0, of 32 / 8 of 128 (two) 37.1 / 24.1; 16 of 75 of 12 / 12 of 64 (two and a half)
//    26.0 / 16.4; behind 700 keys (one) 119.9 / 71.5.  Of three tiles a workgroup, 192 rows of 32 / 4 heads of 64: one segment
//    39.2 / 40.4, 700 keys 1.47 times as long by one wave;
//  - more workgroups than compute units and little work in each: heads of 16 from two and a half workgroups a compute unit on (8 rows of
//    250 of 40 / 2 heads 59.5 / 43.2, 3,000 tokens 453 / 368; 588 workgroups of 978 keys 0.89 of one wave, 720 of 476 1.02); of 48 and
//    80, whose LDS leaves a compute unit one workgroup and most of it idle, up to two segments (64 rows of 43 of 40 / 2 of 48
//    112 / 71, of 30 of 16 / 2 of 80 29.5 / 25.3, 8 rows of 250 44.7 / 40.3, and more than that on average not).
// Over 700 steps drawn at random 0.93 of four waves everywhere and 0.94 of one, within 0.2 % of the better one of each; up to 1.12 of one
// is left (heads of 80 behind thousands of keys).
static bool alone(int rows, int max_row_tokens, int Hq, int Hkv, int D, int page, int max_context) {
  if (page > 1 << 24) return true;
  const int rep = Hq / Hkv, per_tile = rep <= 16 ? 16 / rep : 1;
  const long heads = (long)Hkv * (rep <= 16 ? 1 : (rep + 15) / 16), cu = mie_compute_units();
  const long tiles = ((long)max_row_tokens + per_tile - 1) / per_tile, groups = (tiles + AF_TILE_WAVES - 1) / AF_TILE_WAVES;
  const long workgroups = groups * heads * rows;
  const bool one_segment = max_context > 0 && max_context <= AF_SEG, two_segments = max_context > 0 && max_context <= 2 * AF_SEG;
  if (one_segment && (D <= 32 || tiles * heads * rows <= 2 * cu)) return true;
  if (workgroups <= cu) return false;
  if (D == 16 && 2 * workgroups > 5 * cu) return true;
  if ((D == 48 || D == 80) && two_segments) return true;
  const int twice = D <= 32 ? 6 : workgroups <= 2 * cu ? (one_segment ? 5 : 4) : one_segment ? 6 : 5;      // twice the tiles a workgroup up to which
  return 2 * tiles <= twice * groups;
}
MIE_EXPORT int mie_attention_f32_alone(int rows, int max_row_tokens, int Hq, int Hkv, int D, int page, int max_context) {
  return Hkv > 0 && Hq >= Hkv && alone(rows, max_row_tokens, Hq, Hkv, D, page, max_context);
}

// Rows [row0, rows) of the step: row r's tokens are [row_start[r], row_start[r + 1]) at positions from row_position[r] on,
// at most max_row_tokens of them; q and out start at the step's token 0.  max_context: no token is at a position beyond it, or 0.
MIE_EXPORT int mie_attention_f32_portions(const float* q, long q_stride, const float* k_cache, const float* v_cache, float* out,
                                          const int* block_tables, int max_blocks, const int* row_start, const int* row_position,
                                          int row0, int rows, int max_row_tokens, int Hq, int Hkv, int D, int page, float scale,
                                          int window, int max_context, hipStream_t s) {
  if (rows <= row0 || max_row_tokens <= 0) return 0;
  AttArgs a = {q, q_stride, k_cache, v_cache, block_tables, max_blocks, Hq, Hkv, page, window, scale};
  if (check(a, out, D)) return -1;
  const int rep = Hq / Hkv, per_tile = rep <= 16 ? 16 / rep : 1, head_tiles = per_tile > 1 ? 1 : (rep + 15) / 16;
  if (Hkv * head_tiles > 65535 || rows - row0 > 65535) MIE_FAIL("attention_f32: %d kv heads, %d rows are beyond the grid", Hkv, rows - row0);
  const int tiles = (max_row_tokens + AF_TILE_WAVES * per_tile - 1) / (AF_TILE_WAVES * per_tile);
  if ((long)tiles * Hkv * head_tiles > 0x7FFFFFFF) MIE_FAIL("attention_f32: %d tokens are beyond the grid", max_row_tokens);
  if (alone(rows - row0, max_row_tokens, Hq, Hkv, D, page, max_context)) {
    const dim3 waves((max_row_tokens + per_tile - 1) / per_tile, Hkv * head_tiles, rows - row0);
#define AF_ALONE(DT) hipLaunchKernelGGL(portion_alone_f32_kernel<DT>, waves, dim3(64), 0, s, a, out, row_start, row_position, row0, per_tile)
    AF_BY_HEAD(D, AF_ALONE)
    MIE_CHECK_LAUNCH("attention_f32 portions");
    return 0;
  }
  const dim3 grid(tiles * Hkv * head_tiles, rows - row0);
#define AF_PORTIONS(DT)                                                                                                              \
  {                                                                                                                                  \
    if (mie_allow_lds((const void*)portion_f32_kernel<DT>, AF_LDS<DT>, "attention_f32")) return -1;                                  \
    hipLaunchKernelGGL(portion_f32_kernel<DT>, grid, dim3(AF_TILE_WAVES * AF_SIDES<DT> * 64), AF_LDS<DT>, s, a, out, row_start,      \
                       row_position, row0, per_tile, tiles);                                                                         \
  }
  AF_BY_HEAD(D, AF_PORTIONS)
  MIE_CHECK_LAUNCH("attention_f32 portions");
  return 0;
}
