// Matrix products of the bfloat16 path with few rows (M <= 16: decode steps, the head on wanted rows),
// where the weights are streamed once from HBM and everything else is noise: one kernel per product,
// with what comes after it folded in, because at these sizes a launch costs as much as the work.
//
//   y[m, n] = sum_k x[m, k] W[n, k]          x [M, K], W [N, K] bfloat16 as stored in a checkpoint
//
// A workgroup of 4 waves owns one to three tiles of 16 rows of W (tiles of C^T = W X^T); each wave streams one contiguous
// quarter of K in chunks of 64; v_mfma_f32_16x16x32_bf16 with A = 16 weight rows x 32 k and B = 32 k x 16
// batch rows; the waves' accumulators are summed through LDS in a fixed order.  A row's result depends on
// nothing but that row, K and the weights: it is bit-identical in any batch.
//
// How the operands reach the matrix instruction.  The instruction wants lane 16 b + r to hold k-block b (8
// values, 16 bytes) of row r.  Loaded in that order, a quarter wave (16 lanes) touches 16 cache lines for 16
// bytes each, and the address unit, which looks lines up one at a time, is then what bounds the kernel.  So a load takes whole
// cache lines, 8 rows of 64 k (lane 8 r + b), and writes the wave's own piece of the LDS directly (no registers, nothing the
// compiler waits for): slots of one chunk.  A slot's fragments are read, the chunk SLOTS further on is asked for into the same
// slot at once, and then they are multiplied.  Within a row the eight blocks are permuted (block b at 16-byte place
// 8 r + (b ^ r % 8)), so that the fragment reads (lane 16 b + r) are spread over all banks.  No barrier in the loop: a wave
// reads only what it brought in itself.  Up to 8 rows bring in half as much x.
// Loads are what these kernels spend their time on (58 bytes a nanosecond and compute unit with their address arithmetic; whole lines
// come in at 75 to 97 where an address is one addition, see tile_gemm_bf16.hip), so none is made for nothing: nothing behind a wave's
// quarter is asked for (three slots of zeros a wave were, a quarter of all loads at K = 2,048), and tiles share a workgroup's x.
// Measured alone (MI355X, us, 1 / 8 / 16 rows, before and now): [2048, 2048] 4.5 / 4.7 / 5.1 and 4.1 / 4.5 / 4.9, [2048, 5632] 7.8 /
// 8.2 / 9.7 and 7.0 / 7.9 / 9.6, [11264, 2048] 10.2 / 10.2 / 11.1 and 9.6 / 9.7 / 9.9, [32000, 2048] 24.9 / 25.1 / 27.2 and 21.7 / 21.3 /
// 22.1, [6144, 4096] 11.4 / 12.6 / 14.4 and 10.8 / 11.2 / 12.3, [28672, 4096] 38.9 / 40.3 / 42.0 and 37.4 / 37.9 / 39.3.
// With the norm in front fused in, as the engine runs them: [11264, 2048] 10.0 / 10.7 / 10.9, [32000, 2048] 23.3 / 24.5 / 26.5, [6144, 4096]
// 11.7 / 12.5 / 14.4, [28672, 4096] 38.0 / 40.8 / 45.4.
//
// Epilogues: STORE (bfloat16 or float32 y), ADD (r[m, n] += y, the residual add of the 32-bit stream),
//   SWIGLU (W holds gate rows then up rows; a tile is 8 gate rows and the matching 8 up rows, and the
//   workgroup writes silu(gate) * up for them).
//   ROPE (the q/k/v projection: rotary on q and k, cache write of k and v).
// The RMSNorm between two products is folded into them as well, see NormArgs below.  (A norm prologue that
// converted the 32-bit stream inside every workgroup was measured and dropped: redoing the conversion of
// all of x per workgroup cost more than a separate norm kernel.)
#include "launch.hpp"
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int SG_WAVES = 4;       // waves a workgroup
constexpr int SG_THREADS = SG_WAVES * 64;

enum { EPI_STORE_BF16 = 0, EPI_STORE_F32 = 1, EPI_ADD = 2, EPI_SWIGLU = 3, EPI_ROPE = 4, EPI_GEGLU = 5, EPI_CLAMPGLU = 6 };
// the gated epilogues differ in the function only: silu(g) u (SWIGLU), the tanh form of gelu(g) u (GEGLU), or, with g at most
// a limit and u within plus and minus that limit, g sigmoid(alpha g) (u + shift) (CLAMPGLU)
#define EPI_GATED(E) ((E) == EPI_SWIGLU || (E) == EPI_GEGLU || (E) == EPI_CLAMPGLU)

// What the rotary epilogue needs beside the product: W is the fused q/k/v projection; the workgroup owns
// columns j0 .. j0 + 7 and j0 + D/2 .. j0 + D/2 + 7 of one head, i.e. 8 rotary pairs.
struct RopeArgs {
  const int* positions;      // [M]
  const float* cos_t;        // [positions, D / 2]
  const float* sin_t;
  const int* slots;          // [M] cache slot of each row's token
  bf16* k_cache;             // [pages, Hkv, page, D]
  bf16* v_cache;             // [pages, Hkv, D, page]
  int Hq, Hkv, D, page;
};

// The RMSNorm between two of these products, without a kernel of its own (NF).  The product that adds
// into the stream (ADD) also writes, for the norm that follows it with weight g, x_next[m, n] =
// bf16(r[m, n] g[n]) and the sum of r[m, n]^2 over its 16 columns (ss_out [M, tiles]); the product that
// consumes the normed value takes x_next as its X, sums ss_in over the tiles and scales its results by
// rstd[m] = 1 / sqrt(sum / width + eps): rstd is a positive scalar per row, so applying it after the
// product, to values rounded before it, is the same relative rounding as rounding the normed value.
struct NormArgs {
  const void* g;             // ADD: weight of the next norm [N]
  int g_f32;
  bf16* x_next;              // ADD: [M, ldx_next]
  long ldx_next;
  float* ss_out;             // ADD: [M, tiles of this product rounded up to a multiple of 4]
  const float* ss_in;        // others: [rows, ss_tiles rounded up to a multiple of 4], indexed by source row
  int ss_tiles;
  float inv_width, eps;
  const int* rows;           // others: optional gather of X's (and ss_in's) rows, int32 [M]
  float glu_limit, glu_alpha, glu_shift;     // CLAMPGLU's constants (with or without a fused norm)
};

// Which weight row column c (0 .. 15) of tile `tile` multiplies, and whether it exists.
//   plain:  n = 16 tile + c
//   gated:  columns 0 .. 7 are gate rows j = 8 tile + c, columns 8 .. 15 the up rows of the same j
//   ROPE:   columns 0 .. 7 are the first members jd = 8 (tile % (D / 16)) + c of eight rotary pairs of head
//           tile / (D / 16), columns 8 .. 15 their partners jd + D / 2
// so that both members of a pair are lanes c and c ^ 8 of one wave after the reduction.  tile_row: the row of column 0 (h = 0) or
// 8 (h = 1), `rows` the rows that exist from there on (may be none or negative).
template <int EPI>
__device__ __forceinline__ long tile_row(int tile, int h, int N, int up_offset, int D, int& rows) {
  if (EPI_GATED(EPI)) {
    rows = N - tile * 8;
    return (long)h * up_offset + tile * 8;
  }
  if (EPI == EPI_ROPE) {
    const int per_head = D >> 4, head = tile / per_head, jd = (tile - head * per_head) * 8;
    rows = head * D < N ? 8 : 0;
    return (long)head * D + jd + h * (D >> 1);
  }
  rows = N - (tile * 16 + h * 8);
  return (long)tile * 16 + h * 8;
}

// XT: groups of 8 x rows: one for up to 8 (columns 8 to 15 of the tile then take rows 0 to 7 again), else two.
// TW: tiles a workgroup, `tiles` of them in all.
template <int EPI, bool NF, int TW, int XT, int SLOTS>
__global__ void __launch_bounds__(SG_THREADS)
skinny_gemm_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw, void* __restrict__ outv,
                   long ldo, int M, int N, int K, int up_offset, int tiles, RopeArgs rope, NormArgs nf) {
  constexpr int L = 2 * TW + XT, SLOT = L * 1024;          // of a slot: TW times 16 weight rows of 64 k (128 bytes), then the x rows
  static_assert((SLOTS - 1) * L <= 63, "more loads in flight than the counter holds");
  extern __shared__ __align__(1024) char ring_lds[];       // SLOTS slots a wave
  __shared__ float s_acc[TW][SG_WAVES][256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  const int tile0 = blockIdx.x * TW;
  const int all = (K + 63) >> 6, own = (all + SG_WAVES - 1) / SG_WAVES;
  const int c0 = wave * own, chunks = all - c0 < own ? all - c0 : own;         // (none: negative or 0)

  // What this lane brings in: row lrow of each group of 8, block lblk of every 64 k.  And the results this thread owns after the
  // waves are summed: x row m, column c of every tile.
  const int lrow = lane >> 3, lblk = (lane & 7) ^ lrow;
  const int m = threadIdx.x >> 4, c = threadIdx.x & 15;
  const bool gather = NF && EPI != EPI_ADD && nf.rows;
  uint32_t xoff[XT];
#pragma unroll
  for (int t = 0; t < XT; ++t) {
    const int r = t * 8 + lrow < M ? t * 8 + lrow : 0;     // rows beyond M read another row along with the lanes that own it
    xoff[t] = (uint32_t)((long)(gather ? nf.rows[r] : r) * ldx * 2) + lblk * 16;
  }
  const int msrc = m < M ? (gather ? nf.rows[m] : m) : 0;
  const char* wbase[TW][2];
  uint32_t woff[TW][2];
  long n_of[TW];
  bool live[TW];
#pragma unroll
  for (int a = 0; a < TW; ++a) {
    const int tile = tile0 + a < tiles ? tile0 + a : tiles - 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int rows;
      const long row = tile_row<EPI>(tile, h, N, up_offset, rope.D, rows);
      // a row that does not exist is never stored: the tile's last one that does (or the weight's first) is read instead
      wbase[a][h] = reinterpret_cast<const char*>(W + (size_t)(rows > 0 ? row : 0) * ldw);
      woff[a][h] = (uint32_t)((long)(rows > 0 ? (lrow < rows ? lrow : rows - 1) : 0) * ldw * 2) + lblk * 16;
      if (h == c >> 3) {
        n_of[a] = row + (c & 7);
        live[a] = tile0 + a < tiles && m < M && (c & 7) < rows;
      }
    }
  }

  // What the epilogue reads beside the product is asked for before the ring, so that it has arrived long before it is used and a
  // wait for it is no wait for the ring.  Every load is unconditional, from an address clamped into the operand.
  float e_old[TW] = {}, e_cos[TW] = {}, e_sin[TW] = {};
  uint32_t e_g[TW] = {};                   // raw bits of the next norm's weight (converted where it is used)
  int e_slot = 0;
  if (EPI == EPI_ROPE) {                   // positions and slots of the wave's four rows by scalar loads, and the angles
    int pos[4], slot[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = wave * 4 + i < M ? wave * 4 + i : 0;
      pos[i] = rope.positions[r];
      slot[i] = rope.slots[r];
    }
    const int i = lane >> 4, e_pos = i == 0 ? pos[0] : i == 1 ? pos[1] : i == 2 ? pos[2] : pos[3];
    e_slot = i == 0 ? slot[0] : i == 1 ? slot[1] : i == 2 ? slot[2] : slot[3];
    const int half = rope.D >> 1, per_head = rope.D >> 4;
#pragma unroll
    for (int a = 0; a < TW; ++a) {
      const int jd = ((tile0 + a) % per_head) * 8 + (c & 7);
      e_cos[a] = rope.cos_t[(size_t)e_pos * half + jd];
      e_sin[a] = rope.sin_t[(size_t)e_pos * half + jd];
    }
  }
  if (EPI == EPI_ADD) {
#pragma unroll
    for (int a = 0; a < TW; ++a) {
      const long nc = live[a] ? n_of[a] : 0;
      e_old[a] = ((const float*)outv)[(size_t)(live[a] ? m : 0) * ldo + nc];
      if (NF) e_g[a] = nf.g_f32 ? ((const uint32_t*)nf.g)[nc] : (uint32_t)((const uint16_t*)nf.g)[nc];
    }
  }
  // Fused norm, consuming side: the partial sums of squares.  16 lanes a row, lane c takes the
  // tiles 4 (c + 16 i) .. + 3: the first SSP fours now, the rest (widths above 4096) after the loop.
  constexpr int SSP = 4;
  f32x4 ssp[SSP];
  const int ss_ld = (nf.ss_tiles + 3) & ~3;
  if (NF && EPI != EPI_ADD) {
#pragma unroll
    for (int i = 0; i < SSP; ++i) {
      const int t = 4 * (c + 16 * i);
      ssp[i] = *reinterpret_cast<const f32x4*>(nf.ss_in + (size_t)msrc * ss_ld + (t < ss_ld ? t : 0));
    }
  }

  const char* xb = reinterpret_cast<const char*>(X);
  const uint32_t mine = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)ring_lds + wave * SLOTS * SLOT;
  auto issue = [&](int s) {
    const size_t k = (size_t)(c0 + s) * 128;
    const uint32_t base = mine + (s % SLOTS) * SLOT;
    // blocks beyond K are read as the chunk's first block, and are zeros by the time they are multiplied
    const uint32_t back = (c0 + s) * 64 + lblk * 8 >= K ? lblk * 16 : 0;
#pragma unroll
    for (int a = 0; a < TW; ++a)
#pragma unroll
      for (int h = 0; h < 2; ++h) mie_load_to_lds_nt(wbase[a][h] + k, woff[a][h] - back, base + (2 * a + h) * 1024);
#pragma unroll
    for (int t = 0; t < XT; ++t) mie_load_to_lds(xb + k, xoff[t] - back, base + (2 * TW + t) * 1024);
  };
  f32x4 acc[TW];
#pragma unroll
  for (int a = 0; a < TW; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SLOTS; ++s)
    if (s < chunks) issue(s);
  bf16x8 wf[2][TW], xf[2];
  auto take = [&](int it) {                                // this lane's fragments of chunk `it`
    const char* at = ring_lds + (wave * SLOTS + it % SLOTS) * SLOT;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int blk = ((4 * u + kb) ^ (col & 7)) * 16;
#pragma unroll
      for (int a = 0; a < TW; ++a) wf[u][a] = *reinterpret_cast<const bf16x8*>(at + a * 2048 + col * 128 + blk);
      xf[u] = *reinterpret_cast<const bf16x8*>(at + TW * 2048 + (XT == 1 ? col & 7 : col) * 128 + blk);
    }
  };
  auto multiply = [&]() {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int a = 0; a < TW; ++a) acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][a], xf[u], acc[a], 0, 0, 0);
  };
  int it = 0;
  for (; it + SLOTS < chunks; ++it) {
    MIE_VMCNT((SLOTS - 1) * L);                            // chunk `it` has landed: at most those after it are on their way
    asm volatile("" ::: "memory");
    take(it);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // read: the slot is free
    issue(it + SLOTS);
    multiply();
  }
  // the last chunks, nothing behind them
  auto last = [&](auto left) {
    constexpr int LEFT = decltype(left)::value;            // chunks behind this one
    if (LEFT >= SLOTS || LEFT >= chunks) return;
    MIE_VMCNT(LEFT < SLOTS ? LEFT * L : 0);
    asm volatile("" ::: "memory");
    take(it++);
    if (LEFT == 0 && c0 + chunks == all && (K & 63)) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if ((all - 1) * 64 + (4 * u + kb) * 8 >= K) {
          xf[u] = __builtin_bit_cast(bf16x8, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int a = 0; a < TW; ++a) wf[u][a] = xf[u];
        }
    }
    multiply();
  };
  static_assert(SLOTS <= 5, "the calls below");
  last(std::integral_constant<int, 4>());
  last(std::integral_constant<int, 3>());
  last(std::integral_constant<int, 2>());
  last(std::integral_constant<int, 1>());
  last(std::integral_constant<int, 0>());

  float rstd = 1.f;
  if (NF && EPI != EPI_ADD) {
    // 1 / sqrt(mean of squares + eps) of this thread's row, summed in a fixed order by the row's 16 lanes
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < SSP; ++i) {
      asm volatile("" : "+v"(ssp[i]));                     // (not added up, and so not waited for, before the loop)
      const int t = 4 * (c + 16 * i);
      sum += (t < nf.ss_tiles ? ssp[i][0] : 0.f) + (t + 1 < nf.ss_tiles ? ssp[i][1] : 0.f) +
             (t + 2 < nf.ss_tiles ? ssp[i][2] : 0.f) + (t + 3 < nf.ss_tiles ? ssp[i][3] : 0.f);
    }
    if (nf.ss_tiles > 64 * SSP)
      for (int t = 64 * SSP + c; t < nf.ss_tiles; t += 16) sum += nf.ss_in[(size_t)msrc * ss_ld + t];
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    sum += __shfl_xor(sum, 4, 64);
    sum += __shfl_xor(sum, 8, 64);
    rstd = 1.0f / sqrtf(sum * nf.inv_width + nf.eps);
  }

  // sum the waves: acc[i] of lane (col, kb) is weight row 4 kb + i (column of the tile), x row col
#pragma unroll
  for (int a = 0; a < TW; ++a) *reinterpret_cast<f32x4*>(&s_acc[a][wave][lane * 4]) = acc[a];
  __syncthreads();
#pragma unroll
  for (int a = 0; a < TW; ++a) {
    const long n = n_of[a];
    float v = 0.f;
    {
      const int src = (((c >> 2) << 4) + m) * 4 + (c & 3);
#pragma unroll
      for (int w = 0; w < SG_WAVES; ++w) v += s_acc[a][w][src];
    }

    if (EPI == EPI_ADD) {
      const float r = e_old[a] + v;
      if (live[a]) ((float*)outv)[(size_t)m * ldo + n] = r;
      if (NF) {
        const float g = nf.g_f32 ? __uint_as_float(e_g[a]) : __uint_as_float(e_g[a] << 16);
        if (live[a]) nf.x_next[(size_t)m * nf.ldx_next + n] = __float2bfloat16(r * g);
        float q = live[a] ? r * r : 0.f;     // the 16 lanes of a row: sum of squares over this tile's columns
        q += __shfl_xor(q, 1, 64);
        q += __shfl_xor(q, 2, 64);
        q += __shfl_xor(q, 4, 64);
        q += __shfl_xor(q, 8, 64);
        if (c == 0 && m < M && tile0 + a < tiles) nf.ss_out[(size_t)m * ((tiles + 3) & ~3) + tile0 + a] = q;
      }
      continue;
    }
    const float mine_v = v * rstd;
    float other = 0.f;
    if (EPI == EPI_ROPE || EPI_GATED(EPI)) other = __shfl_xor(mine_v, 8, 64);   // the pair's other member
    if (!live[a]) continue;
    if (EPI == EPI_ROPE) {
      const int D = rope.D;
      const int head = (int)(n / D), jd = (int)(n - (long)head * D);   // column inside the head
      const int slot = e_slot;
      if (head < rope.Hq + rope.Hkv) {
        // first member (c < 8): x1 cos - x2 sin; second: x2 cos + x1 sin, x1 being the first member's value
        const float o = c < 8 ? mine_v * e_cos[a] - other * e_sin[a] : mine_v * e_cos[a] + other * e_sin[a];
        if (head < rope.Hq)
          ((bf16*)outv)[(size_t)m * ldo + n] = __float2bfloat16(o);
        else
          rope.k_cache[(((size_t)(slot / rope.page) * rope.Hkv + (head - rope.Hq)) * rope.page + slot % rope.page) * D + jd] =
              __float2bfloat16(o);
      } else {
        rope.v_cache[(((size_t)(slot / rope.page) * rope.Hkv + (head - rope.Hq - rope.Hkv)) * D + jd) * rope.page +
                     slot % rope.page] = __float2bfloat16(mine_v);
      }
    } else if (EPI == EPI_STORE_BF16) {
      ((bf16*)outv)[(size_t)m * ldo + n] = __float2bfloat16(mine_v);
    } else if (EPI == EPI_STORE_F32) {
      ((float*)outv)[(size_t)m * ldo + n] = mine_v;
    } else if (c < 8) {                      // gated: mine = gate, other = up
      if (EPI == EPI_CLAMPGLU) {
        const float g = fminf(mine_v, nf.glu_limit), u = fminf(fmaxf(other, -nf.glu_limit), nf.glu_limit);
        ((bf16*)outv)[(size_t)m * ldo + n] = __float2bfloat16(g * mie_sigmoid(nf.glu_alpha * g) * (u + nf.glu_shift));
      } else {
        const float f = EPI == EPI_GEGLU ? mie_gelu_tanh(mine_v) : mine_v / (1.0f + expf(-mine_v));
        ((bf16*)outv)[(size_t)m * ldo + n] = __float2bfloat16(f * other);
      }
    }
  }
}

MIE_EXPORT const char* gemm_bf16_last_error() { return g_mie_error; }
MIE_EXPORT int mie_skinny_max_rows() { return 16; }

template <bool NF, int TW, int XT, int SLOTS>
static int launch_epi(int epi, hipStream_t s, const bf16* X, long ldx, const bf16* W, long ldw, void* out,
                      long ldo, int M, int N, int K, int up_offset, int tiles, const RopeArgs& rope, const NormArgs& nf, int* held) {
  constexpr int lds = SG_WAVES * SLOTS * (2 * TW + XT) * 1024;
  const dim3 grid((tiles + TW - 1) / TW);
#define SG_LAUNCH(E)                                                                                                    \
  {                                                                                                                     \
    auto kernel = skinny_gemm_kernel<E, NF, TW, XT, SLOTS>;                                                             \
    if (mie_allow_lds((const void*)kernel, lds, "skinny_gemm")) return -1;                                              \
    if (held) return hipOccupancyMaxActiveBlocksPerMultiprocessor(held, kernel, SG_THREADS, lds) == hipSuccess ? 0 : -1; \
    hipLaunchKernelGGL(kernel, grid, dim3(SG_THREADS), lds, s, X, ldx, W, ldw, out, ldo, M, N, K, up_offset, tiles, rope, nf); \
  }
  switch (epi) {
    case EPI_STORE_BF16: SG_LAUNCH(EPI_STORE_BF16); break;
    case EPI_STORE_F32: SG_LAUNCH(EPI_STORE_F32); break;
    case EPI_ADD: SG_LAUNCH(EPI_ADD); break;
    case EPI_SWIGLU: SG_LAUNCH(EPI_SWIGLU); break;
    case EPI_GEGLU: SG_LAUNCH(EPI_GEGLU); break;
    case EPI_CLAMPGLU: SG_LAUNCH(EPI_CLAMPGLU); break;
    case EPI_ROPE: SG_LAUNCH(EPI_ROPE); break;
    default: MIE_FAIL("skinny_gemm: epilogue code %d", epi);
  }
#undef SG_LAUNCH
  MIE_CHECK_LAUNCH("skinny_gemm");
  return 0;
}

// Tiles a workgroup has.  One while every tile has a compute unit of its own; two where one would leave some compute units with
// two workgroups and others with one ([6144, 4096] at 8 rows: 12.2 us with one tile, 11.2 with two).  Beyond, up to 8 rows one again,
// three workgroups a compute unit ([28672, 4096] at 1 / 8 rows 37.4 / 37.9 us, two tiles 38.8 / 39.7), until the rounds are many
// ([128256, 4096]: 160.8 / 157.3 with one, 157.6 / 155.5 with two); from 9 rows on x weighs twice as much: three tiles while
// that gives every compute unit one workgroup ([11264, 2048] at 16 rows 10.7 with one, 9.9 with three), else two ([32000, 2048] 24.0,
// 22.1).  The sums do not depend on it.
static int tiles_for(int M, int tiles) {
  const int cu = mie_compute_units();
  if (tiles <= cu) return 1;
  if (tiles <= 2 * cu) return 2;
  if (M <= 8) return tiles <= 16 * cu ? 1 : 2;
  return tiles <= 3 * cu ? 3 : 2;
}

static int launch_rows(int tiles, int epi, hipStream_t s, const bf16* X, long ldx, const bf16* W, long ldw, void* out,
                       long ldo, int M, int N, int K, int up_offset, const RopeArgs& rope, const NormArgs& n, bool fused,
                       int* held = nullptr) {        // held: nothing is launched, the workgroups that a compute unit holds at once
  const int tw = tiles_for(M, tiles);
#define SG_ROWS(NF, TW, XT, SLOTS) return launch_epi<NF, TW, XT, SLOTS>(epi, s, X, ldx, W, ldw, out, ldo, M, N, K, up_offset, tiles, rope, n, held)
#define SG_TILES(TW, XT, SLOTS)                  \
  {                                              \
    if (fused) SG_ROWS(true, TW, XT, SLOTS);     \
    SG_ROWS(false, TW, XT, SLOTS);               \
  }
  // Slots: what lets a compute unit have its workgroups at once (two of 80 KB at most, the waves' sums with them, or three of 52);
  // one more where it has a single one ([2048, 5632] at 1 row: four slots 8.1 us, five 7.1).  So nothing else is in the LDS: with 64 bytes
  // more, for the rows' factors, a compute unit held one workgroup of two tiles and 9 to 16 rows behind a norm ([28672, 4096] at 9 rows 46.2
  // us for 42.0, [32000, 2048] at 16 30.5 for 26.5).
  if (M <= 8) {
    if (tw == 2) SG_TILES(2, 1, 3);
    if (tiles <= mie_compute_units()) SG_TILES(1, 1, 5);
    SG_TILES(1, 1, 4);
  }
  if (tw == 1) SG_TILES(1, 2, 5);
  if (tw == 2) SG_TILES(2, 2, 3);
  SG_TILES(3, 2, 2);
#undef SG_TILES
#undef SG_ROWS
}

static int check_operands(const char* what, const void* X, long ldx, const void* W, long ldw, int M, int K) {
  if (M > 16) MIE_FAIL("%s: %d rows (at most 16)", what, M);
  if (K <= 0 || (K & 7)) MIE_FAIL("%s: K = %d must be a positive multiple of 8", what, K);
  if (ldx < K || ldw < K || (ldw & 7) || (ldx & 7)) MIE_FAIL("%s: leading dims %ld, %ld for K %d", what, ldx, ldw, K);
  // 32-bit offsets: of up to 64 gathered rows from x, of 8 weight rows from the first of them
  if (ldx > 1L << 24 || ldw > 1L << 28) MIE_FAIL("%s: leading dims %ld, %ld (at most 2^24, 2^28)", what, ldx, ldw);
  if (((uintptr_t)X | (uintptr_t)W) & 15) MIE_FAIL("%s: operands must be 16-byte aligned", what);
  return 0;
}

// The fused norm, both sides.  Producer (epi 2 only): next_g (weight of the norm that follows, bfloat16 or
// float32), x_next [M, ldx_next] bfloat16 and ss_out [M, ceil(N / 16) rounded up to a multiple of 4] float32
// (16-byte aligned) are written beside the add.
// Consumer (other epilogues): X is a producer's x_next, ss_in its ss_out with ss_tiles tiles, width the
// norm's width (= K), rows an optional int32 [M] gather of X's rows.  Pass ss_in = next_g = null for none.
static int fill_norm_args(NormArgs& nf, int epi, const void* next_g, int next_g_f32, void* x_next, long ldx_next,
                          float* ss_out, const float* ss_in, int ss_tiles, int width, float eps, const int* rows,
                          int N) {
  nf = NormArgs{};
  if (epi == EPI_ADD) {
    if (!next_g || !x_next || !ss_out || ldx_next < N) MIE_FAIL("skinny_gemm: fused norm output operands");
    nf.g = next_g; nf.g_f32 = next_g_f32; nf.x_next = (bf16*)x_next; nf.ldx_next = ldx_next; nf.ss_out = ss_out;
  } else {
    if (!ss_in || ss_tiles <= 0 || width <= 0) MIE_FAIL("skinny_gemm: fused norm input operands");
    nf.ss_in = ss_in; nf.ss_tiles = ss_tiles; nf.inv_width = 1.0f / (float)width; nf.eps = eps; nf.rows = rows;
  }
  return 0;
}

// X [M, K] and W bfloat16.  epi: 0 bfloat16 y, 1 float32 y, 2 out[m, n] += y (float32), 3 silu(gate) * up with
// W = [gate rows (N of them); up rows] and N = the intermediate size, 5 the same with gelu_tanh(gate).
MIE_EXPORT int mie_skinny_gemm(const void* X, long ldx, const void* W, long ldw, void* out, long ldo, int epi, int M,
                               int N, int K, const void* next_g, int next_g_f32, void* x_next, long ldx_next,
                               float* ss_out, const float* ss_in, int ss_tiles, float eps, const int* rows,
                               hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (epi < 0 || (epi > EPI_SWIGLU && epi != EPI_GEGLU)) MIE_FAIL("skinny_gemm: epilogue code %d", epi);
  if (check_operands("skinny_gemm", X, ldx, W, ldw, M, K)) return -1;
  if (ldo < N) MIE_FAIL("skinny_gemm: output leading dim %ld < %d", ldo, N);
  RopeArgs none = {};
  NormArgs nf = {};
  const bool fused = next_g || ss_in;
  if (fused && fill_norm_args(nf, epi, next_g, next_g_f32, x_next, ldx_next, ss_out, ss_in, ss_tiles, K, eps, rows, N)) return -1;
  if (!fused && rows) MIE_FAIL("skinny_gemm: a row gather comes with the fused norm only");
  return launch_rows(EPI_GATED(epi) ? (N + 7) / 8 : (N + 15) / 16, epi, s, (const bf16*)X, ldx, (const bf16*)W, ldw, out, ldo, M, N, K, N, none,
                     nf, fused);
}

// Tiles that a workgroup of such a product has.
MIE_EXPORT int mie_skinny_tiles(int epi, int M, int N) { return tiles_for(M, EPI_GATED(epi) ? (N + 7) / 8 : (N + 15) / 16); }

// Workgroups of a product of M rows on a weight [N, K] (gated epilogues: N columns of gate and up) that a compute unit holds at once,
// with a norm fused in or not.
MIE_EXPORT int mie_skinny_held(int epi, int M, int N, int fused) {
  int held = 0;
  const int tiles = EPI_GATED(epi) ? (N + 7) / 8 : (N + 15) / 16;
  return launch_rows(tiles, epi, nullptr, nullptr, 0, nullptr, 0, nullptr, 0, M, N, 0, N, RopeArgs{}, NormArgs{}, fused != 0, &held) ? -1 : held;
}

// g sigmoid(alpha g) (u + shift) with g = min(gate, limit), u = clamp(up, -limit, limit); W = [gate rows (N of them); up rows],
// N the intermediate size, out bfloat16 [M, ldo].  With ss_in: X is a fused-norm producer's x_next (see above).
MIE_EXPORT int mie_skinny_clamped_glu(const void* X, long ldx, const void* W, long ldw, void* out, long ldo, int M, int N, int K,
                                      float limit, float alpha, float shift, const float* ss_in, int ss_tiles, float eps,
                                      const int* rows, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands("skinny_clamped_glu", X, ldx, W, ldw, M, K)) return -1;
  if (ldo < N || !(limit > 0.f)) MIE_FAIL("skinny_clamped_glu: output leading dim %ld < %d, limit %g", ldo, N, (double)limit);
  if (!ss_in && rows) MIE_FAIL("skinny_clamped_glu: a row gather comes with the fused norm only");
  RopeArgs none = {};
  NormArgs nf = {};
  if (ss_in && fill_norm_args(nf, EPI_CLAMPGLU, nullptr, 0, nullptr, 0, nullptr, ss_in, ss_tiles, K, eps, rows, N)) return -1;
  nf.glu_limit = limit; nf.glu_alpha = alpha; nf.glu_shift = shift;
  return launch_rows((N + 7) / 8, EPI_CLAMPGLU, s, (const bf16*)X, ldx, (const bf16*)W, ldw, out, ldo, M, N, K, N, none, nf, ss_in != nullptr);
}

// The fused q/k/v projection of single-token rows with what follows it: W [(Hq + 2 Hkv) D, K]; rotary
// (half-split pairs over the whole head, angles from cos/sin [positions, D / 2] float32) on the q and k
// heads in 32-bit, q [M, Hq D] written to q_out, rotated k and v written to cache slot slots[m]
// (k_cache [pages, Hkv, page, D], v_cache [pages, Hkv, D, page]).  D must be a multiple of 16.
// With ss_in: X is a fused-norm producer's x_next (see above).
MIE_EXPORT int mie_skinny_qkv_rope(const void* X, long ldx, const void* W, long ldw, void* q_out, long ldq,
                                   const int* positions, const float* cos_t, const float* sin_t, const int* slots,
                                   void* k_cache, void* v_cache, int M, int Hq, int Hkv, int D, int page, int K,
                                   const float* ss_in, int ss_tiles, float eps, hipStream_t s) {
  if (M <= 0) return 0;
  if (D <= 0 || (D & 15)) MIE_FAIL("skinny_qkv_rope: head_dim %d must be a multiple of 16", D);
  if (Hq <= 0 || Hkv <= 0 || page <= 0) MIE_FAIL("skinny_qkv_rope: heads %d / %d, page %d", Hq, Hkv, page);
  if (!positions || !cos_t || !sin_t || !slots || !k_cache || !v_cache || !q_out) MIE_FAIL("skinny_qkv_rope: null operand");
  if (check_operands("skinny_qkv_rope", X, ldx, W, ldw, M, K)) return -1;
  if (ldq < (long)Hq * D) MIE_FAIL("skinny_qkv_rope: q leading dim %ld < %d", ldq, Hq * D);
  RopeArgs rope = {positions, cos_t, sin_t, slots, (bf16*)k_cache, (bf16*)v_cache, Hq, Hkv, D, page};
  const int heads = Hq + 2 * Hkv;
  NormArgs nf = {};
  if (ss_in && fill_norm_args(nf, EPI_ROPE, nullptr, 0, nullptr, 0, nullptr, ss_in, ss_tiles, K, eps, nullptr, heads * D)) return -1;
  return launch_rows(heads * (D / 16), EPI_ROPE, s, (const bf16*)X, ldx, (const bf16*)W, ldw, q_out, ldq, M, heads * D, K,
                     D / 2, rope, nf, ss_in != nullptr);
}
