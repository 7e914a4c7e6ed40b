// Matrix products of the bfloat16 path with more than 128 rows, where more than the library's product is gained beside it:
//
//   gate and up with silu(gate) * up on their float32 sums (the separate pass over the library's output reads and writes both
//   once more), and narrow weights over a long K in parts of K, whose sums meet in the add + norm kernel that follows anyway
//   (reduce_rows in gemm_mid_bf16.hip).          x [M, K], W [N, K] bfloat16, float32 sums
//
// A workgroup makes BM x BN outputs with waves of 64 x 64 (v_mfma_f32_16x16x32_bf16, A = 16 weight rows, B = 16 x rows).
// Stages of 64 k come into a ring in the LDS by loads that write it directly, 8 rows x 128 bytes a load: whole cache lines
// (in halves of 64 bytes large tiles were up to a third slower: the L2s are asked twice for every line).  Row r's block b of
// 16 bytes stands at 8 r + (b ^ r % 8), so that the fragment reads (lane 16 g + r: row r, block g) spread over all banks.
//
// What bounds it: what a compute unit takes in, 58 bytes a nanosecond at most (a kernel that only loads, whatever the access pattern
// or who shares the lines), 36 to 48 with these tiles, rings and numbers of workgroups (the library's kernels move 43); reading the
// next fragments while one set is multiplied, across the barrier too, changed nothing.  So what counts is bytes a workgroup brings in, and that every compute unit has one: TILE_STAGE_US, the
// time of a stage of each tile, times the rounds of its grid picks the tile.
#include "launch.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { TG_F32, TG_SWIGLU };

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(a)) | ((uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(b)) << 16);
}

// grid: tiles over m (fastest), then n, then units of K, re-dealt so that an XCD takes a contiguous run of them.
// K in units of stages; unit z's sums go to out + z * unit_stride.
template <int WR, int WC, int STAGES, int EPI>
__global__ void __launch_bounds__(WR * WC * 64)
tile_gemm_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw, void* __restrict__ outv, long ldo,
                 int M, int N, int stages_all, int stages_unit, long unit_stride, int mt, int nt, int up_offset) {
  constexpr int WAVES = WR * WC, BM = WR * 64, BN = WC * 64, XL = BM / 8, LOADS = XL + BN / 8;
  constexpr int STAGE = LOADS * 1024, L = (LOADS + WAVES - 1) / WAVES;
  static_assert((STAGES - 2) * L <= 63, "more loads in flight than the counter holds");
  extern __shared__ __align__(1024) char tg_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  // workgroup i runs on XCD i % 8: give every XCD a run of neighbours, so that a weight tile is fetched into one L2
  int id = blockIdx.x;
  {
    const int total = gridDim.x, q = total >> 3, r = total & 7, x = id & 7, y = id >> 3;
    id = x * q + (x < r ? x : r) + y;
  }
  const int tm = id % mt, rest = id / mt, tn = rest % nt, unit = rest / nt;
  const int m0 = tm * BM;
  const int st0 = unit * stages_unit;
  const int nst = st0 + stages_unit < stages_all ? stages_unit : stages_all - st0;

  const int lrow = lane >> 3, lblk = (lane & 7) ^ lrow;          // this lane's place in a load of 8 rows
  uint32_t off[L], at[L];
  bool is_w[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    const int f = wave * L + j < LOADS ? wave * L + j : LOADS - 1;      // (the last one again)
    is_w[j] = f >= XL;
    long row;
    if (f < XL) {
      row = m0 + f * 8 + lrow;
      if (row >= M) row = M - 1;
      off[j] = (uint32_t)(row * ldx * 2) + lblk * 16;
    } else {
      const int r = (f - XL) * 8 + lrow;
      if (EPI == TG_SWIGLU) {                  // a wave's 64 weight rows: 32 gate rows, then the up rows of the same columns
        row = (long)tn * (BN / 2) + (r >> 6) * 32 + (r & 31);
        if (row >= N) row = N - 1;
        row += ((r >> 5) & 1) * (long)up_offset;
      } else {
        row = (long)tn * BN + r;
        if (row >= N) row = N - 1;
      }
      off[j] = (uint32_t)(row * ldw * 2) + lblk * 16;
    }
    at[j] = f * 1024;
  }
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)tg_lds;
  auto issue = [&](int s) {
    const char* xb = reinterpret_cast<const char*>(X) + (size_t)(st0 + s) * 128;
    const char* wb = reinterpret_cast<const char*>(W) + (size_t)(st0 + s) * 128;
    const uint32_t base = lds0 + (s % STAGES) * STAGE;
#pragma unroll
    for (int j = 0; j < L; ++j) mie_load_to_lds(is_w[j] ? wb : xb, off[j], base + at[j]);
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wr = wave % WR, wc = wave / WR;
  const char* xl = tg_lds + (wr * 64 + col) * 128;
  const char* wl = tg_lds + (BM + wc * 64 + col) * 128;

  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nst) issue(s);
  for (int it = 0; it < nst; ++it) {
    if (it + STAGES - 1 <= nst) MIE_VMCNT((STAGES - 2) * L);      // this wave's loads of stage `it` have landed
    else MIE_VMCNT(0);
    __builtin_amdgcn_s_barrier();                                // and everybody else's; everybody is done with stage it - 1
    asm volatile("" ::: "memory");
    if (it + STAGES - 1 < nst) issue(it + STAGES - 1);
    const int stage = (it % STAGES) * STAGE;
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      const int blk = stage + ((4 * kc + kb) ^ (col & 7)) * 16;
      bf16x8 wf[4], xf[4];
#pragma unroll
      for (int a = 0; a < 4; ++a) wf[a] = *reinterpret_cast<const bf16x8*>(wl + blk + a * 2048);
#pragma unroll
      for (int b = 0; b < 4; ++b) xf[b] = *reinterpret_cast<const bf16x8*>(xl + blk + b * 2048);
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[a], xf[b], acc[a][b], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // this wave has read the stage before the next barrier
  }

  // acc[a][b][i] of lane (col, kb): weight row 16 a + 4 kb + i of the wave's 64, x row 16 b + col
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int m = m0 + wr * 64 + b * 16 + col;
    if (m >= M) continue;
    if (EPI == TG_SWIGLU) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int n = tn * (BN / 2) + wc * 32 + a * 16 + 4 * kb;
        if (n >= N) continue;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float g = acc[a][b][i];
          o[i] = g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f)) * acc[a + 2][b][i];
        }
        *reinterpret_cast<uint2*>((bf16*)outv + (size_t)m * ldo + n) = make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
      }
      continue;
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int n = tn * BN + wc * 64 + a * 16 + 4 * kb;
      if (n >= N) continue;                    // N is a multiple of 4
      *reinterpret_cast<f32x4*>((float*)outv + unit * unit_stride + (size_t)m * ldo + n) = acc[a][b];
    }
  }
}

// The same by eight waves of TB x TA tiles of 16 x 16, four waves over x and two over W: wherever it was measured faster.  Three things
// beside the shape: loads go out from scalar addresses (no lane arithmetic), one between every TB matrix instructions (a load that finds
// the queue full stops its wave; all at once behind the barrier they stop every wave), and the second half's first fragments
// are asked for in the first half.  What each gave at 256 x 384 (2,048 rows of [11264, 2048], 240 tiles, MI355X; 256 x 192 tiles of the kernel
// above take 93.8 us): waves of 128 x 96, which spill registers, 106; addresses by lane arithmetic 97; scalar addresses, all loads at
// once 91; between the matrix instructions 85; the fragments 81.  Tiles of 256 x 384 bring in 80 KB a stage for the matrix instructions of
// six 128 x 128 tiles, which bring in 192 KB.
// SWIGLU: a wave's weight rows are TA / 2 tiles of gate rows, then the up rows of the same columns.  N is a multiple of 8.
template <int TA, int TB, int STAGES, int EPI>
__global__ void __launch_bounds__(512)
tile_spread_kernel(const bf16* __restrict__ X, uint32_t ldx, const bf16* __restrict__ W, uint32_t ldw, void* __restrict__ outv, long ldo,
                   int M, int N, int stages_all, int stages_unit, long unit_stride, int mt, int nt) {
  constexpr int WR = 4, WC = 2, BM = WR * TB * 16, BN = WC * TA * 16, XL = BM / 8, LOADS = XL + BN / 8, L = LOADS / 8;
  constexpr int STAGE = LOADS * 1024, HALF = TA * 8, COLS = EPI == TG_SWIGLU ? BN / 2 : BN;
  static_assert(LOADS % 8 == 0, "every wave brings in as many");
  static_assert(L < 2 * TA, "a load between every TB matrix instructions, from the second on");
  static_assert((STAGES - 2) * L <= 63, "more loads in flight than the counter holds");
  extern __shared__ __align__(1024) char tg_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  int id = blockIdx.x;
  {
    const int total = gridDim.x, q = total >> 3, r = total & 7, x = id & 7, y = id >> 3;
    id = x * q + (x < r ? x : r) + y;
  }
  const int tm = id % mt, rest = id / mt, tn = rest % nt, unit = rest / nt;
  const int m0 = tm * BM, n0 = tn * COLS;
  const int st0 = unit * stages_unit, nst = st0 + stages_unit < stages_all ? stages_unit : stages_all - st0;
  const int lrow = lane >> 3;
  const uint32_t lblk = ((lane & 7) ^ lrow) * 16;
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)tg_lds;
  // a load of 8 rows from a scalar address; of x's last 8 some may not exist, and those read the last one that does
  const int last_x = (M - 1) & ~7;
  const uint32_t xo = lrow * ldx * 2 + lblk, wo = lrow * ldw * 2 + lblk, xo_last = (lrow < M - last_x ? lrow : M - 1 - last_x) * ldx * 2 + lblk;
  auto load = [&](int s, int j) {              // the wave's j-th load of stage s
    const int f = wave * L + j;
    const uint32_t to = lds0 + (s % STAGES) * STAGE + f * 1024;
    const size_t k = (size_t)(st0 + s) * 128;
    if (f < XL) {
      const int g = m0 + f * 8, from = g < last_x ? g : last_x;
      mie_load_to_lds(reinterpret_cast<const char*>(X) + (size_t)from * ldx * 2 + k, g + 8 <= M ? xo : xo_last, to);
    } else {
      const int r = (f - XL) * 8;
      int g = n0 + r, behind = 0;
      if (EPI == TG_SWIGLU) {                  // 8 rows of one wave's gate or up rows
        const int w = r / (2 * HALF), at = r - w * 2 * HALF, up = at >= HALF;
        g = n0 + w * HALF + at - up * HALF;
        behind = up ? N : 0;
      }
      mie_load_to_lds(reinterpret_cast<const char*>(W) + (size_t)((g < N ? g : N - 8) + behind) * ldw * 2 + k, wo, to);
    }
  };
  f32x4 acc[TA][TB];
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wr = wave % WR, wc = wave / WR;
  const char* xl = tg_lds + (wr * TB * 16 + col) * 128;
  const char* wl = tg_lds + (BM + wc * TA * 16 + col) * 128;

  for (int t = 0; t < STAGES - 1; ++t)
    if (t < nst)
#pragma unroll
      for (int j = 0; j < L; ++j) load(t, j);
  for (int it = 0; it < nst; ++it) {
    if (it + STAGES - 1 <= nst) MIE_VMCNT((STAGES - 2) * L);      // this wave's loads of stage `it` have landed
    else MIE_VMCNT(0);
    __builtin_amdgcn_s_barrier();                                // and everybody else's; everybody is done with stage it - 1
    asm volatile("" ::: "memory");
    const bool more = it + STAGES - 1 < nst;
    const int stage = (it % STAGES) * STAGE, blk1 = stage + ((4 + kb) ^ (col & 7)) * 16;
    int next = 0;
    bf16x8 xf[2][TB], wf[2];
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      const int blk = stage + ((4 * kc + kb) ^ (col & 7)) * 16;
      if (kc == 0) {
#pragma unroll
        for (int b = 0; b < TB; ++b) xf[0][b] = *reinterpret_cast<const bf16x8*>(xl + blk + b * 2048);
        wf[0] = *reinterpret_cast<const bf16x8*>(wl + blk);
      }
#pragma unroll
      for (int a = 0; a < TA; ++a) {
        if (a + 1 < TA) wf[(a + 1) & 1] = *reinterpret_cast<const bf16x8*>(wl + blk + (a + 1) * 2048);
        else if (kc == 0) wf[(a + 1) & 1] = *reinterpret_cast<const bf16x8*>(wl + blk1);
        if (kc == 0 && a + TB >= TA) xf[1][a + TB - TA] = *reinterpret_cast<const bf16x8*>(xl + blk1 + (a + TB - TA) * 2048);
        if (kc * TA + a >= 1 && next < L) {
          if (more) load(it + STAGES - 1, next);
          ++next;
        }
#pragma unroll
        for (int b = 0; b < TB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[a & 1], xf[kc][b], acc[a][b], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // this wave has read the stage before the next barrier
  }

  // acc[a][b][i] of lane (col, kb): weight row 16 a + 4 kb + i of the wave's, x row 16 b + col
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    const int m = m0 + (wr * TB + b) * 16 + col;
    if (m >= M) continue;
    if (EPI == TG_SWIGLU) {
#pragma unroll
      for (int a = 0; a < TA / 2; ++a) {
        const int n = n0 + wc * HALF + a * 16 + 4 * kb;
        if (n >= N) continue;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float g = acc[a][b][i];
          o[i] = g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f)) * acc[a + TA / 2][b][i];
        }
        *reinterpret_cast<uint2*>((bf16*)outv + (size_t)m * ldo + n) = make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
      }
      continue;
    }
#pragma unroll
    for (int a = 0; a < TA; ++a) {
      const int n = n0 + (wc * TA + a) * 16 + 4 * kb;
      if (n >= N) continue;
      *reinterpret_cast<f32x4*>((float*)outv + unit * unit_stride + (size_t)m * ldo + n) = acc[a][b];
    }
  }
}

MIE_EXPORT const char* tile_gemm_bf16_last_error() { return g_mie_error; }

template <int WR, int WC, int STAGES, int EPI>
static int launch(const bf16* X, long ldx, const bf16* W, long ldw, void* out, long ldo, int M, int N, int K, int units, hipStream_t s) {
  constexpr int BM = WR * 64, BN = WC * 64, cols = EPI == TG_SWIGLU ? BN / 2 : BN;
  constexpr int lds = STAGES * (BM + BN) * 128;
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = tile_gemm_kernel<WR, WC, STAGES, EPI>;
  if (mie_allow_lds((const void*)kernel, lds, "tile_gemm")) return -1;
  const int mt = (M + BM - 1) / BM, nt = (N + cols - 1) / cols, stages = K / 64, per = (stages + units - 1) / units;
  if ((long)mt * nt * units > 0x7FFFFFFF) MIE_FAIL("tile_gemm: %d x %d tiles are beyond the grid", mt, nt);
  hipLaunchKernelGGL(kernel, dim3(mt * nt * units), dim3(WR * WC * 64), lds, s, X, ldx, W, ldw, out, ldo, M, N, stages, per,
                     (long)M * N, mt, nt, N);
  MIE_CHECK_LAUNCH("tile_gemm");
  return 0;
}

template <int TA, int TB, int STAGES, int EPI>
static int launch_spread(const bf16* X, long ldx, const bf16* W, long ldw, void* out, long ldo, int M, int N, int K, int units, hipStream_t s) {
  constexpr int BM = TB * 64, BN = TA * 32, cols = EPI == TG_SWIGLU ? BN / 2 : BN, lds = STAGES * (BM + BN) * 128;
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = tile_spread_kernel<TA, TB, STAGES, EPI>;
  if (mie_allow_lds((const void*)kernel, lds, "tile_gemm")) return -1;
  const int mt = (M + BM - 1) / BM, nt = (N + cols - 1) / cols, stages = K / 64, per = (stages + units - 1) / units;
  if ((long)mt * nt * units > 0x7FFFFFFF) MIE_FAIL("tile_gemm: %d x %d tiles are beyond the grid", mt, nt);
  hipLaunchKernelGGL(kernel, dim3(mt * nt * units), dim3(512), lds, s, X, (uint32_t)ldx, W, (uint32_t)ldw, out, ldo, M, N, stages, per,
                     (long)M * N, mt, nt);
  MIE_CHECK_LAUNCH("tile_gemm");
  return 0;
}

static int check_operands(const void* X, long ldx, const void* W, long ldw, const void* out, int M, long w_rows, int N, int K) {
  if (K <= 0 || (K & 63) || (N & 7)) MIE_FAIL("tile_gemm: K = %d (multiples of 64), N = %d (of 8)", K, N);
  if (ldx < K || ldw < K || (ldx & 7) || (ldw & 7)) MIE_FAIL("tile_gemm: leading dims %ld, %ld for K %d", ldx, ldw, K);
  if (((uintptr_t)X | (uintptr_t)W | (uintptr_t)out) & 15) MIE_FAIL("tile_gemm: operands must be 16-byte aligned");
  if ((long)M * ldx > 0x40000000L || w_rows * ldw > 0x40000000L) MIE_FAIL("tile_gemm: an operand of more than 2 GiB");
  return 0;
}


// Time of a stage (64 k) of a grid that gives every compute unit one workgroup, with its share of the start and the end, us: measured at
// 160 to 2,048 rows of [11264, 2048] (MI355X).  256 x 384, the second 128 x 128 and those behind it are tile_spread_kernel's, the others
// tile_gemm_kernel's, of which 128 x 128 is for the estimate alone (mie_tile_gemm_swiglu_cost).  Own tile of
// before / now, us: 160 rows 25.2 / 22.4, 256 26.0 / 23.9, 384 36.8 / 30.2, 512 34.1 / 31.1, 768 45.7 / 36.3, 1,536 73.0 / 62.6, 2,048 93.8 / 76.9;
// at 1,024 and 1,132 rows 256 x 256 of sixteen waves of 64 x 64 stays (45.6 and 50.5 us; of eight of 64 x 128 54.6 and 53.7).
constexpr struct { int bm, bn; float us; } TILE_STAGE_US[] = {
  {128, 128, 0.76f}, {192, 128, 0.98f}, {256, 128, 0.99f}, {256, 192, 1.33f}, {256, 256, 1.57f}, {256, 384, 2.35f},
  {128, 128, 0.72f}, {128, 192, 0.96f}, {192, 192, 1.12f}, {256, 320, 1.94f}};

constexpr int TILES_TAKEN = 1, TILES_ESTIMATED = 6, TILES = 10;       // taken: from the first on; estimated: those before the second

// of tiles first .. behind - 1 the one with the least time
static int best_tile(int M, long cols, int first, int behind, float& us) {
  int best = first;
  us = 1e30f;
  for (int i = first; i < behind; ++i) {
    const long tiles = (long)((M + TILE_STAGE_US[i].bm - 1) / TILE_STAGE_US[i].bm) * ((cols + TILE_STAGE_US[i].bn - 1) / TILE_STAGE_US[i].bn);
    const long rounds = (tiles + mie_compute_units() - 1) / mie_compute_units();
    if (rounds * TILE_STAGE_US[i].us < us) {
      us = rounds * TILE_STAGE_US[i].us;
      best = i;
    }
  }
  return best;
}

// What mie_tile_gemm_swiglu takes at most, in units of 0.01 us, for the decision against the library.  It leaves out the tiles of the spread
// kernel but 256 x 384: with them the decision, whose estimate of the library is rough, would change for the better at some sizes and
// for the worse at others (us, own / library / library's kernel chosen by timing: 1,300 rows of [11264, 2048] 63.8 / 71.7 / 72.6, 550 rows
// 36.2 / 36.7 / 36.8, but 256 rows of [8192, 2048] 22.6 / 24.8 / 19.6).
MIE_EXPORT int mie_tile_gemm_swiglu_cost(int M, int N, int K) {
  float us;
  best_tile(M, 2L * N, 0, TILES_ESTIMATED, us);
  return (int)(100.f * us * (K / 64));
}
// The tile that mie_tile_gemm_swiglu takes: 1,000 times its rows plus its columns.
MIE_EXPORT int mie_tile_gemm_swiglu_tile(int M, int N) {
  float us;
  const auto& t = TILE_STAGE_US[best_tile(M, 2L * N, TILES_TAKEN, TILES, us)];
  return t.bm * 1000 + t.bn;
}

// out [M, ldo] bfloat16 = silu(x Wg^T) * (x Wu^T), W = [gate rows (N of them); up rows].
MIE_EXPORT int mie_tile_gemm_swiglu(const void* X, long ldx, const void* W, long ldw, void* out, long ldo, int M, int N, int K, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands(X, ldx, W, ldw, out, M, 2L * N, N, K)) return -1;
  if (ldo < N || (ldo & 3)) MIE_FAIL("tile_gemm_swiglu: output leading dim %ld for %d columns", ldo, N);
  const bf16 *x = (const bf16*)X, *w = (const bf16*)W;
  float us;
  switch (best_tile(M, 2L * N, TILES_TAKEN, TILES, us)) {
    case 1: return launch<3, 2, 2, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    case 2: return launch<4, 2, 3, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    case 3: return launch<4, 3, 2, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    case 4: return launch<4, 4, 2, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    case 5: return launch_spread<12, 4, 2, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    case 6: return launch_spread<4, 2, 4, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    case 7: return launch_spread<6, 2, 4, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    case 8: return launch_spread<6, 3, 3, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
    default: return launch_spread<10, 4, 2, TG_SWIGLU>(x, ldx, w, ldw, out, ldo, M, N, K, 1, s);
  }
}

// part [units, M, N] float32: the sums over unit u's part of K.  Every unit has at least one stage of 64 k.
MIE_EXPORT int mie_tile_gemm_units(const void* X, long ldx, const void* W, long ldw, float* part, int M, int N, int K, int units, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands(X, ldx, W, ldw, part, M, N, N, K)) return -1;
  const int stages = K / 64, per = units > 0 ? (stages + units - 1) / units : 0;
  if (units < 1 || (units - 1) * per >= stages) MIE_FAIL("tile_gemm_units: %d units of %d stages", units, stages);
  const bf16 *x = (const bf16*)X, *w = (const bf16*)W;
  // a workgroup a compute unit and a deep ring, or two and a short one (512 rows of [2048, 5632] in four parts 21.4 us by four waves of 64 x
  // 64, 20.7 by eight; of [4096, 14336] in two 81.1 and 77.1)
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128) * units;
  return tiles <= mie_compute_units() ? launch_spread<4, 2, 4, TG_F32>(x, ldx, w, ldw, part, N, M, N, K, units, s)
                                  : launch<2, 2, 2, TG_F32>(x, ldx, w, ldw, part, N, M, N, K, units, s);
}
