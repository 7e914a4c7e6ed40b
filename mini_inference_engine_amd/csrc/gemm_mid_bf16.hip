// Matrix products of the bfloat16 path with 17 to 128 rows: decode steps of many requests.
//
//   part[s, m, n] = sum over the k of split s of x[m, k] W[n, k]         (narrow weights: q/k/v, o, down)
//   out[m, j]     = silu(gate[m, j]) * up[m, j]  on their float32 sums   (gate and up, all of K in one workgroup)
//
// The few-row kernel (gemm_bf16.hip) gives every 16 weight rows a workgroup that reads all of x, which at 64 rows is four
// times the weights' bytes; a library product runs a narrow weight on a few dozen workgroups.  What a compute unit takes in
// is what bounds these products: 58 bytes a nanosecond, out of the L2 as well as from memory, by loads whose addresses cost some
// forty scalar instructions each as here (75 to 97 where an address is one addition, see tile_gemm_bf16.hip).  So a workgroup owns TW tiles of 16
// weight rows, as many as give every compute unit one workgroup, and x is read once per 16 TW weight rows.
//
// Its waves share no loads and meet at no barrier in the loop: chunks of 64 k are dealt to them in turn, a wave brings a
// chunk of all its weight rows and all x rows into its own slots of the LDS by loads that write the LDS directly (8 rows of
// 128 bytes a load, whole cache lines; block b of row r at 16-byte place 8 r + (b ^ r % 8), so that the fragment reads are
// spread over all banks), reads all fragments into registers, asks for the chunk after into the same slot at once and then
// multiplies (v_mfma_f32_16x16x32_bf16).  The waves' sums meet in the LDS, in wave order.  Weights by nontemporal loads.
// Before, four waves that shared a ring of stages met at a barrier a stage: a stage of 16 KB took 0.4 to 0.6 us whatever it
// loaded.  Measured (MI355X, us, before / now): with the sums' kernel and the norm, 24 rows of [2048, 2048] 8.5 / 7.3, [2560, 2048]
// 9.9 / 8.4, [2048, 5632] 11.9 / 9.7, [4096, 14336] 34.3 / 24.9; 64 rows 9.9 / 8.9, 11.2 / 10.2, 13.2 / 12.3, 33.4 / 30.2.  Of
// two or three chunks a wave 64 and 128 rows gain nothing ([3072, 3072] 13.4 / 13.8 and 17.3 / 18.3, [4096, 2048] 13.2 / 13.9 and 17.8 / 18.2,
// but 32 and 96 rows 12.3 / 11.2 and 17.0 / 16.1, 11.9 / 11.3 and 16.6 / 16.1; other numbers of splits 0.1 to 0.4 us at most).  Gate and
// up against the library's product and silu_mul: [11264, 2048] 17 / 64 / 128 rows 17.6 / 10.9, 19.9 / 13.7, 22.7 / 18.4;
// [28672, 4096] 17 / 64 rows 55.4 / 43, 57.1 / 47.5.
// The number of splits and of tiles a workgroup depends on the weight's shape alone and chunks go to waves by their place in
// K, so a row's result does not depend on the batch it is in.
//
// The kernels that follow add the partial results up in split order and do what comes after the product:
//   reduce_rows:     store (bfloat16 / float32), or add into the 32-bit stream, or add and RMSNorm for
//                    the norm that reads the stream next (one workgroup a row, as the norm kernel);
//   reduce_rope_kv:  the q/k/v projection: rotary on q and k, q out, k and v into their cache slots.
#include "launch.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void store_bf16x4(bf16* p, float4 v) {
  uint2 u;
  u.x = (uint32_t)__bfloat16_as_ushort(__float2bfloat16(v.x)) | ((uint32_t)__bfloat16_as_ushort(__float2bfloat16(v.y)) << 16);
  u.y = (uint32_t)__bfloat16_as_ushort(__float2bfloat16(v.z)) | ((uint32_t)__bfloat16_as_ushort(__float2bfloat16(v.w)) << 16);
  *reinterpret_cast<uint2*>(p) = u;
}

enum { MID_PART = 0, MID_SWIGLU = 1 };
constexpr int MID_WAVES = 4;      // more waves (six, eight) and fewer slots a wave: no faster at any shape

// MT: tiles of 16 x rows.  TW: tiles of 16 weight rows; with SWIGLU a tile is 8 gate rows and the up rows of
// the same columns, W = [gate rows (N of them); up rows].  TAIL: K is no multiple of 64.
// grid (weight tiles / TW, splits), `per` chunks a split; part [splits, M, N] float32, or out [M, ldo] bfloat16.
template <int TW, int MT, int SLOTS, int EPI, bool TAIL>
__global__ void __launch_bounds__(MID_WAVES * 64)
mid_gemm_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw, void* __restrict__ outv, long ldo,
                int M, int N, int K, int per) {
  constexpr int SLOT = (TW + MT) * 2048, L = 2 * (TW + MT);
  static_assert((SLOTS - 1) * L <= 63, "more loads in flight than the counter holds");
  extern __shared__ __align__(1024) char mid_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  const int lrow = lane >> 3, lblk = (lane & 7) ^ lrow;      // this lane's place in a load of 8 rows
  constexpr int COLS = EPI == MID_SWIGLU ? 8 : 16;           // columns of a tile
  const int j0 = blockIdx.x * TW * COLS;
  const int all = (K + 63) >> 6, c0 = blockIdx.y * per, chunks = all - c0 < per ? all - c0 : per;

  // offsets from the workgroup's first weight row (of the gate rows; the up rows lie a constant behind) and from x; a row that does
  // not exist reads the last one and is never stored
  constexpr int WO = EPI == MID_SWIGLU ? TW : 2 * TW;
  uint32_t woff[WO], xoff[2 * MT];
#pragma unroll
  for (int t = 0; t < WO; ++t) {
    const int r = t * 8 + lrow;
    woff[t] = (uint32_t)((long)(j0 + r < N ? r : N - 1 - j0) * ldw * 2) + lblk * 16;
  }
#pragma unroll
  for (int t = 0; t < 2 * MT; ++t) {
    const int r = t * 8 + lrow;
    xoff[t] = (uint32_t)((long)(r < M ? r : M - 1) * ldx * 2) + lblk * 16;
  }
  const char *wb = reinterpret_cast<const char*>(W + (size_t)j0 * ldw), *xb = reinterpret_cast<const char*>(X);
  const char* ub = wb + (size_t)N * ldw * 2;
  const uint32_t mine = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)mid_lds + wave * SLOTS * SLOT;
  auto issue = [&](int s) {
    const int c = c0 + s * MID_WAVES + wave;
    const size_t k = (size_t)c * 128;
    const uint32_t base = mine + (s % SLOTS) * SLOT;
    // blocks beyond K are read as the chunk's first block, and are zeros by the time they are multiplied
    const uint32_t back = TAIL && c * 64 + lblk * 8 >= K ? lblk * 16 : 0;
#pragma unroll
    for (int t = 0; t < 2 * TW; ++t) {
      if (EPI == MID_SWIGLU) mie_load_to_lds_nt((t & 1 ? ub : wb) + k, woff[t / (2 * TW / WO)] - back, base + t * 1024);
      else mie_load_to_lds_nt(wb + k, woff[t / (2 * TW / WO)] - back, base + t * 1024);
    }
#pragma unroll
    for (int t = 0; t < 2 * MT; ++t) mie_load_to_lds(xb + k, xoff[t] - back, base + TW * 2048 + t * 1024);
  };

  f32x4 acc[TW][MT];
#pragma unroll
  for (int a = 0; a < TW; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int n = (chunks - wave + MID_WAVES - 1) / MID_WAVES;      // this wave's chunks: wave, wave + 4, ...
#pragma unroll
  for (int s = 0; s < SLOTS; ++s)
    if (s < n) issue(s);
  for (int it = 0; it < n; ++it) {
    if (it + SLOTS <= n) MIE_VMCNT((SLOTS - 1) * L);              // chunk `it` has landed
    else MIE_VMCNT(0);
    asm volatile("" ::: "memory");
    const char* at = mid_lds + (wave * SLOTS + it % SLOTS) * SLOT;
    bf16x8 f[2][TW + MT];
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      const int blk = ((4 * kc + kb) ^ (col & 7)) * 16;
#pragma unroll
      for (int t = 0; t < TW; ++t) f[kc][t] = *reinterpret_cast<const bf16x8*>(at + t * 2048 + col * 128 + blk);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        f[kc][TW + t] = *reinterpret_cast<const bf16x8*>(at + TW * 2048 + t * 2048 + col * 128 + blk);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // read: the slot is free
    if (it + SLOTS < n) issue(it + SLOTS);
    if (TAIL && c0 + it * MID_WAVES + wave == all - 1) {
#pragma unroll
      for (int kc = 0; kc < 2; ++kc)
        if ((all - 1) * 64 + (4 * kc + kb) * 8 >= K) {
#pragma unroll
          for (int t = 0; t < TW + MT; ++t) f[kc][t] = __builtin_bit_cast(bf16x8, u32x4{0, 0, 0, 0});
        }
    }
#pragma unroll
    for (int kc = 0; kc < 2; ++kc)
#pragma unroll
      for (int a = 0; a < TW; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[kc][a], f[kc][TW + b], acc[a][b], 0, 0, 0);
  }

  __syncthreads();                                               // every wave is done with its slots
  // acc[a][b][i] of lane (col, kb): weight row 4 kb + i of tile a, x row 16 b + col.  PART reads neighbouring columns of a row together, 4 TW
  // of them for every x row: a lane's place within its 16 turned by 4 a + kb, so that those are in different banks.
  auto place = [&](int a, int l) { return EPI == MID_PART && TW <= 4 ? l ^ ((4 * a + (l >> 4)) * (4 / TW) & 15) : l; };
  f32x4* sums = reinterpret_cast<f32x4*>(mid_lds);
#pragma unroll
  for (int a = 0; a < TW; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) sums[((wave * TW + a) * MT + b) * 64 + place(a, lane)] = acc[a][b];
  __syncthreads();
  auto joined = [&](int a, int b, int l) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < MID_WAVES; ++w) v += sums[((w * TW + a) * MT + b) * 64 + place(a, l)];
    return v;
  };
  if (EPI == MID_SWIGLU) {
    for (int i = threadIdx.x; i < TW * MT * 32; i += MID_WAVES * 64) {
      const int l = i & 31, ab = i >> 5, a = ab % TW, b = ab / TW;
      const int m = b * 16 + (l & 15), j = j0 + a * 8 + (l >> 4) * 4;
      if (m >= M || j >= N) continue;
      f32x4 g = joined(a, b, l), u = joined(a, b, l + 32);       // gate rows at kb 0 and 1, up rows at kb 2 and 3
      float o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] = g[q] / (1.0f + expf(-g[q])) * u[q];
      store_bf16x4(reinterpret_cast<bf16*>(outv) + (size_t)m * ldo + j, make_float4(o[0], o[1], o[2], o[3]));
    }
  } else {
    float* out = reinterpret_cast<float*>(outv) + (size_t)blockIdx.y * M * N;
    for (int i = threadIdx.x; i < TW * MT * 64; i += MID_WAVES * 64) {
      const int q = i % (4 * TW), m = i / (4 * TW), j = j0 + q * 4;
      if (m >= M || j >= N) continue;
      *reinterpret_cast<f32x4*>(out + (size_t)m * N + j) = joined(q >> 2, m >> 4, (q & 3) * 16 + (m & 15));
    }
  }
}

// ---------------------------------------------------------------------------- after the product
enum { RED_STORE_BF16 = 0, RED_STORE_F32 = 1, RED_ADD = 2, RED_ADD_NORM = 3 };
constexpr int RED_THREADS = 512;
constexpr int RED_VEC = 4;        // float4 a thread: rows up to 8192 wide

// One workgroup a row; N a multiple of 4, at most 4 * RED_THREADS * RED_VEC.  y = sum of the splits in
// split order.  STORE: out[m, :] = y.  ADD: stream[m, :] += y.  ADD_NORM: also x_next[m, :] =
// bf16(stream * rsqrt(mean(stream^2) + eps) * g), the RMSNorm that reads the stream next.
template <int MODE>
__global__ void __launch_bounds__(RED_THREADS)
reduce_rows_kernel(const float* __restrict__ part, int splits, size_t split_stride, int N, void* __restrict__ out,
                   long ldo, float* __restrict__ stream, const void* __restrict__ g, int g_f32,
                   bf16* __restrict__ x_next, long ldx_next, float eps) {
  __shared__ float scratch[16];
  const int m = blockIdx.x;
  const float* pr = part + (size_t)m * N;
  f32x4 y[RED_VEC];
  float4 w[RED_VEC];
#pragma unroll
  for (int k = 0; k < RED_VEC; ++k) {
    const int i = (threadIdx.x + k * RED_THREADS) * 4;
    y[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    w[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < N) {
      if (MODE == RED_ADD || MODE == RED_ADD_NORM) y[k] = *reinterpret_cast<const f32x4*>(stream + (size_t)m * N + i);
      if (MODE == RED_ADD_NORM) {
        if (g_f32) {
          w[k] = *reinterpret_cast<const float4*>((const float*)g + i);
        } else {
          const uint2 u = *reinterpret_cast<const uint2*>((const uint16_t*)g + i);
          w[k] = make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xFFFF0000u), __uint_as_float(u.y << 16),
                             __uint_as_float(u.y & 0xFFFF0000u));
        }
      }
      add_splits(y[k], reinterpret_cast<const f32x4*>(pr + i), splits, split_stride / 4);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < RED_VEC; ++k) {
    const int i = (threadIdx.x + k * RED_THREADS) * 4;
    if (i >= N) continue;
    const float4 v = make_float4(y[k][0], y[k][1], y[k][2], y[k][3]);
    if (MODE == RED_STORE_BF16) store_bf16x4((bf16*)out + (size_t)m * ldo + i, v);
    if (MODE == RED_STORE_F32) *reinterpret_cast<float4*>((float*)out + (size_t)m * ldo + i) = v;
    if (MODE == RED_ADD || MODE == RED_ADD_NORM) *reinterpret_cast<float4*>(stream + (size_t)m * N + i) = v;
    ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss);
    ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
  }
  if (MODE != RED_ADD_NORM) return;
  const float total = block_sum(ss, scratch);
  const float rstd = 1.0f / sqrtf(total / (float)N + eps);
#pragma unroll
  for (int k = 0; k < RED_VEC; ++k) {
    const int i = (threadIdx.x + k * RED_THREADS) * 4;
    if (i >= N) continue;
    store_bf16x4(x_next + (size_t)m * ldx_next + i,
                 make_float4(y[k][0] * rstd * w[k].x, y[k][1] * rstd * w[k].y, y[k][2] * rstd * w[k].z, y[k][3] * rstd * w[k].w));
  }
}

// The q/k/v projection's partial results, grid (rows, ceil(heads / 4)), a wave a head (q heads, then k heads,
// then v heads): rotary (half-split pairs over the whole head, 32-bit angles) on the q and k heads,
// q [M, Hq D] out, k and v into cache slot slots[m] (k_cache [pages, Hkv, page, D], v_cache [pages, Hkv, D, page]).
__global__ void __launch_bounds__(256)
reduce_rope_kv_kernel(const float* __restrict__ part, int splits, size_t split_stride, bf16* __restrict__ q_out, long ldq,
                      const int* __restrict__ positions, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                      const int* __restrict__ slots, bf16* __restrict__ k_cache, bf16* __restrict__ v_cache, int Hq,
                      int Hkv, int D, int page) {
  const int m = blockIdx.x;
  const int head = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (head >= Hq + 2 * Hkv) return;
  const int N = (Hq + 2 * Hkv) * D;
  const float* pr = part + (size_t)m * N + (size_t)head * D;
  const int half = D >> 1;
  const int pos = positions[m], slot = slots[m];
  if (head < Hq + Hkv) {
    const float* cr = cos_t + (size_t)pos * half;
    const float* sr = sin_t + (size_t)pos * half;
    bf16* dst = head < Hq ? q_out + (size_t)m * ldq + (size_t)head * D
                          : k_cache + (((size_t)(slot / page) * Hkv + (head - Hq)) * page + (size_t)(slot % page)) * D;
    for (int j = lane; j < half; j += 64) {
      const float c = cr[j], sn = sr[j];
      float x1 = 0.f, x2 = 0.f;
      add_splits(x1, pr + j, splits, split_stride);
      add_splits(x2, pr + j + half, splits, split_stride);
      float o1, o2;
      rotate_pair(x1, x2, c, sn, o1, o2);
      dst[j] = __float2bfloat16(o1);
      dst[j + half] = __float2bfloat16(o2);
    }
  } else {
    bf16* dst = v_cache + ((size_t)(slot / page) * Hkv + (head - Hq - Hkv)) * page * D + (size_t)(slot % page);
    for (int d = lane; d < D; d += 64) {
      float v = 0.f;
      add_splits(v, pr + d, splits, split_stride);
      dst[(size_t)d * page] = __float2bfloat16(v);
    }
  }
}

MIE_EXPORT const char* gemm_mid_bf16_last_error() { return g_mie_error; }
MIE_EXPORT int mie_mid_max_rows() { return 128; }

// Weight rows a workgroup of mie_mid_gemm owns, from the weight's rows alone: 32 while that many leave room for three splits on
// a compute unit each, else 64 (24 rows of [4096, 4096] 12.6 us with 64 in four splits, 12.9 with 32 in two).
static int tile_rows(int N) { return (N + 31) / 32 <= 85 ? 32 : 64; }
MIE_EXPORT int mie_mid_tile_rows(int N) { return tile_rows(N); }

// How the caller has to cut K: chunks of 64 k a split for ``splits`` wanted splits, and the number of splits that gives.
static void cut_k(int K, int wanted, int* per, int* splits) {
  const int chunks = (K + 63) / 64;
  *per = (chunks + wanted - 1) / wanted;
  *splits = (chunks + *per - 1) / *per;
}

// The number of splits mie_mid_gemm will really make of ``wanted`` (the caller sizes ``part`` by it).
MIE_EXPORT int mie_mid_splits(int K, int wanted) {
  if (K <= 0 || wanted <= 0) return 0;
  int per, splits;
  cut_k(K, wanted, &per, &splits);
  return splits;
}

struct MidArgs {
  const bf16 *X, *W;
  long ldx, ldw, ldo;
  void* out;
  int M, N, K, per, splits;
};

template <int TW, int MT, int SLOTS, int EPI>
static int launch_mid(const MidArgs& a, hipStream_t s) {
  constexpr int ring = MID_WAVES * SLOTS * (TW + MT) * 2048, sums = MID_WAVES * TW * MT * 1024;
  constexpr int lds = ring > sums ? ring : sums, rows = TW * (EPI == MID_SWIGLU ? 8 : 16);
  if constexpr (lds > 160 * 1024) {
    return launch_mid<TW, MT, SLOTS - 1, EPI>(a, s);
  } else {
    auto kernel = a.K & 63 ? mid_gemm_kernel<TW, MT, SLOTS, EPI, true> : mid_gemm_kernel<TW, MT, SLOTS, EPI, false>;
    if (mie_allow_lds((const void*)kernel, lds, "mid_gemm")) return -1;
    hipLaunchKernelGGL(kernel, dim3((a.N + rows - 1) / rows, a.splits), dim3(MID_WAVES * 64), lds, s, a.X, a.ldx, a.W, a.ldw, a.out, a.ldo,
                       a.M, a.N, a.K, a.per);
    MIE_CHECK_LAUNCH("mid_gemm");
    return 0;
  }
}

template <int TW, int SLOTS, int EPI>
static int launch_rows(const MidArgs& a, hipStream_t s) {
  if (a.M <= 32) return launch_mid<TW, 2, SLOTS, EPI>(a, s);
  if (a.M <= 48) return launch_mid<TW, 3, SLOTS, EPI>(a, s);
  if (a.M <= 64) return launch_mid<TW, 4, SLOTS, EPI>(a, s);
  if constexpr (TW <= 4) {
    if (a.M <= 96) return launch_mid<TW, 6, SLOTS, EPI>(a, s);
    return launch_mid<TW, 8, SLOTS, EPI>(a, s);
  }
  MIE_FAIL("mid_gemm: %d rows with %d tiles", a.M, TW);
}

static int check_operands(const char* what, const void* X, long ldx, const void* W, long ldw, int M, int K) {
  if (M > 128) MIE_FAIL("%s: %d rows (at most 128)", what, M);
  if (K <= 0 || (K & 7)) MIE_FAIL("%s: K = %d must be a positive multiple of 8", what, K);
  if (ldx < K || ldw < K || (ldw & 7) || (ldx & 7)) MIE_FAIL("%s: leading dims %ld, %ld for K %d", what, ldx, ldw, K);
  // 32-bit offsets: of up to 128 rows from x, of up to 64 weight rows from a workgroup's first
  if (ldx > 1L << 24 || ldw > 1L << 24) MIE_FAIL("%s: leading dims %ld, %ld (at most 2^24)", what, ldx, ldw);
  if (((uintptr_t)X | (uintptr_t)W) & 15) MIE_FAIL("%s: operands must be 16-byte aligned", what);
  return 0;
}

// X [M, K], W [N, K] bfloat16 (16-byte aligned, leading dims multiples of 8, K a multiple of 8), M <= 128, N a multiple of 4.
// part [mie_mid_splits(K, wanted_splits), M, N] float32.  zeros has a place in the interface and is not read.
MIE_EXPORT int mie_mid_gemm(const void* X, long ldx, const void* W, long ldw, float* part, int M, int N, int K,
                            int wanted_splits, const void* zeros, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands("mid_gemm", X, ldx, W, ldw, M, K)) return -1;
  if (!part || ((uintptr_t)part & 15) || (N & 3)) MIE_FAIL("mid_gemm: partial sums of %d columns (16-byte aligned, a multiple of 4)", N);
  if (wanted_splits < 1 || wanted_splits > 64) MIE_FAIL("mid_gemm: %d splits", wanted_splits);
  MidArgs a = {(const bf16*)X, (const bf16*)W, ldx, ldw, 0, part, M, N, K, 0, 0};
  cut_k(K, wanted_splits, &a.per, &a.splits);
  return tile_rows(N) == 32 ? launch_rows<2, 2, MID_PART>(a, s) : launch_rows<4, 2, MID_PART>(a, s);
}

// Tiles a workgroup of the gated product has: those for which rounds of the grid times what a workgroup brings in a chunk (its
// weight rows and x) is least, of 1, 2, 3, 4, 6 and 7 (to 64 rows; to 4 beyond, where the waves' sums would not fit the LDS).  64 rows, us: [11264,
// 2048] 3 tiles 13.6, 4 15.1, 2 15; [22016, 4096] 6 tiles 34.9, 3 42.0, 7 37.7; [28672, 4096] 7 tiles 47.5, 4 48.7, 3 56.5.
static int swiglu_tiles(int M, int N) {
  const long tiles = (N + 7) / 8, cu = mie_compute_units();
  const int choices[6] = {1, 2, 3, 4, 6, 7}, x_tiles = (M + 15) / 16;
  int best = 1;
  long least = -1;
  for (int i = 0; i < (M <= 64 ? 6 : 4); ++i) {
    const long cost = ((tiles + choices[i] * cu - 1) / (choices[i] * cu)) * (choices[i] + x_tiles);
    if (least < 0 || cost < least) {
      least = cost;
      best = choices[i];
    }
  }
  return best;
}
MIE_EXPORT int mie_mid_swiglu_tiles(int M, int N) { return swiglu_tiles(M, N); }

// Whether this product gains over the library's and silu_mul: to 64 rows at every width measured (N of 512 to 28,672, K of 512 to 8,192:
// 0.44 to 0.99 of their time); beyond, where x is most of what a workgroup brings in, for K up to 2,048 and while the tiles are at most four
// and a half a compute unit, one round of the grid and a little.  us, library and silu_mul / own, 128 rows: [11264, 2048] 21.7 / 17.4, [16384,
// 2048] 23.9 / 22.9, [18432, 2048] 33.9 / 33.3, but [28672, 2048] 35.7 / 40.9, [28672, 1024] 21.8 / 24.4, [57344, 1024] 35.2 / 46.3, [22016, 2048]
// 31.6 / 35.5 (at 65 rows 29.4 / 27.0), [28672, 4096] 59.1 / 65.6, [22016, 4096] 54.0 / 57.3.
MIE_EXPORT int mie_mid_swiglu_gains(int M, int N, int K) { return M <= 64 || (K <= 2048 && 2L * ((N + 7) / 8) <= 9L * mie_compute_units()); }

// out [M, ldo] bfloat16 = silu(x Wg^T) * (x Wu^T), W = [gate rows (N of them); up rows], N a multiple of 4.
MIE_EXPORT int mie_mid_swiglu(const void* X, long ldx, const void* W, long ldw, void* out, long ldo, int M, int N, int K, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands("mid_swiglu", X, ldx, W, ldw, M, K)) return -1;
  if (!out || ldo < N || (ldo & 3) || (N & 3) || ((uintptr_t)out & 7)) MIE_FAIL("mid_swiglu: output leading dim %ld for %d columns", ldo, N);
  MidArgs a = {(const bf16*)X, (const bf16*)W, ldx, ldw, ldo, out, M, N, K, (K + 63) / 64, 1};
  const int tiles = swiglu_tiles(M, N);
  // two chunks of a wave on their way where a compute unit has one workgroup, one where it has two (64 rows of [28672, 4096] with four
  // tiles: 51.9 us with two chunks, 48.7 with one)
  const bool once = (long)tiles * 8 * mie_compute_units() >= N;
#define MID_TILES(TW) return once ? launch_rows<TW, 2, MID_SWIGLU>(a, s) : launch_rows<TW, 1, MID_SWIGLU>(a, s)
  switch (tiles) {
    case 1: MID_TILES(1);
    case 2: MID_TILES(2);
    case 3: MID_TILES(3);
    case 4: MID_TILES(4);
    case 6: MID_TILES(6);
    default: MID_TILES(7);
  }
#undef MID_TILES
}

// mode 0: out bfloat16 [M, ldo] = sum; 1: out float32; 2: stream [M, N] float32 += sum; 3: as 2, and
// x_next [M, ldx_next] bfloat16 = RMSNorm(stream) with weight g (bfloat16, or float32 if g_f32) and eps.
MIE_EXPORT int mie_mid_reduce(const float* part, int splits, int M, int N, int mode, void* out, long ldo, float* stream,
                              const void* g, int g_f32, void* x_next, long ldx_next, float eps, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (splits < 1 || !part) MIE_FAIL("mid_reduce: %d splits", splits);
  if ((N & 3) || N > 4 * RED_THREADS * RED_VEC) MIE_FAIL("mid_reduce: width %d (multiples of 4 up to %d)", N, 4 * RED_THREADS * RED_VEC);
  const size_t stride = (size_t)M * N;
  dim3 grid(M), block(RED_THREADS);
  switch (mode) {
    case RED_STORE_BF16:
    case RED_STORE_F32:
      if (!out || ldo < N || (ldo & 3) || ((uintptr_t)out & 15)) MIE_FAIL("mid_reduce: output operand");
      if (mode == RED_STORE_BF16)
        hipLaunchKernelGGL(reduce_rows_kernel<RED_STORE_BF16>, grid, block, 0, s, part, splits, stride, N, out, ldo, nullptr, nullptr, 0, nullptr, 0L, 0.f);
      else
        hipLaunchKernelGGL(reduce_rows_kernel<RED_STORE_F32>, grid, block, 0, s, part, splits, stride, N, out, ldo, nullptr, nullptr, 0, nullptr, 0L, 0.f);
      break;
    case RED_ADD:
      if (!stream || ((uintptr_t)stream & 15)) MIE_FAIL("mid_reduce: stream operand");
      hipLaunchKernelGGL(reduce_rows_kernel<RED_ADD>, grid, block, 0, s, part, splits, stride, N, nullptr, 0L, stream, nullptr, 0, nullptr, 0L, 0.f);
      break;
    case RED_ADD_NORM:
      if (!stream || !g || !x_next || ldx_next < N || (ldx_next & 3) || (((uintptr_t)stream | (uintptr_t)g | (uintptr_t)x_next) & 15))
        MIE_FAIL("mid_reduce: norm operands");
      hipLaunchKernelGGL(reduce_rows_kernel<RED_ADD_NORM>, grid, block, 0, s, part, splits, stride, N, nullptr, 0L, stream, g, g_f32,
                         (bf16*)x_next, ldx_next, eps);
      break;
    default: MIE_FAIL("mid_reduce: mode %d", mode);
  }
  MIE_CHECK_LAUNCH("mid_reduce");
  return 0;
}

MIE_EXPORT int mie_mid_reduce_rope_kv(const float* part, int splits, int M, void* q_out, long ldq, const int* positions,
                                      const float* cos_t, const float* sin_t, const int* slots, void* k_cache,
                                      void* v_cache, int Hq, int Hkv, int D, int page, hipStream_t s) {
  if (M <= 0) return 0;
  if (splits < 1 || !part) MIE_FAIL("mid_reduce_rope_kv: %d splits", splits);
  if (D <= 0 || (D & 1)) MIE_FAIL("mid_reduce_rope_kv: head_dim %d", D);
  if (Hq <= 0 || Hkv <= 0 || page <= 0) MIE_FAIL("mid_reduce_rope_kv: heads %d / %d, page %d", Hq, Hkv, page);
  if (!positions || !cos_t || !sin_t || !slots || !k_cache || !v_cache || !q_out) MIE_FAIL("mid_reduce_rope_kv: null operand");
  if (ldq < (long)Hq * D) MIE_FAIL("mid_reduce_rope_kv: q leading dim %ld < %d", ldq, Hq * D);
  const size_t stride = (size_t)M * (Hq + 2 * Hkv) * D;
  hipLaunchKernelGGL(reduce_rope_kv_kernel, dim3(M, (Hq + 2 * Hkv + 3) / 4), dim3(256), 0, s, part, splits, stride, (bf16*)q_out, ldq, positions,
                     cos_t, sin_t, slots, (bf16*)k_cache, (bf16*)v_cache, Hq, Hkv, D, page);
  MIE_CHECK_LAUNCH("mid_reduce_rope_kv");
  return 0;
}
