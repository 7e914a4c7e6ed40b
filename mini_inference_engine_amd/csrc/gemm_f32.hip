// Matrix products of the float32 path on the bfloat16 matrix instruction, every operand in three parts.
//
//   y[m, n] = sum_k x[m, k] W[n, k]          x [M, K], W [N, K], y [M, N] float32
//
// 2^16 times a 32-bit number v of less than 2^111 is the sum of three bfloat16 ones to its last bit (24 bits of mantissa in three
// pieces of 8, the signs take up the roundings): h = bf16(2^16 v), m = bf16(2^16 v - h), l = 2^16 v - h - m.  Without the factor m and
// l would fall below bfloat16's smallest number, 2^-133, for v below 2^-110 (the error of a product of operands of 1 and 2^-118 would be
// 9e-6 for 1e-7); the sums lose the 2^32 of both operands at their end.  Of the nine products six are taken, hh, hm, mh, mm, hl, lh; the
// three left out, ml, lm and ll, are together at most a little more than 2^-24 of |x w|.  A product of two bfloat16 numbers is
// exact in 32 bits, so what rounds is the sums, and those of the five small products run in a chain of their own, where a
// rounding is 2^-8 of one in the sums of hh.  Six v_mfma_f32_16x16x32_bf16 take 96 cycles of a SIMD for what eight
// v_mfma_f32_16x16x4_f32 (true 32-bit products) need 256 for.
//
// One order of summation for every kernel here, whatever M is, so that a row's result is bit-identical however the
// batch around it is cut.  K is taken in steps of 32; the steps are cut into four quarters and every quarter into two
// eighths (sizes from K alone).  An eighth is one chain of steps for hh and one for the small products and ends as their sum, a
// quarter is e0 + e1 and the result ((q0 + q1) + q2) + q3.
//
// Results that are not finite are computed again, in 64 bits (plain_product): a number whose 2^16-fold bfloat16 cannot hold (2^111
// and more, an infinity) has no such parts and gives NaN, and where h(x) h(w) or a sum of them goes beyond the largest number
// (results of 2^95 and more) the parts give an infinity for what may be a finite result.  The rule looks at the whole sum over K alone
// (units' sums are looked at where they are joined), so it is the same for every cut of the batch.  It is there to be right, not fast:
// 512 rows of [2048, 2048] all of whose results are such take 1.2 ms for 0.035.
//
// skinny_f32_kernel (M <= 16): the weights' bytes bound it.  A workgroup owns 16 rows of W; a wave streams a contiguous
//   part of K through a ring of its own in the LDS, filled by loads that write the LDS directly: 8 rows of 32 k a load, lane
//   8 r + b (whole cache lines, where the instruction's own order would touch 16 lines a quarter wave), block b of 16 bytes at
//   8 r + (b ^ r % 8), so that the fragment reads spread over all banks; parts of K meet in the LDS at the end.  Eight waves a
//   workgroup (a deeper queue of loads a compute unit) while the tiles do not fill the compute units, four from there on.
//   A product that goes into a stream whose norm is wanted next takes two workgroups a tile instead, half of K each (a narrow
//   weight's tiles alone leave half of the compute units idle), and the kernel that joins the quarters adds and norms: product, add and
//   norm at 4 rows, before / now: [2048, 2048] 10.6 / 8.9 us, [2048, 5632] 17.5 / 13.8.
// tile_f32_kernel (M > 16): the matrix unit bounds it.  BM x BN outputs a workgroup; a stage of 32 k comes into registers,
//   is split there once for all waves, and goes into the LDS as three planes of bfloat16 (two buffers), while the stage
//   before is multiplied.  Few tiles: the grid is also cut over quarters or eighths, whose sums go to memory and meet in
//   reduce_f32_kernel, or with the norm that follows in reduce_add_norm_kernel (512 rows of [2048, 2048] with add and norm 38.5 / 36.0).
//
// Measured on MI355X against the same kernels on v_mfma_f32_16x16x4_f32, both without the factor of 2^16 (us; those / these): 512 rows of
// [11264, 2048] with SwiGLU 237 / 175, [2048, 5632] 116 / 73, [2048, 2048] 51 / 35; 100 rows 69 / 59, 36 / 29, 21 / 16; 4 rows 21.9 / 19.2,
// 17.0 / 14.8, 8.8 / 8.3.  Without / with the factor, another harness: 512 rows 171 / 166, 71.5 / 70.9, 33.3 / 33.2, 4 rows 18.0 / 18.1,
// 14.9 / 15.1.  Steps of the engine, 22 layers of width 2,048, 32-bit instruction / these: a prompt of 512 tokens 11,637 / 8,775, 4
// rows 1,700 / 1,628.  Relative error of [2048, 2048] against 64 bits 2.1e-7 / 1.0e-7, of [2048, 5632] 3.4e-7 / 1.6e-7, of a whole step's
// logits 2.2e-6 / 1.5e-6 (with the small products in the chain of hh it would be 2.4e-7 and 4.1e-7).  What is left in the tile
// kernel: matrix instructions alone take 63 us for 2,048 rows of [2048, 2048] (the clock falls with every compute unit at them), the
// fragment reads add 15, the splitting the rest of its 93.
#include "launch.hpp"

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __align__(128) const uint32_t mie_zero_words[32] = {0};

// The cut of K, in steps of 32: quarter q is steps [q * quarter, min((q + 1) * quarter, steps)), an eighth `eighth` steps.
struct KCut {
  int steps, quarter, eighth;
};
__host__ __device__ __forceinline__ KCut k_cut(int K) {
  KCut c;
  c.steps = (K + 31) / 32;
  c.quarter = (c.steps + 3) / 4;
  c.eighth = (c.quarter + 1) / 2;
  return c;
}
__host__ __device__ __forceinline__ int least(int a, int b) { return a < b ? a : b; }

// steps [begin, end) of eighth e (0 .. 7); may be empty
__host__ __device__ __forceinline__ void eighth_range(const KCut& c, int e, int& begin, int& end) {
  const int q0 = least((e >> 1) * c.quarter, c.steps), q1 = least(q0 + c.quarter, c.steps);
  begin = least(q0 + (e & 1) * c.eighth, q1);
  end = least(begin + c.eighth, q1);
}

// two numbers as bfloat16, the first in the low half
__device__ __forceinline__ uint32_t round2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
constexpr float GF_SCALE = 65536.f, GF_UNSCALE = 1.f / (65536.f * 65536.f);      // of an operand; of what two scaled ones give
// c minus the low or the high half of h (sel: -1 there, 0 in the other), exact where the difference is a 32-bit number: one
// instruction for the shift or mask and the subtraction.  sel in a scalar register: as a constant the compiler writes -1.0 into the
// instruction, which stands for another half.
__device__ __forceinline__ float less_half(float c, uint32_t h, uint32_t sel) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, h), __builtin_bit_cast(bf16x2, sel), c, false);
}
struct Halves {
  uint32_t low, high;
};
__device__ __forceinline__ Halves minus_one() {
  Halves s;
  asm("s_mov_b32 %0, 0xbf80" : "=s"(s.low));
  asm("s_mov_b32 %0, 0xbf800000" : "=s"(s.high));
  return s;
}
// h, m, l of two numbers.  DOT: the differences by less_half, which pays where splitting bounds a kernel (tiles of 64 x 64 44.8 us against
// 45.9 at 512 rows of [2560, 2048]) and not beside many matrix instructions (128 x 128 tiles 176 against 167 at 512 of [11264, 2048]).
template <bool DOT>
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  const Halves minus = minus_one();
  a *= GF_SCALE;
  b *= GF_SCALE;
  h = round2(a, b);
  a = DOT ? less_half(a, h, minus.low) : a - __uint_as_float(h << 16);
  b = DOT ? less_half(b, h, minus.high) : b - __uint_as_float(h & 0xFFFF0000u);
  m = round2(a, b);
  a = DOT ? less_half(a, m, minus.low) : a - __uint_as_float(m << 16);
  b = DOT ? less_half(b, m, minus.high) : b - __uint_as_float(m & 0xFFFF0000u);
  l = round2(a, b);
}

struct Parts {
  bf16x8 h, m, l;
};
__device__ __forceinline__ Parts split8(const f32x4& a, const f32x4& b) {
  u32x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float p = i < 2 ? a[2 * i] : b[2 * i - 4], q = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
    uint32_t hh, mm, ll;
    split2<true>(p, q, hh, mm, ll);
    h[i] = hh, m[i] = mm, l[i] = ll;
  }
  return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

// One result by 64-bit multiplications and additions, k ascending.
__device__ __forceinline__ float plain_product(const float* x, const float* w, int K) {
  double s = 0.0;
#pragma unroll 4
  for (int k = 0; k < K; k += 4) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(x + k), b = *reinterpret_cast<const f32x4*>(w + k);
#pragma unroll
    for (int i = 0; i < 4; ++i) s = fma((double)a[i], (double)b[i], s);
  }
  return (float)s;
}
__device__ __forceinline__ bool finite(float v) { return fabsf(v) < INFINITY; }
// four results beside each other, x times the rows w, w + ldw, ...: those that are not finite computed again
__device__ __forceinline__ void again_if_not_finite(f32x4& v, const float* x, const float* w, long ldw, int K) {
  if (!__any(!(finite(v[0]) && finite(v[1]) && finite(v[2]) && finite(v[3])))) return;
#pragma unroll 1
  for (int i = 0; i < 4; ++i) {
    const float t = i == 0 ? v[0] : i == 1 ? v[1] : i == 2 ? v[2] : v[3];
    if (finite(t)) continue;
    const float r = plain_product(x, w + i * ldw, K);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = i == j ? r : v[j];
  }
}

enum { GF_STORE = 0, GF_ADD = 1, GF_SWIGLU = 2, GF_ROPE = 3, GF_PART = 4 };

// The q/k/v projection's epilogue: W's rows are q heads, k heads, v heads of D; a tile is 8 rotary pairs of one head.
struct RopeArgs {
  const int* positions;      // [M]
  const float *cos_t, *sin_t;// [positions, D / 2]
  const int* slots;          // [M] cache slot of each row's token
  float *k_cache, *v_cache;  // [pages, Hkv, page, D], [pages, Hkv, D, page]
  int Hq, Hkv, D, page;
};

// ------------------------------------------------------------------------------------------------ few rows
constexpr int GF_NONTEMPORAL = 2;             // the hint of loads whose lines nobody reads again: the weights

// Fragments out of the LDS, read and waited for in one piece of assembly: the compiler knows nothing of the loads that
// write the LDS and would wait for all of them at a read it could see.
__device__ __forceinline__ void ring_read(uint32_t w0, uint32_t w1, uint32_t x0, uint32_t x1, u32x4 (&f)[4]) {
  asm volatile(
    "ds_read_b128 %0, %4\n\t"
    "ds_read_b128 %1, %5\n\t"
    "ds_read_b128 %2, %6\n\t"
    "ds_read_b128 %3, %7\n\t"
    "s_waitcnt lgkmcnt(0)"
    : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3])
    : "v"(w0), "v"(w1), "v"(x0), "v"(x1)
    : "memory");
}
__device__ __forceinline__ void ring_read(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t x0, uint32_t x1, u32x4 (&f)[6]) {
  asm volatile(
    "ds_read_b128 %0, %6\n\t"
    "ds_read_b128 %1, %7\n\t"
    "ds_read_b128 %4, %10\n\t"
    "ds_read_b128 %5, %11\n\t"
    "ds_read_b128 %2, %8\n\t"
    "ds_read_b128 %3, %9\n\t"
    "s_waitcnt lgkmcnt(0)"
    : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3]), "=&v"(f[4]), "=&v"(f[5])
    : "v"(w0), "v"(w1), "v"(w2), "v"(w3), "v"(x0), "v"(x1)
    : "memory");
}
// the other half of every row of 16 lanes
__device__ __forceinline__ bf16x8 other_half(const bf16x8& v) {
  u32x4 r = __builtin_bit_cast(u32x4, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_update_dpp(0, r[i], 0x128, 0xF, 0xF, false);      // row_ror:8
  return __builtin_bit_cast(bf16x8, r);
}

// XL: loads of x a slot: two, or one for up to 8 rows.  Then two steps are taken at once: lanes of columns 0 to 7 read and split the
// first one's x and those of columns 8 to 15 the second one's (an x row is split once, not twice; what columns 8 to 15 add up is
// nobody's result), and one wait serves both: a step of 4 rows
// (22 layers of width 2,048) 1,710 us with a step at a time, 1,616 with two.
// SWIGLU: W is gate rows then up rows (up_offset apart); a tile is 8 gate rows and the 8 up rows of the same columns.
// PART: a workgroup of four waves takes half of K (blockIdx.y), an eighth a wave, and leaves its two quarters' sums in out [4, M, N].
template <int EPI, int WAVES, int SLOTS, int XL>
__global__ void __launch_bounds__(WAVES * 64)
skinny_f32_kernel(const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, float* __restrict__ out,
                  long ldo, const float* __restrict__ bias, int M, int N, int K, int up_offset, RopeArgs rope) {
  constexpr int EPW = EPI == GF_PART ? 1 : 8 / WAVES;              // eighths a wave
  constexpr int U = XL == 1 ? 2 : 1;          // steps at once
  constexpr int L = 2 + XL, SLOT_BYTES = L * 1024;       // loads a slot of 32 k: 16 weight rows of 128 bytes, then the x rows
  static_assert((SLOTS - 1) * L <= 63, "more loads in flight than the counter holds");
  extern __shared__ __align__(16) char gf_lds[];
  char* ring = gf_lds;                                            // WAVES * SLOTS slots
  float* s_acc = reinterpret_cast<float*>(gf_lds);                // [8][256], once every wave is done with its ring
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tile = blockIdx.x;
  const KCut cut = k_cut(K);
  int first_end, ks0, ks1;
  {
    int b;
    const int e = wave * EPW + (EPI == GF_PART ? 4 * blockIdx.y : 0);
    eighth_range(cut, e, ks0, first_end);
    eighth_range(cut, e + EPW - 1, b, ks1);
  }
  const int lrow = lane >> 3, lblk = (lane & 7) ^ lrow;            // this lane's place in a load of 8 rows
  auto weight_row = [&](int r) {              // of the tile's row r; -1: there is none
    int wr = EPI == GF_SWIGLU ? tile * 8 + (r & 7) : tile * 16 + r;
    if (EPI == GF_ROPE) {
      const int per_head = rope.D >> 4, head = tile / per_head;
      wr = head * rope.D + (tile - head * per_head) * 8 + (r & 7) + (r >> 3) * (rope.D >> 1);
    }
    if (wr >= N) return -1;
    return EPI == GF_SWIGLU ? wr + (r >> 3) * up_offset : wr;
  };
  const float *wsrc[2], *xsrc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = lrow + 8 * j, wr = weight_row(r);
    wsrc[j] = W + (size_t)(wr < 0 ? 0 : wr) * ldw + lblk * 4;      // a row that does not exist is never stored
    xsrc[j] = X + (size_t)(r < M ? r : 0) * ldx + lblk * 4;
  }
  const float* zero = reinterpret_cast<const float*>(mie_zero_words) + lblk * 4;
  char* mine = ring + wave * SLOTS * SLOT_BYTES;
  auto issue = [&](int s) {
    char* base = mine + (s % SLOTS) * SLOT_BYTES;
    const int ks = ks0 + s;
    const bool kok = ks < ks1 && ks * 32 + lblk * 4 < K;
    const size_t k = (size_t)ks * 32;
    const float* src[4] = {kok ? wsrc[0] + k : zero, kok ? wsrc[1] + k : zero, kok ? xsrc[0] + k : zero, kok ? xsrc[1] + k : zero};
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const auto* from = (const __attribute__((address_space(1))) void*)src[j];
      auto* to = (__attribute__((address_space(3))) void*)(base + j * 1024);
      if (j < 2) __builtin_amdgcn_global_load_lds(from, to, 16, 0, GF_NONTEMPORAL);
      else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    }
  };
#pragma unroll
  for (int s = 0; s < SLOTS - U; ++s) issue(s);
  const int col = lane & 15, kb = lane >> 4;
  const uint32_t ring0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)mine;
  const uint32_t blk0 = ((2 * kb) ^ (col & 7)) * 16, blk1 = ((2 * kb + 1) ^ (col & 7)) * 16;
  const uint32_t wrow = ring0 + col * 128, xrow = ring0 + 2048 + (XL == 1 ? col & 7 : col) * 128;
  f32x4 main[EPW], small[EPW];
#pragma unroll
  for (int i = 0; i < EPW; ++i) main[i] = small[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int ks, const Parts& w, const Parts& x) {       // (a step beyond ks1 is zeros)
#pragma unroll
    for (int i = 0; i < EPW; ++i)
      if (EPW == 1 || (i == 0) == (ks < first_end)) {
        main[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.h, x.h, main[i], 0, 0, 0);
        small[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.m, x.h, small[i], 0, 0, 0);
        small[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.h, x.m, small[i], 0, 0, 0);
        small[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.l, x.h, small[i], 0, 0, 0);
        small[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.h, x.l, small[i], 0, 0, 0);
        small[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.m, x.m, small[i], 0, 0, 0);
      }
  };
  auto parts = [](const u32x4& a, const u32x4& b) { return split8(__builtin_bit_cast(f32x4, a), __builtin_bit_cast(f32x4, b)); };
  for (int it = 0; it < ks1 - ks0; it += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) issue(it + SLOTS - U + u);       // into the slots that were read a round ago
    MIE_VMCNT((SLOTS - U) * L);                // slots `it` (and it + 1) have landed
    const uint32_t at0 = (it % SLOTS) * SLOT_BYTES, at1 = ((it + 1) % SLOTS) * SLOT_BYTES;
    if constexpr (U == 2) {
      u32x4 f[6];
      const uint32_t w0 = wrow + at0, w1 = wrow + at1, x0 = xrow + (col < 8 ? at0 : at1);
      ring_read(w0 + blk0, w0 + blk1, w1 + blk0, w1 + blk1, x0 + blk0, x0 + blk1, f);
      const Parts x = parts(f[4], f[5]);
      step(ks0 + it, parts(f[0], f[1]), x);
      step(ks0 + it + 1, parts(f[2], f[3]), {other_half(x.h), other_half(x.m), other_half(x.l)});
    } else {
      u32x4 f[4];
      ring_read(wrow + at0 + blk0, wrow + at0 + blk1, xrow + at0 + blk0, xrow + at0 + blk1, f);
      step(ks0 + it, parts(f[0], f[1]), parts(f[2], f[3]));
    }
  }
  MIE_VMCNT(0);                                // nothing of this wave is writing the LDS any more
  __syncthreads();
#pragma unroll
  for (int i = 0; i < EPW; ++i) *reinterpret_cast<f32x4*>(s_acc + (wave * EPW + i) * 256 + lane * 4) = main[i] + small[i];
  __syncthreads();
  if (threadIdx.x >= 256) return;
  // this thread's result: x row m, column c of the tile
  const int m = threadIdx.x >> 4, c = threadIdx.x & 15;
  const int src = (((c >> 2) << 4) + m) * 4 + (c & 3);
  if (EPI == GF_PART) {
    const int n = tile * 16 + c;
    if (m >= M || n >= N) return;
#pragma unroll
    for (int q = 0; q < 2; ++q)
      out[(size_t)(2 * blockIdx.y + q) * M * N + (size_t)m * N + n] = s_acc[2 * q * 256 + src] + s_acc[(2 * q + 1) * 256 + src];
    return;
  }
  float v = 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float t = 0.f;
#pragma unroll
    for (int e = 0; e < 2; ++e) t += s_acc[(2 * q + e) * 256 + src];
    v += t;
  }
  v *= GF_UNSCALE;
  if (!finite(v) && m < M && weight_row(c) >= 0) v = plain_product(X + (size_t)m * ldx, W + (size_t)weight_row(c) * ldw, K);
  float other = 0.f;
  if (EPI == GF_SWIGLU || EPI == GF_ROPE) other = __shfl_xor(v, 8, 64);
  if (EPI == GF_ROPE) {
    if (m >= M) return;
    const int D = rope.D, half = D >> 1, per_head = D >> 4, head = tile / per_head;
    const int j = (tile - head * per_head) * 8 + (c & 7), d = j + (c >> 3) * half, slot = rope.slots[m];
    const size_t page = slot / rope.page, at = slot % rope.page;
    if (head >= rope.Hq + rope.Hkv) {
      rope.v_cache[((page * rope.Hkv + (head - rope.Hq - rope.Hkv)) * D + d) * rope.page + at] = v;
      return;
    }
    const size_t angle = (size_t)rope.positions[m] * half + j;
    float o1, o2;
    rotate_pair(c < 8 ? v : other, c < 8 ? other : v, rope.cos_t[angle], rope.sin_t[angle], o1, o2);
    float* o = head < rope.Hq ? out + (size_t)m * ldo + (size_t)head * D
                              : rope.k_cache + ((page * rope.Hkv + (head - rope.Hq)) * rope.page + at) * D;
    o[d] = c < 8 ? o1 : o2;
    return;
  }
  const int n = EPI == GF_SWIGLU ? tile * 8 + (c & 7) : tile * 16 + c;
  if (m >= M || n >= N) return;
  if (EPI == GF_SWIGLU) {
    if (c < 8) out[(size_t)m * ldo + n] = v / (1.0f + expf(-v)) * other;
  } else {
    if (bias) v += bias[n];
    float* o = out + (size_t)m * ldo + n;
    *o = EPI == GF_ADD ? *o + v : v;
  }
}

// ------------------------------------------------------------------------------------------------ many rows
// LEVELS 0: the unit is an eighth (grid.z 8), 1: a quarter (grid.z 4), 2: all of K (grid.z 1, result or C += result).
// GATED (all of K): out = silu(gate) * up; of a wave's weight rows the first half are gate rows, the others the up rows of the same columns.
// A row of W from `half` on lies `gap` rows further (gate and up rows of some columns of a larger weight; GATED: the up rows lie gap
// behind).
// In the LDS, a buffer: planes h, m, l of BM + BN rows of 64 bytes; row r's block b of 16 bytes at 4 r + (b ^ (r / 2) % 4), so that
// both the writes (a thread has 4 k) and the fragment reads (lane 16 g + r: row r, block g) spread over all banks.
template <int BM, int BN, int WR, int WC, int LEVELS, bool TAIL, bool GATED = false>
__global__ void __launch_bounds__(WR * WC * 64)
tile_f32_kernel(const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, float* __restrict__ out,
                long ldo, const float* __restrict__ bias, int add, int M, int N, int K, int half, long gap) {
  constexpr int THREADS = WR * WC * 64, WM = BM / WR, WN = BN / WC, TM = WM / 16, TN = WN / 16, ROWS = BM + BN;
  constexpr int PLANE = ROWS * 64, BUFFER = 3 * PLANE, XL = BM * 8 / THREADS, LOADS = ROWS * 8 / THREADS;      // 16-byte loads a thread and stage
  constexpr bool DOT = TM * TN <= 2;          // few matrix instructions a number that is split (see split2)
  static_assert(BM * 8 % THREADS == 0 && BN * 8 % THREADS == 0, "loads of a thread are of x or of W");
  extern __shared__ __align__(16) char gf_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * (GATED ? BN / 2 : BN);
  const KCut cut = k_cut(K);
  int ks0, ks1;
  if (LEVELS == 0) eighth_range(cut, blockIdx.z, ks0, ks1);
  else if (LEVELS == 1) { ks0 = least(blockIdx.z * cut.quarter, cut.steps); ks1 = least(ks0 + cut.quarter, cut.steps); }
  else { ks0 = 0; ks1 = cut.steps; }

  const float* src[LOADS];
  const int blk = tid & 7;                    // this thread's 4 k of every row it loads
  int at[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = (tid >> 3) + THREADS / 8 * i;
    if (i < XL) {
      src[i] = X + (size_t)(m0 + r < M ? m0 + r : M - 1) * ldx + blk * 4;
    } else {
      const int c = r - BM, w = c / WN, in = c % WN;
      int row = GATED ? n0 + w * (WN / 2) + in % (WN / 2) : n0 + c;
      row = row < N ? row : N - 1;
      src[i] = W + (size_t)(row + ((GATED ? in >= WN / 2 : row >= half) ? gap : 0)) * ldw + blk * 4;
    }
    at[i] = r * 64 + ((blk >> 1) ^ ((r >> 1) & 3)) * 16 + (blk & 1) * 8;
  }
  f32x4 staged[2][LOADS];                     // two steps on their way
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](f32x4 (&staged)[LOADS], int ks) {      // step ks; TAIL: what lies beyond K is zero, its load is from the row's end
    const int k = TAIL ? least(ks * 32, K - 4 - blk * 4) : ks * 32;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) staged[i] = *reinterpret_cast<const f32x4*>(src[i] + k);
    if (TAIL && ks * 32 + blk * 4 >= K) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) staged[i] = none;
    }
  };
  auto put = [&](const f32x4 (&staged)[LOADS], int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      uint2 h, m, l;
      split2<DOT>(staged[i][0], staged[i][1], h.x, m.x, l.x);
      split2<DOT>(staged[i][2], staged[i][3], h.y, m.y, l.y);
      char* p = gf_lds + buf * BUFFER + at[i];
      *reinterpret_cast<uint2*>(p) = h;
      *reinterpret_cast<uint2*>(p + PLANE) = m;
      *reinterpret_cast<uint2*>(p + 2 * PLANE) = l;
    }
  };

  f32x4 main[TN][TM], small[TN][TM], quarter[LEVELS >= 1 ? TN : 1][LEVELS >= 1 ? TM : 1], total[LEVELS >= 2 ? TN : 1][LEVELS >= 2 ? TM : 1];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) {
      main[a][b] = small[a][b] = none;
      if (LEVELS >= 1) quarter[LEVELS >= 1 ? a : 0][LEVELS >= 1 ? b : 0] = none;
      if (LEVELS >= 2) total[LEVELS >= 2 ? a : 0][LEVELS >= 2 ? b : 0] = none;
    }
  const int wm = (wave % WR) * WM, wn = (wave / WR) * WN;
  const int r16 = lane & 15, g = lane >> 4;
  const int frag = r16 * 64 + (g ^ ((r16 >> 1) & 3)) * 16;

  int quarter_end = LEVELS >= 2 ? least(cut.quarter, cut.steps) : ks1;
  int eighth_end = LEVELS >= 1 ? least(ks0 + cut.eighth, quarter_end) : ks1;
  bf16x8 wf[3][TN], xf[3][TM];
  auto take = [&](int p, int buf) {           // this wave's fragments of plane p
    const char* base = gf_lds + buf * BUFFER + p * PLANE + frag;
#pragma unroll
    for (int a = 0; a < TN; ++a) wf[p][a] = *reinterpret_cast<const bf16x8*>(base + (BM + wn + a * 16) * 64);
#pragma unroll
    for (int b = 0; b < TM; ++b) xf[p][b] = *reinterpret_cast<const bf16x8*>(base + (wm + b * 16) * 64);
  };
  auto products = [&](int p, int q, f32x4 (&acc)[TN][TM]) {
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[p][a], xf[q][b], acc[a][b], 0, 0, 0);
  };
  if (ks0 < ks1) {                            // (behind the unit's end the last step once more, which nobody multiplies)
    fetch(staged[0], ks0);
    fetch(staged[1], least(ks0 + 1, ks1 - 1));
    put(staged[0], 0);
    fetch(staged[0], least(ks0 + 2, ks1 - 1));
  }
  __syncthreads();
  int buf = 0;
  auto stage = [&](int ks, f32x4 (&next)[LOADS]) {       // next: the registers that hold step ks + 1
#pragma unroll
    for (int p = 0; p < 3; ++p) take(p, buf);
    buf ^= 1;
    put(next, buf);                           // (everybody has read this buffer before the last barrier)
    fetch(next, least(ks + 3, ks1 - 1));
    products(0, 0, main);
    products(1, 0, small);
    products(0, 1, small);
    products(2, 0, small);
    products(0, 2, small);
    products(1, 1, small);
    // matrix instructions and the splitting in turn (two of it each: 172 us for 167 at 512 rows of [11264, 2048], in tiles of 64 x 64 46.0
    // for 44.8 at 512 of [2560, 2048])
#pragma unroll
    for (int i = 0; i < 6 * TM * TN; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, DOT ? 1 : 3, 0);
    }
    if (LEVELS >= 1 && ks + 1 == eighth_end) {
      const bool quarter_done = LEVELS >= 2 && eighth_end == quarter_end;
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) {
          f32x4& q = quarter[LEVELS >= 1 ? a : 0][LEVELS >= 1 ? b : 0];
          q += main[a][b] + small[a][b];
          main[a][b] = small[a][b] = none;
          if (quarter_done) {
            total[LEVELS >= 2 ? a : 0][LEVELS >= 2 ? b : 0] += q;
            q = none;
          }
        }
      if (quarter_done) quarter_end = least(quarter_end + cut.quarter, cut.steps);
      eighth_end = least(eighth_end + cut.eighth, quarter_end);
    }
    __syncthreads();
  };
  for (int ks = ks0; ks < ks1;) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      stage(ks, staged[j ^ 1]);
      if (++ks >= ks1) break;
    }
  }
  // acc[i] of lane (r16, g): weight row 4 g + i of the 16, x row r16
  float* dst = out + (LEVELS < 2 ? (size_t)blockIdx.z * M * N : 0);
  const long ld = LEVELS < 2 ? N : ldo;
#pragma unroll
  for (int b = 0; b < TM; ++b) {
    const int m = m0 + wm + b * 16 + r16;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < TN; ++a) {
      if constexpr (GATED) {
        const int n = n0 + wn / 2 + a * 16 + 4 * g;
        if (a >= TN / 2 || n >= N) continue;
        f32x4 v = total[a][b] * GF_UNSCALE, u = total[(a + TN / 2) % TN][b] * GF_UNSCALE;
        again_if_not_finite(v, X + (size_t)m * ldx, W + (size_t)n * ldw, ldw, K);
        again_if_not_finite(u, X + (size_t)m * ldx, W + (size_t)(n + gap) * ldw, ldw, K);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + expf(-v[i])) * u[i];
        *reinterpret_cast<f32x4*>(dst + (size_t)m * ld + n) = v;
        continue;
      }
      const int n = n0 + wn + a * 16 + 4 * g;
      if (n >= N) continue;                   // N is a multiple of 4
      f32x4 v = LEVELS == 0 ? main[a][b] + small[a][b] : LEVELS == 1 ? quarter[LEVELS >= 1 ? a : 0][LEVELS >= 1 ? b : 0]
                                                                     : total[LEVELS >= 2 ? a : 0][LEVELS >= 2 ? b : 0];
      f32x4* o = reinterpret_cast<f32x4*>(dst + (size_t)m * ld + n);
      if (LEVELS == 2) {
        v *= GF_UNSCALE;
        again_if_not_finite(v, X + (size_t)m * ldx, W + (size_t)n * ldw, ldw, K);
        if (bias) v += *reinterpret_cast<const f32x4*>(bias + n);
        if (add) v = *o + v;
      }
      *o = v;
    }
  }
}

// The sums of PARTS (4 quarters or 8 eighths) units joined in the order above, then stored, added into `out`, or, with
// gate sums in columns [0, N) and up sums in [N, 2 N) (`part` has 2 N columns), silu(gate) * up.
template <int PARTS>
__device__ __forceinline__ f32x4 join_parts(const f32x4* p, size_t stride) {
  f32x4 v[PARTS];
#pragma unroll
  for (int i = 0; i < PARTS; ++i) v[i] = p[i * stride];
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  f32x4 total = none;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 t = none;
    if (PARTS == 4) t = v[q];
    else {
#pragma unroll
      for (int e = 0; e < 2; ++e) t += v[(2 * q + e) % PARTS];
    }
    total += t;
  }
  return total * GF_UNSCALE;
}

template <int PARTS, int EPI>
__global__ void __launch_bounds__(256)
reduce_f32_kernel(const float* __restrict__ part, float* __restrict__ out, long ldo, const float* __restrict__ bias, int M, int N,
                  const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, int K, long up_rows) {
  const int cols = EPI == GF_SWIGLU ? 2 * N : N, per_row = N >> 2;
  const size_t stride = (size_t)M * cols / 4, total = (size_t)M * per_row;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    const size_t m = e / per_row, n = (e - m * per_row) * 4;
    const f32x4* p = reinterpret_cast<const f32x4*>(part + m * cols + n);
    f32x4 v = join_parts<PARTS>(p, stride);
    again_if_not_finite(v, X + m * ldx, W + n * ldw, ldw, K);
    f32x4* o = reinterpret_cast<f32x4*>(out + m * ldo + n);
    if (EPI == GF_SWIGLU) {
      f32x4 u = join_parts<PARTS>(p + (N >> 2), stride);
      again_if_not_finite(u, X + m * ldx, W + (up_rows + n) * ldw, ldw, K);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + expf(-v[i])) * u[i];
      *o = v;
    } else {
      if (bias) v += *reinterpret_cast<const f32x4*>(bias + n);
      *o = EPI == GF_ADD ? *o + v : v;
    }
  }
}

// The same joined into the 32-bit stream [M, N], with the RMSNorm that reads the stream next: y [M, N] = stream * rsqrt(mean(stream^2) +
// eps) * g.  A workgroup a row; threads, groups of four and the order of the squares' sum are those of the add + norm kernel
// (embed_norm.hip), so a row has the same bits whichever of the two makes it.  Rows of up to 4,096 numbers: of more, a thread's eight
// groups and their parts do not fit the registers, and joining by itself has more workgroups than rows (product, add and norm, this
// kernel / two: 20 rows of [6144, 2048] 28.3 / 25.4 us, of [8192, 2048] 32.0 / 28.9, of [5120, 13824] 88.0 / 85.5; 512 rows of [5120, 5120]
// 193.5 / 189.0; but of [4096, 4096] 20 rows 27.7 / 28.4, 512 113.3 / 116.8).
constexpr int GF_NORM_THREADS = 256, GF_NORM_MOST = 4 * GF_NORM_THREADS * 4;
__device__ __forceinline__ f32x4 norm_weight4(const float* g) { return *reinterpret_cast<const f32x4*>(g); }
__device__ __forceinline__ f32x4 norm_weight4(const bf16* g) {
  const uint2 u = *reinterpret_cast<const uint2*>(g);
  return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xFFFF0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xFFFF0000u)};
}
template <int PARTS, typename TW, int VEC>
__global__ void __launch_bounds__(GF_NORM_THREADS)
reduce_add_norm_kernel(const float* __restrict__ part, float* __restrict__ stream, const TW* __restrict__ g, float* __restrict__ y, int M,
                       int N, float eps, const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, int K) {
  __shared__ float scratch[16];
  const size_t m = blockIdx.x, stride = (size_t)M * N / 4;
  f32x4 r[VEC], w[VEC], old[VEC];
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    const int i = (threadIdx.x + k * GF_NORM_THREADS) * 4;
    r[k] = w[k] = old[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (i < N) {
      old[k] = *reinterpret_cast<const f32x4*>(stream + m * N + i);
      w[k] = norm_weight4(g + i);
      r[k] = join_parts<PARTS>(reinterpret_cast<const f32x4*>(part + m * N + i), stride);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    const int i = (threadIdx.x + k * GF_NORM_THREADS) * 4;
    if (i < N) {
      again_if_not_finite(r[k], X + m * ldx, W + (size_t)i * ldw, ldw, K);
      r[k] = old[k] + r[k];
      *reinterpret_cast<f32x4*>(stream + m * N + i) = r[k];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) ss = fmaf(r[k][j], r[k][j], ss);
  }
  const float total = block_sum(ss, scratch);
  const float rstd = 1.0f / sqrtf(total / (float)N + eps);
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    const int i = (threadIdx.x + k * GF_NORM_THREADS) * 4;
    if (i < N) {
      f32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = r[k][j] * rstd * w[k][j];
      *reinterpret_cast<f32x4*>(y + m * N + i) = o;
    }
  }
}

// ------------------------------------------------------------------------------------------------ host
MIE_EXPORT const char* gemm_f32_last_error() { return g_mie_error; }

static int check_operands(const char* what, const void* X, long ldx, const void* W, long ldw, const void* out, long ldo, int N, int K) {
  if (K <= 0 || (K & 3) || (N & 3)) MIE_FAIL("%s: K = %d and N = %d must be positive multiples of 4", what, K, N);
  if (ldx < K || ldw < K || ldo < N || (ldx & 3) || (ldw & 3) || (ldo & 3)) MIE_FAIL("%s: leading dims %ld, %ld, %ld for K %d, N %d", what, ldx, ldw, ldo, K, N);
  if (((uintptr_t)X | (uintptr_t)W | (uintptr_t)out) & 15) MIE_FAIL("%s: operands must be 16-byte aligned", what);
  return 0;
}

// The tile of a workgroup and how many units K is cut into (1, 4 or 8) for M rows (more than 16): the cheapest by what was
// measured (MI355X, 17 to 2,048 rows of [11264, 2048], [2560, 2048], [2048, 2048], [2048, 5632], [768, 1536] and two small
// weights).  A step of 32 k costs a compute unit fixed + each x the workgroups it has, whether they run side by side or in
// turn; a start 2.9 us; units' sums cost a kernel of 1.9 us and 1.6 us a million of them.  Large tiles split and read an operand for
// more outputs, small ones and units of K give every compute unit work: us of 128 x 128 / 128 x 64 / 64 x 64, each at its best cut: 512
// rows of [11264, 2048] 176 / 169 / 180, 2,048 rows 543 / 638 / 684, 512 rows of [2048, 2048] 35 / 40 / 39, 100 rows 20 / 17 / 16, 32 rows of
// [2048, 5632] 36 / 27 / 20.  gated: the product's gate and up columns are joined where the units' sums are, else by a pass of its own.
// The units' sums take at most GF_PART_FLOATS, 128 MiB: 512 rows of [11264, 2048] have 92 MB of them (quarters 187 us, uncut 212 and a
// pass of 10), and without a bound their memory would grow with the weight's size to gigabytes.
constexpr long GF_PART_FLOATS = 1L << 25;
constexpr struct { int bm, bn; float fixed, each; } GF_TILES[3] = {{128, 128, 0.f, 1.40f}, {128, 64, 0.f, 0.87f}, {64, 64, 0.07f, 0.45f}};
struct TilePlan {
  int tile, units;
};
static TilePlan tile_plan(int M, int N, int K, bool gated, float* cost = nullptr) {
  TilePlan best = {2, 8};
  float least_us = 1e30f;
  const KCut cut = k_cut(K);
  const float outputs = (float)M * N;
  for (int t = 0; t < 3; ++t) {
    const long tiles = (long)((M + GF_TILES[t].bm - 1) / GF_TILES[t].bm) * ((N + GF_TILES[t].bn - 1) / GF_TILES[t].bn);
    for (int units = 1; units <= 8; units += units == 1 ? 3 : 4) {
      if (units > 1 && units * (long)M * N > GF_PART_FLOATS) break;
      const int steps = units == 1 ? cut.steps : units == 4 ? cut.quarter : cut.eighth;
      const long each = (tiles * units + mie_compute_units() - 1) / mie_compute_units();
      float us = 2.9f + steps * (GF_TILES[t].fixed + GF_TILES[t].each * each);
      if (units > 1 || gated) us += 1.9f + outputs * units * 1.6e-6f;
      if (us < least_us) {
        least_us = us;
        best = {t, units};
      }
    }
  }
  if (cost) *cost = least_us;
  return best;
}

// Columns of a gated product [M, N] (N gate and N up rows of W) that are made by uncut 128 x 128 tiles with silu(gate) * up behind them: as
// many as fill whole rounds of the grid, where those and the others (the plan above) are estimated to take less than the plan for all
// of them.  0: none.  A round uncut costs a tile's steps and no sums of parts in memory: 512 rows of [11264, 2048] are 256 tiles, one
// round, and 96 that the plan cuts into quarters, 158 us; all in quarters, 5.5 rounds of 6 and 92 MB of sums, 178; 384 rows 115 and 150, 512 of [28672, 4096] 695 and 776.
static int whole_columns(int M, int N, int K) {
  float all_us, rest_us = 0.f;
  tile_plan(M, 2 * N, K, true, &all_us);
  const int mt = (M + 127) / 128, nt = (N + 63) / 64, cu = mie_compute_units();
  const int rounds = (int)((long)mt * nt / cu), whole = rounds > 0 ? (int)((long)cu * rounds / mt) * 64 : 0;
  if (M <= 16 || whole <= 0) return 0;
  const int rest = whole < N ? N - whole : 0;
  if (rest && tile_plan(M, 2 * rest, K, true, &rest_us).units == 1) return 0;
  return rounds * (2.9f + k_cut(K).steps * GF_TILES[0].each) + rest_us < 0.97f * all_us ? N - rest : 0;
}
MIE_EXPORT int mie_f32_whole_columns(int M, int N, int K) { return whole_columns(M, N, K); }
MIE_EXPORT int mie_f32_units(int M, int N, int K, int gated) { return tile_plan(M, N, K, gated != 0).units; }

template <int EPI>
static int launch_skinny(const float* X, long ldx, const float* W, long ldw, float* out, long ldo, const float* bias, int M, int N,
                         int K, hipStream_t s, const RopeArgs& rope = RopeArgs{}) {
  const int tiles = EPI == GF_SWIGLU ? (N + 7) / 8 : (N + 15) / 16;
  // 8 waves, 144 KB of ring (128 from 9 rows on) and one workgroup a compute unit, or 4 waves, 48 KB and three
#define GF_SKINNY(WAVES, SLOTS, XL)                                                                                       \
  {                                                                                                                       \
    auto kernel = skinny_f32_kernel<EPI, WAVES, SLOTS, XL>;                                                               \
    constexpr int lds = WAVES * SLOTS * (2 + XL) * 1024;                                                                  \
    if (mie_allow_lds((const void*)kernel, lds, "gemm_f32")) return -1;                                                   \
    hipLaunchKernelGGL(kernel, dim3(tiles, EPI == GF_PART ? 2 : 1), dim3(WAVES * 64), lds, s, X, ldx, W, ldw, out, ldo, bias, M, N, K, N, rope); \
  }
  if constexpr (EPI == GF_PART) {             // (few slots: those behind a wave's few steps bring zeros; 6 to 12 are up to 1.4 us slower)
    if (M <= 8) GF_SKINNY(4, 4, 1) else GF_SKINNY(4, 4, 2)
  } else if (tiles <= 256) {
    if (M <= 8) GF_SKINNY(8, 6, 1) else GF_SKINNY(8, 4, 2)
  } else {
    if (M <= 8) GF_SKINNY(4, 4, 1) else GF_SKINNY(4, 3, 2)
  }
#undef GF_SKINNY
  MIE_CHECK_LAUNCH("skinny_f32");
  return 0;
}

template <int BM, int BN, int WR, int WC, int LEVELS>
static int launch_tile(const float* X, long ldx, const float* W, long ldw, float* out, long ldo, const float* bias, int add, int M,
                       int N, int K, int units, hipStream_t s, int half = 0x7FFFFFFF, long gap = 0) {
  constexpr int lds = 2 * (BM + BN) * 192;
  auto kernel = K & 31 ? tile_f32_kernel<BM, BN, WR, WC, LEVELS, true> : tile_f32_kernel<BM, BN, WR, WC, LEVELS, false>;
  if ((M + BM - 1) / BM > 65535) MIE_FAIL("gemm_f32: M = %d is beyond the grid", M);
  if (mie_allow_lds((const void*)kernel, lds, "gemm_f32")) return -1;
  hipLaunchKernelGGL(kernel, dim3((N + BN - 1) / BN, (M + BM - 1) / BM, units), dim3(WR * WC * 64), lds, s, X, ldx, W, ldw, out, ldo, bias, add, M, N, K, half, gap);
  MIE_CHECK_LAUNCH("tile_f32");
  return 0;
}

static int launch_tiles(const float* X, long ldx, const float* W, long ldw, float* out, long ldo, const float* bias, int add, int M,
                        int N, int K, const TilePlan& plan, hipStream_t s, int half = 0x7FFFFFFF, long gap = 0) {
#define GF_TILE(BM, BN, WR, WC)                                                                                             \
  return plan.units == 1   ? launch_tile<BM, BN, WR, WC, 2>(X, ldx, W, ldw, out, ldo, bias, add, M, N, K, 1, s, half, gap)           \
         : plan.units == 4 ? launch_tile<BM, BN, WR, WC, 1>(X, ldx, W, ldw, out, ldo, bias, add, M, N, K, 4, s, half, gap)           \
                           : launch_tile<BM, BN, WR, WC, 0>(X, ldx, W, ldw, out, ldo, bias, add, M, N, K, 8, s, half, gap)
  if (plan.tile == 0) GF_TILE(128, 128, 4, 2);
  if (plan.tile == 1) GF_TILE(128, 64, 4, 2);
  GF_TILE(64, 64, 2, 4);
#undef GF_TILE
}

template <int EPI>
static int launch_reduce(int units, const float* part, float* out, long ldo, const float* bias, int M, int N, const float* X, long ldx,
                         const float* W, long ldw, int K, hipStream_t s, long up_rows = 0) {
  if (!up_rows) up_rows = N;
  long blocks = ((long)M * (N / 4) + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (units == 4)
    hipLaunchKernelGGL((reduce_f32_kernel<4, EPI>), dim3((unsigned)blocks), dim3(256), 0, s, part, out, ldo, bias, M, N, X, ldx, W, ldw, K, up_rows);
  else
    hipLaunchKernelGGL((reduce_f32_kernel<8, EPI>), dim3((unsigned)blocks), dim3(256), 0, s, part, out, ldo, bias, M, N, X, ldx, W, ldw, K, up_rows);
  MIE_CHECK_LAUNCH("reduce_f32");
  return 0;
}

// epi 0: out = x W^T (+ bias), 1: out += x W^T (+ bias), 2: out = silu(gate) * up with W = [gate rows (N of them); up rows].
// part: mie_f32_units(M, columns of x W^T, K, epi == 2) * M * columns floats, 16-byte aligned, when M > 16 and that is more than
// one unit.
MIE_EXPORT int mie_gemm_f32(const float* X, long ldx, const float* W, long ldw, float* out, long ldo, int epi, const float* bias,
                            float* part, int M, int N, int K, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (epi < GF_STORE || epi > GF_SWIGLU) MIE_FAIL("gemm_f32: epilogue code %d", epi);
  if (epi == GF_SWIGLU && bias) MIE_FAIL("gemm_f32: no bias beside the gated epilogue");
  if (((uintptr_t)bias | (uintptr_t)part) & 15) MIE_FAIL("gemm_f32: bias and partial sums must be 16-byte aligned");
  if (check_operands("gemm_f32", X, ldx, W, ldw, out, ldo, N, K)) return -1;
  if (M <= 16)
    return epi == GF_STORE ? launch_skinny<GF_STORE>(X, ldx, W, ldw, out, ldo, bias, M, N, K, s)
         : epi == GF_ADD ? launch_skinny<GF_ADD>(X, ldx, W, ldw, out, ldo, bias, M, N, K, s)
                         : launch_skinny<GF_SWIGLU>(X, ldx, W, ldw, out, ldo, bias, M, N, K, s);
  const int cols = epi == GF_SWIGLU ? 2 * N : N;
  const TilePlan plan = tile_plan(M, cols, K, epi == GF_SWIGLU);
  const int units = plan.units;
  if (units == 1 && epi != GF_SWIGLU) return launch_tiles(X, ldx, W, ldw, out, ldo, bias, epi == GF_ADD, M, N, K, plan, s);
  if (epi == GF_SWIGLU && units == 1) MIE_FAIL("gemm_f32: %d rows of %d columns are one unit: take the product and silu_mul", M, cols);
  if (!part) MIE_FAIL("gemm_f32: %d units need memory for their sums", units);
  if (launch_tiles(X, ldx, W, ldw, part, cols, nullptr, 0, M, cols, K, plan, s)) return -1;
  return epi == GF_STORE ? launch_reduce<GF_STORE>(units, part, out, ldo, bias, M, N, X, ldx, W, ldw, K, s)
       : epi == GF_ADD ? launch_reduce<GF_ADD>(units, part, out, ldo, bias, M, N, X, ldx, W, ldw, K, s)
                       : launch_reduce<GF_SWIGLU>(units, part, out, ldo, bias, M, N, X, ldx, W, ldw, K, s);
}

// out [M, N] = silu(x Wg^T) * (x Wu^T), its first mie_f32_whole_columns(M, N, K) columns (not 0) by uncut tiles, the others in
// mie_f32_units(M, 2 * others, K, 1) units, whose sums take units * M * 2 * others floats of part (16-byte aligned).
MIE_EXPORT int mie_gemm_f32_gated(const float* X, long ldx, const float* W, long ldw, float* out, long ldo, float* part, int M, int N, int K,
                                  hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands("gemm_f32_gated", X, ldx, W, ldw, out, ldo, N, K)) return -1;
  const int whole = whole_columns(M, N, K), rest = N - whole;
  if (!whole) MIE_FAIL("gemm_f32_gated: no columns of %d rows of [%d, %d] fill the grid", M, 2 * N, K);
  if (rest && (!part || ((uintptr_t)part & 15))) MIE_FAIL("gemm_f32_gated: the units' sums need memory, 16-byte aligned");
  constexpr int lds = 2 * (128 + 128) * 192;
  auto kernel = K & 31 ? tile_f32_kernel<128, 128, 4, 2, 2, true, true> : tile_f32_kernel<128, 128, 4, 2, 2, false, true>;
  if ((M + 127) / 128 > 65535) MIE_FAIL("gemm_f32: M = %d is beyond the grid", M);
  if (mie_allow_lds((const void*)kernel, lds, "gemm_f32")) return -1;
  hipLaunchKernelGGL(kernel, dim3((whole + 63) / 64, (M + 127) / 128, 1), dim3(512), lds, s, X, ldx, W, ldw, out, ldo, nullptr, 0, M, whole, K,
                     0, (long)N);
  MIE_CHECK_LAUNCH("tile_f32");
  if (!rest) return 0;
  const TilePlan plan = tile_plan(M, 2 * rest, K, true);
  const float* Wr = W + (size_t)whole * ldw;
  if (launch_tiles(X, ldx, Wr, ldw, part, 2 * rest, nullptr, 0, M, 2 * rest, K, plan, s, rest, (long)whole)) return -1;
  return launch_reduce<GF_SWIGLU>(plan.units, part, out + whole, ldo, nullptr, M, rest, X, ldx, Wr, ldw, K, s, N);
}

// How many units K is cut into where the product is added into a stream whose RMSNorm is wanted next (mie_gemm_f32_add_norm), 0: the
// product with the add and the norm by themselves.  More than 16 rows: the units that the product is cut into anyway.  Up to 16
// rows: quarters, two a workgroup, while that gives every compute unit at most one workgroup and a wave some steps.
MIE_EXPORT int mie_f32_norm_units(int M, int N, int K) {
  if (M <= 0 || (N & 3) || N > GF_NORM_MOST || K <= 0) return 0;
  if (M <= 16) return K >= 1024 && 2 * ((N + 15) / 16) <= mie_compute_units() ? 4 : 0;
  const int units = tile_plan(M, N, K, false).units;
  return units > 1 ? units : 0;
}

// stream [M, N] += x W^T and y [M, N] = RMSNorm(stream) with weight g (float32 if g_f32, else bfloat16).  part: mie_f32_norm_units(M, N, K)
// (which is not 0) * M * N floats.  Everything 16-byte aligned.
MIE_EXPORT int mie_gemm_f32_add_norm(const float* X, long ldx, const float* W, long ldw, float* stream, const void* g, int g_f32, float* y,
                                     float* part, int M, int N, int K, float eps, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  const int units = mie_f32_norm_units(M, N, K);
  if (!units) MIE_FAIL("gemm_f32_add_norm: %d rows of [%d, %d] are not cut into units", M, N, K);
  if (!stream || !g || !y || !part || ((uintptr_t)g | (uintptr_t)y | (uintptr_t)part) & 15) MIE_FAIL("gemm_f32_add_norm: operands must be 16-byte aligned");
  if (check_operands("gemm_f32_add_norm", X, ldx, W, ldw, stream, N, N, K)) return -1;
  if (M <= 16) {
    if (launch_skinny<GF_PART>(X, ldx, W, ldw, part, N, nullptr, M, N, K, s)) return -1;
  } else if (launch_tiles(X, ldx, W, ldw, part, N, nullptr, 0, M, N, K, tile_plan(M, N, K, false), s)) return -1;
  const int groups = (N / 4 + GF_NORM_THREADS - 1) / GF_NORM_THREADS;
#define GF_NORM(PARTS, TW, VEC)                                                                                                  \
  hipLaunchKernelGGL((reduce_add_norm_kernel<PARTS, TW, VEC>), dim3(M), dim3(GF_NORM_THREADS), 0, s, part, stream, (const TW*)g, y, M, N, \
                     eps, X, ldx, W, ldw, K)
#define GF_NORM_VEC(PARTS, TW)            \
  if (groups <= 2) GF_NORM(PARTS, TW, 2); \
  else GF_NORM(PARTS, TW, 4)
  if (units == 4) {
    if (g_f32) { GF_NORM_VEC(4, float); } else { GF_NORM_VEC(4, bf16); }
  } else {
    if (g_f32) { GF_NORM_VEC(8, float); } else { GF_NORM_VEC(8, bf16); }
  }
#undef GF_NORM_VEC
#undef GF_NORM
  MIE_CHECK_LAUNCH("gemm_f32_add_norm");
  return 0;
}

// The q/k/v projection of up to 16 rows with what follows it: W [(Hq + 2 Hkv) D, K]; q and k rotated (half-split pairs over the
// whole head), q to q_out [M, ldq], k and v to cache slot slots[m].  The tile's 16 columns are 8 pairs, so both halves of a
// pair are 8 lanes apart; the kernel that did this alone cost 4.6 us a layer, most of it its start (a step of 4 rows of 512
// keys, 22 layers of width 2,048: 1,784 -> 1,691 us, MI355X).
MIE_EXPORT int mie_qkv_rope_f32(const float* X, long ldx, const float* W, long ldw, float* q_out, long ldq, const int* positions,
                                const float* cos_t, const float* sin_t, const int* slots, float* k_cache, float* v_cache, int M,
                                int Hq, int Hkv, int D, int page, int K, hipStream_t s) {
  if (M <= 0) return 0;
  if (M > 16) MIE_FAIL("qkv_rope_f32: %d rows (at most 16)", M);
  if (Hq <= 0 || Hkv <= 0 || page <= 0 || D <= 0 || (D & 15)) MIE_FAIL("qkv_rope_f32: heads %d / %d of %d, page %d", Hq, Hkv, D, page);
  if (!positions || !cos_t || !sin_t || !slots || !k_cache || !v_cache || !q_out) MIE_FAIL("qkv_rope_f32: null operand");
  if (ldq < (long)Hq * D) MIE_FAIL("qkv_rope_f32: q leading dim %ld for %d columns", ldq, Hq * D);
  const int N = (Hq + 2 * Hkv) * D;
  if (check_operands("qkv_rope_f32", X, ldx, W, ldw, X, N, N, K)) return -1;      // (q_out's place needs no alignment)
  return launch_skinny<GF_ROPE>(X, ldx, W, ldw, q_out, ldq, nullptr, M, N, K, s,
                                RopeArgs{positions, cos_t, sin_t, slots, k_cache, v_cache, Hq, Hkv, D, page});
}
