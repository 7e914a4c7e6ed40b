// Matrix products of the float32 path on the 32-bit matrix instruction.
//
//   y[m, n] = sum_k x[m, k] W[n, k]          x [M, K], W [N, K], y [M, N] float32
//
// One order of summation for every kernel here, whatever M is, so that a row's result is bit-identical however the
// batch around it is cut.  K is taken in steps of 16 (four v_mfma_f32_16x16x4_f32: the matrix unit adds true 32-bit
// products); the steps are cut into four quarters and every quarter into four segments (sizes from K alone).  A
// segment is one chain of matrix instructions, a quarter is ((s0 + s1) + s2) + s3 and the result ((q0 + q1) + q2) + q3:
// the rounding error of a long sum grows with K / 16 + 16 terms.  Inside a step the sixteen k are taken as the
// instruction takes them from 16-byte pieces: instruction j multiplies k = j, 4 + j, 8 + j, 12 + j.
//
// skinny_f32_kernel (M <= 16): the weights' bytes bound it.  A workgroup owns 16 rows of W; a wave streams a contiguous
//   part of K through a ring of its own in the LDS, filled by loads that write the LDS directly: 8 rows of 32 k a load, lane
//   8 r + b (whole cache lines, where the instruction's own order would touch 16 lines a quarter wave), block b of 16 bytes at
//   8 r + (b ^ r % 8), so that the fragment reads spread over all banks; segments meet in the LDS at the end.  Eight waves a
//   workgroup (a deeper queue of loads a compute unit) while the tiles do not fill the compute units, four from there on.
// tile_f32_kernel (M > 16): the matrix unit bounds it.  BM x BN outputs a workgroup, two buffers of 32 k in the LDS, the
//   next stage on its way to registers while one is multiplied; several waves a SIMD, since one alone waits out its reads
//   of the LDS (128 x 128 on four waves: 44 to 60 TFLOP/s).  Few tiles: the grid is also cut over quarters or segments,
//   whose sums go to memory and meet in reduce_f32_kernel.
//
// Measured on MI355X against the vector-unit kernel gemm_nt_kernel (gemm.hip) with its 64 x 64 tiles walking all of K:
// a step's products at 4 rows 47 -> 6.1 ms with the kernels beside them unchanged, and whole cache lines a load (half lines and
// 16 rows of x before) took a whole step 2,057 -> 1,853 us; 512 rows of [2048, 2048] 330 -> 50 us, of [11264, 2048] 475 -> 225
// (105 TFLOP/s of the 157 that the 32-bit matrix unit has).  Error against 64 bits of a 22-layer step's logits 2.5e-6 -> 2.1e-6.
#include "launch.hpp"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __align__(128) const uint32_t mie_zero_words[32] = {0};

// The cut of K, in steps of 16: quarter q is steps [q * quarter, min((q + 1) * quarter, steps)), a segment `segment` steps.
struct KCut {
  int steps, quarter, segment;
};
__host__ __device__ __forceinline__ KCut k_cut(int K) {
  KCut c;
  c.steps = (K + 15) / 16;
  c.quarter = (c.steps + 3) / 4;
  c.segment = (c.quarter + 3) / 4;
  return c;
}
__host__ __device__ __forceinline__ int least(int a, int b) { return a < b ? a : b; }

// steps [begin, end) of segment s (0 .. 15); may be empty
__host__ __device__ __forceinline__ void segment_range(const KCut& c, int s, int& begin, int& end) {
  const int q0 = least((s >> 2) * c.quarter, c.steps), q1 = least(q0 + c.quarter, c.steps);
  begin = least(q0 + (s & 3) * c.segment, q1);
  end = least(begin + c.segment, q1);
}

__device__ __forceinline__ f32x4 step_mfma(const f32x4& w, const f32x4& x, f32x4 acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], acc, 0, 0, 0);
  return acc;
}

enum { GF_STORE = 0, GF_ADD = 1, GF_SWIGLU = 2, GF_ROPE = 3 };

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
constexpr int GF_U = 2;                       // steps a slot of a wave's ring

// The fragments of a slot out of the LDS, read and waited for in one piece of assembly: the compiler knows nothing of the
// loads that write the LDS and would wait for all of them at a read it could see.
__device__ __forceinline__ void ring_read(uint32_t w0, uint32_t x0, uint32_t w1, uint32_t x1, u32x4 (&f)[4]) {
  asm volatile(
    "ds_read_b128 %0, %4\n\t"
    "ds_read_b128 %1, %5\n\t"
    "ds_read_b128 %2, %6\n\t"
    "ds_read_b128 %3, %7\n\t"
    "s_waitcnt lgkmcnt(0)"
    : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3])
    : "v"(w0), "v"(x0), "v"(w1), "v"(x1)
    : "memory");
}

// XL: loads of x a slot: one for up to 8 rows (columns 8 to 15 of the tile then take rows 0 to 7 again), else two.
// SWIGLU: W is gate rows then up rows (up_offset apart); a tile is 8 gate rows and the 8 up rows of the same columns.
template <int EPI, int WAVES, int SLOTS, int XL>
__global__ void __launch_bounds__(WAVES * 64)
skinny_f32_kernel(const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, float* __restrict__ out,
                  long ldo, const float* __restrict__ bias, int M, int N, int K, int up_offset, RopeArgs rope) {
  constexpr int SPW = 16 / WAVES;             // segments a wave
  constexpr int L = 2 + XL, SLOT_BYTES = L * 1024;       // loads a slot: 16 weight rows of 128 bytes, then the x rows
  static_assert((SLOTS - 1) * L <= 63, "more loads in flight than the counter holds");
  extern __shared__ __align__(16) char gf_lds[];
  char* ring = gf_lds;                                            // WAVES * SLOTS slots
  float* s_acc = reinterpret_cast<float*>(gf_lds);                // [16][256], once every wave is done with its ring
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tile = blockIdx.x;
  const KCut cut = k_cut(K);
  int seg_end[SPW], ks0, ks1;
  {
    int b, e;
    segment_range(cut, wave * SPW, ks0, e);
#pragma unroll
    for (int i = 0; i < SPW; ++i) segment_range(cut, wave * SPW + i, b, seg_end[i]);
    ks1 = seg_end[SPW - 1];
  }
  const int lrow = lane >> 3, lblk = (lane & 7) ^ lrow;            // this lane's place in a load of 8 rows
  const float *wsrc[2], *xsrc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = lrow + 8 * j;
    int wr = EPI == GF_SWIGLU ? tile * 8 + (r & 7) : tile * 16 + r;
    if (EPI == GF_ROPE) {
      const int per_head = rope.D >> 4, head = tile / per_head;
      wr = head * rope.D + (tile - head * per_head) * 8 + (r & 7) + (r >> 3) * (rope.D >> 1);
    }
    if (wr >= N) wr = 0;                      // a row that does not exist is never stored
    if (EPI == GF_SWIGLU) wr += (r >> 3) * up_offset;
    wsrc[j] = W + (size_t)wr * ldw + lblk * 4;
    xsrc[j] = X + (size_t)(r < M ? r : 0) * ldx + lblk * 4;
  }
  const float* zero = reinterpret_cast<const float*>(mie_zero_words) + lblk * 4;
  char* mine = ring + wave * SLOTS * SLOT_BYTES;
  auto issue = [&](int s) {
    char* base = mine + (s % SLOTS) * SLOT_BYTES;
    const int ks = ks0 + s * GF_U;
    const bool kok = ks + (lblk >> 2) < ks1 && ks * 16 + lblk * 4 < K;
    const size_t k = (size_t)ks * 16;
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
  for (int s = 0; s < SLOTS - 1; ++s) issue(s);
  const int col = lane & 15, kb = lane >> 4;
  const uint32_t ring0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)mine;
  const uint32_t blk0 = (kb ^ (col & 7)) * 16, blk1 = ((4 + kb) ^ (col & 7)) * 16;
  const uint32_t wrow0 = ring0 + col * 128, xrow0 = ring0 + 2048 + (XL == 1 ? col & 7 : col) * 128;
  f32x4 acc[SPW];
#pragma unroll
  for (int i = 0; i < SPW; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int rounds = ks1 > ks0 ? (ks1 - ks0 + GF_U - 1) / GF_U : 0;
  for (int it = 0; it < rounds; ++it) {
    issue(it + SLOTS - 1);                    // into the slot that was read a round ago
    MIE_VMCNT((SLOTS - 1) * L);                // slot `it` has landed
    u32x4 f[2 * GF_U];
    const uint32_t w0 = wrow0 + (it % SLOTS) * SLOT_BYTES, x0 = xrow0 + (it % SLOTS) * SLOT_BYTES;
    ring_read(w0 + blk0, x0 + blk0, w0 + blk1, x0 + blk1, f);
#pragma unroll
    for (int u = 0; u < GF_U; ++u) {
      const int ks = ks0 + it * GF_U + u;     // a step beyond ks1 loaded zeros and joins the last segment: it adds nothing
      const f32x4 w4 = __builtin_bit_cast(f32x4, f[2 * u]), x4 = __builtin_bit_cast(f32x4, f[2 * u + 1]);
#pragma unroll
      for (int i = 0; i < SPW; ++i)
        if (i == SPW - 1 ? (SPW == 1 || ks >= seg_end[SPW > 1 ? SPW - 2 : 0]) : (ks < seg_end[i] && (i == 0 || ks >= seg_end[i > 0 ? i - 1 : 0])))
          acc[i] = step_mfma(w4, x4, acc[i]);
    }
  }
  MIE_VMCNT(0);                                // nothing of this wave is writing the LDS any more
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SPW; ++i) *reinterpret_cast<f32x4*>(s_acc + (wave * SPW + i) * 256 + lane * 4) = acc[i];
  __syncthreads();
  if (threadIdx.x >= 256) return;
  // this thread's result: x row m, column c of the tile
  const int m = threadIdx.x >> 4, c = threadIdx.x & 15;
  const int src = (((c >> 2) << 4) + m) * 4 + (c & 3);
  float v = 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float t = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) t += s_acc[(4 * q + s) * 256 + src];
    v += t;
  }
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
// LEVELS 0: the unit is a segment (grid.z 16), 1: a quarter (grid.z 4), 2: all of K (grid.z 1, result or C += result).
template <int BM, int BN, int WR, int WC, int LEVELS>
__global__ void __launch_bounds__(WR * WC * 64)
tile_f32_kernel(const float* __restrict__ X, long ldx, const float* __restrict__ W, long ldw, float* __restrict__ out,
                long ldo, const float* __restrict__ bias, int add, int M, int N, int K) {
  constexpr int THREADS = WR * WC * 64, WM = BM / WR, WN = BN / WC, TM = WM / 16, TN = WN / 16;
  constexpr int XL = BM * 8 / THREADS, WL = BN * 8 / THREADS;      // 16-byte loads a thread and stage
  extern __shared__ __align__(16) char gf_lds[];
  f32x4* xs = reinterpret_cast<f32x4*>(gf_lds);                    // [2][BM][8]: row r's block b at 8 r + (b ^ (r / 2) % 8)
  f32x4* ws = xs + 2 * BM * 8;                                     // [2][BN][8]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const KCut cut = k_cut(K);
  int ks0, ks1;
  if (LEVELS == 0) segment_range(cut, blockIdx.z, ks0, ks1);
  else if (LEVELS == 1) { ks0 = least(blockIdx.z * cut.quarter, cut.steps); ks1 = least(ks0 + cut.quarter, cut.steps); }
  else { ks0 = 0; ks1 = cut.steps; }

  const float* xsrc[XL];
  const float* wsrc[WL];
  int xat[XL], wat[WL], xblk[XL], wblk[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int idx = tid + THREADS * i, r = idx >> 3, b = idx & 7, row = m0 + r;
    xsrc[i] = X + (size_t)(row < M ? row : M - 1) * ldx + b * 4;
    xblk[i] = b * 4;
    xat[i] = r * 8 + (b ^ ((r >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int idx = tid + THREADS * i, r = idx >> 3, b = idx & 7, row = n0 + r;
    wsrc[i] = W + (size_t)(row < N ? row : N - 1) * ldw + b * 4;
    wblk[i] = b * 4;
    wat[i] = r * 8 + (b ^ ((r >> 1) & 7));
  }
  f32x4 xr[XL], wreg[WL];
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int ks) {                  // steps ks, ks + 1; what lies beyond K is zero, its load is from the row's end
    const int k = ks * 16;
    if (k + 32 <= K) {                        // (a unit may start at an odd step: the last stage can be cut short for any K)
#pragma unroll
      for (int i = 0; i < XL; ++i) xr[i] = *reinterpret_cast<const f32x4*>(xsrc[i] + k);
#pragma unroll
      for (int i = 0; i < WL; ++i) wreg[i] = *reinterpret_cast<const f32x4*>(wsrc[i] + k);
      return;
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) xr[i] = *reinterpret_cast<const f32x4*>(xsrc[i] + least(k, K - 4 - xblk[i]));
#pragma unroll
    for (int i = 0; i < WL; ++i) wreg[i] = *reinterpret_cast<const f32x4*>(wsrc[i] + least(k, K - 4 - wblk[i]));
#pragma unroll
    for (int i = 0; i < XL; ++i) if (k + xblk[i] >= K) xr[i] = none;
#pragma unroll
    for (int i = 0; i < WL; ++i) if (k + wblk[i] >= K) wreg[i] = none;
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XL; ++i) xs[buf * BM * 8 + xat[i]] = xr[i];
#pragma unroll
    for (int i = 0; i < WL; ++i) ws[buf * BN * 8 + wat[i]] = wreg[i];
  };

  f32x4 acc[TN][TM], quarter[LEVELS >= 1 ? TN : 1][LEVELS >= 1 ? TM : 1], total[LEVELS >= 2 ? TN : 1][LEVELS >= 2 ? TM : 1];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) {
      acc[a][b] = none;
      if (LEVELS >= 1) quarter[LEVELS >= 1 ? a : 0][LEVELS >= 1 ? b : 0] = none;
      if (LEVELS >= 2) total[LEVELS >= 2 ? a : 0][LEVELS >= 2 ? b : 0] = none;
    }
  const int wm = (wave % WR) * WM, wn = (wave / WR) * WN;
  const int r16 = lane & 15, g = lane >> 4;

  int quarter_end = LEVELS >= 2 ? least(cut.quarter, cut.steps) : ks1;
  int segment_end = LEVELS >= 1 ? least(ks0 + cut.segment, quarter_end) : ks1;
  if (ks0 < ks1) fetch(ks0);
  int buf = 0;
  for (int ks = ks0; ks < ks1; ks += 2, buf ^= 1) {
    put(buf);
    __syncthreads();                          // (a buffer is written again two stages on, behind the barrier in between)
    if (ks + 2 < ks1) fetch(ks + 2);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (ks + u >= ks1) break;
      f32x4 wf[TN], xf[TM];
#pragma unroll
      for (int a = 0; a < TN; ++a) { const int r = wn + a * 16 + r16; wf[a] = ws[buf * BN * 8 + r * 8 + ((4 * u + g) ^ ((r >> 1) & 7))]; }
#pragma unroll
      for (int b = 0; b < TM; ++b) { const int r = wm + b * 16 + r16; xf[b] = xs[buf * BM * 8 + r * 8 + ((4 * u + g) ^ ((r >> 1) & 7))]; }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
          for (int b = 0; b < TM; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[a][j], xf[b][j], acc[a][b], 0, 0, 0);
      if (LEVELS >= 1 && ks + u + 1 == segment_end) {
        const bool quarter_done = LEVELS >= 2 && segment_end == quarter_end;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
          for (int b = 0; b < TM; ++b) {
            f32x4& q = quarter[LEVELS >= 1 ? a : 0][LEVELS >= 1 ? b : 0];
            q += acc[a][b];
            acc[a][b] = none;
            if (quarter_done) {
              total[LEVELS >= 2 ? a : 0][LEVELS >= 2 ? b : 0] += q;
              q = none;
            }
          }
        if (quarter_done) quarter_end = least(quarter_end + cut.quarter, cut.steps);
        segment_end = least(segment_end + cut.segment, quarter_end);
      }
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
      const int n = n0 + wn + a * 16 + 4 * g;
      if (n >= N) continue;                   // N is a multiple of 4
      f32x4 v = LEVELS == 0 ? acc[a][b] : LEVELS == 1 ? quarter[LEVELS >= 1 ? a : 0][LEVELS >= 1 ? b : 0]
                                                      : total[LEVELS >= 2 ? a : 0][LEVELS >= 2 ? b : 0];
      f32x4* o = reinterpret_cast<f32x4*>(dst + (size_t)m * ld + n);
      if (LEVELS == 2) {
        if (bias) v += *reinterpret_cast<const f32x4*>(bias + n);
        if (add) v = *o + v;
      }
      *o = v;
    }
  }
}

// The sums of PARTS (4 quarters or 16 segments) units joined in the order above, then stored, added into `out`, or, with
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
      for (int s = 0; s < 4; ++s) t += v[(4 * q + s) % PARTS];
    }
    total += t;
  }
  return total;
}

template <int PARTS, int EPI>
__global__ void __launch_bounds__(256)
reduce_f32_kernel(const float* __restrict__ part, float* __restrict__ out, long ldo, const float* __restrict__ bias, int M, int N) {
  const int cols = EPI == GF_SWIGLU ? 2 * N : N, per_row = N >> 2;
  const size_t stride = (size_t)M * cols / 4, total = (size_t)M * per_row;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (size_t)gridDim.x * 256) {
    const size_t m = e / per_row, n = (e - m * per_row) * 4;
    const f32x4* p = reinterpret_cast<const f32x4*>(part + m * cols + n);
    f32x4 v = join_parts<PARTS>(p, stride);
    f32x4* o = reinterpret_cast<f32x4*>(out + m * ldo + n);
    if (EPI == GF_SWIGLU) {
      const f32x4 u = join_parts<PARTS>(p + (N >> 2), stride);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + expf(-v[i])) * u[i];
      *o = v;
    } else {
      if (bias) v += *reinterpret_cast<const f32x4*>(bias + n);
      *o = EPI == GF_ADD ? *o + v : v;
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

// The tile of a workgroup (wide: 128 rows of x by 64 of W and eight waves, else 64 by 64 and four) and how many units K is
// cut into for M rows (more than 16): 1, 4 or 16.  Measured over 32 to 2,048 rows at [2560, 2048], [2048, 2048],
// [11264, 2048] and [2048, 5632] (MI355X, us): the wide tile reads a third less out of the L2s and wins from two
// workgroups a compute unit on (512 rows of [11264, 2048] 225 against 241, 2,048 rows of [2048, 2048] 150 against 165),
// unless its last rows would be empty (300 rows of [11264, 2048] 184 against 157).  64 by 64 in quarters from 128 tiles
// on (512 rows of [2048, 2048] 51 against 61 in segments and 62 whole, 200 of [11264, 2048] 121 against 127 whole),
// in segments below (32 rows of [2048, 5632] 22 against 44).
static void tile_plan(int M, int N, bool& wide, int& units) {
  auto tiles = [&](int a, int b) { return (long)((M + a - 1) / a) * ((N + b - 1) / b); };
  wide = tiles(128, 64) >= 512 && (M + 127) / 128 * 128 * 10 <= (M + 63) / 64 * 64 * 11;
  const long t = tiles(64, 64);
  units = wide || t >= 1024 ? 1 : t >= 128 ? 4 : 16;
}
MIE_EXPORT int mie_f32_units(int M, int N) {
  bool wide;
  int units;
  tile_plan(M, N, wide, units);
  return units;
}

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
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(WAVES * 64), lds, s, X, ldx, W, ldw, out, ldo, bias, M, N, K, N, rope);  \
  }
  if (tiles <= 256) {
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
                       int N, int K, int units, hipStream_t s) {
  constexpr int lds = 2 * (BM + BN) * 128;
  auto kernel = tile_f32_kernel<BM, BN, WR, WC, LEVELS>;
  if ((M + BM - 1) / BM > 65535) MIE_FAIL("gemm_f32: M = %d is beyond the grid", M);
  if (mie_allow_lds((const void*)kernel, lds, "gemm_f32")) return -1;
  hipLaunchKernelGGL(kernel, dim3((N + BN - 1) / BN, (M + BM - 1) / BM, units), dim3(WR * WC * 64), lds, s, X, ldx, W, ldw, out, ldo, bias, add, M, N, K);
  MIE_CHECK_LAUNCH("tile_f32");
  return 0;
}

static int launch_tiles(const float* X, long ldx, const float* W, long ldw, float* out, long ldo, const float* bias, int add, int M,
                        int N, int K, bool wide, int units, hipStream_t s) {
  if (wide) return launch_tile<128, 64, 4, 2, 2>(X, ldx, W, ldw, out, ldo, bias, add, M, N, K, 1, s);
  return units == 1   ? launch_tile<64, 64, 2, 2, 2>(X, ldx, W, ldw, out, ldo, bias, add, M, N, K, 1, s)
         : units == 4 ? launch_tile<64, 64, 2, 2, 1>(X, ldx, W, ldw, out, ldo, bias, add, M, N, K, 4, s)
                      : launch_tile<64, 64, 2, 2, 0>(X, ldx, W, ldw, out, ldo, bias, add, M, N, K, 16, s);
}

template <int EPI>
static int launch_reduce(int units, const float* part, float* out, long ldo, const float* bias, int M, int N, hipStream_t s) {
  long blocks = ((long)M * (N / 4) + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (units == 4)
    hipLaunchKernelGGL((reduce_f32_kernel<4, EPI>), dim3((unsigned)blocks), dim3(256), 0, s, part, out, ldo, bias, M, N);
  else
    hipLaunchKernelGGL((reduce_f32_kernel<16, EPI>), dim3((unsigned)blocks), dim3(256), 0, s, part, out, ldo, bias, M, N);
  MIE_CHECK_LAUNCH("reduce_f32");
  return 0;
}

// epi 0: out = x W^T (+ bias), 1: out += x W^T (+ bias), 2: out = silu(gate) * up with W = [gate rows (N of them); up rows].
// part: mie_f32_units(M, columns of x W^T) * M * columns floats, 16-byte aligned, when M > 16 and that is more than one
// unit or epi is 2 (then at least one unit's worth).
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
  bool wide;
  int units;
  tile_plan(M, cols, wide, units);
  if (units == 1 && epi != GF_SWIGLU) return launch_tiles(X, ldx, W, ldw, out, ldo, bias, epi == GF_ADD, M, N, K, wide, 1, s);
  if (epi == GF_SWIGLU && units == 1) MIE_FAIL("gemm_f32: %d rows of %d columns are one unit: take the product and silu_mul", M, cols);
  if (!part) MIE_FAIL("gemm_f32: %d units need memory for their sums", units);
  if (launch_tiles(X, ldx, W, ldw, part, cols, nullptr, 0, M, cols, K, wide, units, s)) return -1;
  return epi == GF_STORE ? launch_reduce<GF_STORE>(units, part, out, ldo, bias, M, N, s)
       : epi == GF_ADD ? launch_reduce<GF_ADD>(units, part, out, ldo, bias, M, N, s)
                       : launch_reduce<GF_SWIGLU>(units, part, out, ldo, bias, M, N, s);
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
