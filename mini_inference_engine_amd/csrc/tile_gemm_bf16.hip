// Matrix products of the bfloat16 path with more than 128 rows, with what follows each of them folded in:
//
//   add:      stream[m, n] += sum_k x[m, k] W[n, k]                  (o and down; the 32-bit stream)
//   q/k/v:    rotary on the float32 sums of q and k, q out, k and v into their cache slots
//   SwiGLU:   out[m, j] = silu(gate[m, j]) * up[m, j] on their float32 sums
//   parts:    part[u, m, n] = the sums over unit u's part of K, which meet in the add + norm kernel that follows anyway
//             (reduce_rows in gemm_mid_bf16.hip)          x [M, K], W [N, K] bfloat16, float32 sums
//
// A workgroup makes BM x BN outputs (v_mfma_f32_16x16x32_bf16, A = 16 weight rows, B = 16 x rows), its waves WR x WC tiles of them.
// Stages of 64 k come into a ring in the LDS by loads that write it directly, 8 rows x 128 bytes a load: whole cache lines.  Row r's
// block b of 16 bytes stands at 8 r + (b ^ r % 8), so that the fragment reads (lane 16 g + r: row r, block g) spread over all banks.
//
// What bounds it, and what was wrong with the kernels before.  They took a compute unit's intake for the limit, 58 bytes a nanosecond: that
// was the time of their own instructions, some 40 scalar ones a load for its address.  A kernel that only loads, offsets in registers, gets
// 75 to 97 bytes a nanosecond in this pattern (128 x 128 to 256 x 384 tiles) and 128 of lines that are in the L2.  So:
//   - a load is one scalar addition and the load: this lane's offset of each of a wave's loads stays in a register;
//   - the fragments of half a stage are read while the other half is multiplied, across the one barrier a stage, in its middle, and loads go
//     out between the matrix instructions (2,048 rows of [2048, 5632], weights in the caches, us: read behind the barrier 49, so 44);
//   - weights that come from memory in pieces of 128 bytes a row cost 10 us of that product more than weights in the memory-side cache, at
//     any depth of the ring; so a wave beside the others reads a word of every 64 bytes of the rows eight stages (1 KB a row) ahead: 57 -> 47;
//   - what follows the product is in its epilogue (q/k/v's rotation had a kernel of 8 us), two tiles' numbers of a row stored as 16 bytes.
// Large products are bound by the matrix instructions and the clock they leave (1.9 to 2.2 GHz): the library's largest tiles stay there.
#include "launch.hpp"
#include <math.h>
#include <type_traits>
#include <utility>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_on_8 __attribute__((aligned(8)));      // 16 bytes that begin on 8: one store all the same

enum { TG_F32, TG_ADD, TG_SWIGLU, TG_ROPE };

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(a)) | ((uint32_t)__builtin_bit_cast(uint16_t, __float2bfloat16(b)) << 16);
}

// What the rotary epilogue needs beside the product: W is the fused q/k/v projection.
struct TileRope {
  const int* positions;      // [M]
  const float* cos_t;        // [positions, D / 2]
  const float* sin_t;
  const int* slots;          // [M] cache slot of each row's token
  bf16* k_cache;             // [pages, Hkv, page, D]
  bf16* v_cache;             // [pages, Hkv, D, page]
  int Hq, Hkv, D, page;
};

struct TileArgs {
  const bf16 *X, *W;
  void* out;
  long ldo, unit_stride;
  uint32_t ldx, ldw;         // in bytes
  int M, N, stages_all, stages_unit, mt, nt, panel;     // stages of 64 k; tiles over m and n, columns of tiles an XCD walks together
};

// 16 bytes a lane to the LDS at byte ring + AT + 16 lane (mie_load_to_lds with the place's constant part folded into its one move)
template <int AT>
__device__ __forceinline__ void load_to_ring(const void* base, uint32_t offset, uint32_t ring) {
  uint32_t written;
  asm volatile(
    "s_add_u32 m0, %1, %4\n\t"
    "s_nop 0\n\t"
    "global_load_lds_dwordx4 %2, %3"
    : "={m0}"(written)
    : "s"(ring), "v"(offset), "s"(base), "n"(AT)
    : "memory", "scc");
}

template <int N> using Int = std::integral_constant<int, N>;

// Two tiles' four bfloat16 numbers a lane become one tile's eight: lanes of kb 0 and 2 get tile a's numbers of kb 0, 1 and of 2, 3, the
// lanes of kb 1 and 3 tile b's.
__device__ __forceinline__ uint4 eight_of_two(uint2 a, uint2 b) {
  const auto x = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false), y = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
  return make_uint4(x[0], y[0], x[1], y[1]);
}

// silu(gate) * up of x row m: acc[a] gate, acc[a + TA / 2] up, n the first column of the wave's first tile
template <int TA, int TB>
__device__ __forceinline__ void store_swiglu(const TileArgs& t, const f32x4 (&acc)[TA][TB], int b, int m, int n, int kb) {
  auto four = [&](int a) {
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float g = acc[a][b][i];
      o[i] = g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f)) * acc[a + TA / 2][b][i];
    }
    return make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
  };
  bf16* row = (bf16*)t.out + (size_t)m * t.ldo;
#pragma unroll
  for (int a = 0; a + 1 < TA / 2; a += 2) {
    const uint4 v = eight_of_two(four(a), four(a + 1));
    const int at = n + (a + (kb & 1)) * 16 + 8 * (kb >> 1);          // N is a multiple of 8
    if (m < t.M && at < t.N) *reinterpret_cast<u32x4_on_8*>(row + at) = u32x4_on_8{v.x, v.y, v.z, v.w};      // (ldo is one of 4)
  }
  if (TA / 2 % 2) {
    const uint2 v = four(TA / 2 - 1);
    const int at = n + (TA / 2 - 1) * 16 + 4 * kb;
    if (m < t.M && at < t.N) *reinterpret_cast<uint2*>(row + at) = v;
  }
}

// The work of a wave that computes nothing: it reads a word of every 64 bytes of the tile's weight rows AHEAD stages before the stages that
// need them, AHEAD * 128 neighbouring bytes of a row at once, and meets the others at their barriers.  The workgroups of the same weight
// rows share them.  (The words go to 256 bytes of the LDS that nobody reads.  Of rows dealt by heads those are touched that lie in the
// tile's place: the workgroups beside this one touch the others.)
template <int BN, int AHEAD, bool GATED>
__device__ __forceinline__ void touch_weights(const TileArgs& t, int tm, int n0, int st0, int nst, uint32_t scrap) {
  constexpr int PIECES = 2 * AHEAD, ROWS = 64 / PIECES;     // of 64 bytes; rows a load takes
  static_assert(ROWS >= 1, "at most 32 stages");
  const int lane = threadIdx.x & 63, share = (BN + t.mt - 1) / t.mt, first = tm * share;
  auto touch = [&](int s) {                                // stages s .. s + AHEAD - 1
    const int piece = lane % PIECES < 2 * (nst - s) ? lane % PIECES : 2 * (nst - s) - 1;
    const char* from = reinterpret_cast<const char*>(t.W) + (size_t)(st0 + s) * 128;
    for (int r = 0; r < share; r += ROWS) {
      const int in = first + r + lane / PIECES, at = in < BN ? in : BN - 1, up = GATED && at >= BN / 2;
      const int row = n0 + at - up * (BN / 2);
      const uint32_t offset = (uint32_t)((row < t.N ? row : t.N - 1) + up * t.N) * t.ldw + piece * 64;
      uint32_t written;
      asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dword %2, %3"
        : "={m0}"(written)
        : "s"(scrap), "v"(offset), "s"(from)
        : "memory");
    }
  };
  touch(0);
  __builtin_amdgcn_s_barrier();
  for (int s = 0; s < nst; ++s) {
    if (s % AHEAD == 0 && s + AHEAD < nst) touch(s + AHEAD);
    __builtin_amdgcn_s_barrier();
  }
  MIE_VMCNT(0);
}

// K in units of stages; unit z's sums go to out + z * unit_stride.  N: columns of the result (TG_SWIGLU: of gate and of up each).
// Weight rows of a wave's TA tiles of 16, by what follows the product:
//   SWIGLU  TA / 2 tiles of gate rows, then the up rows of the same columns
//   ROPE    a tile is 8 first members jd .. jd + 7 of a head's rotary pairs, then their partners jd + D / 2 ..
template <int WR, int WC, int TA, int TB, int RING, int AHEAD, int EPI>
__global__ void __launch_bounds__((WR * WC + (AHEAD > 0)) * 64)
tile_gemm_kernel(TileArgs t, TileRope rope) {
  constexpr int WAVES = WR * WC, BM = WR * TB * 16, BN = WC * TA * 16, STAGE = (BM + BN) * 128;
  constexpr int XL = BM / 8, LOADS = XL + BN / 8, L = (LOADS + WAVES - 1) / WAVES;
  constexpr bool EVEN = LOADS % WAVES == 0;
  constexpr int NM = TA * TB, NF = TA + TB;
  static_assert(RING >= 2 && (RING - 1) * L <= 63, "more loads in flight than the counter holds");
  static_assert(EPI != TG_SWIGLU || TA % 2 == 0, "gate and up tiles");
  extern __shared__ __align__(1024) char tg_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  // workgroup i runs on XCD i % 8: every XCD gets a run of neighbours, tiles in panels of `panel` columns of tiles, across a panel first
  int id = blockIdx.x;
  {
    const int total = gridDim.x, q = total >> 3, r = total & 7, x = id & 7, y = id >> 3;
    id = x * q + (x < r ? x : r) + y;
  }
  const int tiles = t.mt * t.nt, unit = id / tiles;
  id -= unit * tiles;
  const int pn = id / (t.panel * t.mt), rest = id - pn * t.panel * t.mt;
  const int width = t.nt - pn * t.panel < t.panel ? t.nt - pn * t.panel : t.panel;
  const int tm = rest / width, tn = pn * t.panel + rest - tm * width;
  const int m0 = tm * BM, n0 = tn * (EPI == TG_SWIGLU ? BN / 2 : BN);
  const int st0 = unit * t.stages_unit, nst = st0 + t.stages_unit < t.stages_all ? t.stages_unit : t.stages_all - st0;

  // the weight row that is row r of the tile
  auto weight_row = [&](int r) {
    int row, behind = 0;
    if (EPI == TG_SWIGLU) {
      constexpr int HALF = TA * 8;
      const int w = r / (2 * HALF), at = r - w * 2 * HALF, up = at >= HALF;
      row = n0 + w * HALF + at - up * HALF;
      behind = up * t.N;
    } else if (EPI == TG_ROPE) {
      const int tile = (n0 + r) >> 4, per_head = rope.D >> 4, head = tile / per_head;
      row = head * rope.D + (tile - head * per_head) * 8 + ((r >> 3) & 1) * (rope.D >> 1) + (r & 7);
    } else {
      row = n0 + r;
    }
    return (uint32_t)((row < t.N ? row : t.N - 1) + behind);
  };
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)tg_lds;
  if constexpr (AHEAD > 0)
    if (wave == WAVES) {
      touch_weights<BN, AHEAD, EPI == TG_SWIGLU>(t, tm, n0, st0, nst, lds0 + RING * STAGE);
      return;
    }

  // the offset of every load of this wave from the first row of x or of W, kept for the whole loop: a load costs one scalar addition
  const int lrow = lane >> 3;
  const uint32_t lblk = ((lane & 7) ^ lrow) * 16;
  const char *xb = reinterpret_cast<const char*>(t.X) + (size_t)st0 * 128, *wb = reinterpret_cast<const char*>(t.W) + (size_t)st0 * 128;
  uint32_t off[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    const int f = EVEN || wave * L + j < LOADS ? wave * L + j : LOADS - 1;      // (the last one again)
    if (f < XL) {
      const int row = m0 + f * 8 + lrow;
      off[j] = (uint32_t)(row < t.M ? row : t.M - 1) * t.ldx + lblk;
    } else {
      off[j] = weight_row((f - XL) * 8 + lrow) * t.ldw + lblk;
    }
  }
  const uint32_t mine = lds0 + wave * L * 1024;
  uint32_t ri = 0;                                     // place in the ring of the stage that is asked for next
  auto load = [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    if constexpr (EVEN && XL % L == 0) load_to_ring<j * 1024>(wave < XL / L ? xb : wb, off[j], mine + ri);
    else {
      const int f = wave * L + j;
      const char* base = f < XL ? xb : wb;
      if constexpr (EVEN) load_to_ring<j * 1024>(base, off[j], mine + ri);
      else load_to_ring<0>(base, off[j], lds0 + (f < LOADS ? f : LOADS - 1) * 1024 + ri);
    }
  };
  auto loads = [&](auto from, auto to) {
    constexpr int F = decltype(from)::value, T = decltype(to)::value;
    [&]<int... J>(std::integer_sequence<int, J...>) { (load(Int<F + J>()), ...); }(std::make_integer_sequence<int, T - F>());
  };
  auto advance = [&]() {
    xb += 128;
    wb += 128;
    ri += STAGE;
    if (ri == RING * STAGE) ri = 0;
  };

  f32x4 acc[TA][TB];
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wr = wave % WR, wc = wave / WR;
  const char* xl = tg_lds + (wr * TB * 16 + col) * 128;
  const char* wl = tg_lds + (BM + wc * TA * 16 + col) * 128;
  const uint32_t b0 = (kb ^ (col & 7)) * 16, b1 = ((4 + kb) ^ (col & 7)) * 16;

#pragma unroll
  for (int s = 0; s < RING; ++s)
    if (s < nst) {
      loads(Int<0>(), Int<L>());
      advance();
    }
  bf16x8 f[2][NF];                                      // x fragments, then weight fragments; a set for each half of a stage
  auto read = [&](int set, uint32_t at, int i) {
    f[set][i] = i < TB ? *reinterpret_cast<const bf16x8*>(xl + at + i * 2048) : *reinterpret_cast<const bf16x8*>(wl + at + (i - TB) * 2048);
  };
  // Half a stage: the products of set `cur`; between them the other set is read and loads F .. T - 1 of a stage go out.
  auto half = [&](auto curc, uint32_t at, auto from, auto to) {
    constexpr int cur = decltype(curc)::value, F = decltype(from)::value, T = decltype(to)::value, NL = T - F, SP = NM * 3 / 4 > 0 ? NM * 3 / 4 : 1;
    [&]<int... I>(std::integer_sequence<int, I...>) {
      ([&] {
        constexpr int a = I / TB, b = I % TB;
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[cur][TB + a], f[cur][b], acc[a][b], 0, 0, 0);
        constexpr int r0 = (I < SP ? I : SP) * NF / SP, r1 = (I + 1 < SP ? I + 1 : SP) * NF / SP;
        constexpr int l0 = I * NL / NM, l1 = (I + 1) * NL / NM;
        if constexpr (r1 > r0 || l1 > l0) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = r0; i < r1; ++i) read(cur ^ 1, at, i);
          loads(Int<F + l0>(), Int<F + l1>());
          __builtin_amdgcn_sched_barrier(0);
        }
      }(), ...);
    }(std::make_integer_sequence<int, NM>());
  };
  if (nst >= RING) MIE_VMCNT((RING - 1) * L);
  else MIE_VMCNT(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < NF; ++i) read(0, b0, i);
  uint32_t rd = 0;
  constexpr int LH = RING == 2 ? L : L / 2;                              // loads behind the barrier of a stage; the others go out in the next one's first half
  // pend: the second part of a stage's loads is still to go out; more: the first part of another one's goes out here; left: stages
  // that may still be on their way when the next one is waited for
  auto stage = [&](auto pendc, auto morec, auto leftc) {
    constexpr bool PEND = decltype(pendc)::value, MORE = decltype(morec)::value;
    constexpr int LEFT = decltype(leftc)::value;
    const uint32_t nx = rd + STAGE == RING * STAGE ? 0 : rd + STAGE;
    half(Int<0>(), rd + b1, Int<PEND ? LH : L>(), Int<L>());
    if (PEND && LH < L) advance();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave has read all of the stage
    MIE_VMCNT((LEFT > 0 ? LEFT : 0) * L);                // its loads of the next one have landed
    __builtin_amdgcn_s_barrier();                        // and everybody else's
    asm volatile("" ::: "memory");
    half(Int<1>(), nx + b0, Int<0>(), Int<MORE ? LH : 0>());
    if (MORE && LH == L) advance();
    rd = nx;
  };
  if (nst > RING) {
    stage(std::false_type(), std::true_type(), Int<RING - 2>());
    for (int it = 1; it + RING < nst; ++it) stage(std::true_type(), std::true_type(), Int<RING - 2>());
    stage(std::true_type(), std::false_type(), Int<RING - 2>());
    [&]<int... I>(std::integer_sequence<int, I...>) {
      (stage(std::false_type(), std::false_type(), Int<RING - 3 - I>()), ...);
    }(std::make_integer_sequence<int, RING - 1>());
  } else {
    for (int it = 0; it < nst; ++it) stage(std::false_type(), std::false_type(), Int<0>());
  }

  // acc[a][b][i] of lane (col, kb): weight row 16 a + 4 kb + i of the wave's, x row 16 b + col
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    const int m = m0 + (wr * TB + b) * 16 + col;
    if (EPI != TG_ROPE && EPI != TG_SWIGLU && m >= t.M) continue;
    if constexpr (EPI == TG_SWIGLU) {
      store_swiglu<TA, TB>(t, acc, b, m, n0 + wc * TA * 8, kb);
    } else if constexpr (EPI == TG_ROPE) {
      // lanes of kb 0 and 1 hold first members, those of kb 2 and 3 (32 lanes on) their partners
      const int mm = m < t.M ? m : t.M - 1, half_d = rope.D >> 1, per_head = rope.D >> 4;
      const int slot = rope.slots[mm], page_of = slot / rope.page, in_page = slot - page_of * rope.page;
      const float *cr = rope.cos_t + (size_t)rope.positions[mm] * half_d, *sr = rope.sin_t + (size_t)rope.positions[mm] * half_d;
      bf16* q_row = (bf16*)t.out + (size_t)m * t.ldo;
      bf16* k_row = rope.k_cache + ((size_t)page_of * rope.Hkv * rope.page + in_page) * rope.D;
      bf16* v_row = rope.v_cache + (size_t)page_of * rope.Hkv * rope.D * rope.page + in_page;
      const int tile0 = (n0 >> 4) + wc * TA;
      auto place = [&](int a, int& head, int& jd) {        // tile a of the wave: its head and the first of its eight pairs
        head = (tile0 + a) / per_head;
        jd = (tile0 + a - head * per_head) * 8;
      };
      auto turned = [&](int a, int jd) {                   // this lane's four numbers of tile a, rotated and rounded
        const f32x4 c = *reinterpret_cast<const f32x4*>(cr + jd + 4 * (kb & 1)), s = *reinterpret_cast<const f32x4*>(sr + jd + 4 * (kb & 1));
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t v = __float_as_uint(acc[a][b][i]);
          const auto x = __builtin_amdgcn_permlane32_swap(v, v, false, false);      // the pair's first member, the second
          float o1, o2;
          rotate_pair(__uint_as_float(x[0]), __uint_as_float(x[1]), c[i], s[i], o1, o2);
          o[i] = kb < 2 ? o1 : o2;
        }
        return make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
      };
      auto home = [&](int head) {
        return head < rope.Hq ? q_row + (size_t)head * rope.D : k_row + (size_t)(head - rope.Hq) * rope.page * rope.D;
      };
      auto store_v = [&](int a, int head, int jd) {
        const int d = jd + 4 * (kb & 1) + (kb >> 1) * half_d;
        if (m < t.M)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v_row[((size_t)(head - rope.Hq - rope.Hkv) * rope.D + d + i) * rope.page] = __float2bfloat16(acc[a][b][i]);
      };
#pragma unroll
      for (int a = 0; a < TA; a += 2) {
        int head[2], jd[2];
        place(a, head[0], jd[0]);
        place(a + 1, head[1], jd[1]);
        if (a + 1 < TA && head[1] < rope.Hq + rope.Hkv) {
          const uint4 v = eight_of_two(turned(a, jd[0]), turned(a + 1 < TA ? a + 1 : a, jd[1]));
          bf16* dst = kb & 1 ? home(head[1]) + jd[1] : home(head[0]) + jd[0];
          if (m < t.M) *reinterpret_cast<uint4*>(dst + (kb >> 1) * half_d) = v;
          continue;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (a + h >= TA || head[h] >= rope.Hq + 2 * rope.Hkv) continue;
          if (head[h] < rope.Hq + rope.Hkv) {
            const uint2 v = turned(a + h, jd[h]);
            if (m < t.M) *reinterpret_cast<uint2*>(home(head[h]) + jd[h] + 4 * (kb & 1) + (kb >> 1) * half_d) = v;
          } else {
            store_v(a + h, head[h], jd[h]);
          }
        }
      }
    } else {
      float* row = (float*)t.out + unit * t.unit_stride + (size_t)m * t.ldo;
      f32x4 old[TA];
      if (EPI == TG_ADD) {
#pragma unroll
        for (int a = 0; a < TA; ++a) {
          const int n = n0 + (wc * TA + a) * 16 + 4 * kb;
          old[a] = *reinterpret_cast<const f32x4*>(row + (n < t.N ? n : 0));
        }
      }
#pragma unroll
      for (int a = 0; a < TA; ++a) {
        const int n = n0 + (wc * TA + a) * 16 + 4 * kb;
        if (n >= t.N) continue;                          // N is a multiple of 8
        *reinterpret_cast<f32x4*>(row + n) = EPI == TG_ADD ? old[a] + acc[a][b] : acc[a][b];
      }
    }
  }
}

// Gate and up, and parts of K, by waves without room for a second set of fragments: a stage is read behind its barrier, in one of two ways.
//   SPREAD  few waves of many sums (256 x 320 and 256 x 384, eight of them): the weight fragments one ahead, a load between every TB matrix
//           instructions; a load that finds the queue full stops its wave, and all at once behind the barrier they stop every wave.
//   else    many waves (256 x 192 by twelve, 256 x 256 by sixteen of 64 x 64): while one waits another one multiplies, so each reads all
//           fragments of half a stage before its products, and the loads of the next stage, which in a ring of two has only this stage's time
//           to arrive, all go out first.  [11264, 2048], weights from memory, us, so / spread / by eight waves (of 64 x 96 with two sets
//           of fragments, of 64 x 128 spread): 800 rows 46.4 / 49.8 / 50.3, 1,132 50.2 / 56.5 / 55.8, 1,280 51.7 / 57.3 / 57.5; [16384, 2048] 700 rows
//           47.5 / 56.3 / 56.9, 2,048 107 / 117 / 120.  Two workgroups a compute unit, each with a ring of two, are the same at parts of K.
template <int WR, int WC, int TA, int TB, int STAGES, bool SPREAD, int EPI>
__global__ void __launch_bounds__(WR * WC * 64)
tile_lean_kernel(TileArgs t) {
  constexpr int WAVES = WR * WC, BM = WR * TB * 16, BN = WC * TA * 16, XL = BM / 8, LOADS = XL + BN / 8, L = (LOADS + WAVES - 1) / WAVES;
  constexpr int STAGE = LOADS * 1024, HALF = TA * 8;
  constexpr bool EVEN = LOADS % WAVES == 0;
  static_assert(!SPREAD || L < 2 * TA, "a load between every TB matrix instructions, from the second on");
  static_assert(!SPREAD || (TB <= TA && TA % 2 == 0), "the second half's x fragments are read in the first, its first weights in the slot that is free");
  static_assert((STAGES - 2) * L <= 63, "more loads in flight than the counter holds");
  static_assert(EPI == TG_SWIGLU || EPI == TG_F32, "what follows");
  extern __shared__ __align__(1024) char tg_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  int id = blockIdx.x;
  {
    const int total = gridDim.x, q = total >> 3, r = total & 7, x = id & 7, y = id >> 3;
    id = x * q + (x < r ? x : r) + y;
  }
  const int tm = id % t.mt, rest = id / t.mt, unit = EPI == TG_F32 ? rest / t.nt : 0, tn = rest - unit * t.nt;
  const int m0 = tm * BM, n0 = tn * (EPI == TG_SWIGLU ? BN / 2 : BN);
  const int st0 = unit * t.stages_unit, left = t.stages_all - st0, nst = EPI == TG_F32 && t.stages_unit < left ? t.stages_unit : left;
  const int lrow = lane >> 3;
  const uint32_t lblk = ((lane & 7) ^ lrow) * 16;
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)tg_lds;
  const char *xb = reinterpret_cast<const char*>(t.X) + (size_t)st0 * 128, *wb = reinterpret_cast<const char*>(t.W) + (size_t)st0 * 128;
  uint32_t off[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    const int f = EVEN || wave * L + j < LOADS ? wave * L + j : LOADS - 1;      // (the last one again)
    uint32_t row;
    if (f < XL) {
      row = m0 + f * 8 + lrow;
      if ((int)row >= t.M) row = t.M - 1;
      off[j] = row * t.ldx + lblk;
      continue;
    }
    const int r = (f - XL) * 8, w = EPI == TG_SWIGLU ? r / (2 * HALF) : 0, at = r - w * 2 * HALF, up = EPI == TG_SWIGLU && at >= HALF;
    row = n0 + w * HALF + at - up * HALF + lrow;
    if ((int)row >= t.N) row = t.N - 1;
    off[j] = (row + up * t.N) * t.ldw + lblk;
  }
  const uint32_t mine = lds0 + wave * L * 1024;
  uint32_t ri = 0;
  auto load = [&](auto jc) {                   // the wave's j-th load of the stage that is asked for next
    constexpr int j = decltype(jc)::value;
    const int f = wave * L + j;
    const char* base = f < XL ? xb : wb;
    if constexpr (EVEN) load_to_ring<j * 1024>(base, off[j], mine + ri);
    else load_to_ring<0>(base, off[j], lds0 + (f < LOADS ? f : LOADS - 1) * 1024 + ri);
  };
  auto loads = [&]() { [&]<int... J>(std::integer_sequence<int, J...>) { (load(Int<J>()), ...); }(std::make_integer_sequence<int, L>()); };
  auto advance = [&]() {
    xb += 128;
    wb += 128;
    ri += STAGE;
    if (ri == STAGES * STAGE) ri = 0;
  };
  f32x4 acc[TA][TB];
#pragma unroll
  for (int a = 0; a < TA; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wr = wave % WR, wc = wave / WR;
  const char* xl = tg_lds + (wr * TB * 16 + col) * 128;
  const char* wl = tg_lds + (BM + wc * TA * 16 + col) * 128;

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nst) {
      loads();
      advance();
    }
  uint32_t stage = 0;
  auto body = [&](auto morec) {
    constexpr bool MORE = decltype(morec)::value;
    if (MORE) MIE_VMCNT((STAGES - 2) * L);                        // this wave's loads of the stage have landed
    else MIE_VMCNT(0);
    __builtin_amdgcn_s_barrier();                                // and everybody else's; everybody is done with the stage before
    asm volatile("" ::: "memory");
    const uint32_t blk0 = stage + (kb ^ (col & 7)) * 16, blk1 = stage + ((4 + kb) ^ (col & 7)) * 16;
    if constexpr (SPREAD) {
      bf16x8 xf[2][TB], wf[2];
#pragma unroll
      for (int b = 0; b < TB; ++b) xf[0][b] = *reinterpret_cast<const bf16x8*>(xl + blk0 + b * 2048);
      wf[0] = *reinterpret_cast<const bf16x8*>(wl + blk0);
      [&]<int... I>(std::integer_sequence<int, I...>) {
        ([&] {
          constexpr int kc = I / TA, a = I % TA;
          const uint32_t blk = kc ? blk1 : blk0;
          if constexpr (a + 1 < TA) wf[(a + 1) & 1] = *reinterpret_cast<const bf16x8*>(wl + blk + (a + 1) * 2048);
          else if constexpr (kc == 0) wf[(a + 1) & 1] = *reinterpret_cast<const bf16x8*>(wl + blk1);
          if constexpr (kc == 0 && a + TB >= TA) xf[1][a + TB - TA] = *reinterpret_cast<const bf16x8*>(xl + blk1 + (a + TB - TA) * 2048);
          if constexpr (MORE && I >= 1 && I <= L) load(Int<I - 1>());
#pragma unroll
          for (int b = 0; b < TB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[a & 1], xf[kc][b], acc[a][b], 0, 0, 0);
        }(), ...);
      }(std::make_integer_sequence<int, 2 * TA>());
    } else {
      if (MORE) loads();
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const uint32_t blk = kc ? blk1 : blk0;
        bf16x8 xf[TB], wf[TA];
#pragma unroll
        for (int a = 0; a < TA; ++a) wf[a] = *reinterpret_cast<const bf16x8*>(wl + blk + a * 2048);
#pragma unroll
        for (int b = 0; b < TB; ++b) xf[b] = *reinterpret_cast<const bf16x8*>(xl + blk + b * 2048);
#pragma unroll
        for (int a = 0; a < TA; ++a)
#pragma unroll
          for (int b = 0; b < TB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[a], xf[b], acc[a][b], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // this wave has read the stage before the next barrier
    if (MORE) advance();
    stage = stage + STAGE == STAGES * STAGE ? 0 : stage + STAGE;
  };
  int it = 0;
  for (; it + STAGES - 1 < nst; ++it) body(std::true_type());
  for (; it < nst; ++it) body(std::false_type());

#pragma unroll
  for (int b = 0; b < TB; ++b) {
    const int m = m0 + (wr * TB + b) * 16 + col;
    if constexpr (EPI == TG_SWIGLU) {
      store_swiglu<TA, TB>(t, acc, b, m, n0 + wc * HALF, kb);
    } else if (m < t.M) {
      float* row = (float*)t.out + unit * t.unit_stride + (size_t)m * t.ldo;
#pragma unroll
      for (int a = 0; a < TA; ++a) {
        const int n = n0 + (wc * TA + a) * 16 + 4 * kb;
        if (n < t.N) *reinterpret_cast<f32x4*>(row + n) = acc[a][b];       // N is a multiple of 8
      }
    }
  }
}

MIE_EXPORT const char* tile_gemm_bf16_last_error() { return g_mie_error; }

static int grid_of(TileArgs& t, int bm, int cols, int K, int units, int* grid) {
  t.mt = (t.M + bm - 1) / bm;
  t.nt = (t.N + cols - 1) / cols;
  t.stages_all = K / 64;
  t.stages_unit = (t.stages_all + units - 1) / units;
  if ((long)t.mt * t.nt * units > 0x7FFFFFFF) MIE_FAIL("tile_gemm: %d x %d tiles are beyond the grid", t.mt, t.nt);
  *grid = t.mt * t.nt * units;
  // an XCD's run of tiles as square as its rows of x and W allow
  const float run = *grid / 8.f, wide = sqrtf(run * bm / cols);
  t.panel = wide < 1.f ? 1 : wide > t.nt ? t.nt : (int)(wide + 0.5f);
  return 0;
}

template <int WR, int WC, int TA, int TB, int RING, int AHEAD, int EPI>
static int launch(TileArgs t, const TileRope& rope, int K, int units, hipStream_t s) {
  constexpr int BM = WR * TB * 16, BN = WC * TA * 16, lds = RING * (BM + BN) * 128 + (AHEAD > 0 ? 256 : 0);
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = tile_gemm_kernel<WR, WC, TA, TB, RING, AHEAD, EPI>;
  if (mie_allow_lds((const void*)kernel, lds, "tile_gemm")) return -1;
  int grid;
  if (grid_of(t, BM, EPI == TG_SWIGLU ? BN / 2 : BN, K, units, &grid)) return -1;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3((WR * WC + (AHEAD > 0)) * 64), lds, s, t, rope);
  MIE_CHECK_LAUNCH("tile_gemm");
  return 0;
}

// The same with the wave that reads the weights ahead where three or more rows of tiles share that reading.  Of one or two rows each such wave
// has 64 rows or more of every eight stages to itself, and the others wait for it at the barriers: [11264, 2048], us, with / without it (128 x 128):
// 129 rows 23.9 / 18.9, 256 23.6 / 22.1; [16384, 2048] 129 rows 27.3 / 23.1, 256 27.3 / 24.2, 450 (256 x 128) 37.1 / 31.4, 300 (192 x 128) 31.7 /
// 26.4, 384 32.3 / 28.9; [28672, 2048] 160 rows (192 x 128) 40.6 / 32.9; [22528, 2048] 129 rows (128 x 192) 36.8 / 27.5, 256 37.6 / 31.7.  Of three and more
// 450 rows of [11264, 2048] (128 x 192) 28.0 / 26.6, 512 28.3 / 28.2, of [5632, 2048] 22.8 / 24.0 and 23.1 / 26.2; 384 rows of [8192, 2048] 21.2 / 21.7, 512 21.0 / 21.5, 1,024 of [2048, 2048] 16.8 / 18.4.  Parts of K: 129 rows of [4096, 14336] in
// four 42.9 / 35.8, 256 45.3 / 42.2, 129 of [2048, 5632] in eight 13.2 / 12.3, 256 of [8192, 4096] in two 29.5 / 26.1; of four rows of tiles 512 of
// [4096, 14336] in two 64.6 / 71.8.
template <int WR, int WC, int TA, int TB, int RING, int EPI>
static int launch_ahead(const TileArgs& t, int K, int units, hipStream_t s) {
  return t.M <= 2 * WR * TB * 16 ? launch<WR, WC, TA, TB, RING, 0, EPI>(t, TileRope{}, K, units, s)
                                 : launch<WR, WC, TA, TB, RING, 8, EPI>(t, TileRope{}, K, units, s);
}

template <int WR, int WC, int TA, int TB, int STAGES, bool SPREAD, int EPI>
static int launch_lean(TileArgs t, int K, int units, hipStream_t s) {
  constexpr int BM = WR * TB * 16, BN = WC * TA * 16, lds = STAGES * (BM + BN) * 128;
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = tile_lean_kernel<WR, WC, TA, TB, STAGES, SPREAD, EPI>;
  if (mie_allow_lds((const void*)kernel, lds, "tile_gemm")) return -1;
  int grid;
  if (grid_of(t, BM, EPI == TG_SWIGLU ? BN / 2 : BN, K, units, &grid)) return -1;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(WR * WC * 64), lds, s, t);
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

static TileArgs arguments(const void* X, long ldx, const void* W, long ldw, void* out, long ldo, int M, int N) {
  TileArgs t = {};
  t.X = (const bf16*)X; t.W = (const bf16*)W; t.out = out; t.ldo = ldo;
  t.ldx = (uint32_t)ldx * 2; t.ldw = (uint32_t)ldw * 2; t.M = M; t.N = N;
  return t;
}

// Tiles of the products that are added or rotated: time of a stage of 64 k and of start and end, us (MI355X, weights from memory), and
// workgroups that a compute unit holds at once.  Measured at 160 to 2,048 rows of [2048, 2048], [2048, 5632], [2560, 2048], [4096, 4096],
// [4096, 14336] and [6144, 4096].
constexpr struct { int bm, bn; float us, fixed; int held; } PRODUCT_TILES[] = {
  {64, 64, 0.235f, 2.8f, 2}, {64, 80, 0.27f, 2.8f, 2}, {64, 96, 0.29f, 2.8f, 1}, {64, 128, 0.33f, 3.2f, 1}, {80, 128, 0.34f, 6.0f, 1},
  {96, 128, 0.375f, 6.0f, 1}, {128, 128, 0.45f, 8.0f, 1}, {128, 160, 0.54f, 10.0f, 1}, {128, 192, 0.68f, 8.5f, 1}, {256, 128, 0.78f, 12.0f, 1}};
constexpr int PRODUCT_TILES_N = sizeof(PRODUCT_TILES) / sizeof(PRODUCT_TILES[0]);

static long tiles_of(int i, int M, int N) {
  const auto& p = PRODUCT_TILES[i];
  return (long)((M + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn);
}

// The tile with the least estimate among those whose workgroups all run at once; -1 where none has so few: there the library's largest
// tiles are faster (us, own / library: 2,048 rows of [6144, 4096] 103 / 88, of [8192, 4096] 122 / 114, of [28672, 4096] 480 / 428).  Two
// workgroups a compute unit take 1.55 times one's time.  With one round, us, own / library (which for q/k/v leaves the rotation, 8 to 9 us
// more, to a kernel of its own): added, [2048, 2048] 160 rows 9.7 / 12.3, 512 10.4 / 12.2, 1,132 16.9 / 19.5, 2,048 22.4 / 23.5; [2048, 5632]
// 768 31.8 / 33.3, 1,132 35.7 / 44.7, 2,048 47.3 / 55.1; [4096, 4096] 2,048 62.1 / 66.3; [4096, 14336] 1,024 113 / 132, 2,048
// 187 / 197; q/k/v, [2560, 2048] 160 rows 10.7 / 12.7, 512 12.6 / 14.6, 1,132 19.6 / 20.8, 2,048 28.8 / 28.4; [6144, 4096] 256 27.8 / 26.7, 512
// 38.5 / 36.6, 1,024 52.9 / 52.4.
static int tile_for(int M, int N, int K) {
  int best = -1;
  float least = 1e30f;
  for (int i = 0; i < PRODUCT_TILES_N; ++i) {
    const auto& p = PRODUCT_TILES[i];
    const long tiles = tiles_of(i, M, N), cu = mie_compute_units();
    if (tiles > p.held * cu) continue;
    const float us = (p.us * (K / 64) + p.fixed) * (tiles > cu ? 1.55f : 1.f);
    if (us < least) {
      least = us;
      best = i;
    }
  }
  return best;
}

// 1,000 times the rows plus the columns of the tile that such a product takes, 0: it is the library's.
MIE_EXPORT int mie_tile_gemm_tile(int M, int N, int K) {
  const int i = tile_for(M, N, K);
  return i < 0 ? 0 : PRODUCT_TILES[i].bm * 1000 + PRODUCT_TILES[i].bn;
}

// Whether the tile that tile_for picks for q/k/v also beats the library's product with the rotary kernel, 8 us, behind it.  It does not where
// a few compute units walk a long K, which the library cuts, us, own / library and rotary kernel: 129 rows of [768, 3072] 13.4 / 12.3, of
// [640, 2560] 12.5 / 10.9 (36 and 30 tiles), 300 rows of [768, 4096] 18.1 / 17.2, of [768, 8192] 30.5 / 25.0, 192 of [1280, 5120] 24.6 / 19.9 (60 tiles).  On the other
// side 256 rows of [768, 3072] 13.2 / 13.4 (48 tiles), 350 of [768, 4096] 16.8 / 20.6 (72), 129 of [768, 2048] 10.2 / 12.8; of 365 products of 129 to 2,048
// rows 2 remain that the library makes up to 1.6 % faster; all of them together take 0.72 times its time.
MIE_EXPORT int mie_tile_gemm_rope_gains(int M, int N, int K) {
  const int i = tile_for(M, N, K);
  if (i < 0) return 0;
  const long tiles = tiles_of(i, M, N), cu = mie_compute_units();
  return !(64 * tiles <= 15 * cu && K > 3072) && !(64 * tiles <= 9 * cu && K > 2048);
}

// Whether the tile that tile_for picks for a product that is added also beats the library's.  It does not, us, weights from memory, own / library:
//   - on a tenth to a quarter of the compute units with more than 16 stages each, where the library cuts K: 129 to 256 rows of [1024, 2048]
//     9.2 / 8.4, of [1024, 3072] 14.7 / 10.4, of [1536, 1536] 7.9 / 7.5 (but of [1024, 1024] 6.3 / 8.2, 300 rows of [1024, 3072] 14.2 / 15.6);
//   - on 256 x 128 tiles for three quarters of the compute units or fewer: 1,536 rows of [4096, 4096] 59.3 / 56.2, of [4096, 1024] 23.0 / 22.1, 768 of
//     [8192, 8192] 114 / 102 (1,700 and 1,800 rows of [4096, 4096], 224 and 256 of them, 58.8 / 62.3 and 62.2 / 63.6);
//   - on the two widest tiles for 8,192 columns and more over a K of 2,048 or less, whose start and end weigh most: 600 rows 32.4 / 29.8, 900 40.7 /
//     38.8, 1,024 42.7 / 40.7 (of [8192, 8192] 123 / 127).
// Of 397 products of 129 to 2,048 rows 8 remain that the library makes up to 15 % faster (384 rows of [4096, 2048] 16.4 / 15.7, 129 of [8192, 2048]
// 20.0 / 17.0); all of them together take 0.88 times the library's time.
MIE_EXPORT int mie_tile_gemm_add_gains(int M, int N, int K) {
  const int i = tile_for(M, N, K);
  if (i < 0) return 0;
  const auto& p = PRODUCT_TILES[i];
  const long tiles = tiles_of(i, M, N), cu = mie_compute_units();
  if (32 * tiles <= 9 * cu && K > 1024) return 0;
  if (p.bm == 256 && 4 * tiles <= 3 * cu) return 0;
  return !(p.bm * p.bn >= 128 * 192 && N >= 8192 && K <= 2048);
}

// Stages that a wave reads the weights of an added product ahead, 0: none does.  It saves the product time by itself at any size (2,048 rows of
// [4096, 14336], weights from memory, 100 ms on end: 189 us with it, 197 without, 204 by the library), but a product of 200 us takes its power from
// the kernels around it, and in whole steps of such products the saving was gone: 2,048 tokens behind 4,096 in four layers of [4096, 4096]
// and [4096, 14336], three runs, us, with it / without for the second / library: 4,042 / 4,033 / 4,076, 4,055 / 4,010 / 4,086, 4,032 / 4,014 / 4,061.
// Smaller ones keep it: [4096, 11008], 2,048 rows 3,295 / 3,376 / 3,445 a step, [4096, 14336], 1,700 rows 3,265 / 3,348 / 3,359.
MIE_EXPORT int mie_tile_gemm_add_ahead(int M, int N, int K) { return (double)M * N * K > 1.1e11 ? 0 : 8; }

template <int EPI>
static int launch_tile(const TileArgs& t, const TileRope& rope, int K, hipStream_t s) {
  switch (tile_for(t.M, t.N, K)) {
    case 0: return launch<2, 2, 2, 2, 4, 8, EPI>(t, rope, K, 1, s);
    case 1: return launch<4, 1, 5, 1, 4, 8, EPI>(t, rope, K, 1, s);
    case 2: return launch<2, 2, 3, 2, 4, 8, EPI>(t, rope, K, 1, s);
    case 3: return launch<2, 2, 4, 2, 4, 8, EPI>(t, rope, K, 1, s);
    case 4: return launch<1, 4, 2, 5, 4, 8, EPI>(t, rope, K, 1, s);
    case 5: return launch<2, 2, 4, 3, 4, 8, EPI>(t, rope, K, 1, s);
    case 6: return launch<2, 2, 4, 4, 4, 8, EPI>(t, rope, K, 1, s);
    case 7: return launch<2, 2, 5, 4, 4, 8, EPI>(t, rope, K, 1, s);
    case 8: return launch<2, 2, 6, 4, 3, 8, EPI>(t, rope, K, 1, s);
    case 9:
      if constexpr (EPI == TG_ADD)
        if (!mie_tile_gemm_add_ahead(t.M, t.N, K)) return launch<4, 2, 4, 4, 3, 0, EPI>(t, rope, K, 1, s);
      return launch<4, 2, 4, 4, 3, 8, EPI>(t, rope, K, 1, s);
  }
  MIE_FAIL("tile_gemm: %d rows of [%d, %d] are no one round of any tile", t.M, t.N, K);
}

// stream [M, ldo] float32 += x W^T.
MIE_EXPORT int mie_tile_gemm_add(const void* X, long ldx, const void* W, long ldw, float* stream, long ldo, int M, int N, int K, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands(X, ldx, W, ldw, stream, M, N, N, K)) return -1;
  if (ldo < N || (ldo & 3)) MIE_FAIL("tile_gemm_add: leading dim %ld for %d columns", ldo, N);
  return launch_tile<TG_ADD>(arguments(X, ldx, W, ldw, stream, ldo, M, N), TileRope{}, K, s);
}

// The q/k/v projection with the rotation of q and k, q_out [M, ldq] and the caches bfloat16.  D must be a multiple of 16.
MIE_EXPORT int mie_tile_gemm_qkv_rope(const void* X, long ldx, const void* W, long ldw, void* q_out, long ldq, const int* positions,
                                      const float* cos_t, const float* sin_t, const int* slots, void* k_cache, void* v_cache, int M, int Hq,
                                      int Hkv, int D, int page, int K, hipStream_t s) {
  if (M <= 0) return 0;
  if (D <= 0 || (D & 15)) MIE_FAIL("tile_gemm_qkv_rope: head_dim %d must be a multiple of 16", D);
  if (Hq <= 0 || Hkv <= 0 || page <= 0) MIE_FAIL("tile_gemm_qkv_rope: heads %d / %d, page %d", Hq, Hkv, page);
  if (!positions || !cos_t || !sin_t || !slots || !k_cache || !v_cache || !q_out) MIE_FAIL("tile_gemm_qkv_rope: null operand");
  const int N = (Hq + 2 * Hkv) * D;
  if (check_operands(X, ldx, W, ldw, q_out, M, N, N, K)) return -1;
  if (ldq < (long)Hq * D || (ldq & 7)) MIE_FAIL("tile_gemm_qkv_rope: q leading dim %ld < %d", ldq, Hq * D);
  if ((((uintptr_t)cos_t | (uintptr_t)sin_t) & 15) || ((uintptr_t)k_cache & 15)) MIE_FAIL("tile_gemm_qkv_rope: operands must be 16-byte aligned");
  TileRope rope = {positions, cos_t, sin_t, slots, (bf16*)k_cache, (bf16*)v_cache, Hq, Hkv, D, page};
  return launch_tile<TG_ROPE>(arguments(X, ldx, W, ldw, q_out, ldq, M, N), rope, K, s);
}

// Time of a stage (64 k) of a grid that gives every compute unit one workgroup, with its share of the start and the end, us: the numbers
// that the choice goes by, measured on kernels before these.  256 x 192 and wider are tile_lean_kernel's, the others
// tile_gemm_kernel's, of which the first 128 x 128 is for the estimate alone (mie_tile_gemm_swiglu_cost).  The present kernels' at [11264, 2048]
// (MI355X, weights from memory, one round, few to all rows of the tiles): 128 x 128 0.58 to 0.71, 128 x 192 0.72 to 0.93, 192 x 128 0.73 to 0.85,
// 256 x 128 0.84 to 0.95, 192 x 192 0.87 to 1.08, 256 x 192 1.29 to 1.48, 256 x 256 1.31 to 1.68, 256 x 320 1.79 to 2.06, 256 x 384 1.92 to 2.36.  The
// order is the same, and so is the choice: of 22 numbers of rows from 129 to 2,048, with every tile timed, it was within 3 % of the best tile,
// but at 300 and 333, where 192 x 128 takes 23.8 and 25.3 us for 26.2 of 128 x 192.
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

// What mie_tile_gemm_swiglu takes at most, in units of 0.01 us, for the decision against the library.  It leaves out the
// tiles behind 256 x 384: with them the decision, whose estimate of the library is rough, would change for the better at some sizes and
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
  const TileArgs t = arguments(X, ldx, W, ldw, out, ldo, M, N);
  float us;
  switch (best_tile(M, 2L * N, TILES_TAKEN, TILES, us)) {
    case 1: return launch_ahead<2, 2, 4, 6, 3, TG_SWIGLU>(t, K, 1, s);
    case 2: return launch_ahead<4, 2, 4, 4, 3, TG_SWIGLU>(t, K, 1, s);
    case 3: return launch_lean<4, 3, 4, 4, 2, false, TG_SWIGLU>(t, K, 1, s);
    case 4: return launch_lean<4, 4, 4, 4, 2, false, TG_SWIGLU>(t, K, 1, s);
    case 5: return launch_lean<4, 2, 12, 4, 2, true, TG_SWIGLU>(t, K, 1, s);
    case 6: return launch_ahead<2, 2, 4, 4, 4, TG_SWIGLU>(t, K, 1, s);
    case 7: return launch_ahead<2, 2, 6, 4, 3, TG_SWIGLU>(t, K, 1, s);
    case 8: return launch<2, 2, 6, 6, 3, 0, TG_SWIGLU>(t, TileRope{}, K, 1, s);
    default: return launch_lean<4, 2, 10, 4, 2, true, TG_SWIGLU>(t, K, 1, s);
  }
}

// part [units, M, N] float32: the sums over unit u's part of K.  Every unit has at least one stage of 64 k.
MIE_EXPORT int mie_tile_gemm_units(const void* X, long ldx, const void* W, long ldw, float* part, int M, int N, int K, int units, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (check_operands(X, ldx, W, ldw, part, M, N, N, K)) return -1;
  const int stages = K / 64, per = units > 0 ? (stages + units - 1) / units : 0;
  if (units < 1 || (units - 1) * per >= stages) MIE_FAIL("tile_gemm_units: %d units of %d stages", units, stages);
  TileArgs t = arguments(X, ldx, W, ldw, part, N, M, N);
  t.unit_stride = (long)M * N;
  // a workgroup a compute unit and a deep ring, or two and a short one each: weights from memory, us, deep / short, 300 rows of [4096, 14336] in
  // five parts 56.8 / 51.3, 384 65.7 / 53.9, of [4096, 4096] 26.3 / 20.9; 384 rows of [8192, 4096] in two 46.5 / 37.5
  const long groups = (long)((M + 127) / 128) * ((N + 127) / 128) * units;
  return groups > mie_compute_units() ? launch_lean<4, 2, 4, 2, 2, false, TG_F32>(t, K, units, s) : launch_ahead<2, 2, 4, 4, 4, TG_F32>(t, K, units, s);
}
