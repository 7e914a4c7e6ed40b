// Attention of single-token rows on the matrix cores of gfx950 (decode_attention, below), as a function of one workgroup: a kernel of
// its own takes it (attention_bf16.hip), and one that serves a step's portions beside them (prefill_attention_bf16.hip).
// Caches: keys [pages, Hkv, page, D], values [pages, Hkv, D, page].
//
// decode_attention: single-token rows.  One workgroup per (row, kv head, 16 query heads of its group,
// split of the context); its waves take 32-key blocks of the split in turn.  With v_mfma_f32_16x16x32_bf16
//   S^T[key, head]  = K[key, d]  . Q^T[d, head]      A = 16 keys x 32 dims, straight from the key page
//   O^T[d, head]   += V^T[d, key] . P^T[key, head]   A = 16 dims x 32 keys, straight from the value page
// The scores come out with lane % 16 = head and 4 consecutive keys per lane group; that is already
// the layout P^T needs as the B operand of the second product if the 32 keys of its reduction are
// taken in the order (lane group, tile, i), and the value operand is loaded in that same order, so the
// probabilities never leave registers.  Softmax state is one value per lane: the maximum of its head, the sum over
// its own keys of the head's (a head's four lanes join after the last block); exponentials are base 2 with scale * log2(e) folded into the scores.  The waves of a workgroup are
// merged through LDS; splits write normalised partials and base-2 log-sum-exps, merged by a second,
// small kernel.  Keys outside [lo, p] get probability 0 by selection and their values are zeroed, so stale
// or poisoned slots never reach the sums.
//
// How keys and values come in (head sizes 64, 96 and 128): each wave brings its blocks of 32 keys into slots of its own
// in the LDS by loads that write the LDS directly, whole cache lines, and reads the fragments back; a slot is refilled as soon as
// its fragments are in registers, so all of a wave's slots are on their way while it computes.  Straight into registers in the
// matrix instruction's order a quarter wave touches 16 rows for 16 (keys) or 8 bytes (values), and the address unit's line look-ups
// keep a compute unit far below the 75 to 97 bytes a nanosecond that whole lines come in at.  Measured (MI355X, attention and merge, us, before / now): 32 / 4
// heads of 64, 64 rows of 200 to 1,990 keys 21.8 / 20.5, 96 rows 32.9 / 28.6, 32 rows of 150 to 900 13.4 / 11.8, 8 of 2,040 10.7 / 10.5; 32 / 8
// heads of 128, 8 rows of 1,000 to 6,000 41.6 / 35.3, 64 of 200 to 1,990 73.0 / 63.9.  At head size 32 registers are the faster way (64
// rows of 2,040 keys 17.3 us, 19.1 through the LDS).
// The 32 keys of a block are dealt to the score tiles' rows so that a lane's eight probabilities belong to eight neighbouring keys,
// 16 bytes of a value row: lane group g has keys 8 g .. 8 g + 7.
#pragma once
#include "attention_bf16_common.hpp"
#include "launch.hpp"

constexpr int NW_SPLIT = D > 128 ? 2 : 4;    // waves per workgroup (bounded by the LDS the merge of the waves needs)
// When rows and heads alone fill the GPU the context is not split and there is no second kernel; a workgroup then
// has a whole context to read, and eight waves keep twice the loads in flight for it: as long as there are
// fewer than two workgroups a compute unit.  With more, the compute units are kept busy by the number of
// workgroups, and four waves each are faster (256 rows x 4 kv heads of 512 keys: 24.8 against 32.9 us; 64 rows of
// 2,048 keys: 27.8 against 24.1).
constexpr int NW_WHOLE = D > 128 ? 2 : (D > 64 ? 4 : 8);
constexpr bool RINGED = D % 32 == 0 && D >= 64 && D <= 128;
// Blocks of a wave on their way: 32 to 64 KB a workgroup of four waves, 128 of eight (two blocks a wave of four leave room for two
// workgroups a compute unit: head size 64, 128 rows of 100 to 1,990 keys 33.4 us with one, 36.5 with two, 256 of 512 29.1 and 33.6)
constexpr int slots_of(int nw, bool ring = RINGED) { return !ring ? 0 : nw == 8 ? 2 : 1; }
constexpr int BLOCK_LOADS = D / 8;           // of 1 KB: keys and values of 32 keys
// Dynamic LDS of a workgroup of nw waves: the slots, and later, in the same place, the waves' sums.
constexpr int da_lds_bytes(int nw, bool ring) {
  const int slots = nw * slots_of(nw, ring) * BLOCK_KEYS * D * 4, sums = nw * 16 * (D + 1) * 4;
  return slots > sums ? slots : sums;
}
// Workgroups up to which one is NW_WHOLE waves: while each has a compute unit's LDS to itself (ringed), or fewer than two a compute unit.
static long whole_most() { return RINGED ? mie_compute_units() : 2L * mie_compute_units() - 1; }

// What the kernel needs to finish the q/k/v projection of its row itself (FROM_SUMS): the projection's
// float32 sums, split over K or not, instead of q; the angle tables; where the row's new key and value go.
// A workgroup then owns everything of its (row, kv head): it adds the splits up, rotates its group's q heads
// (kept in the LDS) and its k head, writes k and v to their cache slot, and goes on as if another kernel had.
// Only for unsplit contexts and groups of up to 16 heads (one workgroup per row and kv head).
struct ProjectionSums {
  const float* part;         // [splits, rows, ld]: q heads, k heads, v heads
  int splits;
  size_t split_stride;       // floats from one split to the next
  long ld;
  const float* cos_t;        // [positions, D / 2]
  const float* sin_t;
  const int* slots;          // [rows] cache slot of each row's token
};

// DB: a bias on the softmax's scores by the key's distance, from a table a head (its last entry for everything further
// back), added after the scale.
// SIG: sigmoid weights instead of a softmax.  A visible key counts with sigmoid(cap(score) + the head's bias),
// cap(x) = c tanh(x / c) or x itself; a chunk size n (0: none) hides the keys before floor(position / n) n.  There
// is no maximum and no denominator: waves and splits simply add up (the merge sees maxima of 0 and one unit sum
// a workgroup, and the kernel that joins the splits is told not to divide).  scale_log2 then carries the plain scale.
// KEEP: beside the window the row sees its request's first ``keep`` keys.  The blocks that hold them come before the
// window's in the order the splits and waves walk: index x of that order is key x up to the end of the kept blocks, key
// x + gap behind it, gap a whole number of blocks.
// CHUNK: the softmax over the keys of the row's own chunk of positions (from floor(position / chunk) chunk on).
// RING: keys and values through the slots.  Caches off 16 bytes, which those loads do not take, come into registers (RING false), at the
// ringed head sizes in the slots' order of keys, so that the result has the same bits.
// The workgroup of row b, of `unit` of the kv heads and their tiles of 16 query heads, and of split s.
template <int NW, bool FROM_SUMS, bool SIG, bool DB, bool KEEP, bool CHUNK, bool RING>
__device__ __forceinline__ void
decode_attention_body(const int b, const int unit, const int s, const bf16* __restrict__ q, long q_stride, bf16* k_cache, bf16* v_cache,
                      bf16* __restrict__ out, float* __restrict__ o_part,
                      float* __restrict__ lse_part, const int* __restrict__ block_tables, int max_blocks,
                      const int* __restrict__ positions, int Hq, int Hkv, int head_tiles, int page,
                      float scale_log2, int window, int partition, int num_splits, ProjectionSums proj,
                      float sink_log2, int chunk, float softcap, const float* __restrict__ head_bias,
                      const float* __restrict__ dist_bias, int dist_n, int keep, const float* __restrict__ head_sinks) {
  static_assert(!(DB && (SIG || FROM_SUMS)), "the distance bias is built for the softmax over finished queries");
  static_assert(!(KEEP && (SIG || FROM_SUMS || DB)), "kept first keys are built for the plain softmax over finished queries");
  static_assert(!(CHUNK && (SIG || FROM_SUMS || DB || KEEP)), "chunks are built for the plain softmax over finished queries, and for sigmoids");
  __shared__ float s_m[NW][16], s_l[NW][16], s_M[16], s_L[16];
  extern __shared__ __align__(1024) char da_lds[];               // the waves' slots, then s_o [NW][16][D + 1]
  float* s_o = reinterpret_cast<float*>(da_lds);
  __shared__ __align__(16) bf16 s_q[FROM_SUMS ? 16 : 1][D];
  __shared__ __align__(16) bf16 s_k[FROM_SUMS ? D : 1], s_v[FROM_SUMS ? D : 1];   // the row's own new key and value
  const int kvh = unit / head_tiles, ht = unit - kvh * head_tiles;
  const int G = Hq / Hkv;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // the same in all lanes: kept in a scalar register
  const int col = lane & 15, kb = lane >> 4;
  const int g = ht * 16 + col;
  const bool head_ok = g < G;
  const int head = kvh * G + (head_ok ? g : 0);
  const int* bt = block_tables + (size_t)b * max_blocks;

  // Everything that can be asked for before the row's length is known is asked for first: the queries
  // and, without a window, the first block of keys and values (pages are looked up by key index alone,
  // clamped to the table; entries past the row's pages name the scratch page, whose contents are masked).
  Frag qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = ks * 32 + kb * 8;
    qf[ks].q = make_uint4(0, 0, 0, 0);
    if (!FROM_SUMS && head_ok && d0 < D) qf[ks].q = *reinterpret_cast<const uint4*>(q + (size_t)b * q_stride + (size_t)head * D + d0);
  }
  struct KeyBlock {
    Frag a[2][KS];      // keys: 16 keys x 32 dims each
    Frag va[DT];        // values: 16 dims x 32 keys each, in the order the probabilities sit in registers
  };
  // Pages hold a multiple of 16 keys, so each half of a block lies in one page: looked up through the scalar unit, a block
  // ahead.  Looked up by vector loads in front of a block's own, they made every block wait for all of the one before (vector
  // loads return in order), and nothing was on its way beside the block being computed.
  const auto* pages = (const __attribute__((address_space(4))) int*)(uintptr_t)bt;
  const int last_page = max_blocks - 1;
  const int page_shift = (page & (page - 1)) == 0 ? __builtin_ctz(page) : -1;
  struct Places {
    int pg[2], off[2];  // page and first key in it of keys 0 .. 15 and 16 .. 31 of a block
  };
  auto find = [&](int blk) {
    Places p;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key = blk + 16 * t, pi = page_shift >= 0 ? key >> page_shift : key / page;
      p.pg[t] = pages[pi < last_page ? pi : last_page];
      p.off[t] = key - pi * page;
    }
    return p;
  };
  auto load_block = [&](KeyBlock& B, const Places& p) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int half = RINGED ? col >> 3 : t, r = RINGED ? (col >> 2 & 1) * 8 + 4 * t + (col & 3) : col;      // of the block; the key in it
      const bf16* kp = k_cache + (((size_t)(half ? p.pg[1] : p.pg[0]) * Hkv + kvh) * page + (half ? p.off[1] : p.off[0])) * D;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int d0 = ks * 32 + kb * 8;
        B.a[t][ks].q = *reinterpret_cast<const uint4*>(kp + (r * D + (d0 < D ? d0 : 0)));
      }
    }
    const bf16* v0 = v_cache + ((size_t)p.pg[0] * Hkv + kvh) * D * page + p.off[0];
    const bf16* v1 = v_cache + ((size_t)p.pg[1] * Hkv + kvh) * D * page + p.off[1];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int at = (dt * 16 + col) * page + (RINGED ? 8 * (kb & 1) : 4 * kb);
      const bf16 *f0 = RINGED && kb >> 1 ? v1 : v0, *f1 = RINGED ? f0 + 4 : v1;
      B.va[dt].h[0] = *reinterpret_cast<const uint2*>(f0 + at);
      B.va[dt].h[1] = *reinterpret_cast<const uint2*>(f1 + at);
    }
  };
  // The slots.  Keys: row k of 32 as it stands in its page, 16-byte block b at place b ^ f(k) of it, f = k % 4 + 4 (k / 8 % 2) as far as
  // the row's blocks allow; values: a page's 16 keys of a dim are two blocks, swapped for every second four dims.  Both so
  // that eight lanes' fragment reads are in different banks.
  constexpr int SLOTS = slots_of(NW, RING), AHEAD_LOADS = RING ? (SLOTS - 1) * BLOCK_LOADS : 0;
  static_assert(AHEAD_LOADS <= 63, "more loads in flight than the counter holds");
  constexpr int NBLK = D / 8, TURN = NBLK % 8 == 0 ? 7 : 3, KL = RING ? D / 32 : 1;
  uint32_t koff[KL];
#pragma unroll
  for (int j = 0; j < KL; ++j) {
    const int i = j * 64 + lane, r = i / NBLK, place = i - r * NBLK;
    koff[j] = r * D * 2 + (place ^ (((r & 3) | ((r >> 3) << 2)) & TURN)) * 16;
  }
  const uint32_t voff = (lane >> 1) * page * 2 + ((lane & 1) ^ ((lane >> 3) & 1)) * 16;
  char* mine = da_lds + wave * SLOTS * 128 * D;
  const uint32_t mine0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)mine;
  auto issue = [&](int slot, const Places& p) {
    const uint32_t to = mine0 + slot * 128 * D;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bf16* kp = k_cache + (((size_t)p.pg[t] * Hkv + kvh) * page + p.off[t]) * D;
#pragma unroll
      for (int j = 0; j < KL; ++j) mie_load_to_lds(kp, koff[j], to + t * 32 * D + j * 1024);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bf16* vp = v_cache + ((size_t)p.pg[t] * Hkv + kvh) * D * page + p.off[t];
#pragma unroll
      for (int j = 0; j < KL; ++j) mie_load_to_lds(vp + (size_t)32 * j * page, voff, to + 64 * D + t * 32 * D + j * 1024);
    }
  };
  auto take = [&](KeyBlock& B, int slot) {
    const char* at = mine + slot * 128 * D;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        B.a[t][ks].q = *reinterpret_cast<const uint4*>(at + (8 * (col >> 2) + 4 * t + (col & 3)) * D * 2 + ((4 * ks + kb) ^ (col & TURN)) * 16);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      B.va[dt].q = *reinterpret_cast<const uint4*>(at + 64 * D + (kb >> 1) * 32 * D + (dt * 16 + col) * 32 + ((kb & 1) ^ ((col >> 2) & 1)) * 16);
  };
  // which key of a block: a lane's j-th probability, and the row of score tile t that lane column c holds
  auto key_at = [&](int blk, int j) { return RINGED ? blk + 8 * kb + j : blk + 16 * (j >> 2) + 4 * kb + (j & 3); };
  auto row_key = [&](int blk, int t) { return RINGED ? blk + 8 * (col >> 2) + 4 * t + (col & 3) : blk + 16 * t + col; };
  constexpr bool AHEAD = D <= 128;          // two blocks on their way; larger heads have no room for it
  KeyBlock b0, b1;
  const int pos_raw = positions[b];
  int begin0 = s * partition;               // the split's first key when there is no window
  const bool early = AHEAD && !CHUNK && window <= 0 && (!SIG || chunk <= 0);
  if (early) {
    if constexpr (RING) issue(0, find(begin0 + BLOCK_KEYS * wave));
    else load_block(b0, find(begin0 + BLOCK_KEYS * wave));
  }

  const int pos = pos_raw;
  if (FROM_SUMS) {
    // the row's own q, k and v from the projection's sums (the expressions of the kernel that does this alone)
    const int slot = proj.slots[b], half = D >> 1;
    const float* pr = proj.part + (size_t)b * proj.ld;
    const float* cr = proj.cos_t + (size_t)pos * half;
    const float* sr = proj.sin_t + (size_t)pos * half;
    bf16* kdst = k_cache + (((size_t)(slot / page) * Hkv + kvh) * page + (size_t)(slot % page)) * D;
    for (int t = threadIdx.x; t < (G + 1) * half; t += NW * 64) {
      const int hh = t / half, j = t - hh * half;
      const float* src = pr + (size_t)(hh < G ? kvh * G + hh : Hq + kvh) * D + j;
      float x1 = 0.f, x2 = 0.f;
      add_splits(x1, src, proj.splits, proj.split_stride);
      add_splits(x2, src + half, proj.splits, proj.split_stride);
      const float c = cr[j], sn = sr[j];
      float o1, o2;
      rotate_pair(x1, x2, c, sn, o1, o2);
      bf16* dst = hh < G ? s_q[hh] : s_k;
      dst[j] = __float2bfloat16(o1);
      dst[j + half] = __float2bfloat16(o2);
      if (hh == G) {
        kdst[j] = __float2bfloat16(o1);
        kdst[j + half] = __float2bfloat16(o2);
      }
    }
    bf16* vdst = v_cache + ((size_t)(slot / page) * Hkv + kvh) * page * D + (size_t)(slot % page);
    for (int d = threadIdx.x; d < D; d += NW * 64) {
      float v = 0.f;
      add_splits(v, pr + (size_t)(Hq + Hkv + kvh) * D + d, proj.splits, proj.split_stride);
      vdst[(size_t)d * page] = __float2bfloat16(v);
      s_v[d] = __float2bfloat16(v);
    }
    // The waves meet over what went into the LDS only; the stores to the cache are not waited for, because
    // nobody here reads them back: the block that holds the row's own key takes it from the LDS (compute()).
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = ks * 32 + kb * 8;
      if (head_ok && d0 < D) qf[ks].q = *reinterpret_cast<const uint4*>(&s_q[g][d0]);
    }
  }
  int lo = window > 0 ? (pos - window + 1 > 0 ? pos - window + 1 : 0) : 0;
  // DB: the lane's head's row of the distance table (entries already times log2 e)
  const float* __restrict__ db_row = DB ? dist_bias + (size_t)head * dist_n : nullptr;
  float sg_c1 = 0.f, sg_c2 = 0.f, sg_c3 = 0.f;
  if constexpr (SIG || CHUNK) {
    if (chunk > 0 && pos / chunk * chunk > lo) lo = pos / chunk * chunk;
  }
  if constexpr (SIG) {
    const float hb = head_bias ? head_bias[head] : 0.f;
    const float L2E = 1.4426950408889634f;
    if (softcap > 0.f) {
      sg_c1 = 2.f * L2E * scale_log2 / softcap;
      sg_c2 = 2.f * L2E * softcap;
      sg_c3 = -L2E * (softcap + hb);
    } else {
      sg_c1 = -L2E * scale_log2;
      sg_c3 = -L2E * hb;
    }
  }
  int gap = 0, kept_end = 0;
  if constexpr (KEEP) {
    kept_end = (keep + BLOCK_KEYS - 1) & ~(BLOCK_KEYS - 1);
    gap = (lo & ~(BLOCK_KEYS - 1)) - kept_end;
    gap = gap > 0 ? gap : 0;
  }
  const int last_x = pos - gap;                // place of the row's own key in the order the blocks are walked
  auto key_of = [&](int x) { return !KEEP || x < kept_end ? x : x + gap; };
  const int begin = (KEEP ? 0 : lo & ~(BLOCK_KEYS - 1)) + s * partition;
  const int end = begin + partition < last_x + 1 ? begin + partition : last_x + 1;

  if (begin > last_x) {
    if (RING) MIE_VMCNT(0);      // nothing of this wave may still be writing the LDS when it ends
    // this split lies beyond the row's keys (uniform over the workgroup)
    if (num_splits > 1 && threadIdx.x < 16 && ht * 16 + (int)threadIdx.x < G)
      lse_part[((size_t)b * Hq + kvh * G + ht * 16 + threadIdx.x) * num_splits + s] = -INFINITY;
    return;
  }

  float m = -INFINITY, l = 0.f;
  f32x4 O[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](KeyBlock& B, int blk) {
    if (FROM_SUMS && pos >= blk && pos < blk + BLOCK_KEYS) {       // (the same for the whole wave)
      // what was loaded for the row's own key is whatever its slot held: the key and value come from the LDS
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if (row_key(blk, t) == pos) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            const int d0 = ks * 32 + kb * 8;
            B.a[t][ks].q = *reinterpret_cast<const uint4*>(&s_k[d0 < D ? d0 : 0]);
          }
        }
#pragma unroll
      for (int wi = 0; wi < 4; ++wi) {                           // word wi of a value fragment: two keys
        const int key = key_at(blk, 2 * wi);
        const bool low = key == pos, high = key + 1 == pos;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const uint32_t nv = (uint32_t)__bfloat16_as_ushort(s_v[dt * 16 + col]);
          const uint32_t w = B.va[dt].w[wi];
          B.va[dt].w[wi] = low ? (w & 0xFFFF0000u) | nv : (high ? (w & 0x0000FFFFu) | (nv << 16) : w);
        }
      }
    }
    if (D % 32 != 0) {
      // the last 32-dim step of the keys is half empty: its upper lanes were loaded from dim 0
#pragma unroll
      for (int t = 0; t < 2; ++t)
        if ((KS - 1) * 32 + kb * 8 >= D) B.a[t][KS - 1].q = make_uint4(0, 0, 0, 0);
    }
    // ---- scores of 32 keys x 16 heads
    f32x4 S[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      S[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        S[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B.a[t][ks].v, qf[ks].v, S[t], 0, 0, 0);
    }
    const bool partial = blk + BLOCK_KEYS > pos + 1 || (blk < lo && (!KEEP || blk + BLOCK_KEYS > keep));
    if constexpr (SIG) {
      bool ok[8];
      float p[8];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key_at(blk, 4 * t + i);
          ok[t * 4 + i] = key >= lo && key <= pos;
          float w;
          if (softcap > 0.f) {
            const float r = __builtin_amdgcn_rcpf(1.f + fast_exp2(S[t][i] * sg_c1));
            w = __builtin_amdgcn_rcpf(1.f + fast_exp2(fmaf(r, sg_c2, sg_c3)));
          } else {
            w = __builtin_amdgcn_rcpf(1.f + fast_exp2(fmaf(S[t][i], sg_c1, sg_c3)));
          }
          p[t * 4 + i] = ok[t * 4 + i] ? w : 0.f;
        }
      Frag pb;
#pragma unroll
      for (int j = 0; j < 4; ++j) pb.w[j] = pack_bf16(p[2 * j], p[2 * j + 1]);
      if (partial) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            uint32_t w = B.va[dt].w[j];
            if (!ok[2 * j]) w &= 0xFFFF0000u;
            if (!ok[2 * j + 1]) w &= 0x0000FFFFu;
            B.va[dt].w[j] = w;
          }
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) O[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B.va[dt].v, pb.v, O[dt], 0, 0, 0);
      return;
    }
    // ---- online softmax, one head per lane column
    float sv[8];
    bool ok[8];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key_at(blk, 4 * t + i);
        ok[t * 4 + i] = (key >= lo || (KEEP && key < keep)) && key <= pos;
        if constexpr (DB) {
          int n = pos - key;
          n = n < 0 ? 0 : (n < dist_n ? n : dist_n - 1);            // a key after the row's own is masked
          sv[t * 4 + i] = ok[t * 4 + i] ? fmaf(S[t][i], scale_log2, db_row[n]) : -INFINITY;
        } else {
          sv[t * 4 + i] = ok[t * 4 + i] ? S[t][i] * scale_log2 : -INFINITY;
        }
        mx = fmaxf(mx, sv[t * 4 + i]);
      }
    const float m_new = fmaxf(m, quad_max(mx));         // finite: every block taken holds a visible key
    // exp2f: weights and factors below 2^-126 keep what a 32-bit number holds of them, where the hardware's exponential alone gives 0 (64
    // rows of 200 to 1,990 keys 20.9 us for 20.5, 8 of 1,000 to 6,000 34.3 for 33.8; exp2f only in blocks that have such a weight 20.6
    // and 37.9, MI355X).
    const float alpha = exp2f(m - m_new);
    float p[8], rs = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = ok[j] ? exp2f(sv[j] - m_new) : 0.f;
      rs += p[j];
    }
    l = l * alpha + rs;                                 // of this lane's keys; the head's four lanes join after the last block
    m = m_new;
    Frag pb;
#pragma unroll
    for (int j = 0; j < 4; ++j) pb.w[j] = pack_bf16(p[2 * j], p[2 * j + 1]);
    if (partial) {
      // zero the values of keys outside [lo, pos]: 0 * (stale NaN) must not reach the sum
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t w = B.va[dt].w[j];
          if (!ok[2 * j]) w &= 0xFFFF0000u;
          if (!ok[2 * j + 1]) w &= 0x0000FFFFu;
          B.va[dt].w[j] = w;
        }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      O[dt] *= alpha;
      O[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B.va[dt].v, pb.v, O[dt], 0, 0, 0);
    }
  };

  constexpr int STEP = BLOCK_KEYS * NW;     // keys from one block of a wave to its next
  const int first = begin + BLOCK_KEYS * wave;
  if constexpr (RING) {
    const int count = first < end ? (end - first + STEP - 1) / STEP : 0;       // this wave's blocks: nothing beyond the split's own keys
#pragma unroll
    for (int i = 0; i < SLOTS; ++i)
      if (i < count && !(i == 0 && early)) issue(i, find(key_of(first + i * STEP)));
    Places next = find(key_of(first + SLOTS * STEP));
    for (int it = 0; it < count; ++it) {
      if (it + SLOTS <= count) MIE_VMCNT(AHEAD_LOADS);                  // block `it` has landed
      else MIE_VMCNT(0);
      asm volatile("" ::: "memory");
      take(b0, it % SLOTS);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                       // read: the slot is free
      if (it + SLOTS < count) {
        issue(it % SLOTS, next);
        next = find(key_of(first + (it + SLOTS + 1) * STEP));
      }
      compute(b0, key_of(first + it * STEP));
    }
    MIE_VMCNT(0);                           // (a wave without a block may have asked for one early)
  } else if (AHEAD) {
    if (CHUNK || window > 0 || (SIG && chunk > 0)) load_block(b0, find(key_of(first)));  // with a window the split's start had to wait for the row's length
    const int part_end = begin + partition;   // nothing is asked for beyond the split's own keys
    Places next = find(key_of(first + STEP));
    for (int blk = first; blk < end; blk += 2 * STEP) {
      if (blk + STEP < part_end) load_block(b1, next);                         // in flight while block 0 is computed
      next = find(key_of(blk + 2 * STEP));
      compute(b0, key_of(blk));
      if (blk + 2 * STEP < part_end) load_block(b0, next);
      next = find(key_of(blk + 3 * STEP));
      if (blk + STEP < end) compute(b1, key_of(blk + STEP));
    }
  } else {
    for (int blk = first; blk < end; blk += STEP) {
      load_block(b0, find(key_of(blk)));
      compute(b0, key_of(blk));
    }
  }

  // ---- merge the waves of the workgroup
  if constexpr (SIG) {
    m = 0.f;
    l = wave == 0 ? 1.f : 0.f;
  } else {
    l = quad_sum(l);
  }
  if (kb == 0) {
    s_m[wave][col] = m;
    s_l[wave][col] = l;
  }
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, s_m[w][col]);
  float L = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float mw = s_m[w][col];
    L += mw == -INFINITY ? 0.f : exp2f(mw - M) * s_l[w][col];
  }
  const float f = m == -INFINITY ? 0.f : exp2f(m - M);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) s_o[(wave * 16 + col) * (D + 1) + dt * 16 + 4 * kb + i] = O[dt][i] * f;
  if (wave == 0 && kb == 0) {
    s_M[col] = M;
    s_L[col] = L;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * D; e += NW * 64) {
    const int hc = e / D, d = e - hc * D;
    const int gg = ht * 16 + hc;
    if (gg >= G) continue;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += s_o[(w * 16 + hc) * (D + 1) + d];
    const size_t hh = (size_t)b * Hq + kvh * G + gg;
    if (num_splits == 1) {
      // a sink (sink_log2 > -inf) is one more term in the denominator; with splits the merge kernel adds it
      const float sk = head_sinks ? head_sinks[kvh * G + gg] : sink_log2;
      out[hh * D + d] = __float2bfloat16(sum / (s_L[hc] + exp2f(sk - s_M[hc])));
    } else {
      const float val = sum / s_L[hc];
      o_part[(hh * num_splits + s) * D + d] = val;
      if (d == 0) lse_part[hh * num_splits + s] = s_M[hc] + log2f(s_L[hc]);
    }
  }
}

// One wave per (row, head): lane s takes the log-sum-exp of split s (the wave reduces max and sum with
// shuffles), then the lanes spread over D and add the splits' partials with all loads of a chunk of 16
// splits issued together: two memory round trips in all, whatever the number of splits.
// (Merging inside the attention kernel by the split that arrives last was tried: the partials have to
// cross the per-XCD L2s, and the device-scope fences that takes cost far more than this launch.)
__global__ void __launch_bounds__(64)
merge_splits_kernel(const float* __restrict__ o_part, const float* __restrict__ lse_part, bf16* __restrict__ out,
                    int num_splits, float sink_log2, int plain_sum, const float* __restrict__ head_sinks, int Hq) {
  constexpr int DL = (D + 63) / 64;
  const size_t hh = blockIdx.x;
  const int lane = threadIdx.x;
  const float* lse = lse_part + hh * num_splits;
  const float* op = o_part + hh * num_splits * D;
  float acc[DL];
#pragma unroll
  for (int i = 0; i < DL; ++i) acc[i] = 0.f;
  // Sixteen splits' partial outputs at a time.  The first sixteen are asked for before their weights are
  // known, so that the kernel waits for memory once and not twice; every load is unconditional, from an
  // address clamped into the operand (what is read for a split or a dim that does not exist is not used).
  float part[16][DL];
  auto ask = [&](int first) {
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
      for (int i = 0; i < DL; ++i) {
        const int d = lane + 64 * i, sp = first + j;
        part[j][i] = op[(size_t)(sp < num_splits ? sp : num_splits - 1) * D + (d < D ? d : 0)];
      }
  };
  ask(0);
  if (head_sinks) sink_log2 = head_sinks[hh % Hq];
  float W = 0.f;
  float M = -INFINITY;                       // the maximum over all splits first (64 a round)
  for (int s0 = 0; s0 < num_splits; s0 += 64) {
    const float v = lse[s0 + lane < num_splits ? s0 + lane : 0];
    M = fmaxf(M, wave_max(s0 + lane < num_splits ? v : -INFINITY));
  }
  for (int s0 = 0; s0 < num_splits; s0 += 64) {
    const float vv = lse[s0 + lane < num_splits ? s0 + lane : 0];
    const float v = s0 + lane < num_splits ? vv : -INFINITY;
    const float w = v == -INFINITY ? 0.f : exp2f(v - M);
    W += wave_sum(w);
    const int n = num_splits - s0 < 64 ? num_splits - s0 : 64;
    for (int c = 0; c < n; c += 16) {
      if (s0 + c > 0) ask(s0 + c);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float wj = __shfl(w, (c + j) & 63, 64);
#pragma unroll
        for (int i = 0; i < DL; ++i)
          if (c + j < n && wj != 0.f && lane + 64 * i < D) acc[i] += wj * part[j][i];    // a split without keys holds no data
      }
    }
  }
  // the sink's term, if there is one (else exp2(-inf) = 0); sigmoid weights (plain_sum) are not normalised
  const float inv = plain_sum ? 1.0f : 1.0f / (W + exp2f(sink_log2 - M));
#pragma unroll
  for (int i = 0; i < DL; ++i) {
    const int d = lane + 64 * i;
    if (d < D) out[hh * D + d] = __float2bfloat16(acc[i] * inv);
  }
}
