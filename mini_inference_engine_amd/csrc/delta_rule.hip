// The delta-rule recurrence over a step's rows, with the request's state in its slot; everything is 32-bit.
//
// Per head a state S [d, d] (key channel i, value channel j):
//     S <- diag(decay) S - (a * u) (u^T S) + k v^T   (both terms of the old S),   o = S^T r.
// delta_prepare: a workgroup a token, from the projection's float32 sums: decay = exp(-decay_scale *
//     sigmoid(W tanh(inner) + bias)) (the product over the inner size in FMAs, ascending), a = sigmoid(a + bias),
//     the unit key u = k / sqrt(sum(k^2) + 1e-6) of each head -> prep [T, 3, H d] = decay, a * u, u.
// delta_scan: a workgroup a (row, chunk, head), thread j owns column j of S in registers (every term of the update of
//     column j reads that column only), tokens in order.  What all columns share (decay, a * u, u, k, r of a token) comes
//     in through the LDS, eight tokens at a time, the next eight on their way meanwhile.  The head's output is divided by
//     its root mean square, times the weight and the sigmoid of the output gate, and rounded once.
//
// Rows run whole (one chunk: S from state[slot], left there afterwards), or, long rows, in chunks on the matrix cores (below) or,
// what those do not take, in chunks of L tokens side by side in three passes, since a chunk acts on the state it starts from as S_end = P S_start + B with P and B of the
// chunk's own tokens:  (1) every chunk but a row's last computes P (the recurrence without k v^T on the identity) and
// B (the recurrence on zero), a thread carrying the same column of both;  (2) per row and head, chunk after chunk, S_start(c + 1) = P_c S_start(c) + B_c from
// state[slot] (16 columns a workgroup; columns do not mix);  (3) every chunk runs its tokens from its S_start and writes
// the outputs, a row's last chunk leaves state[slot].  The two ways differ by the rounding of pass 2 alone.
#include "launch.hpp"

constexpr int PT_MAX = 16;       // most tokens a workgroup of delta_prepare takes: a channel's row of the decay matrix is read once for all of them

// RMAX > 0: inner sizes up to RMAX, the channel's row of the matrix in registers; 0: any inner size, the row read from memory
template <int RMAX>
__global__ void __launch_bounds__(256)
delta_prepare_kernel(const float* __restrict__ sums, long ld, int k_col, int a_col, int w_col, const float* __restrict__ w_decay,
                     int rank, const float* __restrict__ decay_bias, float decay_scale, const float* __restrict__ removal_bias,
                     float* __restrict__ prep, int tokens, int H, int d, int heads_here, int PT) {
  extern __shared__ __align__(16) float prep_lds[];
  const int rank4 = RMAX > 0 ? RMAX : (rank + 3) & ~3;
  float* inner = prep_lds;                       // [PT][rank4]: the decay's inner activations after their tanh
  float* ssq = prep_lds + (size_t)PT * rank4;    // [PT][heads_here]: sum of squares of the keys of the heads this workgroup touches
  const int t0 = blockIdx.x * PT, n = H * d;
  const int nt = tokens - t0 < PT ? tokens - t0 : PT;
  const int c0 = blockIdx.y * 256, h0 = c0 / d;
  for (int e = threadIdx.x; e < nt * rank4; e += blockDim.x) {
    const int tt = e / rank4, j = e % rank4;
    inner[e] = j < rank ? tanhf(sums[(size_t)(t0 + tt) * ld + w_col + j]) : 0.f;
  }
  for (int e = threadIdx.x; e < nt * heads_here; e += blockDim.x) {
    const int tt = e / heads_here, h = h0 + e % heads_here;
    float s = 0.f;
    if (h < H) {
      const float* kh = sums + (size_t)(t0 + tt) * ld + k_col + (size_t)h * d;
      if ((d & 3) == 0 && (((uintptr_t)kh) & 15) == 0) {          // the same order whatever the step holds, either way
#pragma unroll 4
        for (int i = 0; i < d; i += 4) {
          const float4 v = *reinterpret_cast<const float4*>(kh + i);
          s = fmaf(v.x, v.x, s);
          s = fmaf(v.y, v.y, s);
          s = fmaf(v.z, v.z, s);
          s = fmaf(v.w, v.w, s);
        }
      } else {
        for (int i = 0; i < d; ++i) s = fmaf(kh[i], kh[i], s);
      }
    }
    ssq[e] = s;
  }
  __syncthreads();
  const int c = c0 + threadIdx.x;                // a thread a channel
  if (c >= n) return;
  const float* w = w_decay + (size_t)c * rank;
  const float zb = decay_bias[c], rb = removal_bias[c];
  const int hl = c / d - h0;
  const bool vec = (rank & 3) == 0 && (((uintptr_t)w_decay) & 15) == 0;
  float wreg[RMAX > 0 ? RMAX : 1];
  if (RMAX > 0) {
#pragma unroll
    for (int j = 0; j < RMAX; ++j) wreg[j] = j < rank ? w[j] : 0.f;
  }
  for (int tt = 0; tt < nt; ++tt) {
    float z = zb;
    const float* in = inner + (size_t)tt * rank4;
    if (RMAX > 0) {
#pragma unroll
      for (int j = 0; j < RMAX; j += 4) {          // inner is zero beyond the inner size
        const float4 iv = *reinterpret_cast<const float4*>(in + j);
        z = fmaf(wreg[j], iv.x, z);
        z = fmaf(wreg[j + 1], iv.y, z);
        z = fmaf(wreg[j + 2], iv.z, z);
        z = fmaf(wreg[j + 3], iv.w, z);
      }
    } else if (vec) {
      for (int j = 0; j < rank; j += 4) {        // the row of the matrix stays in the cache nearest this thread over the tokens
        const float4 wv = *reinterpret_cast<const float4*>(w + j);
        const float4 iv = *reinterpret_cast<const float4*>(in + j);
        z = fmaf(wv.x, iv.x, z);
        z = fmaf(wv.y, iv.y, z);
        z = fmaf(wv.z, iv.z, z);
        z = fmaf(wv.w, iv.w, z);
      }
    } else {
      for (int j = 0; j < rank; ++j) z = fmaf(w[j], in[j], z);
    }
    const float* row = sums + (size_t)(t0 + tt) * ld;
    const float a = mie_sigmoid(row[a_col + c] + rb);
    const float u = row[k_col + c] / sqrtf(ssq[tt * heads_here + hl] + 1e-6f);
    float* out = prep + (size_t)(t0 + tt) * 3 * n;
    out[c] = expf(-decay_scale * mie_sigmoid(z));
    out[n + c] = a * u;
    out[2 * n + c] = u;
  }
}

enum { SCAN_WHOLE = 0, SCAN_SUMMARY = 1, SCAN_FROM_START = 2 };
constexpr int TB = 8;            // tokens a block of the LDS
constexpr int NV = 6;            // vectors a token: decay, a * u, u, k, r, v

struct ScanArgs {
  const float* sums; long ld; int r_col, k_col, v_col, g_col;
  const float* prep; const float* norm_weight; float eps;
  float* state; const int* row_start; const int* slots; void* out;
  float* summaries;      // [rows * max_chunks, H, 2, d, d]: B, P of a chunk
  float* starts;         // [rows * max_chunks, H, d, d]: the state a chunk starts from
  int H, d, L, max_chunks, mode;
};

template <int DMAX, typename TO, bool SUMMARY>
__global__ void __launch_bounds__(DMAX < 64 ? 64 : DMAX)
delta_scan_kernel(ScanArgs a) {
  constexpr int NT = DMAX < 64 ? 64 : DMAX;
  __shared__ float scratch[16];
  __shared__ __align__(16) float stage[TB][NV][DMAX];   // channels beyond the head's size hold zeros
  const int row = blockIdx.x / a.max_chunks, chunk = blockIdx.x % a.max_chunks, h = blockIdx.y, j = threadIdx.x;
  const int d = a.d, n = a.H * d;
  const int row_end = a.row_start[row + 1];
  const int t0 = a.row_start[row] + chunk * a.L;
  if (t0 >= row_end) return;                                   // the whole workgroup: this row has no such chunk
  const int t1 = t0 + a.L < row_end ? t0 + a.L : row_end;
  const bool last = t1 == row_end;
  constexpr bool summary = SUMMARY;                            // one thread carries column j of B (in S) and of P (in Q)
  if (summary && last) return;                                 // nobody starts from the end of a row's last chunk
  const bool live = j < d;
  const int jj = live ? j : 0;
  float* sp = a.state + ((size_t)a.slots[row] * a.H + h) * d * d;
  const size_t ch = (size_t)blockIdx.x * a.H + h;
  float S[DMAX];
  float Q[SUMMARY ? DMAX : 1];
  if (summary) {
#pragma unroll
    for (int i = 0; i < DMAX; ++i) S[i] = 0.f;
#pragma unroll
    for (int i = 0; i < (SUMMARY ? DMAX : 1); ++i) Q[i] = live && i == j ? 1.f : 0.f;
  } else {
    const float* from = a.mode == SCAN_FROM_START ? a.starts + ch * d * d : sp;
#pragma unroll
    for (int i = 0; i < DMAX; ++i) S[i] = i < d ? from[(size_t)i * d + jj] : 0.f;
  }
  const float nw = a.norm_weight[h * d + jj];
  int lane0;
  asm volatile("v_mov_b32 %0, 0" : "=v"(lane0));
  // thread j brings channel j of a token's six vectors in, for TB tokens at a time (zeros beyond the head's size and
  // beyond the chunk, so that the loops below need no bounds: a channel that is not there keeps S at zero)
  constexpr int PER = TB * NV;
  float nxt[PER];
  const size_t hj = (size_t)h * d + jj;
  auto fetch = [&](int tb) {
#pragma unroll
    for (int tt = 0; tt < TB; ++tt) {
      const int t = tb + tt < t1 ? tb + tt : t1 - 1;            // clamped: what is read beyond the chunk is not used
      const bool ok = live && tb + tt < t1;
      const float* prow = a.prep + (size_t)t * 3 * n + hj;
      const float* srow = a.sums + (size_t)t * a.ld + hj;
      nxt[tt * NV + 0] = ok ? prow[0] : 0.f;
      nxt[tt * NV + 1] = ok ? prow[n] : 0.f;
      nxt[tt * NV + 2] = ok ? prow[2 * n] : 0.f;
      nxt[tt * NV + 3] = ok ? srow[a.k_col] : 0.f;
      nxt[tt * NV + 4] = ok ? srow[a.r_col] : 0.f;
      nxt[tt * NV + 5] = ok ? srow[a.v_col] : 0.f;
    }
  };
  fetch(t0);
  TO* out = (TO*)a.out;
  for (int tb = t0; tb < t1; tb += TB) {
    __syncthreads();                                           // the block before is used up
    if (j < DMAX) {
#pragma unroll
      for (int p = 0; p < PER; ++p) stage[p / NV][p % NV][j] = nxt[p];
    }
    __syncthreads();
    if (tb + TB < t1) fetch(tb + TB);
    const int nt = t1 - tb < TB ? t1 - tb : TB;
    for (int tt = 0; tt < nt; ++tt) {
      // What every column shares is read by every lane from the same LDS address.  ``lane0`` is a zero the compiler
      // cannot see through: without it the values count as uniform, are moved to scalar registers, and those run out.
      const float* decay = stage[tt][0] + lane0;
      const float* au = stage[tt][1] + lane0;
      const float* u = stage[tt][2] + lane0;
      const float* k = stage[tt][3] + lane0;
      const float* r = stage[tt][4] + lane0;
      const float v = stage[tt][5][jj];
      float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f, q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
#pragma unroll
      for (int i = 0; i < DMAX; i += 4) {
        s0 = fmaf(u[i], S[i], s0);
        s1 = fmaf(u[i + 1], S[i + 1], s1);
        s2 = fmaf(u[i + 2], S[i + 2], s2);
        s3 = fmaf(u[i + 3], S[i + 3], s3);
        if (summary) {
          q0 = fmaf(u[i], Q[i], q0);
          q1 = fmaf(u[i + 1], Q[i + 1], q1);
          q2 = fmaf(u[i + 2], Q[i + 2], q2);
          q3 = fmaf(u[i + 3], Q[i + 3], q3);
        }
      }
      const float seen = (s0 + s1) + (s2 + s3), seen_q = (q0 + q1) + (q2 + q3);
      float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;
#pragma unroll
      for (int i = 0; i < DMAX; i += 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          S[i + e] = fmaf(k[i + e], v, fmaf(-au[i + e], seen, decay[i + e] * S[i + e]));
          if (summary) Q[i + e] = fmaf(-au[i + e], seen_q, decay[i + e] * Q[i + e]);       // no k v^T: what the start state becomes
        }
        if (!summary) {
          o0 = fmaf(S[i], r[i], o0);
          o1 = fmaf(S[i + 1], r[i + 1], o1);
          o2 = fmaf(S[i + 2], r[i + 2], o2);
          o3 = fmaf(S[i + 3], r[i + 3], o3);
        }
      }
      if (!summary) {
        const float o = (o0 + o1) + (o2 + o3);
        const float sq = live ? o * o : 0.f;
        const float total = DMAX <= 64 ? wave_sum(sq) : block_sum(sq, scratch);
        const float rstd = 1.0f / sqrtf(total / (float)d + a.eps);
        const int t = tb + tt;
        if (live)
          out[(size_t)t * n + h * d + j] = from_float<TO>(o * rstd * nw * mie_sigmoid(a.sums[(size_t)t * a.ld + a.g_col + h * d + j]));
      }
    }
  }
  if (!live) return;
  float* to = summary ? a.summaries + ch * 2 * d * d : sp;
  if (summary || last) {
#pragma unroll
    for (int i = 0; i < DMAX; ++i)
      if (i < d) to[(size_t)i * d + j] = S[i];
  }
  if (summary) {
#pragma unroll
    for (int i = 0; i < (SUMMARY ? DMAX : 1); ++i)
      if (i < d) to[(size_t)(d + i) * d + j] = Q[i];
  }
}

// Pass 2: per (row, head, block of 16 columns), chunk after chunk: start(c + 1) = P_c start(c) + B_c, start(0) = state[slot].
// The column block of start(c) and the whole of P_c sit in the LDS; a thread makes four neighbouring columns of a row.
__global__ void __launch_bounds__(256)
delta_fold_kernel(const float* __restrict__ summaries, float* __restrict__ starts, const float* __restrict__ state,
                  const int* __restrict__ row_start, const int* __restrict__ slots, int H, int d, int L, int max_chunks) {
  extern __shared__ __align__(16) float fold_lds[];
  float* col = fold_lds;                         // [d][16]
  float* pm = fold_lds + (size_t)d * 16;         // [d][d + 1]
  const int row = blockIdx.x, h = blockIdx.y, j0 = blockIdx.z * 16;
  const int tokens = row_start[row + 1] - row_start[row];
  const int chunks = (tokens + L - 1) / L;
  const float* sp = state + ((size_t)slots[row] * H + h) * d * d;
  for (int e = threadIdx.x; e < d * 16; e += blockDim.x) {
    const int i = e / 16, jl = e % 16;
    col[e] = j0 + jl < d ? sp[(size_t)i * d + j0 + jl] : 0.f;
  }
  __syncthreads();
  // P of a chunk comes in through registers while the chunk before is folded (d * d / 256 numbers a thread)
  const int per = (d * d + 255) / 256;
  float pre[16];                                 // the first 16 of them; the rest, for d > 64, is read when needed
  auto ask = [&](int c) {
    const float* P = summaries + ((((size_t)row * max_chunks + c) * H + h) * 2 + 1) * d * d;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int e = threadIdx.x + k * 256;
      pre[k] = (k < per && e < d * d) ? P[e] : 0.f;
    }
  };
  if (chunks > 1) ask(0);
  for (int c = 0; c < chunks; ++c) {
    const size_t ch = ((size_t)row * max_chunks + c) * H + h;
    float* st = starts + ch * d * d;
    for (int e = threadIdx.x; e < d * 16; e += blockDim.x)
      if (j0 + e % 16 < d) st[(size_t)(e / 16) * d + j0 + e % 16] = col[e];
    if (c + 1 == chunks) break;
    const float* B = summaries + ch * 2 * d * d;
    const float* P = B + (size_t)d * d;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int e = threadIdx.x + k * 256;
      if (k < per && e < d * d) pm[(e / d) * (d + 1) + e % d] = pre[k];
    }
    for (int e = threadIdx.x + 16 * 256; e < d * d; e += blockDim.x) pm[(e / d) * (d + 1) + e % d] = P[e];
    __syncthreads();
    if (c + 2 < chunks) ask(c + 1);
    // every thread's new values first (up to four quads of columns at d = 256), then all of them into the LDS
    float4 fresh[4];
#pragma unroll
    for (int cnt = 0; cnt < 4; ++cnt) {
      const int q = threadIdx.x + cnt * 256;
      if (q >= d * 4) break;
      const int i = q / 4, jq = (q % 4) * 4;
      float4 acc;
      acc.x = j0 + jq < d ? B[(size_t)i * d + j0 + jq] : 0.f;
      acc.y = j0 + jq + 1 < d ? B[(size_t)i * d + j0 + jq + 1] : 0.f;
      acc.z = j0 + jq + 2 < d ? B[(size_t)i * d + j0 + jq + 2] : 0.f;
      acc.w = j0 + jq + 3 < d ? B[(size_t)i * d + j0 + jq + 3] : 0.f;
      const float* pr = pm + (size_t)i * (d + 1);
      for (int m = 0; m < d; ++m) {
        const float p = pr[m];
        const float4 sv = *reinterpret_cast<const float4*>(col + m * 16 + jq);
        acc.x = fmaf(p, sv.x, acc.x);
        acc.y = fmaf(p, sv.y, acc.y);
        acc.z = fmaf(p, sv.z, acc.z);
        acc.w = fmaf(p, sv.w, acc.w);
      }
      fresh[cnt] = acc;
    }
    __syncthreads();
#pragma unroll
    for (int cnt = 0; cnt < 4; ++cnt) {
      const int q = threadIdx.x + cnt * 256;
      if (q < d * 4) *reinterpret_cast<float4*>(col + (q / 4) * 16 + (q % 4) * 4) = fresh[cnt];
    }
    __syncthreads();
  }
}

// ---- long rows on the matrix cores: chunks of 64 tokens, heads of up to 64, in 32-bit (v_mfma_f32_16x16x4_f32)
//
// With w = a * u, P_t the product of a chunk's decays up to token t (a number a channel) and y_t = S_(t-1)^T u_t, unrolled from
// the state S_0 the chunk starts from (the triangular-solve form of the chunked delta rule: the WY representation of a product of
// rank-one updates, with a decay a channel):
//     S_t = P_t S_0 + sum_(s <= t) P_t / P_s (k_s v_s^T - w_s y_s^T)
//     (I + A) y = (P_(t-1) u) S_0 + B v,      A_ts = sum_i u_ti w_si P_(t-1)i / P_si  (s < t),   B the same with k_s for w_s
//     o = (P_t r) S_0 + Qk v - Qw y,          Qk_ts = sum_i r_ti k_si P_ti / P_si  (s <= t),     Qw the same with w_s
// so with [W | U] = (I + A)^-1 [P_(t-1) u | B v] a chunk acts on S_0 by four 64 x 64 matrices:
//     S_end = P S_0 + E,  P = P_end - (P_end / P_s w)^T W,  E = (P_end / P_s k)^T v - (P_end / P_s w)^T U
//     o = R S_0 + F,      R = P_t r - Qw W,                 F = Qk v - Qw U
// (1) chunk_solve, a workgroup a (chunk, head): from the projection's sums to P, E, R, F;  (2) chunk_fold, per (row, head, 16
// columns), chunk after chunk: S_0 of every chunk;  (3) chunk_outputs: o, its norm, weight and gate.
// The products run on the matrix cores, so a quotient P_t / P_s is the factor of t from the start of its 16 on, the decays of the
// 16s between, and the factor of s up to the end of its own 16; inside one 16 the reciprocal of s's factor from its start on.
// Every factor is a product of decays, and every sum of 64 terms is four chains of 16 that meet at the end: each number is then
// a few roundings from true, as in the token-by-token recurrence.  (Powers of differences of summed logarithms carry a logarithm's
// absolute rounding, and one chain over 64 or 128 terms four times as many roundings.)  Relative error of the state
// against 64 bits, 1e-8, 512 tokens of heads of 64, decay scales 0.61 / 1 / 2 / 4 (MI355X): 9.6 / 8.2 / 9.1 / 9.5; with powers and
// long chains 24 / 24 / 33 / 55; token by token 9.6 / 8.4 / 8.8 / 9.5.  Beyond DELTA_SCALE_MAX the token-by-token chunks are up to
// a third more exact with other weights (heads of 32, scale 4: 4.4 against 6.2), so they take what lies there.
// What bounds it: the solve's chain of small products (about 440 matrix instructions a SIMD and chunk) and its 32-bit arithmetic,
// a workgroup a compute unit.  2,048 tokens of 16 heads of 64 (MI355X): 40 + 168 + 142 + 175 us (preparation, summaries, fold,
// chunks, token by token through the LDS) -> 73 + 31 + 18 us.  The token-by-token chunks stay for heads of 65 to 128, other inner
// sizes and stronger decays.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int CH = 64, MS = CH + 4;
constexpr float DELTA_SCALE_MAX = 1.f;
constexpr int SOLVE_THREADS = 512;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// four chains of a sum meet
__device__ __forceinline__ f32x4 meet(const f32x4 (&p)[4]) { return (p[0] + p[1]) + (p[2] + p[3]); }
// 1 / x to within a rounding or so, x a normal number
__device__ __forceinline__ float reciprocal(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}
// The waves meet over the LDS only: loads and stores of global memory stay on their way (__syncthreads would wait for them)
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

struct ChunkArgs {
  const float* sums; long ld; int r_col, k_col, v_col, g_col, a_col, w_col;
  const float* w_decay; int rank; const float* decay_bias; float decay_scale; const float* removal_bias;
  const float* norm_weight; float eps;
  float* state; const int* row_start; const int* slots; void* out;
  float *P, *E, *R, *F, *S0;       // [units * H][DP or 64][DP]; S0 [units * H][DP][DP]
  int H, d, first_row, rows, units;           // rows [first_row, first_row + rows), their chunks in `units` places
};

// Places for the chunks of `rows` rows of together `tokens` tokens.  The chunks of the rows' k-th begin at place
// chunk_places(tokens before it, k): a row of n tokens is then ceil(n / 64) = chunk_places(n, 1) or more from the next one's,
// without a sum over the rows' chunks, and what lies between is less than a place a row.  (As many places a row as the longest has
// chunks were 2.1 GB a layer for a prompt of 1,000 tokens beside 100 portions of 10, 16 heads of 64; so 0.16 GB.)
__host__ __device__ __forceinline__ int chunk_places(int tokens, int rows) { return (int)((tokens + (long)(CH - 1) * rows) / CH); }

// Every wave looks for its place's row, 64 rows at a time: the last that begins at it or before
__device__ __forceinline__ int row_of_place(const ChunkArgs& a, int place) {
  if (a.rows == 1) return 0;           // (the prompt by itself need not wait for the loads below)
  const int* __restrict__ start = a.row_start + a.first_row;
  const int lane = threadIdx.x & 63, t0 = start[0];
  int k = 0;
  for (int base = 0; base < a.rows; base += 64) {
    const int at = base + lane;
    const int n = __popcll(__builtin_amdgcn_ballot_w64(at < a.rows && chunk_places(start[at < a.rows ? at : 0] - t0, at) <= place));
    k += n;
    if (n < 64) break;
  }
  return k - 1;
}

#define CHUNK_OF_ROW                                                                                                    \
  const int place = blockIdx.y + gridDim.y * blockIdx.z;                                                                \
  if (place >= a.units) return;                                                                                         \
  const int rr = row_of_place(a, place), row = a.first_row + rr, h = blockIdx.x;                                        \
  const int ci = place - (rr ? chunk_places(a.row_start[row] - a.row_start[a.first_row], rr) : 0);                      \
  const int t0 = a.row_start[row] + ci * CH, t_end = a.row_start[row + 1];                                              \
  if (t0 >= t_end) return;                                                                                              \
  const int nt = t_end - t0 < CH ? t_end - t0 : CH;                                                                     \
  const size_t unit = (size_t)place * a.H + h

template <int DP>
__global__ void __launch_bounds__(SOLVE_THREADS)
chunk_solve_kernel(ChunkArgs a) {
  constexpr int DS = DP + 4, CT = DP / 16, WAVES = SOLVE_THREADS / 64;
  extern __shared__ __align__(16) float lds[];
  float* sU = lds;                   // [64][DS] unit keys, then P_(t-1) u
  float* sK = sU + CH * DS;          // keys, then P_end / P_s k
  float* sW = sK + CH * DS;          // a * u, then P_end / P_s w
  float* sR = sW + CH * DS;          // r, then P_t r
  float* sG = sR + CH * DS;          // decays, their products from the start of a token's 16 on; then [64][MS] B
  float* M = sG + CH * MS;           // [64][MS] the inner activations; then A
  float* X = M + CH * MS;            // [64][MS] (I + A)^-1
  float* Qw = X + CH * MS;
  float* Qk = Qw + CH * MS;
  float* sT = Qk;                    // first [64][DS] products from a token's next to the end of its 16
  float* so = Qk + CH * MS;          // [4][DP] products of a 16's decays, then P_end
  CHUNK_OF_ROW;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = a.d, nH = a.H * d;
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  // ---- a wave eight tokens, lane a channel
  {
    const int i = lane < d ? lane : d - 1, c = h * d + i;
    const float rb = a.removal_bias[c];
    float k[8], r[8], al[8], in[8], kk[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int tt = 8 * wave + q;
      const float* src = a.sums + (size_t)(t0 + (tt < nt ? tt : nt - 1)) * a.ld;
      k[q] = src[a.k_col + c];
      r[q] = src[a.r_col + c];
      al[q] = src[a.a_col + c];
      in[q] = src[a.w_col + (lane < a.rank ? lane : a.rank - 1)];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) kk[q] = lane < d ? k[q] * k[q] : 0.f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int q = 0; q < 8; ++q) kk[q] += __shfl_xor(kk[q], o, 64);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int tt = 8 * wave + q;
      const bool ok = lane < d && tt < nt;
      const float u = k[q] / sqrtf(kk[q] + 1e-6f);
      if (lane < DP) {
        sU[tt * DS + lane] = ok ? u : 0.f;
        sK[tt * DS + lane] = ok ? k[q] : 0.f;
        sR[tt * DS + lane] = ok ? r[q] : 0.f;
        sW[tt * DS + lane] = ok ? mie_sigmoid(al[q] + rb) * u : 0.f;
      }
      M[tt * MS + lane] = lane < a.rank && tt < nt ? tanhf(in[q]) : 0.f;
    }
  }
  lds_barrier();
  // ---- decays: (inner activations) (matrix of the head's channels)^T
  for (int tile = wave; tile < 4 * CT; tile += WAVES) {
    const int x = tile & 3, c = (tile >> 2) * 16 + n;
    const int cc = h * d + (c < d ? c : d - 1);
    const float* __restrict__ wd = a.w_decay + (size_t)cc * a.rank + 4 * g;
    f32x4 zs[4] = {none, none, none, none};
    for (int kb = 0; kb < a.rank; kb += 16) {
      const f32x4 w = *reinterpret_cast<const f32x4*>(wd + kb);
      const f32x4 in = *reinterpret_cast<const f32x4*>(M + (16 * x + n) * MS + kb + 4 * g);
#pragma unroll
      for (int j = 0; j < 4; ++j) zs[j] = mfma4(in[j], w[j], zs[j]);
    }
    const f32x4 z = meet(zs);
    const float b = a.decay_bias[cc];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * x + 4 * g + e;
      sG[t * DS + c] = t < nt && c < d ? expf(-a.decay_scale * mie_sigmoid(z[e] + b)) : 1.f;
    }
  }
  lds_barrier();
  // ---- products over the tokens of a 16 (over all 64 they could reach zero)
  if (tid < 4 * DP) {
    const int i = tid % DP, part = tid / DP;
    float run = 1.f, decay[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) decay[t] = sG[(16 * part + t) * DS + i];
#pragma unroll
    for (int t = 15; t >= 0; --t) {
      sT[(16 * part + t) * DS + i] = run;
      run *= decay[t];
    }
    run = 1.f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      run *= decay[t];
      sG[(16 * part + t) * DS + i] = run;
    }
    so[part * DP + i] = run;
  }
  lds_barrier();
  // ---- A, B, Qw, Qk: the ten 16 x 16 blocks on and below the diagonal over the waves, results kept until all have read
  f32x4 accA[2], accB[2], accW[2], accK[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    accA[q] = accB[q] = accW[q] = accK[q] = none;
    const int blk = wave + WAVES * q;
    if (blk >= 10) break;
    const int x = blk < 4 ? 3 : blk < 7 ? 2 : blk < 9 ? 1 : 0, y = blk - (blk < 4 ? 0 : blk < 7 ? 4 : blk < 9 ? 7 : 9);
    const int t = 16 * x + n, s = 16 * y + n;
    const float* gb = sG + (t - (n > 0 ? 1 : 0)) * DS;
    f32x4 pA[4] = {none, none, none, none}, pB[4] = {none, none, none, none}, pW[4] = {none, none, none, none}, pK[4] = {none, none, none, none};
    const f32x4 ones = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int i = 4 * g; i < DP; i += 16) {
      f32x4 gp = *reinterpret_cast<const f32x4*>(gb + i);
      if (n == 0) gp = ones;                                        // before the 16's first token: nothing
      const f32x4 gt = *reinterpret_cast<const f32x4*>(sG + t * DS + i);
      f32x4 es;                                                     // from s's next token to the end of its 16 and on to t's
      if (x == y) {
        const f32x4 gs = *reinterpret_cast<const f32x4*>(sG + s * DS + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) es[e] = reciprocal(gs[e]);
      } else {
        es = *reinterpret_cast<const f32x4*>(sT + s * DS + i);
        for (int z = y + 1; z < x; ++z) es *= *reinterpret_cast<const f32x4*>(so + z * DP + i);
      }
      const f32x4 u = *reinterpret_cast<const f32x4*>(sU + t * DS + i), r = *reinterpret_cast<const f32x4*>(sR + t * DS + i);
      const f32x4 w = *reinterpret_cast<const f32x4*>(sW + s * DS + i), k = *reinterpret_cast<const f32x4*>(sK + s * DS + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lu = u[e] * gp[e], lr = r[e] * gt[e], rw = w[e] * es[e], rk = k[e] * es[e];
        pA[e] = mfma4(lu, rw, pA[e]);
        pB[e] = mfma4(lu, rk, pB[e]);
        pW[e] = mfma4(lr, rw, pW[e]);
        pK[e] = mfma4(lr, rk, pK[e]);
      }
    }
    accA[q] = meet(pA);
    accB[q] = meet(pB);
    accW[q] = meet(pW);
    accK[q] = meet(pK);
  }
  lds_barrier();
  // ---- the vectors times their decays, in place, P_end beside them
  for (int e = tid; e < CH * DP; e += SOLVE_THREADS) {
    const int t = e / DP, i = e % DP, x = t >> 4;
    const float G = sG[t * DS + i], Gb = t & 15 ? sG[(t - 1) * DS + i] : 1.f;
    float before = 1.f, to_end = sT[t * DS + i];
    for (int z = 0; z < x; ++z) before *= so[z * DP + i];
    for (int z = x + 1; z < 4; ++z) to_end *= so[z * DP + i];
    sU[t * DS + i] *= before * Gb;
    sR[t * DS + i] *= before * G;
    sK[t * DS + i] *= to_end;
    sW[t * DS + i] *= to_end;
    if (t == CH - 1) so[4 * DP + i] = before * G;
  }
  for (int e = tid; e < CH * MS; e += SOLVE_THREADS) M[e] = X[e] = Qw[e] = 0.f;
  lds_barrier();
  for (int e = tid; e < CH * MS; e += SOLVE_THREADS) sG[e] = Qk[e] = 0.f;
  lds_barrier();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int blk = wave + WAVES * q;
    if (blk >= 10) break;
    const int x = blk < 4 ? 3 : blk < 7 ? 2 : blk < 9 ? 1 : 0, y = blk - (blk < 4 ? 0 : blk < 7 ? 4 : blk < 9 ? 7 : 9);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * x + 4 * g + e, s = 16 * y + n;
      M[t * MS + s] = s < t ? accA[q][e] : 0.f;
      sG[t * MS + s] = s < t ? accB[q][e] : 0.f;
      Qw[t * MS + s] = s <= t ? accW[q][e] : 0.f;
      Qk[t * MS + s] = s <= t ? accK[q][e] : 0.f;
    }
  }
  lds_barrier();
  // ---- the inverse: diagonal blocks by substitution, a lane a column; X_ab = -X_aa sum_c M_ac X_cb below them
  if (wave < 4) {
    const float* __restrict__ m = M + 16 * wave * MS + 16 * wave;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float v = t == n ? 1.f : 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) v = fmaf(-m[t * MS + s], x[s], v);
      x[t] = v;
    }
    if (g == 0) {
#pragma unroll
      for (int t = 0; t < 16; ++t) X[(16 * wave + t) * MS + 16 * wave + n] = x[t];
    }
  }
  lds_barrier();
#pragma unroll 1
  for (int dist = 1; dist < 4; ++dist) {
    if (wave + dist < 4) {
      const int x = wave + dist, y = wave;
      f32x4 ps[4] = {none, none, none, none}, r = none;
      for (int c = y; c < x; ++c) {
        const f32x4 m = *reinterpret_cast<const f32x4*>(M + (16 * x + n) * MS + 16 * c + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j) ps[j] = mfma4(m[j], X[(16 * c + 4 * g + j) * MS + 16 * y + n], ps[j]);
      }
      const f32x4 s = meet(ps);
      // a result's rows 4 g + e are what the next product's operand wants as its rows 4 g + j
      const f32x4 xx = *reinterpret_cast<const f32x4*>(X + (16 * x + n) * MS + 16 * x + 4 * g);
#pragma unroll
      for (int j = 0; j < 4; ++j) r = mfma4(xx[j], s[j], r);
#pragma unroll
      for (int e = 0; e < 4; ++e) X[(16 * x + 4 * g + e) * MS + 16 * y + n] = -r[e];
    }
    lds_barrier();
  }
  // ---- the four matrices, a wave 16 columns: first W, R, P, then U, F, E
  auto lower = [&](const float* L, const f32x4 (&b)[4], f32x4 (&acc)[4], float sign) {      // acc += sign L b, L lower triangular
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      f32x4 p[4] = {none, none, none, none};
#pragma unroll
      for (int y = 0; y <= x; ++y) {
        const f32x4 m = *reinterpret_cast<const f32x4*>(L + (16 * x + n) * MS + 16 * y + 4 * g) * sign;
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = mfma4(m[j], b[y][j], p[j]);
      }
      acc[x] += meet(p);
    }
  };
  auto turned = [&](const float* T, const f32x4 (&b)[4], f32x4 (&acc)[CT], float sign) {    // acc += sign T^T b, T [64][DS]
#pragma unroll
    for (int x = 0; x < CT; ++x) {
      f32x4 p[4] = {none, none, none, none};
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = mfma4(sign * T[(16 * y + 4 * g + j) * DS + 16 * x + n], b[y][j], p[j]);
      acc[x] += meet(p);                 // (on top of the other sum, a chain would round at its size)
    }
  };
  for (int ct = wave; ct < 2 * CT; ct += WAVES) {
    const bool of_v = ct >= CT;
    const int c = (of_v ? ct - CT : ct) * 16 + n;
    f32x4 b[4], w[4], o[4], st[CT];
#pragma unroll
    for (int x = 0; x < 4; ++x) w[x] = o[x] = none;
#pragma unroll
    for (int x = 0; x < CT; ++x) st[x] = none;
    if (of_v) {
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int s = 16 * y + 4 * g + j;
          b[y][j] = s < nt && c < d ? a.sums[(size_t)(t0 + s) * a.ld + a.v_col + h * d + c] : 0.f;
        }
      lower(Qk, b, o, 1.f);
      turned(sK, b, st, 1.f);
      lower(sG, b, w, 1.f);              // B v
#pragma unroll
      for (int y = 0; y < 4; ++y) { b[y] = w[y]; w[y] = none; }
    } else {
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          b[y][j] = sU[(16 * y + 4 * g + j) * DS + c];
          o[y][j] = sR[(16 * y + 4 * g + j) * DS + c];
        }
    }
    lower(X, b, w, 1.f);                 // W or U
    lower(Qw, w, o, -1.f);
    turned(sW, w, st, -1.f);
    float* __restrict__ to = (of_v ? a.F : a.R) + unit * CH * DP + c;
    float* __restrict__ se = (of_v ? a.E : a.P) + unit * DP * DP + c;
    const float diagonal = of_v ? 0.f : so[4 * DP + c];                  // P_end
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) to[(size_t)(16 * x + 4 * g + e) * DP] = o[x][e];
#pragma unroll
    for (int x = 0; x < CT; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) se[(size_t)(16 * x + 4 * g + e) * DP] = st[x][e] + (16 * x + 4 * g + e == c ? diagonal : 0.f);
  }
}

// (2) grid (H, rows, DP / 16): a wave 16 rows of the state's 16 columns; every chunk's S_0 out, S = P S + E
template <int DP>
__global__ void __launch_bounds__(DP * 4)
chunk_fold_kernel(ChunkArgs a) {
  constexpr int CS = 20, KB = DP / 16;
  __shared__ __align__(16) float sS[2][DP * CS];
  const int h = blockIdx.x, rr = blockIdx.y, row = a.first_row + rr, col = blockIdx.z * 16 + (threadIdx.x & 15);
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int d = a.d, tokens = a.row_start[row + 1] - a.row_start[row], chunks = (tokens + CH - 1) / CH;
  if (chunks <= 0) return;
  const int place = rr ? chunk_places(a.row_start[row] - a.row_start[a.first_row], rr) : 0;
  float* __restrict__ st = a.state + ((size_t)a.slots[row] * a.H + h) * d * d;
  f32x4 S;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 16 * wave + 4 * g + e;
    S[e] = r < d && col < d ? st[(size_t)r * d + col] : 0.f;
  }
  struct Ahead { f32x4 p[KB], e; };      // what a chunk needs, asked for two chunks ahead
  auto fetch = [&](Ahead& A, int c) {
    const size_t unit = (size_t)(place + (c < chunks ? c : chunks - 1)) * a.H + h;
    const float* __restrict__ P = a.P + unit * DP * DP + (size_t)(16 * wave + n) * DP + 4 * g;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) A.p[kb] = *reinterpret_cast<const f32x4*>(P + 16 * kb);
    const float* __restrict__ E = a.E + unit * DP * DP + (size_t)(16 * wave + 4 * g) * DP + col;
#pragma unroll
    for (int e = 0; e < 4; ++e) A.e[e] = E[(size_t)e * DP];
  };
  auto step = [&](Ahead& A, int c) {
    float* __restrict__ s = sS[c & 1];
    float* __restrict__ S0 = a.S0 + ((size_t)(place + c) * a.H + h) * DP * DP + (size_t)(16 * wave + 4 * g) * DP + col;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[(16 * wave + 4 * g + e) * CS + n] = S[e];
      S0[(size_t)e * DP] = S[e];
    }
    lds_barrier();                       // (two buffers: the one written next was read before this barrier)
    const f32x4 none = {0.f, 0.f, 0.f, 0.f};
    f32x4 acc[4] = {none, none, none, none};
    float right[KB][4];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) right[kb][j] = s[(16 * kb + 4 * g + j) * CS + n];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = mfma4(A.p[kb][j], right[kb][j], acc[j]);
    S = A.e + meet(acc);
    fetch(A, c + 2);
  };
  Ahead even, odd;
  fetch(even, 0);
  fetch(odd, 1);
  for (int c = 0; c < chunks; c += 2) {
    step(even, c);
    if (c + 1 < chunks) step(odd, c + 1);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 16 * wave + 4 * g + e;
    if (r < d && col < d) st[(size_t)r * d + col] = S[e];
  }
}

// A chunk's tokens one by one from S_0 (in the LDS, a stride of SS a row; used up), one wave, lane a channel and a column; vec: 5 DP.
template <int DP, typename TO>
__device__ __forceinline__ void chunk_one_by_one(const ChunkArgs& a, float* S, float* vec, int h, int t0, int nt) {
  constexpr int SS = DP + 4;
  const int lane = threadIdx.x & 63, d = a.d;
  const bool live = lane < d;
  const int c = h * d + (live ? lane : 0);
  const float* __restrict__ wd = a.w_decay + (size_t)c * a.rank;
#pragma unroll 1
  for (int tt = 0; tt < nt; ++tt) {
    const size_t t = t0 + tt;
    const float* __restrict__ src = a.sums + t * a.ld;
    const float k = live ? src[a.k_col + c] : 0.f, inner = lane < a.rank ? tanhf(src[a.w_col + lane]) : 0.f;
    const float u = k / sqrtf(wave_sum(k * k) + 1e-6f);
    float z = a.decay_bias[c];
#pragma unroll 1
    for (int j = 0; j < a.rank; ++j) z = fmaf(wd[j], __shfl(inner, j, 64), z);
    if (live) {
      vec[lane] = expf(-a.decay_scale * mie_sigmoid(z));
      vec[DP + lane] = mie_sigmoid(src[a.a_col + c] + a.removal_bias[c]) * u;
      vec[2 * DP + lane] = u;
      vec[3 * DP + lane] = k;
      vec[4 * DP + lane] = src[a.r_col + c];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // (one wave: what it wrote is there)
    float o = 0.f;
    if (live) {
      const float v = src[a.v_col + c];
      float seen = 0.f;
#pragma unroll 1
      for (int i = 0; i < d; ++i) seen = fmaf(vec[2 * DP + i], S[i * SS + lane], seen);
#pragma unroll 1
      for (int i = 0; i < d; ++i) {
        const float x = fmaf(vec[3 * DP + i], v, fmaf(-vec[DP + i], seen, vec[i] * S[i * SS + lane]));
        S[i * SS + lane] = x;
        o = fmaf(x, vec[4 * DP + i], o);
      }
    }
    const float rstd = 1.0f / sqrtf(wave_sum(o * o) / (float)d + a.eps);
    if (live) ((TO*)a.out)[t * a.H * d + c] = from_float<TO>(o * rstd * a.norm_weight[c] * mie_sigmoid(src[a.g_col + c]));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// (3) a wave 16 tokens of a head: o = R S_0 + F, S_0 through the LDS; then the norm, the weight and the gate.  A product takes
// 0 times what a later token of its 16 holds, and where that is not a number or infinite, 0 times it is not 0: a chunk with such a
// result takes its tokens one by one, each from the state before it (the state behind such a token is no number either way).
template <int DP, typename TO>
__global__ void __launch_bounds__(256)
chunk_outputs_kernel(ChunkArgs a) {
  constexpr int CT = DP / 16, SS = DP + 4;
  __shared__ __align__(16) float sS[DP * SS];
  __shared__ float sVec[5 * DP];
  __shared__ int sOdd;
  CHUNK_OF_ROW;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = a.d;
  if (tid == 0) sOdd = 0;
  const float* __restrict__ S0 = a.S0 + unit * DP * DP;
  const float* __restrict__ R = a.R + unit * CH * DP + (size_t)(16 * wave + n) * DP + 4 * g;
  const float* __restrict__ F = a.F + unit * CH * DP + (size_t)(16 * wave + 4 * g) * DP + n;
  f32x4 r[CT], o[CT];
#pragma unroll
  for (int kb = 0; kb < CT; ++kb) r[kb] = *reinterpret_cast<const f32x4*>(R + 16 * kb);
#pragma unroll
  for (int x = 0; x < CT; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[x][e] = F[(size_t)e * DP + 16 * x];
  for (int e = tid; e < DP * DP / 4; e += 256) {
    const int i = e / (DP / 4), c = e % (DP / 4);
    *reinterpret_cast<f32x4*>(sS + i * SS + 4 * c) = *reinterpret_cast<const f32x4*>(S0 + 4 * e);
  }
  __syncthreads();
#pragma unroll
  for (int x = 0; x < CT; ++x) {
    const f32x4 none = {0.f, 0.f, 0.f, 0.f};
    f32x4 p[4] = {none, none, none, none};
#pragma unroll
    for (int kb = 0; kb < CT; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) p[j] = mfma4(r[kb][j], sS[(16 * kb + 4 * g + j) * SS + 16 * x + n], p[j]);
    o[x] += meet(p);
  }
  bool odd = false;
#pragma unroll
  for (int x = 0; x < CT; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e) odd |= !(fabsf(o[x][e]) < INFINITY);     // (tokens and channels that are not there are zeros)
  if (odd) sOdd = 1;
  __syncthreads();
  if (sOdd) {                            // the same for the whole workgroup
    if (wave == 0) chunk_one_by_one<DP, TO>(a, sS, sVec, h, t0, nt);
    return;
  }
  float ss[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    ss[e] = 0.f;
#pragma unroll
    for (int x = 0; x < CT; ++x) ss[e] = fmaf(o[x][e], o[x][e], ss[e]);
  }
#pragma unroll
  for (int q = 8; q > 0; q >>= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) ss[e] += __shfl_xor(ss[e], q, 64);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int tt = 16 * wave + 4 * g + e;
    if (tt >= nt) continue;
    const float rstd = 1.0f / sqrtf(ss[e] / (float)d + a.eps);
    const size_t t = t0 + tt;
#pragma unroll
    for (int x = 0; x < CT; ++x) {
      const int c = 16 * x + n;
      if (c < d)
        ((TO*)a.out)[t * a.H * d + h * d + c] =
            from_float<TO>(o[x][e] * rstd * a.norm_weight[h * d + c] * mie_sigmoid(a.sums[t * a.ld + a.g_col + h * d + c]));
    }
  }
}

MIE_EXPORT const char* delta_rule_last_error() { return g_mie_error; }

template <int DP>
static int chunks_launch(const ChunkArgs& a, int rows, int out_dtype, hipStream_t s) {
  const size_t lds = ((size_t)4 * CH * (DP + 4) + (size_t)5 * CH * MS + 5 * DP) * sizeof(float);
  if (mie_allow_lds(reinterpret_cast<const void*>(chunk_solve_kernel<DP>), (int)lds, "delta_rule")) return -1;
  const dim3 units(a.H, a.units < 32768 ? a.units : 32768, (a.units + 32767) / 32768);
  hipLaunchKernelGGL(chunk_solve_kernel<DP>, units, dim3(SOLVE_THREADS), lds, s, a);
  MIE_CHECK_LAUNCH("delta_rule (chunks: solve)");
  hipLaunchKernelGGL(chunk_fold_kernel<DP>, dim3(a.H, rows, DP / 16), dim3(DP * 4), 0, s, a);
  MIE_CHECK_LAUNCH("delta_rule (chunks: fold)");
  if (out_dtype == MIE_F32) hipLaunchKernelGGL((chunk_outputs_kernel<DP, float>), units, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((chunk_outputs_kernel<DP, bf16>), units, dim3(256), 0, s, a);
  MIE_CHECK_LAUNCH("delta_rule (chunks: outputs)");
  return 0;
}

// Whether mie_delta_rule_chunks takes heads of d, an inner size and a decay's scale.
MIE_EXPORT int mie_delta_rule_chunks_take(int d, int rank, float decay_scale) {
  return d >= 1 && d <= 64 && rank >= 16 && rank <= 64 && rank % 16 == 0 && decay_scale >= 0.f && decay_scale <= DELTA_SCALE_MAX;
}
// places of the chunks of `rows` rows of together `tokens` tokens, and floats of scratch a (place, head) takes
MIE_EXPORT int mie_delta_rule_places(int tokens, int rows) { return chunk_places(tokens, rows); }
MIE_EXPORT int mie_delta_rule_unit_floats(int d) { const int DP = d <= 32 ? 32 : 64; return 2 * CH * DP + 3 * DP * DP; }

// Rows [first_row, first_row + rows), of together `tokens` tokens, in chunks of 64 tokens; scratch: mie_delta_rule_places(tokens, rows)
// * H * mie_delta_rule_unit_floats(d) floats.
MIE_EXPORT int mie_delta_rule_chunks(const float* sums, long ld, int r_col, int k_col, int v_col, int g_col, int a_col, int w_col,
                                     const float* w_decay, int rank, const float* decay_bias, float decay_scale,
                                     const float* removal_bias, const float* norm_weight, float eps, float* state,
                                     const int* row_start, const int* slots, void* out, int out_dtype, int first_row, int rows,
                                     int H, int d, int tokens, float* scratch, hipStream_t s) {
  if (rows <= 0 || tokens <= 0) return 0;
  if (H <= 0 || first_row < 0 || !mie_delta_rule_chunks_take(d, rank, decay_scale))
    MIE_FAIL("delta_rule: chunks of %d heads of %d, inner size %d, decays' scale %g", H, d, rank, (double)decay_scale);
  if (rows > 65535 || H > 65535) MIE_FAIL("delta_rule: %d rows, %d heads are beyond the grid", rows, H);
  if (out_dtype != MIE_F32 && out_dtype != MIE_BF16) MIE_FAIL("delta_rule: out dtype code %d", out_dtype);
  if (!scratch || (((uintptr_t)scratch | (uintptr_t)w_decay) & 15)) MIE_FAIL("delta_rule: scratch and the decay's matrix must be 16-byte aligned");
  const int DP = d <= 32 ? 32 : 64;
  const int places = chunk_places(tokens, rows);
  const size_t units = (size_t)places * H;
  ChunkArgs a{sums, ld, r_col, k_col, v_col, g_col, a_col, w_col, w_decay, rank, decay_bias, decay_scale, removal_bias, norm_weight,
              eps, state, row_start, slots, out, nullptr, nullptr, nullptr, nullptr, nullptr, H, d, first_row, rows, places};
  float* at = scratch;
  auto take = [&](size_t per) { float* q = at; at += units * per; return q; };
  a.P = take((size_t)DP * DP);
  a.E = take((size_t)DP * DP);
  a.S0 = take((size_t)DP * DP);
  a.R = take((size_t)CH * DP);
  a.F = take((size_t)CH * DP);
  return DP == 32 ? chunks_launch<32>(a, rows, out_dtype, s) : chunks_launch<64>(a, rows, out_dtype, s);
}

// prep: scratch of tokens * 3 * H * d floats.  chunk_tokens 0: rows run whole.  Else rows run in chunks of that many
// tokens, at most max_chunks a row, with scratch summaries [rows * max_chunks * H * 2 * d * d] and starts
// [rows * max_chunks * H * d * d] floats.
MIE_EXPORT int mie_delta_rule(const float* sums, long ld, int r_col, int k_col, int v_col, int g_col, int a_col, int w_col,
                              const float* w_decay, int rank, const float* decay_bias, float decay_scale,
                              const float* removal_bias, const float* norm_weight, float eps, float* state,
                              const int* row_start, const int* slots, float* prep, void* out, int out_dtype, int tokens,
                              int rows, int H, int d, int chunk_tokens, int max_chunks, float* summaries, float* starts,
                              hipStream_t s) {
  if (tokens <= 0 || rows <= 0) return 0;
  if (H <= 0 || d <= 0 || d > 256 || rank <= 0) MIE_FAIL("delta_rule: %d heads of %d, inner size %d (heads up to 256)", H, d, rank);
  if (H > 65535) MIE_FAIL("delta_rule: %d heads is beyond the grid", H);
  if (chunk_tokens > 0 && d > 128) MIE_FAIL("delta_rule: heads of %d run whole, not in chunks (up to 128)", d);
  if (chunk_tokens < 0 || (chunk_tokens > 0 && (max_chunks < 1 || !summaries || !starts)))
    MIE_FAIL("delta_rule: chunks of %d tokens, %d a row, need their scratch", chunk_tokens, max_chunks);
  const int heads_here = 255 / d + 2;           // heads a workgroup's 256 channels can touch
  // few tokens: a workgroup a token; many: up to PT_MAX tokens a workgroup, the matrix read once for them
  const int pt = tokens <= 64 ? 1 : tokens < 64 * PT_MAX ? (tokens + 63) / 64 : PT_MAX;
  const int rmax = rank <= 16 ? 16 : rank <= 64 ? 64 : 0;
  const size_t lds = ((size_t)pt * (rmax ? rmax : (rank + 3) & ~3) + (size_t)pt * heads_here) * sizeof(float);
  if (lds > 60 * 1024) MIE_FAIL("delta_rule: an inner size of %d does not fit the LDS", rank);
  if ((H * d + 255) / 256 > 65535) MIE_FAIL("delta_rule: %d channels is beyond the grid", H * d);
#define DP_LAUNCH(RMAX_)                                                                                                     \
  hipLaunchKernelGGL(delta_prepare_kernel<RMAX_>, dim3((tokens + pt - 1) / pt, (H * d + 255) / 256), dim3(256), lds, s, sums, ld, \
                     k_col, a_col, w_col, w_decay, rank, decay_bias, decay_scale, removal_bias, prep, tokens, H, d, heads_here, pt)
  if (rmax == 16) DP_LAUNCH(16);
  else if (rmax == 64) DP_LAUNCH(64);
  else DP_LAUNCH(0);
#undef DP_LAUNCH
  MIE_CHECK_LAUNCH("delta_rule (prepare)");
  ScanArgs a{sums, ld, r_col, k_col, v_col, g_col, prep, norm_weight, eps, state, row_start, slots, out, summaries, starts,
             H, d, chunk_tokens > 0 ? chunk_tokens : 1 << 30, chunk_tokens > 0 ? max_chunks : 1, SCAN_WHOLE};
#define DR_LAUNCH(DMAX_, TO_, GRID_, SUM_) \
  hipLaunchKernelGGL((delta_scan_kernel<DMAX_, TO_, SUM_>), GRID_, dim3(DMAX_ < 64 ? 64 : DMAX_), 0, s, a)
#define DR_SIZES(TO_, GRID_, SUM_)                      \
  if (d <= 16) DR_LAUNCH(16, TO_, GRID_, SUM_);         \
  else if (d <= 32) DR_LAUNCH(32, TO_, GRID_, SUM_);    \
  else if (d <= 64) DR_LAUNCH(64, TO_, GRID_, SUM_);    \
  else if (d <= 128) DR_LAUNCH(128, TO_, GRID_, SUM_);  \
  else DR_LAUNCH(256, TO_, GRID_, SUM_)
#define DR_DTYPES(GRID_, SUM_)                                   \
  if (out_dtype == MIE_F32) { DR_SIZES(float, GRID_, SUM_); }    \
  else if (out_dtype == MIE_BF16) { DR_SIZES(bf16, GRID_, SUM_); } \
  else MIE_FAIL("delta_rule: out dtype code %d", out_dtype)
  if (chunk_tokens == 0) {
    DR_DTYPES(dim3(rows, H), false);
    MIE_CHECK_LAUNCH("delta_rule (scan)");
    return 0;
  }
  if ((long)rows * max_chunks > 2147483647L) MIE_FAIL("delta_rule: %d rows of %d chunks is beyond the grid", rows, max_chunks);
  a.mode = SCAN_SUMMARY;
  DR_SIZES(float, dim3(rows * max_chunks, H), true);              // writes no outputs: one instantiation serves both dtypes
  MIE_CHECK_LAUNCH("delta_rule (chunk summaries)");
  const size_t fold_lds = ((size_t)d * 16 + (size_t)d * (d + 1)) * sizeof(float);
  if (fold_lds > 64 * 1024) {
    static bool allowed = false;
    if (!allowed) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(delta_fold_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)fold_lds);
      if (e != hipSuccess) MIE_FAIL("delta_rule: %zu bytes of LDS refused: %s", fold_lds, hipGetErrorString(e));
      allowed = true;
    }
  }
  hipLaunchKernelGGL(delta_fold_kernel, dim3(rows, H, (d + 15) / 16), dim3(256), fold_lds, s, summaries,
                     starts, state, row_start, slots, H, d, chunk_tokens, max_chunks);
  MIE_CHECK_LAUNCH("delta_rule (fold)");
  a.mode = SCAN_FROM_START;
  DR_DTYPES(dim3(rows * max_chunks, H), false);
  MIE_CHECK_LAUNCH("delta_rule (chunks)");
  return 0;
#undef DR_DTYPES
#undef DR_SIZES
#undef DR_LAUNCH
}
