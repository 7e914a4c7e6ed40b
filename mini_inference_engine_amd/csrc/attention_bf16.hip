// bfloat16 attention of single-token rows: the kernel around decode_attention_bf16.hpp and its entry points, for one head size per build
// (-DHEAD_DIM=N, a multiple of 16 up to 256).
#include "decode_attention_bf16.hpp"

template <int NW, bool FROM_SUMS, bool SIG, bool DB, bool KEEP, bool CHUNK, bool RING>
__global__ void __launch_bounds__(NW * 64)
decode_attention_kernel(const bf16* __restrict__ q, long q_stride, bf16* k_cache, bf16* v_cache,
                        bf16* __restrict__ out, float* __restrict__ o_part,
                        float* __restrict__ lse_part, const int* __restrict__ block_tables, int max_blocks,
                        const int* __restrict__ positions, int Hq, int Hkv, int head_tiles, int page,
                        float scale_log2, int window, int partition, int num_splits, ProjectionSums proj,
                        float sink_log2, int chunk, float softcap, const float* __restrict__ head_bias,
                        const float* __restrict__ dist_bias, int dist_n, int keep, const float* __restrict__ head_sinks) {
  decode_attention_body<NW, FROM_SUMS, SIG, DB, KEEP, CHUNK, RING>(
    blockIdx.x, blockIdx.y, blockIdx.z, q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions, Hq,
    Hkv, head_tiles, page, scale_log2, window, partition, num_splits, proj, sink_log2, chunk, softcap, head_bias, dist_bias, dist_n,
    keep, head_sinks);
}

MIE_EXPORT const char* attention_bf16_last_error() { return g_mie_error; }
MIE_EXPORT int mie_attention_bf16_head_dim() { return D; }
#define DA_KIND(...) __VA_ARGS__
// KIND: FROM_SUMS, SIG, DB, KEEP, CHUNK in brackets; `off16` is the caller's
#define DA_LAUNCH(NW, KIND, STREAM, ...)                                                                                           \
  do {                                                                                                                             \
    auto kernel_ = off16 ? decode_attention_kernel<NW, DA_KIND KIND, false> : decode_attention_kernel<NW, DA_KIND KIND, RINGED>;    \
    const int lds_ = da_lds_bytes(NW, RINGED && !off16);                                                                           \
    if (mie_allow_lds((const void*)kernel_, lds_, "decode_attention")) return -1;                                                   \
    hipLaunchKernelGGL(kernel_, grid, dim3(NW * 64), lds_, STREAM, __VA_ARGS__);                                                   \
  } while (0)
static bool caches_off16(const void* k_cache, const void* v_cache) { return RINGED && (((uintptr_t)k_cache | (uintptr_t)v_cache) & 15); }

MIE_EXPORT int mie_decode_block_keys() { return BLOCK_KEYS * NW_SPLIT; }

// q: token b is row b (single-token rows lead the flattened batch).  partition: keys per split, a
// multiple of mie_decode_block_keys().  o_part [rows, Hq, splits, D] and lse_part [rows, Hq, splits]
// float are needed when num_splits > 1.
static int decode_attention_launch(const void* q, long q_stride, const void* k_cache, const void* v_cache, void* out,
                                   float* o_part, float* lse_part, const int* block_tables, int max_blocks,
                                   const int* positions, int rows, int Hq, int Hkv, int head_dim, int page,
                                   float scale, int window, int partition, int num_splits, float sink_log2,
                                   hipStream_t stream, bool sigmoid = false, int chunk = 0, float softcap = 0.f,
                                   const float* head_bias = nullptr, const float* dist_bias = nullptr, int dist_n = 0,
                                   int keep = 0, const float* head_sinks = nullptr) {
  if (rows <= 0) return 0;
  if (keep < 0 || (keep > 0 && (window <= 0 || sigmoid || dist_bias)))
    MIE_FAIL("decode_attention: %d kept first keys belong beside a window, plain softmax only", keep);
  if (dist_bias && (sigmoid || dist_n < 1)) MIE_FAIL("decode_attention: a distance bias of %d entries a head, softmax only", dist_n);
  if (chunk < 0 || softcap < 0.f) MIE_FAIL("decode_attention: chunk %d, score cap %g", chunk, (double)softcap);
  if (head_dim != D) MIE_FAIL("decode_attention: built for head_dim %d, called with %d", D, head_dim);
  if (Hkv <= 0 || Hq % Hkv) MIE_FAIL("decode_attention: %d query heads on %d kv heads", Hq, Hkv);
  if (page < 16 || page % 16) MIE_FAIL("decode_attention: page size %d (multiples of 16)", page);
  if (partition <= 0 || partition % (BLOCK_KEYS * NW_SPLIT)) MIE_FAIL("decode_attention: partition %d is no multiple of %d", partition, BLOCK_KEYS * NW_SPLIT);
  if (num_splits < 1 || num_splits > 65535) MIE_FAIL("decode_attention: %d splits", num_splits);
  if (num_splits > 1 && (!o_part || !lse_part)) MIE_FAIL("decode_attention: splits need partial buffers");
  if (q_stride < (long)Hq * D || (q_stride % 8) || ((uintptr_t)q % 16)) MIE_FAIL("decode_attention: q stride %ld / alignment", q_stride);
  if (max_blocks <= 0) MIE_FAIL("decode_attention: max_blocks %d", max_blocks);
  const int G = Hq / Hkv, head_tiles = (G + 15) / 16;
  if ((long)Hkv * head_tiles > 65535) MIE_FAIL("decode_attention: too many head tiles for the grid");
  dim3 grid(rows, Hkv * head_tiles, num_splits);
  // (the kernel writes the caches only when it is given the projection's sums)
  bf16* kc = (bf16*)const_cast<void*>(k_cache);
  bf16* vc = (bf16*)const_cast<void*>(v_cache);
  const bool off16 = caches_off16(k_cache, v_cache);
  const bool whole = num_splits == 1 && NW_WHOLE != NW_SPLIT && (long)rows * Hkv * head_tiles <= whole_most();
  if (chunk > 0 && !sigmoid && (keep > 0 || dist_bias)) MIE_FAIL("decode_attention: chunks beside kept keys or a distance bias are not built");
  if (chunk > 0 && !sigmoid && whole)
    DA_LAUNCH(NW_WHOLE, (false, false, false, false, true), stream,
                       (const bf16*)q, q_stride, kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv,
                       head_tiles, page, scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, chunk, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, 0, head_sinks);
  else if (chunk > 0 && !sigmoid)
    DA_LAUNCH(NW_SPLIT, (false, false, false, false, true), stream,
                       (const bf16*)q, q_stride, kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv,
                       head_tiles, page, scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, chunk, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, 0, head_sinks);
  else if (keep > 0 && whole)
    DA_LAUNCH(NW_WHOLE, (false, false, false, true, false), stream, (const bf16*)q,
                       q_stride, kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, 0, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, keep, head_sinks);
  else if (keep > 0)
    DA_LAUNCH(NW_SPLIT, (false, false, false, true, false), stream, (const bf16*)q,
                       q_stride, kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, 0, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, keep, head_sinks);
  else if (dist_bias && whole)
    DA_LAUNCH(NW_WHOLE, (false, false, true, false, false), stream, (const bf16*)q, q_stride,
                       kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, 0, 0.f,
                       (const float*)nullptr, dist_bias, dist_n, 0, head_sinks);
  else if (dist_bias)
    DA_LAUNCH(NW_SPLIT, (false, false, true, false, false), stream, (const bf16*)q, q_stride,
                       kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, 0, 0.f,
                       (const float*)nullptr, dist_bias, dist_n, 0, head_sinks);
  else if (sigmoid && whole)
    DA_LAUNCH(NW_WHOLE, (false, true, false, false, false), stream, (const bf16*)q, q_stride,
                       kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale, window, partition, num_splits, ProjectionSums{}, sink_log2, chunk, softcap, head_bias, (const float*)nullptr, 0, 0,
                       head_sinks);
  else if (sigmoid)
    DA_LAUNCH(NW_SPLIT, (false, true, false, false, false), stream, (const bf16*)q, q_stride,
                       kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale, window, partition, num_splits, ProjectionSums{}, sink_log2, chunk, softcap, head_bias, (const float*)nullptr, 0, 0,
                       head_sinks);
  else if (whole)
    DA_LAUNCH(NW_WHOLE, (false, false, false, false, false), stream, (const bf16*)q, q_stride,
                       kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, 0, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, 0, head_sinks);
  else
    DA_LAUNCH(NW_SPLIT, (false, false, false, false, false), stream, (const bf16*)q, q_stride,
                       kc, vc, (bf16*)out, o_part, lse_part, block_tables, max_blocks, positions, Hq, Hkv, head_tiles, page,
                       scale * 1.4426950408889634f, window, partition, num_splits, ProjectionSums{}, sink_log2, 0, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, 0, head_sinks);
  MIE_CHECK_LAUNCH("decode_attention");
  if (num_splits > 1) {
    hipLaunchKernelGGL(merge_splits_kernel, dim3(rows * Hq), dim3(64), 0, stream, o_part, lse_part, (bf16*)out, num_splits,
                       sink_log2, (int)sigmoid, head_sinks, Hq);
    MIE_CHECK_LAUNCH("merge_splits");
  }
  return 0;
}

MIE_EXPORT int mie_decode_attention(const void* q, long q_stride, const void* k_cache, const void* v_cache, void* out,
                                    float* o_part, float* lse_part, const int* block_tables, int max_blocks,
                                    const int* positions, int rows, int Hq, int Hkv, int head_dim, int page,
                                    float scale, int window, int partition, int num_splits, hipStream_t stream) {
  return decode_attention_launch(q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions,
                                 rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits, -INFINITY, stream);
}

// The same with a sink: one more term exp(sink) in every softmax's denominator that has no value.
MIE_EXPORT int mie_decode_attention_sink(const void* q, long q_stride, const void* k_cache, const void* v_cache, void* out,
                                         float* o_part, float* lse_part, const int* block_tables, int max_blocks,
                                         const int* positions, int rows, int Hq, int Hkv, int head_dim, int page,
                                         float scale, int window, int partition, int num_splits, float sink,
                                         hipStream_t stream) {
  return decode_attention_launch(q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions,
                                 rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits,
                                 sink * 1.4426950408889634f, stream);
}


// Sigmoid weights instead of a softmax: a visible key counts with sigmoid(cap(score) + head_bias[head]) (head_bias
// float32 [Hq] or null), cap(x) = softcap tanh(x / softcap) (0: none); chunk n (0: none) hides the keys before
// floor(position / n) n.  Nothing is normalised.
MIE_EXPORT int mie_decode_attention_sigmoid(const void* q, long q_stride, const void* k_cache, const void* v_cache, void* out,
                                            float* o_part, float* lse_part, const int* block_tables, int max_blocks,
                                            const int* positions, int rows, int Hq, int Hkv, int head_dim, int page,
                                            float scale, int window, int partition, int num_splits, int chunk, float softcap,
                                            const float* head_bias, hipStream_t stream) {
  return decode_attention_launch(q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions,
                                 rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits, -INFINITY, stream, true,
                                 chunk, softcap, head_bias);
}

// The q/k/v projection's end and the attention in one kernel, for steps whose rows and kv heads alone fill
// the GPU (contexts unsplit).  part [splits, rows, ld] float32: the projection's sums (q heads, k heads, v
// heads), to be added up in split order; rotary over the whole head with angles from cos / sin [positions,
// D / 2]; the row's k and v go to cache slot slots[row], which must be the slot of key positions[row] in the
// row's block table.  Groups of up to 16 query heads a kv head.  partition as for mie_decode_attention (at least the
// longest context).
MIE_EXPORT int mie_decode_attention_from_sums(const float* part, int splits, long split_stride, long ld, const float* cos_t,
                                              const float* sin_t, const int* slots, void* k_cache, void* v_cache, void* out,
                                              const int* block_tables, int max_blocks, const int* positions, int rows, int Hq,
                                              int Hkv, int head_dim, int page, float scale, int window, int partition,
                                              hipStream_t stream) {
  if (rows <= 0) return 0;
  if (head_dim != D) MIE_FAIL("decode_attention_from_sums: built for head_dim %d, called with %d", D, head_dim);
  if (Hkv <= 0 || Hq % Hkv) MIE_FAIL("decode_attention_from_sums: %d query heads on %d kv heads", Hq, Hkv);
  if (Hq / Hkv > 16) MIE_FAIL("decode_attention_from_sums: groups of %d query heads (at most 16)", Hq / Hkv);
  if (page < 16 || page % 16) MIE_FAIL("decode_attention_from_sums: page size %d (multiples of 16)", page);
  if (partition <= 0 || partition % (BLOCK_KEYS * NW_SPLIT)) MIE_FAIL("decode_attention_from_sums: partition %d is no multiple of %d", partition, BLOCK_KEYS * NW_SPLIT);
  if (!part || !cos_t || !sin_t || !slots || !k_cache || !v_cache || !out || !positions || !block_tables) MIE_FAIL("decode_attention_from_sums: null operand");
  if (splits < 1 || ld < (long)(Hq + 2 * Hkv) * D || (splits > 1 && split_stride < (long)rows * ld)) MIE_FAIL("decode_attention_from_sums: %d splits, stride %ld, row stride %ld", splits, split_stride, ld);
  if (max_blocks <= 0 || Hkv > 65535) MIE_FAIL("decode_attention_from_sums: max_blocks %d, %d kv heads", max_blocks, Hkv);
  const ProjectionSums proj = {part, splits, (size_t)split_stride, ld, cos_t, sin_t, slots};
  dim3 grid(rows, Hkv, 1);
  const bool off16 = caches_off16(k_cache, v_cache);
  if ((long)rows * Hkv <= whole_most())
    DA_LAUNCH(NW_WHOLE, (true, false, false, false, false), stream, (const bf16*)nullptr, 0L,
                       (bf16*)k_cache, (bf16*)v_cache, (bf16*)out, (float*)nullptr, (float*)nullptr, block_tables, max_blocks,
                       positions, Hq, Hkv, 1, page, scale * 1.4426950408889634f, window, partition, 1, proj, -INFINITY, 0, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, 0, (const float*)nullptr);
  else
    DA_LAUNCH(NW_SPLIT, (true, false, false, false, false), stream, (const bf16*)nullptr, 0L,
                       (bf16*)k_cache, (bf16*)v_cache, (bf16*)out, (float*)nullptr, (float*)nullptr, block_tables, max_blocks,
                       positions, Hq, Hkv, 1, page, scale * 1.4426950408889634f, window, partition, 1, proj, -INFINITY, 0, 0.f,
                       (const float*)nullptr, (const float*)nullptr, 0, 0, (const float*)nullptr);
  MIE_CHECK_LAUNCH("decode_attention_from_sums");
  return 0;
}


// ---- the same for callers that cannot allocate (decode_attention_static.hpp)
#include "decode_attention_static.hpp"
#include <mutex>

// Partial results of a split context: the library's own device memory, one copy on every GPU.
// In host code this name is only a stand-in for the symbol; the device address comes from
// hipGetSymbolAddress, per device, and only that address is ever handed to a kernel.
static __device__ __align__(256) float scratch[MIE_DECODE_STATIC_SCRATCH_BYTES / sizeof(float)];

constexpr int MAX_DEVICES = 64;
static float* g_scratch_of_device[MAX_DEVICES];
static std::mutex g_scratch_lock;

static int scratch_for_current_device(float** ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) MIE_FAIL("decode_attention_static: hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= MAX_DEVICES) MIE_FAIL("decode_attention_static: device %d (at most %d devices)", dev, MAX_DEVICES);
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (!g_scratch_of_device[dev]) {
    float* p = nullptr;
    e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      MIE_FAIL("decode_attention_static: hipGetSymbolAddress on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_of_device[dev] = p;
  }
  *ptr = g_scratch_of_device[dev];
  return 0;
}

MIE_EXPORT int mie_decode_attention_static_setup(void) {
  float* p;
  // (and the LDS beyond the default that the kernels ask for)
#define DA_ALLOW(NW, RING) \
  mie_allow_lds((const void*)decode_attention_kernel<NW, false, false, false, false, false, RING>, da_lds_bytes(NW, RING), "decode_attention_static")
  if (DA_ALLOW(NW_SPLIT, RINGED) || DA_ALLOW(NW_WHOLE, RINGED) || DA_ALLOW(NW_SPLIT, false) || DA_ALLOW(NW_WHOLE, false)) return -1;
#undef DA_ALLOW
  return scratch_for_current_device(&p);
}

MIE_EXPORT long mie_decode_attention_static_capacity(void) { return (long)MIE_DECODE_STATIC_SCRATCH_BYTES; }

MIE_EXPORT int mie_decode_attention_static(const void* q, long q_stride, const void* k_cache, const void* v_cache,
                                           void* out, const int* block_tables, int max_blocks, const int* positions,
                                           int rows, int Hq, int Hkv, int head_dim, int page, float scale, int window,
                                           int partition, int num_splits, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (num_splits <= 1)      // no partial results: the plain entry point allocates nothing either
    return mie_decode_attention(q, q_stride, k_cache, v_cache, out, nullptr, nullptr, block_tables, max_blocks,
                                positions, rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits, stream);
  if (Hq <= 0 || head_dim != D) MIE_FAIL("decode_attention_static: built for head_dim %d, called with %d (%d heads)", D, head_dim, Hq);
  const size_t entries = (size_t)rows * (size_t)Hq * (size_t)num_splits;
  const size_t need = entries * (D + 1) * sizeof(float);
  if (need > MIE_DECODE_STATIC_SCRATCH_BYTES)
    MIE_FAIL("decode_attention_static: %d rows x %d heads x %d splits x head_dim %d need %zu bytes for partial results; "
             "the library holds %u (fewer splits, or the entry point that takes buffers)",
             rows, Hq, num_splits, D, need, (unsigned)MIE_DECODE_STATIC_SCRATCH_BYTES);
  float* base = nullptr;
  if (scratch_for_current_device(&base)) return -1;
  float* o_part = base;                       // [rows, Hq, splits, D]
  float* lse_part = base + entries * D;       // [rows, Hq, splits]
  return mie_decode_attention(q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions,
                              rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits, stream);
}

// The softmax with a bias on the score by the key's distance: dist_bias float32 [Hq, dist_n], its entries already times
// log2 e; a key n positions back of the row's token adds entry min(n, dist_n - 1) of the head's row to score * scale.
MIE_EXPORT int mie_decode_attention_biased(const void* q, long q_stride, const void* k_cache, const void* v_cache, void* out,
                                           float* o_part, float* lse_part, const int* block_tables, int max_blocks,
                                           const int* positions, int rows, int Hq, int Hkv, int head_dim, int page,
                                           float scale, int window, int partition, int num_splits, const float* dist_bias,
                                           int dist_n, hipStream_t stream) {
  if (!dist_bias) MIE_FAIL("decode_attention_biased: no table");
  return decode_attention_launch(q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions,
                                 rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits, -INFINITY, stream, false,
                                 0, 0.f, nullptr, dist_bias, dist_n);
}

// The softmax over a window beside the request's first ``keep`` keys (0: none; window 0: all keys), with a sink per query head:
// head_sinks float32 [Hq] or null, the numbers already times log2 e.  partition counts kept and window keys together: each
// of the two starts on a block of its own.
MIE_EXPORT int mie_decode_attention_kept(const void* q, long q_stride, const void* k_cache, const void* v_cache, void* out,
                                         float* o_part, float* lse_part, const int* block_tables, int max_blocks,
                                         const int* positions, int rows, int Hq, int Hkv, int head_dim, int page,
                                         float scale, int window, int partition, int num_splits, int keep,
                                         const float* head_sinks, hipStream_t stream) {
  return decode_attention_launch(q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions,
                                 rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits, -INFINITY, stream, false,
                                 0, 0.f, nullptr, nullptr, 0, keep, head_sinks);
}

// The softmax over the keys of the row's own chunk of positions, from floor(position / chunk) chunk on (and over the last
// ``window`` of them, if that is not 0).
MIE_EXPORT int mie_decode_attention_chunked(const void* q, long q_stride, const void* k_cache, const void* v_cache, void* out,
                                            float* o_part, float* lse_part, const int* block_tables, int max_blocks,
                                            const int* positions, int rows, int Hq, int Hkv, int head_dim, int page,
                                            float scale, int window, int partition, int num_splits, int chunk,
                                            hipStream_t stream) {
  if (chunk < 1) MIE_FAIL("decode_attention_chunked: chunks of %d positions", chunk);
  return decode_attention_launch(q, q_stride, k_cache, v_cache, out, o_part, lse_part, block_tables, max_blocks, positions,
                                 rows, Hq, Hkv, head_dim, page, scale, window, partition, num_splits, -INFINITY, stream, false,
                                 chunk);
}
