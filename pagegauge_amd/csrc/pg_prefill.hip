// Prompt (prefill) kernels for gfx950: causal attention over a whole prompt and
// the element-wise work between a decoder layer's GEMMs.
//
//   * causal_attention_kernel: [T, Hq, 128] x [T, Hkv, 128] FP16, GQA group
//     4, float32 online softmax (the prompt attention of
//     scripts/benchmark_page_gauge_transformer.py's TransformerDecoder);
//   * rms_norm_kernel: MistralRMSNorm of every row, with the residual add
//     in front of it;
//   * rope_rows_kernel: RoPE of the query and key rows of a fused QKV
//     projection into dense [T, H, 128] tensors;
//   * swiglu_kernel: silu(gate) * up of a fused gate/up projection.
//
// The element-wise kernels round exactly where the torch operators they
// stand for round (each FP16 operation to FP16, float32 statistics), and move
// 16 bytes per lane and access: they are bound by HBM.  At 16384 tokens of a
// 4096 / 14336 wide layer a norm with its add takes 73 us, RoPE 53 us (6.4
// TB/s) and SwiGLU 236 us (6.0 TB/s); as torch operators they took 1.7 ms
// more per layer (two-layer prompt 18.3 against 14.9 ms).
#include "pg_common.h"

namespace pg {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

#define PG_LDS __attribute__((address_space(3)))
#define PG_GLOBAL __attribute__((address_space(1)))

constexpr int kTileKeys = 64;
constexpr int kTileBytes = kTileKeys * kHeadDim * 2;     // 16 KiB
constexpr float kRescaleLimit = 8.0f;                    // log2
constexpr float kNegInf = -__builtin_huge_valf();
// The running maximum before the first finite score.  Finite, so that a tile
// of -inf scores adds probabilities of 0 and not exp2(-inf + inf).
constexpr float kLowest = -__FLT_MAX__;

struct AttentionArgs {
  const uint16_t* query;
  const uint16_t* key;
  const uint16_t* value;
  uint16_t* out;
  int64_t query_stride;
  int64_t key_stride;
  int64_t value_stride;
  int64_t out_stride;
  int tokens;
  int kv_heads;
  int blocks;          // query blocks
  float scale_log2;
};

// One workgroup per (KV head, block of queries): its waves are the 4 query
// heads of the group times blocks of 32 queries, and they share every K and V
// tile of 64 keys through LDS.  A wave keeps its queries as the B operand of
// v_mfma_f32_32x32x16_f16 and computes S^T = K Q^T, so that a lane holds 32
// scores of ONE query: the softmax reduces in registers plus one swap with
// the lane 32 away, the running maximum and the rescale are per-lane scalars,
// and the probabilities are, register for register, the B operand of
// O^T += V^T P^T (V^T through transposing LDS reads, keys permuted alike).
//
// K and V tiles go from memory to LDS directly, double-buffered, one barrier
// per tile; the 16-byte chunks of a row are swizzled by the row (in the
// source address) so that neither the K reads (8 rows per access) nor the
// transposing V reads (4 rows x 32 bytes) meet in a bank.  The scores of tile
// j + 1 are computed beside the softmax of tile j: the two halves of the work
// use the matrix cores and the VALU for about the same time (58 and 54 % of the
// cycles at 16384 tokens), which is what bounds the kernel; the LDS reads (32 KiB
// per wave and tile) take half of either.
//
// The running maximum is raised only when a score exceeds it by more than
// 2^8 (probabilities then reach 256, which FP16 holds at the same relative
// precision): most tiles skip the rescale of the accumulators.  A lane adds its
// probabilities in float32, in two sums: half the chain (16384 tokens 2047 us
// with one, 2044 with two; no difference at 1000 tokens, nor in the error
// against 64 bits at any length).
//
// Blocks are dispatched longest first, and KV heads vary fastest, so that with
// 8 heads each XCD works on one head's keys and values.
//
// Measured, 32 query and 8 KV heads: 16384 tokens 1.99 ms (1105 TFLOP/s of the
// causal half; about 38 ms as matmul, mask, softmax and matmul launches over
// float32 scores in memory), 4096 tokens 139 us (985), 1000 tokens 23 us
// (340, too few workgroups).
template <int kWaves>
__global__ __launch_bounds__(kWave * kWaves, 2) void causal_attention_kernel(AttentionArgs a) {
  constexpr int kQueries = 32 * (kWaves / kGqa);   // query rows per workgroup
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * kTileBytes];   // K0 K1 V0 V1
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave;
  const int kv = blockIdx.x % a.kv_heads;
  const int block = a.blocks - 1 - blockIdx.x / a.kv_heads;
  const int head = kv * kGqa + wave % kGqa;
  const int q0 = block * kQueries + 32 * (wave / kGqa);
  const int half = lane >> 5;
  const int column = lane & 31;
  const int q = q0 + column;
  const int last = a.tokens - 1;
  // key tiles that any row of the workgroup sees
  const int tiles = (min((block + 1) * kQueries, a.tokens) + kTileKeys - 1) / kTileKeys;

  v8h qf[8];
  const uint16_t* qp = a.query + static_cast<int64_t>(min(q, last)) * a.query_stride + head * kHeadDim + 8 * half;
#pragma unroll
  for (int k = 0; k < 8; ++k) qf[k] = *reinterpret_cast<const v8h*>(qp + 16 * k);

  // direct-to-LDS tile loads: one instruction fills 4 rows
  const uint16_t* kg = a.key + kv * kHeadDim;
  const uint16_t* vg = a.value + kv * kHeadDim;
  const int lrow = lane >> 4;
  const int lchunk = lane & 15;
  constexpr int kLoads = 16 / kWaves;      // per wave and tensor
  auto load_k = [&](int tile, int buffer) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int row = 4 * (wave * kLoads + i) + lrow;
      const int key = min(tile * kTileKeys + row, last);
      const uint16_t* src = kg + static_cast<int64_t>(key) * a.key_stride + 8 * (lchunk ^ (row & 15));
      __builtin_amdgcn_global_load_lds(
          (const PG_GLOBAL void*)src,
          (PG_LDS void*)(lds + buffer * kTileBytes + 1024 * (wave * kLoads + i)), 16, 0, 0);
    }
  };
  auto load_v = [&](int tile, int buffer) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int row = 4 * (wave * kLoads + i) + lrow;
      const int key = min(tile * kTileKeys + row, last);
      const uint16_t* src = vg + static_cast<int64_t>(key) * a.value_stride + 8 * (lchunk ^ (4 * (row & 3)));
      __builtin_amdgcn_global_load_lds(
          (const PG_GLOBAL void*)src,
          (PG_LDS void*)(lds + (2 + buffer) * kTileBytes + 1024 * (wave * kLoads + i)), 16, 0, 0);
    }
  };
  // LDS read offsets
  uint32_t k_at[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) k_at[k] = column * 256 + (((2 * k + half) ^ (column & 15)) << 4);
  uint32_t v_at[4];
  {
    const int i = lane & 15, g = lane >> 4;
    const int row = 4 * (g >> 1) + (i >> 2);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int chunk = 4 * d + 2 * (g & 1) + ((i & 3) >> 1);
      v_at[d] = 2 * kTileBytes + row * 256 + ((chunk ^ (4 * (row & 3))) << 4) + 8 * (i & 1);
    }
  }

  v16f o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
  float m = kLowest, l = 0.0f, l1 = 0.0f;

  auto qk = [&](int buffer, v16f (&s)[2]) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[b][r] = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const v8h kf = *reinterpret_cast<const v8h*>(lds + k_at[k] + buffer * kTileBytes + b * 8192);
        s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[k], s[b], 0, 0, 0);
      }
  };
  auto softmax = [&](v16f (&s)[2], v8h (&p)[4]) {
    float mx = s[0][0];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[b][r]);
    mx *= a.scale_log2;
    {
      const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
    }
    if (__builtin_amdgcn_ballot_w64(mx > m + kRescaleLimit)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= alpha;
      l1 *= alpha;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][r], a.scale_log2, -m));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][r + 1], a.scale_log2, -m));
        l += p0;
        l1 += p1;
        p[2 * b + r / 8][r % 8] = static_cast<_Float16>(p0);
        p[2 * b + r / 8][r % 8 + 1] = static_cast<_Float16>(p1);
      }
  };
  auto pv = [&](int buffer, v8h (&p)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint8_t* at = lds + v_at[d] + buffer * kTileBytes + k * 4096;
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PG_LDS v4s*)at);
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PG_LDS v4s*)(at + 2048));
        const v8h vf = __builtin_shufflevector(__builtin_bit_cast(v4h, lo), __builtin_bit_cast(v4h, hi),
                                               0, 1, 2, 3, 4, 5, 6, 7);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, p[k], o[d], 0, 0, 0);
      }
  };
  auto mask = [&](int tile, v16f (&s)[2]) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = tile * kTileKeys + 32 * b + 8 * (r / 4) + 4 * half + r % 4;
        s[b][r] = key > q ? kNegInf : s[b][r];
      }
  };
  auto barrier = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  // iteration j: the scores of tile j are in ``s``; K of tile j + 1 and V of
  // tile j have been requested
  auto body = [&](int j, int parity, v16f (&s)[2], v16f (&next)[2]) {
    barrier();
    if (j + 2 < tiles) load_k(j + 2, parity);
    load_v(j + 1, parity ^ 1);
    v8h p[4];
    qk(parity ^ 1, next);
    softmax(s, p);
    pv(parity, p);
  };
  auto finish = [&](int j, int parity, v16f (&s)[2]) {
    barrier();
    v8h p[4];
    mask(j, s);
    softmax(s, p);
    pv(parity, p);
  };

  v16f s0[2], s1[2];
  load_k(0, 0);
  barrier();
  if (tiles > 1) load_k(1, 1);
  load_v(0, 0);
  qk(0, s0);
  int j = 0;
  for (; j + 2 < tiles; j += 2) {
    body(j, 0, s0, s1);
    body(j + 1, 1, s1, s0);
  }
  if (j + 1 < tiles) {
    body(j, 0, s0, s1);
    finish(j + 1, 1, s1);
  } else {
    finish(j, 0, s0);
  }

  {
    l += l1;
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  if (q >= a.tokens) return;
  const float inv = 1.0f / l;
  uint16_t* out = a.out + static_cast<int64_t>(q) * a.out_stride + head * kHeadDim + 4 * half;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      v4h w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = static_cast<_Float16>(o[d][r + e] * inv);
      *reinterpret_cast<v4h*>(out + 32 * d + 2 * r) = w;
    }
}

// From this many 64-query workgroups on, the 8-wave workgroup, which reads K
// and V half as often; below it the 4-wave one, whose twice as many workgroups
// fill the chip.  8 against 4 waves, 8 KV heads: 1024 tokens (128 workgroups)
// 30.2 against 23.0 us, 2048 54.8 / 49.8, 3072 (384) 90.6 / 91.3, 4096 139 /
// 153, 16384 1990 / 2124.
constexpr int64_t kWideBlocks = 384;

template <int kWaves>
void launch_attention(AttentionArgs a, hipStream_t stream) {
  constexpr int kQueries = 32 * (kWaves / kGqa);
  a.blocks = (a.tokens + kQueries - 1) / kQueries;
  hipLaunchKernelGGL(causal_attention_kernel<kWaves>, dim3(static_cast<unsigned>(a.blocks) * a.kv_heads),
                     dim3(kWave * kWaves), 0, stream, a);
}

__device__ __forceinline__ float to_f(_Float16 h) { return static_cast<float>(h); }
__device__ __forceinline__ _Float16 to_h(float f) { return static_cast<_Float16>(f); }

constexpr int kRowThreads = 256;

struct RmsNormArgs {
  uint16_t* x;             // [rows, width]; with ``delta``, x + delta is written back
  int64_t x_stride;
  const uint16_t* delta;   // [rows, width] or null
  int64_t delta_stride;
  const uint16_t* weight;  // [width]
  uint16_t* out;           // [rows, width]
  int64_t out_stride;
  int width;
  float eps;
};

// One workgroup per row; thread t holds the 8-element vectors t, t + 256, ...
// of its row in registers (kVectors of them), so that a row is read once.
template <int kVectors>
__global__ __launch_bounds__(kRowThreads) void rms_norm_kernel(RmsNormArgs a) {
  __shared__ float sums[kRowThreads / kWave];
  uint16_t* x = a.x + blockIdx.x * a.x_stride;
  const int vectors = a.width / 8;
  v8h v[kVectors];
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kVectors; ++i) {
    const int at = threadIdx.x + i * kRowThreads;
    if (at < vectors) {
      v[i] = *reinterpret_cast<const v8h*>(x + 8 * at);
      if (a.delta != nullptr) {
        const v8h d = *reinterpret_cast<const v8h*>(a.delta + blockIdx.x * a.delta_stride + 8 * at);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = to_h(to_f(v[i][e]) + to_f(d[e]));
        *reinterpret_cast<v8h*>(x + 8 * at) = v[i];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += to_f(v[i][e]) * to_f(v[i][e]);
    }
  }
  ss = wave_sum(ss);
  if (threadIdx.x % kWave == 0) sums[threadIdx.x / kWave] = ss;
  __syncthreads();
  float total = 0.0f;
#pragma unroll
  for (int w = 0; w < kRowThreads / kWave; ++w) total += sums[w];
  const float inv = rsqrtf(total / static_cast<float>(a.width) + a.eps);
  uint16_t* out = a.out + blockIdx.x * a.out_stride;
#pragma unroll
  for (int i = 0; i < kVectors; ++i) {
    const int at = threadIdx.x + i * kRowThreads;
    if (at < vectors) {
      const v8h w = *reinterpret_cast<const v8h*>(a.weight + 8 * at);
      v8h r;
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = to_h(to_f(w[e]) * to_f(to_h(to_f(v[i][e]) * inv)));
      *reinterpret_cast<v8h*>(out + 8 * at) = r;
    }
  }
}

struct RopeRowsArgs {
  const uint16_t* qkv;     // [tokens, >= (query_heads + kv_heads) * 128]
  int64_t qkv_stride;
  const uint16_t* cosine;  // [tokens, 128]
  const uint16_t* sine;
  int64_t rope_stride;
  uint16_t* query;         // [tokens, query_heads, 128]
  uint16_t* key;           // [tokens, kv_heads, 128]
  int query_heads;
  int kv_heads;
  int64_t units;           // tokens * heads * 8
};

// A thread rotates dims 8u..8u+7 and 64+8u..64+8u+7 of one head row.
__global__ __launch_bounds__(kRowThreads) void rope_rows_kernel(RopeRowsArgs a) {
#pragma clang fp contract(off)
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * kRowThreads + threadIdx.x;
  if (unit >= a.units) return;
  const int u = static_cast<int>(unit & 7);
  const int64_t row = unit >> 3;
  const int heads = a.query_heads + a.kv_heads;
  const int64_t token = row / heads;
  const int head = static_cast<int>(row - token * heads);
  const uint16_t* x = a.qkv + token * a.qkv_stride + head * kHeadDim + 8 * u;
  const uint16_t* c = a.cosine + token * a.rope_stride + 8 * u;
  const uint16_t* s = a.sine + token * a.rope_stride + 8 * u;
  const v8h lo = *reinterpret_cast<const v8h*>(x);
  const v8h hi = *reinterpret_cast<const v8h*>(x + 64);
  const v8h c_lo = *reinterpret_cast<const v8h*>(c);
  const v8h c_hi = *reinterpret_cast<const v8h*>(c + 64);
  const v8h s_lo = *reinterpret_cast<const v8h*>(s);
  const v8h s_hi = *reinterpret_cast<const v8h*>(s + 64);
  v8h r_lo, r_hi;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    // x * cos + rotate_half(x) * sin, every operation rounded to FP16
    const _Float16 a0 = lo[e] * c_lo[e];
    const _Float16 a1 = -hi[e] * s_lo[e];
    r_lo[e] = a0 + a1;
    const _Float16 b0 = hi[e] * c_hi[e];
    const _Float16 b1 = lo[e] * s_hi[e];
    r_hi[e] = b0 + b1;
  }
  uint16_t* out = head < a.query_heads
                      ? a.query + (token * a.query_heads + head) * kHeadDim
                      : a.key + (token * a.kv_heads + head - a.query_heads) * kHeadDim;
  *reinterpret_cast<v8h*>(out + 8 * u) = r_lo;
  *reinterpret_cast<v8h*>(out + 64 + 8 * u) = r_hi;
}

struct SwigluArgs {
  const uint16_t* gate_up;  // [rows, 2 * width]: gate, then up
  int64_t stride;
  uint16_t* out;            // [rows, width]
  int64_t out_stride;
  int vectors;              // width / 8
};

// Grid (vectors / 256, rows): a thread takes 8 elements.
__global__ __launch_bounds__(kRowThreads) void swiglu_kernel(SwigluArgs a) {
  const int at = blockIdx.x * kRowThreads + threadIdx.x;
  if (at >= a.vectors) return;
  const uint16_t* x = a.gate_up + blockIdx.y * a.stride + 8 * at;
  const v8h gate = *reinterpret_cast<const v8h*>(x);
  const v8h up = *reinterpret_cast<const v8h*>(x + 8 * a.vectors);
  v8h r;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float g = to_f(gate[e]);
    const _Float16 act = to_h(g / (1.0f + expf(-g)));
    r[e] = to_h(to_f(act) * to_f(up[e]));
  }
  *reinterpret_cast<v8h*>(a.out + blockIdx.y * a.out_stride + 8 * at) = r;
}

bool aligned(const void* p, uintptr_t to) { return reinterpret_cast<uintptr_t>(p) % to == 0; }

}  // namespace
}  // namespace pg

using namespace pg;

extern "C" int32_t pg_causal_attention(const void* query, int64_t query_stride, const void* key,
                                       int64_t key_stride, const void* value, int64_t value_stride,
                                       void* out, int64_t out_stride, int32_t tokens,
                                       int32_t query_heads, int32_t kv_heads, float sm_scale,
                                       void* stream) {
  clear_error();
  if (!query || !key || !value || !out) return fail(PG_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  if (tokens <= 0) return fail(PG_ERROR_INVALID_ARGUMENT, "the prompt must hold at least one token");
  if (kv_heads <= 0 || query_heads != static_cast<int64_t>(kGqa) * kv_heads)
    return fail(PG_ERROR_UNSUPPORTED, "the attention kernel requires GQA group size 4");
  // key and block numbers are int32, up to a block past the last token
  if (tokens > 0x7fffffff - 64 || (static_cast<int64_t>(tokens) + 31) / 32 * kv_heads > 0x7fffffff)
    return fail(PG_ERROR_INVALID_ARGUMENT, "too many tokens");
  const int64_t q_row = static_cast<int64_t>(query_heads) * kHeadDim;
  const int64_t kv_row = static_cast<int64_t>(kv_heads) * kHeadDim;
  if (query_stride < q_row || out_stride < q_row || key_stride < kv_row || value_stride < kv_row ||
      query_stride % 8 || key_stride % 8 || value_stride % 8 || out_stride % 4)
    return fail(PG_ERROR_INVALID_ARGUMENT, "token strides must cover the rows and keep 16-byte alignment");
  if (!aligned(query, 16) || !aligned(key, 16) || !aligned(value, 16) || !aligned(out, 8))
    return fail(PG_ERROR_INVALID_ARGUMENT, "attention rows must be 16-byte aligned");
  if (!(sm_scale > 0.0f) || !__builtin_isfinite(sm_scale))
    return fail(PG_ERROR_INVALID_ARGUMENT, "sm_scale must be positive and finite");
  AttentionArgs a{};
  a.query = static_cast<const uint16_t*>(query);
  a.key = static_cast<const uint16_t*>(key);
  a.value = static_cast<const uint16_t*>(value);
  a.out = static_cast<uint16_t*>(out);
  a.query_stride = query_stride;
  a.key_stride = key_stride;
  a.value_stride = value_stride;
  a.out_stride = out_stride;
  a.tokens = tokens;
  a.kv_heads = kv_heads;
  a.scale_log2 = sm_scale * 1.4426950408889634f;
  const int64_t wide = (static_cast<int64_t>(tokens) + 63) / 64 * kv_heads;
  if (wide >= kWideBlocks) {
    launch_attention<8>(a, as_stream(stream));
  } else {
    launch_attention<4>(a, as_stream(stream));
  }
  return check_launch("causal_attention");
}

extern "C" int32_t pg_rms_norm(void* x, int64_t x_stride, const void* delta, int64_t delta_stride,
                               const void* weight, float eps, void* out, int64_t out_stride,
                               int64_t rows, int32_t width, void* stream) {
  clear_error();
  if (!x || !weight || !out) return fail(PG_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  if (rows <= 0 || rows > 0x7fffffff || width <= 0)
    return fail(PG_ERROR_INVALID_ARGUMENT, "rows and width must be positive");
  if (width % 8 || width > 8 * 8 * kRowThreads)
    return fail(PG_ERROR_UNSUPPORTED, "the row width must be a multiple of 8, at most 16384");
  if (x_stride < width || out_stride < width || (delta && delta_stride < width) || x_stride % 8 ||
      out_stride % 8 || (delta && delta_stride % 8) || !aligned(x, 16) || !aligned(weight, 16) ||
      !aligned(out, 16) || !aligned(delta, 16))
    return fail(PG_ERROR_INVALID_ARGUMENT, "rows must be 16-byte aligned and their strides cover the width");
  RmsNormArgs a{};
  a.x = static_cast<uint16_t*>(x);
  a.x_stride = x_stride;
  a.delta = static_cast<const uint16_t*>(delta);
  a.delta_stride = delta_stride;
  a.weight = static_cast<const uint16_t*>(weight);
  a.out = static_cast<uint16_t*>(out);
  a.out_stride = out_stride;
  a.width = width;
  a.eps = eps;
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(rows)), dim3(kRowThreads), 0,
                       as_stream(stream), a);
  };
  // vectors per thread: the smallest register block that holds the row
  const int per_thread = (width / 8 + kRowThreads - 1) / kRowThreads;
  if (per_thread <= 2) launch(rms_norm_kernel<2>);
  else if (per_thread <= 4) launch(rms_norm_kernel<4>);
  else launch(rms_norm_kernel<8>);
  return check_launch("rms_norm");
}

extern "C" int32_t pg_rope_rows(const void* qkv, int64_t qkv_stride, const void* cosine,
                                const void* sine, int64_t rope_stride, void* query, void* key,
                                int64_t tokens, int32_t query_heads, int32_t kv_heads,
                                void* stream) {
  clear_error();
  if (!qkv || !cosine || !sine || !query || !key)
    return fail(PG_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  if (tokens <= 0 || query_heads <= 0 || kv_heads <= 0)
    return fail(PG_ERROR_INVALID_ARGUMENT, "tokens and head counts must be positive");
  const int64_t heads = static_cast<int64_t>(query_heads) + kv_heads;
  if (heads > 0x7fffffff / kHeadDim || tokens > 0x7fffffffffff / (heads * 8))
    return fail(PG_ERROR_INVALID_ARGUMENT, "too many tokens");
  if (qkv_stride < heads * kHeadDim || qkv_stride % 8 ||
      rope_stride < kHeadDim || rope_stride % 8 || !aligned(qkv, 16) || !aligned(cosine, 16) ||
      !aligned(sine, 16) || !aligned(query, 16) || !aligned(key, 16))
    return fail(PG_ERROR_INVALID_ARGUMENT, "rows must be 16-byte aligned and their strides cover the heads");
  RopeRowsArgs a{};
  a.qkv = static_cast<const uint16_t*>(qkv);
  a.qkv_stride = qkv_stride;
  a.cosine = static_cast<const uint16_t*>(cosine);
  a.sine = static_cast<const uint16_t*>(sine);
  a.rope_stride = rope_stride;
  a.query = static_cast<uint16_t*>(query);
  a.key = static_cast<uint16_t*>(key);
  a.query_heads = query_heads;
  a.kv_heads = kv_heads;
  a.units = tokens * heads * 8;
  const int64_t blocks = (a.units + kRowThreads - 1) / kRowThreads;
  if (blocks > 0x7fffffff) return fail(PG_ERROR_INVALID_ARGUMENT, "too many tokens");
  hipLaunchKernelGGL(rope_rows_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kRowThreads), 0,
                     as_stream(stream), a);
  return check_launch("rope_rows");
}

extern "C" int32_t pg_swiglu(const void* gate_up, int64_t stride, void* out, int64_t out_stride,
                             int64_t rows, int32_t width, void* stream) {
  clear_error();
  if (!gate_up || !out) return fail(PG_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  if (rows <= 0 || width <= 0)
    return fail(PG_ERROR_INVALID_ARGUMENT, "rows and width must be positive");
  if (width % 8 || stride < 2 * static_cast<int64_t>(width) || stride % 8 || out_stride < width ||
      out_stride % 8 || !aligned(gate_up, 16) || !aligned(out, 16))
    return fail(PG_ERROR_INVALID_ARGUMENT, "rows must be 16-byte aligned vectors of 8 and their strides cover them");
  SwigluArgs a{};
  a.stride = stride;
  a.out_stride = out_stride;
  a.vectors = width / 8;
  const unsigned columns = static_cast<unsigned>((a.vectors + kRowThreads - 1) / kRowThreads);
  // the grid's y extent holds 65535 rows
  for (int64_t row = 0; row < rows; row += 65535) {
    a.gate_up = static_cast<const uint16_t*>(gate_up) + row * stride;
    a.out = static_cast<uint16_t*>(out) + row * out_stride;
    const unsigned count = static_cast<unsigned>(rows - row < 65535 ? rows - row : 65535);
    hipLaunchKernelGGL(swiglu_kernel, dim3(columns, count), dim3(kRowThreads), 0,
                       as_stream(stream), a);
  }
  return check_launch("swiglu");
}
