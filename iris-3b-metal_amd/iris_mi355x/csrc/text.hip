// Kernels of the layer-wise text adapter (src/iris3b/nn/embeddings.py:110-141, 209-266) that
// the GEMM, row and flash-attention kernels do not cover: the self-attention of each text
// token across its encoder layers (a sequence of a dozen states per token, so one wave per
// (token, head) with the whole sequence in LDS), and the learned pool over those layers.
#include "iris_common.hpp"

#include <algorithm>

namespace iris {
namespace {

constexpr int kMaxSeq = 16;    // encoder layers per token
constexpr int kMaxHeadDim = 128;
constexpr int kMaxWavesPerBlock = 4;
constexpr int kLdsBudget = 64 * 1024;  // bytes of LDS per workgroup the launch may ask for

// LDS floats of one wave: q, k, v of L tokens of d values, and the L x L probabilities.
__host__ __device__ constexpr int layer_attention_floats(int L, int d) { return 3 * L * d + L * L; }

// One wave per (sequence s, head h): q, k, v rows of the L tokens of sequence s are columns
// h*d, D + h*d, 2D + h*d of qkv rows s*L .. s*L + L - 1 (D = heads * d). out = softmax(q k^T *
// scale) v in FP32 from BF16 inputs, stored BF16 at out rows s*L + i, columns h*d. A block holds
// blockDim.x / 64 waves, each with its own LDS slice.
__global__ __launch_bounds__(64 * kMaxWavesPerBlock) void layer_attention_kernel(const bf16* __restrict__ qkv,
                                                                              bf16* __restrict__ out, long seqs,
                                                                              int L, int heads, int d, float scale) {
  extern __shared__ float smem[];
  const int wv = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const long item = static_cast<long>(blockIdx.x) * (blockDim.x >> 6) + wv;
  const bool active = item < seqs * heads;  // every wave reaches the barriers
  float* sq = smem + wv * layer_attention_floats(L, d);
  float* sk = sq + L * d;
  float* sv = sk + L * d;
  float* sp = sv + L * d;
  const long s = active ? item / heads : 0;
  const int h = active ? static_cast<int>(item % heads) : 0;
  const int D = heads * d;
  if (active) {
    for (int e = lane; e < L * d; e += kWave) {
      const int i = e / d, c = e - i * d;
      const bf16* row = qkv + (s * L + i) * 3L * D + h * d + c;
      sq[e] = to_f32(row[0]);
      sk[e] = to_f32(row[D]);
      sv[e] = to_f32(row[2 * D]);
    }
  }
  __syncthreads();
  if (active) {
    for (int e = lane; e < L * L; e += kWave) {
      const int i = e / L, j = e - i * L;
      float acc = 0.0f;
      for (int c = 0; c < d; ++c) acc += sq[i * d + c] * sk[j * d + c];
      sp[e] = acc * scale;
    }
  }
  __syncthreads();
  if (active && lane < L) {
    float* pr = sp + lane * L;
    float m = -INFINITY;
    for (int j = 0; j < L; ++j) m = fmaxf(m, pr[j]);
    float sum = 0.0f;
    for (int j = 0; j < L; ++j) {
      const float p = expf(pr[j] - m);
      pr[j] = p;
      sum += p;
    }
    const float inv = 1.0f / sum;
    for (int j = 0; j < L; ++j) pr[j] *= inv;
  }
  __syncthreads();
  if (active) {
    for (int e = lane; e < L * d; e += kWave) {
      const int i = e / d, c = e - i * d;
      float acc = 0.0f;
      for (int j = 0; j < L; ++j) acc += sp[i * L + j] * sv[j * d + c];
      out[(s * L + i) * static_cast<long>(D) + h * d + c] = from_f32<bf16>(acc);
    }
  }
}

// The same attention on MFMAs for heads of whole 16-value blocks (d = 16 DT), straight from global
// memory to fragments: no LDS, no barrier, one wave per (sequence, head).
// S^T = K Q^T is 16 x 16 x 32 BF16 (the products of BF16 values are exact, the sums FP32, as before);
// the accumulator leaves lane (g = l / 16, i = l % 16) with the scores of query i against the keys
// 4 g + e, e = 0..3, so the softmax of a query is four registers and two exchanges, and register e is
// the B operand of O^T += V^T P^T on 16 x 16 x 4 FP32 over the keys {4 g + e}: the probabilities stay
// FP32. V enters as pairs (lane: key 4 g + e, dims 32 t + 2 i + {0, 1}), 64 bytes a row per load; the
// two products of a pair block then hold eight consecutive dims of a query, stored as 16 bytes.
// What bounds it: HBM (74 MB at 300 tokens of 12 x 2560). The kernel above adds every product from
// LDS one by one: 116 us at 300 tokens x 12 layers x 32 heads of 80 against 21 us here (3.5 TB/s; 59
// against 11 us at 154 tokens; with V loaded value by value 32 us).
template <int DT>
__global__ __launch_bounds__(256) void layer_attention_mfma_kernel(const bf16* __restrict__ qkv, bf16* __restrict__ out,
                                                                   long items, int L, int heads, float scale) {
  constexpr int KS = (DT + 1) / 2;  // 32-value k-steps of a head
  const int lane = threadIdx.x & 63;
  const long item = static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (item >= items) return;
  const long s = item / heads;
  const int h = static_cast<int>(item - s * heads);
  const int d = 16 * DT;
  const long D = static_cast<long>(heads) * d;
  const int i16 = lane & 15, g = lane >> 4;
  const bf16* base = qkv + s * L * 3 * D + static_cast<long>(h) * d;
  const bool row_ok = i16 < L;
  bf16x8 q[KS], k[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int c = 32 * ks + 8 * g;
    const bool ok = row_ok && (DT % 2 == 0 || ks + 1 < KS || c < d);
    const bf16* row = base + i16 * 3 * D + c;
    q[ks] = ok ? *reinterpret_cast<const bf16x8*>(row) : bf16x8{};
    k[ks] = ok ? *reinterpret_cast<const bf16x8*>(row + D) : bf16x8{};
  }
  // dims 32 t + 2 i + {0, 1} of row j in block t, and with an odd DT dim 32 (DT / 2) + i of a last one
  bf16x2 v2[4][DT / 2 + 1];
  bf16 v1[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int j = 4 * g + e;
    const bf16* row = base + j * 3 * D + 2 * D;
#pragma unroll
    for (int t = 0; t < DT / 2; ++t) v2[e][t] = j < L ? *reinterpret_cast<const bf16x2*>(row + 32 * t + 2 * i16) : bf16x2{};
    v1[e] = DT % 2 && j < L ? row[32 * (DT / 2) + i16] : static_cast<bf16>(0.0f);
  }
  f32x4 p{};
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[ks], q[ks], p, 0, 0, 0);
  float m = -INFINITY;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    p[e] = 4 * g + e < L ? p[e] * scale : -INFINITY;
    m = fmaxf(m, p[e]);
  }
  m = fmaxf(m, __shfl_xor(m, 16));
  m = fmaxf(m, __shfl_xor(m, 32));
  float sum = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    p[e] = 4 * g + e < L ? expf(p[e] - m) : 0.0f;
    sum += p[e];
  }
  sum += __shfl_xor(sum, 16);
  sum += __shfl_xor(sum, 32);
  const float inv = 1.0f / sum;
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] *= inv;
  auto weigh = [&](const float (&v)[4]) {  // O^T of one 16-dim block: the keys {4 g + e}, e in turn
    f32x4 o{};
#pragma unroll
    for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], p[e], o, 0, 0, 0);
    return o;
  };
  bf16* dst = out + (s * L + i16) * D + static_cast<long>(h) * d;
#pragma unroll
  for (int t = 0; t < DT / 2; ++t) {
    f32x4 o[2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
      o[b] = weigh({to_f32(v2[0][t][b]), to_f32(v2[1][t][b]), to_f32(v2[2][t][b]), to_f32(v2[3][t][b])});
    if (row_ok) {
      const float y[8] = {o[0][0], o[1][0], o[0][1], o[1][1], o[0][2], o[1][2], o[0][3], o[1][3]};
      store8(dst + 32 * t + 8 * g, y);
    }
  }
  if constexpr (DT % 2 != 0) {
    const f32x4 o = weigh({to_f32(v1[0]), to_f32(v1[1]), to_f32(v1[2]), to_f32(v1[3])});
    if (row_ok) store4(dst + 32 * (DT / 2) + 4 * g, o);
  }
}

// 0/1 key bytes [batch, n_pad] from a [batch, >= n] mask of 1-, 4- or 8-byte elements (bool /
// uint8, int32, float32, int64: nonzero = keep, as mask.bool()); positions n .. n_pad - 1 are 0.
__global__ __launch_bounds__(256) void key_mask_kernel(const void* __restrict__ mask, int kind, long ld, int batch,
                                                       int n, int n_pad, unsigned char* __restrict__ out) {
  const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<long>(batch) * n_pad) return;
  const long b = i / n_pad;
  const int j = static_cast<int>(i - b * n_pad);
  bool keep = false;
  if (j < n) {
    const long at = b * ld + j;
    switch (kind) {
      case 0:
        keep = static_cast<const unsigned char*>(mask)[at] != 0;
        break;
      case 1:
        keep = static_cast<const int*>(mask)[at] != 0;
        break;
      case 2:
        keep = static_cast<const float*>(mask)[at] != 0.0f;
        break;
      default:
        keep = static_cast<const long long*>(mask)[at] != 0;
        break;
    }
  }
  out[i] = keep ? 1 : 0;
}

// out[r, c] = sum_l weight[l] * (h + branch)[r*L + l, c] + bias, in layer order (nn.Linear(L, 1)
// over the layer axis, after the last block's residual add); four columns per thread.
template <typename TO>
__global__ __launch_bounds__(256) void layer_pool_kernel(const float* __restrict__ h, const bf16* __restrict__ branch,
                                                         const float* __restrict__ weight,
                                                         const float* __restrict__ bias, long rows, int L, int width,
                                                         TO* __restrict__ out) {
  const long i4 = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  const long nv = width >> 2;
  if (i4 >= rows * nv) return;
  const long r = i4 / nv;
  const int c = static_cast<int>(i4 - r * nv) * 4;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int l = 0; l < L; ++l) {
    f32x4 v = load4(h + (r * L + l) * width + c);
    if (branch) {
      const f32x4 bv = load4(branch + (r * L + l) * width + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += bv[e];
    }
    const float wl = weight[l];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += wl * v[e];
  }
  const float b = bias ? bias[0] : 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] += b;
  store4(out + r * width + c, acc);
}

}  // namespace
}  // namespace iris

using namespace iris;

extern "C" int iris_layer_attention(const void* qkv, void* out, long seqs, int seq_len, int heads, int head_dim,
                                    float scale, hipStream_t stream) {
  IRIS_REQUIRE(seqs >= 0 && seq_len > 0 && seq_len <= kMaxSeq && heads > 0 && head_dim > 0 &&
                   head_dim <= kMaxHeadDim,
               "layer_attention: sequences of 1..%d tokens with heads of at most %d (got %d, %d)", kMaxSeq,
               kMaxHeadDim, seq_len, head_dim);
  IRIS_REQUIRE(qkv && out && qkv != out, "layer_attention: bad pointers");
  if (seqs == 0) return IRIS_OK;
  const long items = seqs * heads;
  // whole 16-value blocks with 16-byte rows: on MFMAs (other widths: the general kernel)
  if (head_dim % 16 == 0 && aligned(qkv, 16) && aligned(out, 16) && (items + 3) / 4 < (1L << 31)) {
    const dim3 grid(static_cast<unsigned>((items + 3) / 4));
    const bf16* in = static_cast<const bf16*>(qkv);
    bf16* to = static_cast<bf16*>(out);
    switch (head_dim / 16) {
#define IRIS_DT_CASE(DT)                                                                              \
  case DT:                                                                                            \
    layer_attention_mfma_kernel<DT><<<grid, 256, 0, stream>>>(in, to, items, seq_len, heads, scale);  \
    break;
      IRIS_DT_CASE(1)
      IRIS_DT_CASE(2)
      IRIS_DT_CASE(3)
      IRIS_DT_CASE(4)
      IRIS_DT_CASE(5)
      IRIS_DT_CASE(6)
      IRIS_DT_CASE(7)
      IRIS_DT_CASE(8)
#undef IRIS_DT_CASE
    }
    return check_launch("layer_attention");
  }
  const size_t per_wave = sizeof(float) * layer_attention_floats(seq_len, head_dim);  // <= 25.6 KB
  const int waves = static_cast<int>(std::min<size_t>(kMaxWavesPerBlock, kLdsBudget / per_wave));
  IRIS_REQUIRE((items + waves - 1) / waves < (1L << 31), "layer_attention: grid too large");
  const dim3 grid(static_cast<unsigned>((items + waves - 1) / waves));
  layer_attention_kernel<<<grid, 64 * waves, per_wave * waves, stream>>>(static_cast<const bf16*>(qkv),
                                                                         static_cast<bf16*>(out), seqs, seq_len,
                                                                         heads, head_dim, scale);
  return check_launch("layer_attention");
}

extern "C" int iris_text_key_mask(const void* mask, int elem_kind, long ld, int batch, long n, long n_pad, void* out,
                                  hipStream_t stream) {
  IRIS_REQUIRE(elem_kind >= 0 && elem_kind <= 3, "text_key_mask: element kind 0 (1 byte), 1 (int32), 2 (float32), 3 (int64)");
  IRIS_REQUIRE(batch >= 0 && n > 0 && n_pad >= n && n_pad % 64 == 0 && n_pad < (1L << 24) && ld >= n,
               "text_key_mask: bad shape");
  IRIS_REQUIRE(mask && out && aligned(out, 4), "text_key_mask: bad pointers");
  if (batch == 0) return IRIS_OK;
  const long total = batch * n_pad;
  key_mask_kernel<<<dim3(static_cast<unsigned>((total + 255) / 256)), 256, 0, stream>>>(
      mask, elem_kind, ld, batch, static_cast<int>(n), static_cast<int>(n_pad), static_cast<unsigned char*>(out));
  return check_launch("text_key_mask");
}

extern "C" int iris_layer_pool(const float* h, const void* branch, const float* weight, const float* bias, long rows,
                               int layers, int width, void* out, int out_dtype, hipStream_t stream) {
  IRIS_REQUIRE(rows >= 0 && layers > 0 && width > 0 && width % 4 == 0, "layer_pool: bad shape");
  IRIS_REQUIRE(out_dtype == IRIS_F32 || out_dtype == IRIS_BF16, "layer_pool: unknown output dtype");
  IRIS_REQUIRE(h && weight && out && aligned(h, 16) && aligned(out, 8) && (!branch || aligned(branch, 8)),
               "layer_pool: bad pointers");
  if (rows == 0) return IRIS_OK;
  const long n = rows * (width / 4);
  const dim3 grid(static_cast<unsigned>((n + 255) / 256));
  if (out_dtype == IRIS_F32)
    layer_pool_kernel<float><<<grid, 256, 0, stream>>>(h, static_cast<const bf16*>(branch), weight, bias, rows, layers,
                                                       width, static_cast<float*>(out));
  else
    layer_pool_kernel<bf16><<<grid, 256, 0, stream>>>(h, static_cast<const bf16*>(branch), weight, bias, rows, layers,
                                                      width, static_cast<bf16*>(out));
  return check_launch("layer_pool");
}
