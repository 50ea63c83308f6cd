// BF16-weight matrix-vector products for the per-step conditioning: the timestep MLP and
// the shared adaLN cores (M = batch <= 4 per launch). HBM-bound on the weight read.
//
// gemv_rows_kernel: a wave owns R consecutive weight rows and streams them with 16-byte loads,
// DEPTH rows ahead, against its slice of the (activated) input vectors held in registers (lane l
// has the 8-element chunks l, l + 64, ..), so nothing but weights moves in the row loop. The
// inputs are activated once per workgroup and reach the registers through LDS. R = 8 where that
// still gives every CU a workgroup or two (the per-block copies of an output then leave as 32-byte
// pieces), else 2; figures at launch_rows.
// gemv_kernel: any k and batch whose inputs do not fit the registers (more than 20 chunks per lane).
// Both add a row's products in the same order, so they agree bit for bit.
#include "iris_common.hpp"

namespace iris {
namespace {

constexpr int kMaxBatch = 4;
constexpr int kRowsPerWave = 2;
constexpr int kRowsPerBlock = 4 * kRowsPerWave;

template <int NCH, int NB, int R>
__global__ __launch_bounds__(256, 2) void gemv_rows_kernel(const bf16* __restrict__ w, const float* __restrict__ x, int n,
                                                        int k, const float* __restrict__ bias,
                                                        const float* __restrict__ extra, int n_extra,
                                                        float* __restrict__ out, long out_bstride, long out_jstride,
                                                        int in_act, int out_act) {
  constexpr int DEPTH = R < 4 ? R : (NB * NCH > 10 ? 2 : 4);  // rows in flight
  extern __shared__ float xs[];  // NB * k
  const int lane = threadIdx.x & 63;
  const int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
  const int chunks = k >> 3;
  bf16x8 wv[DEPTH][NCH];
  auto load_row = [&](int r) {
    const bf16* wr = w + static_cast<long>(min(row0 + r, n - 1)) * k;  // (rows past n read a valid one)
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + kWave * i;  // (only the last chunk of a lane can lie past the row)
      wv[r % DEPTH][i] = i + 1 < NCH || c < chunks ? *reinterpret_cast<const bf16x8*>(wr + 8 * c) : bf16x8{};
    }
  };
#pragma unroll
  for (int r = 0; r < DEPTH; ++r) load_row(r);
  for (int i = 4 * threadIdx.x; i < NB * k; i += 4 * 256) {
    f32x4 v = load4(x + i);
    if (in_act == IRIS_ACT_SILU) v = f32x4{silu(v[0]), silu(v[1]), silu(v[2]), silu(v[3])};
    store4(xs + i, v);
  }
  __syncthreads();
  if (row0 >= n) return;
  float xv[NB][NCH][8];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + kWave * i;
      if (i + 1 < NCH || c < chunks) {
        load8(xs + b * k + 8 * c, xv[b][i]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[b][i][e] = 0.0f;
      }
    }
  float y[NB][R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      float wf[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) wf[e] = to_f32(wv[r % DEPTH][i][e]);
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[b] = __builtin_fmaf(wf[e], xv[b][i][e], acc[b]);
    }
    if (r + DEPTH < R) load_row(r + DEPTH);
#pragma unroll
    for (int b = 0; b < NB; ++b) y[b][r] = wave_sum(acc[b]);  // (every lane holds the sum)
  }
  // lane l finishes row l % R: one activation per row, then the outputs in pieces of R floats
  const int rr = lane % R;
  const int row = row0 + rr;
  if (row >= n) return;
  const float bv = bias ? bias[row] : 0.0f;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    float v = y[b][0];
#pragma unroll
    for (int r = 1; r < R; ++r) v = rr == r ? y[b][r] : v;
    if (bias) v += bv;
    if (out_act == IRIS_ACT_SILU) v = silu(v);
    if (n_extra == 0) {
      if (lane < R) out[b * out_bstride + row] = v;
    } else {
      for (int j = lane / R; j < n_extra; j += kWave / R)
        out[j * out_jstride + b * out_bstride + row] = v + extra[static_cast<long>(j) * n + row];
    }
  }
}

__global__ __launch_bounds__(256) void gemv_kernel(const bf16* __restrict__ w, const float* __restrict__ x,
                                                   int nb, int n, int k, const float* __restrict__ bias,
                                                   const float* __restrict__ extra, int n_extra,
                                                   float* __restrict__ out, long out_bstride, long out_jstride,
                                                   int in_act, int out_act) {
  extern __shared__ float xs[];  // nb * k
  for (int i = threadIdx.x; i < nb * k; i += 256) {
    const float v = x[i];
    xs[i] = in_act == IRIS_ACT_SILU ? silu(v) : v;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int row0 = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6) * kRowsPerWave;
  const int chunks = k >> 3;
#pragma unroll
  for (int rr = 0; rr < kRowsPerWave; ++rr) {
    const int row = row0 + rr;
    if (row >= n) break;  // uniform across the wave
    float acc[kMaxBatch] = {0.0f, 0.0f, 0.0f, 0.0f};
    const bf16* wr = w + static_cast<long>(row) * k;
    for (int c = lane; c < chunks; c += kWave) {
      float wv[8];
      load8(wr + 8 * c, wv);
#pragma unroll
      for (int b = 0; b < kMaxBatch; ++b) {
        if (b < nb) {
          const float* xb = xs + b * k + 8 * c;
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[b] = __builtin_fmaf(wv[e], xb[e], acc[b]);
        }
      }
    }
#pragma unroll
    for (int b = 0; b < kMaxBatch; ++b) {
      if (b >= nb) break;
      float y = wave_sum(acc[b]);  // (every lane holds the sum)
      if (bias) y += bias[row];
      if (out_act == IRIS_ACT_SILU) y = silu(y);
      if (n_extra == 0) {
        if (lane == 0) out[b * out_bstride + row] = y;
      } else {  // the per-block copies, one per lane
        for (int j = lane; j < n_extra; j += kWave)
          out[j * out_jstride + b * out_bstride + row] = y + extra[static_cast<long>(j) * n + row];
      }
    }
  }
}

struct GemvArgs {
  const bf16* w;
  const float* x;
  int n, k;
  const float *bias, *extra;
  int n_extra;
  float* out;
  long out_bstride, out_jstride;
  int in_act, out_act;
};

// Measured on one box, us per call (TB/s of weight), HIP-graph replays with every weight from HBM:
//                                    batch 1        2             3             4
//   15360 x 2560, 24 bias rows, before 28.8 (2.7)   48.2 (1.6)    73.2 (1.1)    99.4 (0.8)
//                               now    16.7 (4.7)   19.2 (4.1)    21.2 (3.7)    28.8 (2.7)
//   2560 x 2560                 before 11.7 (1.1)   16.6          22.5          28.7
//                               now     6.0 (2.2)    7.0           8.4           9.6
// (before: gemv_kernel, whose input reads from LDS grew with the batch). A copy of this size class
// moves 4.8 TB/s; batch 4 has two waves per SIMD to hide its latency (250 VGPRs).
template <int NCH, int NB>
void launch_rows(const GemvArgs& a, hipStream_t stream) {
  const size_t lds = static_cast<size_t>(NB) * a.k * sizeof(float);
  const bool many = a.n >= 4 * 8 * device_cus();  // 8 rows per wave still fill the CUs
  const int per_wg = 4 * (many ? 8 : 2);
  const dim3 grid((a.n + per_wg - 1) / per_wg);
  if (many)
    gemv_rows_kernel<NCH, NB, 8><<<grid, 256, lds, stream>>>(a.w, a.x, a.n, a.k, a.bias, a.extra, a.n_extra, a.out,
                                                             a.out_bstride, a.out_jstride, a.in_act, a.out_act);
  else
    gemv_rows_kernel<NCH, NB, 2><<<grid, 256, lds, stream>>>(a.w, a.x, a.n, a.k, a.bias, a.extra, a.n_extra, a.out,
                                                             a.out_bstride, a.out_jstride, a.in_act, a.out_act);
}

template <int NCH>
bool launch_batch(const GemvArgs& a, int nb, hipStream_t stream) {
  switch (nb) {
    case 1: launch_rows<NCH, 1>(a, stream); return true;
    case 2: launch_rows<NCH, 2>(a, stream); return true;
    case 3: if constexpr (3 * NCH <= 20) { launch_rows<NCH, 3>(a, stream); return true; } break;
    case 4: if constexpr (4 * NCH <= 20) { launch_rows<NCH, 4>(a, stream); return true; } break;
  }
  return false;
}

// The register form where it is instantiated (the chunks per lane of the widths in use: 256, 2560).
bool launch_registers(const GemvArgs& a, int nb, hipStream_t stream) {
  if (!aligned(a.x, 16)) return false;
  const int nch = (a.k / 8 + kWave - 1) / kWave;
  if (nch == 1) return launch_batch<1>(a, nb, stream);
  if (nch == 5) return launch_batch<5>(a, nb, stream);
  return false;
}

}  // namespace
}  // namespace iris

using namespace iris;

extern "C" int iris_gemv_bf16(const void* w, const float* x, int batch, int n, int k, const float* bias,
                              const float* extra_bias, int n_extra, float* out, int in_act, int out_act,
                              hipStream_t stream) {
  IRIS_REQUIRE(batch >= 0 && n > 0 && k > 0 && k % 8 == 0 && k <= 4096, "gemv: need k %% 8 == 0 and k <= 4096");
  IRIS_REQUIRE(n_extra >= 0 && (n_extra == 0 || extra_bias), "gemv: extra biases missing");
  IRIS_REQUIRE((in_act == IRIS_ACT_NONE || in_act == IRIS_ACT_SILU) &&
                   (out_act == IRIS_ACT_NONE || out_act == IRIS_ACT_SILU),
               "gemv: unknown activation");
  IRIS_REQUIRE(w && x && out, "gemv: null pointer");
  IRIS_REQUIRE(aligned(w, 16), "gemv: weight must be 16-byte aligned");
  const long out_bstride = n;
  const long out_jstride = static_cast<long>(batch) * n;
  for (int b0 = 0; b0 < batch; b0 += kMaxBatch) {
    const int nb = batch - b0 < kMaxBatch ? batch - b0 : kMaxBatch;
    const GemvArgs args{static_cast<const bf16*>(w), x + static_cast<long>(b0) * k, n, k, bias, extra_bias, n_extra,
                        out + static_cast<long>(b0) * n, out_bstride, out_jstride, in_act, out_act};
    if (!launch_registers(args, nb, stream)) {
      const dim3 grid((n + kRowsPerBlock - 1) / kRowsPerBlock);
      const size_t lds = static_cast<size_t>(nb) * k * sizeof(float);
      gemv_kernel<<<grid, 256, lds, stream>>>(args.w, args.x, nb, n, k, bias, extra_bias, n_extra, args.out, out_bstride,
                                              out_jstride, in_act, out_act);
    }
    const int rc = check_launch("gemv");
    if (rc) return rc;
  }
  return IRIS_OK;
}
