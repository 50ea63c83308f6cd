// BF16-weight matrix-vector products for the per-step conditioning: the timestep MLP and
// the shared adaLN cores (M = batch <= 4 per launch). HBM-bound on the weight read.
//
// gemv_rows_kernel: a wave owns R consecutive weight rows and streams them with 16-byte loads,
// DEPTH rows ahead, against its slice of the (activated) input vectors held in registers (lane l
// has the 8-element chunks l, l + 64, ..), so nothing but weights moves in the row loop. The
// inputs are activated once per workgroup and reach the registers through LDS. R = 8 where that
// still gives every CU a workgroup or two (the per-block copies of an output then leave as 32-byte
// pieces), else 2; figures at launch_rows.
// One launch runs the image and the text core (they share their inputs), and the first timestep
// layer computes the sinusoidal features it reads, so the chain is three launches: 51 -> 44 us per
// denoise step.
// It is instantiated for the widths in use, one or five chunks per lane: k <= 512 and 2056 <= k <= 2560.
// gemv_kernel: every other k, and inputs that are not 16-byte aligned.
// Both add a row's products in the same order, so they agree bit for bit.
#include "iris_common.hpp"

namespace iris {
namespace {

constexpr int kMaxBatch = 4;
constexpr int kRowsPerWave = 2;
constexpr int kRowsPerBlock = 4 * kRowsPerWave;

// One product over the inputs of a launch.
struct GemvJob {
  const bf16* w;
  int n;
  const float *bias, *extra;
  int n_extra;
  float* out;
  long out_bstride, out_jstride;
};
// A launch: one job, or two on the same inputs (workgroups from `blocks0` on run the second). With
// freqs the inputs are the timestep features [cos | sin](x[b] freqs) of k / 2 frequencies.
struct GemvLaunch {
  GemvJob job[2];
  int blocks0;
  const float *x, *freqs;
  int k, in_act, out_act;
};

template <int NCH, int NB, int R>
__global__ __launch_bounds__(256, 2) void gemv_rows_kernel(GemvLaunch a) {
  constexpr int DEPTH = R < 4 ? R : (NB * NCH > 10 ? 2 : 4);  // rows in flight
  extern __shared__ float xs[];  // NB * k
  const bool second = static_cast<int>(blockIdx.x) >= a.blocks0;
  const GemvJob& job = second ? a.job[1] : a.job[0];
  const bf16* __restrict__ w = job.w;
  const float* __restrict__ x = a.x;
  const float* __restrict__ bias = job.bias;
  const float* __restrict__ extra = job.extra;
  float* __restrict__ out = job.out;
  const int n = job.n, k = a.k, n_extra = job.n_extra;
  const long out_bstride = job.out_bstride, out_jstride = job.out_jstride;
  const int lane = threadIdx.x & 63;
  const int row0 = ((static_cast<int>(blockIdx.x) - (second ? a.blocks0 : 0)) * 4 + (threadIdx.x >> 6)) * R;
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
  if (a.freqs) {
    const int half = k >> 1;
    for (int i = threadIdx.x; i < NB * half; i += 256) {
      const int b = i / half, j = i - b * half;
      const float phase = x[b] * a.freqs[j];
      xs[b * k + j] = cosf(phase);
      xs[b * k + half + j] = sinf(phase);
    }
  } else {
    for (int i = 4 * threadIdx.x; i < NB * k; i += 4 * 256) {
      f32x4 v = load4(x + i);
      if (a.in_act == IRIS_ACT_SILU) v = f32x4{silu(v[0]), silu(v[1]), silu(v[2]), silu(v[3])};
      store4(xs + i, v);
    }
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
    if (a.out_act == IRIS_ACT_SILU) v = silu(v);
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

// Measured on one box, us per call (TB/s of weight), HIP-graph replays with every weight from HBM:
//                                    batch 1        2             3             4
//   15360 x 2560, 24 bias rows, before 28.8 (2.7)   48.2 (1.6)    73.2 (1.1)    99.4 (0.8)
//                               now    16.7 (4.7)   19.2 (4.1)    21.2 (3.7)    28.8 (2.7)
//   2560 x 2560                 before 11.7 (1.1)   16.6          22.5          28.7
//                               now     6.0 (2.2)    7.0           8.4           9.6
// (before: gemv_kernel, whose input reads from LDS grew with the batch). A copy of this size class
// moves 4.8 TB/s; batch 4 has two waves per SIMD to hide its latency (250 VGPRs).
template <int NCH, int NB>
void launch_rows(GemvLaunch& a, int jobs, hipStream_t stream) {
  const size_t lds = static_cast<size_t>(NB) * a.k * sizeof(float);
  const int rows = a.job[0].n + (jobs > 1 ? a.job[1].n : 0);
  const bool many = rows >= 4 * 8 * device_cus();  // 8 rows per wave still fill the CUs
  const int per_wg = 4 * (many ? 8 : 2);
  a.blocks0 = (a.job[0].n + per_wg - 1) / per_wg;
  const dim3 grid(a.blocks0 + (jobs > 1 ? (a.job[1].n + per_wg - 1) / per_wg : 0));
  if (many)
    gemv_rows_kernel<NCH, NB, 8><<<grid, 256, lds, stream>>>(a);
  else
    gemv_rows_kernel<NCH, NB, 2><<<grid, 256, lds, stream>>>(a);
}

template <int NCH>
bool launch_batch(GemvLaunch& a, int jobs, int nb, hipStream_t stream) {
  switch (nb) {
    case 1: launch_rows<NCH, 1>(a, jobs, stream); return true;
    case 2: launch_rows<NCH, 2>(a, jobs, stream); return true;
    case 3: launch_rows<NCH, 3>(a, jobs, stream); return true;
    case 4: launch_rows<NCH, 4>(a, jobs, stream); return true;
  }
  return false;
}

// The register form where it is instantiated: one chunk per lane (timestep features, also those that
// a launch computes itself: at most 512 wide) or five (the model's width).
bool launch_registers(GemvLaunch& a, int jobs, int nb, hipStream_t stream) {
  if (!a.freqs && !aligned(a.x, 16)) return false;
  const int nch = (a.k / 8 + kWave - 1) / kWave;
  if (nch == 1) return launch_batch<1>(a, jobs, nb, stream);
  if (nch == 5) return launch_batch<5>(a, jobs, nb, stream);
  return false;
}

// `jobs` products of all batch items, four items per launch; the jobs' outputs are [n_extra,] batch, n.
int gemv_launch(const GemvLaunch& whole, int jobs, int batch, hipStream_t stream) {
  for (int b0 = 0; b0 < batch; b0 += kMaxBatch) {
    const int nb = batch - b0 < kMaxBatch ? batch - b0 : kMaxBatch;
    GemvLaunch a = whole;
    a.x += static_cast<long>(b0) * (a.freqs ? 1 : a.k);
    for (int j = 0; j < jobs; ++j) {
      a.job[j].out_bstride = a.job[j].n;
      a.job[j].out_jstride = static_cast<long>(batch) * a.job[j].n;
      a.job[j].out += static_cast<long>(b0) * a.job[j].n;
    }
    if (!launch_registers(a, jobs, nb, stream)) {
      for (int j = 0; j < jobs; ++j) {
        const GemvJob& g = a.job[j];
        const dim3 grid((g.n + kRowsPerBlock - 1) / kRowsPerBlock);
        const size_t lds = static_cast<size_t>(nb) * a.k * sizeof(float);
        gemv_kernel<<<grid, 256, lds, stream>>>(g.w, a.x, nb, g.n, a.k, g.bias, g.extra, g.n_extra, g.out,
                                                g.out_bstride, g.out_jstride, a.in_act, a.out_act);
      }
    }
    const int rc = check_launch("gemv");
    if (rc) return rc;
  }
  return IRIS_OK;
}

int check_job(const GemvJob& job, int k) {
  IRIS_REQUIRE(job.n > 0 && k > 0 && k % 8 == 0 && k <= 4096, "gemv: need k %% 8 == 0 and k <= 4096");
  IRIS_REQUIRE(job.n_extra >= 0 && (job.n_extra == 0 || job.extra), "gemv: extra biases missing");
  IRIS_REQUIRE(job.w && job.out, "gemv: null pointer");
  IRIS_REQUIRE(aligned(job.w, 16), "gemv: weight must be 16-byte aligned");
  return IRIS_OK;
}

bool valid_act(int act) { return act == IRIS_ACT_NONE || act == IRIS_ACT_SILU; }

}  // namespace
}  // namespace iris

using namespace iris;

extern "C" int iris_gemv_bf16(const void* w, const float* x, int batch, int n, int k, const float* bias,
                              const float* extra_bias, int n_extra, float* out, int in_act, int out_act,
                              hipStream_t stream) {
  GemvLaunch a{};
  a.job[0] = GemvJob{static_cast<const bf16*>(w), n, bias, extra_bias, n_extra, out, 0, 0};
  a.x = x;
  a.k = k;
  a.in_act = in_act;
  a.out_act = out_act;
  IRIS_REQUIRE(batch >= 0 && x, "gemv: bad batch or input");
  IRIS_REQUIRE(valid_act(in_act) && valid_act(out_act), "gemv: unknown activation");
  const int rc = check_job(a.job[0], k);
  return rc ? rc : gemv_launch(a, 1, batch, stream);
}

extern "C" int iris_gemv_bf16_pair(const void* const* w, const float* x, int batch, const int* n, int k,
                                   const float* const* bias, const float* const* extra_bias, const int* n_extra,
                                   float* const* out, int in_act, int out_act, hipStream_t stream) {
  IRIS_REQUIRE(w && n && bias && extra_bias && n_extra && out, "gemv: null pointer");
  IRIS_REQUIRE(batch >= 0 && x, "gemv: bad batch or input");
  IRIS_REQUIRE(valid_act(in_act) && valid_act(out_act), "gemv: unknown activation");
  GemvLaunch a{};
  a.x = x;
  a.k = k;
  a.in_act = in_act;
  a.out_act = out_act;
  for (int j = 0; j < 2; ++j) {
    a.job[j] = GemvJob{static_cast<const bf16*>(w[j]), n[j], bias[j], extra_bias[j], n_extra[j], out[j], 0, 0};
    const int rc = check_job(a.job[j], k);
    if (rc) return rc;
  }
  return gemv_launch(a, 2, batch, stream);
}

extern "C" int iris_timestep_gemv_bf16(const float* t, const float* freqs, int half, const void* w, int batch, int n,
                                       const float* bias, float* out, int out_act, hipStream_t stream) {
  IRIS_REQUIRE(batch >= 0 && t && freqs && half > 0 && half % 4 == 0 && half <= 256,
               "timestep_gemv: need 4 to 256 frequencies, a multiple of 4");
  IRIS_REQUIRE(valid_act(out_act), "gemv: unknown activation");
  GemvLaunch a{};
  a.job[0] = GemvJob{static_cast<const bf16*>(w), n, bias, nullptr, 0, out, 0, 0};
  a.x = t;
  a.freqs = freqs;
  a.k = 2 * half;
  a.in_act = IRIS_ACT_NONE;
  a.out_act = out_act;
  const int rc = check_job(a.job[0], a.k);
  return rc ? rc : gemv_launch(a, 1, batch, stream);
}
