// The decision head after the last projection: each request row's option logits from its own adapter's readout, then
// the masked, tempered softmax (the reference's readout_rows: engine/batched_kernels.py:492-559, with
// DecisionModel.forward's mask and temperature).
//  - readout_logits_kernel: one workgroup per (up to 16 rows of one adapter, 64 options), so a readout is read once for
//    16 of its requests. Its 4 waves slice the hidden dimension (32 inputs in turn); a wave multiplies 4 blocks of 16
//    readout rows by the 16 hidden vectors with 16x16x32 bf16 MFMAs, operands straight from memory (16 rows of 64 bytes an
//    instruction), and the waves' float32 sums are added in wave order, rounded to bf16 and stored as float32. Bound by
//    the readouts' bytes: when every row read its own copy and each logit took a shuffle tree, 512 rows over 128 adapters
//    took 64 us (0.5 GB through the caches, a chain of six lane exchanges a logit).
//  - option_softmax_kernel: one wave per row; options from the row's count on get the logit -1e9, the logits are
//    divided by the adapter's temperature and the softmax taken over all options (max and sum by fixed shuffle trees).
#include "mlora_common.h"

namespace {

using namespace mlora;

constexpr int kRoOptionsPerBlock = 64;
constexpr int kRoThreads = 256;
constexpr int kRoWaves = kRoThreads / 64;
constexpr int kRoBlocks = kRoOptionsPerBlock / 16;  // 16-option MFMA blocks a wave takes
constexpr int kRoRows = 16;                         // rows of one adapter a workgroup takes
constexpr int kRoWindow = 1024;                     // ... among this many consecutive rows
constexpr int kRoAhead = 4;                         // steps whose loads are in flight together

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

__global__ __launch_bounds__(kRoThreads) void readout_logits_kernel(const uint16_t* __restrict__ hidden,
                                                                   int64_t hidden_stride, int32_t dim,
                                                                   const uint16_t* __restrict__ pool,
                                                                   int64_t pool_stride, int32_t options,
                                                                   int32_t pool_rows,
                                                                   const int32_t* __restrict__ adapters, int32_t rows,
                                                                   float* __restrict__ logits) {
  __shared__ float red[kRoWaves][kRoBlocks][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto adapter_of = [&](int i) {
    const int a = adapters[i];
    return a < 0 || a >= pool_rows ? 0 : a;  // an index outside the pool reads row 0: every read stays inside the pool
  };
  // Block b leads if the rows of its adapter before it in its window are a multiple of 16; it then takes itself and the
  // adapter's next 15 rows of the window, lane l the row l & 15 (past the last: its own again, never stored).
  const int b = blockIdx.x;
  const int a = adapter_of(b);
  const int w0 = b - b % kRoWindow, w1 = min(w0 + kRoWindow, rows);
  int before = 0;
  for (int i = w0; i < b; i += 64) {
    const int j = i + lane;
    before += __popcll(__ballot(j < b && adapter_of(min(j, rows - 1)) == a));
  }
  if (before % kRoRows != 0) return;
  int row = b, n = 1;
  for (int i = b + 1; i < w1 && n < kRoRows; i += 64) {
    const int j = i + lane;
    uint64_t m = __ballot(j < w1 && adapter_of(min(j, rows - 1)) == a);
    while (m != 0 && n < kRoRows) {
      if ((lane & 15) == n) row = i + __ffsll((unsigned long long)m) - 1;
      ++n;
      m &= m - 1;
    }
  }
  // operands: lane l holds row (option or request) l & 15, inputs 32 step + 8 (l >> 4) .. +7; options past the last re-read
  // it (their sums are not stored), inputs past the dimension are zero
  const int o0 = blockIdx.y * kRoOptionsPerBlock;
  const uint16_t* hrow = hidden + (int64_t)row * hidden_stride + 8 * (lane >> 4);
  const uint16_t* wrow[kRoBlocks];
#pragma unroll
  for (int q = 0; q < kRoBlocks; ++q)
    wrow[q] = pool + (int64_t)a * pool_stride + (int64_t)min(o0 + 16 * q + (lane & 15), options - 1) * dim + 8 * (lane >> 4);
  f32x4_t acc[kRoBlocks];
#pragma unroll
  for (int q = 0; q < kRoBlocks; ++q) acc[q] = f32x4_t{};
  const int steps = (dim + 31) / 32;
  for (int s0 = wave; s0 < steps; s0 += kRoWaves * kRoAhead) {
    uint4 hv[kRoAhead], wv[kRoAhead][kRoBlocks];
#pragma unroll
    for (int i = 0; i < kRoAhead; ++i) {
      const int c = 32 * (s0 + kRoWaves * i);
      const bool in = c + 8 * (lane >> 4) < dim;
      hv[i] = in ? *reinterpret_cast<const uint4*>(hrow + c) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < kRoBlocks; ++q)
        wv[i][q] = in ? *reinterpret_cast<const uint4*>(wrow[q] + c) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < kRoAhead; ++i)
#pragma unroll
      for (int q = 0; q < kRoBlocks; ++q)
        acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wv[i][q]), as_bf16x8(hv[i]), acc[q], 0, 0, 0);
  }
  // lane l holds request l & 15, options 16 q + 4 (l >> 4) + e
#pragma unroll
  for (int q = 0; q < kRoBlocks; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][q][e][lane] = acc[q][e];
  __syncthreads();
  if ((lane & 15) >= n) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v = red[0][wave][e][lane];
#pragma unroll
    for (int i = 1; i < kRoWaves; ++i) v += red[i][wave][e][lane];
    const int o = o0 + 16 * wave + 4 * (lane >> 4) + e;
    if (o < options) logits[(int64_t)row * options + o] = bf16_to_f32(f32_to_bf16(v));
  }
}

static_assert(kRoBlocks == kRoWaves, "wave q stores block q");

__global__ __launch_bounds__(64) void option_softmax_kernel(const float* __restrict__ logits, int32_t options,
                                                           const int32_t* __restrict__ adapters,
                                                           const int32_t* __restrict__ counts,
                                                           const float* __restrict__ temp_pool, int32_t pool_rows,
                                                           float* __restrict__ out) {
  const int b = blockIdx.x, lane = threadIdx.x;
  int a = adapters[b];
  if (a < 0 || a >= pool_rows) a = 0;
  const int count = counts[b];
  const float t = temp_pool[a];
  constexpr int kPer = 4;  // options per lane: at most 256
  float x[kPer];
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int o = lane + 64 * k;
    float v = -INFINITY;
    if (o < options) {
      v = o < count ? logits[(int64_t)b * options + o] : -1e9f;
      v = v / t;
    }
    x[k] = v;
    m = fmaxf(m, v);
  }
  m = wave_max(m);
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    x[k] = lane + 64 * k < options ? expf(x[k] - m) : 0.0f;
    s += x[k];
  }
  s = wave_sum(s);
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int o = lane + 64 * k;
    if (o < options) out[(int64_t)b * options + o] = x[k] / s;
  }
}

}  // namespace

int launch_readout_logits(const uint16_t* hidden, int64_t hidden_stride, int32_t dim, const uint16_t* pool,
                          int64_t pool_stride, int32_t options, int32_t pool_rows, const int32_t* adapters,
                          int32_t rows, float* logits, hipStream_t stream) {
  if (rows == 0) return MLORA_OK;
  const dim3 grid((unsigned)rows, (unsigned)((options + kRoOptionsPerBlock - 1) / kRoOptionsPerBlock));
  hipLaunchKernelGGL(readout_logits_kernel, grid, dim3(kRoThreads), 0, stream, hidden, hidden_stride, dim, pool,
                     pool_stride, options, pool_rows, adapters, rows, logits);
  return hipGetLastError() == hipSuccess ? MLORA_OK : MLORA_ELAUNCH;
}

int launch_option_softmax(const float* logits, int32_t options, const int32_t* adapters, const int32_t* counts,
                          const float* temp_pool, int32_t pool_rows, int32_t rows, float* probs, hipStream_t stream) {
  if (rows == 0) return MLORA_OK;
  hipLaunchKernelGGL(option_softmax_kernel, dim3((unsigned)rows), dim3(64), 0, stream, logits, options, adapters,
                     counts, temp_pool, pool_rows, probs);
  return hipGetLastError() == hipSuccess ? MLORA_OK : MLORA_ELAUNCH;
}
