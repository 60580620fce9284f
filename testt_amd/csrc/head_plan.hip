// The small steps around the head's chunk kernels, each one launch and none of them waiting on the
// host (solution/head.py:93-137 sorts the rows, reads the counts back, and scales and scatters
// the gradient with a dozen torch operations):
//
//   soupk_head_plan    per row of a chunk its slot among the chunk's labelled rows (-1: ignored),
//                      the labelled rows per chunk, and the gradient's scale and unit
//   soupk_head_finish  loss = sum(token loss) / denominator, and the argmax hits as bytes
//   soupk_head_dh      [rows, H] gradient of the hidden states from the packed chunk rows
//
// All three are bound by launch latency at the sizes of a training step (2048 rows: 16 KB of
// labels, 12 MB of gradient); what they replace is about 30 torch launches of 2 - 5 us each, one
// device-to-host copy and its wait (head loss forward + backward at 24 rows 406 -> 217 us, at 700
// rows 924 -> 698 us on MI355X).

#include "soupk_common.hpp"

namespace soupk {
namespace {

constexpr int64_t kIgnore = -100;
constexpr int kPlanThreads = 1024;

// The power of two G nearest 64 * max(d, 1e-6) on a log scale, clamped to [1, 2^16]
// (solution/head.py:79-84) for an integer d: 2^(round(log2 d) + 6), where log2 d rounds up
// when d^2 > 2^(2e + 1), e = floor(log2 d) (equality is impossible).
__device__ double grad_unit(int64_t d) {
  if (d <= 0) return 1.0;            // log2(1e-6) + 6 < 0
  if (d >= 2048) return 65536.0;
  const int e = 31 - __clz(static_cast<int>(d));
  const int r = e + (d * d > (int64_t{1} << (2 * e + 1)) ? 1 : 0) + 6;
  return static_cast<double>(1 << min(r, 16));
}

// One workgroup per chunk: ranks by wavefront ballots, 1024 rows at a time.
__global__ __launch_bounds__(kPlanThreads) void head_plan_kernel(
    const int64_t* __restrict__ target, int64_t rows, int64_t chunk, int32_t* __restrict__ slot,
    int32_t* __restrict__ counts, const int64_t* __restrict__ denominator, float scale,
    float unit, float* __restrict__ scal) {
  __shared__ int wave_n[kPlanThreads / kWave];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t r0 = blockIdx.x * chunk, r1 = min(r0 + chunk, rows);
  int base = 0;
  for (int64_t r = r0; r < r1; r += kPlanThreads) {
    const int64_t i = r + threadIdx.x;
    const bool lab = i < r1 && target[i] != kIgnore;
    const uint64_t mask = __ballot(lab);
    __syncthreads();                       // wave_n of the last round has been read
    if (lane == 0) wave_n[w] = __popcll(mask);
    __syncthreads();
    int before = base;
#pragma unroll
    for (int k = 0; k < kPlanThreads / kWave; ++k) {
      const int n = wave_n[k];
      before += k < w ? n : 0;
      base += n;
    }
    if (i < r1) slot[i] = lab ? before + __popcll(mask & ((uint64_t{1} << lane) - 1)) : -1;
  }
  if (threadIdx.x == 0) {
    counts[blockIdx.x] = base;
    if (blockIdx.x == 0) {
      if (denominator != nullptr) {
        const int64_t d = *denominator;
        const double u = grad_unit(d);
        unit = static_cast<float>(u);
        scale = static_cast<float>(u / fmax(static_cast<double>(d), 1e-6));
      }
      scal[0] = scale;
      scal[1] = unit;
    }
  }
}

// Sum in 64 bits over strided lanes (a fixed order), one rounding, then the fp32 division that
// torch makes of an fp32 sum and an integer or Python denominator.
__global__ __launch_bounds__(kPlanThreads) void head_finish_kernel(
    const float* __restrict__ token_loss, const int32_t* __restrict__ correct, int64_t rows,
    const int64_t* __restrict__ denominator, float den, float* __restrict__ loss,
    uint8_t* __restrict__ hit) {
  __shared__ double part[kPlanThreads / kWave];
  double s = 0.0;
  for (int64_t i = threadIdx.x; i < rows; i += kPlanThreads) {
    s += static_cast<double>(token_loss[i]);
    hit[i] = correct[i] != 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int k = 0; k < kPlanThreads / kWave; ++k) t += part[k];
    const float d = denominator != nullptr ? static_cast<float>(*denominator) : den;
    *loss = static_cast<float>(t) / d;
  }
}

// dh[m] = fp16(fp32(packed row of m) * (grad_loss / unit)), zeros for an ignored row; a chunk's
// packed rows start at the chunk's first row.
__global__ __launch_bounds__(256) void head_dh_kernel(
    const u32x4* __restrict__ packed, const int32_t* __restrict__ slot,
    const float* __restrict__ grad_loss, const float* __restrict__ scal, u32x4* __restrict__ dh,
    int64_t n8, int h8, int64_t chunk) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n8) return;
  const int64_t m = i / h8;
  const int s = slot[m];
  u32x4 out = {0u, 0u, 0u, 0u};
  if (s >= 0 && s < chunk) {
    const float f = *grad_loss / scal[1];
    const u32x4 v = packed[(m / chunk * chunk + s) * h8 + (i - m * h8)];
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = pack_h2(lo_h(v[k]) * f, hi_h(v[k]) * f);
  }
  dh[i] = out;
}

bool bad16(const void* p) { return p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15); }

}  // namespace
}  // namespace soupk

using namespace soupk;

extern "C" __attribute__((visibility("default"))) int soupk_head_plan(
    const int64_t* target, int64_t rows, int64_t chunk, int32_t* slot, int32_t* counts,
    const int64_t* denominator, float scale, float unit, float* scal, void* stream) {
  if (rows < 0 || chunk < 1 || chunk > 0x7fffffff) return kInvalid;
  if (rows == 0) return kOk;
  if (!target || !slot || !counts || !scal) return kInvalid;
  const int64_t n = (rows + chunk - 1) / chunk;
  if (n > 0x7fffffff) return kInvalid;
  return launch_kernel(head_plan_kernel, dim3(static_cast<unsigned>(n)), dim3(kPlanThreads),
                       static_cast<hipStream_t>(stream), target, rows, chunk, slot, counts,
                       denominator, scale, unit, scal);
}

extern "C" __attribute__((visibility("default"))) int soupk_head_finish(
    const float* token_loss, const int32_t* correct, int64_t rows, const int64_t* denominator,
    float den, float* loss, uint8_t* hit, void* stream) {
  if (rows < 0) return kInvalid;
  if (rows == 0) return kOk;
  if (!token_loss || !correct || !loss || !hit) return kInvalid;
  return launch_kernel(head_finish_kernel, dim3(1), dim3(kPlanThreads),
                       static_cast<hipStream_t>(stream), token_loss, correct, rows, denominator,
                       den, loss, hit);
}

extern "C" __attribute__((visibility("default"))) int soupk_head_dh(
    const uint16_t* packed, const int32_t* slot, const float* grad_loss, const float* scal,
    uint16_t* dh, int64_t rows, int32_t H, int64_t chunk, void* stream) {
  if (rows < 0 || H <= 0 || H % 8 || chunk < 1) return kInvalid;
  if (rows == 0) return kOk;
  if (bad16(packed) || bad16(dh) || !slot || !grad_loss || !scal) return kInvalid;
  const int64_t n8 = rows * (H / 8);
  if ((n8 + 255) / 256 > 0x7fffffff) return kInvalid;
  return launch_kernel(head_dh_kernel, dim3(static_cast<unsigned>((n8 + 255) / 256)), dim3(256),
                       static_cast<hipStream_t>(stream), reinterpret_cast<const u32x4*>(packed),
                       slot, grad_loss, scal, reinterpret_cast<u32x4*>(dh), n8, H / 8, chunk);
}
