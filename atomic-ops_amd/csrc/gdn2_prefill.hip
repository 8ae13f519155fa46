// Checks and reset flags of a prefill (chunk_forward_inference) in one pass before its kernels: the
// extremes of the gate g, whether a document boundary lies inside a full chunk, and the reset bytes
// of the chunks and of the tail's tokens.  As torch operations these were some twenty small launches
// and a 23 us reduction, and the device idled while the host read them back; now the prefill is
// enqueued behind this kernel and the caller waits for its statistics alone.  B2 H16 L3000, bf16,
// four documents: 406 -> 313 us a call.
#include "gdn2_kernels.hpp"

namespace gdn2 {

// NaN propagates, as in torch.aminmax (and the caller then lets it pass)
__device__ __forceinline__ float min_nan(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float max_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }

template <bool BF>
__device__ __forceinline__ void g_extremes(const PrefillPrepArgs& a) {
  __shared__ float slo[4], shi[4];
  float lo = __builtin_inff(), hi = -__builtin_inff();
  const size_t n4 = a.n_g / 4, step = (size_t)PREP_G_BLOCKS * 256;
  auto take = [&](float x) {
    lo = min_nan(lo, x);
    hi = max_nan(hi, x);
  };
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += step) {
    float4 x;
    if constexpr (BF) {
      const uint2 u = reinterpret_cast<const uint2*>(a.g)[i];
      x = make_float4(bf16_val(u.x & 0xffffu), bf16_val(u.x >> 16), bf16_val(u.y & 0xffffu), bf16_val(u.y >> 16));
    } else {
      x = reinterpret_cast<const float4*>(a.g)[i];
    }
    take(x.x);
    take(x.y);
    take(x.z);
    take(x.w);
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    lo = min_nan(lo, __shfl_xor(lo, m));
    hi = max_nan(hi, __shfl_xor(hi, m));
  }
  if (lane_id() == 0) {
    slo[wave_id()] = lo;
    shi[wave_id()] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    a.stats[2 * blockIdx.x] = min_nan(min_nan(slo[0], slo[1]), min_nan(slo[2], slo[3]));
    a.stats[2 * blockIdx.x + 1] = max_nan(max_nan(shi[0], shi[1]), max_nan(shi[2], shi[3]));
  }
}

// One wave per (batch row, chunk), then one per batch row for the tail.
__global__ __launch_bounds__(256) void prefill_prep_kernel(PrefillPrepArgs a) {
  if (blockIdx.x < PREP_G_BLOCKS) {
    if (a.g_bf16) g_extremes<true>(a);
    else g_extremes<false>(a);
    return;
  }
  const int wv = (blockIdx.x - PREP_G_BLOCKS) * 4 + wave_id(), l = lane_id();
  if (wv >= a.B * (a.n_full + 1)) return;
  const int b = wv / (a.n_full + 1), c = wv - b * (a.n_full + 1);
  auto id = [&](int t) -> int64_t {
    const size_t i = (size_t)b * a.L + t;
    return a.seg64 ? static_cast<const int64_t*>(a.seg)[i] : static_cast<const int32_t*>(a.seg)[i];
  };
  if (c < a.n_full) {
    const int64_t first = id(c * a.bt);
    bool differs = false;
    for (int t = l; t < a.bt; t += WAVE) differs = differs || id(c * a.bt + t) != first;
    const bool bad = __ballot(differs) != 0;
    if (l == 0) a.stats[2 * PREP_G_BLOCKS + b * a.n_full + c] = bad ? 1.f : 0.f;
    const uint8_t chg = c > 0 && id((c - 1) * a.bt) != first;
    const int G = a.bt / T, n64 = a.n_full * G;      // the chunk's first 64-token part carries the flag
    for (int i = l; i < a.H * G; i += WAVE) {
      const int h = i / G, j = i - h * G;
      a.flags[((size_t)b * a.H + h) * n64 + c * G + j] = j == 0 ? chg : 0;
    }
  } else {
    const int t0 = a.n_full * a.bt, n = a.L - t0;
    for (int i = l; i < n; i += WAVE) a.tail_flags[(size_t)b * n + i] = t0 + i > 0 && id(t0 + i) != id(t0 + i - 1);
  }
}

hipError_t launch_prefill_prep(const PrefillPrepArgs& a, hipStream_t s) {
  const int seg_blocks = a.seg ? (a.B * (a.n_full + 1) + 3) / 4 : 0;
  hipLaunchKernelGGL(prefill_prep_kernel, dim3(PREP_G_BLOCKS + seg_blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace gdn2
