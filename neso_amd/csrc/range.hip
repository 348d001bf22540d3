// Largest |x| of up to three fp32 tensors in one launch, read by the host
// while later work of the stream runs.
//
// The split-precision kernels need the magnitude of their inputs on the host
// (to rescale, or to refuse, before the caller sees a result).  Each
// workgroup reduces its share of one tensor and stores the maximum's bits
// straight to its own slot of pinned host memory, where the host polls for
// them (neso_abs_max_wait): no counter or accumulator to clear, no copy, and
// no stream synchronisation, so a launch queued behind this one keeps the
// GPU busy while the host looks at the result.
//
// Bound: HBM, every element once.  Maxima are taken on the bit patterns of
// |x|, so any NaN gives a NaN and else any infinity gives an infinity.
#include <chrono>

#include "common.h"
#include "neso_internal.h"

namespace neso {

namespace {

constexpr int kRangeThreads = 256;
constexpr int kRangeLoads = 4;  // 16-byte loads in flight per thread

// FLAT: every tensor is one contiguous run and nothing is added.
template <bool FLAT>
__global__ __launch_bounds__(kRangeThreads) void abs_max_kernel(RangeArgs a, uint32_t* slots) {
  const int t = blockIdx.y;
  const float* x = a.x[t];
  const int quads = a.dim / 4;
  const uint32_t total = (uint32_t)a.batch * a.rows[t] * quads;
  const uint32_t step = gridDim.x * kRangeThreads;
  uint32_t m = 0;
  auto load = [&](uint32_t i) {
    if constexpr (FLAT) return *reinterpret_cast<const float4v*>(x + 4 * (int64_t)i);
    const uint32_t row = i / quads, c = 4 * (i % quads), b = row / a.rows[t];
    float4v v = *reinterpret_cast<const float4v*>(x + b * a.batch_stride[t] +
                                                  (row - b * a.rows[t]) * (int64_t)a.row_stride[t] + c);
    if (t == 0 && a.add) v += *reinterpret_cast<const float4v*>(a.add + (int64_t)b * a.dim + c);
    return v;
  };
  for (uint32_t i = blockIdx.x * kRangeThreads + threadIdx.x; i < total; i += kRangeLoads * step) {
    float4v v[kRangeLoads];
#pragma unroll
    for (int u = 0; u < kRangeLoads; ++u) v[u] = load(min(i + u * step, total - 1));
#pragma unroll
    for (int u = 0; u < kRangeLoads; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) m = max(m, __float_as_uint(v[u][e]) & 0x7fffffffu);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, kWave));
  __shared__ uint32_t part[kRangeThreads / kWave];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kRangeThreads / kWave; ++w) m = max(m, part[w]);
    __hip_atomic_store(&slots[blockIdx.y * gridDim.x + blockIdx.x], m, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

// Workgroups per tensor: one per kRangeLoads loads of each thread, at most
// one per CU.
int abs_max_slots(const RangeArgs& a) {
  int64_t most = 0;
  for (int t = 0; t < a.count; ++t) most = max(most, (int64_t)a.batch * a.rows[t] * (a.dim / 4));
  const int64_t want = (most + kRangeThreads * kRangeLoads - 1) / (kRangeThreads * kRangeLoads);
  return (int)max((int64_t)1, min(want, (int64_t)kRangeSlots));
}

hipError_t launch_abs_max(const RangeArgs& a, int slots_each, uint32_t* slots, hipStream_t s) {
  bool flat = !a.add;
  for (int t = 0; t < a.count; ++t)
    flat = flat && (a.rows[t] <= 1 || a.row_stride[t] == a.dim) &&
           (a.batch <= 1 || a.batch_stride[t] == (int64_t)a.rows[t] * a.dim);
  const dim3 grid(slots_each, a.count), block(kRangeThreads);
  return flat ? launch<&abs_max_kernel<true>>(ktag("abs_max_kernel", true), grid, block, s, a, slots)
              : launch<&abs_max_kernel<false>>(ktag("abs_max_kernel", false), grid, block, s, a, slots);
}

hipError_t wait_abs_max(const uint32_t* slots, int n, hipStream_t s) {
  const volatile uint32_t* v = slots;
  const auto begin = std::chrono::steady_clock::now();
  for (int i = 0; i < n;) {
    if (v[i] != kRangeEmpty) {
      ++i;
      continue;
    }
    __builtin_ia32_pause();
    // A long queue ahead, or a stream in error: leave the wait to HIP.
    if (std::chrono::steady_clock::now() - begin > std::chrono::milliseconds(20)) {
      const hipError_t e = hipStreamSynchronize(s);
      if (e != hipSuccess) return e;
      for (int k = 0; k < n; ++k)
        if (v[k] == kRangeEmpty) return hipErrorUnknown;
      break;
    }
  }
  return hipSuccess;
}

}  // namespace neso
