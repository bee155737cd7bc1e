// The verify accept step, the greedy draft pick (argmax_rows) and the exp check kernel.
#include "sampler_device.h"
#include "launch.h"
#include "../../include/artemis_sampler.h"

using namespace as_dev;

namespace {

// spec/step.rs:347-379 over picks that all k+1 rows already made: the first pick that is a stop id
// (turn.rs:350-352) or differs from the draft after it ends the burst. One thread: k <= 15.
__global__ void accept_kernel(const uint32_t* __restrict__ picks, const uint32_t* __restrict__ status,
                              const uint32_t* __restrict__ drafts, uint32_t k,
                              const uint32_t* __restrict__ stop_ids, uint32_t n_stop,
                              uint64_t* __restrict__ rng_state, uint32_t draws_per_row,
                              uint32_t* __restrict__ result) {
  if (threadIdx.x != 0) return;
  uint32_t read = 0, flags = 0;
  for (uint32_t i = 0; i <= k; ++i) {
    if (status[i] & AS_ROW_NONFINITE) {
      flags |= 2u;
      break;
    }
    const uint32_t y = picks[i];
    read = i + 1;
    if (status[i] & AS_ROW_EXACT_PATH) flags |= 0x100u;
    bool stop = false;
    for (uint32_t j = 0; j < n_stop; ++j) stop = stop || stop_ids[j] == y;
    if (stop) {
      flags |= 1u;
      break;
    }
    if (i < k && drafts[i] != y) break;
  }
  // The stream advances by one draw per row the sampler read.
  if (draws_per_row) {
    uint64_t s[4] = {rng_state[0], rng_state[1], rng_state[2], rng_state[3]};
    for (uint32_t i = 0; i < read; ++i) rng_next(s);
    for (int j = 0; j < 4; ++j) rng_state[j] = s[j];
  }
  result[0] = read;
  result[1] = read > 0 ? read - 1 : 0;
  result[2] = read > 0 ? picks[read - 1] : AS_NO_DRAFT;
  result[3] = flags;
}

constexpr int kArgThreads = 256;
constexpr uint32_t kArgLoads = 8;  // 16-byte loads in flight per thread

// argmax_rows.comp: the largest finite value, ties to the lower index (-0 and +0 tie), NO_DRAFT for
// none; the embedding-row address of the pick. Each row is cut into `parts` slices of `len` values, a
// workgroup each (workgroup row * parts + part). A slice's best is one u64, ordered as the pick is
// (value key with -0 as +0, then the lower index; 0: no finite value). With one slice per row the
// workgroup writes the row; else it stores its best device-coherent, waits for it and counts itself in
// the row's `arrived`, and the slice that brings the count to `parts` reads the slices' bests
// (device-coherent), writes the row and clears the count for the next call.
// One workgroup's loads bound a lone row (1 MB at 10 GB/s with one 16-byte load per thread in flight):
// a row of 248,320 values and embed_rows of its pick took 98.8 us, and take 11.2 as 49 slices of 5,120.
template <bool kVec>
__global__ __launch_bounds__(kArgThreads) void argmax_kernel(const float* __restrict__ logits,
                                                             uint64_t row_stride, uint32_t n, uint32_t parts,
                                                             uint32_t len, uint64_t* best, uint32_t* arrived,
                                                             uint32_t* __restrict__ ids,
                                                             uint64_t* __restrict__ rows_out,
                                                             uint64_t embd, uint32_t row_bytes,
                                                             uint32_t slot) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  __shared__ uint64_t red[kArgThreads / kWave];
  __shared__ uint32_t last;
  const uint32_t row = blockIdx.x / parts, part = blockIdx.x % parts, tid = threadIdx.x, lane = tid & (kWave - 1);
  const uint32_t b0 = part * len, b1 = b0 + min(len, n - b0);  // parts = ceil(n / len)
  const float* src = logits + (uint64_t)row * row_stride;
  float bv = -__builtin_inff();
  uint32_t bi = kNone;
  // Each thread sees its values in index order, so a strict `>` keeps the lowest index of a tie.
  auto see = [&](float v, uint32_t i) {
    if (v > bv && v <= __FLT_MAX__) {
      bv = v;
      bi = i;
    }
  };
  uint32_t tail = b0;  // the first value the 16-byte groups leave
  if (kVec) {
    // The slice starts on a multiple of 1,024 values and the rows are 16-byte aligned.
    const uint32_t groups = (b1 - b0) / 4;
    for (uint32_t g0 = tid; g0 < groups; g0 += kArgLoads * kArgThreads) {
      f32x4 q[kArgLoads];
#pragma unroll
      for (uint32_t u = 0; u < kArgLoads; ++u) {
        const uint32_t g = g0 + u * kArgThreads;
        if (g < groups) q[u] = *reinterpret_cast<const f32x4*>(src + b0 + 4 * g);
      }
#pragma unroll
      for (uint32_t u = 0; u < kArgLoads; ++u) {
        const uint32_t g = g0 + u * kArgThreads;
        if (g < groups)
#pragma unroll
          for (int c = 0; c < 4; ++c) see(q[u][c], b0 + 4 * g + c);
      }
    }
    tail = b0 + 4 * groups;
  }
  // (In 64 bits: a slice may end within one step of 2^32.)
  for (uint64_t i0 = (uint64_t)tail + tid; i0 < b1; i0 += kArgLoads * kArgThreads) {
    float q[kArgLoads];
#pragma unroll
    for (uint32_t u = 0; u < kArgLoads; ++u) {
      const uint64_t i = i0 + u * kArgThreads;
      if (i < b1) q[u] = src[i];
    }
#pragma unroll
    for (uint32_t u = 0; u < kArgLoads; ++u) {
      const uint64_t i = i0 + u * kArgThreads;
      if (i < b1) see(q[u], (uint32_t)i);
    }
  }
  uint64_t key = wave_max_u64(bi == kNone ? 0ull : pack(total_key(bv == 0.0f ? 0.0f : bv), bi));
  if (lane == 0) red[tid / kWave] = key;
  __syncthreads();
  for (int w = 0; w < kArgThreads / kWave; ++w) key = max(key, red[w]);
  if (parts > 1) {
    uint64_t* rb = best + (uint64_t)row * parts;
    if (tid == 0) {
      __hip_atomic_store(rb + part, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const uint32_t old = __hip_atomic_fetch_add(arrived + row, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = old + 1 == parts ? 1u : 0u;
    }
    __syncthreads();
    if (!last || tid >= kWave) return;
    key = 0;
    for (uint32_t s = lane; s < parts; s += kWave)
      key = max(key, __hip_atomic_load(rb + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    key = wave_max_u64(key);
    if (tid == 0) __hip_atomic_store(arrived + row, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (tid == 0) {
    ids[slot + row] = key ? packed_id(key) : AS_NO_DRAFT;
    rows_out[slot + row] = embd + (uint64_t)(key ? packed_id(key) : 0u) * (uint64_t)row_bytes;
  }
}

__global__ void exp_kernel(const double* __restrict__ x, double* __restrict__ y, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = as_exp::exp(x[i]);
}

// The hardware 2^x (V_EXP_F32) the scan's sums are built on.
__global__ void exp2f_kernel(const float* __restrict__ x, float* __restrict__ y, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = __builtin_amdgcn_exp2f(x[i]);
}

}  // namespace

namespace as_launch {

hipError_t accept(hipStream_t stream, const uint32_t* picks, const uint32_t* status,
                  const uint32_t* drafts, uint32_t k, const uint32_t* stop_ids, uint32_t n_stop,
                  uint64_t* rng_state, uint32_t draws_per_row, uint32_t* result) {
  hipLaunchKernelGGL(accept_kernel, dim3(1), dim3(64), 0, stream, picks, status, drafts, k, stop_ids,
                     n_stop, rng_state, draws_per_row, result);
  return hipGetLastError();
}

// Slices per row: as many as make three workgroups per CU over the call's rows, of at least 4,096 values
// (greedy_kernel's least) and, rounded up, of a multiple of 1,024, so that their 16-byte groups stay aligned:
// at 248,320 values 49 of 5,120 for one row, 41 of 6,144 for 16, 3 of 82,944 for 256. From
// kArgGroups rows on a row is one workgroup's, so n_rows * parts stays under 2 * kArgGroups wherever
// the slices' bests are used. Without scratch (a captured call) every row is one workgroup's: a lone row of
// 248,320 values 31.5 us in a replayed graph (97 with one load per thread in flight), against 4.8 in slices.
hipError_t argmax_rows(hipStream_t stream, bool vec, const float* logits, uint64_t row_stride,
                       uint32_t n, uint32_t n_rows, uint64_t* best, uint32_t* arrived, uint32_t* ids,
                       uint64_t* rows_out, uint64_t embd, uint32_t row_bytes, uint32_t slot) {
  uint32_t parts = best && n_rows < kArgGroups ? (kArgGroups + n_rows - 1) / n_rows : 1u;
  parts = max(1u, min(parts, n / 4096));
  const uint64_t per = ((uint64_t)n + parts - 1) / parts;
  const uint32_t len = parts > 1 ? (uint32_t)((per + 1023) / 1024 * 1024) : n;
  if (parts > 1) parts = (uint32_t)(((uint64_t)n + len - 1) / len);
  const dim3 grid(n_rows * parts);
  hipLaunchKernelGGL(vec ? argmax_kernel<true> : argmax_kernel<false>, grid, dim3(kArgThreads), 0, stream, logits,
                     row_stride, n, parts, len, best, arrived, ids, rows_out, embd, row_bytes, slot);
  return hipGetLastError();
}

hipError_t debug_exp(hipStream_t stream, const double* x, double* y, uint32_t n) {
  hipLaunchKernelGGL(exp_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, x, y, n);
  return hipGetLastError();
}

hipError_t debug_exp2f(hipStream_t stream, const float* x, float* y, uint32_t n) {
  hipLaunchKernelGGL(exp2f_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, x, y, n);
  return hipGetLastError();
}

}  // namespace as_launch
