// The output head's matvec, with the greedy draft step fused into it.
//
// matvec (crates/kernels/shaders/matvec.glsl, matvec_{type}.comp; dispatch Kernels::matvec):
// y = W x for `rows` rows of k values of a weight type (quant.glsl's six), each output as the
// reference computes it, bit for bit: lane l of a 32-lane row group sums the row's 32-value units
// l, l + 32, ... in order from 0 (quant.glsl's lane_sum; each unit_dot adds its rounded products in
// order), and the 32 partials meet in the tree p[i] += p[i + s] for s = 16, 8, 4, 2, 1
// (tree32.glsl; twin/mod.rs:15-25). The library is built without contraction, so every product is
// rounded before its add, as the reference's `precise` arithmetic is.
//
// F32, BF16, Q8_0 and some Q6_K tables (matvec_kernel): on CDNA4 a wave of 64 lanes holds two 32-lane row
// groups (a 32-lane xor shuffle stays inside its half); each group computes two rows per step, so that two
// units' loads are in flight per lane, and a 256-thread workgroup walks 16-row steps grid-stride, with a grid that fits the
// chip in one round. x is staged once per workgroup in LDS, unit u at xs[33 u ..] (the pad of one float
// puts the 32 lanes' reads of 32 different units in 32 different banks). Weights are read once, straight
// from HBM; the compiler merges a unit's 2-byte reads into 16-byte loads (the target allows unaligned
// global access, and Q8_0's 34-byte and Q6_K's 210-byte blocks are only 2-byte aligned). The K-quants take
// quad_kernel, below, but for the Q6_K tables that row_threads names.
//
// head_argmax: the same rows with argmax_rows' epilogue (crates/kernels/shaders/argmax_rows.comp):
// the largest finite output, ties to the lower index (-0 and +0 tie), computed as the outputs are
// produced: each workgroup keeps its best as one u64 key, and a one-workgroup kernel takes the
// largest key and writes ids[slot] and rows_out[slot] = embd + id * row_bytes (AS_NO_DRAFT and row
// 0's address when no output is finite). The logits need not be written or read again.
#include <type_traits>

#include "sampler_device.h"
#include "launch.h"
#include "../../include/artemis_sampler.h"

using namespace as_dev;

namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kRowsPerStep = 2 * (kThreads / 32);  // 8 groups of 32 lanes, two rows each
constexpr uint32_t kFinalThreads = 1024;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float half_u16(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }
// 32 bytes at a 2-byte aligned address as 8 words (two 2-byte reads each; the compiler merges the
// reads into wide loads), and byte l of them.
__device__ __forceinline__ void load32(const uint16_t* p, uint32_t (&q)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = (uint32_t)p[2 * i] | ((uint32_t)p[2 * i + 1] << 16);
}
__device__ __forceinline__ uint32_t byte_of(const uint32_t (&q)[8], uint32_t l) {
  return (q[l >> 2] >> (8 * (l & 3))) & 0xFFu;
}

// Four 6-bit quants q = lo + 16 hi at once, one a byte (lo: the low nibbles of l's bytes, hi: the low pairs of
// h's), each byte holding q - 32 as a signed byte: lo in its low nibble and hi - 2 (mod 16) in its high one,
// which v_perm_b32 looks up per byte (byte hi of 0x1000F0E0: 0xE0, 0xF0, 0x00, 0x10). Each value is then one
// sign-extending byte-to-float conversion; float(q - 32) is exactly the reference's float(q) - 32.
__device__ __forceinline__ uint32_t q6_bytes(uint32_t l, uint32_t h) {
  return (l & 0x0F0F0F0Fu) | __builtin_amdgcn_perm(0u, 0x1000F0E0u, h & 0x03030303u);
}

// quant.glsl unit_dot (twin/matvec.rs:21-84) for unit u of the row; x: the unit's 32 inputs in LDS.
template <uint32_t kType>
__device__ __forceinline__ float unit_dot(const uint8_t* __restrict__ row, uint32_t u, const float* x) {
  if constexpr (kType == AS_WTYPE_F32) {
    const uint32_t* w = reinterpret_cast<const uint32_t*>(row + 128u * u);
    uint32_t wv[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) wv[i] = w[i];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) s = s + __uint_as_float(wv[i]) * x[i];
    return s;
  } else if constexpr (kType == AS_WTYPE_BF16) {
    const uint32_t* w = reinterpret_cast<const uint32_t*>(row + 64u * u);
    uint32_t wv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) wv[i] = w[i];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s = s + __uint_as_float(wv[i] << 16) * x[2 * i];
      s = s + __uint_as_float(wv[i] & 0xFFFF0000u) * x[2 * i + 1];
    }
    return s;
  } else if constexpr (kType == AS_WTYPE_Q8_0) {
    const uint16_t* b = reinterpret_cast<const uint16_t*>(row + 34u * u);
    uint32_t q[8];
    load32(b + 1, q);
    const float d = half_u16(b[0]);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) s = s + (float)(int8_t)byte_of(q, i) * x[i];
    return d * s;
  } else {
    // Q6_K: unit j of a block is half n = j / 4, quarter m = j % 4.
    static_assert(kType == AS_WTYPE_Q6_K, "Q4_K and Q5_K take quad_kernel");
    const uint16_t* b = reinterpret_cast<const uint16_t*>(row + 210u * (u / 8));
    const uint32_t j = u % 8, n = j / 4, m = j % 4;
    uint32_t ql[8], qh[8];
    load32(b + 32 * n + 16 * (m & 1), ql);
    load32(b + 64 + 16 * n, qh);
    const uint32_t scs = b[96 + 4 * n + m], dh = b[104];
    float sa = 0.0f, sb = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t s4 = q6_bytes(ql[i] >> (4 * (m >> 1)), qh[i] >> (2 * m));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float prod = (float)(int8_t)(uint8_t)(s4 >> (8 * e)) * x[4 * i + e];
        if (i < 4) sa = sa + prod;
        else sb = sb + prod;
      }
    }
    const float pa = (float)(int8_t)(scs & 0xFFu) * sa, pb = (float)(int8_t)(scs >> 8) * sb;
    return half_u16(dh) * (pa + pb);
  }
}

// argmax_rows' order as one u64: finite values by value (-0 as +0), then the lower index; 0 for a
// non-finite value (below every finite key).
__device__ __forceinline__ uint64_t draft_key(float v, uint32_t i) {
  return is_finite_bits(v) ? pack(total_key(v == 0.0f ? 0.0f : v), i) : 0ull;
}

// Lane l's partials of two rows a and b: units l, l + 32, ... added in order from 0 (quant.glsl
// lane_sum). The two rows' dot products of a unit are independent and read the same inputs, so their
// loads are in flight together.
template <uint32_t kType>
__device__ __forceinline__ float lane_sum2(const uint8_t* wr, uint32_t lane, uint32_t units, const float* xs,
                                           float* acc_b, const uint8_t* wr_b, bool has_b) {
  float a = 0.0f, b = 0.0f;
  for (uint32_t u = lane; u < units; u += 32) {
    const float da = unit_dot<kType>(wr, u, xs + u * 33);
    const float db = has_b ? unit_dot<kType>(wr_b, u, xs + u * 33) : 0.0f;
    a = a + da;
    b = b + db;
  }
  *acc_b = b;
  return a;
}

// tree32.glsl over a 32-lane group (lanes past a short row's units hold +0.0).
__device__ __forceinline__ float tree32(float acc) {
  acc = acc + __shfl_xor(acc, 16, 32);
  acc = acc + __shfl_xor(acc, 8, 32);
  acc = acc + __shfl_xor(acc, 4, 32);
  acc = acc + __shfl_xor(acc, 2, 32);
  acc = acc + __shfl_xor(acc, 1, 32);
  return acc;
}

// Each 32-lane group computes two rows per step (a workgroup 16), rows 2s and 2s + 1 of the step.
template <uint32_t kType, bool kArgmax>
__global__ __launch_bounds__(kThreads) void matvec_kernel(const uint8_t* __restrict__ w, uint64_t row_bytes,
                                                          uint32_t rows, uint32_t k, const float* __restrict__ x,
                                                          float* __restrict__ y, uint64_t* __restrict__ partials) {
  extern __shared__ float xs[];  // k / 32 units of 33 floats
  __shared__ uint64_t red[kThreads / kWave];
  const uint32_t tid = threadIdx.x, units = k / 32;
  for (uint32_t i = tid; i < k; i += kThreads) xs[(i / 32) * 33 + (i % 32)] = x[i];
  __syncthreads();
  const uint32_t lane = tid & 31, slot = tid / 32;
  const uint32_t n_steps = (rows + kRowsPerStep - 1) / kRowsPerStep;
  uint64_t best = 0;
  for (uint32_t g = blockIdx.x; g < n_steps; g += gridDim.x) {
    const uint32_t r0 = g * kRowsPerStep + 2 * slot, r1 = r0 + 1;
    float acc0 = 0.0f, acc1 = 0.0f;
    if (r0 < rows)
      acc0 = lane_sum2<kType>(w + (uint64_t)r0 * row_bytes, lane, units, xs, &acc1, w + (uint64_t)r1 * row_bytes,
                              r1 < rows);
    acc0 = tree32(acc0);
    acc1 = tree32(acc1);
    if (lane == 0) {
      if (r0 < rows) {
        if (y) y[r0] = acc0;
        if (kArgmax) best = max(best, draft_key(acc0, r0));
      }
      if (r1 < rows) {
        if (y) y[r1] = acc1;
        if (kArgmax) best = max(best, draft_key(acc1, r1));
      }
    }
  }
  if constexpr (kArgmax) {
    best = wave_max_u64(best);
    if ((tid & (kWave - 1)) == 0) red[tid / kWave] = best;
    __syncthreads();
    if (tid == 0) {
      for (uint32_t i = 1; i < kThreads / kWave; ++i) best = max(best, red[i]);
      partials[blockIdx.x] = best;
    }
  }
}

// ---- the K-quants: four units per thread ------------------------------------------------------------
//
// A K-quant block's bytes are shared between units: Q6_K's 16 bytes of ql serve two units and its qh
// four; Q4_K's and Q5_K's 32 bytes of nibbles two, Q5_K's high bits eight. With a unit per lane each lane
// loaded its unit's 64 bytes for the 26 (Q6_K) that are its own, 2-byte aligned 16-byte pieces all, and
// the kernel waited on its loads' issue (128 us for 70 us of VALU work at the 248,320 x 2,048 Q6_K head).
// Here a thread takes a quad, units 4q .. 4q + 3 (half a block), and loads each byte once; kT threads (4, 8
// or 16, inside one DPP row) take a row's quads q = t, t + kT, .... The four units' sums are independent
// chains, so their dependent adds overlap, and every shift of the unpacking is a constant.
//
// The order stays the reference's: unit u belongs to lane u % 32 of its 32 partials and a lane adds its
// units in order. Thread t < 8 keeps partials 4t .. 4t + 3; with 8 threads the quads it takes are theirs, in
// order. With 16, per step of 16 quads, it adds its own quad (units 4t .. of the step's first 32) and then
// thread t + 8's (the second 32), moved by DPP. A quad past the row's end adds +0.0, which changes nothing
// (a partial starts from +0.0 and is never -0.0).
//
// At 248,320 x 2,048, by events (us; a unit per lane before): Q6_K 127.7 to 86.8, 4.8 TB/s of weights and, by the
// counters, 5.0 VALU instructions per weight (65 us at full issue); Q5_K 127.7 to 72.3, 5.2 per weight (68 us);
// Q4_K 111.6 to 54.2, 3.8 per weight (49 us).
constexpr uint32_t kQuadStride = 132;  // LDS floats per quad of x (see quad_kernel)
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_u __attribute__((ext_vector_type(2), aligned(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int kShift>
__device__ __forceinline__ float row_shl(float x) {  // lane i of a 16-lane row gets lane i + kShift's (0 past the row)
  return __builtin_bit_cast(float, dpp_u32<0x100 + kShift>(__builtin_bit_cast(uint32_t, x)));
}

// Byte e of a word of quants 0 .. 15, two at a time: read as FP8 (E4M3) a byte q < 16 is q 2^-9 exactly (the
// subnormals and the first binade are one even scale), which the conversion's scale of 2^9 makes float(q).
// One instruction per two weights.
__device__ __forceinline__ f32x2 nibbles_lo(uint32_t w) { return __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, 512.0f, false); }
__device__ __forceinline__ f32x2 nibbles_hi(uint32_t w) { return __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, 512.0f, true); }

// Four values through an empty asm: the selects that follow would otherwise have each unit's whole sum sunk
// into a branch of its own, with every input held in registers until then.
__device__ __forceinline__ void hold(float (&v)[4]) { __asm__ volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])); }

// A row's quad as loaded, and its four units' dot products (quant.glsl unit_dot, twin/matvec.rs:21-84).
template <uint32_t kType, bool kWords>
struct Quad;

// kWords: the table is 4-byte aligned. Every second block (210 bytes) then starts 2 bytes into a word,
// where a 16-byte load costs the vector memory unit more: the words that hold the quad are loaded whole and
// moved together two bytes at a time (v_alignbyte_b32), one instruction per four low nibbles' word. A block
// that starts mid-word reads the 2 bytes before it, the block's before; the first one does not.
// (248,320 x 2,048: 98 us with the loads as they fall, 88 with words.)
template <bool kWords>
struct Quad<AS_WTYPE_Q6_K, kWords> {
  static constexpr uint32_t kBlock = 210;
  u32x4_u ql[4], qh[2];  // the half block's 64 bytes of low nibbles and 32 of high pairs
  uint32_t ql_end, qh_end, by;  // kWords: the words after them, and how far into its first word each starts
  u32x2_u sc;            // its 8 scales
  uint16_t d;
  float sa[4], sb[4];
  typedef uint32_t u32x4_w __attribute__((ext_vector_type(4), aligned(4)));
  using Load = typename std::conditional<kWords, u32x4_w, u32x4_u>::type;
  // Words i of the nibbles and of the pairs.
  __device__ __forceinline__ uint32_t low(int i) const {
    if constexpr (!kWords) return ql[i / 4][i % 4];
    else return __builtin_amdgcn_alignbyte(i < 15 ? ql[(i + 1) / 4][(i + 1) % 4] : ql_end, ql[i / 4][i % 4], by);
  }
  __device__ __forceinline__ uint32_t high(int i) const {
    if constexpr (!kWords) return qh[i / 4][i % 4];
    else return __builtin_amdgcn_alignbyte(i < 7 ? qh[(i + 1) / 4][(i + 1) % 4] : qh_end, qh[i / 4][i % 4], by);
  }
  __device__ __forceinline__ void load(const uint8_t* row, uint32_t q) {
    const uint8_t* blk = row + kBlock * (q / 2);
    const uint32_t n = q % 2;
    const uint8_t* at = blk;
    if constexpr (kWords) {
      by = (uint32_t)(uintptr_t)blk & 2u;
      at = blk - by;
      ql_end = *reinterpret_cast<const uint32_t*>(at + 64 * n + 64);
      qh_end = *reinterpret_cast<const uint32_t*>(at + 128 + 32 * n + 32);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) ql[i] = *reinterpret_cast<const Load*>(at + 64 * n + 16 * i);
#pragma unroll
    for (int i = 0; i < 2; ++i) qh[i] = *reinterpret_cast<const Load*>(at + 128 + 32 * n + 16 * i);
    sc = *reinterpret_cast<const u32x2_u*>(blk + 192 + 8 * n);
    d = *reinterpret_cast<const uint16_t*>(blk + 208);
#pragma unroll
    for (int m = 0; m < 4; ++m) sa[m] = sb[m] = 0.0f;
  }
  // Values 4i .. 4i + 3 of the four units.
  __device__ __forceinline__ void step(int i, const f32x4 (&x)[4]) {
    const uint32_t h = high(i), l0 = low(i), l1 = low(8 + i);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const uint32_t s4 = q6_bytes((m & 1 ? l1 : l0) >> (4 * (m >> 1)), h >> (2 * m));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float prod = (float)(int8_t)(uint8_t)(s4 >> (8 * e)) * x[m][e];
        if (i < 4) sa[m] = sa[m] + prod;
        else sb[m] = sb[m] + prod;
      }
    }
  }
  __device__ __forceinline__ void hold_sums() {
    hold(sa);
    hold(sb);
  }
  __device__ __forceinline__ float dot(int m, const float*) const {
    const uint32_t s = sc[m / 2] >> (16 * (m & 1));
    const float pa = (float)(int8_t)(s & 0xFFu) * sa[m], pb = (float)(int8_t)((s >> 8) & 0xFFu) * sb[m];
    return half_u16(d) * (pa + pb);
  }
};

template <bool kQ5>
struct QuadK {
  static constexpr uint32_t kBlock = kQ5 ? 176 : 144;
  u32x4_u hd;              // d, dmin, 12 bytes of scales and mins
  u32x4_u qs[4];           // the half block's 64 bytes of nibbles
  u32x4_u qh[kQ5 ? 2 : 1]; // Q5_K: the block's 32 bytes of high bits
  uint32_t half;           // which half of the block
  float sq[4];
  __device__ __forceinline__ void load(const uint8_t* row, uint32_t q) {
    const uint8_t* blk = row + kBlock * (q / 2);
    half = q % 2;
    hd = *reinterpret_cast<const u32x4_u*>(blk);
    if constexpr (kQ5) {
#pragma unroll
      for (int i = 0; i < 2; ++i) qh[i] = *reinterpret_cast<const u32x4_u*>(blk + 16 + 16 * i);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) qs[i] = *reinterpret_cast<const u32x4_u*>(blk + (kQ5 ? 48 : 16) + 64 * half + 16 * i);
#pragma unroll
    for (int m = 0; m < 4; ++m) sq[m] = 0.0f;
  }
  // Values 4i .. 4i + 3 of the four units, four quants at once (quant.glsl kq_dot): unit m's nibbles at
  // bit 4 (m & 1) of word i of 32-byte run m / 2 and, for Q5_K, bit 4 half + m of the high bytes at bit 4;
  // float(q) is exact, so the products are the reference's.
  __device__ __forceinline__ void step(int i, const f32x4 (&x)[4]) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      uint32_t q4 = (qs[2 * (m / 2) + i / 4][i % 4] >> (4 * (m & 1))) & 0x0F0F0F0Fu;
      float f[4];
      if constexpr (kQ5) {
        q4 |= ((qh[i / 4][i % 4] >> (4 * half + m)) & 0x01010101u) << 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = (float)((q4 >> (8 * e)) & 0xFFu);
      } else {
        const f32x2 a = nibbles_lo(q4), b = nibbles_hi(q4);
        f[0] = a[0];
        f[1] = a[1];
        f[2] = b[0];
        f[3] = b[1];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) sq[m] = sq[m] + f[e] * x[m][e];
    }
  }
  __device__ __forceinline__ void hold_sums() { hold(sq); }
  // sx: the sums of the four units' inputs, in order.
  __device__ __forceinline__ float dot(int m, const float* sx) const {
    // ggml's get_scale_min_k4 over the 12 bytes at offset 4 (quant.glsl scale_min_k4), unit j = 4 half + m.
    const uint32_t a = hd[1] >> (8 * m), b = hd[2] >> (8 * m), c = hd[3] >> (8 * m);
    const uint32_t sc = half ? (c & 0xFu) | ((a >> 2) & 0x30u) : a & 63u;
    const uint32_t mn = half ? ((c >> 4) & 0xFu) | ((b >> 2) & 0x30u) : b & 63u;
    const float p = (half_u16(hd[0] & 0xFFFFu) * (float)sc) * sq[m];
    const float r = (half_u16(hd[0] >> 16) * (float)mn) * sx[m];
    return p - r;
  }
};
template <bool kWords>
struct Quad<AS_WTYPE_Q4_K, kWords> : QuadK<false> {};
template <bool kWords>
struct Quad<AS_WTYPE_Q5_K, kWords> : QuadK<true> {};

// x lies in LDS with quad q's 128 inputs at xs[kQuadStride q ..]: 16 threads reading the same place of 16
// consecutive quads by 16 bytes each hit 16 different groups of four banks. After them, per quad, the
// sums of its four units' inputs (Q4_K and Q5_K subtract their minimum times it: the same for every row,
// so each unit is summed once per workgroup rather than once per row).
template <uint32_t kType, bool kWords, uint32_t kT, bool kArgmax>
__global__ __launch_bounds__(kThreads) void quad_kernel(const uint8_t* __restrict__ w, uint64_t row_bytes,
                                                        uint32_t rows, uint32_t k, const float* __restrict__ x,
                                                        float* __restrict__ y, uint64_t* __restrict__ partials) {
  extern __shared__ float xs[];
  __shared__ uint64_t red[kThreads / kWave];
  constexpr bool kSums = kType != AS_WTYPE_Q6_K;
  const uint32_t tid = threadIdx.x, quads = k / 128;
  for (uint32_t i = tid; i < k; i += kThreads) xs[(i / 128) * kQuadStride + i % 128] = x[i];
  __syncthreads();
  float* sums = xs + quads * kQuadStride;
  if constexpr (kSums) {
    for (uint32_t u = tid; u < 4 * quads; u += kThreads) {
      const float* xu = xs + (u / 4) * kQuadStride + 32 * (u % 4);
      float s = 0.0f;
      for (int i = 0; i < 32; ++i) s = s + xu[i];
      sums[u] = s;
    }
    __syncthreads();
  }
  const uint32_t t = tid % kT, group = tid / kT;
  constexpr uint32_t kStep = kThreads / kT;
  const uint32_t n_steps = (rows + kStep - 1) / kStep;
  uint64_t best = 0;
  for (uint32_t g = blockIdx.x; g < n_steps; g += gridDim.x) {
    const uint32_t r = g * kStep + group;
    const uint8_t* wr = w + (uint64_t)min(r, rows - 1) * row_bytes;
    float p[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t q0 = 0; q0 < quads; q0 += kT) {
      const bool mine = q0 + t < quads;
      const uint32_t q = mine ? q0 + t : quads - 1;
      Quad<kType, kWords> qd;
      qd.load(wr, q);
      const float* xq = xs + q * kQuadStride;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // (Each step's LDS reads and conversions stay in it: hoisted, they would take the registers of
        // one wave in eight.)
        __builtin_amdgcn_sched_barrier(0);
        f32x4 xv[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) xv[m] = *reinterpret_cast<const f32x4*>(xq + 32 * m + 4 * i);
        qd.step(i, xv);
      }
      qd.hold_sums();
      float d[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) d[m] = qd.dot(m, sums + 4 * q);
      hold(d);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        d[m] = mine ? d[m] : 0.0f;
        p[m] = p[m] + d[m];
        if (kT == 16) p[m] = p[m] + row_shl<8>(d[m]);
      }
    }
    // tree32.glsl over partials 4t + m, t < 8 (kT 4: the others are +0.0): strides 16, 8 and 4 across
    // threads, 2 and 1 within one.
    if (kT >= 8)
#pragma unroll
      for (int m = 0; m < 4; ++m) p[m] = p[m] + row_shl<4>(p[m]);
#pragma unroll
    for (int m = 0; m < 4; ++m) p[m] = p[m] + row_shl<2>(p[m]);
#pragma unroll
    for (int m = 0; m < 4; ++m) p[m] = p[m] + row_shl<1>(p[m]);
    const float v = (p[0] + p[2]) + (p[1] + p[3]);
    if (t == 0 && r < rows) {
      if (y) y[r] = v;
      if (kArgmax) best = max(best, draft_key(v, r));
    }
  }
  if constexpr (kArgmax) {
    best = wave_max_u64(best);
    if ((tid & (kWave - 1)) == 0) red[tid / kWave] = best;
    __syncthreads();
    if (tid == 0) {
      for (uint32_t i = 1; i < kThreads / kWave; ++i) best = max(best, red[i]);
      partials[blockIdx.x] = best;
    }
  }
}

__global__ __launch_bounds__(kFinalThreads) void draft_final_kernel(const uint64_t* __restrict__ partials,
                                                                    uint32_t n_partials, uint32_t* __restrict__ ids,
                                                                    uint64_t* __restrict__ rows_out, uint64_t embd,
                                                                    uint32_t row_bytes, uint32_t slot) {
  __shared__ uint64_t red[kFinalThreads / kWave];
  uint64_t best = 0;
  for (uint32_t i = threadIdx.x; i < n_partials; i += kFinalThreads) best = max(best, partials[i]);
  best = wave_max_u64(best);
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t i = 1; i < kFinalThreads / kWave; ++i) best = max(best, red[i]);
    const uint32_t id = best ? packed_id(best) : AS_NO_DRAFT;
    ids[slot] = id;
    rows_out[slot] = embd + (uint64_t)(best ? id : 0u) * (uint64_t)row_bytes;
  }
}

// Workgroups for `rows`: as many as the chip holds at once (the kernel's occupancy at this LDS size
// times the CUs), so every workgroup runs in the first round, and no more than there are steps.
template <typename K>
uint32_t grid_for(K kernel, size_t lds, uint32_t rows, uint32_t step) {
  int dev = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kThreads, lds) != hipSuccess || per_cu < 1 || cus < 1)
    per_cu = 1, cus = 256;
  uint64_t g = (uint64_t)per_cu * (uint64_t)cus;
  const uint32_t n_steps = (rows + step - 1) / step;
  if (g > as_launch::kMatvecGroups) g = as_launch::kMatvecGroups;
  return (uint32_t)(g < n_steps ? g : n_steps);
}

// A K-quant row's threads: 4, 8 or 16 of quad_kernel's, or 32, a unit per lane (matvec_kernel; Q6_K only).
//  - Up to 4 quads, 4 threads hold the row whole (its first 16 partials, the others +0.0): 16 would leave 12
//    idle (Q4_K, 120,000 x 512: 9.7 us against 30.9, and 26.9 for a unit per lane). Up to 8, 8 threads do, in
//    one step (248,320 x 1,024: Q5_K 32.0 us against 57.1 with 16, Q6_K 37.0 against 67.4 and 49.3 for a unit
//    per lane).
//  - Longer rows take the quads in steps of 8 or 16 threads. 16 leave half a step or more idle when the last
//    step holds 8 quads or fewer; 8 do not, but need 16,384 rows for two waves per SIMD, without which each
//    step's loads are waited for (2,560 values, 65,536 and 8,192 rows, 8 against 16 threads: Q5_K 26.6 and
//    31.4 us, 8.3 and 7.6). Elsewhere 16 measured best for Q5_K and Q6_K (238,095 x 2,048: Q6_K 82.7 against
//    93.0), and 8 for Q4_K, whose weights cost the fewest instructions beside the tree that half as many
//    threads share (248,320 x 2,048: 52.8 against 57.8).
//  - Q6_K between the two, where 16 threads idle and rows are few: a unit per lane, which fills its 32 lanes
//    (2,560 values: 6,144 rows 7.6 us, against 7.9 with 8 threads and 8.0 with 16; 20,480 rows 14.4 against 15.5 and
//    15.5; 32,768 rows 20.9 against 20.1 with 8).
uint32_t row_threads(uint32_t wtype, uint32_t quads, uint32_t rows) {
  if (quads <= 4) return 4;
  if (quads <= 8) return 8;
  const bool half_idle = quads % 16 != 0 && quads % 16 <= 8;
  if (wtype == AS_WTYPE_Q6_K) return !half_idle ? 16 : (rows < 32768 ? 32 : 8);
  return rows >= 16384 && (half_idle || wtype == AS_WTYPE_Q4_K) ? 8 : 16;
}

template <bool kArgmax>
hipError_t launch(hipStream_t stream, const void* w, uint32_t wtype, uint64_t row_bytes, uint32_t rows, uint32_t k,
                  const float* x, float* y, uint64_t* partials, uint32_t* groups) {
  const size_t lds = (size_t)(k / 32) * 33 * sizeof(float);
  const size_t qlds = (size_t)(k / 128) * (kQuadStride + 4) * sizeof(float);
  const uint8_t* wb = static_cast<const uint8_t*>(w);
  const dim3 block(kThreads);
  const uint32_t threads = row_threads(wtype, k / 128, rows);
  switch (wtype) {
#define AS_MV_RUN(T)                                                                                                 \
  {                                                                                                                  \
    *groups = grid_for(matvec_kernel<T, kArgmax>, lds, rows, kRowsPerStep);                                          \
    hipLaunchKernelGGL((matvec_kernel<T, kArgmax>), dim3(*groups), block, lds, stream, wb, row_bytes, rows, k, x, y, \
                       partials);                                                                                    \
    break;                                                                                                           \
  }
#define AS_MV(T) case T: AS_MV_RUN(T)
    AS_MV(AS_WTYPE_F32)
    AS_MV(AS_WTYPE_BF16)
    AS_MV(AS_WTYPE_Q8_0)
#define AS_QUAD_T(T, W, N)                                                                                           \
  {                                                                                                                  \
    *groups = grid_for(quad_kernel<T, W, N, kArgmax>, qlds, rows, kThreads / N);                                     \
    hipLaunchKernelGGL((quad_kernel<T, W, N, kArgmax>), dim3(*groups), block, qlds, stream, wb, row_bytes, rows, k,  \
                       x, y, partials);                                                                              \
    break;                                                                                                           \
  }
#define AS_QUAD(T, W)                                                                                                \
  {                                                                                                                  \
    if (threads == 4) AS_QUAD_T(T, W, 4)                                                                             \
    if (threads == 8) AS_QUAD_T(T, W, 8)                                                                             \
    AS_QUAD_T(T, W, 16)                                                                                              \
  }
    case AS_WTYPE_Q4_K: AS_QUAD(AS_WTYPE_Q4_K, false)
    case AS_WTYPE_Q5_K: AS_QUAD(AS_WTYPE_Q5_K, false)
    case AS_WTYPE_Q6_K:
      if (threads == 32) AS_MV_RUN(AS_WTYPE_Q6_K)
      if ((uintptr_t)w % 4 == 0) AS_QUAD(AS_WTYPE_Q6_K, true)
      AS_QUAD(AS_WTYPE_Q6_K, false)
#undef AS_QUAD
#undef AS_QUAD_T
#undef AS_MV
#undef AS_MV_RUN
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

namespace as_launch {

hipError_t matvec(hipStream_t stream, const void* w, uint32_t wtype, uint64_t row_bytes, uint32_t rows, uint32_t k,
                  const float* x, float* y) {
  uint32_t groups = 0;
  return launch<false>(stream, w, wtype, row_bytes, rows, k, x, y, nullptr, &groups);
}

hipError_t head_argmax(hipStream_t stream, const void* w, uint32_t wtype, uint64_t row_bytes, uint32_t rows,
                       uint32_t k, const float* x, float* y, uint64_t* partials, uint32_t* ids, uint64_t* rows_out,
                       uint64_t embd, uint32_t embd_row_bytes, uint32_t slot) {
  uint32_t groups = 0;
  hipError_t e = launch<true>(stream, w, wtype, row_bytes, rows, k, x, y, partials, &groups);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(draft_final_kernel, dim3(1), dim3(kFinalThreads), 0, stream, partials, groups, ids, rows_out,
                     embd, embd_row_bytes, slot);
  return hipGetLastError();
}

}  // namespace as_launch
