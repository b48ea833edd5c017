// Per-tensor scales of K and V rows (gfx950), in one launch.
//
// Semantics of PagedKVCache.prefill for "int8_per_tensor"
// (benchmarks/int8_bridge/paged_cache.py:101-102), for fp16 or bf16 rows:
//   scale = max(fp32(t(amax|x| / 127)), 1e-8)     (t = the input type; NaN stays NaN)
//
// Half of the work-groups take K, half V.  Each reduces the magnitude bits of its
// share (ordered like the values, with NaN above infinity) and leaves them as a
// partial; the last of a tensor to arrive folds the partials and writes the scale.
// The read of the rows bounds it, and below some 20 MB the arrivals, one
// device-scope atomic each on one address per tensor: hence few, large work-groups
// and a counter for each tensor.  MI355X, 2 x 4001 x 8 x 128 fp16 (16.4 MB): 7.5 us, with
// one counter for both 8.8; 65 MB 14.5 (one counter 15.9).  torch's abs, amax, division,
// conversion and clamp of the two tensors took 10 launches, 42 us on the device.
#include <algorithm>

#include "pa_device.hpp"
#include "pa_internal.hpp"

namespace pa {

namespace {

constexpr int kAmaxThreads = 512;
constexpr int kAmaxLoads = 8;   // 16-byte loads a thread keeps in flight
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

struct AmaxArgs {
  const uint16_t* x[2];     // K, V
  int64_t ts[2], hs[2];     // element strides of a token and of a head
  long long pieces;         // 16-byte pieces of one tensor
  int hkv, dg;              // kv heads, 8-dim groups of a row
  int flat[2];              // the tensor's rows are contiguous
  float* scale[2];
  uint32_t* counter;        // K's arrivals; V's kSchedQueueStride words on (another line)
  uint32_t* partials;       // K's groups, then V's
  int groups;               // per tensor
};

__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t u = (uint32_t)__shfl_xor((int)v, o, kWave);
    v = u > v ? u : v;
  }
  return v;
}

template <bool BF>
__device__ __forceinline__ float tensor_scale(uint32_t am) {
  float s;
  if constexpr (BF) {
    // one rounding to bf16; the product with fl(1/127) rounds as the quotient
    // does (a / 127 of an 8-bit significand lies farther than 2^-17 from
    // every bf16 midpoint)
    const float q = bitsf(am << 16) * (1.0f / 127.0f);
    const uint32_t b = fbits(q);
    const uint32_t r = (q != q) ? ((b >> 16) | 0x40u) : ((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
    s = bitsf(r << 16);
  } else {
    // (equal to fp16(a / 127) for every fp16 value, as in the write kernel)
    s = (float)(half_t)((float)__builtin_bit_cast(half_t, (uint16_t)am) * (1.0f / 127.0f));
  }
  return s < 1e-8f ? 1e-8f : s;   // NaN stays
}

template <bool BF>
__global__ void __launch_bounds__(kAmaxThreads) tensor_scales_kernel(AmaxArgs a) {
  __shared__ uint32_t red[kAmaxThreads / kWave];
  __shared__ int last;
  const int is_v = blockIdx.x & 1, grp = blockIdx.x >> 1;
  const uint16_t* x = a.x[is_v];
  uint32_t* const counter = a.counter + is_v * kSchedQueueStride;
  const long long stride = (long long)a.groups * kAmaxThreads;
  u16x2_t am2 = {0, 0};
  for (long long p0 = (long long)grp * kAmaxThreads + threadIdx.x; p0 < a.pieces;
       p0 += stride * kAmaxLoads) {
    uint4 v[kAmaxLoads];
#pragma unroll
    for (int k = 0; k < kAmaxLoads; ++k) {
      long long p = p0 + k * stride;
      p = p < a.pieces ? p : a.pieces - 1;   // (a piece read twice changes no maximum)
      long long at = p * 8;
      if (!a.flat[is_v]) {
        const long long row = p / a.dg;
        const long long tok = row / a.hkv;
        at = tok * a.ts[is_v] + (row - tok * a.hkv) * a.hs[is_v] + (p - row * a.dg) * 8;
      }
      v[k] = *reinterpret_cast<const uint4*>(x + at);
    }
#pragma unroll
    for (int k = 0; k < kAmaxLoads; ++k) {
      const uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        am2 = __builtin_elementwise_max(am2, __builtin_bit_cast(u16x2_t, w[i] & 0x7FFF7FFFu));
    }
  }
  const uint32_t am = wave_umax(am2[0] > am2[1] ? am2[0] : am2[1]);
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x >> 6] = am;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < kAmaxThreads / kWave; ++i) m = red[i] > m ? red[i] : m;
    // the partial is in memory (acknowledged) before the arrival is counted
    __hip_atomic_store(a.partials + is_v * kAmaxGroups + grp, m, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           (uint32_t)(a.groups - 1);
  }
  __syncthreads();
  if (!last || threadIdx.x >= kWave) return;
  uint32_t m = 0;
  for (int i = threadIdx.x; i < a.groups; i += kWave) {
    const uint32_t u = __hip_atomic_load(a.partials + is_v * kAmaxGroups + i, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    m = u > m ? u : m;
  }
  m = wave_umax(m);
  if (threadIdx.x == 0) {
    *a.scale[is_v] = tensor_scale<BF>(m);
    __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

}  // namespace

hipError_t launch_tensor_scales(const WriteLaunch& l, bool bf16, float* k_scale, float* v_scale,
                                uint32_t* counter, uint32_t* partials) {
  AmaxArgs a{};
  a.x[0] = static_cast<const uint16_t*>(l.key);
  a.x[1] = static_cast<const uint16_t*>(l.value);
  a.ts[0] = l.key_token_stride;
  a.ts[1] = l.value_token_stride;
  a.hs[0] = l.key_head_stride;
  a.hs[1] = l.value_head_stride;
  a.hkv = l.num_kv_heads;
  a.dg = l.head_dim / 8;
  a.pieces = (long long)l.num_tokens * a.hkv * a.dg;
  for (int i = 0; i < 2; ++i)
    a.flat[i] = a.hs[i] == l.head_dim && a.ts[i] == (int64_t)l.head_dim * a.hkv;
  a.scale[0] = k_scale;
  a.scale[1] = v_scale;
  a.counter = counter;
  a.partials = partials;
  const long long per_group = (long long)kAmaxThreads * kAmaxLoads;
  a.groups = (int)std::min<long long>(kAmaxGroups, (a.pieces + per_group - 1) / per_group);
  const dim3 grid(2 * a.groups);
  if (bf16) tensor_scales_kernel<true><<<grid, kAmaxThreads, 0, l.stream>>>(a);
  else tensor_scales_kernel<false><<<grid, kAmaxThreads, 0, l.stream>>>(a);
  return hipGetLastError();
}

}  // namespace pa
