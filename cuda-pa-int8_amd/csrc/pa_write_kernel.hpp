// Paged-cache writes (gfx950): per-token INT8 quantize, per-tensor INT8
// quantize, and fp16 placement, one kernel.
//
// Semantics (bit-exact with the reference's torch code):
//   quantize_per_token, tests/paged_decode_attn.py:106-112
//     amax  = max_d |x_d|                 (in the input type, exact)
//     scale = fp32(t(max(amax, t(1e-8)) / 127))   (t = fp16 or bf16, the input
//                                                  type; the division rounded once)
//     q_d   = int8(clamp(rne(fp32(x_d) / scale), -127, 127)), NaN -> 0
//   placement, tests/paged_decode_attn.py:85-99,190-197 and
//   benchmarks/int8_bridge/paged_cache.py:116-130,145-154
//     k_cache[blk, h, :, off, :] = q.view(D/8, 8)
//     v_cache[blk, h, :, off]    = q
//     scales[blk, h, off]        = scale,   with slot = blk * block_size + off.
//   per-tensor mode (PagedKVCache "int8_per_tensor",
//   benchmarks/int8_bridge/paged_cache.py:99-106,140-142): the caller passes
//   one fp32 scale for all of K and one for all of V (device pointers), and
//     q_d = int8(clamp(rne(fp32(x_d) / scale), -127, 127)), scale stored per slot.
//   fp16 mode: the rows themselves, no scales.
//
// Work.  A window is 16 consecutive input tokens.  A wave reads the slots around
// its window and finds, with scalar bit operations on wave ballots, the
// *runs*: 16 tokens that fill one aligned 16-slot cell.  At most one run starts
// inside a window (at any of its 16 tokens), and the wave that owns the start
// writes the whole run: a batch of prompts of any lengths, or of chunks that
// continue sequences at any position, is written in whole cells whatever the
// position of its tokens in the input.  The window's *loose* tokens, which
// belong to no run (the ends of a sequence, decode appends, scattered slots), are
// stored one by one.  (The form for few rows takes a window as it is.)
//
// What bounds it: HBM, mixed reads and writes; small launches, latency.  Many
// rows: one wave per (window, head), K then V, both loads out together; the
// hardware replaces finished waves, which balances the windows with loose
// tokens, and 7-8 waves per SIMD keep enough loads in flight (a resident grid
// that walked the items with two rows prefetched took 87 VGPRs, 5 waves, and ran 68
// us where this form runs 61).  Plain input loads: a row's 128-byte lines are
// read half by one instruction and half by the next, and non-temporal
// lines can be gone in between (72 against 68 us).  MI355X, against the kernel that
// took whole cells only where a window's first token sat on one: 48 ragged bf16
// prompts (47,601 tokens x 8 heads, 296 MB) INT8 108 -> 61 us; 32 fp16 chunks of 200-1024
// tokens x 8 heads 62 -> 37 us; 131,072 aligned tokens x 2 heads INT8 44.0 -> 41.6 us
// (4.9 TB/s), fp16 53.9 -> 52.5 (5.1 TB/s); 32,768 x 8 in blocks of 64 84 -> 47 us.
//
// Lane l holds 8 dims (one 16-byte load) of one token per step: dim groups
// (l >> 4) + 4j of token lane_token(l & 15).  K leaves as it came, 8 dims per
// lane.  V is transposed in registers: two quad exchanges and one row
// rotation by 8 leave lane l with 8 consecutive tokens of one dim, and the 8
// lanes that share a dim group with the 8 dims of that group; a store
// instruction of a run therefore covers whole 128-byte lines of V at block size
// 16, as it does of K, and no LDS is used.  Tokens outside runs are stored
// element by element (write_loose).
//
// Quantizing multiplies by the reciprocal of the scale; an element whose
// product lies too close to a rounding tie (or is not finite) is redone with
// the IEEE division, so every byte equals the reference's.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "pa_device.hpp"
#include "pa_internal.hpp"

namespace pa {

typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

// The fast path multiplies by r, the hardware reciprocal of s (within 1 ulp
// of 1/s), instead of dividing.  With |x / s| < 128:
//   |fl(x * r) - x / s| <= 128 * (2^-23 + 2^-24) ~ 2.3e-5   (r, then the product)
//   |fl(x / s) - x / s| <= 2^-18 ~ 3.8e-6                    (the reference's quotient)
// so a product farther than 2.7e-5 from every half-integer rounds to the same
// integer as the IEEE quotient the reference computes.  The guard keeps a margin.
constexpr float kTieGuard = 4.0e-5f;
constexpr float kRoundMagic = 12582912.0f;   // 1.5 * 2^23: y + magic rounds y to an integer (RNE)
// fp16(a / 127) == fp16(fl(a * fl(1/127))) for every fp16 value a and for the
// clamp value 1e-8: a / 127 is never an fp16 rounding midpoint and stays more
// than 2^-18 (relative) away from one, beyond the 2^-23 error of the product
// (checked exhaustively on the CPU).
constexpr float kInv127 = 1.0f / 127.0f;

// The two elements of a 32-bit word of fp16 (BF false) or bf16 (BF true)
// input, widened to fp32 (exactly).
template <bool BF>
__device__ __forceinline__ void widen2(uint32_t w, float& lo, float& hi) {
  if constexpr (BF) {
    lo = __builtin_bit_cast(float, w << 16);
    hi = __builtin_bit_cast(float, w & 0xFFFF0000u);
  } else {
    const half2_t h = __builtin_bit_cast(half2_t, w);
    lo = (float)h.x;
    hi = (float)h.y;
  }
}

// fp32 -> bf16 -> fp32, round to nearest even; a NaN stays a (quiet) NaN.
__device__ __forceinline__ float round_bf16(float f) {
  const uint32_t b = __builtin_bit_cast(uint32_t, f);
  const uint32_t r = (f != f) ? ((b >> 16) | 0x40u) : ((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
  return __builtin_bit_cast(float, r << 16);
}

// Exact path: rne(x / s) with IEEE division, clamped to [-127, 127], NaN -> 0.
__device__ __forceinline__ uint32_t quant_exact_byte(float x, float s) {
  float r = __builtin_rintf(x / s);
  r = (r != r) ? 0.f : fminf(fmaxf(r, -127.f), 127.f);
  return (uint32_t)((int)r) & 0xFFu;
}

// Quantizes the 8 fp16 values of one 16-B group to 8 bytes with the
// reciprocal.  `slow` is set when some element's product lies within
// kTieGuard of a half-integer: the fast byte is then not provably the
// reference's and the caller redoes the group exactly.  With a normal fp16
// scale, |x / s| <= 127 * (1 + 2^-11) < 127.5 for every element of the row, so
// no range check is needed, and the inputs are finite (a NaN or inf in the row
// makes the scale non-normal, which takes the exact path): the largest
// distance to an integer over the group decides with one comparison.
template <bool BF>
__device__ __forceinline__ uint2 quant_group_fast(uint4 xv, float r, bool& slow) {
  const uint32_t wv[4] = {xv.x, xv.y, xv.z, xv.w};
  uint32_t bytes[8];
  float dmax = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float xs[2];
    widen2<BF>(wv[k], xs[0], xs[1]);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float y = xs[e] * r;
      dmax = fmaxf(dmax, __builtin_fabsf(y - __builtin_rintf(y)));
      bytes[2 * k + e] = __builtin_bit_cast(uint32_t, y + kRoundMagic);   // low byte = rne(y) mod 256
    }
  }
  slow = slow || !(dmax < 0.5f - kTieGuard);
  uint2 out;
  out.x = __builtin_amdgcn_perm(__builtin_amdgcn_perm(bytes[3], bytes[2], 0x0c0c0400u),
                                __builtin_amdgcn_perm(bytes[1], bytes[0], 0x0c0c0400u), 0x05040100u);
  out.y = __builtin_amdgcn_perm(__builtin_amdgcn_perm(bytes[7], bytes[6], 0x0c0c0400u),
                                __builtin_amdgcn_perm(bytes[5], bytes[4], 0x0c0c0400u), 0x05040100u);
  return out;
}

// The same with a scale given by the caller (per-tensor mode), where the
// quotient can exceed the int8 range: a product of magnitude >= 127 gives
// +-127 (the IEEE quotient then exceeds 126.5, the reciprocal being a normal
// number, so it rounds to >= 127 and clamps there); the rest lies below 127
// and rounds as above.
template <bool BF>
__device__ __forceinline__ uint2 quant_group_fast_sat(uint4 xv, float r, bool& slow) {
  const uint32_t wv[4] = {xv.x, xv.y, xv.z, xv.w};
  uint32_t bytes[8];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float xs[2];
    widen2<BF>(wv[k], xs[0], xs[1]);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float y = xs[e] * r;
      const bool sat = __builtin_fabsf(y) >= 127.f;
      slow = slow || (!sat && !(__builtin_fabsf(y - __builtin_rintf(y)) < 0.5f - kTieGuard));
      bytes[2 * k + e] = sat ? (y > 0.f ? 0x7Fu : 0x81u)
                             : __builtin_bit_cast(uint32_t, y + kRoundMagic);
    }
  }
  uint2 out;
  out.x = __builtin_amdgcn_perm(__builtin_amdgcn_perm(bytes[3], bytes[2], 0x0c0c0400u),
                                __builtin_amdgcn_perm(bytes[1], bytes[0], 0x0c0c0400u), 0x05040100u);
  out.y = __builtin_amdgcn_perm(__builtin_amdgcn_perm(bytes[7], bytes[6], 0x0c0c0400u),
                                __builtin_amdgcn_perm(bytes[5], bytes[4], 0x0c0c0400u), 0x05040100u);
  return out;
}

// The exact path for one 16-B group.
template <bool BF>
__device__ __forceinline__ uint2 quant_group_exact(uint4 xv, float s) {
  const uint32_t wv[4] = {xv.x, xv.y, xv.z, xv.w};
  uint32_t b[8];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float lo, hi;
    widen2<BF>(wv[k], lo, hi);
    b[2 * k] = quant_exact_byte(lo, s);
    b[2 * k + 1] = quant_exact_byte(hi, s);
  }
  return make_uint2(b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24),
                    b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24));
}

// Cache policy of a run's stores (buffer store aux bits).  With blocks of 16
// tokens a store instruction covers whole 128-byte lines and nt, the streaming
// policy, is the faster one; with larger blocks a V line is completed by the
// windows that follow, and plain stores let the L2 put it together (MI355X,
// 32768 tokens x 8 heads, INT8, blocks of 64: plain 52 us, nt 70 us; 131072 tokens x 2
// heads, blocks of 16: plain 43.7 us, nt 41.9 us; ragged fp16, blocks of 16: 33.0 / 26.2 us).
constexpr int kStorePlain = 0, kStoreStream = 2;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)bytes, 0x00020000);
}

// What a write stores: the rows themselves (fp16), or INT8 with each token's own
// scale or with one given scale per tensor.
enum class WriteMode { kF16, kTokenScale, kGivenScale };

constexpr int kWriteWaves = 4;   // waves (windows) of a work-group

struct WriteArgs {
  const uint16_t* key;
  const uint16_t* value;
  int64_t kts, khs, vts, vhs;   // element strides of a token and of a head
  const int64_t* slots;         // num_tokens entries
  int num_tokens;               // tokens with a slot
  int num_rows;                 // of them, tokens with an input row (>= 1); the rest are zeros
  int hkv;
  void* kc;
  void* vc;
  float* ksc;                   // INT8 modes
  float* vsc;
  const float* k_scale_in;      // kGivenScale
  const float* v_scale_in;
  int64_t pool;                 // slots of the cache
  int bs, bs_log2;
  int wpb_log2;                 // log2 of the windows per cache block (many rows)
};

// Token of a lane of a 16-lane row: bits 2 and 3 change places, so that the
// row rotation by 8 pairs the lanes of neighbouring token quads (its own inverse).
__device__ __forceinline__ int lane_token(int r) {
  return (r & 3) | ((r >> 1) & 4) | ((r << 1) & 8);
}

typedef uint32_t wu2_t __attribute__((ext_vector_type(2)));
typedef uint32_t wu4_t __attribute__((ext_vector_type(4)));
template <int POLICY>
__device__ __forceinline__ void store_tile(__amdgpu_buffer_rsrc_t tile, int at, uint2 g) {
  __builtin_amdgcn_raw_buffer_store_b64((wu2_t){g.x, g.y}, tile, at, 0, POLICY);
}
template <int POLICY>
__device__ __forceinline__ void store_tile(__amdgpu_buffer_rsrc_t tile, int at, uint4 g) {
  __builtin_amdgcn_raw_buffer_store_b128((wu4_t){g.x, g.y, g.z, g.w}, tile, at, 0, POLICY);
}

constexpr int kRowRor8 = 0x128;   // lane i <- (i + 8) % 16 of its row

// Lane selectors of the V transpose (bytes or halves), fixed per lane.
struct TransposeSel {
  uint32_t s1, s2;   // v_perm selectors of the two quad exchanges
  bool hi2, hi8;     // lane bits 1 and 3
};
template <bool HALVES>
__device__ __forceinline__ TransposeSel transpose_sel(int lane) {
  TransposeSel t;
  const bool odd = lane & 1;
  t.hi2 = lane & 2;
  t.hi8 = lane & 8;
  // 2 x 2 exchange of neighbouring lanes: bytes (0, 2 | 1, 3) or halves (0 | 1)
  t.s1 = HALVES ? (odd ? 0x03020706u : 0x05040100u) : (odd ? 0x03070105u : 0x06020400u);
  t.s2 = t.hi2 ? 0x03020706u : 0x05040100u;   // halves between lanes 2 apart
  return t;
}

// 8 dims x 1 token per lane -> 8 tokens x 1 dim, INT8: in, the 8 bytes of the
// lane's token (dims 8o .. 8o + 7); out, dim 8o + 4 * (lane bit 3) + (lane & 3)
// of tokens 8 * (lane bit 2) .. + 7.
__device__ __forceinline__ uint2 transpose_v(uint2 q, const TransposeSel& t) {
  uint32_t w[2] = {q.x, q.y};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    w[i] = __builtin_amdgcn_perm(dpp_mov_u<kQuadXor1>(w[i]), w[i], t.s1);
    w[i] = __builtin_amdgcn_perm(dpp_mov_u<kQuadXor2>(w[i]), w[i], t.s2);
  }
  const uint32_t recv = dpp_mov_u<kRowRor8>(t.hi8 ? w[0] : w[1]);
  return t.hi8 ? make_uint2(recv, w[1]) : make_uint2(w[0], recv);
}

// The same for 2-byte elements.
__device__ __forceinline__ uint4 transpose_v(uint4 x, const TransposeSel& t) {
  uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w[i] = __builtin_amdgcn_perm(dpp_mov_u<kQuadXor1>(w[i]), w[i], t.s1);
  uint2 p[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t recv = dpp_mov_u<kQuadXor2>(t.hi2 ? w[2 * i] : w[2 * i + 1]);
    p[i] = t.hi2 ? make_uint2(recv, w[2 * i + 1]) : make_uint2(w[2 * i], recv);
  }
  const uint32_t r0 = dpp_mov_u<kRowRor8>(t.hi8 ? p[0].x : p[1].x);
  const uint32_t r1 = dpp_mov_u<kRowRor8>(t.hi8 ? p[0].y : p[1].y);
  return t.hi8 ? make_uint4(r0, r1, p[1].x, p[1].y) : make_uint4(p[0].x, p[0].y, r0, r1);
}

__device__ __forceinline__ int64_t readlane64(int64_t v, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const int hi = __builtin_amdgcn_readlane((int)(v >> 32), lane);
  return ((int64_t)hi << 32) | lo;
}

// One token row of a lane: JQ 16-byte groups as loaded.
template <int D>
struct WriteRow {
  static constexpr int DG = D / 8;          // 8-dim groups of a row
  // 16-byte groups per lane; with head_dim % 32 != 0 the last j is a group only
  // for lane quarters with qq + 4j < DG (the others load the row's last
  // group, in bounds, and store nothing).
  static constexpr int JQ = (DG + 3) / 4;
  uint4 x[JQ];
};

// The scale of a lane's token and what its quantization needs.
struct RowScale {
  float s = 0.f, rcp = 0.f;
  bool normal = true;   // the reciprocal path is provably exact away from ties
};

template <int D, WriteMode MODE, bool BF, bool PROBE>
__device__ __forceinline__ RowScale row_scale(const WriteRow<D>& r, const float* given) {
  RowScale q;
  if constexpr (PROBE) {
    q.s = 1.f;
  } else if constexpr (MODE == WriteMode::kGivenScale) {
    q.s = given[0];
    // A caller's scale takes the IEEE reciprocal; the saturating fast path
    // needs it normal and finite.
    q.rcp = 1.0f / q.s;
    q.normal = q.rcp >= 1.17549435e-38f && q.rcp <= 3.40282347e+38f;
  } else if constexpr (MODE == WriteMode::kTokenScale) {
    // amax over the token's D values as fp16 / bf16 magnitude bits (ordered
    // like the values; a NaN input gives NaN bits above +inf, so the scale
    // becomes NaN as in torch).  A padding group repeats the row's last one.
    u16x2_t am2 = {0, 0};
#pragma unroll
    for (int j = 0; j < WriteRow<D>::JQ; ++j) {
      const uint32_t wv[4] = {r.x[j].x, r.x[j].y, r.x[j].z, r.x[j].w};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        am2 = __builtin_elementwise_max(am2, __builtin_bit_cast(u16x2_t, wv[k] & 0x7FFF7FFFu));
    }
    uint32_t am = am2[0] > am2[1] ? am2[0] : am2[1];
    am = rows_umax(am);
    if constexpr (BF) {
      // bf16: amax and clamp_min(bf16(1e-8)) are exact in fp32; the quotient
      // is the IEEE one rounded to bf16 (one rounding, as torch's).
      const float amax = __builtin_bit_cast(float, am << 16);
      const float lo = __builtin_bit_cast(float, 0x322C0000u);   // bf16(1e-8), RNE
      const float v = (amax < lo) ? lo : amax;             // clamp_min, NaN-preserving
      q.s = round_bf16(v / 127.f);
      // bf16 keeps fp32's exponent range: only NaN / inf leave the fast path
      // (a normal bf16 scale keeps |x / s| <= 127 (1 + 2^-8) < 127.5).
      q.normal = q.s >= 1.17549435e-38f && q.s <= 3.38953139e+38f;
    } else {
      const float amax = (float)__builtin_bit_cast(half_t, (uint16_t)am);
      const float v = (amax < 1e-8f) ? 1e-8f : amax;      // clamp_min, NaN-preserving
      q.s = (float)(half_t)(v * kInv127);                 // == fp16(v / 127), RNE
      // A scale that is not a normal fp16 number (zero, subnormal, NaN, inf)
      // sends the token's elements to the exact path.
      q.normal = q.s >= 6.103515625e-05f && q.s <= 65504.0f;
    }
    // Per-token scales are normal fp16 / bf16 numbers on the fast path, so the
    // hardware reciprocal is finite and within the guard's error budget.
    q.rcp = __builtin_amdgcn_rcpf(q.s);
  }
  return q;
}

// The stored form of one 8-dim group: 8 INT8 bytes or 8 fp16 values.
template <WriteMode MODE>
using WriteGroup = typename std::conditional<MODE == WriteMode::kF16, uint4, uint2>::type;

template <WriteMode MODE, bool BF, bool PROBE>
__device__ __forceinline__ WriteGroup<MODE> row_group(uint4 x, const RowScale& q) {
  if constexpr (MODE == WriteMode::kF16) {
    return x;
  } else if constexpr (PROBE) {
    return make_uint2(__builtin_amdgcn_perm(x.y, x.x, 0x07050301u),
                      __builtin_amdgcn_perm(x.w, x.z, 0x07050301u));
  } else {
    bool slow = !q.normal;
    uint2 g = MODE == WriteMode::kGivenScale ? quant_group_fast_sat<BF>(x, q.rcp, slow)
                                             : quant_group_fast<BF>(x, q.rcp, slow);
    if (__builtin_amdgcn_ballot_w64(slow) != 0) {
      if (slow) g = quant_group_exact<BF>(x, q.s);   // rare: the reference's division
    }
    return g;
  }
}

// Per-lane constants of a write kernel.
template <bool I8>
struct WriteLane {
  int lane, qq, i;   // lane quarter, token of the sixteen
  int tg, vd;        // V after the transpose: tokens tg .. tg + 7 of dim 8o + vd
  TransposeSel ts;
  __device__ __forceinline__ WriteLane() {
    lane = threadIdx.x & 63;
    qq = lane >> 4;
    i = lane_token(lane & 15);
    tg = 2 * (lane & 4);
    vd = ((lane >> 1) & 4) + (lane & 3);
    ts = transpose_sel<!I8>(lane);
  }
};

// The slots around the window at t0: lane b holds those of tokens t0 - 16 + b and
// t0 - 15 + b (b < 48).
struct WindowSlots {
  int64_t s0, s1;
  __device__ __forceinline__ void load(const WriteArgs& a, int t0, int lane) {
    const int tl = t0 - 16 + lane;
    s0 = a.slots[min(max(tl, 0), a.num_tokens - 1)];
    s1 = a.slots[min(max(tl + 1, 0), a.num_tokens - 1)];
  }
};

// What a window holds (uniform over the wave).
struct Window {
  bool run;            // a run starts in the window,
  int start;           // at token t0 + start,
  int64_t slot;        // at this slot
  uint32_t loose;      // bit k: token t0 + k has a slot and belongs to no run
};

__device__ __forceinline__ Window find_runs(const WriteArgs& a, int t0, int lane,
                                            const WindowSlots& ws) {
  const int T = a.num_tokens;
  const int tl = t0 - 16 + lane;
  const bool ok0 = lane < 48 && tl >= 0 && tl < T && ws.s0 >= 0 && ws.s0 < a.pool;
  const uint64_t ok = __builtin_amdgcn_ballot_w64(ok0);
  const uint64_t al = __builtin_amdgcn_ballot_w64(ok0 && (ws.s0 & 15) == 0 && a.bs >= 16);
  const uint64_t nx = __builtin_amdgcn_ballot_w64(ok0 && tl + 1 < T && ws.s1 == ws.s0 + 1);
  uint64_t f = nx & (nx >> 1);
  f &= f >> 2;
  f &= f >> 4;
  f &= f >> 7;      // 15 successors in a row
  f &= al;          // bit b: a run starts at token t0 - 16 + b
  uint64_t cov = f | (f << 1);
  cov |= cov << 2;
  cov |= cov << 4;
  cov |= cov << 8;  // the runs' tokens
  const uint32_t own = (uint32_t)(f >> 16) & 0xFFFFu;
  Window w;
  w.run = own != 0;
  w.start = own != 0 ? __builtin_ctz(own) : 0;
  w.slot = own != 0 ? readlane64(ws.s0, 16 + w.start) : 0;
  w.loose = (uint32_t)((ok & ~cov) >> 16) & 0xFFFFu;
  return w;
}

// The K (V) input row of head h for the tokens tb + i.
template <int D>
__device__ __forceinline__ void load_row(const WriteArgs& a, bool v, int h, int tb, int i, int qq,
                                         WriteRow<D>& r) {
  const int64_t tok = min(tb + i, a.num_rows - 1);
  const uint16_t* src = v ? a.value + tok * a.vts + (int64_t)h * a.vhs
                          : a.key + tok * a.kts + (int64_t)h * a.khs;
#pragma unroll
  for (int j = 0; j < WriteRow<D>::JQ; ++j) {
    const int o = qq + 4 * j < WriteRow<D>::DG ? qq + 4 * j : WriteRow<D>::DG - 1;
    r.x[j] = *reinterpret_cast<const uint4*>(src + o * 8);
  }
}

// Writes one row of the run at `slot`, whose tokens are tb + i.
template <int D, WriteMode MODE, bool BF, bool PROBE>
__device__ __forceinline__ void write_run(const WriteArgs& a,
                                          const WriteLane<MODE != WriteMode::kF16>& ln, bool v,
                                          int h, int tb, int64_t slot, const WriteRow<D>& r) {
  constexpr bool I8 = MODE != WriteMode::kF16;
  constexpr int ESZ = I8 ? 1 : 2;
  const int bs = a.bs;
  const int64_t bh = (slot >> a.bs_log2) * a.hkv + h;
  const int off = (int)(slot & (bs - 1));
  const bool pad = tb + ln.i >= a.num_rows;
  const RowScale q = row_scale<D, MODE, BF, PROBE>(r, v ? a.v_scale_in : a.k_scale_in);
  const uint32_t tile_bytes = (uint32_t)(D * bs * ESZ);
  const auto tile =
      tile_rsrc(static_cast<uint8_t*>(v ? a.vc : a.kc) + (size_t)bh * tile_bytes, tile_bytes);
  auto at_v = [&](int o) { return ((8 * o + ln.vd) * bs + off + ln.tg) * ESZ; };
#pragma unroll
  for (int j = 0; j < WriteRow<D>::JQ; ++j) {
    const int o = ln.qq + 4 * j;           // dim group: dims 8o .. 8o + 7
    if (o >= WriteRow<D>::DG) continue;    // padding group (whole 16-lane rows): nothing to write
    WriteGroup<MODE> g = row_group<MODE, BF, PROBE>(r.x[j], q);
    if (pad) g = WriteGroup<MODE>{};
    if (!v) store_tile<kStoreStream>(tile, (o * bs + off + ln.i) * 8 * ESZ, g);
    else if (bs == 16) store_tile<kStoreStream>(tile, at_v(o), transpose_v(g, ln.ts));
    else store_tile<kStorePlain>(tile, at_v(o), transpose_v(g, ln.ts));
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (I8) {
    if (ln.qq == 0) (v ? a.vsc : a.ksc)[bh * bs + off + ln.i] = pad ? 0.f : q.s;
  }
}

// Writes one row of the window's loose tokens (t0 + k for the bits k of `loose`),
// each at its own slot; sl: the slot of token t0 + i.  V goes out element by element: from the
// transposed registers, 8 dims of a token per store instruction and 8 lanes, or, where most of the
// tokens are neighbours in the cache (`together`), as loaded, 16 tokens of a dim (MI355X, INT8,
// 8 chunks of 256 x 8 heads at slot 8: 7.1 / 6.8 us at block size 16, 10.9 / 6.8 at 64, fp16 9.4 / 7.1
// and 12.9 / 6.6; 256 appends fp16 5.0 / 7.2).
template <int D, WriteMode MODE, bool BF, bool PROBE>
__device__ __forceinline__ void write_loose(const WriteArgs& a,
                                            const WriteLane<MODE != WriteMode::kF16>& ln, bool v,
                                            int h, int t0, uint32_t loose, int64_t sl,
                                            const WriteRow<D>& r, bool together) {
  constexpr bool I8 = MODE != WriteMode::kF16;
  constexpr int ESZ = I8 ? 1 : 2;
  constexpr int DG = WriteRow<D>::DG, JQ = WriteRow<D>::JQ;
  using Group = WriteGroup<MODE>;
  const int bs = a.bs;
  const bool mine = (loose >> ln.i) & 1;
  const bool pad = t0 + ln.i >= a.num_rows;
  const int64_t bh = (mine ? sl >> a.bs_log2 : 0) * a.hkv + h;
  const int off = mine ? (int)(sl & (bs - 1)) : 0;
  const RowScale q = row_scale<D, MODE, BF, PROBE>(r, v ? a.v_scale_in : a.k_scale_in);
  Group g[JQ];
#pragma unroll
  for (int j = 0; j < JQ; ++j) {
    g[j] = row_group<MODE, BF, PROBE>(r.x[j], q);
    if (pad) g[j] = Group{};
  }
  if (!v) {
    uint8_t* const dst = static_cast<uint8_t*>(a.kc) + (bh * DG * bs + off) * 8 * ESZ;
    if (mine) {
#pragma unroll
      for (int j = 0; j < JQ; ++j)
        if (ln.qq + 4 * j < DG)
          *reinterpret_cast<Group*>(dst + (size_t)((ln.qq + 4 * j) * bs * 8 * ESZ)) = g[j];
    }
  } else if (together) {
    if (mine) {
      uint8_t* const dst =
          static_cast<uint8_t*>(a.vc) + ((bh * D + 8 * ln.qq) * bs + off) * (int64_t)ESZ;
#pragma unroll
      for (int j = 0; j < JQ; ++j) {
        if (ln.qq + 4 * j >= DG) continue;
        uint32_t d[sizeof(Group) / 4];
        __builtin_memcpy(d, &g[j], sizeof(Group));
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          uint8_t* const e = dst + (size_t)((32 * j + k) * bs * ESZ);
          if constexpr (I8) *e = (uint8_t)(d[k / 4] >> (8 * (k & 3)));
          else *reinterpret_cast<uint16_t*>(e) = (uint16_t)(d[k / 2] >> (16 * (k & 1)));
        }
      }
    }
  } else {
    const int64_t col = bh * D * bs + off;   // the token's column of its V tile
#pragma unroll
    for (int j = 0; j < JQ; ++j) g[j] = transpose_v(g[j], ln.ts);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      // token tg + k's column, from a lane that holds the token
      const int src = lane_token(ln.tg + k);
      const int64_t c = (int64_t)(uint32_t)__shfl((int)(uint32_t)col, src, kWave) |
                        ((int64_t)__shfl((int)(col >> 32), src, kWave) << 32);
      if ((loose >> (ln.tg + k)) & 1) {
        uint8_t* const dst =
            static_cast<uint8_t*>(a.vc) + (c + (int64_t)(8 * ln.qq + ln.vd) * bs) * ESZ;
#pragma unroll
        for (int j = 0; j < JQ; ++j) {
          if (ln.qq + 4 * j >= DG) continue;
          uint32_t d[sizeof(Group) / 4];
          __builtin_memcpy(d, &g[j], sizeof(Group));
          uint8_t* const e = dst + (size_t)(32 * j * bs * ESZ);
          if constexpr (I8) *e = (uint8_t)(d[k / 4] >> (8 * (k & 3)));
          else *reinterpret_cast<uint16_t*>(e) = (uint16_t)(d[k / 2] >> (16 * (k & 1)));
        }
      }
    }
  }
  if constexpr (I8) {
    if (ln.qq == 0 && mine) (v ? a.vsc : a.ksc)[bh * bs + off] = pad ? 0.f : q.s;
  }
}

// The form for many rows: a wave for each window and kv head, K then V (both rows'
// loads go out together).  The windows of a cache block come first, then the
// heads: the waves of a work-group write neighbouring rows.
// BF: INT8 modes only, the inputs are bf16 (bit patterns) instead of fp16.
// PROBE (the benchmark's write-stream probe, not a write op): the same work,
// loads and stores, with the quantization replaced by the high byte of each
// input element and the scale by 1, so that its time is the memory system's
// for exactly this kernel's address stream.
template <int D, WriteMode MODE, bool BF, bool PROBE = false>
__global__ void __launch_bounds__(kWriteWaves * kWave) paged_write_kernel(WriteArgs a) {
  static_assert(D % 8 == 0, "head_dim must be a multiple of 8");
  static_assert(MODE != WriteMode::kF16 || !BF, "the fp16 mode moves fp16 rows");
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long group = (long long)blockIdx.y * gridDim.x + blockIdx.x;
  const long long item = group * kWriteWaves + w;
  const long long rest = item >> a.wpb_log2;
  const int blk = (int)(rest / a.hkv);
  const int h = (int)(rest - (long long)blk * a.hkv);
  const int t0 = ((blk << a.wpb_log2) + (int)(item & ((1 << a.wpb_log2) - 1))) * 16;
  if (t0 >= a.num_tokens) return;
  const WriteLane<MODE != WriteMode::kF16> ln;
  WindowSlots ws;
  ws.load(a, t0, ln.lane);
  const Window win = find_runs(a, t0, ln.lane, ws);
  if (win.run) {
    WriteRow<D> rk, rv;
    load_row<D>(a, false, h, t0 + win.start, ln.i, ln.qq, rk);
    load_row<D>(a, true, h, t0 + win.start, ln.i, ln.qq, rv);
    __builtin_amdgcn_sched_barrier(0);
    write_run<D, MODE, BF, PROBE>(a, ln, false, h, t0 + win.start, win.slot, rk);
    write_run<D, MODE, BF, PROBE>(a, ln, true, h, t0 + win.start, win.slot, rv);
  }
  if (win.loose != 0) {
    const int64_t sl = a.slots[min(t0 + ln.i, a.num_tokens - 1)];
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
      WriteRow<D> r;
      load_row<D>(a, part != 0, h, t0, ln.i, ln.qq, r);
      write_loose<D, MODE, BF, PROBE>(a, ln, part != 0, h, t0, win.loose, sl, r, false);
    }
  }
}

// The form for few rows (decode appends, short prompts and chunks), which are bound by
// latency: one wave for each window, head, K or V.  The row is loaded together with the
// slots, at the window's own tokens, and nothing waits for a second load: a window whose 16
// tokens fill one cell is written as a run, all others token by token.  (Searching runs as the
// form for many rows does, a run that starts inside its window had its row loaded again once
// the slots were known, beside idle waves for the kind of token a window has none of.)
// MI355X, with that search -> this, us: INT8 23 chunks of 32-42 tokens x 8 heads at odd
// positions 5.9 -> 4.8, one of 601 5.6 -> 4.4 (blocks of 64 5.6 -> 4.2); 3 prompts of 1500-2000 x 1
// head 6.1 -> 4.65; fp16 23 chunks, blocks of 64, 6.2 -> 3.8; 8 chunks of 192-256 x 8 heads INT8
// 8.2 -> 6.8, fp16 6.6 -> 7.1 (7.25 before the search).
template <int D, WriteMode MODE, bool BF, bool PROBE = false>
__global__ void __launch_bounds__(kWriteWaves * kWave) paged_write_small_kernel(WriteArgs a) {
  const int item = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int win_no = item / (2 * a.hkv), sub = item - win_no * 2 * a.hkv;
  const int t0 = win_no * 16, h = sub >> 1;
  const bool v = sub & 1;
  if (t0 >= a.num_tokens) return;
  const WriteLane<MODE != WriteMode::kF16> ln;
  const int tok = t0 + ln.i;
  const bool in = tok < a.num_tokens;
  int64_t sl = a.slots[in ? tok : a.num_tokens - 1];
  WriteRow<D> r;
  load_row<D>(a, v, h, t0, ln.i, ln.qq, r);
  const bool ok = in && sl >= 0 && sl < a.pool;
  const int64_t slot = readlane64(sl, 0);   // token t0's (lane 0 holds it)
  const bool run = a.bs >= 16 && (slot & 15) == 0 &&
                   __builtin_amdgcn_ballot_w64(!ok || sl != slot + ln.i) == 0;
  if (run) {
    write_run<D, MODE, BF, PROBE>(a, ln, v, h, t0, slot, r);
  } else {
    // bit k: token t0 + k, which lane lane_token(k) of every 16 holds
    const uint32_t held = (uint32_t)__builtin_amdgcn_ballot_w64(ok) & 0xFFFFu;
    const uint32_t loose = (held & 0xF00Fu) | ((held & 0x0F00u) >> 4) | ((held & 0x00F0u) << 4);
    // neighbours of the window's first or last token in the cache
    const int64_t last = readlane64(sl, 15);
    const bool near = ok && (sl == slot + ln.i || sl == last - (15 - ln.i));
    const bool together = __popcll(__builtin_amdgcn_ballot_w64(near)) >= 32;
    if (loose != 0) write_loose<D, MODE, BF, PROBE>(a, ln, v, h, t0, loose, sl, r, together);
  }
}

// Where the small form ends (its waves: two per window and head) and up to where it runs in
// one-wave work-groups (which spread over more CUs).  MI355X, time of the small form over the
// large one's, geometric mean of prompts and chunks x 8 heads, INT8 (bf16 rows and one given
// scale alike) / fp16, by waves: 1700-2100 0.81 / 0.98, 2600-3100 0.77 / 0.94, 3100-3700 0.86 /
// 1.01, 3700-4200 0.95 / 1.08 at head_dim 128; 2100-2600 0.83 / 0.97, 2600-3100 0.77 / 1.03, 3100-3700
// 0.95 / 1.09, 3700-4200 1.08 / 1.26 at 256.  Work-groups of one wave against four: 300-370 waves
// INT8 0.94, fp16 0.84; 512 0.97; 704 0.94, 0.92; 750-980 of one head 1.05, 1.10.
template <int D, WriteMode MODE>
constexpr int kSmallWaves = MODE == WriteMode::kF16 ? (D > 128 ? 2048 : 3072)
                                                    : (D > 128 ? 3072 : 4096);
constexpr int kSmallSpreadWaves = 704;

template <int D, WriteMode MODE, bool BF, bool PROBE = false>
hipError_t launch_write(const WriteLaunch& l) {
  WriteArgs a{};
  a.key = static_cast<const uint16_t*>(l.key);
  a.value = static_cast<const uint16_t*>(l.value);
  a.kts = l.key_token_stride;
  a.khs = l.key_head_stride;
  a.vts = l.value_token_stride;
  a.vhs = l.value_head_stride;
  a.slots = l.slot_mapping;
  a.num_tokens = l.num_tokens + l.pad_tokens;
  a.num_rows = l.num_tokens;
  a.hkv = l.num_kv_heads;
  a.kc = l.k_cache;
  a.vc = l.v_cache;
  a.ksc = l.k_scales;
  a.vsc = l.v_scales;
  a.k_scale_in = l.k_scale_in;
  a.v_scale_in = l.v_scale_in;
  a.bs = l.block_size;
  a.bs_log2 = __builtin_ctz((unsigned)l.block_size);
  a.pool = (int64_t)l.num_blocks * l.block_size;
  const long long windows = (a.num_tokens + 15ll) / 16;
  const long long small = 2 * windows * l.num_kv_heads;
  if (small <= kSmallWaves<D, MODE>) {
    const int nw = small <= kSmallSpreadWaves ? 1 : kWriteWaves;
    paged_write_small_kernel<D, MODE, BF, PROBE>
        <<<((int)small + nw - 1) / nw, nw * kWave, 0, l.stream>>>(a);
    return hipGetLastError();
  }
  a.wpb_log2 = std::max(0, a.bs_log2 - 4);
  const long long blocks = (windows + (1 << a.wpb_log2) - 1) >> a.wpb_log2;
  const long long items = (blocks << a.wpb_log2) * l.num_kv_heads;
  const long long groups = (items + kWriteWaves - 1) / kWriteWaves;
  // (a dispatch counts its work-items per dimension in 32 bits)
  const long long gx = std::min<long long>(groups, 1 << 22);
  const dim3 grid((unsigned)gx, (unsigned)((groups + gx - 1) / gx));
  paged_write_kernel<D, MODE, BF, PROBE><<<grid, kWriteWaves * kWave, 0, l.stream>>>(a);
  return hipGetLastError();
}

}  // namespace pa
