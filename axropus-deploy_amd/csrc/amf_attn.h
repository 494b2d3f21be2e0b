// amf_attn.h - what the dense attention kernels share: the arguments, the
// split-partial layout and the loads of one lane's share of a K/V row (dense
// elements, or INT4_SYM codes dequantized in registers).
#pragma once

#include "amf_internal.h"
#include "amf_kernel_util.h"

namespace amf {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.4426950408889634f;

struct AttnArgs {
  const void* q;
  const void* k;
  const void* v;
  const float* mask;
  int64_t ms0, ms1, ms2, ms3;  // mask strides over (batch, q head, q row, kv token)
  void* out;
  int64_t batch;
  int32_t num_q_heads, num_kv_heads;
  int64_t q_len, kv_len;
  int32_t head_dim;
  float scale;
  // INT4_SYM K/V (split path only): k and v point at packed codes (element
  // 8 w + n of a row in nibble n of code word w), these at the fp16
  // per-channel scales [head_dim].
  const _Float16* k_scales;
  const _Float16* v_scales;
};

// Scores, maxima and the splits' m are base-2 logarithms (scaled by log2(e))
// without a mask.  With one they stay natural logarithms and their differences
// are scaled before 2^x: a mask's lowest finite value times log2(e) would be
// -inf, and a row masked with it everywhere NaN instead of its tokens' mean.
__host__ __device__ inline float score_scale(const AttnArgs& a) {
  return a.mask ? a.scale : a.scale * kLog2e;
}
__host__ __device__ inline float exp2_factor(const AttnArgs& a) { return a.mask ? kLog2e : 1.0f; }

constexpr int kPartPad = 4;            // a split partial: acc[D], m, l, 2 pad (16-byte rows)
constexpr int64_t kXcds = 8;           // XCDs of the chip, dealt workgroups round-robin

inline bool split_head_dim(int32_t D) { return D == 64 || D == 128 || D == 256; }

// INT4 = true: K and V are INT4_SYM codes, dequantized as the codec's restore
// does, (code - 8) * scale in fp32 rounded to DT (the dtype the restore would
// write and q's dtype), so the scores see the values a decompressed tensor
// holds.  (code - 8) * s is taken as fma(code, s, -8 s): the exact product
// fits fp32 (4 + 11 bits), so the single rounding of the fma is exact too.
// The nibbles go to bytes first (even elements in w & 0x0F0F0F0F, odd ones
// in (w >> 4) & 0x0F0F0F0F), so that v_cvt_f32_ubyte0..3 convert them; the
// empty asm keeps the compiler from folding that back into a bit-field
// extract per element.
template <int DT>
__device__ __forceinline__ float round_to(float y) {
  if constexpr (DT == AMF_DTYPE_BF16) {
    return (float)(__bf16)y;
  } else if constexpr (DT == AMF_DTYPE_F16) {
    keep_f32(y);
    return (float)(_Float16)y;
  } else {
    return y;
  }
}

// The 8 exact products (code - 8) * scale of one code word, before rounding.
__device__ __forceinline__ void int4_sym_vals(uint32_t w, const float (&s)[8], const float (&z)[8],
                                              float (&y)[8]) {
  uint32_t ev = w & 0x0F0F0F0Fu, od = (w >> 4) & 0x0F0F0F0Fu;
  asm("" : "+v"(ev));
  asm("" : "+v"(od));
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    y[2 * i] = __builtin_fmaf((float)((ev >> (8 * i)) & 0xFFu), s[2 * i], z[2 * i]);
    y[2 * i + 1] = __builtin_fmaf((float)((od >> (8 * i)) & 0xFFu), s[2 * i + 1], z[2 * i + 1]);
  }
}

// One lane's 8 elements of a K/V row as loaded (lane c of a row group holds
// dims 8c .. 8c + 7 of a head_dim-D row): a code word for INT4, else 16
// (bf16/fp16) or 32 (fp32) bytes.  decode() gives them as fp32; pairs()
// (bf16/fp16 only) as four DT pairs, elements 2i and 2i + 1 in word i.
template <int DT, bool INT4>
struct RawRow {  // bf16 / fp16
  u32x4 w;
  static __device__ __forceinline__ RawRow load(const void* base, int64_t r, int c, int D) {
    return RawRow{*reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(base) + r * D +
                                                  8 * c)};
  }
  __device__ __forceinline__ void decode(const float (&)[8], const float (&)[8],
                                         float (&x)[8]) const {
    unpack8<DT == AMF_DTYPE_BF16>(w, x);
  }
  __device__ __forceinline__ void pairs(const float (&)[8], const float (&)[8],
                                        uint32_t (&pr)[4]) const {
    pr[0] = w.x;
    pr[1] = w.y;
    pr[2] = w.z;
    pr[3] = w.w;
  }
};

template <>
struct RawRow<AMF_DTYPE_F32, false> {
  f32x4 lo, hi;
  static __device__ __forceinline__ RawRow load(const void* base, int64_t r, int c, int D) {
    const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(base) + r * D + 8 * c);
    return RawRow{p[0], p[1]};
  }
  __device__ __forceinline__ void decode(const float (&)[8], const float (&)[8],
                                         float (&x)[8]) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = lo[e];
      x[4 + e] = hi[e];
    }
  }
};

template <int DT>
struct RawRow<DT, true> {
  uint32_t w;
  static __device__ __forceinline__ RawRow load(const void* base, int64_t r, int c, int D) {
    return RawRow{static_cast<const uint32_t*>(base)[r * (D / 8) + c]};
  }
  __device__ __forceinline__ void decode(const float (&s)[8], const float (&z)[8],
                                         float (&x)[8]) const {
    float y[8];
    int4_sym_vals(w, s, z, y);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = round_to<DT>(y[e]);
  }
  __device__ __forceinline__ void pairs(const float (&s)[8], const float (&z)[8],
                                        uint32_t (&pr)[4]) const {
    float y[8];
    int4_sym_vals(w, s, z, y);
    // round to nearest even, as decode() and the restore do
#pragma unroll
    for (int i = 0; i < 4; ++i) pr[i] = pack2<DT == AMF_DTYPE_BF16>(y[2 * i], y[2 * i + 1]);
  }
};

// Four consecutive outputs at element i (a multiple of 4), rounded to an
// AMF_DTYPE_* output.
__device__ __forceinline__ void store4(void* out, int out_dtype, int64_t i, f32x4 x) {
  if (out_dtype == AMF_DTYPE_F32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(out) + i) = x;
  } else {
    const u32x2 w = out_dtype == AMF_DTYPE_BF16
                        ? u32x2{pack2<true>(x[0], x[1]), pack2<true>(x[2], x[3])}
                        : u32x2{pack2<false>(x[0], x[1]), pack2<false>(x[2], x[3])};
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(out) + i) = w;
  }
}

}  // namespace amf
