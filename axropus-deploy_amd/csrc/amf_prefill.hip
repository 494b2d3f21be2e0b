// amf_prefill.hip - dense attention of many query rows (chunked prefill,
// verification of drafted tokens) on MFMA tiles: the q_len > 1 form of
// amf_dense_attn and of the masked / head_dim 64 and 256 forms of
// amf_int4_sym_dense_attn, for bf16 and fp16.
//
// The query rows of one (batch, KV head) - its GQA group's heads times q_len
// - are the columns of 32x32x16 tiles, so each K/V tile staged in LDS serves
// 32 rows per wave.  The scores are formed transposed, S^T = K Q^T: a lane
// then holds one query row (column lane % 32) with 16 tokens of a 32-token
// tile, the softmax statistics of a row are per-lane scalars (one exchange
// with lane ^ 32 for the maximum), and the weights are already in the
// B-operand layout of O^T = V^T P^T, whose k slots take the tokens in the
// order the scores leave them.  V^T comes out of LDS through the transposing
// read (ds_read_b64_tr_b16).
//
// Precision.  The bf16 / fp16 products of Q and K are exact and summed in
// fp32, as the one-row kernel's v_dot2 does.  The softmax weights are fp32
// and enter the PV tiles as three bf16 terms, whose sum is exactly the weight;
// an fp16 V enters as two, which hold its 11 bits exactly as well.  (fp16
// terms would lose the weights below 2^-14 of the row's largest, and two bf16
// terms, a tenth faster at 32 / 8 heads, 512 rows, 4096 tokens, are 16 bits.)
// Accumulators, maxima and sums are fp32.
#include <algorithm>
#include <type_traits>

#include "amf_attn.h"
#include "amf_prefill.h"

namespace {

using namespace amf;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef s16x4 __attribute__((address_space(3))) lds_s16x4;

template <int DT>
__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
  if constexpr (DT == AMF_DTYPE_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// Tokens of a staged tile: 64, or 32 where 64 rows would take too much LDS
// (head_dim 256) or too many registers in flight per lane (one wave).
constexpr int tile_tokens(int D, int NW) { return D == 256 || NW == 1 ? 32 : 64; }

// LDS row strides in bytes.  K rows are read as 16-byte vectors of 32
// consecutive rows: 16 more than the row moves each by 4 banks.  V rows are
// read by the transposing read, 4 rows of 64 bytes per half wave: 64 more
// than the row puts them 16 banks apart.
constexpr int k_stride(int D) { return 2 * D + 16; }
constexpr int v_stride(int D) { return 2 * D + 64; }

// bf16 terms of a softmax weight.
constexpr int kTerms = 3;

// The terms of the weights p0 and p1 (low and high half of each word).  A
// positive weight has only positive terms, a zero one only zeros: inf in V
// then gives inf under a positive weight (mixed signs or a zero term would
// make it NaN) and NaN under a zero one, as the product with the weight itself
// does.  Each term is the top half of the bit pattern below the remainder's,
// so the next remainder is positive and exact and the third fits 8 bits.
__device__ __forceinline__ void weight_split(float p0, float p1, uint32_t (&w)[kTerms]) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t a = __builtin_elementwise_sub_sat(f2u(p0), 1u) & 0xFFFF0000u;
    const uint32_t b = __builtin_elementwise_sub_sat(f2u(p1), 1u) & 0xFFFF0000u;
    w[k] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    p0 -= u2f(a);
    p1 -= u2f(b);
  }
  w[2] = __builtin_amdgcn_perm(f2u(p1), f2u(p0), 0x07060302u);
}

// A pair of fp16 V values as two bf16 pairs, hi + lo: the top 8 bits of each
// value's 11 and the rest, below 2^8.  The clamp only meets the NaN of an
// infinite value's remainder and makes it -256: hi alone is then infinite.
__device__ __forceinline__ void v_split(uint32_t w, uint32_t& hi, uint32_t& lo) {
  const uint32_t a = f2u(half_lo<false>(w)), b = f2u(half_hi<false>(w));
  hi = __builtin_amdgcn_perm(b, a, 0x07060302u);
  const float ra = __builtin_amdgcn_fmed3f(u2f(a) - u2f(a & 0xFFFF0000u), -256.0f, 256.0f);
  const float rb = __builtin_amdgcn_fmed3f(u2f(b) - u2f(b & 0xFFFF0000u), -256.0f, 256.0f);
  lo = __builtin_amdgcn_perm(f2u(rb), f2u(ra), 0x07060302u);
}

// Measured (32 / 8 heads, head_dim 128, causal mask): bf16 512 rows x 4096
// tokens 1285 -> 85 us (25 -> 380 TFLOP/s), 128 rows x 8192 tokens 913 -> 56 us;
// fp16 1490 -> 118 and 938 -> 71 us; the one-row kernel ran every row's products
// on the VALU and read K/V from L2 once per row.  Now bound by the matrix cores
// and the VALU beside them at two waves per SIMD: QK^T and three PV terms are 69
// GFLOP of tiles, 55 us at the rate a large library product reaches here, and
// the softmax and the weights' terms take about as many cycles.  A second LDS
// buffer (one barrier per tile instead of two) and other orders of the PV tiles
// measured the same.
//
// Registers: at head_dim 64 and 128 nothing spills.  What kept it from that was
// a second copy of the tile's body for the split's last tile (42 VGPRs in
// scratch at 128), the int4 scales (in LDS now), and the mask's scalar
// addresses.  At head_dim 256 the tile after next is not prefetched and the
// mask is read after the scores, so that four waves keep 8 to 15 VGPRs in
// scratch (before 69 to 80; 256 rows x 4096 tokens, 16 / 2 heads 77 -> 67 us),
// and one wave, of which LDS lets four on a CU, may use 512 (4 heads x 16 x 16
// rows x 4096 tokens 379 -> 66 us).
//
// NW waves of 32 query rows each share the K/V tiles.  Unit u is (b, KV head,
// split), served by `tiles` workgroups; with xcd_map they take consecutive
// slots of one XCD (its L2 holds the unit's K/V), else they are consecutive
// workgroups.
template <int DT, int D, int NW, bool INT4>
__global__ __launch_bounds__(64 * NW, D == 256 && NW == 1 ? 1 : 2) void prefill_attn_kernel(
    AttnArgs a, int out_dtype, float* part, int64_t split_tokens, int64_t n_splits, int64_t units,
    int tiles, bool xcd_map) {
  constexpr int BT = tile_tokens(D, NW), KS = k_stride(D), VS = v_stride(D);
  constexpr int LPR = D / 8;                     // 16-byte chunks per K/V row
  constexpr int CH = BT * LPR / (64 * NW);       // chunks per lane of a tile
  constexpr int RSTEP = 64 * NW / LPR;           // rows between a lane's chunks
  static_assert(CH >= 1 && (64 * NW) % LPR == 0, "a tile is whole chunks per lane");
  // fp16 V: split where it is staged, for all waves of the workgroup, or, for a
  // single wave, where it is read (as much work, and half the LDS)
  constexpr bool F16 = DT == AMF_DTYPE_F16, SPLIT_STAGE = F16 && NW > 1;
  constexpr bool AHEAD = D <= 128;  // the next tile's rows and the mask read early
  using Raw = RawRow<DT, INT4>;
  __shared__ __attribute__((aligned(16))) uint8_t k_lds[BT * KS];
  __shared__ __attribute__((aligned(16))) uint8_t v_lds[(SPLIT_STAGE ? 2 : 1) * BT * VS];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lc = lane & 31, h = lane >> 5;
  const int64_t id = blockIdx.x;
  int64_t u;
  int tile;
  if (xcd_map) {
    const int64_t slot = id / kXcds;
    tile = (int)(slot % tiles);
    u = (slot / tiles) * kXcds + id % kXcds;
  } else {
    tile = (int)(id % tiles);
    u = id / tiles;
  }
  if (u >= units) return;
  const int64_t split = u % n_splits, bkv = u / n_splits;
  const int hkv = (int)(bkv % a.num_kv_heads);
  const int64_t b = bkv / a.num_kv_heads;
  const int G = a.num_q_heads / a.num_kv_heads;
  const int64_t T = a.kv_len;
  const int64_t t_begin = split * split_tokens, t_end = min(T, t_begin + split_tokens);
  const int64_t kv_base = (b * a.num_kv_heads + hkv) * T;

  // This lane's query row: rows run over (query token, head of the group),
  // head fastest, so the lanes of a wave share mask rows.
  const int64_t M = (int64_t)G * a.q_len;
  const int64_t row = ((int64_t)tile * NW + wave) * 32 + lc;
  const bool row_ok = row < M;
  const int64_t tq = (row_ok ? row : 0) / G;
  const int head = hkv * G + (int)((row_ok ? row : 0) % G);
  const int64_t qrow = (b * a.num_q_heads + head) * a.q_len + tq;
  u32x4 qb[D / 16];  // B operand: dims 16 ks + 8 h .. + 7
  {
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + qrow * D + 8 * h;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) qb[ks] = *reinterpret_cast<const u32x4*>(qp + 16 * ks);
  }
  const float qs = score_scale(a), e2 = exp2_factor(a);
  const float* mrow = a.mask ? a.mask + b * a.ms0 + (int64_t)head * a.ms1 + tq * a.ms2 : nullptr;
  // staging: chunk (row r0 + RSTEP i, dims 8 c ..) of the tile
  const int c = tid % LPR, r0 = tid / LPR;
  // int4: K and V channel scales (read per tile: 32 registers less across it)
  __shared__ __attribute__((aligned(16))) float s_lds[INT4 ? 2 * D : 4];
  if constexpr (INT4) {
    for (int d = tid; d < D; d += 64 * NW) {
      s_lds[d] = (float)a.k_scales[d];
      s_lds[D + d] = (float)a.v_scales[d];
    }
  }
  // this lane's scales s and -8 s of K or V
  auto scales = [&](int base, float (&sc)[8], float (&z)[8]) {
    if constexpr (INT4) {
      const f32x4* p = reinterpret_cast<const f32x4*>(s_lds + base + 8 * c);
      const f32x4 x = p[0], y = p[1];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        sc[e] = e < 4 ? x[e & 3] : y[e & 3];
        z[e] = -8.0f * sc[e];
      }
    }
  };
  Raw kr[CH], vr[CH];
  constexpr int RB = INT4 ? D / 2 : 2 * D, CB = INT4 ? 4 : 16;  // bytes of a row, of a chunk
  const uint32_t lane_off = (uint32_t)(r0 * RB + c * CB);
  // Loads of the tile at t0: a uniform base and one fixed offset per lane, or
  // (a tile that the split's end cuts) rows clamped into the split.
  auto fetch = [&](int64_t t0) {
    if (t0 + BT <= t_end) {
      const uint8_t* kb = static_cast<const uint8_t*>(a.k) + (kv_base + t0) * RB;
      const uint8_t* vb = static_cast<const uint8_t*>(a.v) + (kv_base + t0) * RB;
#pragma unroll
      for (int i = 0; i < CH; ++i) kr[i] = Raw::load(kb + i * RSTEP * RB + lane_off, 0, 0, D);
#pragma unroll
      for (int i = 0; i < CH; ++i) vr[i] = Raw::load(vb + i * RSTEP * RB + lane_off, 0, 0, D);
    } else if (t0 < t_end) {
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int64_t t = t0 + r0 + RSTEP * i;
        kr[i] = Raw::load(a.k, kv_base + (t < t_end ? t : t_begin), c, D);
        vr[i] = Raw::load(a.v, kv_base + (t < t_end ? t : t_begin), c, D);
      }
    }
  };
  auto stage = [&](int64_t t0, bool full) {
    float sc[8], z[8];
    scales(0, sc, z);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      uint32_t kp[4];
      kr[i].pairs(sc, z, kp);
      *reinterpret_cast<u32x4*>(k_lds + (r0 + RSTEP * i) * KS + 16 * c) =
          u32x4{kp[0], kp[1], kp[2], kp[3]};
    }
    scales(D, sc, z);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      uint8_t* dst = v_lds + (r0 + RSTEP * i) * VS + 16 * c;
      uint32_t vp[4];
      vr[i].pairs(sc, z, vp);
      if constexpr (SPLIT_STAGE) {
        u32x4 vh, vl;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          uint32_t x, y;
          v_split(vp[w], x, y);
          vh[w] = x;
          vl[w] = y;
        }
        *reinterpret_cast<u32x4*>(dst) = vh;
        *reinterpret_cast<u32x4*>(dst + BT * VS) = vl;
      } else {
        *reinterpret_cast<u32x4*>(dst) = u32x4{vp[0], vp[1], vp[2], vp[3]};
      }
    }
    if (!full) {  // V rows past the split: zeros (their scores are -inf below)
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int r = r0 + RSTEP * i;
        if (t0 + r < t_end) continue;
        *reinterpret_cast<u32x4*>(v_lds + r * VS + 16 * c) = u32x4{0, 0, 0, 0};
        if constexpr (SPLIT_STAGE)
          *reinterpret_cast<u32x4*>(v_lds + BT * VS + r * VS + 16 * c) = u32x4{0, 0, 0, 0};
      }
    }
  };

  float m_run = -INFINITY, l_run = 0.0f;  // l_run: this lane's tokens
  f32x16 acc[D / 32];
#pragma unroll
  for (int d = 0; d < D / 32; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d][i] = 0.0f;

  // addresses of this lane's LDS reads
  const uint8_t* k_rd = k_lds + lc * KS + 16 * h;
  const int l16 = lane & 15;
  const uint8_t* v_rd = v_lds + (4 * h + (l16 >> 2)) * VS + 32 * ((lane >> 4) & 1) + 8 * (l16 & 3);

  // A operand of V^T: dims 32 d .. + 31, 16 tokens in the order of the scores
  auto read_v = [](const uint8_t* vp) {
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vp));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vp + 8 * VS));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2[0], l2[1], h2[0], h2[1]};
  };

  // One tile; `full` when it lies inside the split: nothing is clamped or
  // masked per element then.
  auto tile_step = [&](int64_t t0, auto full) {
    if constexpr (!AHEAD) fetch(t0);
    __syncthreads();  // the previous tile has been read
    stage(t0, full);
    __syncthreads();
    // token of score element i of block tb: t0 + 32 tb + 8 (i / 4) + 4 h + i % 4
    // A contiguous mask row is read four values at once (at any multiple of 4
    // bytes), others and the row's end one at a time.
    f32x4 mk[BT / 32][4];
    auto load_mask = [&] {
      if (a.ms3 == 1 && full) {
        const float* mp = mrow + t0 + 4 * h;
#pragma unroll
        for (int tb = 0; tb < BT / 32; ++tb)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            mk[tb][g] = *reinterpret_cast<const f32x4u*>(mp + 32 * tb + 8 * g);
      } else if (full) {
        const float* mp = mrow + (t0 + 4 * h) * a.ms3;
#pragma unroll
        for (int tb = 0; tb < BT / 32; ++tb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            mk[tb][i >> 2][i & 3] = *mp;
            mp += (i & 3) == 3 ? 5 * a.ms3 : a.ms3;
            asm("" : "+v"(mp));  // one address at a time
          }
      } else {
#pragma unroll
        for (int tb = 0; tb < BT / 32; ++tb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int64_t t = t0 + 32 * tb + 8 * (i >> 2) + 4 * h + (i & 3);
            mk[tb][i >> 2][i & 3] = mrow[(t < t_end ? t : t_begin) * a.ms3];
          }
      }
    };
    if (AHEAD && mrow) load_mask();
    if constexpr (AHEAD) fetch(t0 + BT);

    f32x16 s[BT / 32];
#pragma unroll
    for (int tb = 0; tb < BT / 32; ++tb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[tb][i] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks)
        s[tb] = mfma32<DT>(*reinterpret_cast<const u32x4*>(k_rd + 32 * tb * KS + 32 * ks), qb[ks],
                           s[tb]);
    }
    if (mrow) {
      if constexpr (!AHEAD) load_mask();
#pragma unroll
      for (int tb = 0; tb < BT / 32; ++tb)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[tb][i] = fmaf(s[tb][i], qs, mk[tb][i >> 2][i & 3]);
    } else {
#pragma unroll
      for (int tb = 0; tb < BT / 32; ++tb)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[tb][i] *= qs;
    }
    if (!full) {
#pragma unroll
      for (int tb = 0; tb < BT / 32; ++tb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (t0 + 32 * tb + 8 * (i >> 2) + 4 * h + (i & 3) >= t_end) s[tb][i] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int tb = 0; tb < BT / 32; ++tb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[tb][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    // a row with every score so far -inf keeps l = 0 and acc = 0
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    if (__any(m_new > m_run)) {
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * e2);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < D / 32; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] *= alpha;
    }
    m_run = m_new;

#pragma unroll
    for (int st = 0; st < BT / 16; ++st) {
      // weights of the step's 16 tokens in bf16 terms, 8 per lane
      u32x4 pb[kTerms];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float d0 = s[st >> 1][8 * (st & 1) + 2 * j] - m_use;
        const float d1 = s[st >> 1][8 * (st & 1) + 2 * j + 1] - m_use;
        const float p0 = __builtin_amdgcn_exp2f(d0 * e2);
        const float p1 = __builtin_amdgcn_exp2f(d1 * e2);
        l_run += p0;
        l_run += p1;
        uint32_t w[kTerms];
        weight_split(p0, p1, w);
#pragma unroll
        for (int k = 0; k < kTerms; ++k) pb[k][j] = w[k];
      }
#pragma unroll
      for (int d = 0; d < D / 32; ++d) {
        const uint8_t* vp = v_rd + 16 * st * VS + 64 * d;
        const u32x4 va = read_v(vp);
        if constexpr (F16) {
          u32x4 vh = va, vl;
          if constexpr (SPLIT_STAGE) {
            vl = read_v(vp + BT * VS);
          } else {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              uint32_t x, y;
              v_split(va[w], x, y);
              vh[w] = x;
              vl[w] = y;
            }
          }
#pragma unroll
          for (int k = 0; k < kTerms; ++k) {
            acc[d] = mfma32<AMF_DTYPE_BF16>(vh, pb[k], acc[d]);
            acc[d] = mfma32<AMF_DTYPE_BF16>(vl, pb[k], acc[d]);
          }
        } else {
#pragma unroll
          for (int k = 0; k < kTerms; ++k) acc[d] = mfma32<DT>(va, pb[k], acc[d]);
        }
      }
    }
  };
  if constexpr (AHEAD) fetch(t_begin);
  if constexpr (D == 64) {
    int64_t t0 = t_begin;
    for (; t0 + BT <= t_end; t0 += BT) tile_step(t0, std::true_type{});
    if (t0 < t_end) tile_step(t0, std::false_type{});
  } else {
    // one copy of the body, with uniform branches: a second one spilled 42 VGPRs
    // at head_dim 128 (head_dim 64 has the registers, and is 5% faster with two)
    for (int64_t t0 = t_begin; t0 < t_end; t0 += BT) tile_step(t0, t0 + BT <= t_end);
  }

  const float l = l_run + __shfl_xor(l_run, 32);
  if (!row_ok) return;
  if (n_splits == 1) {
    // a row whose scores are all -inf: 0 / 0 = NaN, as softmax gives
#pragma unroll
    for (int d = 0; d < D / 32; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int64_t o = qrow * D + 32 * d + 8 * g + 4 * h;
        const f32x4 x = {acc[d][4 * g] / l, acc[d][4 * g + 1] / l, acc[d][4 * g + 2] / l,
                         acc[d][4 * g + 3] / l};
        store4(a.out, out_dtype, o, x);
      }
  } else {
    float* pr = part + (qrow * n_splits + split) * (int64_t)(D + kPartPad);
#pragma unroll
    for (int d = 0; d < D / 32; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(pr + 32 * d + 8 * g + 4 * h) =
            f32x4{acc[d][4 * g], acc[d][4 * g + 1], acc[d][4 * g + 2], acc[d][4 * g + 3]};
    if (h == 0) {
      pr[D] = m_run;
      pr[D + 1] = l;
    }
  }
}

// out = sum_k f_k acc_k / sum_k f_k l_k, f_k = 2^((m_k - M) e2), over a row's splits,
// one lane per four dims, each reading every (m, l) of its row itself; all of
// the at most N splits' loads are in flight together (in a loop over the splits
// they followed each other: a call of 64 rows x 1024 tokens, 8 heads over one of
// 128 dims, 14.5 us instead of 11.5).  More than
// kFewSplits splits go to the one-row kernel's merge (a workgroup per row).
constexpr int kFewSplits = 8;

template <int D, int N>
__global__ __launch_bounds__(256) void prefill_merge_kernel(void* out, int out_dtype, int64_t rows,
                                                            const float* part, int n_splits,
                                                            float e2) {
  constexpr int Q = D / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = i / Q;
  const int quad = (int)(i % Q);
  if (row >= rows) return;
  const float* pr = part + row * n_splits * (int64_t)(D + kPartPad);
  f32x2 ml[N];
  f32x4 x[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {  // past the last split: that one again
    const float* p = pr + min(k, n_splits - 1) * (D + kPartPad);
    ml[k] = *reinterpret_cast<const f32x2*>(p + D);
    x[k] = *reinterpret_cast<const f32x4*>(p + 4 * quad);
  }
  float M = ml[0][0];
#pragma unroll
  for (int k = 1; k < N; ++k) M = fmaxf(M, ml[k][0]);
  float den = 0.0f;
  f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int k = 0; k < N; ++k) {
    if (k < n_splits) {
      const float m = ml[k][0];
      const float f = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m - M) * e2);
      den = fmaf(ml[k][1], f, den);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = fmaf(x[k][e], f, o[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = o[e] / den;
  store4(out, out_dtype, row * D + 4 * quad, o);
}

template <int DT, int D, int NW, bool INT4>
void launch_one(const AttnArgs& a, int32_t out_dtype, float* part, const PrefillPlan& p,
                hipStream_t st) {
  const int64_t units = a.batch * a.num_kv_heads * p.n_splits;
  const bool xcd = units % kXcds == 0;
  const dim3 grid((unsigned)(units * p.tiles));
  prefill_attn_kernel<DT, D, NW, INT4><<<grid, 64 * NW, 0, st>>>(
      a, out_dtype, part, p.split_tokens, p.n_splits, units, (int)p.tiles, xcd);
  const int64_t rows = a.batch * a.num_q_heads * a.q_len;
  if (p.n_splits > kFewSplits) {
    launch_merge(a, out_dtype, rows, part, p.n_splits, st);
  } else if (p.n_splits > 1) {
    const dim3 mgrid((unsigned)((rows * (D / 4) + 255) / 256));
#define AMF_MERGE(N)                                                                   \
  prefill_merge_kernel<D, N><<<mgrid, 256, 0, st>>>(a.out, out_dtype, rows, part,      \
                                                    (int)p.n_splits, exp2_factor(a))
    if (p.n_splits <= 2)
      AMF_MERGE(2);
    else if (p.n_splits <= 4)
      AMF_MERGE(4);
    else
      AMF_MERGE(kFewSplits);
#undef AMF_MERGE
  }
}

template <int DT, bool INT4>
void launch_shape(const AttnArgs& a, int32_t out_dtype, float* part, const PrefillPlan& p,
                  hipStream_t st) {
#define AMF_PREFILL(DD)                                                           \
  (p.waves == 1 ? launch_one<DT, DD, 1, INT4>(a, out_dtype, part, p, st)   \
                : launch_one<DT, DD, 4, INT4>(a, out_dtype, part, p, st))
  if (a.head_dim == 64)
    AMF_PREFILL(64);
  else if (a.head_dim == 128)
    AMF_PREFILL(128);
  else
    AMF_PREFILL(256);
#undef AMF_PREFILL
}

}  // namespace

namespace amf {

bool prefill_plan(int64_t batch, int32_t num_q_heads, int32_t num_kv_heads, int64_t q_len,
                  int64_t kv_len, int32_t head_dim, int64_t max_splits, PrefillPlan* p) {
  const int64_t M = (int64_t)(num_q_heads / num_kv_heads) * q_len;
  if (q_len < 2 || M < kPrefillMinRows || !split_head_dim(head_dim)) return false;
  p->waves = M <= 32 ? 1 : 4;
  p->tiles = (M + 32 * p->waves - 1) / (32 * p->waves);
  const int64_t base = batch * num_kv_heads * p->tiles;
  const int64_t want = p->waves == 1 ? kPrefillGroups1 : kPrefillGroups4;
  const int64_t chunks = (kv_len + 63) / 64;
  int64_t n = (want + base - 1) / base;
  const int64_t mc = p->waves == 1 ? kPrefillMinChunks1 : kPrefillMinChunks4;
  n = std::min<int64_t>(n, (chunks + mc - 1) / mc);
  const int64_t most = std::max<int64_t>(kPrefillSplits, kMaxPrefillSplits / base);
  n = std::max<int64_t>(1, std::min<int64_t>({n, max_splits, most}));
  const int64_t per = (chunks + n - 1) / n;
  p->split_tokens = per * 64;
  p->n_splits = (chunks + per - 1) / per;
  return base <= (0x7FFFFFFF) / p->n_splits;
}

bool prefill_pays(const PrefillPlan& p, int64_t batch, int32_t num_q_heads, int32_t num_kv_heads,
                  int64_t q_len, int64_t kv_len, int32_t head_dim, bool fp16) {
  if (head_dim < 256 || num_q_heads / num_kv_heads % (fp16 ? 4 : 2) == 0) return true;
  int64_t least = kPrefillMinPairs;
  if (fp16) least *= 2;
  if (p.waves > 1 && p.n_splits > 1) least *= 2;
  return (double)batch * num_q_heads * q_len * kv_len > (double)least;
}

int64_t prefill_split_bytes(int64_t batch, int32_t num_q_heads, int64_t q_len, int32_t head_dim) {
  return batch * num_q_heads * q_len * (int64_t)(head_dim + kPartPad) * (int64_t)sizeof(float);
}

void launch_prefill(const AttnArgs& a, int32_t dtype, int32_t out_dtype, bool int4, float* part,
                    const PrefillPlan& p, hipStream_t st) {
  if (dtype == AMF_DTYPE_BF16)
    int4 ? launch_shape<AMF_DTYPE_BF16, true>(a, out_dtype, part, p, st)
         : launch_shape<AMF_DTYPE_BF16, false>(a, out_dtype, part, p, st);
  else
    int4 ? launch_shape<AMF_DTYPE_F16, true>(a, out_dtype, part, p, st)
         : launch_shape<AMF_DTYPE_F16, false>(a, out_dtype, part, p, st);
}

}  // namespace amf
