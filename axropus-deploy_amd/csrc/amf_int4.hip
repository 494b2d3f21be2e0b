// amf_int4.hip - INT4 codecs of the compressed VRAM pool, fused with the
// paged gather (save) and paged scatter (restore).
//
// Formats (layouts in include/amf_hip.h):
//  - AMF_FMT_INT4_SYM_BLOCK: INT4PerBlockCodec on a page tensor
//    (korith_vllm_ext/codecs/amf_codec.py:358-447): the page is the 16-token
//    axis padded to the codec's 128-token block, so one scale per (plane,
//    page) over every head.
//  - AMF_FMT_INT4_SYM: INT4PerChannelCodec (amf_codec.py:305-343): one scale
//    per head_dim channel over a whole layer, K and V together.
//  - AMF_FMT_INT4_ASYM_G32: asymmetric 32-dim groups, fp16 (scale, zero).
// Nibble order of the symmetric formats follows _pack_int4 / _unpack_int4
// (amf_codec.py:502-539): element 2i in the low nibble, u = q + 8.
#include "amf_internal.h"
#include "amf_kernel_util.h"

namespace {

using namespace amf;

constexpr int kThreads = 256;
constexpr float kSymMax = 7.0f;
constexpr float kAsymLevels = 15.0f;

// Nibble n (0..7) of a dword, as fp32.
__device__ __forceinline__ float nib(uint32_t w, int n) {
  return (float)__builtin_amdgcn_ubfe(w, 4 * n, 4);
}

// ------------------------------------------------------------ symmetric ----

struct SymGeom {
  int n_rows;     // block_size * num_heads
  int head_dim;
  int cpr_log2;   // log2(head_dim / 32): 32-element chunks per row
  int pps;        // planes per scale group (per-channel format)
};

// 32 cache elements at byte address `p` -> fp32.
template <int DT>
__device__ __forceinline__ void load32(const uint8_t* p, float* x) {
#pragma unroll
  for (int q = 0; q < 4; ++q) load8<DT>(p + q * (8 * elem_bytes<DT>()), x + 8 * q);
}

// Code words a sym-restore lane keeps in flight before its stores.
#ifndef AMF_SYM_RESTORE_UNROLL
#define AMF_SYM_RESTORE_UNROLL AMF_RESTORE_UNROLL
#endif

// CHANNEL = false: INT4_SYM_BLOCK (params: [n_pages] fp16);
// CHANNEL = true : INT4_SYM       (params: [head_dim] fp16 per scale group).
// One lane = one 8-element chunk (4 code bytes in, one 16-byte vector out):
// wave-wide stores cover 1 KiB contiguously.  A page of more than 8 passes
// of the workgroup is cut into `parts` workgroups of whole passes (a dense
// tensor's page can hold millions of elements).
// SLOTS: the rows go to the cache rows of the tokens' slots.
template <int DT, bool CHANNEL, bool SLOTS, int TEAM>
__global__ __launch_bounds__(kThreads) void int4_sym_dequant_scatter_kernel(
    const uint64_t* __restrict__ code_planes, const uint64_t* __restrict__ param_planes,
    const uint64_t* __restrict__ cache_planes, int64_t cache_stride,
    const int32_t* __restrict__ block_ids, int64_t pool, int64_t n_pages, int n_planes,
    int parts, SymGeom g, SlotRows rows, int32_t* err_flag) {
  __shared__ int64_t s_row[SLOTS ? kMaxSlotPage : 1];
  const PageWork pw = xcd_page_work<TEAM>(n_pages * parts, n_planes);
  if (!pw.valid) return;
  const int64_t j = pw.j / parts;
  const int part = (int)(pw.j % parts);
  const int plane = pw.plane;
  uint8_t* __restrict__ out = reinterpret_cast<uint8_t*>(cache_planes[plane]);
  if constexpr (SLOTS) {
    slot_row_offsets(rows, j, s_row, err_flag);
  } else {
    const int64_t dp = block_ids ? (int64_t)block_ids[j] : j;
    if (dp < 0 || dp >= pool) {
      if (threadIdx.x % TEAM == 0 && err_flag) atomicOr(err_flag, AMF_ERRFLAG_BLOCK_RANGE);
      return;
    }
    out += dp * cache_stride;
  }
  const int page_elems = g.n_rows * g.head_dim;
  const int n8 = page_elems >> 3;
  // this workgroup's chunks: [k_begin, k_end), k_begin a multiple of TEAM
  const int span = (n8 + parts - 1) / parts;
  const int k_begin = part * ((span + TEAM - 1) / TEAM * TEAM);
  const int k_end = min(n8, k_begin + (span + TEAM - 1) / TEAM * TEAM);
  const uint32_t* __restrict__ codes =
      reinterpret_cast<const uint32_t*>(code_planes[plane]) + j * (int64_t)n8;
  const _Float16* __restrict__ params = reinterpret_cast<const _Float16*>(param_planes[plane]);
  const int tid = threadIdx.x % TEAM;
  const float s_page = CHANNEL ? 0.0f : (float)params[j];
  // Channel scales of this lane's 8 dims; fixed while 8 * TEAM is a
  // multiple of head_dim (checked on the host).
  float s_ch[8];
  if (CHANNEL) {
    const int d0 = (tid * 8) % g.head_dim;
#pragma unroll
    for (int q = 0; q < 8; ++q) s_ch[q] = (float)params[d0 + q];
  }
  const uint32_t cpt = SLOTS ? (uint32_t)n8 / (uint32_t)rows.page_tokens : 1;  // chunks per row
  constexpr int U = AMF_SYM_RESTORE_UNROLL;
  for (int base = k_begin + tid; base < k_end; base += U * TEAM) {
    uint32_t c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = base + u * TEAM;
      if (k < k_end) c[u] = ld_stream(codes + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = base + u * TEAM;
      if (k < k_end) {
        float x[8];
#pragma unroll
        for (int n = 0; n < 8; ++n) x[n] = (nib(c[u], n) - 8.0f) * (CHANNEL ? s_ch[n] : s_page);
        if constexpr (SLOTS) {
          const uint32_t t = (uint32_t)k / cpt;
          const int64_t off = s_row[t];
          if (off >= 0) store8<DT>(out + off + (k - t * cpt) * (8 * elem_bytes<DT>()), x);
        } else {
          store8<DT>(out + (int64_t)k * (8 * elem_bytes<DT>()), x);
        }
      }
    }
  }
}

constexpr int kBigThreads = 1024;

// INT4_SYM_BLOCK save: page absmax -> scale -> codes; the page stays in
// registers.  One lane = CPL 8-element chunks NT apart, so each load
// instruction of a wave covers 1 KiB of whole lines (non-temporal: read once)
// and each code store 256 contiguous bytes.  A lane holds at most 8 chunks up
// to pages of 8192 chunks (at most 64 VGPRs: two workgroups of 1024 lanes a
// CU, so that one loads while the other quantizes) and 16 up to 16384, a
// dense entry's block of 128 tokens x 8 heads x 128 dims.  64 planes, bf16,
// before (256 lanes: 32 chunks a lane up to 8192, two reads beyond) and now:
// 32 blocks of 8 heads 225 -> 144 us (4.66 TB/s), 64 blocks of 4 heads 198 ->
// 108 us (6.19 TB/s); one layer's 64 blocks of 8 heads 39 -> 16 us.
// SLOTS: the page's rows are cache rows named by token slots (zeros past the
// sequence's end), read in place instead of from a gathered copy.
// NT = 64: a wave per (small) page, four to a workgroup.
template <bool BF16, int CPL, int NT, bool SLOTS>
__global__ __launch_bounds__(NT < kThreads ? kThreads : NT,
                             CPL <= 8 && (NT > kThreads || !BF16) ? 8 : 1) void
int4_symblock_quant_gather_kernel(
    const uint64_t* __restrict__ cache_planes, int64_t cache_stride,
    const int32_t* __restrict__ block_ids, int64_t pool, int64_t n_pages,
    const uint64_t* __restrict__ code_planes, const uint64_t* __restrict__ param_planes,
    SymGeom g, SlotRows rows, int32_t* err_flag) {
  static_assert(NT >= kThreads || (NT == 64 && !SLOTS), "the slot form takes whole workgroups");
  constexpr int kPages = NT < kThreads ? kThreads / NT : 1;
  const int64_t j =
      (int64_t)blockIdx.x * kPages +
      (kPages > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0);
  if (kPages > 1 && j >= n_pages) return;
  const int tid = kPages > 1 ? threadIdx.x % NT : threadIdx.x;
  const int plane = blockIdx.y;
  __shared__ int64_t s_row[SLOTS ? kMaxSlotPage : 1];
  const int n8 = (int)((int64_t)g.n_rows * g.head_dim / 8);
  const uint8_t* __restrict__ src = reinterpret_cast<const uint8_t*>(cache_planes[plane]);
  if constexpr (SLOTS) {
    slot_row_offsets(rows, j, s_row, err_flag);
  } else {
    const int64_t sp = block_ids ? (int64_t)block_ids[j] : j;
    if (sp < 0 || sp >= pool) {
      if (tid == 0 && err_flag) atomicOr(err_flag, AMF_ERRFLAG_BLOCK_RANGE);
      return;
    }
    src += sp * cache_stride;
  }
  uint32_t* __restrict__ codes = reinterpret_cast<uint32_t*>(code_planes[plane]) + j * n8;
  _Float16* __restrict__ params = reinterpret_cast<_Float16*>(param_planes[plane]);

  u32x4 v[CPL];
  if constexpr (SLOTS) {
    const uint32_t cpt = (uint32_t)n8 / (uint32_t)rows.page_tokens;  // chunks per token row
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      const uint32_t k = tid + i * NT;
      v[i] = u32x4{0, 0, 0, 0};
      if (k < (uint32_t)n8) {
        const uint32_t t = k / cpt;
        const int64_t off = s_row[t];
        if (off >= 0) v[i] = ld_stream(reinterpret_cast<const u32x4*>(src + off) + (k - t * cpt));
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      const int k = tid + i * NT;
      if (k < n8) v[i] = ld_stream(reinterpret_cast<const u32x4*>(src) + k);
    }
  }
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    if (tid + i * NT < n8) {
      float x[8];
      unpack8<BF16>(v[i], x);
#pragma unroll
      for (int n = 0; n < 8; ++n) m = fmaxf(m, fabsf(x[n]));
    }
  }
  float amax = wave_max_xor(m, 64);
  if constexpr (NT > 64) {
    __shared__ float s_wmax[NT / 64];
    if ((tid & 63) == 0) s_wmax[tid >> 6] = amax;
    __syncthreads();
    amax = s_wmax[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) amax = fmaxf(amax, s_wmax[w]);
  }
  // amf_codec.py:392-394: absmax.clamp_min(1e-8) / 7 in fp32.
  const float scale = fmaxf(amax, 1e-8f) / kSymMax;
  const float rscale = 1.0f / scale;
  if (tid == 0) params[j] = (_Float16)scale;
  // In the large workgroups, and for fp16, the words are unpacked again: kept
  // from the maximum they would take twice the registers of the page itself
  // (234 us instead of 144).
  if constexpr (NT > kThreads || !BF16) {
#pragma unroll
    for (int i = 0; i < CPL; ++i) asm("" : "+v"(v[i]));
  }
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    const int k = tid + i * NT;
    if (k < n8) {
      float x[8];
      unpack8<BF16>(v[i], x);
      uint32_t w = 0;
#pragma unroll
      for (int n = 0; n < 8; ++n)
        w = push_code(w, div_rn_code(x[n], scale, rscale), -8.0f, 7.0f, 8.0f);
      st_stream(w, codes + k);
    }
  }
}

// INT4_SYM_BLOCK save of pages larger than the register-resident kernels
// hold, and of fp32 caches: the page absmax in a first read, the codes in a
// second (which hits in cache).  One lane = one 8-element chunk per step,
// U of them loaded before any is used: a page is one workgroup
// however large it is, so the bytes that workgroup keeps in flight set its
// rate (a page of 2M elements 500 -> 121 us with 1024 lanes of 4 chunks for 256
// of one).  An fp32 page of at most kLoopChunks chunks leaves such a workgroup
// mostly idle and takes 256 lanes of one (32 x 300 pages of 1 x 64 71 / 21 us
// with 1024 / 256 lanes, 32 x 250 of 5 x 128 205 / 195, 32 x 200 of 8 x 128 224 /
// 248).  Same arithmetic as int4_symblock_quant_gather_kernel.
constexpr int64_t kLoopChunks = 1536;

template <int DT, int NT, int U>
__global__ __launch_bounds__(NT) void int4_symblock_quant_looped_kernel(
    const uint64_t* __restrict__ cache_planes, int64_t cache_stride,
    const int32_t* __restrict__ block_ids, int64_t pool, const uint64_t* __restrict__ code_planes,
    const uint64_t* __restrict__ param_planes, SymGeom g, int32_t* err_flag) {
  constexpr int ES = elem_bytes<DT>();
  const int64_t j = blockIdx.x;
  const int plane = blockIdx.y;
  const int64_t sp = block_ids ? (int64_t)block_ids[j] : j;
  if (sp < 0 || sp >= pool) {
    if (threadIdx.x == 0 && err_flag) atomicOr(err_flag, AMF_ERRFLAG_BLOCK_RANGE);
    return;
  }
  const int64_t n8 = (int64_t)g.n_rows * g.head_dim / 8;
  const uint8_t* __restrict__ src =
      reinterpret_cast<const uint8_t*>(cache_planes[plane]) + sp * cache_stride;
  uint32_t* __restrict__ codes = reinterpret_cast<uint32_t*>(code_planes[plane]) + j * n8;
  _Float16* __restrict__ params = reinterpret_cast<_Float16*>(param_planes[plane]);
  float m = 0.0f;
  for (int64_t k0 = threadIdx.x; k0 < n8; k0 += U * NT) {
    float x[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = k0 + u * NT;  // past the end: the lane's first chunk again
      load8<DT>(src + (k < n8 ? k : k0) * (8 * ES), x[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int n = 0; n < 8; ++n) m = fmaxf(m, fabsf(x[u][n]));
  }
  m = wave_max_xor(m, 64);
  __shared__ float s_wmax[NT / 64];
  if ((threadIdx.x & 63) == 0) s_wmax[threadIdx.x >> 6] = m;
  __syncthreads();
  float amax = s_wmax[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) amax = fmaxf(amax, s_wmax[w]);
  const float scale = fmaxf(amax, 1e-8f) / kSymMax;
  const float rscale = 1.0f / scale;
  if (threadIdx.x == 0) params[j] = (_Float16)scale;
  for (int64_t k0 = threadIdx.x; k0 < n8; k0 += U * NT) {
    float x[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = k0 + u * NT;
      load8<DT>(src + (k < n8 ? k : k0) * (8 * ES), x[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = k0 + u * NT;
      uint32_t w = 0;
#pragma unroll
      for (int n = 0; n < 8; ++n)
        w = push_code(w, div_rn_code(x[u][n], scale, rscale), -8.0f, 7.0f, 8.0f);
      if (k < n8) st_stream(w, codes + k);
    }
  }
}

// INT4_SYM save, pass 1: per-channel absmax over a scale group.  One lane =
// one 8-element chunk, as in pass 2 (kThreads * 8 is a multiple of head_dim,
// so a lane's 8 channels stay fixed): every load instruction of a wave covers
// 1 KiB of whole lines, and a page's chunks are all in flight at once.  Each
// workgroup folds a strided set of pages, reduces the lanes that share
// channels (shuffles, then an LDS table), and issues one global atomic max
// per channel into ws[group][head_dim].
constexpr int kAbsmaxUnroll = 8;

// Small pages are read PPI at a time, so that as many loads are in flight.
template <int DT, int PPI>
__global__ __launch_bounds__(kThreads) void int4_channel_absmax_kernel(
    const uint64_t* __restrict__ cache_planes, int64_t cache_stride,
    const int32_t* __restrict__ block_ids, int64_t pool, int64_t n_pages, SymGeom g,
    uint32_t* ws, int32_t* err_flag) {
  constexpr int U = kAbsmaxUnroll / PPI;
  const int plane = blockIdx.y;
  __shared__ uint32_t s_max[1024];
  for (int d = threadIdx.x; d < g.head_dim; d += kThreads) s_max[d] = 0;
  const int n8 = (int)((int64_t)g.n_rows * g.head_dim / 8);
  float m[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) m[q] = 0.0f;
  for (int64_t j0 = blockIdx.x; j0 < n_pages; j0 += (int64_t)gridDim.x * PPI) {
    const uint8_t* src[PPI];
#pragma unroll
    for (int p = 0; p < PPI; ++p) {
      const int64_t j = j0 + (int64_t)p * gridDim.x;
      src[p] = nullptr;
      if (j < n_pages) {
        const int64_t sp = block_ids ? (int64_t)block_ids[j] : j;
        if (sp >= 0 && sp < pool)
          src[p] = reinterpret_cast<const uint8_t*>(cache_planes[plane]) + sp * cache_stride;
        else if (threadIdx.x == 0 && err_flag)
          atomicOr(err_flag, AMF_ERRFLAG_BLOCK_RANGE);
      }
    }
    if (PPI == 1 && !src[0]) continue;
    // PPI > 1: the page fits one step
    for (int base = threadIdx.x; base < n8; base += kThreads * U) {
      float x[PPI][U][8];
#pragma unroll
      for (int p = 0; p < PPI; ++p)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = base + u * kThreads;
          if ((PPI == 1 || src[p]) && k < n8) load8_stream<DT>(src[p] + (int64_t)k * (8 * elem_bytes<DT>()), x[p][u]);
        }
#pragma unroll
      for (int p = 0; p < PPI; ++p)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if ((PPI == 1 || src[p]) && base + u * kThreads < n8) {
#pragma unroll
            for (int q = 0; q < 8; ++q) m[q] = fmaxf(m[q], fabsf(x[p][u][q]));
          }
        }
    }
  }
  // Lanes lane, lane + L, lane + 2L, ... of a wave (L = head_dim / 8 chunks
  // per row) hold the same channels.
  const int lpr = g.head_dim / 8;
#pragma unroll
  for (int q = 0; q < 8; ++q)
    for (int o = 32; o >= lpr; o >>= 1) m[q] = fmaxf(m[q], __shfl_xor(m[q], o));
  __syncthreads();  // s_max cleared
  if ((threadIdx.x & 63) < lpr) {
    const int d0 = (threadIdx.x * 8) % g.head_dim;
#pragma unroll
    for (int q = 0; q < 8; ++q) atomicMax(&s_max[d0 + q], f2u(m[q]));
  }
  __syncthreads();
  for (int d = threadIdx.x; d < g.head_dim; d += kThreads)
    atomicMax(ws + (int64_t)(plane / g.pps) * g.head_dim + d, s_max[d]);
}

__global__ void fill_u32_kernel(uint32_t* p, int64_t n, uint32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// INT4_SYM save, pass 2: one lane = one 8-element chunk (16 bytes of bf16 in,
// one 4-byte code word out), so a wave stores 256 contiguous bytes.  Chunk k
// covers channels (8 k) % head_dim ..+7 and k advances by kThreads, a
// multiple of head_dim / 8: a lane's 8 channels, and so its scales and
// reciprocals, stay fixed for the whole page.
#ifndef AMF_CHAN_UNROLL
#define AMF_CHAN_UNROLL 4
#endif
constexpr int kChanUnroll = AMF_CHAN_UNROLL;

// TEAM lanes take a page: a wave for small pages.
template <int DT, int TEAM>
__global__ __launch_bounds__(kThreads) void int4_channel_quant_gather_kernel(
    const uint64_t* __restrict__ cache_planes, int64_t cache_stride,
    const int32_t* __restrict__ block_ids, int64_t pool, int64_t n_pages,
    const uint64_t* __restrict__ code_planes, const uint64_t* __restrict__ param_planes, SymGeom g, const uint32_t* __restrict__ ws,
    int32_t* err_flag) {
  constexpr int kPages = kThreads / TEAM;
  const int64_t j =
      (int64_t)blockIdx.x * kPages +
      (kPages > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / TEAM) : 0);
  if (kPages > 1 && j >= n_pages) return;
  const int tid = kPages > 1 ? threadIdx.x % TEAM : threadIdx.x;
  const int plane = blockIdx.y;
  // The group's fp16 scales (amf_codec.py:312-313), written once per group
  // by its first plane's first page.
  if (j == 0 && plane % g.pps == 0) {
    _Float16* p = reinterpret_cast<_Float16*>(param_planes[plane]);
    const uint32_t* gw = ws + (int64_t)(plane / g.pps) * g.head_dim;
    for (int d = tid; d < g.head_dim; d += TEAM)
      p[d] = (_Float16)(fmaxf(u2f(gw[d]), 1e-8f) / kSymMax);
  }
  const int64_t sp = block_ids ? (int64_t)block_ids[j] : j;
  if (sp < 0 || sp >= pool) {
    if (tid == 0 && err_flag) atomicOr(err_flag, AMF_ERRFLAG_BLOCK_RANGE);
    return;
  }
  const int64_t page_elems = (int64_t)g.n_rows * g.head_dim;
  const int n8 = (int)(page_elems / 8);
  const uint8_t* __restrict__ src =
      reinterpret_cast<const uint8_t*>(cache_planes[plane]) + sp * cache_stride;
  uint32_t* __restrict__ codes =
      reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(code_planes[plane]) + j * (page_elems / 2));
  const int d0 = (tid * 8) % g.head_dim;
  const uint32_t* lw = ws + (int64_t)(plane / g.pps) * g.head_dim + d0;
  float sc[8], rc[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    sc[q] = fmaxf(u2f(lw[q]), 1e-8f) / kSymMax;  // amf_codec.py:312-313
    rc[q] = 1.0f / sc[q];
  }
  for (int base = tid; base < n8; base += TEAM * kChanUnroll) {
    float x[kChanUnroll][8];
#pragma unroll
    for (int u = 0; u < kChanUnroll; ++u) {
      const int k = base + u * TEAM;
      if (k < n8) load8_stream<DT>(src + (int64_t)k * (8 * elem_bytes<DT>()), x[u]);
    }
#pragma unroll
    for (int u = 0; u < kChanUnroll; ++u) {
      const int k = base + u * TEAM;
      if (k < n8) {
        uint32_t w = 0;
#pragma unroll
        for (int n = 0; n < 8; ++n)
          w = push_code(w, div_rn_code(x[u][n], sc[n], rc[n]), -8.0f, 7.0f, 8.0f);
        st_stream(w, codes + k);
      }
    }
  }
}

// ----------------------------------------------------------- asymmetric ----
//
// Page geometry: block_size 16, G = head_dim / 32 groups.  Per (page, head):
// K codes [16][D/2], K params [16][G]; V codes tiled dim-major, V params [G][16].

struct AsymGeom {
  int num_heads;
  int head_dim;
  int groups;          // head_dim / 32
  int hb_code_bytes;   // 16 * head_dim / 2   (one (page, head) code block)
  int hb_param_words;  // 16 * groups
  int kpr_log2, h_log2;  // log2(head_dim / 8) and log2(num_heads), -1 unless powers of two
};

// Group quantizer: min / max over 32 values, then
// scale = max(mx - mn, 1e-8) / 15 and q = clamp(rint((x - mn) / scale), 0, 15).
struct AsymParams {
  float mn, scale, rscale;
};

__device__ __forceinline__ AsymParams asym_params(const float* x) {
  float mn = x[0], mx = x[0];
#pragma unroll
  for (int n = 1; n < 32; ++n) {
    mn = fminf(mn, x[n]);
    mx = fmaxf(mx, x[n]);
  }
  AsymParams p;
  p.mn = mn;
  p.scale = fmaxf(mx - mn, 1e-8f) / kAsymLevels;
  p.rscale = 1.0f / p.scale;
  return p;
}

// Code n of eight into w, in order.  The wave-per-page save pushes it
// (push_code), which needs fewer operations; with a workgroup per page the
// compiler then holds so many chains at once that waves are lost (32 layers x
// 500 pages of 4 x 128: 145 us against 133).
template <int TEAM>
__device__ __forceinline__ uint32_t asym_insert(uint32_t w, int n, float x,
                                                const AsymParams& p) {
  if constexpr (TEAM == 64)
    return push_code(w, div_rn_code(x - p.mn, p.scale, p.rscale), 0.0f, kAsymLevels, 0.0f);
  float q = __builtin_rintf(div_rn(x - p.mn, p.scale, p.rscale));
  q = fminf(fmaxf(q, 0.0f), kAsymLevels);
  return w | (uint32_t)q << (4 * n);
}

__device__ __forceinline__ uint32_t asym_param_word(const AsymParams& p) {
  uint32_t s = __builtin_bit_cast(uint16_t, (_Float16)p.scale);
  uint32_t z = __builtin_bit_cast(uint16_t, (_Float16)p.mn);
  return s | (z << 16);
}

__device__ __forceinline__ float param_scale(uint32_t w) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu));
}
__device__ __forceinline__ float param_zero(uint32_t w) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
}

// Restore of one page of one plane; even planes are K, odd planes V (tiled
// layout).  Items:
//  K: (head, token, group): 16 code bytes + 1 param word -> 32 outputs of a row
//  V: (head, 8-dim block, token half): 32 code bytes + 8 param words ->
//     8 tokens x 8 dims.
#ifndef AMF_ASYM_K_UNROLL
#define AMF_ASYM_K_UNROLL 4
#endif
constexpr int kKUnroll = AMF_ASYM_K_UNROLL;

// TEAM lanes take a page (four pages a workgroup when it is small), and a V
// item writes 8 / VSPLIT of its tokens, so that a page of few heads still has
// an item for each lane.  P2: head_dim and the head count are powers of two,
// so the items' indices are shifts (others divide, a workgroup to a page: no
// model of the sizes served here has such pages).  fp32 pages, twice the bytes,
// keep a workgroup each.  80 layers x 777 pages of 1 x 128 235 ->
// 113 us, 32 x 1000 of 2 x 128 153 -> 115 us (6.0 TB/s), 32 x 512 of 8 x 128
// 245 -> 241 us.
template <int DT, int TEAM, int VSPLIT, bool P2>
__global__ __launch_bounds__(kThreads) void int4_asym_dequant_scatter_kernel(
    const uint64_t* __restrict__ code_planes, const uint64_t* __restrict__ param_planes,
    const uint64_t* __restrict__ cache_planes, int64_t cache_stride,
    const int32_t* __restrict__ block_ids, int64_t pool, int64_t n_pages, AsymGeom g,
    int32_t* err_flag) {
  // A (page, plane) grid, page-major: all XCDs work on one plane at a time,
  // which measured faster here than the XCD-contiguous map of the other
  // restores (1.025 vs 1.065 ms at 32 layers x 2048 pages).
  constexpr int kPages = kThreads / TEAM;
  const int64_t j =
      (int64_t)blockIdx.x * kPages +
      (kPages > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / TEAM) : 0);
  if (kPages > 1 && j >= n_pages) return;
  const int tid = threadIdx.x % TEAM;
  const int plane = blockIdx.y;
  const bool is_v = (plane & 1) != 0;
  const int64_t dp = block_ids ? (int64_t)block_ids[j] : j;
  if (dp < 0 || dp >= pool) {
    if (tid == 0 && err_flag) atomicOr(err_flag, AMF_ERRFLAG_BLOCK_RANGE);
    return;
  }
  const int H = g.num_heads, D = g.head_dim, G = g.groups;
  const int kpr = D / 8;  // 8-dim blocks per row
  // quotient by, and remainder of, the block count and the head count
  auto by_kpr = [&](int x) { return P2 ? x >> g.kpr_log2 : x / kpr; };
  auto of_kpr = [&](int x) { return P2 ? x & (kpr - 1) : x % kpr; };
  auto by_h = [&](int x) { return P2 ? x >> g.h_log2 : x / H; };
  auto of_h = [&](int x) { return P2 ? x & (H - 1) : x % H; };
  const uint8_t* __restrict__ codes = reinterpret_cast<const uint8_t*>(code_planes[plane]) +
                                      j * (int64_t)H * g.hb_code_bytes;
  const uint32_t* __restrict__ params = reinterpret_cast<const uint32_t*>(param_planes[plane]) +
                                        j * (int64_t)H * g.hb_param_words;
  uint8_t* __restrict__ out = reinterpret_cast<uint8_t*>(cache_planes[plane]) + dp * cache_stride;

  if (!is_v) {
    // Items (token, head, 8-dim block) in cache order: lane k writes the k-th
    // 16-byte vector of the page, reads 4 code bytes and its group's param word.
    // kKUnroll items per lane have their code and param loads in flight
    // before any is converted.
    const int n_items = 16 * H * kpr;
    for (int it0 = tid; it0 < n_items; it0 += TEAM * kKUnroll) {
      uint32_t c[kKUnroll], pw[kKUnroll];
#pragma unroll
      for (int u = 0; u < kKUnroll; ++u) {
        const int it = it0 + u * TEAM;
        if (it < n_items) {
          const int kk = of_kpr(it);
          const int th = by_kpr(it);  // token * H + head
          const int t = by_h(th), h = of_h(th);
          const int ht = h * 16 + t;
          c[u] = ld_stream(reinterpret_cast<const uint32_t*>(codes + (int64_t)ht * (D / 2)) + kk);
          pw[u] = params[ht * G + (kk >> 2)];
        }
      }
#pragma unroll
      for (int u = 0; u < kKUnroll; ++u) {
        const int it = it0 + u * TEAM;
        if (it < n_items) {
          const float s = param_scale(pw[u]), z = param_zero(pw[u]);
          float x[8];
#pragma unroll
          for (int n = 0; n < 8; ++n) x[n] = nib(c[u], n) * s + z;
          store8<DT>(out + (int64_t)it * (8 * elem_bytes<DT>()), x);
        }
      }
    }
  } else {
    // Items (head, token half, part, 8-dim block), the block fastest: lanes
    // next to each other write next to each other.
    constexpr int NT = 8 / VSPLIT;  // tokens of an item
    const int n_items = H * kpr * 2 * VSPLIT;
    for (int it = tid; it < n_items; it += TEAM) {
      const int b = of_kpr(it);
      const int r = by_kpr(it);
      const int i0 = r % VSPLIT * NT;
      const int th = r / VSPLIT & 1;
      const int h = r / (2 * VSPLIT);
      const u32x4* cp =
          reinterpret_cast<const u32x4*>(codes + (int64_t)h * g.hb_code_bytes + 64 * b + 32 * th);
      const u32x4 c0 = ld_stream(cp);
      const u32x4 c1 = ld_stream(cp + 1);
      const uint32_t w[8] = {c0[0], c0[1], c0[2], c0[3], c1[0], c1[1], c1[2], c1[3]};
      const uint32_t* pp = params + h * g.hb_param_words + (b >> 2) * 16 + 8 * th + i0;
      uint32_t pw[NT];
#pragma unroll
      for (int i = 0; i < NT; ++i) pw[i] = pp[i];
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const float s = param_scale(pw[i]), z = param_zero(pw[i]);
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = nib(w[k], i0 + i) * s + z;
        const int t = 8 * th + i0 + i;
        store8<DT>(out + elem_bytes<DT>() * ((int64_t)(t * H + h) * D + 8 * b), x);
      }
    }
  }
}

// The lanes that save a page: the workgroup, or one wave of it (small pages,
// four to a workgroup).  A wave's LDS accesses complete in order, so its sync
// only keeps the compiler from moving them.
template <int TEAM>
__device__ __forceinline__ int team_lane() {
  return (int)(TEAM == kThreads ? threadIdx.x : threadIdx.x % TEAM);
}
template <int TEAM>
__device__ __forceinline__ void team_sync() {
  if constexpr (TEAM == 64) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// A page's bytes -> LDS, kStageUnroll 16-byte vectors per lane in flight.
// (Padding the rows against the bank conflicts of the quantizers' 64-byte
// reads measured slower: 140 vs 133 us at 32 layers x 500 pages of 4 x 128.)
#ifndef AMF_ASYM_STAGE_UNROLL
#define AMF_ASYM_STAGE_UNROLL 8
#endif
constexpr int kStageUnroll = AMF_ASYM_STAGE_UNROLL;

template <int TEAM>
__device__ __forceinline__ void stage_page(const uint8_t* __restrict__ src, int page_bytes,
                                           uint8_t* lds) {
  for (int o0 = team_lane<TEAM>() * 16; o0 < page_bytes; o0 += TEAM * 16 * kStageUnroll) {
    u32x4 v[kStageUnroll];
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const int o = o0 + u * TEAM * 16;
      if (o < page_bytes) v[u] = ld_stream(reinterpret_cast<const u32x4*>(src + o));
    }
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const int o = o0 + u * TEAM * 16;
      if (o < page_bytes) *reinterpret_cast<u32x4*>(lds + o) = v[u];
    }
  }
}

// Save of one page of a K plane: items (head, token, group) read 64 cache
// bytes, write 16 code bytes and one param word.
#ifndef AMF_ASYM_KSAVE_UNROLL
#define AMF_ASYM_KSAVE_UNROLL 2
#endif
constexpr int kKSaveUnroll = AMF_ASYM_KSAVE_UNROLL;
template <int DT, int TEAM, int KU>
__device__ __forceinline__ void asym_quant_k(const uint8_t* __restrict__ src,
                                             uint8_t* __restrict__ codes,
                                             uint32_t* __restrict__ params, const AsymGeom& g) {
  const int H = g.num_heads, D = g.head_dim, G = g.groups;
  const int n_items = 16 * H * G;
  // Items in cache order (token, head, group) so the loads are contiguous;
  // KU items per lane are loaded before any is quantized.
  for (int it0 = team_lane<TEAM>(); it0 < n_items; it0 += TEAM * KU) {
    float x[KU][32];
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int it = it0 + u * TEAM;
      if (it < n_items)
        load32<DT>(src + elem_bytes<DT>() * ((int64_t)(it / G) * D + 32 * (it % G)), x[u]);
    }
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int it = it0 + u * TEAM;
      if (it < n_items) {
        const int gi = it % G;
        const int th = it / G;  // token * H + head
        const int t = th / H, h = th % H;
        const AsymParams p = asym_params(x[u]);
        u32x4 c;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t w = 0;
#pragma unroll
          for (int n = 0; n < 8; ++n)
            w = asym_insert<TEAM>(w, n, x[u][8 * q + n], p);
          c[q] = w;
        }
        const int ht = h * 16 + t;
        st_stream(c, reinterpret_cast<u32x4*>(codes + (int64_t)ht * (D / 2) + 16 * gi));
        params[ht * G + gi] = asym_param_word(p);
      }
    }
  }
}

// Save of one page of a V plane.  Groups run along head_dim while the code
// tiles run along tokens: phase 1 computes every group's (mn, scale) into LDS
// tables, phase 2 builds the 8-token x 8-dim tiles.  STAGED copies the page
// into LDS first (when it fits); otherwise both phases read the page from
// global memory, where the second read hits in cache.
constexpr int kAsymLdsBytes = 64 * 1024;

template <int DT, bool STAGED, int TEAM>
__device__ __forceinline__ void asym_quant_v(const uint8_t* __restrict__ src,
                                             uint8_t* __restrict__ codes,
                                             uint32_t* __restrict__ params, const AsymGeom& g,
                                             uint8_t* lds) {
  constexpr int ES = elem_bytes<DT>();
  const int H = g.num_heads, D = g.head_dim, G = g.groups;
  const int page_bytes = STAGED ? 16 * H * D * ES : 0;
  // phase 0: page -> LDS (cache layout)
  if (STAGED) stage_page<TEAM>(src, page_bytes, lds);
  const uint8_t* data = STAGED ? lds : src;
  float* s_mn = reinterpret_cast<float*>(lds + page_bytes);          // [H][G][16]
  float* s_sc = s_mn + 16 * H * G;                                   // [H][G][16]
  float* s_rc = s_sc + 16 * H * G;                                   // [H][G][16]
  team_sync<TEAM>();
  const int n_groups = 16 * H * G;
  for (int it = team_lane<TEAM>(); it < n_groups; it += TEAM) {
    // it = (head, group, token): params are written in V order.
    const int t = it & 15;
    const int hg = it >> 4;
    const int h = hg / G, gi = hg % G;
    float x[32];
    load32<DT>(data + ES * ((t * H + h) * D + 32 * gi), x);
    const AsymParams p = asym_params(x);
    s_mn[it] = p.mn;
    s_sc[it] = p.scale;
    s_rc[it] = p.rscale;
    params[it] = asym_param_word(p);
  }
  team_sync<TEAM>();
  const int nb = D / 8;
  const int n_items = H * nb * 2;
  for (int it = team_lane<TEAM>(); it < n_items; it += TEAM) {
    const int th = it & 1;
    const int b = (it >> 1) % nb;
    const int h = (it >> 1) / nb;
    uint32_t w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = 8 * th + i;
      const int pi = (h * G + (b >> 2)) * 16 + t;
      AsymParams p;
      p.mn = s_mn[pi];
      p.scale = s_sc[pi];
      p.rscale = s_rc[pi];
      float x[8];
      load8<DT>(data + ES * ((t * H + h) * D + 8 * b), x);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        w[k] = asym_insert<TEAM>(w[k], i, x[k], p);
    }
    u32x4* cp = reinterpret_cast<u32x4*>(codes + (int64_t)h * g.hb_code_bytes + 64 * b + 32 * th);
    st_stream(u32x4{w[0], w[1], w[2], w[3]}, cp);
    st_stream(u32x4{w[4], w[5], w[6], w[7]}, cp + 1);
  }
}

// One page per team; KU: K items a lane loads at once.  A wave per page for
// small pages (four to a workgroup; one K item per lane for one head, whose
// registers allow 8 waves per SIMD): 80 layers x 777 pages of 1 x 128 213 ->
// 122 us, 32 x 1000 of 2 x 128 152 -> 119 us (5.8 TB/s), where a workgroup per
// page had 64 and 128 items for its 256 lanes.
template <int DT, bool STAGED, int TEAM, int KU>
__global__ __launch_bounds__(kThreads, TEAM == kThreads ? 1 : KU == 1 ? 8 : 5) void
int4_asym_quant_gather_kernel(
    const uint64_t* __restrict__ cache_planes, int64_t cache_stride,
    const int32_t* __restrict__ block_ids, int64_t pool, int64_t n_pages,
    const uint64_t* __restrict__ code_planes, const uint64_t* __restrict__ param_planes,
    AsymGeom g, int team_lds, int32_t* err_flag) {
  extern __shared__ __attribute__((aligned(16))) uint8_t shared_lds[];
  constexpr int kPages = kThreads / TEAM;
  const int team = kPages > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / TEAM) : 0;
  uint8_t* lds = shared_lds + team * team_lds;
  const int64_t j = (int64_t)blockIdx.x * kPages + team;
  if (kPages > 1 && j >= n_pages) return;
  const int plane = blockIdx.y;
  const int64_t sp = block_ids ? (int64_t)block_ids[j] : j;
  if (sp < 0 || sp >= pool) {
    if (team_lane<TEAM>() == 0 && err_flag) atomicOr(err_flag, AMF_ERRFLAG_BLOCK_RANGE);
    return;
  }
  const int H = g.num_heads;
  const uint8_t* __restrict__ src =
      reinterpret_cast<const uint8_t*>(cache_planes[plane]) + sp * cache_stride;
  uint8_t* __restrict__ codes =
      reinterpret_cast<uint8_t*>(code_planes[plane]) + j * (int64_t)H * g.hb_code_bytes;
  uint32_t* __restrict__ params =
      reinterpret_cast<uint32_t*>(param_planes[plane]) + j * (int64_t)H * g.hb_param_words;
  if ((plane & 1) == 0) {
    if (STAGED) {
      // The page enters LDS by whole-line non-temporal loads (1 KiB per wave
      // instruction); the items' 64-byte reads then come from LDS.  Reading
      // the items straight from memory splits every line over four load
      // instructions, which the non-temporal policy would fetch repeatedly.
      stage_page<TEAM>(src, 16 * H * g.head_dim * elem_bytes<DT>(), lds);
      team_sync<TEAM>();
      asym_quant_k<DT, TEAM, KU>(lds, codes, params, g);
    } else {
      asym_quant_k<DT, TEAM, KU>(src, codes, params, g);
    }
  } else {
    asym_quant_v<DT, STAGED, TEAM>(src, codes, params, g, lds);
  }
}

// Chunks of a page the register-resident INT4_SYM_BLOCK save holds.
constexpr int64_t kMaxRegChunks = 16 * kBigThreads;

// The register-resident INT4_SYM_BLOCK save of pages of n8 <= kMaxRegChunks
// chunks of 8 bf16 / fp16 elements.
template <bool SLOTS>
void launch_symblock_quant(bool bf16, int64_t n8, int64_t n_pages, int n_planes, hipStream_t s,
                           const uint64_t* cache_planes, int64_t cache_stride,
                           const int32_t* block_ids, int64_t pool, const uint64_t* code_planes,
                           const uint64_t* param_planes, const SymGeom& g, const SlotRows& rows,
                           int32_t* err_flag) {
  const dim3 grid((unsigned)n_pages, (unsigned)n_planes);
  const dim3 wgrid((unsigned)((n_pages + kThreads / 64 - 1) / (kThreads / 64)),
                   (unsigned)n_planes);
#define AMF_LAUNCH(C, NT)                                                                     \
  (bf16 ? int4_symblock_quant_gather_kernel<true, C, NT, SLOTS>                               \
              <<<NT == 64 ? wgrid : grid, NT == 64 ? kThreads : NT, 0, s>>>(                  \
                  cache_planes, cache_stride, block_ids, pool, n_pages, code_planes,          \
                  param_planes, g, rows, err_flag)                                            \
        : int4_symblock_quant_gather_kernel<false, C, NT, SLOTS>                              \
              <<<NT == 64 ? wgrid : grid, NT == 64 ? kThreads : NT, 0, s>>>(                  \
                  cache_planes, cache_stride, block_ids, pool, n_pages, code_planes,          \
                  param_planes, g, rows, err_flag))
  if constexpr (!SLOTS) {
    // a wave per small page once there are pages enough to wait for: 2560 pages
    // of 1 x 128 6.2 / 6.5 us as workgroups / waves, 4096 7.8 / 7.2
    const bool many = n_pages * n_planes >= 4096;
    if (many && n8 <= 256) {
      AMF_LAUNCH(4, 64);
      return;
    }
    if (many && n8 <= kSmallPageChunks) {
      AMF_LAUNCH(8, 64);
      return;
    }
  }
  if (n8 <= 256) AMF_LAUNCH(1, 256);
  else if (n8 <= 512) AMF_LAUNCH(2, 256);
  else if (n8 <= 1024) AMF_LAUNCH(4, 256);
  else if (n8 <= 2048) AMF_LAUNCH(8, 256);
  else if (n8 <= 4096) AMF_LAUNCH(8, 512);
  else if (n8 <= 8192) AMF_LAUNCH(8, kBigThreads);
  else AMF_LAUNCH(16, kBigThreads);
#undef AMF_LAUNCH
}

// The symmetric restore (page or slot form) after validation.
template <bool SLOTS>
int launch_sym_restore(const char* who, int32_t format, int64_t n_pages, hipStream_t s,
                       const uint64_t* code_planes, const uint64_t* param_planes,
                       const uint64_t* cache_planes, int64_t cache_stride, int32_t cache_dtype,
                       const int32_t* block_ids, int64_t pool, int32_t n_planes,
                       const SymGeom& g, const SlotRows& rows, int32_t* err_flag) {
  const bool ch = format == AMF_FMT_INT4_SYM;
  if (ch && (8 * kThreads) % g.head_dim != 0)
    return fail(AMF_ERR_UNSUPPORTED, "%s: head_dim %d must divide %d", who, g.head_dim,
                8 * kThreads);
  if (n_pages == 0) return ok();
  // pages beyond 8 workgroup passes are split over workgroups of 8 passes
  const int64_t n8 = (int64_t)g.n_rows * g.head_dim / 8;
  const int parts = (int)std::max<int64_t>(1, n8 / (8 * kThreads));
  if (n_pages * parts * n_planes > 0x7FFFFFF0ll)
    return fail(AMF_ERR_UNSUPPORTED, "%s: %lld pages x %d parts x %d planes exceed one launch",
                who, (long long)n_pages, parts, n_planes);
#define AMF_LAUNCH(C, TEAM)                                                                  \
  int4_sym_dequant_scatter_kernel<DT, C, SLOTS, TEAM>                                        \
      <<<xcd_page_grid<TEAM>(n_pages * parts, n_planes), kThreads, 0, s>>>(                  \
          code_planes, param_planes, cache_planes, cache_stride, block_ids, pool, n_pages,   \
          n_planes, parts, g, rows, err_flag)
  if constexpr (!SLOTS) {
    // a wave's pass of 512 elements keeps a lane's channels as well
    if (small_restore_page(n8, cache_dtype) && (!ch || 512 % g.head_dim == 0)) {
      AMF_WITH_DTYPE(cache_dtype, if (ch) AMF_LAUNCH(true, 64); else AMF_LAUNCH(false, 64));
      return check_launch(who);
    }
  }
  AMF_WITH_DTYPE(cache_dtype,
                 if (ch) AMF_LAUNCH(true, kPageTeam); else AMF_LAUNCH(false, kPageTeam));
#undef AMF_LAUNCH
  return check_launch(who);
}

int check_int4_format(const char* who, int32_t format) {
  if (format != AMF_FMT_INT4_SYM_BLOCK && format != AMF_FMT_INT4_SYM &&
      format != AMF_FMT_INT4_ASYM_G32)
    return fail(AMF_ERR_INVALID_ARG, "%s: format %d is not an INT4 format", who, format);
  return ok();
}

int make_sym_geom(const char* who, int32_t block_size, int32_t num_heads, int32_t head_dim,
                  int32_t pps, SymGeom* g) {
  const int cpr = head_dim / 32;
  if (cpr > kThreads || (cpr & (cpr - 1)) != 0)
    return fail(AMF_ERR_UNSUPPORTED, "%s: head_dim/32 = %d must be a power of two <= %d", who,
                cpr, kThreads);
  g->n_rows = block_size * num_heads;
  g->head_dim = head_dim;
  g->cpr_log2 = __builtin_ctz(cpr);
  g->pps = pps > 0 ? pps : 1;
  return ok();
}

// lds_staged: LDS of the V save with the page staged (the page in the cache
// dtype + three fp32 tables of 16*H*G entries); lds_tables: the tables alone.
int make_asym_geom(const char* who, int32_t block_size, int32_t num_heads, int32_t head_dim,
                   int32_t elem_size, int32_t n_planes, AsymGeom* g, size_t* lds_staged,
                   size_t* lds_tables) {
  if (block_size != 16)
    return fail(AMF_ERR_UNSUPPORTED, "%s: INT4_ASYM_G32 needs block_size 16 (got %d)", who,
                block_size);
  if (n_planes % 2 != 0)
    return fail(AMF_ERR_INVALID_ARG, "%s: INT4_ASYM_G32 needs (K, V) plane pairs", who);
  g->num_heads = num_heads;
  g->head_dim = head_dim;
  g->groups = head_dim / 32;
  g->hb_code_bytes = 16 * head_dim / 2;
  g->hb_param_words = 16 * g->groups;
  auto log2_or = [](int x) { return (x & (x - 1)) == 0 ? __builtin_ctz(x) : -1; };
  g->kpr_log2 = log2_or(head_dim / 8);
  g->h_log2 = log2_or(num_heads);
  *lds_tables = (size_t)3 * 4 * 16 * num_heads * g->groups;
  *lds_staged = (size_t)16 * num_heads * head_dim * elem_size + *lds_tables;
  if (*lds_tables > (size_t)kAsymLdsBytes)
    return fail(AMF_ERR_UNSUPPORTED, "%s: %d heads x %d dims exceed the LDS parameter tables", who,
                num_heads, head_dim);
  return ok();
}

}  // namespace

extern "C" int amf_int4_dequant_scatter(int32_t format, const uint64_t* code_planes,
                                        const uint64_t* param_planes, const uint64_t* cache_planes,
                                        int64_t cache_page_stride, int32_t cache_dtype,
                                        const int32_t* block_ids, int64_t pool_pages,
                                        int32_t n_planes, int64_t n_pages, int32_t block_size,
                                        int32_t num_heads, int32_t head_dim, int32_t* err_flag,
                                        void* stream) {
  const char* who = "amf_int4_dequant_scatter";
  int rc = check_int4_format(who, format);
  if (rc) return rc;
  rc = check_codec_geometry(who, cache_planes, cache_page_stride, cache_dtype, block_ids,
                            pool_pages, code_planes, param_planes, n_planes, n_pages, block_size,
                            num_heads, head_dim);
  if (rc) return rc;
  hipStream_t s = as_stream(stream);
  if (n_pages * n_planes > 0x7FFFFFF0ll)
    return fail(AMF_ERR_UNSUPPORTED, "%s: %lld pages x %d planes exceed one launch", who,
                (long long)n_pages, n_planes);
  if (format == AMF_FMT_INT4_ASYM_G32) {
    AsymGeom g;
    size_t lds_staged, lds_tables;
    if ((rc = make_asym_geom(who, block_size, num_heads, head_dim, cache_elem_bytes(cache_dtype),
                             n_planes, &g, &lds_staged, &lds_tables)))
      return rc;
    if (n_pages == 0) return ok();
#define AMF_LAUNCH(TEAM, VSPLIT, P2)                                                           \
  AMF_WITH_DTYPE(cache_dtype,                                                                  \
                 int4_asym_dequant_scatter_kernel<DT, TEAM, VSPLIT, P2>                        \
                 <<<dim3((unsigned)((n_pages + kThreads / TEAM - 1) / (kThreads / TEAM)),      \
                         (unsigned)n_planes),                                                  \
                    kThreads, 0, s>>>(code_planes, param_planes, cache_planes,                 \
                                      cache_page_stride, block_ids, pool_pages, n_pages, g,    \
                                      err_flag))
    const int64_t v_items = (int64_t)num_heads * head_dim / 8 * 2;
    const bool small = cache_dtype != AMF_DTYPE_F32 && 8 * v_items <= kSmallPageChunks;
    if (g.kpr_log2 < 0 || g.h_log2 < 0) AMF_LAUNCH(256, 1, false);
    else if (!small && v_items < kThreads) AMF_LAUNCH(256, 2, true);
    else if (!small) AMF_LAUNCH(256, 1, true);
    else if (v_items <= 16) AMF_LAUNCH(64, 4, true);
    else if (v_items <= 32) AMF_LAUNCH(64, 2, true);
    else AMF_LAUNCH(64, 1, true);
#undef AMF_LAUNCH
    return check_launch(who);
  }
  SymGeom g;
  if ((rc = make_sym_geom(who, block_size, num_heads, head_dim, 1, &g))) return rc;
  return launch_sym_restore<false>(who, format, n_pages, as_stream(stream), code_planes,
                                   param_planes, cache_planes, cache_page_stride, cache_dtype,
                                   block_ids, pool_pages, n_planes, g, SlotRows{}, err_flag);
}

extern "C" int amf_int4_dequant_scatter_slots(
    int32_t format, const uint64_t* code_planes, const uint64_t* param_planes,
    const uint64_t* cache_planes, int64_t cache_page_stride, int32_t cache_block,
    int32_t cache_dtype, const int64_t* slot_mapping, int64_t pool_slots, int32_t n_planes,
    int64_t n_slots, int32_t page_tokens, int32_t num_heads, int32_t head_dim, int32_t* err_flag,
    void* stream) {
  const char* who = "amf_int4_dequant_scatter_slots";
  int rc = check_int4_format(who, format);
  if (rc) return rc;
  if (format == AMF_FMT_INT4_ASYM_G32)
    return fail(AMF_ERR_UNSUPPORTED, "%s: the symmetric formats only", who);
  SlotRows rows;
  int64_t n_pages = 0;
  rc = check_slot_codec(who, cache_planes, cache_page_stride, cache_block, cache_dtype,
                        slot_mapping, pool_slots, code_planes, param_planes, n_planes, n_slots,
                        page_tokens, num_heads, head_dim, &rows, &n_pages);
  if (rc) return rc;
  SymGeom g;
  if ((rc = make_sym_geom(who, page_tokens, num_heads, head_dim, 1, &g))) return rc;
  return launch_sym_restore<true>(who, format, n_pages, as_stream(stream), code_planes,
                                  param_planes, cache_planes, cache_page_stride, cache_dtype,
                                  nullptr, 0, n_planes, g, rows, err_flag);
}

extern "C" int amf_int4_quant_gather_slots(
    int32_t format, const uint64_t* cache_planes, int64_t cache_page_stride, int32_t cache_block,
    int32_t cache_dtype, const int64_t* slot_mapping, int64_t pool_slots,
    const uint64_t* code_planes, const uint64_t* param_planes, int32_t n_planes, int64_t n_slots,
    int32_t page_tokens, int32_t num_heads, int32_t head_dim, int32_t* err_flag, void* stream) {
  const char* who = "amf_int4_quant_gather_slots";
  int rc = check_int4_format(who, format);
  if (rc) return rc;
  SlotRows rows;
  int64_t n_pages = 0;
  rc = check_slot_codec(who, cache_planes, cache_page_stride, cache_block, cache_dtype,
                        slot_mapping, pool_slots, code_planes, param_planes, n_planes, n_slots,
                        page_tokens, num_heads, head_dim, &rows, &n_pages);
  if (rc) return rc;
  SymGeom g;
  if ((rc = make_sym_geom(who, page_tokens, num_heads, head_dim, 1, &g))) return rc;
  const int64_t n8 = (int64_t)g.n_rows * g.head_dim / 8;
  if (format != AMF_FMT_INT4_SYM_BLOCK || cache_dtype == AMF_DTYPE_F32 || n8 > kMaxRegChunks)
    return fail(AMF_ERR_UNSUPPORTED,
                "%s: INT4_SYM_BLOCK pages of at most %lld bf16 / fp16 elements only", who,
                (long long)(8 * kMaxRegChunks));
  if (n_pages == 0) return ok();
  launch_symblock_quant<true>(cache_dtype == AMF_DTYPE_BF16, n8, n_pages, n_planes,
                              as_stream(stream), cache_planes, cache_page_stride, nullptr, 0, code_planes,
                              param_planes, g, rows, err_flag);
  return check_launch(who);
}

extern "C" int amf_int4_quant_gather(int32_t format, const uint64_t* cache_planes,
                                     int64_t cache_page_stride, int32_t cache_dtype,
                                     const int32_t* block_ids, int64_t pool_pages,
                                     const uint64_t* code_planes, const uint64_t* param_planes,
                                     int32_t n_planes, int32_t planes_per_scale, int64_t n_pages,
                                     int32_t block_size, int32_t num_heads, int32_t head_dim,
                                     float* workspace,
                                     int64_t workspace_bytes, int32_t* err_flag, void* stream) {
  const char* who = "amf_int4_quant_gather";
  int rc = check_int4_format(who, format);
  if (rc) return rc;
  rc = check_codec_geometry(who, cache_planes, cache_page_stride, cache_dtype, block_ids,
                            pool_pages, code_planes, param_planes, n_planes, n_pages, block_size,
                            num_heads, head_dim);
  if (rc) return rc;
  const bool bf16 = cache_dtype == AMF_DTYPE_BF16;
  hipStream_t s = as_stream(stream);
  dim3 grid((unsigned)n_pages, (unsigned)n_planes);
  if (format == AMF_FMT_INT4_ASYM_G32) {
    AsymGeom g;
    size_t lds_staged, lds_tables;
    if ((rc = make_asym_geom(who, block_size, num_heads, head_dim, cache_elem_bytes(cache_dtype),
                             n_planes, &g, &lds_staged, &lds_tables)))
      return rc;
    if (n_pages == 0) return ok();
    const bool staged = lds_staged <= (size_t)kAsymLdsBytes;
#define AMF_LAUNCH(ST, TEAM, KU)                                                               \
  int4_asym_quant_gather_kernel<DT, ST, TEAM, KU>                                              \
      <<<dim3((unsigned)((n_pages + kThreads / TEAM - 1) / (kThreads / TEAM)),                 \
              (unsigned)n_planes),                                                             \
         kThreads, (ST ? lds_staged : lds_tables) * (kThreads / TEAM), s>>>(                   \
          cache_planes, cache_page_stride, block_ids, pool_pages, n_pages, code_planes,        \
          param_planes, g, (int)(ST ? lds_staged : lds_tables), err_flag)
    // four small pages to a workgroup while their staging fits
    if (16 * num_heads * head_dim <= 8 * kSmallPageChunks &&
        4 * lds_staged <= (size_t)kAsymLdsBytes) {
      AMF_WITH_DTYPE(cache_dtype, if (16 * num_heads * g.groups <= 64) AMF_LAUNCH(true, 64, 1);
                     else AMF_LAUNCH(true, 64, kKSaveUnroll));
      return check_launch(who);
    }
    AMF_WITH_DTYPE(cache_dtype, if (staged) AMF_LAUNCH(true, kThreads, kKSaveUnroll);
                   else AMF_LAUNCH(false, kThreads, kKSaveUnroll));
#undef AMF_LAUNCH
    return check_launch(who);
  }
  if (format == AMF_FMT_INT4_SYM &&
      (planes_per_scale <= 0 || n_planes % planes_per_scale != 0))
    return fail(AMF_ERR_INVALID_ARG, "%s: planes_per_scale %d does not divide n_planes %d", who,
                planes_per_scale, n_planes);
  SymGeom g;
  if ((rc = make_sym_geom(who, block_size, num_heads, head_dim, planes_per_scale, &g))) return rc;
  if (n_pages == 0) return ok();
  if (format == AMF_FMT_INT4_SYM_BLOCK) {
    const int64_t n8 = (int64_t)g.n_rows * g.head_dim / 8;
    // Pages that fit lanes' registers (at most kMaxRegChunks chunks) take the
    // single-read kernel; larger pages and fp32 caches the two-read one.
    if (cache_dtype == AMF_DTYPE_F32 || n8 > kMaxRegChunks) {
#define AMF_LAUNCH(DT, NT, U)                                                          \
  int4_symblock_quant_looped_kernel<DT, NT, U><<<grid, NT, 0, s>>>(                    \
      cache_planes, cache_page_stride, block_ids, pool_pages, code_planes, param_planes, g, err_flag)
      if (n8 <= kLoopChunks)
        AMF_LAUNCH(AMF_DTYPE_F32, kThreads, 1);
      else
        AMF_WITH_DTYPE(cache_dtype, AMF_LAUNCH(DT, kBigThreads, 4));
#undef AMF_LAUNCH
      return check_launch(who);
    }
    launch_symblock_quant<false>(bf16, n8, n_pages, n_planes, s, cache_planes, cache_page_stride, block_ids,
                                 pool_pages, code_planes, param_planes, g, SlotRows{}, err_flag);
    return check_launch(who);
  }
  // AMF_FMT_INT4_SYM: absmax pass, then the quant pass (which also writes the fp16 scales).
  if (head_dim > 1024) return fail(AMF_ERR_UNSUPPORTED, "%s: head_dim > 1024", who);
  const int64_t need = amf_quant_workspace_bytes(format, n_planes, planes_per_scale, head_dim);
  if (!workspace || workspace_bytes < need)
    return fail(AMF_ERR_WORKSPACE, "%s: needs %lld workspace bytes", who, (long long)need);
  uint32_t* ws = reinterpret_cast<uint32_t*>(workspace);
  const int64_t n_ws = need / 4;
  fill_u32_kernel<<<(unsigned)((n_ws + 255) / 256), 256, 0, s>>>(ws, n_ws, 0u);
#ifndef AMF_ABSMAX_WGS
#define AMF_ABSMAX_WGS 64
#endif
  dim3 rgrid((unsigned)(n_pages < AMF_ABSMAX_WGS ? n_pages : AMF_ABSMAX_WGS), (unsigned)n_planes);
  const int64_t lane_chunks = ((int64_t)g.n_rows * head_dim / 8 + kThreads - 1) / kThreads;
#define AMF_LAUNCH(P)                                                                   \
  int4_channel_absmax_kernel<DT, P><<<rgrid, kThreads, 0, s>>>(                         \
      cache_planes, cache_page_stride, block_ids, pool_pages, n_pages, g, ws, err_flag)
  // several pages at a time where a workgroup has more than one (fp32, 32 x 300
  // pages of 3 x 64: 102 / 109 us one / four at a time)
  const int64_t step =
      cache_dtype != AMF_DTYPE_F32 && n_pages > AMF_ABSMAX_WGS ? lane_chunks : 0;
  AMF_WITH_DTYPE(cache_dtype, if (step == 1) AMF_LAUNCH(8);
                 else if (step == 2) AMF_LAUNCH(4); else AMF_LAUNCH(1));
#undef AMF_LAUNCH
#define AMF_LAUNCH(TEAM)                                                                      \
  AMF_WITH_DTYPE(cache_dtype, int4_channel_quant_gather_kernel<DT, TEAM>                      \
                 <<<dim3((unsigned)((n_pages + kThreads / TEAM - 1) / (kThreads / TEAM)),     \
                         (unsigned)n_planes),                                                 \
                    kThreads, 0, s>>>(cache_planes, cache_page_stride, block_ids, pool_pages, \
                                      n_pages, code_planes, param_planes, g, ws, err_flag))
  // a wave's pass of 512 elements keeps a lane's channels as well
  // (fp32: up to half the chunks, 32 x 300 pages of 1 x 64 58 / 47 us with a
  // workgroup / a wave, of 3 x 64 105 / 110)
  const int64_t small = kSmallPageChunks / (cache_dtype == AMF_DTYPE_F32 ? 2 : 1);
  if ((int64_t)g.n_rows * head_dim <= 8 * small && 512 % head_dim == 0) AMF_LAUNCH(64);
  else AMF_LAUNCH(kThreads);
#undef AMF_LAUNCH
  return check_launch(who);
}
