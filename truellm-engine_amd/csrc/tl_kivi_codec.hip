// tl_kivi_codec.hip -- KIVI INT4 codecs for gfx950.
//
// 1. The reference vector codec (kivi_cache.cu:23-198): per vector, the top
//    n_outliers |x| channels stored raw as fp16 with a u8 index, the other
//    channels min/max quantised to 4 bits in groups of group_size with an
//    fp16 (step, zero) pair.  Bit-exact with the reference's fp32 IEEE
//    arithmetic: correctly rounded division, rint, no contraction of
//    (x - gmin) * scale, and the fused multiply-add nvcc forms for
//    nibble * step + zero on decode.
//
// 2. The paged KIVI format: per kv head, a page holds 32 tokens quantised
//    with the same group quantiser, K per channel over the 32 tokens and V
//    per token over groups of 32 channels (KIVI's key/value granularities,
//    config_schema.h:122-129), laid out so a dequantised dword is a ready
//    MFMA operand (see tl_kivi.hpp).  One workgroup builds one page.
#include "tl_device.hpp"
#include "tl_internal.hpp"
#include "tl_kivi.hpp"
#include "tl_kivi_page.hpp"

#include <float.h>

#include <type_traits>

namespace tl {

namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// Least and greatest of packed halves, element by element; a NaN stays.
__device__ __forceinline__ half2v pk_min(half2v a, half2v b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ half2v pk_max(half2v a, half2v b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ half2v as_half2(uint32_t w) { return __builtin_bit_cast(half2v, w); }

// The scans of group_params' caller start from +-FLT_MAX, skip NaN and keep
// the first of equal values.  Over finite values that is the plain least and
// greatest value, but for the sign of a zero minimum: such groups, and those
// with a NaN or an infinity, are scanned in order.
__device__ __forceinline__ bool scan_in_order(float mn, float mx) {
  return !(mn > -FLT_MAX && mx < FLT_MAX) || mn == 0.0f;
}

// The codes of quantise over a group of finite values, before packing: the
// code plus kCodeBias.  x - min is exact in one rounding from the half, the
// product is rounded by itself (no contraction), and it lies in [0, LEVELS]
// up to a rounding, so adding 2^23 leaves its nearest-even integer in the low
// mantissa bits and no clamp is needed.
constexpr uint32_t kCodeBias = 0x4B000000u;                      // 2^23 in fp32
__device__ __forceinline__ uint32_t biased_code(_Float16 x, float one, float gmin, float scale) {
#pragma clang fp contract(off)
  const float d = __builtin_fmaf((float)x, one, -gmin);
  const float p = d * scale;
  return __float_as_uint(p + 8388608.0f);
}

// ---------------------------------------------------------------------------
// The reference vector codec.  8 lanes share a vector, a 64-thread workgroup
// takes 8 vectors: 16 384 vectors are 2048 wavefronts, two per SIMD.  The
// sequential part of the format (which slot an outlier ends in) is kept
// sequential over the channels, but each of its steps is the work of 8
// lanes; the rest (ranks, groups, codes) is spread over them.  Rows and
// records go through LDS, so that memory sees whole lines.  Bound: the
// 128-step scan's dependency chain (about 6 vector instructions a step at up
// to 8 outliers) and the few wavefronts there are to hide the rest.  Compress
// and decompress of 16 384 vectors of 128 channels, 8 outliers, groups of 16:
// 16.8 us; with a minimum over the slots in each step, values widened one by
// one and divisions in the copies 23.8 us; one thread per vector, with its
// slots, flags and values in scratch memory, 1488 us.
// ---------------------------------------------------------------------------
constexpr int kVecLanes = 8, kVecVecs = kWave / kVecLanes;
constexpr int kVecRow = kKiviMaxHeadDim + 8;          // halves per LDS row (16-byte rows, shifted banks)
// Bytes of a record that are written: 3 per outlier, then per group its
// codes and 4 parameter bytes; at most that of 64 outliers and, for groups
// of 2, the other 64 channels and one group left over.
constexpr int kVecRecMax = 3 * kKiviMaxOutliers + ((kKiviMaxHeadDim - kKiviMaxOutliers) / 2 + 1) * 5;
constexpr int kVecRec = (kVecRecMax + 3) / 4 * 4;

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
}
constexpr int kDppShr1 = 0x111;          // lane i <- i - 1 within each row of 16
constexpr int kDppBcast = 0x150;         // + n: lane n of each row to all of it
// Lane 7 of the vector's 8 lanes to all of them (banks 0, 1 hold the row's
// first vector, 2, 3 its second).
__device__ __forceinline__ uint32_t last8(uint32_t v) {
  const int lo = __builtin_amdgcn_update_dpp((int)v, (int)v, kDppBcast + 7, 0xF, 0x3, false);
  return (uint32_t)__builtin_amdgcn_update_dpp(lo, (int)v, kDppBcast + 15, 0xF, 0xC, false);
}
// Over the 8 lanes of a vector.
__device__ __forceinline__ uint32_t or8(uint32_t v) {
  v |= dpp_u32<kDppXor1>(v);
  v |= dpp_u32<kDppXor2>(v);
  return v | dpp_u32<kDppHalfMirror>(v);
}

// A vector's row of d halves between memory and LDS, by its own 8 lanes;
// 16-byte accesses where d is a multiple of 8 and the base 16-byte aligned.
__device__ __forceinline__ void vec_row_in(const uint16_t* src, uint16_t* row, int d, bool wide, int l8) {
  if (wide) {
    for (int i = 8 * l8; i < d; i += 8 * kVecLanes) *reinterpret_cast<u32x4*>(row + i) = load16(src + i);
  } else {
    for (int i = l8; i < d; i += kVecLanes) row[i] = src[i];
  }
}
__device__ __forceinline__ void vec_row_out(uint16_t* dst, const uint16_t* row, int d, bool wide, int l8) {
  if (wide) {
    for (int i = 8 * l8; i < d; i += 8 * kVecLanes)
      *reinterpret_cast<u32x4*>(dst + i) = *reinterpret_cast<const u32x4*>(row + i);
  } else {
    for (int i = l8; i < d; i += kVecLanes) dst[i] = row[i];
  }
}
// The same for a record's n bytes, in dwords where `dwords`.
__device__ __forceinline__ void vec_bytes(uint8_t* dst, const uint8_t* src, int n, bool dwords, int l8) {
  int done = 0;
  if (dwords) {
#pragma unroll 4
    for (int i = 4 * l8; i + 4 <= n; i += 4 * kVecLanes)
      *reinterpret_cast<uint32_t*>(dst + i) = *reinterpret_cast<const uint32_t*>(src + i);
    done = n & ~3;
  }
  for (int i = done + l8; i < n; i += kVecLanes) dst[i] = src[i];
}

// Bytes of a record that are written (the stride can be longer: the last
// group's missing codes).
__host__ __device__ inline int kivi_record_bytes(int head_dim, int n_outliers, int group_size) {
  const int n_res = head_dim - n_outliers;
  const int n_groups = (n_res + group_size - 1) / group_size;
  if (n_groups == 0) return 3 * n_outliers;
  const int last = n_res - (n_groups - 1) * group_size;
  return 3 * n_outliers + (n_groups - 1) * (group_size / 2 + 4) + (last + 1) / 2 + 4;
}

// SPL: outlier slots per lane (slot i * 8 + lane), at least n_outliers / 8.
template <int SPL>
__global__ __launch_bounds__(kWave) void kivi_vec_compress_kernel(
    const uint16_t* __restrict__ in, uint8_t* __restrict__ out, int n_vecs, int head_dim, int n_outliers,
    int group_size, int stride, int rec_bytes, bool wide, bool dwords) {
  __shared__ __attribute__((aligned(16))) uint16_t s_x[kVecVecs * kVecRow];
  __shared__ __attribute__((aligned(16))) uint16_t s_res[kVecVecs * kVecRow];
  __shared__ __attribute__((aligned(16))) uint8_t s_rec[kVecVecs * kVecRec];
  const int lane = threadIdx.x, l8 = lane % kVecLanes, vi = lane / kVecLanes;
  const int64_t v0 = (int64_t)blockIdx.x * kVecVecs;
  const int nv = (int)min<int64_t>(kVecVecs, n_vecs - v0);
  uint16_t* x = s_x + vi * kVecRow;
  uint16_t* res = s_res + vi * kVecRow;
  uint8_t* rec = s_rec + vi * kVecRec;
  if (vi < nv) vec_row_in(in + (v0 + vi) * head_dim, x, head_dim, wide, l8);
  // channels up to the next multiple of 8: NaN, which the scan skips
  if (vi < nv && head_dim + l8 < (head_dim + 7) / 8 * 8) x[head_dim + l8] = 0x7FFF;
  __syncthreads();

  // Top-n_outliers |x| by the reference's replace-the-first-minimum scan.  A
  // slot is one word: (|x| as ordered bits + 1, 0 when empty) << 16 | slot
  // << 8 | 255 - channel.  The words stand in descending order over places
  // 8 i + l8 (the last n_outliers of them), so the first slot of least
  // magnitude is the last place, and its slot goes to the channel that
  // replaces it: that word enters at its place and those below it move on
  // by one, all of which is the median of (own word, word before, new word).
  // A channel no greater than the least falls below the last place: at equal
  // magnitude its word has that slot and a smaller channel field.
  uint32_t key[SPL];
#pragma unroll
  for (int i = 0; i < SPL; ++i) {
    const int s = SPL * kVecLanes - 1 - (i * kVecLanes + l8);
    key[i] = s < n_outliers ? (uint32_t)s << 8 | 0xFFu : 0xFFFFFFFFu;
  }
  if (n_outliers > 0) {
    const uint32_t top = l8 == 0 ? 0xFFFFFFFFu : 0u;
    for (int d0 = 0; d0 < head_dim; d0 += 8) {
      const u32x4 c = *reinterpret_cast<const u32x4*>(x + d0);
      const uint32_t w[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t h = (w[e / 2] >> (16 * (e & 1))) & 0x7FFFu;
        const uint32_t m = (h <= 0x7C00u ? (h + 1u) << 16 : 0u) | (uint32_t)(255 - d0 - e);   // NaN is never greater
        uint32_t last[SPL], before[SPL];
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
          last[i] = last8(key[i]);
          before[i] = dpp_u32<kDppShr1>(key[i]) | top;
          if (i > 0) before[i] = l8 == 0 ? last[i - 1] : before[i];
        }
        const uint32_t put = (last[SPL - 1] & 0xFF00u) | m;
#pragma unroll
        for (int i = 0; i < SPL; ++i) key[i] = max(key[i], min(put, before[i]));
      }
    }
  }

  // the outliers' records, and the mask of their channels (an empty slot
  // holds channel 0, as the reference's does)
  uint32_t mask[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < SPL; ++i) {
    if (key[i] != 0xFFFFFFFFu) {
      const int s = key[i] >> 8 & 0xFF, ch = 255 - (key[i] & 0xFF);
      const uint16_t h = x[ch];
      rec[3 * s] = (uint8_t)ch;
      rec[3 * s + 1] = (uint8_t)(h & 0xff);
      rec[3 * s + 2] = (uint8_t)(h >> 8);
#pragma unroll
      for (int w = 0; w < 4; ++w) mask[w] |= ch / 32 == w ? 1u << (ch % 32) : 0u;
    }
  }
#pragma unroll
  for (int w = 0; w < 4; ++w) mask[w] = or8(mask[w]);

  // the other channels, ascending: lane l8 places channels 16 l8 .. + 15
  const int n_res = head_dim - n_outliers;
  {
    const uint32_t mine = l8 < 2 ? mask[0] : l8 < 4 ? mask[1] : l8 < 6 ? mask[2] : mask[3];
    int before = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) before += w < l8 / 2 ? __builtin_popcount(mask[w]) : 0;
    if (l8 & 1) before += __builtin_popcount(mine & 0xFFFFu);
    const uint32_t own = (l8 & 1) ? mine >> 16 : mine;
    int r = 16 * l8 - before;
    const u32x4 c[2] = {*reinterpret_cast<const u32x4*>(x + 16 * l8), *reinterpret_cast<const u32x4*>(x + 16 * l8 + 8)};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const bool put = !((own >> e) & 1u) && 16 * l8 + e < head_dim;
      if (put && r < n_res) res[r] = (uint16_t)(word(c[e / 8], e % 8 / 2) >> (16 * (e & 1)));
      r += put ? 1 : 0;
    }
  }
  __syncthreads();

  const int n_groups = (n_res + group_size - 1) / group_size;
  for (int g = l8; g < n_groups; g += kVecLanes) {
    const int g0 = g * group_size, g1 = min(g0 + group_size, n_res);
    // groups start at even indices: pairs are whole words
    const uint32_t* pairs = reinterpret_cast<const uint32_t*>(res + g0);
    const int n = g1 - g0;
    uint8_t* p = rec + 3 * n_outliers + g * (group_size / 2 + 4);
    float gmin = FLT_MAX, gmax = -FLT_MAX;
    bool in_order = true;
    if (n % 2 == 0) {
      half2v a = as_half2(pairs[0]), b = a;
#pragma unroll 4
      for (int i = 1; i < n / 2; ++i) {
        a = pk_min(a, as_half2(pairs[i]));
        b = pk_max(b, as_half2(pairs[i]));
      }
      gmin = (float)__builtin_elementwise_minimum(a.x, a.y);
      gmax = (float)__builtin_elementwise_maximum(b.x, b.y);
      in_order = scan_in_order(gmin, gmax);
    }
    if (in_order) {
      gmin = FLT_MAX;
      gmax = -FLT_MAX;
      for (int i = 0; i < n; ++i) {
        const float a = f16_to_f32(res[g0 + i]);
        if (a < gmin) gmin = a;
        if (a > gmax) gmax = a;
      }
    }
    const GroupQ q = group_params(gmin, gmax);
    if (!in_order) {
#pragma unroll 4
      for (int i = 0; i < n / 2; ++i) {
        const half2v w = as_half2(pairs[i]);
        p[i] = (uint8_t)(biased_code(w.x, 1.0f, q.gmin, q.scale) + (biased_code(w.y, 1.0f, q.gmin, q.scale) << 4));
      }
    } else {
      for (int i = 0; i < n; i += 2) {
        const int q0 = quantise(f16_to_f32(res[g0 + i]), q);
        const int q1 = i + 1 < n ? quantise(f16_to_f32(res[g0 + i + 1]), q) : 0;
        p[i / 2] = (uint8_t)((q1 << 4) | q0);
      }
    }
    p += (n + 1) / 2;
    p[0] = (uint8_t)(q.step & 0xff); p[1] = (uint8_t)(q.step >> 8);
    p[2] = (uint8_t)(q.zero & 0xff); p[3] = (uint8_t)(q.zero >> 8);
  }
  __syncthreads();

  if (vi < nv) vec_bytes(out + (v0 + vi) * stride, rec, rec_bytes, dwords, l8);
}

__global__ __launch_bounds__(kWave) void kivi_vec_decompress_kernel(
    const uint8_t* __restrict__ in, uint16_t* __restrict__ out, int n_vecs, int head_dim, int n_outliers,
    int group_size, int stride, int rec_bytes, bool wide, bool dwords) {
  __shared__ __attribute__((aligned(16))) uint16_t s_x[kVecVecs * kVecRow];
  __shared__ __attribute__((aligned(16))) uint16_t s_res[kVecVecs * kVecRow];
  __shared__ __attribute__((aligned(16))) uint8_t s_rec[kVecVecs * kVecRec];
  const int lane = threadIdx.x, l8 = lane % kVecLanes, vi = lane / kVecLanes;
  const int64_t v0 = (int64_t)blockIdx.x * kVecVecs;
  const int nv = (int)min<int64_t>(kVecVecs, n_vecs - v0);
  uint8_t* rec = s_rec + vi * kVecRec;
  uint16_t* x = s_x + vi * kVecRow;
  uint16_t* res = s_res + vi * kVecRow;
  if (vi < nv) vec_bytes(rec, in + (v0 + vi) * stride, rec_bytes, dwords, l8);
  __syncthreads();
  const int n_res = head_dim - n_outliers;
  if (vi < nv) {
    // the groups' values, ascending, a group per lane
    const int n_groups = (n_res + group_size - 1) / group_size;
    for (int g = l8; g < n_groups; g += kVecLanes) {
      const int n = min(group_size, n_res - g * group_size), nb = (n + 1) / 2;
      const uint8_t* pack = rec + 3 * n_outliers + g * (group_size / 2 + 4);
      const uint8_t* p = pack + nb;
      const float st = f16_to_f32((uint16_t)(p[0] | (p[1] << 8)));
      const float ze = f16_to_f32((uint16_t)(p[2] | (p[3] << 8)));
      // groups start at even indices: pairs are whole words (the last pair's
      // second value is not read when there is none)
      uint32_t* pairs = reinterpret_cast<uint32_t*>(res + g * group_size);
#pragma unroll 4
      for (int i = 0; i < nb; ++i) {
        const int b = pack[i];
        pairs[i] = f32_to_f16(__builtin_fmaf((float)(b & 0x0f), st, ze)) |
                   (uint32_t)f32_to_f16(__builtin_fmaf((float)(b >> 4), st, ze)) << 16;
      }
    }
  }
  __syncthreads();
  if (vi < nv) {
    // lane l8 owns channels 16 l8 .. + 15; every lane reads every outlier,
    // so that of two for one channel the later stands
    uint32_t own = 0;
#pragma unroll 4
    for (int i = 0; i < n_outliers; ++i) {
      const int ch = rec[3 * i];
      const uint16_t h = (uint16_t)(rec[3 * i + 1] | (rec[3 * i + 2] << 8));
      if (ch / 16 == l8 && ch < head_dim) {
        own |= 1u << (ch % 16);
        x[ch] = f32_to_f16(f16_to_f32(h));
      }
    }
    // the other channels' ranks: those of the lanes before first
    const int owned = max(min(16 * l8 + 16, head_dim) - 16 * l8, 0);
    const int free_own = owned - __builtin_popcount(own);
    int before = 0;
#pragma unroll
    for (int o = 1; o < kVecLanes; ++o) {
      const int n = __shfl(free_own, (lane & ~(kVecLanes - 1)) + ((l8 - o) & (kVecLanes - 1)), kWave);
      before += o <= l8 ? n : 0;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      // channels past the values (two outliers for one channel) read as zero
      const int r = before + e - __builtin_popcount(own & ((1u << e) - 1u));
      const uint16_t v = r < n_res ? res[r] : (uint16_t)0;
      if (e < owned && !((own >> e) & 1u)) x[16 * l8 + e] = v;
    }
  }
  __syncthreads();
  if (vi < nv) vec_row_out(out + (v0 + vi) * head_dim, x, head_dim, wide, l8);
}

// ---------------------------------------------------------------------------
// Paged KIVI append: the new token of each (sequence, kv head) into the fp16
// pool [N, n_kv, 128, BS], and the page (32 tokens x 128 channels) that it
// completes, or, with build-ahead, its piece of the next page.
// ---------------------------------------------------------------------------
template <int BITS>
__global__ __launch_bounds__(128) void kivi_append_kernel(PageJob j) {
  __shared__ __attribute__((aligned(16))) KiviBuildSmem<BITS> sm;
  const int tid = threadIdx.x;
  const int kvh = blockIdx.x % j.num_kv_heads, seq = blockIdx.x / j.num_kv_heads;
  const int L = j.seq_lens[seq];
  const int lq = kivi_quantized_len(L, j.residual_length);
  kivi_append_token<128>(j, seq, kvh, tid);
  if (j.build_ahead) {
    // the pages this append completes were written in pieces by the
    // appends before it; this one writes its piece of the next page:
    // wavefront 0 stages its fp16, then each wavefront quantises two of
    // its quarters
    int ahead_page;
    const int piece = kivi_ahead_piece(L, j.residual_length, ahead_page);
    if (piece < 0) return;
    __shared__ int s_pid;
    uint16_t* raw = reinterpret_cast<uint16_t*>(&sm.qk[0][0]);
    const int lane = tid % kWave, wave = tid / kWave;
    if (wave == 0) {
      KiviPiece pc = kivi_piece_plan(j, seq, ahead_page, piece, lane);
      kivi_piece_load(j, pc, kvh, ahead_page, lane);
      kivi_piece_stage(pc, lane, raw);
      if (lane == 0) s_pid = pc.piece >= 0 ? pc.pid : -1;
    }
    __syncthreads();
    const int pid = s_pid;
    if (pid < 0) return;
    for (int q = wave; q < 4; q += 128 / kWave)
      kivi_piece_quarter<BITS>(j, pid, piece, kvh, q, lane, kivi_piece_quarter_values(piece, q, lane, raw),
                               &sm.qv[0][0] + 256 * q);
    return;
  }
  if (lq == 0 || lq == kivi_quantized_len(L - 1, j.residual_length)) return;
  kivi_build_page<128, BITS>(sm, j, seq, kvh, lq / kKiviPageTokens - 1, L, tid);
}

// ---------------------------------------------------------------------------
// Prefix build: every page of a prefix, one workgroup of two wavefronts per
// (page, kv head), one on K and one on V, with the values in registers.
//
// kivi_build_page above gives one thread one group of 32 values that it reads
// from LDS, and runs each value through some 16 VALU instructions and four
// LDS accesses of a byte or two; that, and 30 KiB of LDS per workgroup, took
// 80 us for a build whose bytes need 26.  Here a value costs about 5: min and
// max over packed halves three at a time, x - min straight from the half
// (v_fma_mix), one multiply, the rounding as an addition of 2^23 and one
// shift-add into the packed codes; codes reach their page dwords by exchanges
// between lanes of a quad or octet.  The page's bytes are kivi_build_page's.
//
// 8 prompts of 4096 tokens, 8 kv heads, INT4 (171 MB): 37.9 us = 4.5 TB/s
// (79.9 before).  Held to fewer registers for 5 or 6 wavefronts per SIMD (116
// here, 4) it spills: 46 and 54 us.
// ---------------------------------------------------------------------------

// N codes of BITS each (8 of 4 bits, 4 of 8) into a dword, code i at bit
// shift_of(i).
template <int BITS, int N, bool IN_ORDER, class Value, class Group, class Shift>
__device__ __forceinline__ uint32_t pack_codes(float one, Value value, Group group, Shift shift_of) {
  uint32_t acc = 0;
  if constexpr (IN_ORDER) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      acc |= (uint32_t)quantise<KiviFmt<BITS>::kLevels>((float)value(i), group(i)) << shift_of(i);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) acc -= kCodeBias << shift_of(i);
#pragma unroll
    for (int i = 0; i < N; ++i)
      acc += biased_code(value(i), one, group(i).gmin, group(i).scale) << shift_of(i);
  }
  return acc;
}

// Exchanges with lane ^ M of one bit of the element position in a dword: the
// upper of each pair of 16-bit halves, bytes or nibbles goes to the lane with
// bit M clear, the lower one to the other.
template <int M>
__device__ __forceinline__ uint32_t swap_halves(uint32_t own, bool up) {
  return __builtin_amdgcn_perm(own, lane_xor_u<M>(own), up ? 0x07060302u : 0x01000504u);
}
template <int M>
__device__ __forceinline__ uint32_t swap_bytes(uint32_t own, bool up) {
  return __builtin_amdgcn_perm(own, lane_xor_u<M>(own), up ? 0x07030501u : 0x02060004u);
}
template <int M>
__device__ __forceinline__ uint32_t swap_nibbles(uint32_t own, bool up) {
  const uint32_t o = lane_xor_u<M>(own), mask = up ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
  return (own & mask) | (__builtin_amdgcn_alignbit(o, o, up ? 4 : 28) & ~mask);
}

// The block of token `tok` of a sequence, or -1.
__device__ __forceinline__ int block_of_token(const PageJob& j, const int32_t* btab, int tok) {
  const int lb = tok / j.block_size;
  const int phys = lb < j.max_blocks_per_seq ? btab[lb] : -1;
  return phys < 0 || phys >= j.num_blocks ? -1 : phys;
}
__device__ __forceinline__ const uint16_t* pool_at(const PageJob& j, const uint16_t* pool, int phys, int kvh, int c,
                                                   int tok) {
  return pool + (((int64_t)phys * j.num_kv_heads + kvh) * kKiviHead + c) * j.block_size + tok % j.block_size;
}

// K of a page.  Lane (tt, jj, ci) = (lane / 32, lane / 8 % 4, lane % 8) takes
// tokens 16 tt .. 16 tt + 15 of channels 8 (jj + 4 m) + ci, m = 0 .. 3: the
// channels of one chunk position, whose codes of 8 tokens the lanes of an
// octet exchange for 8 channels of a token each.
template <int BITS>
__device__ __forceinline__ void build_page_k(const PageJob& j, const int32_t* btab, int kvh, int page, uint8_t* dst,
                                             uint32_t* stage, int lane) {
  using F = KiviFmt<BITS>;
  constexpr int LV = F::kLevels, PER = 32 / BITS, DW = 16 / PER;   // codes of a dword, dwords of 16 tokens
  const int tt = lane >> 5, jj = lane >> 3 & 3, ci = lane & 7;
  const int tok = page * kKiviPageTokens + 16 * tt;
  const int phys[2] = {block_of_token(j, btab, tok), block_of_token(j, btab, tok + 8)};
  uint32_t x[4][8];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const u32x4 v = load16(pool_at(j, j.k_cache, max(phys[r], 0), kvh, 32 * m + 8 * jj + ci, tok + 8 * r));
      x[m][4 * r] = v.x; x[m][4 * r + 1] = v.y; x[m][4 * r + 2] = v.z; x[m][4 * r + 3] = v.w;
    }
  if (__builtin_amdgcn_ballot_w64(phys[0] < 0 || phys[1] < 0)) {  // a block table hole reads as zeros
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int i = 0; i < 8; ++i) x[m][i] = phys[i / 4] < 0 ? 0u : x[m][i];
  }
  float one = 1.0f;
  asm volatile("" : "+s"(one));                                  // x - min as one v_fma_mix
  uint32_t out[4][DW];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    auto value = [&](int i) { return as_half2(x[m][i / 2])[i & 1]; };
    half2v a = as_half2(x[m][0]), b = a;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      a = pk_min(a, as_half2(x[m][i]));
      b = pk_max(b, as_half2(x[m][i]));
    }
    // the token halves of the channel sit 32 lanes apart
    a = pk_min(a, as_half2(lane_xor_u<32>(__builtin_bit_cast(uint32_t, a))));
    b = pk_max(b, as_half2(lane_xor_u<32>(__builtin_bit_cast(uint32_t, b))));
    float mn = (float)__builtin_elementwise_minimum(a.x, a.y), mx = (float)__builtin_elementwise_maximum(b.x, b.y);
    const bool in_order = __builtin_amdgcn_ballot_w64(scan_in_order(mn, mx)) != 0;
    if (in_order) {
      mn = FLT_MAX;
      mx = -FLT_MAX;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float v = (float)value(i);
        if (v < mn) mn = v;
        if (v > mx) mx = v;
      }
      scan_combine_lanes<32, 32>(mn, mx, lane);
    }
    const GroupQ g = group_params<LV>(mn, mx);
    reinterpret_cast<uint16_t*>(dst + F::kKParams + (jj + 4 * m) * 32)[8 * tt + ci] = tt ? g.zero : g.step;
    // token e of a dword where channel e belongs in the page's
    auto shift = [&](int e) { return BITS == 4 ? 16 * (e & 1) + 4 * (e >> 1) : 8 * (e >> 1) + 16 * (e & 1); };
    auto group = [&](int) -> const GroupQ& { return g; };
#pragma unroll
    for (int k = 0; k < DW; ++k) {
      auto val = [&](int e) { return value(PER * k + e); };
      uint32_t w = in_order ? pack_codes<BITS, PER, true>(one, val, group, shift)
                            : pack_codes<BITS, PER, false>(one, val, group, shift);
      w = swap_halves<1>(w, lane & 1);
      if constexpr (BITS == 4) {
        w = swap_nibbles<2>(w, lane & 2);
        w = swap_bytes<4>(w, lane & 4);
      } else {
        w = swap_bytes<2>(w, lane & 2);
      }
      out[m][k] = w;
    }
  }
  if constexpr (BITS == 4) {
    // dwords m = 0 .. 3 of tokens 16 tt + 8 k + ci: whole chunks
#pragma unroll
    for (int k = 0; k < DW; ++k)
      reinterpret_cast<u32x4*>(dst + F::kKCodes)[64 * tt + 16 * jj + 8 * k + ci] =
          u32x4{out[0][k], out[1][k], out[2][k], out[3][k]};
  } else {
    // dword 2 m + ci / 4 of tokens 16 tt + 4 k + ci % 4
#pragma unroll
    for (int k = 0; k < DW; ++k)
#pragma unroll
      for (int m = 0; m < 4; ++m)
        stage[(64 * tt + 16 * jj + 4 * k + (ci & 3)) * 8 + 2 * m + (ci >> 2)] = out[m][k];
    build_barrier<kWave>();
#pragma unroll
    for (int i = 0; i < F::kChunk * 2; i += 16)                  // 128 chunks of kChunk bytes, 16 per lane and step
      reinterpret_cast<u32x4*>(dst + F::kKCodes)[i * 4 + lane] = reinterpret_cast<const u32x4*>(stage)[i * 4 + lane];
  }
}

// V of a page.  Lane (g, r, p) = (lane / 16, lane / 4 % 4, lane % 4) takes
// the two tokens of slots 2 p, 2 p + 1 of lane group r over the 32 channels
// of group g, so a (token, group)'s least and greatest value need no other
// lane; the lanes of a quad exchange their tokens' codes of four channels (a
// pair, of two) for eight (four) slots of one.
template <int BITS>
__device__ __forceinline__ void build_page_v(const PageJob& j, const int32_t* btab, int kvh, int page, uint8_t* dst,
                                             uint32_t* stage, int lane) {
  using F = KiviFmt<BITS>;
  constexpr int LV = F::kLevels, CH = 16 / BITS;                 // channels of a packed dword
  const int g = lane >> 4, r = lane >> 2 & 3, p = lane & 3;
  const int tok = page * kKiviPageTokens + kivi_v_token(r, 2 * p);
  const int phys = block_of_token(j, btab, tok);
  const uint16_t* at = pool_at(j, j.v_cache, max(phys, 0), kvh, 32 * g, tok);
  uint32_t x[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) x[i] = *reinterpret_cast<const uint32_t*>(at + i * j.block_size);
  if (__builtin_amdgcn_ballot_w64(phys < 0)) {
#pragma unroll
    for (int i = 0; i < 32; ++i) x[i] = phys < 0 ? 0u : x[i];
  }
  half2v a = as_half2(x[0]), b = a;
#pragma unroll
  for (int i = 1; i < 32; ++i) {
    a = pk_min(a, as_half2(x[i]));
    b = pk_max(b, as_half2(x[i]));
  }
  float mn[2] = {(float)a.x, (float)a.y}, mx[2] = {(float)b.x, (float)b.y};
  const bool in_order =
      __builtin_amdgcn_ballot_w64(scan_in_order(mn[0], mx[0]) || scan_in_order(mn[1], mx[1])) != 0;
  if (in_order) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      mn[e] = FLT_MAX;
      mx[e] = -FLT_MAX;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const float v = (float)as_half2(x[i])[e];
        if (v < mn[e]) mn[e] = v;
        if (v > mx[e]) mx[e] = v;
      }
    }
  }
  const GroupQ q[2] = {group_params<LV>(mn[0], mx[0]), group_params<LV>(mn[1], mx[1])};
  uint32_t* params = reinterpret_cast<uint32_t*>(dst + F::kVParams + (4 * g + r) * 32);
  params[p] = q[0].step | (uint32_t)q[1].step << 16;
  params[4 + p] = q[0].zero | (uint32_t)q[1].zero << 16;

  float one = 1.0f;
  asm volatile("" : "+s"(one));
  // chunks of the stage are permuted (by 4 r or 2 r) against bank conflicts
  // between the lane groups
  constexpr int SW = BITS == 4 ? 4 : 2, CD = F::kChunk / 4;
  auto chunk = [&](int c) { return (64 * (g >> 1) + 16 * r + ((c & 15) ^ (SW * r))) * CD; };
  // code e of a dword: channel e / 2 of its CH, token e % 2; the second
  // token in the upper half
  auto shift = [&](int e) { return 16 * (e & 1) + BITS * (e >> 1); };
  auto group = [&](int e) -> const GroupQ& { return q[e & 1]; };
#pragma unroll
  for (int k = 0; k < 32 / CH; ++k) {
    auto val = [&](int e) { return as_half2(x[CH * k + (e >> 1)])[e & 1]; };
    uint32_t w = in_order ? pack_codes<BITS, 2 * CH, true>(one, val, group, shift)
                          : pack_codes<BITS, 2 * CH, false>(one, val, group, shift);
    if constexpr (BITS == 4) {
      w = swap_nibbles<1>(w, lane & 1);
      w = swap_bytes<2>(w, lane & 2);
      const int c = 4 * k + p;                                   // of the group's 32
      stage[chunk(c) + 2 * (g & 1) + (c >> 4)] = w;
    } else {
      w = swap_bytes<1>(w, lane & 1);
      const int c = 2 * k + (p & 1);
      stage[chunk(c) + 4 * (g & 1) + 2 * (c >> 4) + (p >> 1)] = w;
    }
  }
  build_barrier<kWave>();
#pragma unroll
  for (int i = 0; i < F::kChunk * 2; i += 16) {
    const int at16 = i * 4 + lane, c = at16 / (CD / 4);          // 16 bytes of chunk c
    const int from = (c ^ (SW * (c >> 4 & 3))) * (CD / 4) + at16 % (CD / 4);
    reinterpret_cast<u32x4*>(dst + F::kVCodes)[at16] = reinterpret_cast<const u32x4*>(stage)[from];
  }
}

template <int BITS>
__global__ __launch_bounds__(2 * kWave) void kivi_prefix_kernel(PageJob j) {
  using F = KiviFmt<BITS>;
  __shared__ __attribute__((aligned(16))) uint32_t stage[2][128 * F::kChunk / 4];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int bid = blockIdx.x;
  const int kvh = bid % j.num_kv_heads; bid /= j.num_kv_heads;
  const int page = bid % j.pages_per_seq_grid;
  const int seq = bid / j.pages_per_seq_grid;
  const int L = j.seq_lens[seq];
  // build-ahead: the next page too once its first piece is due (every piece
  // written so far and the rest ahead of time: the same bytes)
  int ahead_page;
  const int piece = j.build_ahead ? kivi_ahead_piece(L, j.residual_length, ahead_page) : -1;
  if (page >= kivi_quantized_len(L, j.residual_length) / kKiviPageTokens && !(piece >= 0 && page == ahead_page)) return;
  if (page >= j.max_pages_per_seq) return;
  const int pid = j.page_tables[(int64_t)seq * j.max_pages_per_seq + page];
  if (pid < 0 || pid >= j.num_pages) return;
  uint8_t* dst = j.pages + ((int64_t)pid * j.num_kv_heads + kvh) * F::kBytes;
  const int32_t* btab = j.block_tables + (int64_t)seq * j.max_blocks_per_seq;
  if (wave == 0)
    build_page_k<BITS>(j, btab, kvh, page, dst, stage[0], lane);
  else
    build_page_v<BITS>(j, btab, kvh, page, dst, stage[1], lane);
}

}  // namespace

int launch_kivi_vec(const void* in, void* out, int n_vecs, int head_dim, int n_outliers,
                    int group_size, int stride, bool compress, hipStream_t stream) {
  const int rec_bytes = kivi_record_bytes(head_dim, n_outliers, group_size);
  const uint16_t* kv = (const uint16_t*)(compress ? in : out);
  const uint8_t* rec = (const uint8_t*)(compress ? out : in);
  const bool wide = head_dim % 8 == 0 && (uintptr_t)kv % 16 == 0;
  const bool dwords = stride % 4 == 0 && (uintptr_t)rec % 4 == 0;
  // a launch of 2^32 threads or more (2^29 vectors) wraps
  constexpr int kMost = 1 << 28;
  for (int first = 0, n; first < n_vecs; first += n) {
    n = min(n_vecs - first, kMost);
    const dim3 grid((unsigned)((n + kVecVecs - 1) / kVecVecs));
    const uint16_t* x = kv + (int64_t)first * head_dim;
    const uint8_t* r = rec + (int64_t)first * stride;
    if (compress) {
      auto go = [&](auto spl) {
        hipLaunchKernelGGL(kivi_vec_compress_kernel<decltype(spl)::value>, grid, dim3(kWave), 0, stream, x,
                           const_cast<uint8_t*>(r), n, head_dim, n_outliers, group_size, stride, rec_bytes, wide,
                           dwords);
      };
      if (n_outliers <= kVecLanes) go(std::integral_constant<int, 1>());
      else if (n_outliers <= 2 * kVecLanes) go(std::integral_constant<int, 2>());
      else if (n_outliers <= 4 * kVecLanes) go(std::integral_constant<int, 4>());
      else go(std::integral_constant<int, 8>());
    } else {
      hipLaunchKernelGGL(kivi_vec_decompress_kernel, grid, dim3(kWave), 0, stream, r, const_cast<uint16_t*>(x), n,
                         head_dim, n_outliers, group_size, stride, rec_bytes, wide, dwords);
    }
  }
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

int launch_kivi_pages(const KiviPageLaunch& a) {
  if (!a.append && a.max_pages_to_build <= 0) return 0;
  const PageJob j = make_page_job(a);
  const dim3 grid((unsigned)(a.num_seqs * j.pages_per_seq_grid * a.num_kv_heads));
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(128), 0, a.stream, j); };
  if (a.append) {
    if (a.bits == 8) go(kivi_append_kernel<8>); else go(kivi_append_kernel<4>);
  } else {
    if (a.bits == 8) go(kivi_prefix_kernel<8>); else go(kivi_prefix_kernel<4>);
  }
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

}  // namespace tl
