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

// ---------------------------------------------------------------------------
// The reference vector codec.  8 lanes share a vector, a 64-thread workgroup
// takes 8 vectors: 16 384 vectors are 2048 wavefronts, two per SIMD.  The
// sequential part of the format (which slot an outlier ends in) is kept
// sequential over the channels, but each of its steps is the work of 8
// lanes; the rest (ranks, groups, codes) is spread over them.  Rows and
// records go through LDS, so that memory sees whole lines.  Bound: the
// 128-step scan's dependency chain (about 12 vector instructions a step at
// up to 8 outliers).  Compress and decompress of 16 384 vectors of 128
// channels, 8 outliers, groups of 16: 23.9 us; one thread per vector, with
// its slots, flags and values in scratch memory, took 1488 us (783 + 706).
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
// Over the 8 lanes of a vector.
__device__ __forceinline__ uint32_t min8(uint32_t v) {
  v = min(v, dpp_u32<kDppXor1>(v));
  v = min(v, dpp_u32<kDppXor2>(v));
  return min(v, dpp_u32<kDppHalfMirror>(v));
}
__device__ __forceinline__ uint32_t or8(uint32_t v) {
  v |= dpp_u32<kDppXor1>(v);
  v |= dpp_u32<kDppXor2>(v);
  return v | dpp_u32<kDppHalfMirror>(v);
}

// nv rows of d halves between memory and LDS rows of kVecRow halves; 16-byte
// accesses where d is a multiple of 8 and the base 16-byte aligned.
__device__ __forceinline__ void vec_rows_in(const uint16_t* src, uint16_t* rows, int nv, int d, bool wide, int lane) {
  if (wide) {
    const int per = d / 8;
    for (int i = lane; i < nv * per; i += kWave)
      *reinterpret_cast<u32x4*>(rows + i / per * kVecRow + i % per * 8) = load16(src + 8 * i);
  } else {
    for (int i = lane; i < nv * d; i += kWave) rows[i / d * kVecRow + i % d] = src[i];
  }
}
__device__ __forceinline__ void vec_rows_out(uint16_t* dst, const uint16_t* rows, int nv, int d, bool wide, int lane) {
  if (wide) {
    const int per = d / 8;
    for (int i = lane; i < nv * per; i += kWave)
      *reinterpret_cast<u32x4*>(dst + 8 * i) = *reinterpret_cast<const u32x4*>(rows + i / per * kVecRow + i % per * 8);
  } else {
    for (int i = lane; i < nv * d; i += kWave) dst[i] = rows[i / d * kVecRow + i % d];
  }
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
  vec_rows_in(in + v0 * head_dim, s_x, nv, head_dim, wide, lane);
  // channels up to the next multiple of 8: NaN, which the scan skips
  if (vi < nv && head_dim + l8 < (head_dim + 7) / 8 * 8) x[head_dim + l8] = 0x7FFF;
  __syncthreads();

  // Top-n_outliers |x| by the reference's replace-the-first-minimum scan.  A
  // slot is one word: (|x| as ordered bits + 1, 0 when empty) << 16 | slot
  // << 8 | channel, so the least word of the vector's slots is the first
  // slot of least magnitude.
  uint32_t key[SPL];
#pragma unroll
  for (int i = 0; i < SPL; ++i) {
    const int s = i * kVecLanes + l8;
    key[i] = s < n_outliers ? (uint32_t)s << 8 : 0xFFFFFFFFu;
  }
  if (n_outliers > 0) {
    uint32_t least = 0;                               // slot 0, empty
    for (int d0 = 0; d0 < head_dim; d0 += 8) {
      const u32x4 c = *reinterpret_cast<const u32x4*>(x + d0);
      const uint32_t w[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t m = ((w[e / 2] >> (16 * (e & 1))) & 0x7FFFu) + 1u;
        const bool take = m > (least >> 16) && m <= 0x7C01u;      // greater, and not NaN
        const uint32_t put = m << 16 | (least & 0xFF00u) | (uint32_t)(d0 + e);
        const uint32_t at = take ? least : 0xFFFFFFFEu;           // no slot holds that word
        uint32_t lo = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
          key[i] = key[i] == at ? put : key[i];
          lo = min(lo, key[i]);
        }
        least = min8(lo);
      }
    }
  }

  // the outliers' records, and the mask of their channels (an empty slot
  // holds channel 0, as the reference's does)
  uint32_t mask[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < SPL; ++i) {
    const int s = i * kVecLanes + l8;
    if (s < n_outliers) {
      const int ch = key[i] & 0xFF;
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
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int d = 16 * l8 + e;
      const bool put = !((own >> e) & 1u) && d < head_dim;
      if (put && r < n_res) res[r] = x[d];
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
    float gmin = FLT_MAX, gmax = -FLT_MAX;
#pragma unroll 4
    for (int i = 0; i < n; i += 2) {
      const uint32_t w = pairs[i / 2];
      const float a = f16_to_f32((uint16_t)w), b = i + 1 < n ? f16_to_f32((uint16_t)(w >> 16)) : a;
      if (a < gmin) gmin = a;
      if (a > gmax) gmax = a;
      if (b < gmin) gmin = b;
      if (b > gmax) gmax = b;
    }
    const GroupQ q = group_params(gmin, gmax);
    uint8_t* p = rec + 3 * n_outliers + g * (group_size / 2 + 4);
#pragma unroll 4
    for (int i = 0; i < n; i += 2) {
      const uint32_t w = pairs[i / 2];
      const int q0 = quantise(f16_to_f32((uint16_t)w), q);
      const int q1 = i + 1 < n ? quantise(f16_to_f32((uint16_t)(w >> 16)), q) : 0;
      *p++ = (uint8_t)((q1 << 4) | q0);
    }
    p[0] = (uint8_t)(q.step & 0xff); p[1] = (uint8_t)(q.step >> 8);
    p[2] = (uint8_t)(q.zero & 0xff); p[3] = (uint8_t)(q.zero >> 8);
  }
  __syncthreads();

  uint8_t* dst = out + v0 * stride;
  const int words = rec_bytes / 4;
  int done = 0;
  if (dwords) {
    for (int i = lane; i < nv * words; i += kWave) {
      const int v = i / words, w = i % words;
      *reinterpret_cast<uint32_t*>(dst + (int64_t)v * stride + 4 * w) =
          *reinterpret_cast<const uint32_t*>(s_rec + v * kVecRec + 4 * w);
    }
    done = 4 * words;
  }
  const int rest = rec_bytes - done;
  for (int i = lane; i < nv * rest; i += kWave) {
    const int v = i / rest, b = done + i % rest;
    dst[(int64_t)v * stride + b] = s_rec[v * kVecRec + b];
  }
}

__global__ __launch_bounds__(kWave) void kivi_vec_decompress_kernel(
    const uint8_t* __restrict__ in, uint16_t* __restrict__ out, int n_vecs, int head_dim, int n_outliers,
    int group_size, int stride, int rec_bytes, bool wide, bool dwords) {
  __shared__ __attribute__((aligned(16))) uint16_t s_x[kVecVecs * kVecRow];
  __shared__ __attribute__((aligned(16))) uint8_t s_rec[kVecVecs * kVecRec];
  const int lane = threadIdx.x, l8 = lane % kVecLanes, vi = lane / kVecLanes;
  const int64_t v0 = (int64_t)blockIdx.x * kVecVecs;
  const int nv = (int)min<int64_t>(kVecVecs, n_vecs - v0);
  const uint8_t* src = in + v0 * stride;
  {
    const int words = rec_bytes / 4;
    int done = 0;
    if (dwords) {
      for (int i = lane; i < nv * words; i += kWave) {
        const int v = i / words, w = i % words;
        *reinterpret_cast<uint32_t*>(s_rec + v * kVecRec + 4 * w) =
            *reinterpret_cast<const uint32_t*>(src + (int64_t)v * stride + 4 * w);
      }
      done = 4 * words;
    }
    const int rest = rec_bytes - done;
    for (int i = lane; i < nv * rest; i += kWave) {
      const int v = i / rest, b = done + i % rest;
      s_rec[v * kVecRec + b] = src[(int64_t)v * stride + b];
    }
  }
  __syncthreads();
  if (vi < nv) {
    const uint8_t* rec = s_rec + vi * kVecRec;
    uint16_t* x = s_x + vi * kVecRow;
    // lane l8 owns channels 16 l8 .. + 15; every lane reads every outlier,
    // so that of two for one channel the later stands
    uint32_t own = 0;
    for (int i = 0; i < n_outliers; ++i) {
      const int ch = rec[3 * i];
      if (ch / 16 == l8 && ch < head_dim) {
        own |= 1u << (ch % 16);
        x[ch] = f32_to_f16(f16_to_f32((uint16_t)(rec[3 * i + 1] | (rec[3 * i + 2] << 8))));
      }
    }
    // the other channels' ranks: those of the lanes before first
    const int c1 = min(16 * l8 + 16, head_dim);
    const int owned = max(c1 - 16 * l8, 0);
    const int free_own = owned - __builtin_popcount(own);
    int before = 0;
#pragma unroll
    for (int o = 1; o < kVecLanes; ++o) {
      const int n = __shfl(free_own, (lane & ~(kVecLanes - 1)) + ((l8 - o) & (kVecLanes - 1)), kWave);
      before += o <= l8 ? n : 0;
    }
    const int n_res = head_dim - n_outliers;
    const int last0 = (n_res - 1) / group_size * group_size;        // first index of the last group
    int r = before;
    for (int e = 0; e < owned; ++e) {
      if ((own >> e) & 1u) continue;
      float val = 0.f;
      if (r < n_res) {
        const int g = r / group_size, k = r - g * group_size;
        const uint8_t* pack = rec + 3 * n_outliers + g * (group_size / 2 + 4);
        const int n = g * group_size == last0 ? n_res - last0 : group_size;
        const uint8_t* p = pack + (n + 1) / 2;
        const float st = f16_to_f32((uint16_t)(p[0] | (p[1] << 8)));
        const float ze = f16_to_f32((uint16_t)(p[2] | (p[3] << 8)));
        const int nib = (k % 2 == 0) ? (pack[k / 2] & 0x0f) : (pack[k / 2] >> 4);
        val = __builtin_fmaf((float)nib, st, ze);
      }
      x[16 * l8 + e] = f32_to_f16(val);
      ++r;
    }
  }
  __syncthreads();
  vec_rows_out(out + v0 * head_dim, s_x, nv, head_dim, wide, lane);
}

// ---------------------------------------------------------------------------
// Paged KIVI: build one page (32 tokens x 128 channels of one kv head) from
// the fp16 pool [N, n_kv, 128, BS].
// ---------------------------------------------------------------------------
template <int BITS>
__global__ __launch_bounds__(128) void kivi_page_kernel(PageJob j) {
  __shared__ __attribute__((aligned(16))) KiviBuildSmem<BITS> sm;
  const int tid = threadIdx.x;
  int bid = blockIdx.x;
  const int kvh = bid % j.num_kv_heads; bid /= j.num_kv_heads;
  const int pg = bid % j.pages_per_seq_grid;
  const int seq = bid / j.pages_per_seq_grid;
  const int L = j.seq_lens[seq];
  const int lq = kivi_quantized_len(L, j.residual_length);
  int page;
  int ahead_page;
  const int piece = j.build_ahead ? kivi_ahead_piece(L, j.residual_length, ahead_page) : -1;
  if (j.append) {
    kivi_append_token<128>(j, seq, kvh, tid);
    if (j.build_ahead) {
      // the pages this append completes were written in pieces by the
      // appends before it; this one writes its piece of the next page:
      // wavefront 0 stages its fp16, then each wavefront quantises two of
      // its quarters
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
    page = lq / kKiviPageTokens - 1;
  } else {
    page = pg;
    // build-ahead: the next page too once its first piece is due (every
    // piece written so far and the rest ahead of time: the same bytes)
    if (page >= lq / kKiviPageTokens && !(piece >= 0 && page == ahead_page)) return;
  }
  kivi_build_page<128, BITS>(sm, j, seq, kvh, page, L, tid);
}

}  // namespace

int launch_kivi_vec(const void* in, void* out, int n_vecs, int head_dim, int n_outliers,
                    int group_size, int stride, bool compress, hipStream_t stream) {
  const dim3 grid((unsigned)((n_vecs + kVecVecs - 1) / kVecVecs));
  const int rec_bytes = kivi_record_bytes(head_dim, n_outliers, group_size);
  const void* kv = compress ? in : out;
  const void* rec = compress ? out : in;
  const bool wide = head_dim % 8 == 0 && (uintptr_t)kv % 16 == 0;
  const bool dwords = stride % 4 == 0 && (uintptr_t)rec % 4 == 0;
  if (compress) {
    auto go = [&](auto spl) {
      hipLaunchKernelGGL(kivi_vec_compress_kernel<decltype(spl)::value>, grid, dim3(kWave), 0, stream,
                         (const uint16_t*)in, (uint8_t*)out, n_vecs, head_dim, n_outliers, group_size, stride,
                         rec_bytes, wide, dwords);
    };
    if (n_outliers <= kVecLanes) go(std::integral_constant<int, 1>());
    else if (n_outliers <= 2 * kVecLanes) go(std::integral_constant<int, 2>());
    else if (n_outliers <= 4 * kVecLanes) go(std::integral_constant<int, 4>());
    else go(std::integral_constant<int, 8>());
  } else {
    hipLaunchKernelGGL(kivi_vec_decompress_kernel, grid, dim3(kWave), 0, stream, (const uint8_t*)in, (uint16_t*)out,
                       n_vecs, head_dim, n_outliers, group_size, stride, rec_bytes, wide, dwords);
  }
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

int launch_kivi_pages(const KiviPageLaunch& a) {
  if (!a.append && a.max_pages_to_build <= 0) return 0;
  const PageJob j = make_page_job(a);
  const dim3 grid((unsigned)(a.num_seqs * j.pages_per_seq_grid * a.num_kv_heads));
  if (a.bits == 8)
    hipLaunchKernelGGL(kivi_page_kernel<8>, grid, dim3(128), 0, a.stream, j);
  else
    hipLaunchKernelGGL(kivi_page_kernel<4>, grid, dim3(128), 0, a.stream, j);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

}  // namespace tl
