// Depthwise causal convolution as banded Toeplitz products on
// v_mfma_f32_16x16x32_bf16, at fp32 precision (gfx950).
//
// Output block a (16 positions) of a tile is column a of
//     Y = T Xw,   T[i][t] = band[t - i],   Xw[t][a] = src[16 a + t],
// t < 32 S.  The bf16 matrix rate is 16 times the fp32 one, so every fp32
// operand is written as a sum of bf16 values and the product runs once per
// pair of parts.  Each part is what the parts before it leave, rounded to
// nearest; the sum is the operand exactly:
//     fp32: 3 parts (8 + 8 + 8 mantissa bits), fp16: 2 (8 + 3), bf16: 1.
// The pairs (i, j) with i + j <= 2 are kept.  For an operand in [1, 2) part 1
// is at most 2^-8 and part 2 at most 2^-17, so the dropped pairs, (1, 2) and
// (2, 1) above all, are at most 2^-24 of the product: what one fp32 rounding
// may lose, and of either sign.  (Parts cut off instead of rounded reach 2^-7
// and 2^-15 with the operand's sign: 2^-21, always towards zero.)  bf16
// samples against fp32 taps are 3 products (none dropped), i.e. 3/16 of the
// fp32 matrix time.  Operands below 2^-110 lose parts to bf16's smallest
// value.
//
// Lane layout: lane l supplies A[l % 16][8 (l / 16) + e] and B[8 (l / 16) +
// e][l % 16], e < 8, and receives D[4 (l / 16) + r][l % 16].  With the taps as
// A and the samples as B a lane receives four consecutive positions of one
// block, and a wave's result is one contiguous run of 256 positions: stores
// are 8 or 16 bytes per lane.  (With the samples as A a lane receives four
// positions 16 apart, four 2-byte stores.)
#pragma once

#include "direct_conv.h"

namespace nsq {

template <int DT>
constexpr int kParts = DT == NSQ_DTYPE_BF16 ? 1 : DT == NSQ_DTYPE_F16 ? 2 : 3;
constexpr int kTapParts = 3;

// (v0, v1) = sums of the parts, each a pair of bf16 in a word (v0 low), largest first.
template <int P>
__device__ __forceinline__ void split_parts2(float v0, float v1, uint32_t (&b)[P]) {
#pragma unroll
  for (int p = 0; p < P; ++p) {
    b[p] = f32x2_to_bf16x2_bits(v0, v1);
    if (p + 1 < P) {
      v0 -= __uint_as_float(b[p] << 16);
      v1 -= __uint_as_float(b[p] & 0xffff0000u);
    }
  }
}

__device__ __forceinline__ nsq_bf16x8_t as_bf16x8(uint4 u) { return __builtin_bit_cast(nsq_bf16x8_t, u); }

// c += T Xw over one step: the products of parts i of the samples and j of the taps with i + j <= 2.
template <int P>
__device__ __forceinline__ void mma_parts(const nsq_bf16x8_t (&tap)[kTapParts], const nsq_bf16x8_t (&x)[P],
                                          nsq_f32x4_t& c) {
#pragma unroll
  for (int d = kTapParts - 1; d >= 0; --d)  // small products first
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (d - i >= 0) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tap[d - i], x[i], c, 0, 0, 0);
}

// sum_j w[j] x[n - K + 1 + j], tap by tap from memory.
template <int DT>
__device__ __forceinline__ float direct_taps(const RowBuf<DT, false>& x, const float* __restrict__ w, int K, int n) {
  float a = 0.f;
  for (int j = 0; j < K; ++j) a = fmaf(w[j], x.elem_halo(n - K + 1 + j), a);
  return a;
}

// The band of K taps as A operands.  conv: T[i][t] = w[t - i - pad] over the
// window src[m] = x[n0 - KP + m], KP = band_kp<S>() (pad = KP - K + 1 leading
// zero taps); REV: T[i][t] = w[K - 1 - (t - i)] over src[m] = g[n0 + m].
// Samples of the window before the tile's first: a multiple of 16 with KP + 16 <= 32 S columns.
template <int S>
constexpr int band_kp() { return 32 * S - 16 < kConvMaxK ? 32 * S - 16 : kConvMaxK; }
// Whether the last step's upper 16 columns are zero in both bands (S = 9: K <= 256); lanes 32.. then store nothing.
template <int S>
constexpr bool band_half_last() { return band_kp<S>() + 16 < 32 * S; }
// 16-byte operands of a band in LDS, all parts.
template <int S>
constexpr int band_operands() { return kTapParts * (64 * S - (band_half_last<S>() ? 32 : 0)); }

template <int S, bool REV>
__device__ __forceinline__ float band_tap(const float* wl, int K, int i, int t) {
  constexpr int KP = band_kp<S>();
  const int j = REV ? K - 1 - (t - i) : t - i - (KP - K + 1);
  const bool ok = j >= 0 && j < K;
  const float v = wl[ok ? j : 0];
  return ok ? v : 0.f;
}

// Step s of the band for lane l, as kTapParts 16-byte operands.
template <int S, bool REV>
__device__ __forceinline__ void band_operand(const float* wl, int K, int s, int l, uint4 (&o)[kTapParts]) {
  const int kk = l >> 4, i = l & 15;
  uint32_t u[kTapParts][4];
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    uint32_t a[kTapParts];
    split_parts2<kTapParts>(band_tap<S, REV>(wl, K, i, 32 * s + 8 * kk + e),
                            band_tap<S, REV>(wl, K, i, 32 * s + 8 * kk + e + 1), a);
#pragma unroll
    for (int p = 0; p < kTapParts; ++p) u[p][e / 2] = a[p];
  }
#pragma unroll
  for (int p = 0; p < kTapParts; ++p) o[p] = make_uint4(u[p][0], u[p][1], u[p][2], u[p][3]);
}

// A band in LDS as operands, made by the whole workgroup, and one lane's copy of it.
template <int S, bool REV>
__device__ __forceinline__ void put_band(uint4* to, const float* wl, int K) {
  for (int o = int(threadIdx.x); o < S * 64; o += kConvThreads) {
    const int s = o >> 6, l = o & 63;
    const bool half = band_half_last<S>() && s == S - 1;
    if (half && l >= 32) continue;
    uint4 u[kTapParts];
    band_operand<S, REV>(wl, K, s, l, u);
#pragma unroll
    for (int p = 0; p < kTapParts; ++p) to[s * kTapParts * 64 + p * (half ? 32 : 64) + l] = u[p];
  }
}
template <int S>
__device__ __forceinline__ void get_band(const uint4* from, nsq_bf16x8_t (&tap)[S][kTapParts]) {
  const int l = int(threadIdx.x) & 63;
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int p = 0; p < kTapParts; ++p) {
      if (band_half_last<S>() && s == S - 1) {
        const uint4 u = from[s * kTapParts * 64 + p * 32 + (l & 31)];
        const bool z = l >= 32;
        tap[s][p] = as_bf16x8(make_uint4(z ? 0u : u.x, z ? 0u : u.y, z ? 0u : u.z, z ? 0u : u.w));
      } else {
        tap[s][p] = as_bf16x8(from[(s * kTapParts + p) * 64 + l]);
      }
    }
}

// Rows that are not whole 16-byte chunks (AL false) are read and written as unaligned vectors, and by elements only
// where a chunk crosses the row's end.  Element accesses alone (a lane's eight at a stride of 16 or 32 bytes across
// lanes) took B=4 C=512 L=10007 K=33 from 27 (row-wise loads of the fp32 products) to 51 us forward in bf16.
template <int DT, int N>
struct RowVec {  // N elements of DT as a vector that may start at any element
  static constexpr int W = N * int(sizeof(typename Elem<DT>::T)) / 4;
  typedef uint32_t V __attribute__((ext_vector_type(W), aligned(sizeof(typename Elem<DT>::T))));
};

// row[n, n + N) as words, zero outside [0, L); a chunk before the row lies wholly before it.
template <int DT, int N, int W>
__device__ __forceinline__ void load_any(const typename Elem<DT>::T* __restrict__ row, const RowBuf<DT, false>& rb,
                                         int n, int L, uint32_t (&w)[W]) {
  using R = RowVec<DT, N>;
  static_assert(W == R::W, "load_any: words");
  uint32_t v[W];
#pragma unroll
  for (int i = 0; i < W; ++i) v[i] = 0;
  if (n >= 0 && n + N <= L) {
    const typename R::V m = *reinterpret_cast<const typename R::V*>(row + n);
#pragma unroll
    for (int i = 0; i < W; ++i) v[i] = m[i];
  } else if (n >= 0 && n < L) {
    if constexpr (DT == NSQ_DTYPE_F32) {
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = rb.elem_halo_bits(n + i);
    } else {
#pragma unroll
      for (int i = 0; i < W; ++i) v[i] = rb.elem_halo_bits(n + 2 * i) | (rb.elem_halo_bits(n + 2 * i + 1) << 16);
    }
  }
#pragma unroll
  for (int i = 0; i < W; ++i) w[i] = v[i];
}

// Eight consecutive samples of a row, loaded raw and written out as bf16 parts.
template <int DT, bool AL>
struct PartChunk {
  static constexpr int P = kParts<DT>;
  Win8<DT, true> w;
  __device__ __forceinline__ void load(const typename Elem<DT>::T* __restrict__ row, int n, int L) {
    const RowBuf<DT, false> rb(row, L);
    if constexpr (AL)
      w.load(rb, n);
    else
      load_any<DT, 8>(row, rb, n, L, w.w);
  }
  __device__ __forceinline__ void parts(uint4 (&o)[P]) const {
    if constexpr (DT == NSQ_DTYPE_BF16) {
      o[0] = make_uint4(w.w[0], w.w[1], w.w[2], w.w[3]);
    } else {
      uint32_t u[P][4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        uint32_t a[P];
        split_parts2<P>(w.at(e), w.at(e + 1), a);
#pragma unroll
        for (int p = 0; p < P; ++p) u[p][e / 2] = a[p];
      }
#pragma unroll
      for (int p = 0; p < P; ++p) o[p] = make_uint4(u[p][0], u[p][1], u[p][2], u[p][3]);
    }
  }
};

// Four consecutive outputs at position n of a row (n a multiple of 4), dropped past the end: one 8- or 16-byte store,
// aligned where the rows are (AL), else by elements where it crosses the end.
template <int DT, bool AL>
__device__ __forceinline__ void store4(typename Elem<DT>::T* __restrict__ row, int n, int L, const float (&v)[4]) {
  const RowBuf<DT, false> rb(row, L);
  using R = RowVec<DT, 4>;
  uint32_t u[R::W];
  if constexpr (DT == NSQ_DTYPE_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = __float_as_uint(v[i]);
  } else if constexpr (DT == NSQ_DTYPE_BF16) {
    u[0] = f32x2_to_bf16x2_bits(v[0], v[1]);
    u[1] = f32x2_to_bf16x2_bits(v[2], v[3]);
  } else {
    u[0] = __builtin_bit_cast(uint32_t, __floats2half2_rn(v[0], v[1]));
    u[1] = __builtin_bit_cast(uint32_t, __floats2half2_rn(v[2], v[3]));
  }
  if constexpr (AL) {
    using U2 = uint32_t __attribute__((ext_vector_type(2)));
    using U4 = uint32_t __attribute__((ext_vector_type(4)));
    const int off = n * int(sizeof(typename Elem<DT>::T));
    if constexpr (DT == NSQ_DTYPE_F32)
      __builtin_amdgcn_raw_buffer_store_b128(U4{u[0], u[1], u[2], u[3]}, rb.r, off, 0, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(U2{u[0], u[1]}, rb.r, off, 0, 0);
  } else if (n + 4 <= L) {
    typename R::V m;
#pragma unroll
    for (int i = 0; i < R::W; ++i) m[i] = u[i];
    *reinterpret_cast<typename R::V*>(row + n) = m;
  } else if (n < L) {
#pragma unroll
    for (int r = 0; r < 4; ++r) rb.store_elem(n + r, v[r]);
  }
}

// Four consecutive samples at position n >= 0 of a row as raw bits (zero past the end).
template <int DT, bool AL>
struct Quad {
  static constexpr bool HALF = DT != NSQ_DTYPE_F32;
  uint32_t w[HALF ? 2 : 4];
  __device__ __forceinline__ void load(const typename Elem<DT>::T* __restrict__ row, int n, int L) {
    const RowBuf<DT, false> rb(row, L);
    if constexpr (!AL) {
      load_any<DT, 4>(row, rb, n, L, w);
    } else if constexpr (HALF) {
      const auto m = __builtin_amdgcn_raw_buffer_load_b64(rb.r, n * 2, 0, 0);
      w[0] = m[0]; w[1] = m[1];
    } else {
      const auto m = __builtin_amdgcn_raw_buffer_load_b128(rb.r, n * 4, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = m[i];
    }
  }
  __device__ __forceinline__ float at(int i) const {
    if constexpr (HALF) {
      const uint32_t v = (i & 1) ? (w[i >> 1] >> 16) : (w[i >> 1] & 0xffffu);
      return RowBuf<DT, false>::bits_to_f32(v);
    } else {
      return RowBuf<DT, false>::bits_to_f32(w[i]);
    }
  }
};

// The operand whose contraction runs over the 16-element rows of an LDS array: lane l gets element l % 16 of rows
// 8 (l / 16) + e, e < 8 (p: row 0).  ds_read_b64_tr_b16: the 16 lanes of a group read four rows, 8 bytes a lane, and
// lane i receives column i of them (checked on MI355X).
__device__ __forceinline__ nsq_bf16x8_t tr16_column8(const uint16_t* p) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef v4s __attribute__((address_space(3)))* lds_v4s;
  const int l = int(threadIdx.x) & 63;
  const uint16_t* q = p + (8 * (l >> 4) + ((l >> 2) & 3)) * 16 + 4 * (l & 3);
  const v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(q));
  const v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(q + 64));
  return __builtin_bit_cast(nsq_bf16x8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Steps of 32 window columns for K taps: 32 S >= K + 15.
inline int band_steps_for(int64_t K) { return K <= 17 ? 1 : K <= 49 ? 2 : K <= 81 ? 3 : K <= 145 ? 5 : K <= 209 ? 7 : 9; }

}  // namespace nsq
