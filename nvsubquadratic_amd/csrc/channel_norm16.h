// Norms over channels for 16-bit tensors with 16-byte runs (channel_norm.hip
// includes this after its own kernels; the operators and roundings are
// described there).
//
// Bound by HBM: forward y, v in and out once (6 bytes an element gated),
// backward dout, y, v in and dy, dv out (10 bytes).  The kernels above staged
// every element as fp32 in LDS, which left tiles of 16 positions (32-byte
// pieces of the channels-first rows), read y and v twice and took three
// passes over the tile; B=16 C=384 S=128^2 bf16 gated: forward 228 us,
// backward 679 us (2.7 and 1.5 TB/s).  Here a tile of 32 H positions stays in
// registers as its raw bits: lane l of wave w holds channel 16 (w + W j) +
// l % 16, j < NB, positions 32 h + 8 (l / 16) .. + 7, h < H, so that
//   - the channels-first side is one 16-byte access per (j, h), 64 (H = 1) or
//     128 (H = 2) bytes of a row per 16 lanes x 4;
//   - the channels-last side goes through one 16-bit LDS tile [position]
//     [channel], 16 bytes per lane to and from HBM; the backward's lanes read
//     their column of it with the transposing LDS read;
//   - the sums over channels are lane-halving DPP adds over the 16 lanes of a
//     position run, then one LDS exchange between the waves.  RMS and L2 need
//     one reduction each way: with xhat = u r, sum_c w dout xhat = r sum_c w
//     dout u.
// A lane holds up to three 16-byte vectors of each tensor (128 VGPRs, 4 waves per SIMD): 512 threads for 384
// channels, 1024 for 768; above that the backward spills (100 registers at 1536) and still gains.
// Measured there (us, forward / backward): 137 / 302, 4.4 and 3.3 TB/s.  Other sizes at B = 16, S = 128^2 bf16 gated,
// before -> now: C = 64 32 -> 27 / 116 -> 88, 768 485 -> 276 / 3812 -> 610, 1536 1147 -> 545 / 6929 -> 2067.
#pragma once

namespace nsq {
namespace {

constexpr int kNorm16MaxC = 1536;
// Sixteen bytes as a compiler vector: conditional copies of the uint4 struct go through scratch memory.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// xor-style partners within 16 lanes: 15, 7, 2, 1 (every lane meets all others).
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// One halving step: of N values a lane keeps the upper N / 2 if `up`, else the lower, adding its partner's share.
template <int N, int CTRL>
__device__ __forceinline__ void halve(float (&v)[N], bool up) {
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const float lo = v[i], hi = v[N / 2 + i];
    const float keep = up ? hi : lo, give = up ? lo : hi;
    v[i] = keep + dpp<CTRL>(give);
  }
}

// Sums over the 16 lanes of a row of 8 values; the lane is left with the sum of value lane16_slot(l).
__device__ __forceinline__ float sum16(const float (&a)[8], int l) {
  float v[8], w[4], x[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = a[i];
  halve<8, 0x140>(v, l & 8);
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = v[i];
  halve<4, 0x141>(w, l & 4);
  x[0] = w[0];
  x[1] = w[1];
  halve<2, 0x4E>(x, l & 2);
  return x[0] + dpp<0xB1>(x[0]);
}
__device__ __forceinline__ int lane16_slot(int l) { return ((l & 8) >> 1) + ((l & 4) >> 1) + ((l & 2) >> 1); }

template <int NB_, int H_, int NT_>
struct Norm16Cfg {
  static constexpr int NB = NB_, H = H_, NT = NT_, W = NT / 64, TS = 32 * H;
};
// LDS row stride of the channels-last tile: the channels rounded up to 16 and 16 more (rows 32 bytes apart mod 256
// where C is a multiple of 128, so the four rows of a transposing read fall on different banks).
__host__ __device__ inline int norm16_ld(int C) { return (C + 15) / 16 * 16 + 16; }
template <class F>
inline size_t norm16_lds(int C, int sums) {
  return size_t(F::TS) * norm16_ld(C) * 2 + size_t(F::W + 1) * sums * F::TS * 4;
}

// K sums per position over all channels: part[k] holds the lane's 8 position sums for each h.  Result in tot[k][TS].
template <class F, int K>
__device__ __forceinline__ void norm16_sums(const float (&part)[K][F::H][8], float* red, float* tot) {
  const int t = int(threadIdx.x), l = t & 63, wave = t >> 6;
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int h = 0; h < F::H; ++h) {
      const float s = sum16(part[k][h], l);
      if ((l & 1) == 0) red[(wave * K + k) * F::TS + 32 * h + 8 * (l >> 4) + lane16_slot(l)] = s;
    }
  __syncthreads();
  if (t < K * F::TS) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < F::W; ++w) s += red[w * K * F::TS + t];
    tot[t] = s;
  }
  __syncthreads();
}

template <int DT>
__device__ __forceinline__ void unpack8(const u32x4& q, float (&f)[8]) {
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 8; ++i)
    f[i] = RowBuf<DT, false>::bits_to_f32((i & 1) ? w[i >> 1] >> 16 : w[i >> 1] & 0xffffu);
}
template <int DT>
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == NSQ_DTYPE_BF16)
      w[i] = f32x2_to_bf16x2_bits(f[2 * i], f[2 * i + 1]);
    else
      w[i] = __builtin_bit_cast(uint32_t, __floats2half2_rn(f[2 * i], f[2 * i + 1]));
  }
  return u32x4{w[0], w[1], w[2], w[3]};
}

// The two values of one 32-bit word.
template <int DT>
__device__ __forceinline__ void unpack2(uint32_t w, float (&f)[2]) {
  f[0] = RowBuf<DT, false>::bits_to_f32(w & 0xffffu);
  f[1] = RowBuf<DT, false>::bits_to_f32(w >> 16);
}
template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (DT == NSQ_DTYPE_BF16)
    return f32x2_to_bf16x2_bits(a, b);
  else
    return __builtin_bit_cast(uint32_t, __floats2half2_rn(a, b));
}

// Hides that the bits are those of an earlier use: without it the compiler keeps each sweep's unpacked values, gates
// and products (eight registers a vector each) for the next one across the barriers, or unpacks a conditional load
// where it is issued, and spills.
__device__ __forceinline__ void opaque(u32x4& q) { asm volatile("" : "+v"(q)); }

// 16-byte accesses through a raw buffer that starts at a tile: the range check stands in for the branches, so a
// tile's loads are issued back to back, and one 32-bit offset a vector serves every tensor.  kOutside reads as zero
// and stores nothing.
constexpr int kOutside = int(0x80000000u);
struct Buf16 {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Buf16(const void* p, int64_t bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, int(bytes), 0x00020000)) {}
  __device__ __forceinline__ u32x4 load(int off) const {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  }
  __device__ __forceinline__ void store(int off, u32x4 v) const {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, 0);
  }
};

// Position sums of a lane's 8 positions out of tot (16-byte reads).
__device__ __forceinline__ void take8(const float* tot, float (&o)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(tot), b = *reinterpret_cast<const float4*>(tot + 4);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
  o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
}

// u = round(y round(act(v))), or y (ACT = kNoGate); act(v) rounded in a.
constexpr int kNoGate = -1;
template <int DT, int ACT>
__device__ __forceinline__ float gate_u(float y, float v, float& a) {
#pragma clang fp contract(off)
  if constexpr (ACT == kNoGate) return y;
  a = Elem<DT>::round(gate_act(ACT, v));
  return Elem<DT>::round(y * a);
}

// Chunk q of a channels-last tile of C8 16-byte chunks a row: its position.
__device__ __forceinline__ int chunk_row(int q, float inv_c8) { return int((float(q) + 0.5f) * inv_c8); }

template <int DT, int MODE, int ACT, class F>
__global__ __launch_bounds__(F::NT) __attribute__((amdgpu_waves_per_eu(4))) void chnorm16_fwd_kernel(
    const typename Elem<DT>::T* __restrict__ y, const typename Elem<DT>::T* __restrict__ v,
    const float* __restrict__ w, const float* __restrict__ bias, typename Elem<DT>::T* __restrict__ out, int C,
    int64_t S, int64_t tiles_per_b, int64_t ntiles, float eps, int out_blh) {
#pragma clang fp contract(off)
  using T = typename Elem<DT>::T;
  extern __shared__ __align__(16) float smem[];
  const int ld = norm16_ld(C);
  uint16_t* tile = reinterpret_cast<uint16_t*>(smem);
  float* tot = smem + F::TS * ld / 2;
  float* red = tot + F::TS;
  const int t = int(threadIdx.x), l = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t ti = xcd_remap(blockIdx.x, ntiles);
  const int64_t b = ti / tiles_per_b, s0 = (ti % tiles_per_b) * F::TS;
  const int p0 = 8 * (l >> 4), nval = int(S - s0 < F::TS ? S - s0 : F::TS);
  const int64_t base = b * C * S + s0, left = (int64_t(C) * S - s0) * 2;
  const Buf16 yb(y + base, left), vb((ACT != kNoGate ? v : y) + base, left);
  auto offset = [&](int j, int h) {
    const int c = 16 * (wave + F::W * j) + (l & 15), p = 32 * h + p0;
    return c < C && p < nval ? 2 * (c * int(S) + p) : kOutside;
  };
  u32x4 yr[F::NB][F::H], vr[F::NB][F::H];
#pragma unroll
  for (int j = 0; j < F::NB; ++j)
#pragma unroll
    for (int h = 0; h < F::H; ++h) {
      const int o = offset(j, h);
      yr[j][h] = yb.load(o);
      vr[j][h] = ACT != kNoGate ? vb.load(o) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
  for (int j = 0; j < F::NB; ++j)
#pragma unroll
    for (int h = 0; h < F::H; ++h) {
      opaque(yr[j][h]);
      opaque(vr[j][h]);
    }
  float part[1][F::H][8];
#pragma unroll
  for (int h = 0; h < F::H; ++h)
#pragma unroll
    for (int k = 0; k < 8; ++k) part[0][h][k] = 0.f;
  // u replaces y as its bits (u is exact in the I/O type); zero outside the tensor (act(0) y = 0 with y = 0)
#pragma unroll
  for (int j = 0; j < F::NB; ++j)
#pragma unroll
    for (int h = 0; h < F::H; ++h) {
      float a[8], g[8], ac;
      unpack8<DT>(yr[j][h], a);
      unpack8<DT>(vr[j][h], g);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float u = gate_u<DT, ACT>(a[k], g[k], ac);
        a[k] = u;
        part[0][h][k] = MODE == CHN_LN ? part[0][h][k] + u : fmaf(u, u, part[0][h][k]);
      }
      if constexpr (ACT != kNoGate) yr[j][h] = pack8<DT>(a);
    }
  norm16_sums<F, 1>(part, red, tot);
  float mu[F::H][8], r[F::H][8];
#pragma unroll
  for (int h = 0; h < F::H; ++h) take8(tot + 32 * h + p0, r[h]);
  if constexpr (MODE == CHN_LN) {
#pragma unroll
    for (int h = 0; h < F::H; ++h)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        mu[h][k] = r[h][k] / float(C);
        part[0][h][k] = 0.f;
      }
#pragma unroll
    for (int j = 0; j < F::NB; ++j)
      if (16 * (wave + F::W * j) + (l & 15) < C)
#pragma unroll
        for (int h = 0; h < F::H; ++h) {
          float a[8];
          unpack8<DT>(yr[j][h], a);
#pragma unroll
          for (int k = 0; k < 8; ++k) part[0][h][k] = fmaf(a[k] - mu[h][k], a[k] - mu[h][k], part[0][h][k]);
        }
    norm16_sums<F, 1>(part, red, tot);
#pragma unroll
    for (int h = 0; h < F::H; ++h) take8(tot + 32 * h + p0, r[h]);
  }
#pragma unroll
  for (int h = 0; h < F::H; ++h)
#pragma unroll
    for (int k = 0; k < 8; ++k)
      r[h][k] = MODE == CHN_L2 ? 1.f / fmaxf(Elem<DT>::round(sqrtf(r[h][k])), eps)
                               : rsqrtf(r[h][k] * (1.f / float(C)) + eps);
#pragma unroll
  for (int j = 0; j < F::NB; ++j) {
    const int c = 16 * (wave + F::W * j) + (l & 15);
    const float wc = w && c < C ? w[c] : 1.f, bc = MODE == CHN_LN && bias && c < C ? bias[c] : 0.f;
#pragma unroll
    for (int h = 0; h < F::H; ++h) {
      float a[8];
      unpack8<DT>(yr[j][h], a);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float o = wc * ((MODE == CHN_LN ? a[k] - mu[h][k] : a[k]) * r[h][k]);
        a[k] = MODE == CHN_LN && bias ? o + bc : o;
      }
      const u32x4 q = pack8<DT>(a);
      if (out_blh) {
        const uint32_t e[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (c < C) tile[(32 * h + p0 + k) * ld + c] = uint16_t(e[k >> 1] >> (16 * (k & 1)));
      } else {
        Buf16(out + base, left).store(offset(j, h), q);
      }
    }
  }
  if (!out_blh) return;
  __syncthreads();
  const int C8 = C / 8;
  const float inv = 1.f / float(C8);
  T* o = out + (b * S + s0) * int64_t(C);
  for (int q = t; q < nval * C8; q += F::NT) {
    const int s = chunk_row(q, inv), c = (q - s * C8) * 8;
    *reinterpret_cast<u32x4*>(o + uint32_t(q) * 8) = *reinterpret_cast<const u32x4*>(tile + s * ld + c);
  }
}

// 8 positions of one channel out of the channels-last tile, per 16 lanes of consecutive channels (rows s .. s + 7).
__device__ __forceinline__ u32x4 tile_column8(const uint16_t* tile, int ld, int s, int c0, int l) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef v4s __attribute__((address_space(3)))* lds_v4s;
  const uint16_t* q = tile + (s + ((l >> 2) & 3)) * ld + c0 + 4 * (l & 3);
  const v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(q));
  const v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(q + 4 * ld));
  return __builtin_bit_cast(u32x4, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int DT, int MODE, int ACT, class F>
__global__ __launch_bounds__(F::NT) __attribute__((amdgpu_waves_per_eu(4))) void chnorm16_bwd_kernel(
    const typename Elem<DT>::T* __restrict__ dout, const typename Elem<DT>::T* __restrict__ y,
    const typename Elem<DT>::T* __restrict__ v, const float* __restrict__ w, typename Elem<DT>::T* __restrict__ dy,
    typename Elem<DT>::T* __restrict__ dv, float* __restrict__ dw_part, float* __restrict__ db_part, int C, int64_t S,
    int64_t tiles_per_b, int64_t ntiles, float eps, int in_blh) {
#pragma clang fp contract(off)
  using T = typename Elem<DT>::T;
  constexpr int K = MODE == CHN_LN ? 3 : 2;
  extern __shared__ __align__(16) float smem[];
  const int ld = norm16_ld(C);
  uint16_t* tile = reinterpret_cast<uint16_t*>(smem);
  float* tot = smem + F::TS * ld / 2;
  float* red = tot + K * F::TS;
  const int t = int(threadIdx.x), l = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int p0 = 8 * (l >> 4);
  const int C8 = C / 8;
  const float inv = 1.f / float(C8), invC = 1.f / float(C);
  const int64_t wg = xcd_remap(blockIdx.x, gridDim.x);
  float gw[F::NB], gb[F::NB], wc[F::NB];
#pragma unroll
  for (int j = 0; j < F::NB; ++j) {
    const int c = 16 * (wave + F::W * j) + (l & 15);
    gw[j] = gb[j] = 0.f;
    wc[j] = c < C ? (w ? w[c] : 1.f) : 0.f;
  }
  for (int64_t ti = wg; ti < ntiles; ti += gridDim.x) {
    const int64_t b = ti / tiles_per_b, s0 = (ti % tiles_per_b) * F::TS;
    const int nval = int(S - s0 < F::TS ? S - s0 : F::TS);
    const int64_t base = b * C * S + s0, left = (int64_t(C) * S - s0) * 2;
    const int64_t dbase = in_blh ? (b * S + s0) * int64_t(C) : base;
    const Buf16 yb(y + base, left), vb((ACT != kNoGate ? v : y) + base, left);
    const Buf16 db(dout + dbase, in_blh ? int64_t(nval) * C * 2 : left);
    const Buf16 dyb(dy + base, left), dvb((ACT != kNoGate ? dv : dy) + base, left);
    u32x4 yr[F::NB][F::H], vr[F::NB][F::H], dr[F::NB][F::H];
    auto each = [&](auto&& f) {
#pragma unroll
      for (int j = 0; j < F::NB; ++j)
#pragma unroll
        for (int h = 0; h < F::H; ++h) {
          const int c = 16 * (wave + F::W * j) + (l & 15), p = 32 * h + p0;
          f(j, h, c < C && p < nval ? 2 * (c * int(S) + p) : kOutside);
        }
    };
    constexpr int QN = F::NB * F::H;  // chunks of dout a thread moves at most: TS C8 / NT
    u32x4 q[QN];
    if (in_blh) {
#pragma unroll
      for (int k = 0; k < QN; ++k) {
        const int at = t + k * F::NT;
        q[k] = db.load(at < nval * C8 ? 16 * at : kOutside);
      }
    }
    each([&](int j, int h, int o) {
      yr[j][h] = yb.load(o);
      vr[j][h] = ACT != kNoGate ? vb.load(o) : u32x4{0, 0, 0, 0};
      if (!in_blh) dr[j][h] = db.load(o);
    });
    if (in_blh) {
#pragma unroll
      for (int k = 0; k < QN; ++k) {
        const int at = t + k * F::NT;
        const int s = chunk_row(at, inv), c = (at - s * C8) * 8;
        if (at < nval * C8) *reinterpret_cast<u32x4*>(tile + s * ld + c) = q[k];
      }
      __syncthreads();
      each([&](int j, int h, int o) {
        const int c0 = 16 * (wave + F::W * j);
        dr[j][h] = tile_column8(tile, ld, 32 * h + p0, c0 < C ? c0 : 0, l);
        const uint32_t keep = o == kOutside ? 0u : ~0u;  // what lies past the tile's rows or channels is not dout
        dr[j][h] &= u32x4{keep, keep, keep, keep};
      });
    }
    each([&](int j, int h, int) {
      opaque(yr[j][h]);
      opaque(vr[j][h]);
      opaque(dr[j][h]);
    });
    float part[K][F::H][8];
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int h = 0; h < F::H; ++h)
#pragma unroll
        for (int i = 0; i < 8; ++i) part[k][h][i] = 0.f;
    float mu[F::H][8];
    if constexpr (MODE == CHN_LN) {
      float p1[1][F::H][8];
#pragma unroll
      for (int h = 0; h < F::H; ++h)
#pragma unroll
        for (int i = 0; i < 8; ++i) p1[0][h][i] = 0.f;
      each([&](int j, int h, int) {
        float a[8], g[8], ac;
        unpack8<DT>(yr[j][h], a);
        unpack8<DT>(vr[j][h], g);
#pragma unroll
        for (int k = 0; k < 8; ++k) p1[0][h][k] += gate_u<DT, ACT>(a[k], g[k], ac);
        NSQ_SLOT_FENCE();
      });
      norm16_sums<F, 1>(p1, red, tot);
#pragma unroll
      for (int h = 0; h < F::H; ++h) {
        take8(tot + 32 * h + p0, mu[h]);
#pragma unroll
        for (int k = 0; k < 8; ++k) mu[h][k] = mu[h][k] / float(C);
      }
      // tot is written again after the next barrier
      each([&](int j, int h, int) {
        opaque(yr[j][h]);
        opaque(vr[j][h]);
      });
    }
    // sum of u^2 (LN: of squared deviations), of (w dout) u (LN: deviation), LN: of w dout
    each([&](int j, int h, int o) {
      (void)o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // a word at a time keeps the live values few
        float a[2], g[2], d[2], ac;
        unpack2<DT>(yr[j][h][i], a);
        unpack2<DT>(vr[j][h][i], g);
        unpack2<DT>(dr[j][h][i], d);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int k = 2 * i + e;
          float u = gate_u<DT, ACT>(a[e], g[e], ac);
          if constexpr (MODE == CHN_LN) u = o != kOutside ? u - mu[h][k] : 0.f;
          const float wd = wc[j] * d[e];
          part[0][h][k] = fmaf(u, u, part[0][h][k]);
          part[1][h][k] = fmaf(wd, u, part[1][h][k]);
          if constexpr (MODE == CHN_LN) part[K - 1][h][k] += wd;
        }
        NSQ_SLOT_FENCE();
      }
    });
    norm16_sums<F, K>(part, red, tot);
    each([&](int j, int h, int) {
      opaque(yr[j][h]);
      opaque(vr[j][h]);
      opaque(dr[j][h]);
    });
#pragma unroll
    for (int h = 0; h < F::H; ++h) {
      float r[8], m[8], mg[8];
      take8(tot + 32 * h + p0, r);
      take8(tot + F::TS + 32 * h + p0, m);
      if constexpr (MODE == CHN_LN) take8(tot + (K - 1) * F::TS + 32 * h + p0, mg);
      const bool inside = 32 * h + p0 < nval;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if constexpr (MODE == CHN_L2) {
          const float n = Elem<DT>::round(sqrtf(r[k]));
          r[k] = 1.f / fmaxf(n, eps);
          m[k] = n < eps ? 0.f : m[k] * r[k];
        } else {
          r[k] = rsqrtf(r[k] * invC + eps);
          m[k] = m[k] * r[k] * invC;
          if constexpr (MODE == CHN_LN) mg[k] *= invC;
        }
        // past the tensor u = 0 and, at eps = 0, r = inf: their product would reach gw as NaN
        if (!inside) r[k] = m[k] = 0.f;
      }
#pragma unroll
      for (int j = 0; j < F::NB; ++j) {
        const int c = 16 * (wave + F::W * j) + (l & 15);
        const int off = c < C && 32 * h + p0 < nval ? 2 * (c * int(S) + 32 * h + p0) : kOutside;
        u32x4 o0, o1;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          float a[2], g[2], d[2], e1[2], ac = 0.f;
          unpack2<DT>(yr[j][h][n], a);
          unpack2<DT>(vr[j][h][n], g);
          unpack2<DT>(dr[j][h][n], d);
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int k = 2 * n + e;
            const float u = gate_u<DT, ACT>(a[e], g[e], ac);
            const float xh = (MODE == CHN_LN ? u - mu[h][k] : u) * r[k];
            const float wd = wc[j] * d[e];
            gw[j] = fmaf(d[e], xh, gw[j]);  // dout is zero outside the tensor
            if constexpr (MODE == CHN_LN) gb[j] += d[e];
            const float du = Elem<DT>::round(r[k] * ((MODE == CHN_LN ? wd - mg[k] : wd) - xh * m[k]));
            if constexpr (ACT != kNoGate) {
              e1[e] = Elem<DT>::round(du * a[e]) * gate_dact(ACT, g[e]);
              a[e] = du * ac;
            } else {
              a[e] = e1[e] = du;
            }
          }
          o0[n] = pack2<DT>(a[0], a[1]);
          o1[n] = pack2<DT>(e1[0], e1[1]);
          NSQ_SLOT_FENCE();
        }
        dyb.store(off, o0);
        if constexpr (ACT != kNoGate) dvb.store(off, o1);
        NSQ_SLOT_FENCE();
      }
    }
  }
  // per-channel sums over the lane's positions, then over the position runs of the wave (fixed order)
#pragma unroll
  for (int j = 0; j < F::NB; ++j) {
    const int c = 16 * (wave + F::W * j) + (l & 15);
    float a = gw[j], g = gb[j];
    a += __shfl_xor(a, 16);
    a += __shfl_xor(a, 32);
    if constexpr (MODE == CHN_LN) {
      g += __shfl_xor(g, 16);
      g += __shfl_xor(g, 32);
    }
    if (l < 16 && c < C) {
      if (dw_part) dw_part[wg * C + c] = a;
      if (MODE == CHN_LN && db_part) db_part[wg * C + c] = g;
    }
  }
}

// The configuration for C channels: the fewest blocks a wave that cover them.  The forward takes 256 threads up to 192
// channels, where eight waves would have nothing to do (C = 64, S = 128^2, B = 16 gated: 45 us with 512 threads, the
// tile kernel 32); the backward is held to 512 workgroups by its partial rows and keeps 512 threads.
template <bool BWD, class F>
inline void with_norm16(int C, F&& f) {
  if constexpr (!BWD) {
    if (C <= 64) return f(Norm16Cfg<1, 2, 256>{});
    if (C <= 128) return f(Norm16Cfg<2, 2, 256>{});
    if (C <= 192) return f(Norm16Cfg<3, 1, 256>{});
  } else {
    if (C <= 128) return f(Norm16Cfg<1, 1, 512>{});
  }
  if (C <= 256) return f(Norm16Cfg<2, 1, 512>{});
  if (C <= 384) return f(Norm16Cfg<3, 1, 512>{});
  if (C <= 512) return f(Norm16Cfg<2, 1, 1024>{});
  if (C <= 768) return f(Norm16Cfg<3, 1, 1024>{});
  if (C <= 1024) return f(Norm16Cfg<4, 1, 1024>{});
  return f(Norm16Cfg<6, 1, 1024>{});
}

}  // namespace
}  // namespace nsq
