// The causal 1D convolution on the fused plan (FFT lengths F = 1024 to 16384)
// in the ring z^F = -1, forward (gates included) and backward.
//
// A packed real transform (even and odd samples, fused_fwd_kernel) unpacks the
// Hermitian spectrum through LDS: at F = 16384 two 70 KB tiles in the backward,
// so one workgroup of 8 waves a CU, 13 LDS round trips an image, and 10 us a
// transform per CU where its VALU and LDS work is under 3.  Here, with
// M = F / 2, u[n] - i u[n + M] times W_{4M}^n followed by an M-point complex
// DFT evaluates a real row at the M roots of z^M = -i (the conjugates are the
// other M roots of z^F = -1).  Spectra are M plain complex points, so a
// transform's last pass stays in registers, is multiplied there and is the
// inverse's first pass; one tile serves every transform of a workgroup, and
// M / 8 threads (16 waves at F = 16384) hold 8 points each of the filter's
// spectrum, of the filter gradient's and of the current image's: 4 LDS round
// trips a transform at F = 16384.  Nothing wraps into a kept window:
// F >= L + K - 1 holds every lag of the products.
// Passes: radix 8, the first (and the inverse's last) radix 2 or 4 where 8
// does not divide out, so that every thread always holds 8 points.  A radix-16
// first pass on half of the threads spills (600 us where radix 8 takes 314).
// Rows are read and written as single elements, consecutive across lanes; the
// next row's are in flight during the current transform.
// What bounds it: LDS passes and their barriers; at B=4 H=1024 L=K=8192 bf16
// the forward moves 1.0 TB/s and the backward 0.85.
// Measured (us, packed transform -> ring, shortcut, kernel time), L = K:
//   bf16, B x H x L     forward          backward
//   4 x 1024 x 512      23.4 ->  11.4     76 ->  26
//   4 x 1024 x 1024     31.3 ->  22.0     89 ->  37
//   4 x 1024 x 2048     54.3 ->  36.6    115 ->  58
//   4 x 1024 x 4096      133 ->  76      391 -> 116
//   4 x 1024 x 8192      239 -> 166      513 -> 314
//   1 x  256 x 8192     24.3 ->  20.3     45 ->  30
//   1 x   64 x 4096     13.4 ->  10.8
// with the fold's roots as products; from the table (ring_fold), as now, 2 % more
// at L = 512 and 8192 and 8 to 13 % between.
// fp32 within 6 % of these.  Small grids ran two transforms side by side in
// one workgroup before (the 1-row figures): the ring is faster there too but for
// 64 to 256 rows of F = 4096 with a short filter (9.3 -> 10.3), so it takes every
// grid size.  Error against float64 (B=2 H=128 fp32), packed -> ring: y 1.86 -> 1.79e-7 at L = 512, 2.02 -> 2.05e-7 at
// 2048, 2.16 -> 2.12e-7 at 4096, 2.49 -> 2.15e-7 at 8192; gx and gk below the packed transform's at every length.
#pragma once

#include "gate.h"

namespace nsq {

template <int LOGM_>
struct RingCfg {
  static constexpr int LOGM = LOGM_, M = 1 << LOGM, T = M / 8;
  // log2 of the first pass's radix; the others are radix 8, the last of them in registers
  static constexpr int R0 = LOGM % 3 ? LOGM % 3 : 3, R = 1 << R0, NR = M / R, PER = 8 / R;
  static constexpr int MID = (LOGM - R0) / 3 - 1;
  static_assert(LOGM >= 9 && LOGM <= 13, "RingCfg: length out of range");
};

// W_{4M}^n of a first-pass butterfly's inputs n = j + r M / R, r < R.  Every sample meets one on its way in and out: as
// products of two rounded roots they cost a tenth of the transform's error (2.46e-7 against 2.16e-7 of the packed
// transform at B=2 H=128 L=4096 fp32), so they come from the table.  M = 8192 is beyond its 2^14 segment: there odd j
// are one product (by W_32768), and r = 1 one more (W_8), still 2.3e-7 where the hardware's sine and cosine gave 3.2e-7
// and the packed transform 2.5e-7 (L=8192); two table reads and a select a sample instead cost the backward 10%.
template <class C>
__device__ __forceinline__ void ring_fold(const float2* __restrict__ tw, int j, float2 (&w)[C::R]) {
  constexpr int LOGB = C::LOGM + 2;
  if constexpr (LOGB <= 14) {
#pragma unroll
    for (int r = 0; r < C::R; ++r) w[r] = tw[(1 << LOGB) + j + r * C::NR];
  } else {
    static_assert(LOGB == 15 && C::R == 2, "ring_fold: roots of unity");
    const float2 e = tw[(1 << 14) + (j >> 1)];
    w[0] = cmul_fixed(e, make_float2(1.f, j & 1 ? -1.91747597e-4f : 0.f));  // cos rounds to 1
    w[1] = cmul_fixed(w[0], make_float2(0.70710678118654752440f, -0.70710678118654752440f));
  }
}

// One pass over the thread's 8 points: ld(i, j, v) reads butterfly j's inputs, st(i, base, v) takes outputs base + r NS.
template <int LOGN, int LOGR, int LOGNS, bool INV, int T, class LD, class ST>
__device__ __forceinline__ void ring_pass(LD&& ld, ST&& st, const float2* __restrict__ tw) {
  constexpr int R = 1 << LOGR, NR = 1 << (LOGN - LOGR), NS = 1 << LOGNS, PER = NR / T;
  static_assert(PER * R == 8, "ring_pass: 8 points per thread");
  const int tid = opaque_tid();
  float2 v[PER][R];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int j = tid + i * T, k = j & (NS - 1);
    float2 w[R];
    if constexpr (LOGNS > 0) pass_twiddles<R>(TwTable(tw), NS * R, k, w);
    ld(i, j, v[i]);
    if constexpr (LOGNS > 0)
#pragma unroll
      for (int r = 1; r < R; ++r) v[i][r] = INV ? cmulc(v[i][r], w[r]) : cmul(v[i][r], w[r]);
    dft<R, INV>(v[i]);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int j = tid + i * T, k = j & (NS - 1);
    st(i, ((j - k) << LOGR) + k, v[i]);
  }
  __syncthreads();
}

// The middle radix-8 passes, from 2^LOGNS points done.
template <class C, int LOGNS, bool INV>
__device__ __forceinline__ void ring_middle(float2* lds, const float2* __restrict__ tw) {
  static_for<0, C::MID>([&](auto n) {
    constexpr int NSL = LOGNS + 3 * decltype(n)::value, NS = 1 << NSL;
    ring_pass<C::LOGM, 3, NSL, INV, C::T>(
        [&](int, int j, float2 (&z)[8]) {
          const float2* q = lds + pad16(j);
#pragma unroll
          for (int r = 0; r < 8; ++r) z[r] = q[pad16(r * C::T)];
        },
        [&](int, int base, const float2 (&z)[8]) {
#pragma unroll
          for (int r = 0; r < 8; ++r) lds[pad16(base + r * NS)] = z[r];
        },
        tw);
  });
}

// One real row's first-pass inputs: raw bits of samples n = tid + i T + r M / R.
template <int DT, class C>
struct RingRow {
  uint32_t w[C::PER][C::R];
  __device__ __forceinline__ void load(const RowBuf<DT, false>& b) {
    const int t = opaque_tid();
#pragma unroll
    for (int i = 0; i < C::PER; ++i)
#pragma unroll
      for (int r = 0; r < C::R; ++r) w[i][r] = b.elem_halo_bits(t + i * C::T + r * C::NR);
  }
};

// A row -> the thread's 8 spectral points: lo(i, r, n) is the sample n = tid + i T + r M / R, hi(n) samples from M on
// (WIDE).  TABLE: the last pass's roots all from the table, not four of seven as products (fp32 rows: their results show
// it, 16-bit ones do not).
template <class C, bool WIDE, bool TABLE = false, class LO, class HI>
__device__ __forceinline__ void ring_spectrum(float2* lds, LO&& lo, HI&& hi, float2 (&v)[8],
                                              const float2* __restrict__ tw) {
  ring_pass<C::LOGM, C::R0, 0, false, C::T>(
      [&](int i, int j, float2 (&z)[C::R]) {
        float2 wf[C::R];
        ring_fold<C>(tw, j, wf);
#pragma unroll
        for (int r = 0; r < C::R; ++r) {
          const float2 w = wf[r];
          const float a = lo(i, r, j + r * C::NR), c = WIDE ? hi(j + r * C::NR + C::M) : 0.f;
          z[r] = make_float2(fmaf(c, w.y, a * w.x), fmaf(-c, w.x, a * w.y));
        }
      },
      [&](int, int base, const float2 (&z)[C::R]) {
#pragma unroll
        for (int r = 0; r < C::R; ++r) lds[pad16(base + r)] = z[r];
      },
      tw);
  ring_middle<C, C::R0, false>(lds, tw);
  const int j = opaque_tid();
  float2 w[8];
  if constexpr (TABLE) {
#pragma unroll
    for (int r = 1; r < 8; ++r) w[r] = TwTable(tw).load(C::M, (r * j) & (C::M - 1));
  } else {
    pass_twiddles<8>(TwTable(tw), C::M, j, w);
  }
  const float2* q = lds + pad16(j);
  v[0] = q[0];
#pragma unroll
  for (int r = 1; r < 8; ++r) v[r] = cmul(q[pad16(r * C::T)], w[r]);
  dft<8, false>(v);
}

// The thread's 8 points -> out(n, u[n], u[n + M]), unscaled.  Ends with a barrier.
template <class C, class OUT>
__device__ __forceinline__ void ring_inverse(float2* lds, float2 (&v)[8], OUT&& out, const float2* __restrict__ tw) {
  dft<8, true>(v);
  __syncthreads();  // the spectrum's last pass has read the tile
  {
    const int j = opaque_tid();
#pragma unroll
    for (int r = 0; r < 8; ++r) lds[pad16(8 * j + r)] = v[r];
  }
  __syncthreads();
  ring_middle<C, 3, true>(lds, tw);
  ring_pass<C::LOGM, C::R0, C::LOGM - C::R0, true, C::T>(
      [&](int, int j, float2 (&z)[C::R]) {
        const float2* q = lds + pad16(j);
#pragma unroll
        for (int r = 0; r < C::R; ++r) z[r] = q[pad16(r * C::NR)];
      },
      [&](int, int base, const float2 (&z)[C::R]) {  // base = j < NR: outputs j + r NR
        float2 wf[C::R];
        ring_fold<C>(tw, base, wf);
#pragma unroll
        for (int r = 0; r < C::R; ++r) {
          const float2 a = cmulc(z[r], wf[r]);
          out(base + r * C::NR, a.x, -a.y);
        }
      },
      tw);
}

// Arguments as fused_fwd_kernel's (no fold, no shift): grid (H, ceil(B / b_per_wg)).  GATE: x is the query; the row
// transformed is z = q act1(k), and the outputs are y1 act2(v) and, if kept, y1.
template <int LOGM, int DT, bool WIDE, bool GATE>
__global__ __launch_bounds__(RingCfg<LOGM>::T) __attribute__((amdgpu_waves_per_eu(4))) void ring_fwd_kernel(
    const typename Elem<DT>::T* __restrict__ x, const float* __restrict__ k,
    const typename Elem<DT>::T* __restrict__ s, typename Elem<DT>::T* __restrict__ y, int B, int H, int L, int K,
    int b_per_wg, const float2* __restrict__ tw, int kfilm, GateArgs ga) {
  using C = RingCfg<LOGM>;
  using ET = typename Elem<DT>::T;
  __shared__ float2 lds[Padded<C::M>::SIZE];
  const int h = int(blockIdx.x);
  const int b0 = int(blockIdx.y) * b_per_wg, b1 = min(B, b0 + b_per_wg);
  const int64_t hk = kfilm ? int64_t(b0) * H + h : h;
  const auto row = [&](const void* p, int b) {
    return RowBuf<DT, false>(static_cast<const ET*>(p) + (int64_t(b) * H + h) * L, L);
  };
  RingRow<DT, C> rx, rk;
  const auto load = [&](int b) {
    rx.load(row(x, b));
    if constexpr (GATE) rk.load(row(ga.kg, b));
  };
  load(b0);
  float2 kv[8];
  {
    const RowBuf<NSQ_DTYPE_F32, false> kb(k + hk * K, K);
    RingRow<NSQ_DTYPE_F32, C> kr;
    kr.load(kb);
    ring_spectrum<C, WIDE, DT == NSQ_DTYPE_F32>(
        lds, [&](int i, int r, int) { return __uint_as_float(kr.w[i][r]); }, [&](int n) { return kb.elem(n); }, kv,
        tw);
  }
  const float scale = 1.f / float(C::M);
#pragma unroll
  for (int r = 0; r < 8; ++r) kv[r] = cscale(kv[r], scale);  // a power of two: exact
  const float sv = s ? Elem<DT>::round(Elem<DT>::load(s, h)) : 0.f;
  for (int b = b0; b < b1; ++b) {
    const RowBuf<DT, false> xb = row(x, b), kb = row(GATE ? ga.kg : x, b), yb = row(y, b);
    const auto z = [&](int n) { return GATE ? gate1<DT>(ga.act1, xb.elem(n), kb.elem(n)) : xb.elem(n); };
    float2 v[8];
    ring_spectrum<C, WIDE, DT == NSQ_DTYPE_F32>(
        lds,
        [&](int i, int r, int) {
          const float a = RowBuf<DT, false>::bits_to_f32(rx.w[i][r]);
          return GATE ? gate1<DT>(ga.act1, a, RowBuf<DT, false>::bits_to_f32(rk.w[i][r])) : a;
        },
        z, v, tw);
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = cmul(v[r], kv[r]);
    if (b + 1 < b1) load(b + 1);
    const auto put = [&](int n, float c) {
      c = epilogue<DT>(c, s != nullptr, sv, s ? z(n) : 0.f);
      if constexpr (GATE) {
#pragma clang fp contract(off)
        if (ga.y1) row(ga.y1, b).store_elem(n, c);
        c = c * Elem<DT>::round(gate_act(ga.act2, row(ga.v, b).elem(n)));
      }
      yb.store_elem(n, c);
    };
    ring_inverse<C>(
        lds, v,
        [&](int n, float lo, float hi) {
          put(n, lo);
          if (WIDE) put(n + C::M, hi);
        },
        tw);
  }
}

// Arguments as fused_bwd_kernel's (no fold, no shift): grid (H, kfilm ? B : 1).  WIDE: a row or the filter reaches
// past M samples.
template <int LOGM, int DT, bool WIDE>
__global__ __launch_bounds__(RingCfg<LOGM>::T) __attribute__((amdgpu_waves_per_eu(4))) void ring_bwd_kernel(
    const typename Elem<DT>::T* __restrict__ g, const typename Elem<DT>::T* __restrict__ x,
    const float* __restrict__ k, const typename Elem<DT>::T* __restrict__ s, typename Elem<DT>::T* __restrict__ gx,
    float* __restrict__ gk, float* __restrict__ gs, int B, int H, int L, int K, const float2* __restrict__ tw,
    int kfilm) {
  using C = RingCfg<LOGM>;
  __shared__ float2 lds[Padded<C::M>::SIZE];
  const int h = int(blockIdx.x);
  const int b0 = kfilm ? int(blockIdx.y) : 0, b1 = kfilm ? b0 + 1 : B;
  const int64_t hk = kfilm ? int64_t(b0) * H + h : h;
  const auto row = [&](const typename Elem<DT>::T* p, int b) {
    return RowBuf<DT, false>(p + (int64_t(b) * H + h) * L, L);
  };
  float2 kv[8], q[8];
  {
    const RowBuf<NSQ_DTYPE_F32, false> kb(k + hk * K, K);
    RingRow<NSQ_DTYPE_F32, C> kr;
    kr.load(kb);
    ring_spectrum<C, WIDE>(
        lds, [&](int i, int r, int) { return __uint_as_float(kr.w[i][r]); }, [&](int n) { return kb.elem(n); }, kv,
        tw);
  }
  const float scale = 1.f / float(C::M);
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    kv[r] = cscale(kv[r], scale);  // a power of two: exact
    q[r] = make_float2(0.f, 0.f);
  }
  const float sv = s ? Elem<DT>::round(Elem<DT>::load(s, h)) : 0.f;
  RingRow<DT, C> rx, rg;
  rx.load(row(x, b0));
  for (int b = b0; b < b1; ++b) {
    const RowBuf<DT, false> xb = row(x, b), gb = row(g, b), ob = row(gx, b);
    float2 xs[8], v[8];
    rg.load(gb);
    ring_spectrum<C, WIDE>(
        lds, [&](int i, int r, int) { return RowBuf<DT, false>::bits_to_f32(rx.w[i][r]); },
        [&](int n) { return xb.elem(n); }, xs, tw);
    ring_spectrum<C, WIDE>(
        lds, [&](int i, int r, int) { return RowBuf<DT, false>::bits_to_f32(rg.w[i][r]); },
        [&](int n) { return gb.elem(n); }, v, tw);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      q[r] = cadd(q[r], cmulc(v[r], xs[r]));
      v[r] = cmulc(v[r], kv[r]);
    }
    if (b + 1 < b1) rx.load(row(x, b + 1));
    ring_inverse<C>(
        lds, v,
        [&](int n, float lo, float hi) {
          ob.store_elem(n, epilogue<DT>(lo, s != nullptr, sv, s ? gb.elem(n) : 0.f));
          if (WIDE) ob.store_elem(n + C::M, epilogue<DT>(hi, s != nullptr, sv, s ? gb.elem(n + C::M) : 0.f));
        },
        tw);
  }
  const RowBuf<NSQ_DTYPE_F32, false> kb(gk + hk * K, K);
  ring_inverse<C>(
      lds, q,
      [&](int n, float lo, float hi) {
        kb.store_elem(n, lo * scale);
        if (WIDE) kb.store_elem(n + C::M, hi * scale);
        if (n == 0 && gs) gs[hk] = lo * scale;  // lag 0
      },
      tw);
}

}  // namespace nsq
