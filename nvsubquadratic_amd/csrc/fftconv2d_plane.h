// 2D convolution of small planes, whole images in LDS (forward and backward).
//
// Token grids and small fields (a plane of F0 x F2 <= 128 x 128 real points)
// through the separable passes of fftconv_nd_impl.h cost six kernels and a
// round trip of the padded complex spectrum per pass: at B=64 H=384, 14 x 14
// tokens (F = 32 x 32) an image of 392 bytes moves 4 KB of spectrum six times,
// and the adjoint alone took 146 us.  Here a workgroup of F0 F2 / 16 threads
// owns one channel and a share of the batch, keeps the filter's spectrum in
// registers (8 points a thread) and takes each image from its samples to its
// outputs in LDS; HBM moves x, y (g, x, gx) and the filter only.
//
// Transform.  The last axis uses the ring z^{F2} = -1 instead of z^{F2} = 1:
// with M = F2 / 2, u[n] - i u[n + M] times W_{4M}^n, then an M-point complex
// DFT, evaluates the real row at the M roots of z^M = -i, whose conjugates are
// the other M roots of z^{F2} = -1.  Products of spectra are products in that
// ring, conjugation is index reversal, and a term that leaves the row at F2
// returns with its sign changed.  The kept window of a zero-padded axis holds
// no such term (F2 >= S2 + ceil(K2 / 2)), so the results are the usual ones,
// and a spectrum is F0 x M plain complex points: no Hermitian unpacking, no
// packed DC / Nyquist column, so the last column pass, the product and the
// first inverse column pass are one pass in registers (its radix-8 outputs
// j + r F0 / 8 are the inverse's inputs).  Axis 0 is an ordinary cyclic
// transform: zero-padded or periodic.
//
// Images enter and leave as flat runs of S0 S2 elements, four per lane and
// access: raw bits into LDS (the next image's are loaded before the current
// one is transformed), where the first row pass reads single samples, and the
// kept window as floats into the tile, from which the epilogue (shortcut,
// gates) stores.  Single 2-byte accesses from the row passes themselves made
// 72 vector-memory instructions an image and wave, and those the bound: 436
// against 296 us at B=64 H=384, 64 x 16 (F = 64 x 32), forward + backward.
//
// Bound now by issue and LDS (VALU and LDS each about a third busy, the passes
// of an image one after the other).  Measured forward + backward in bf16 (us,
// separable passes -> here): that shape 698 -> 296; B=64 H=384 16 x 16, K = 31
// 323 -> 155 (gated 405 -> 184); B=8 H=256 64 x 64 260 -> 216; B=2 H=64 7 x 7
// 88 -> 19 (launches).
//
// Shifts (crop offsets, the circular alignment and the adjoints' lags) are
// index arithmetic where a row leaves its last pass: mod F0 along axis 0, with
// the sign of the wrap along axis 2.
#pragma once

#include "gate.h"

namespace nsq {

// F0 x M complex points, 8 per thread.
template <int LOGF0_, int LOGM_>
struct Plane2 {
  static constexpr int LOGF0 = LOGF0_, LOGM = LOGM_, F0 = 1 << LOGF0, M = 1 << LOGM, T = F0 * M / 8;
  static constexpr int RS = Padded<M>::SIZE;  // LDS row stride (complex)
  static_assert(LOGF0 >= 4 && LOGM >= 3 && T >= 64 && T <= 1024, "Plane2: size out of range");
};

struct Plane2Geom {
  int B, H, S0, S2, K0, K2;
  int sh0, o2;  // shift along axis 0 (crop offset or circular alignment), crop offset along axis 2
  int kfilm, per_wg, vec;  // vec: every image starts and ends on a whole access of four elements
};

// Roots in LDS, staged once per workgroup: W_{F0}^j, W_M^j and W_{4M}^n (n < M).  From the table in memory a pass's
// roots are four vector-memory loads that wait behind the images' (or, hoisted out of the image loop, 100 registers).
template <int N>
struct LdsRoots {
  const float2* t;
  __device__ __forceinline__ float2 load(int seg, int idx) const { return t[(idx * (N / seg)) & (N - 1)]; }
};
template <class P>
struct Plane2Roots {
  LdsRoots<P::F0> col;
  LdsRoots<P::M> row;
  const float2* fold;
  static constexpr int SIZE = P::F0 + 2 * P::M;
  // ends with a barrier
  __device__ __forceinline__ Plane2Roots(float2* to, const float2* __restrict__ tw)
      : col{to}, row{to + P::F0}, fold(to + P::F0 + P::M) {
    const TwTable tt(tw);
    const int t = int(threadIdx.x);
    for (int i = t; i < P::F0; i += P::T) to[i] = tt.load(P::F0, i);
    for (int i = t; i < P::M; i += P::T) {
      to[P::F0 + i] = tt.load(P::M, i);
      to[P::F0 + P::M + i] = tt.load(4 * P::M, i);
    }
    __syncthreads();
  }
};

// One radix-2^LOGR Stockham pass over CNT transforms (rows: TMAJOR false; columns: true) of which those with need(m)
// run; ld(m, n) -> value, st(m, n, v).  A barrier separates all reads from the writes and ends the pass.
template <int LOGN, int LOGR, int LOGNS, bool INV, int CNT, int T, bool TMAJOR, class NEED, class LD, class ST,
          class TT>
__device__ __forceinline__ void plane2_pass(NEED&& need, LD&& ld, ST&& st, const TT& tt) {
  constexpr int R = 1 << LOGR, NR = 1 << (LOGN - LOGR), NS = 1 << LOGNS, PER = CNT * NR / T;
  static_assert(CNT * NR % T == 0, "plane2_pass: tile not divisible by threads");
  const int tid = opaque_tid();
  float2 v[PER][R];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int bf = tid + i * T;
    const int m = TMAJOR ? bf % CNT : bf >> (LOGN - LOGR), j = TMAJOR ? bf / CNT : bf & (NR - 1), k = j & (NS - 1);
    if (!need(m)) continue;
    float2 w[R];
    if constexpr (LOGNS > 0) pass_twiddles<R>(tt, NS * R, k, w);
#pragma unroll
    for (int r = 0; r < R; ++r) v[i][r] = ld(m, j + r * NR);
    if constexpr (LOGNS > 0)
#pragma unroll
      for (int r = 1; r < R; ++r) v[i][r] = INV ? cmulc(v[i][r], w[r]) : cmul(v[i][r], w[r]);
    dft<R, INV>(v[i]);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int bf = tid + i * T;
    const int m = TMAJOR ? bf % CNT : bf >> (LOGN - LOGR), j = TMAJOR ? bf / CNT : bf & (NR - 1), k = j & (NS - 1);
    if (!need(m)) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) st(m, ((j - k) << LOGR) + k + r * NS, v[i][r]);
  }
  __syncthreads();
}

template <class P>
__device__ __forceinline__ float2& plane2_at(float2* lds, int row, int n) {
  return lds[row * P::RS + pad16(n)];
}

// Real rows (u(row, n), rows < nrows) -> the thread's 8 spectral points: column tid % M, frequencies tid / M + r F0/8.
// wide: samples n >= M may be nonzero.
template <class P, class U>
__device__ __forceinline__ void plane2_spectrum(float2* lds, U&& u, int nrows, bool wide, float2 (&v)[8],
                                                const Plane2Roots<P>& tw) {
  const auto rows = [&](int m) { return m < nrows; };
  const auto all = [](int) { return true; };
  const auto in = [&](int m, int n) {
    const float2 w = tw.fold[n];
    const float a = u(m, n);
    const float b = wide ? u(m, n + P::M) : 0.f;
    return make_float2(fmaf(b, w.y, a * w.x), fmaf(-b, w.x, a * w.y));
  };
  const auto rd = [&](int m, int n) { return plane2_at<P>(lds, m, n); };
  const auto wr = [&](int m, int n, float2 z) { plane2_at<P>(lds, m, n) = z; };
  plane2_pass<P::LOGM, 3, 0, false, P::F0, P::T, false>(rows, in, wr, tw.row);
  if constexpr (P::LOGM > 3) plane2_pass<P::LOGM, P::LOGM - 3, 3, false, P::F0, P::T, false>(rows, rd, wr, tw.row);
  const auto cin = [&](int c, int n) { return n < nrows ? plane2_at<P>(lds, n, c) : make_float2(0.f, 0.f); };
  const auto crd = [&](int c, int n) { return plane2_at<P>(lds, n, c); };
  const auto cwr = [&](int c, int n, float2 z) { plane2_at<P>(lds, n, c) = z; };
  constexpr int L1 = P::LOGF0 - 3 > 3 ? 1 : P::LOGF0 - 3;  // first radix; 128 points: 2, 8, 8
  plane2_pass<P::LOGF0, L1, 0, false, P::M, P::T, true>(all, cin, cwr, tw.col);
  if constexpr (L1 + 3 < P::LOGF0) plane2_pass<P::LOGF0, 3, L1, false, P::M, P::T, true>(all, crd, cwr, tw.col);
  const int tid = opaque_tid(), c = tid & (P::M - 1), j = tid >> P::LOGM;
  float2 w[8];
  pass_twiddles<8>(tw.col, P::F0, j, w);
  v[0] = crd(c, j);
#pragma unroll
  for (int r = 1; r < 8; ++r) v[r] = cmul(crd(c, j + r * (P::F0 / 8)), w[r]);
  dft<8, false>(v);
}

// The thread's 8 points of a spectrum -> out(row, n, u[n], u[n + M]) of the rows with need(row), unscaled.  Ends
// with a barrier.
template <class P, class NEED, class OUT>
__device__ __forceinline__ void plane2_inverse(float2* lds, float2 (&v)[8], NEED&& need, OUT&& out,
                                               const Plane2Roots<P>& tw) {
  const auto all = [](int) { return true; };
  dft<8, true>(v);
  __syncthreads();  // the spectrum's last pass has read the tile
  const int tid = opaque_tid(), c = tid & (P::M - 1), j = tid >> P::LOGM;
#pragma unroll
  for (int r = 0; r < 8; ++r) plane2_at<P>(lds, 8 * j + r, c) = v[r];
  __syncthreads();
  const auto crd = [&](int cc, int n) { return plane2_at<P>(lds, n, cc); };
  const auto cwr = [&](int cc, int n, float2 z) { plane2_at<P>(lds, n, cc) = z; };
  if constexpr (P::LOGF0 > 6) {
    plane2_pass<P::LOGF0, 3, 3, true, P::M, P::T, true>(all, crd, cwr, tw.col);
    plane2_pass<P::LOGF0, P::LOGF0 - 6, 6, true, P::M, P::T, true>(all, crd, cwr, tw.col);
  } else {
    plane2_pass<P::LOGF0, P::LOGF0 - 3, 3, true, P::M, P::T, true>(all, crd, cwr, tw.col);
  }
  const auto rd = [&](int m, int n) { return plane2_at<P>(lds, m, n); };
  const auto wr = [&](int m, int n, float2 z) { plane2_at<P>(lds, m, n) = z; };
  if constexpr (P::LOGM > 3) plane2_pass<P::LOGM, P::LOGM - 3, 0, true, P::F0, P::T, false>(need, rd, wr, tw.row);
  const auto emit = [&](int m, int n, float2 z) {
    const float2 a = cmulc(z, tw.fold[n]);
    out(m, n, a.x, -a.y);
  };
  plane2_pass<P::LOGM, 3, P::LOGM - 3, true, P::F0, P::T, false>(need, rd, emit, tw.row);
}

// A filter as a range-checked buffer: (row, n) outside reads as zero and stores nothing.
struct Plane2Filter {
  RowBuf<NSQ_DTYPE_F32, false> r;
  int rows, cols;
  __device__ __forceinline__ Plane2Filter(const float* p, int rows_, int cols_)
      : r(p, int64_t(rows_) * cols_), rows(rows_), cols(cols_) {}
  __device__ __forceinline__ int at(int row, int n) const {
    return (unsigned(row) < unsigned(rows) && unsigned(n) < unsigned(cols)) ? row * cols + n : rows * cols;
  }
};

// Four elements of an image per lane and access j < 4 (F0 F2 = 16 T elements at most): element 4 (t + j T).
template <int DT>
struct Plane2Vec {
  static constexpr int W = DT == NSQ_DTYPE_F32 ? 4 : 2;  // words
  using U = uint32_t __attribute__((ext_vector_type(W)));
  U u;
  __device__ __forceinline__ void load(const RowBuf<DT, false>& r, int e, bool vec) {
    if (vec) {
      const int off = e * int(sizeof(typename Elem<DT>::T));
      if constexpr (W == 4)
        u = __builtin_bit_cast(U, __builtin_amdgcn_raw_buffer_load_b128(r.r, off, 0, 0));
      else
        u = __builtin_bit_cast(U, __builtin_amdgcn_raw_buffer_load_b64(r.r, off, 0, 0));
    } else if constexpr (W == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = r.elem_halo_bits(e + i);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) u[i] = r.elem_halo_bits(e + 2 * i) | (r.elem_halo_bits(e + 2 * i + 1) << 16);
    }
  }
  __device__ __forceinline__ void get(float (&f)[4]) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (W == 4)
        f[i] = __uint_as_float(u[i]);
      else
        f[i] = RowBuf<DT, false>::bits_to_f32((i & 1) ? u[i >> 1] >> 16 : u[i >> 1] & 0xffffu);
    }
  }
  __device__ __forceinline__ void set(const float (&f)[4]) {
    if constexpr (W == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = __float_as_uint(f[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (DT == NSQ_DTYPE_BF16)
          u[i] = f32x2_to_bf16x2_bits(f[2 * i], f[2 * i + 1]);
        else
          u[i] = __builtin_bit_cast(uint32_t, __floats2half2_rn(f[2 * i], f[2 * i + 1]));
      }
    }
  }
  __device__ __forceinline__ void store(const RowBuf<DT, false>& r, int e, bool vec) const {
    if (vec) {
      const int off = e * int(sizeof(typename Elem<DT>::T));
      if constexpr (W == 4)
        __builtin_amdgcn_raw_buffer_store_b128(u, r.r, off, 0, 0);
      else
        __builtin_amdgcn_raw_buffer_store_b64(u, r.r, off, 0, 0);
    } else {
      float f[4];
      get(f);
#pragma unroll
      for (int i = 0; i < 4; ++i) r.store_elem(e + i, f[i]);
    }
  }
};

// LDS: the tile, the roots, then one image's raw elements (rounded up to a whole access).
template <class P>
__host__ __device__ constexpr size_t plane2_tile_bytes() {
  return size_t(P::F0 * P::RS + Plane2Roots<P>::SIZE) * sizeof(float2);
}
template <class P, int DT>
inline size_t plane2_lds(const Plane2Geom& g) {
  return plane2_tile_bytes<P>() + (size_t(g.S0) * g.S2 + 3) / 4 * 4 * sizeof(typename Elem<DT>::T);
}

// Index along axis 2 of the adjoints: position p of a row (p >= F2 - o2 wrapped, sign changed) as p + o2.
template <class P>
__device__ __forceinline__ int plane2_lag(int p, int o2, float& v) {
  const int t = p + o2;
  if (t < 2 * P::M) return t;
  v = -v;
  return t - 2 * P::M;
}

// The images of a call: x-side operands (x; gated: q and its gate input kg), and what the epilogues read and write
// beyond the conv's own tensors.
template <int DT, class P, bool GATED>
struct Plane2Io {
  using ET = typename Elem<DT>::T;
  Plane2Geom g;
  int n;       // elements of an image
  ET* raw;     // LDS
  float* flat;  // LDS: the tile, as the kept window
  __device__ __forceinline__ Plane2Io(const Plane2Geom& g_, unsigned char* sm)
      : g(g_), n(g_.S0 * g_.S2), raw(reinterpret_cast<ET*>(sm + plane2_tile_bytes<P>())),
        flat(reinterpret_cast<float*>(sm)) {}
  __device__ __forceinline__ RowBuf<DT, false> image(const void* p, int b, int h) const {
    return RowBuf<DT, false>(static_cast<const ET*>(p) + (int64_t(b) * g.H + h) * n, n);
  }
  template <class F>
  __device__ __forceinline__ void each(F&& f) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = 4 * (int(threadIdx.x) + j * P::T);
      if (e < n) f(j, e);
    }
  }
  __device__ __forceinline__ void load(const void* p, int b, int h, Plane2Vec<DT> (&v)[4]) const {
    const RowBuf<DT, false> r = image(p, b, h);
    each([&](int j, int e) { v[j].load(r, e, g.vec); });
  }
  __device__ __forceinline__ void to_raw(const Plane2Vec<DT> (&v)[4]) const {
    each([&](int j, int e) { *reinterpret_cast<typename Plane2Vec<DT>::U*>(raw + e) = v[j].u; });
  }
  // a act(b), rounded as the gates round, in place of a
  __device__ __forceinline__ void gate(int act, Plane2Vec<DT> (&a)[4], const Plane2Vec<DT> (&b)[4]) const {
    each([&](int j, int) {
      float x[4], y[4];
      a[j].get(x);
      b[j].get(y);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = gate1<DT>(act, x[i], y[i]);
      a[j].set(x);
    });
  }
  __device__ __forceinline__ float sample(int m, int i) const {
    return unsigned(i) < unsigned(g.S2) ? Elem<DT>::load(raw, m * g.S2 + i) : 0.f;
  }
  __device__ __forceinline__ void keep(int row, int i, float c) const {
    if (unsigned(i) < unsigned(g.S2)) flat[row * g.S2 + i] = c;
  }
  __device__ __forceinline__ void get(int e, float (&c)[4], float (&r)[4]) const {
    const float4 f = *reinterpret_cast<const float4*>(flat + e);
    c[0] = f.x; c[1] = f.y; c[2] = f.z; c[3] = f.w;
    Plane2Vec<DT> v;
    v.u = *reinterpret_cast<const typename Plane2Vec<DT>::U*>(raw + e);
    v.get(r);
  }
};

template <int DT, class P, bool GATED>
__global__ __launch_bounds__(P::T) void plane2_fwd_kernel(const typename Elem<DT>::T* __restrict__ x,
                                                          const float* __restrict__ k,
                                                          const typename Elem<DT>::T* __restrict__ s,
                                                          typename Elem<DT>::T* __restrict__ y, Plane2Geom g,
                                                          GatedIO ga, const float2* __restrict__ roots) {
  extern __shared__ __align__(16) unsigned char plane2_sm[];
  float2* lds = reinterpret_cast<float2*>(plane2_sm);
  const Plane2Io<DT, P, GATED> io(g, plane2_sm);
  const Plane2Roots<P> tw(lds + P::F0 * P::RS, roots);
  const int share = int(blockIdx.x / unsigned(g.H)), h = int(blockIdx.x) - share * g.H;
  const int b0 = share * g.per_wg, b1 = min(g.B, b0 + g.per_wg);
  const int64_t hk = g.kfilm ? int64_t(b0) * g.H + h : h;
  Plane2Vec<DT> xv[4], kg[4];
  io.load(x, b0, h, xv);
  if constexpr (GATED) io.load(ga.kg, b0, h, kg);
  float2 kv[8];
  {
    const Plane2Filter kr(k + hk * g.K0 * g.K2, g.K0, g.K2);
    plane2_spectrum<P>(lds, [&](int m, int n) { return kr.r.elem(kr.at(m, n)); }, g.K0, g.K2 > P::M, kv, tw);
  }
  const float scale = 1.f / float(P::F0 * P::M);
#pragma unroll
  for (int r = 0; r < 8; ++r) kv[r] = cscale(kv[r], scale);  // a power of two: exact
  const float sv = s ? Elem<DT>::round(Elem<DT>::load(s, h)) : 0.f;
  for (int b = b0; b < b1; ++b) {
    if constexpr (GATED) io.gate(ga.act1, xv, kg);
    io.to_raw(xv);
    __syncthreads();
    if (b + 1 < b1) {
      io.load(x, b + 1, h, xv);
      if constexpr (GATED) io.load(ga.kg, b + 1, h, kg);
    }
    float2 v[8];
    plane2_spectrum<P>(lds, [&](int m, int n) { return io.sample(m, n); }, g.S0, g.S2 > P::M, v, tw);
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = cmul(v[r], kv[r]);
    plane2_inverse<P>(
        lds, v, [&](int m) { return ((m - g.sh0) & (P::F0 - 1)) < g.S0; },
        [&](int m, int n, float lo, float hi) {
          const int row = (m - g.sh0) & (P::F0 - 1);
          io.keep(row, n - g.o2, lo);
          io.keep(row, n + P::M - g.o2, hi);
        },
        tw);
    const RowBuf<DT, false> yr = io.image(y, b, h);
    io.each([&](int, int e) {
      float c[4], r[4];
      io.get(e, c, r);
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = epilogue<DT>(c[i], s != nullptr, sv, r[i]);
      Plane2Vec<DT> o;
      if constexpr (GATED) {
#pragma clang fp contract(off)
        o.set(c);
        if (ga.y1out) o.store(io.image(ga.y1out, b, h), e, g.vec);
        Plane2Vec<DT> vv;
        vv.load(io.image(ga.v, b, h), e, g.vec);
        float f[4];
        vv.get(f);
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = c[i] * Elem<DT>::round(gate_act(ga.act2, f[i]));
      }
      o.set(c);
      o.store(yr, e, g.vec);
    });
    __syncthreads();
  }
}

// gk: the filter gradient, or with part != 0 the workgroup's share of it at part[blockIdx.x K0 K2] (blockIdx.x =
// share H + h), summed by plane2_reduce_kernel.  GATED: x is q, gy the gradient of the gated output, gx receives dq.
template <int DT, class P, bool GATED>
__global__ __launch_bounds__(P::T) void plane2_bwd_kernel(const typename Elem<DT>::T* __restrict__ gy,
                                                          const typename Elem<DT>::T* __restrict__ x,
                                                          const float* __restrict__ k,
                                                          const typename Elem<DT>::T* __restrict__ s,
                                                          typename Elem<DT>::T* __restrict__ gx,
                                                          float* __restrict__ gk, float* __restrict__ gs,
                                                          float* __restrict__ part, Plane2Geom g, GatedIO ga,
                                                          const float2* __restrict__ roots) {
  extern __shared__ __align__(16) unsigned char plane2_sm[];
  float2* lds = reinterpret_cast<float2*>(plane2_sm);
  const Plane2Io<DT, P, GATED> io(g, plane2_sm);
  const Plane2Roots<P> tw(lds + P::F0 * P::RS, roots);
  const int share = int(blockIdx.x / unsigned(g.H)), h = int(blockIdx.x) - share * g.H;
  const int b0 = share * g.per_wg, b1 = min(g.B, b0 + g.per_wg);
  const int64_t hk = g.kfilm ? int64_t(b0) * g.H + h : h;
  Plane2Vec<DT> xv[4], gv[4], kg[4], vv[4];
  const auto load = [&](int b) {
    io.load(x, b, h, xv);
    io.load(gy, b, h, gv);
    if constexpr (GATED) {
      io.load(ga.kg, b, h, kg);
      io.load(ga.v, b, h, vv);
    }
  };
  load(b0);
  float2 kv[8], q[8];
  {
    const Plane2Filter kr(k + hk * g.K0 * g.K2, g.K0, g.K2);
    plane2_spectrum<P>(lds, [&](int m, int n) { return kr.r.elem(kr.at(m, n)); }, g.K0, g.K2 > P::M, kv, tw);
  }
  const float scale = 1.f / float(P::F0 * P::M);
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    kv[r] = cscale(kv[r], scale);
    q[r] = make_float2(0.f, 0.f);
  }
  const float sv = s ? Elem<DT>::round(Elem<DT>::load(s, h)) : 0.f;
  const auto sample = [&](int m, int n) { return io.sample(m, n); };
  for (int b = b0; b < b1; ++b) {
    float2 xs[8], v[8];
    if constexpr (GATED) {
      io.gate(ga.act1, xv, kg);
      io.gate(ga.act2, gv, vv);
    }
    io.to_raw(xv);
    __syncthreads();
    plane2_spectrum<P>(lds, sample, g.S0, g.S2 > P::M, xs, tw);
    io.to_raw(gv);  // every wave is past the first row pass
    __syncthreads();
    if (b + 1 < b1) load(b + 1);
    plane2_spectrum<P>(lds, sample, g.S0, g.S2 > P::M, v, tw);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      q[r] = cadd(q[r], cmulc(v[r], xs[r]));
      v[r] = cmulc(v[r], kv[r]);
    }
    const auto keep = [&](int row, int p, float c) {
      const int i = plane2_lag<P>(p, g.o2, c);
      io.keep(row, i, c);
    };
    plane2_inverse<P>(
        lds, v, [&](int m) { return ((m + g.sh0) & (P::F0 - 1)) < g.S0; },
        [&](int m, int n, float lo, float hi) {
          const int row = (m + g.sh0) & (P::F0 - 1);
          keep(row, n, lo);
          keep(row, n + P::M, hi);
        },
        tw);
    const RowBuf<DT, false> outr = io.image(gx, b, h);
    io.each([&](int, int e) {
      float c[4], r[4];
      io.get(e, c, r);
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = epilogue<DT>(c[i], s != nullptr, sv, r[i]);  // gated: dz
      Plane2Vec<DT> o;
      if constexpr (GATED) {
#pragma clang fp contract(off)
        Plane2Vec<DT> a;
        float qq[4], kk[4], f[4];
        a.load(io.image(x, b, h), e, g.vec);
        a.get(qq);
        a.load(io.image(ga.kg, b, h), e, g.vec);
        a.get(kk);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f[i] = Elem<DT>::round(c[i] * qq[i]) * gate_dact(ga.act1, kk[i]);
          c[i] = c[i] * Elem<DT>::round(gate_act(ga.act1, kk[i]));
        }
        o.set(f);
        o.store(io.image(ga.dkg, b, h), e, g.vec);
        a.load(io.image(gy, b, h), e, g.vec);
        a.get(qq);
        a.load(io.image(ga.y1, b, h), e, g.vec);
        a.get(f);
        a.load(io.image(ga.v, b, h), e, g.vec);
        a.get(kk);
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = Elem<DT>::round(qq[i] * f[i]) * gate_dact(ga.act2, kk[i]);
        o.set(f);
        o.store(io.image(ga.dv, b, h), e, g.vec);
      }
      o.set(c);
      o.store(outr, e, g.vec);
    });
    __syncthreads();
  }
  const int64_t size = int64_t(g.K0) * g.K2;
  const Plane2Filter kr(part ? part + int64_t(blockIdx.x) * size : gk + hk * size, g.K0, g.K2);
  const auto put = [&](int row, int p, float c) {
    c *= scale;
    const int n2 = plane2_lag<P>(p, g.o2, c);
    kr.r.store_elem(kr.at(row, n2), c);
    if (!part && gs && row == g.sh0 && n2 == g.o2) gs[hk] = c;  // lag 0
  };
  plane2_inverse<P>(
      lds, q, [&](int m) { return ((m + g.sh0) & (P::F0 - 1)) < g.K0; },
      [&](int m, int n, float lo, float hi) {
        const int row = (m + g.sh0) & (P::F0 - 1);
        put(row, n, lo);
        put(row, n + P::M, hi);
      },
      tw);
}

// Calls (fftconv2d_plane_impl.h), one instance per dtype.
}  // namespace nsq
