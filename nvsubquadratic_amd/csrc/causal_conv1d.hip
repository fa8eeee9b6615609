// Depthwise causal direct convolution (k = 1..256), forward and backward.
//
// Replaces the native kernel the reference binds at
// nvsubquadratic/ops/causal_conv1d_custom.py:81-98 (subquadratic_ops_torch
// .causal_conv1d(x, w, bias, activation)), used by the Hyena short-conv slot
// through nvsubquadratic/modules/subq_ops_causal_conv1d.py:77-83.
#include <mutex>

#include "toeplitz_mma.h"

namespace nsq {

// Scratch of nsq_causal_conv1d_bwd_noalloc: one copy per GPU, resident from
// module load to process exit.  In host code `scratch` names a host-side
// stand-in, not device memory: the device address of each GPU's copy comes
// from hipGetSymbolAddress (noalloc_scratch below) and only that address is
// ever handed to kernels.
constexpr size_t kNoAllocScratchBytes = NSQ_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

// Forward for up to 16 taps (short_fwd) from registers: thread t of a tile owns outputs
// n = n0 + 8t + e, e < 8; with the taps left-padded to KP = 4, 8 or 16,
// y[n] = act(bias + sum_j wk[j] x[n - KP + 1 + j]).  Its x window
// [n0 + 8t - 8 XB, n0 + 8t + 8) comes straight from HBM in aligned chunks of 8
// (Win8; the chunks before the thread's own are its neighbours', read again
// from L2), so no LDS staging or barrier.  grid = (B*C, ceil(L / kConvTile)).
template <int DT, bool AL, int ACT, int KP>
__global__ __launch_bounds__(kConvThreads) void cconv_fwd_short_kernel(const typename Elem<DT>::T* __restrict__ x,
                                                                        const float* __restrict__ w,
                                                                        const float* __restrict__ bias,
                                                                        typename Elem<DT>::T* __restrict__ y, int C,
                                                                        int L, int K) {
  static_assert(KP == 4 || KP == 8 || KP == 16, "cconv_fwd_short: taps padded to 4, 8 or 16");
  static_assert(kConvPer == 8, "cconv_fwd_short: 8 outputs per thread");
  constexpr int XB = (KP - 1 + 7) / 8;  // chunks before the outputs: positions >= 1 - KP
  const int64_t row = blockIdx.x;
  const int c = int(row % C);
  const int base = int(blockIdx.y) * kConvTile + kConvPer * int(threadIdx.x);
  float wk[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    const int sl = j - (KP - K);
    wk[j] = sl >= 0 ? w[int64_t(c) * K + (sl >= 0 ? sl : 0)] : 0.f;
  }
  const float b0 = bias ? bias[c] : 0.f;
  const RowBuf<DT, false> xb(x + row * L, L);
  Win8<DT, AL> xc[XB + 1];
#pragma unroll
  for (int i = 0; i <= XB; ++i) xc[i].load(xb, base + 8 * (i - XB));
  auto xat = [&](int p) { return xc[(p + 8 * XB) >> 3].at((p + 8 * XB) & 7); };
  float out[kConvPer];
#pragma unroll
  for (int e = 0; e < kConvPer; ++e) {
    float a = b0;
#pragma unroll
    for (int j = 0; j < KP; ++j) a = fmaf(wk[j], xat(e - KP + 1 + j), a);
    out[e] = act_fwd<ACT>(a);
  }
  store8<DT, AL>(RowBuf<DT, AL>(y + row * L, L), base, out);
}

// Whole rows of 16-byte chunks: every row starts 16-byte aligned and ends on a chunk.
template <int DT>
static bool rows16(int64_t L, const void* a, const void* b, const void* c) {
  return L % (DT == NSQ_DTYPE_F32 ? 4 : 8) == 0 &&
         ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c)) & 15) == 0;
}

constexpr int kConvSegTiles = 4;  // tiles per workgroup of the register backward
// The register kernels run up to 4 taps, the matrix-core ones above 16; between, by what measured faster (us, register /
// matrix-core).  Large calls, B=4 C=4096 L=8192 (2^27 samples):
//   forward, bf16:  identity K = 8 93 / 101, K = 9 112 / 101;  silu K = 4 117 / 105, K = 5 135 / 105;
//   forward, fp32:  K = 4 198 / 201, K = 5 218 / 201, K = 16 226 / 201 (either activation);
//   backward, bf16: silu K = 4 196 / 218, K = 5 274 / 218;  fp32: silu K = 4 339 / 317, K = 5 417 / 317.
// With fewer samples the matrix-core kernels' setup (bands, staging, the tile beside a run's) shows.  Aligned rows,
// forward: fp32 up to 16 taps and 16 bits up to 8 to 2^25 (there fp32 39.5 / 42.0, fp16 33.3 / 35.3, but bf16 35.4 /
//   31.5; B=4 C=1024 L=2048, silu: fp32 K = 16 13.2 / 14.3, bf16 K = 7 9.4 / 11.1); 16 bits up to 16 taps while
//   launches dominate, to 2^19 samples in bf16 (2.4 / 2.6, at 2^20 3.1 / 2.9) and 2^23 in fp16, whose samples are two
//   parts (2^22 5.7 / 5.9).
// Aligned rows, forward + backward, up to 8 taps: fp32 below 2^25 (K = 7 25.6 / 27.2 backward), bf16 to 2^23 (B=2 C=512
//   L=8192 silu K = 5 36.8 / 41.8; at 2^24 62 / 62), fp16 to 2^24 (63 / 71).
// Unaligned rows: the matrix-core kernels read and write them as vectors (toeplitz_mma.h), so they take all calls from 5
// taps but the 16-bit identity forward up to 8 (B=8 C=768 L=777 fp32, K = 7 25.8 / 18.0).
constexpr int kConvShortMax = 4;
constexpr int64_t kConvSmall = int64_t(1) << 25;
template <int DT>
static bool short_fwd(int K, int act, int64_t samples, bool aligned) {
  if (K <= kConvShortMax || (K <= 8 && act == NSQ_ACT_IDENTITY && DT != NSQ_DTYPE_F32)) return true;
  if (!aligned || K > 16) return false;
  const int64_t few = DT == NSQ_DTYPE_F32 ? kConvSmall : int64_t(1) << (DT == NSQ_DTYPE_BF16 ? 19 : 23);
  return samples <= few || (K <= 8 && samples <= kConvSmall - (DT == NSQ_DTYPE_BF16));
}
template <int DT>
static bool short_bwd(int K, int64_t samples, bool aligned) {
  if (K <= kConvShortMax) return true;
  const int64_t few = DT == NSQ_DTYPE_F32 ? kConvSmall - 1 : int64_t(1) << (DT == NSQ_DTYPE_BF16 ? 23 : 24);
  return K <= 8 && aligned && samples <= few;
}

__global__ void cconv_wgrad_reduce_kernel(const float* __restrict__ part, int nparts, int K, float* __restrict__ gw,
                                          float* __restrict__ gb) {
  const int c = blockIdx.x, j = threadIdx.x;
  if (j > K) return;
  const float* pc = part + int64_t(c) * nparts * (K + 1) + j;
  float sacc = 0.f;
  for (int p = 0; p < nparts; ++p) sacc += pc[int64_t(p) * (K + 1)];
  if (j < K)
    gw[int64_t(c) * K + j] = sacc;
  else if (gb)
    gb[c] = sacc;
}

static int64_t cconv_wgrad_parts(int64_t B, int64_t L) {
  return ceil_div(B * ceil_div(L, kConvTile), kConvSegTiles);
}

// ---------------------------------------------------------------------------
// Matrix-core path (more than kConvShortMax taps): banded Toeplitz products
// at fp32 precision on the bf16 matrix cores (toeplitz_mma.h).  A workgroup
// owns one channel and walks a run of its (batch row, 2048-output tile)
// sequence, so the split taps are prepared once per run.
// ---------------------------------------------------------------------------
// Workgroups wanted: 4 or more per resident slot (256 CUs x 2..4) so that they end together, but one where tiles are
// few: a run pays for its bands, and with silu for the gpre of the tile beside it, which is half of a run of one.
// Measured, 1024 / 4096 (us, forward + backward): B=2 C=128 L=16384 K=33 bf16 (2048 tiles) silu 27.0 / 32.5, identity
// 16.7 / 19.7; 8192 tiles 6% better on average, 32768 1.5% worse and up to 9%.
inline int64_t mma_target(int64_t tiles) { return tiles <= 8192 ? 1024 : 4096; }

// A band multiplies every sample of a block's window, later ones too, by some zero tap, and inf leaves NaN among its
// parts (inf - inf; a finite value above the largest bf16 is inf in its first part): a non-finite value makes all the
// sums over its window NaN.  So where all results are finite they are right, and where some are not the kernels take
// the run's results once more at its end, tap by tap from memory.  (Not in place: that path's registers on top of the
// bands' cost one to three waves per SIMD.  Checks of the operands, with flags in LDS, cost 5 to 10% of the time.)
template <int N>
__device__ __forceinline__ bool nonfinite(const float (&v)[N]) {
  float s[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < N; ++i) s[i & 1] = fmaf(v[i], 0.f, s[i & 1]);
  return !(s[0] + s[1] == 0.f);
}

// Tiles per run: as many as leave mma_target workgroups, at least 1.
static int64_t mma_run_tiles(int64_t B, int64_t C, int64_t L) {
  const int64_t tiles = B * ceil_div(L, kConvTile), want = ceil_div(mma_target(C * tiles), C);
  return tiles / want > 1 ? tiles / want : 1;
}
static int64_t mma_runs(int64_t B, int64_t C, int64_t L) {
  return ceil_div(B * ceil_div(L, kConvTile), mma_run_tiles(B, C, L));
}

// The products of S steps for the 16-block M-tiles at blocks a0 and a1: src holds P part arrays of `stride` elements.
template <int S, int P>
__device__ __forceinline__ void band_run2(const nsq_bf16x8_t (&tap)[S][kTapParts], const uint16_t* src, int stride,
                                          int a0, int a1, nsq_f32x4_t& c0, nsq_f32x4_t& c1) {
  const int l = int(threadIdx.x) & 63, kk = l >> 4, a = l & 15;
  const uint16_t* p0 = src + 16 * (a0 + a) + 8 * kk;
  const uint16_t* p1 = src + 16 * (a1 + a) + 8 * kk;
  c0 = nsq_f32x4_t{0.f, 0.f, 0.f, 0.f};
  c1 = nsq_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S; ++s) {
    nsq_bf16x8_t u[P], v[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int o = p * stride + 32 * s;
      if (band_half_last<S>() && s == S - 1) {  // the window ends 16 columns before the step does
        const bool z = kk >= 2;
        const uint4 zero = make_uint4(0, 0, 0, 0);
        u[p] = as_bf16x8(z ? zero : *reinterpret_cast<const uint4*>(p0 + (z ? 0 : o)));
        v[p] = as_bf16x8(z ? zero : *reinterpret_cast<const uint4*>(p1 + (z ? 0 : o)));
      } else {
        u[p] = as_bf16x8(*reinterpret_cast<const uint4*>(p0 + o));
        v[p] = as_bf16x8(*reinterpret_cast<const uint4*>(p1 + o));
      }
    }
    mma_parts<P>(tap[s], u, c0);
    mma_parts<P>(tap[s], v, c1);
  }
}

// y = act(conv + bias).  Bound by HBM (x in, y out) from K = 128 down: 15 MFMAs of 16 cycles per 256 outputs are
// 60 us at B=4 C=4096 L=8192 bf16, where x and y take 100 us at 5.3 TB/s.  Measured there: 101 us at K = 17, 120 at
// K = 128 (152 with silu), 183 at K = 256; the fp32 matrix products before took 409 us at K = 128 with silu.  The window of a tile (KP + 2048 samples as bf16
// parts) is double-buffered in LDS, one barrier per tile, the next tile's samples in flight during the products.
template <int DT, int S, int ACT, bool AL>
__global__ __launch_bounds__(kConvThreads) __attribute__((amdgpu_waves_per_eu(S <= 5 ? 4 : 2))) void
cconv_fwd_mma_kernel(const typename Elem<DT>::T* __restrict__ x, const float* __restrict__ w,
                     const float* __restrict__ bias, typename Elem<DT>::T* __restrict__ y, int B, int C, int L, int K,
                     int run) {
  constexpr int KP = band_kp<S>(), W = KP + kConvTile, P = kParts<DT>;
  // two windows; first the band's operands, made once for the four waves
  constexpr int BAND = band_operands<S>() * 16, WIN = P * W * 2;
  __shared__ __align__(16) unsigned char sm[BAND > 2 * WIN ? BAND : 2 * WIN];
  __shared__ __align__(16) float wl[kConvWeightFloats];
  uint4* band = reinterpret_cast<uint4*>(sm);
  const int c = int(blockIdx.x);
  const int ntiles = (L + kConvTile - 1) / kConvTile;
  const int g0 = int(blockIdx.y) * run, g1 = min(B * ntiles, g0 + run);
  const int t = int(threadIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63;
  stage_weights<false>(wl, w + int64_t(c) * K, K);
  PartChunk<DT, AL> cm, cx;  // samples [8t, 8t + 8) of the window and, for the first threads, [2048 + 8t, ...)
  auto load = [&](int g) {
    const int b = g / ntiles, n0 = (g - b * ntiles) * kConvTile;
    const typename Elem<DT>::T* row = x + (int64_t(b) * C + c) * L;
    cm.load(row, n0 - KP + 8 * t, L);
    if (t < KP / 8) cx.load(row, n0 - KP + kConvTile + 8 * t, L);
  };
  load(g0);
  __syncthreads();  // taps staged
  put_band<S, false>(band, wl, K);
  __syncthreads();
  nsq_bf16x8_t tap[S][kTapParts];
  get_band<S>(band, tap);
  __syncthreads();
  const float b0 = bias ? bias[c] : 0.f;
  const int p0 = 16 * (32 * wave + (l & 15)) + 4 * (l >> 4);  // the lane's positions in M-tile 2 wave; 256 on in the next
  int bad = g1;  // the wave's first tile with a non-finite result
  for (int g = g0; g < g1; ++g) {
    const int b = g / ntiles, n0 = (g - b * ntiles) * kConvTile;
    uint16_t* xb = reinterpret_cast<uint16_t*>(sm + ((g - g0) & 1) * WIN);
    uint4 o[P];
    cm.parts(o);
#pragma unroll
    for (int p = 0; p < P; ++p) *reinterpret_cast<uint4*>(xb + p * W + 8 * t) = o[p];
    if (t < KP / 8) {
      cx.parts(o);
#pragma unroll
      for (int p = 0; p < P; ++p) *reinterpret_cast<uint4*>(xb + p * W + kConvTile + 8 * t) = o[p];
    }
    __syncthreads();  // a wave writes this window again two barriers on, when all have read it
    if (g + 1 < g1) load(g + 1);
    if (n0 + 512 * wave >= L) continue;
    nsq_f32x4_t acc[2];
    band_run2<S, P>(tap, xb, W, 32 * wave, 32 * wave + 16, acc[0], acc[1]);
    float v[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[h][r] = acc[h][r] + b0;
    if (__ballot(nonfinite(reinterpret_cast<const float(&)[8]>(v))) != 0) bad = min(bad, g);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[h][r] = act_fwd<ACT>(v[h][r]);
      store4<DT, AL>(y + (int64_t(b) * C + c) * L, n0 + p0 + 256 * h, L, v[h]);
    }
  }
#pragma unroll 1
  for (int g = bad; g < g1; ++g) {  // each lane its own outputs
    const int b = g / ntiles, n0 = (g - b * ntiles) * kConvTile;
    const RowBuf<DT, false> rb(x + (int64_t(b) * C + c) * L, L), ob(y + (int64_t(b) * C + c) * L, L);
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
      const int n = n0 + p0 + 256 * (i >> 2) + (i & 3);
      if (n < L) ob.store_elem(n, act_fwd<ACT>(direct_taps<DT>(rb, w + int64_t(c) * K, K, n) + b0));
    }
  }
}

// Whole backward of one channel's run of tiles in one pass (the earlier three kernels wrote gpre as fp32 and read it
// twice, 20 bytes a sample against 6 here):
//   gpre = gy silu'(conv(x) + bias) (identity: gy), by the conv band over the tile's 2048 outputs;
//   gx[n] = sum_j w[j] gpre[n + K - 1 - j], by the reversed band;
//   D[i][t] += sum_a gpre[16a + i] x[n0 - KP + 16a + t], gw[j] = sum_i D[i][i + j + pad].
// The tiles of a row run from its end to its start, so the KP positions of gpre past a tile are the first ones of
// the tile before; a run that starts inside a row computes that tile's gpre once more.
// LDS: both bands as operands (reloaded into registers per phase: together they would not fit beside D), the window
// of x and gpre as bf16 parts, in order.  The weight gradient contracts over the blocks a, so its operands are the
// columns of these arrays' 16-wide rows: the transposing LDS read (tr16_column8) forms them, with no second copy.
// The weight gradient is fp32 as the bands are (the same pairs of parts, fp32 sums).
// Bound by issue: at K = 128 with silu 117 MFMAs and about 400 VALU instructions per wave and tile (gpre, its split)
// fill 70% of the cycles at 3 waves per SIMD.  B=4 C=4096 L=8192 bf16: 478 us with silu, 201 identity (155 at K = 17:
// 5.2 TB/s), against 1220 us for the three kernels.
template <int DT, int S, int ACT>
struct CconvBwdCfg {
  static constexpr bool SILU = ACT == NSQ_ACT_SILU;
  static constexpr int KP = band_kp<S>(), W = KP + kConvTile, TG = KP / 16 + 1;
  static constexpr int PX = kParts<DT>, PG = SILU ? 3 : PX;
  static constexpr int TAPS = band_operands<S>();
  static constexpr int O_REV = 0, O_CONV = O_REV + TAPS * 16, O_XL = O_CONV + (SILU ? TAPS * 16 : 0),
                       O_GL = O_XL + PX * W * 2, BYTES = O_GL + PG * W * 2;
  static_assert(16 * 16 * TG * 4 <= TAPS * 16, "cconv_bwd_mma: the final reduction reuses a band");
};

template <int DT, int S, int ACT, bool AL>
__global__ __launch_bounds__(kConvThreads)
__attribute__((amdgpu_waves_per_eu(CconvBwdCfg<DT, S, ACT>::BYTES > 80 * 1024 ? 1 : CconvBwdCfg<DT, S, ACT>::BYTES > 53 * 1024 ? 2 : 3))) void cconv_bwd_mma_kernel(
    const typename Elem<DT>::T* __restrict__ gy, const typename Elem<DT>::T* __restrict__ x,
    const float* __restrict__ w, const float* __restrict__ bias, typename Elem<DT>::T* __restrict__ gx,
    float* __restrict__ part, int B, int C, int L, int K, int run) {
  using F = CconvBwdCfg<DT, S, ACT>;
  constexpr int KP = F::KP, W = F::W, PX = F::PX, PG = F::PG;
  constexpr bool SILU = F::SILU;
  __shared__ __align__(16) unsigned char sm[F::BYTES];
  static_assert((kConvTile + kConvMaxK) * 4 <= F::BYTES, "cconv_bwd_mma: a tile's gpre as fp32 in LDS");
  uint4* rev = reinterpret_cast<uint4*>(sm + F::O_REV);
  uint4* conv = reinterpret_cast<uint4*>(sm + F::O_CONV);
  uint16_t* xl = reinterpret_cast<uint16_t*>(sm + F::O_XL);
  uint16_t* gl = reinterpret_cast<uint16_t*>(sm + F::O_GL);
  float* wl = reinterpret_cast<float*>(sm + F::O_GL);  // the taps until the bands are made; at the end wave sums
  const int c = int(blockIdx.x);
  const int ntiles = (L + kConvTile - 1) / kConvTile;
  const int g0 = int(blockIdx.y) * run, g1 = min(B * ntiles, g0 + run);
  const int t = int(threadIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63;
  const int kk = l >> 4, li = l & 15;
  const int pad = KP - K + 1, tg0 = pad >> 4;
  const float b0 = bias ? bias[c] : 0.f;

  stage_weights<false>(wl, w + int64_t(c) * K, K);
  PartChunk<DT, AL> xm, xx, gm, gx8;
  auto row_of = [&](int g) { return (int64_t(g / ntiles) * C + c) * L; };
  auto load = [&](int g) {
    const int n0 = (g % ntiles) * kConvTile;
    xm.load(x + row_of(g), n0 - KP + 8 * t, L);
    if (t < KP / 8) xx.load(x + row_of(g), n0 - KP + kConvTile + 8 * t, L);
    if constexpr (!SILU) {
      gm.load(gy + row_of(g), n0 + 8 * t, L);
      if (t < KP / 8) gx8.load(gy + row_of(g), n0 + kConvTile + 8 * t, L);
    }
  };
  load(g1 - 1);
  __syncthreads();  // taps staged
  put_band<S, true>(rev, wl, K);
  if constexpr (SILU) put_band<S, false>(conv, wl, K);
  __syncthreads();
  auto stage_x = [&]() {
    uint4 o[PX];
    xm.parts(o);
#pragma unroll
    for (int p = 0; p < PX; ++p) *reinterpret_cast<uint4*>(xl + p * W + 8 * t) = o[p];
    if (t < KP / 8) {
      xx.parts(o);
#pragma unroll
      for (int p = 0; p < PX; ++p) *reinterpret_cast<uint4*>(xl + p * W + kConvTile + 8 * t) = o[p];
    }
  };
  float bacc = 0.f;
  // gpre of tile g into gl (SILU)
  auto make_gpre = [&](int g, bool count) {
    const int n0 = (g % ntiles) * kConvTile;
    Quad<DT, AL> q[2];
    const int p0 = 16 * (32 * wave + li) + 4 * kk;  // the lane's positions in M-tile 2 wave; 256 on in the next
    q[0].load(gy + row_of(g), n0 + p0, L);
    q[1].load(gy + row_of(g), n0 + p0 + 256, L);
    uint32_t b[2][2][PG];  // pairs of positions
    if (n0 + 512 * wave < L) {
      nsq_bf16x8_t tap[S][kTapParts];
      get_band<S>(conv, tap);
      nsq_f32x4_t acc[2];
      band_run2<S, PX>(tap, xl, W, 32 * wave, 32 * wave + 16, acc[0], acc[1]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float gp[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          gp[r] = n0 + p0 + 256 * h + r < L ? q[h].at(r) * dsilu(acc[h][r] + b0) : 0.f;
          if (count) bacc += gp[r];
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) split_parts2<PG>(gp[2 * r], gp[2 * r + 1], b[h][r]);
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int p = 0; p < PG; ++p) b[h][r][p] = 0;
    }
#pragma unroll
    for (int p = 0; p < PG; ++p)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<uint2*>(gl + p * W + p0 + 256 * h) = make_uint2(b[h][0][p], b[h][1][p]);
  };
  // gy itself into gl (identity)
  auto stage_g = [&]() {
    uint4 o[PX];
    gm.parts(o);
#pragma unroll
    for (int p = 0; p < PX; ++p) *reinterpret_cast<uint4*>(gl + p * W + 8 * t) = o[p];
#pragma unroll
    for (int k = 0; k < 8; ++k) bacc += gm.w.at(k);
    if (t < KP / 8) {
      gx8.parts(o);
#pragma unroll
      for (int p = 0; p < PX; ++p) *reinterpret_cast<uint4*>(gl + p * W + kConvTile + 8 * t) = o[p];
    }
  };
  // the KP positions past the tile: the first KP of the tile after it (or zeros past the row)
  auto carry = [&](bool zero) {
    if (t < KP / 8)
#pragma unroll
      for (int p = 0; p < PG; ++p)
        *reinterpret_cast<uint4*>(gl + p * W + kConvTile + 8 * t) =
            zero ? make_uint4(0, 0, 0, 0) : *reinterpret_cast<const uint4*>(gl + p * W + 8 * t);
  };

  nsq_f32x4_t D[F::TG];
#pragma unroll
  for (int tg = 0; tg < F::TG; ++tg) D[tg] = nsq_f32x4_t{0.f, 0.f, 0.f, 0.f};
  if constexpr (SILU) {
    if (g1 % ntiles != 0) {  // the run starts inside a row: gpre of the tile after it
      load(g1);
      stage_x();
      __syncthreads();
      make_gpre(g1, false);
      load(g1 - 1);
      __syncthreads();
    }
  }
  bool bad = false;
  for (int g = g1 - 1; g >= g0; --g) {
    const int n0 = (g % ntiles) * kConvTile;
    if constexpr (SILU) carry(g % ntiles == ntiles - 1);
    stage_x();
    if constexpr (!SILU) stage_g();
    __syncthreads();
    if (g > g0) load(g - 1);
    if constexpr (SILU) {
      make_gpre(g, true);
      __syncthreads();
    }
    if (n0 + 512 * wave < L) {
      nsq_bf16x8_t tap[S][kTapParts];
      get_band<S>(rev, tap);
      nsq_f32x4_t acc[2];
      band_run2<S, PG>(tap, gl, W, 32 * wave, 32 * wave + 16, acc[0], acc[1]);
      float v[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[h][r] = acc[h][r];
      bad = bad || nonfinite(reinterpret_cast<const float(&)[8]>(v));
#pragma unroll
      for (int h = 0; h < 2; ++h) store4<DT, AL>(gx + row_of(g), n0 + 16 * (32 * wave + 16 * h + li) + 4 * kk, L, v[h]);
    }
    {
      // wave w contracts over blocks 32 w .. 32 w + 31
      nsq_bf16x8_t ga[PG];
#pragma unroll
      for (int p = 0; p < PG; ++p) ga[p] = tr16_column8(gl + p * W + 512 * wave);
#pragma unroll
      for (int tg = 0; tg < F::TG; ++tg) {
        if (tg < tg0) continue;
        nsq_bf16x8_t xb[PX];
#pragma unroll
        for (int p = 0; p < PX; ++p) xb[p] = tr16_column8(xl + p * W + 512 * wave + 16 * tg);
#pragma unroll
        for (int d = 2; d >= 0; --d)
#pragma unroll
          for (int p = 0; p < PX; ++p)
            if (d - p >= 0 && d - p < PG)
              D[tg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga[d - p], xb[p], D[tg], 0, 0, 0);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int tg = 0; tg < F::TG; ++tg) {
    const float v[4] = {D[tg][0], D[tg][1], D[tg][2], D[tg][3]};
    bad = bad || nonfinite(v);
  }
  float wsum = 0.f;  // tap t's sum where it is taken directly
  if (__syncthreads_or(bad || !(fabsf(bacc) < INFINITY))) {
#pragma unroll
    for (int tg = 0; tg < F::TG; ++tg) D[tg] = nsq_f32x4_t{0.f, 0.f, 0.f, 0.f};
    bacc = 0.f;
    float* gp = reinterpret_cast<float*>(sm);  // gpre over [n0, n0 + kConvTile + K - 1)
    const float* wc = w + int64_t(c) * K;
#pragma unroll 1
    for (int g = g0; g < g1; ++g) {
      const int n0 = (g % ntiles) * kConvTile, count = min(kConvTile, L - n0);
      const RowBuf<DT, false> xb(x + row_of(g), L), gb(gy + row_of(g), L), ob(gx + row_of(g), L);
#pragma unroll 1
      for (int m = t; m < kConvTile + K - 1; m += kConvThreads) {
        float v = 0.f;
        if (n0 + m < L) v = SILU ? gb.elem(n0 + m) * dsilu(direct_taps<DT>(xb, wc, K, n0 + m) + b0) : gb.elem(n0 + m);
        gp[m] = v;
        if (m < kConvTile) bacc += v;
      }
      __syncthreads();
#pragma unroll 1
      for (int m = t; m < count; m += kConvThreads) {
        float a = 0.f;
#pragma unroll 1
        for (int j = 0; j < K; ++j) a = fmaf(wc[j], gp[m + K - 1 - j], a);
        ob.store_elem(n0 + m, a);
      }
      if (t < K)
#pragma unroll 1
        for (int m = 0; m < count; ++m) wsum = fmaf(gp[m], xb.elem_halo(n0 + m - K + 1 + t), wsum);
      __syncthreads();
    }
  }
  // fixed-order sums over the waves, then along the diagonals
  constexpr int RW = 16 * F::TG;
  float* red = reinterpret_cast<float*>(sm + F::O_REV);
  for (int v = 0; v < kConvWaves; ++v) {
    if (wave == v) {
#pragma unroll
      for (int tg = 0; tg < F::TG; ++tg)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float& dst = red[(4 * kk + r) * RW + 16 * tg + li];
          dst = (v == 0 ? 0.f : dst) + D[tg][r];
        }
    }
    __syncthreads();
  }
  float* pw = part + (int64_t(c) * gridDim.y + blockIdx.y) * (K + 1);
  if (t < K) {
    float s = 0.f;
    for (int i = 0; i < 16; ++i) s += red[i * RW + i + pad + t];
    pw[t] = s + wsum;
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) bacc += __shfl_xor(bacc, o);
  if (l == 0) wl[wave] = bacc;
  __syncthreads();
  if (t == 0) pw[K] = (wl[0] + wl[1]) + (wl[2] + wl[3]);
}

template <class F>
static void with_band(int64_t K, F&& f) {
  switch (band_steps_for(K)) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 5: return f(std::integral_constant<int, 5>{});
    case 7: return f(std::integral_constant<int, 7>{});
    default: return f(std::integral_constant<int, 9>{});
  }
}

template <int DT>
static void launch_fwd_mma(const void* x, const float* w, const float* bias, void* y, int act, int B, int C, int L,
                           int K, hipStream_t st) {
  using ET = typename Elem<DT>::T;
  const dim3 grid(C, unsigned(mma_runs(B, C, L)));
  const int run = int(mma_run_tiles(B, C, L));
  const bool al = rows16<DT>(L, x, y, nullptr);
  with_band(K, [&](auto s) {
    auto go = [&](auto a, auto f) {
      hipLaunchKernelGGL((cconv_fwd_mma_kernel<DT, decltype(s)::value, decltype(f)::value, decltype(a)::value>), grid,
                         dim3(kConvThreads), 0, st, (const ET*)x, w, bias, (ET*)y, B, C, L, K, run);
    };
    using SILU = std::integral_constant<int, NSQ_ACT_SILU>;
    using IDN = std::integral_constant<int, NSQ_ACT_IDENTITY>;
    if (al)
      act == NSQ_ACT_SILU ? go(std::true_type{}, SILU{}) : go(std::true_type{}, IDN{});
    else
      act == NSQ_ACT_SILU ? go(std::false_type{}, SILU{}) : go(std::false_type{}, IDN{});
  });
}

template <int DT>
static void launch_bwd_mma(const void* gy, const void* x, const float* w, const float* bias, void* gx, float* gw,
                           float* gb, int act, int B, int C, int L, int K, float* ws, hipStream_t st) {
  using ET = typename Elem<DT>::T;
  const int nparts = int(mma_runs(B, C, L)), run = int(mma_run_tiles(B, C, L));
  const dim3 grid(C, unsigned(nparts));
  const bool al = rows16<DT>(L, x, gy, gx);
  with_band(K, [&](auto s) {
    auto go = [&](auto a, auto f) {
      hipLaunchKernelGGL((cconv_bwd_mma_kernel<DT, decltype(s)::value, decltype(f)::value, decltype(a)::value>), grid,
                         dim3(kConvThreads), 0, st, (const ET*)gy, (const ET*)x, w, bias, (ET*)gx, ws, B, C, L, K,
                         run);
    };
    using SILU = std::integral_constant<int, NSQ_ACT_SILU>;
    using IDN = std::integral_constant<int, NSQ_ACT_IDENTITY>;
    if (al)
      act == NSQ_ACT_SILU ? go(std::true_type{}, SILU{}) : go(std::true_type{}, IDN{});
    else
      act == NSQ_ACT_SILU ? go(std::false_type{}, SILU{}) : go(std::false_type{}, IDN{});
  });
  hipLaunchKernelGGL(cconv_wgrad_reduce_kernel, dim3(C), dim3(kConvThreads + 64), 0, st, (const float*)ws, nparts, K,
                     gw, gb);
}

// ---------------------------------------------------------------------------
// Backward for up to 8 taps (short_bwd) in one register-resident pass (the Hyena
// short-conv case).  Thread t of a tile owns outputs n = n0 + 8t + e, e < 8.
// With the taps left-padded to KP = 4 or 8 (wk[j] = w[j - (KP - K)]):
//   pre[n]  = bias + sum_j wk[j] x[n - KP + 1 + j],  gpre = gy * silu'(pre) (or gy)
//   gx[n]   = sum_s wr[s] gpre[n + s],                wr[s] = w[K - 1 - s] (s < K)
//   gwk[j] += gpre[n] x[n - KP + 1 + j],              gb += gpre[n]
// gpre is recomputed at the KP - 1 positions past the thread's 8 (its
// neighbour owns them).  x over [n0 + 8t - 8 XB, n0 + 8t + 8 XA) and gy over
// [n0 + 8t, n0 + 8t + 8 XA) come straight from HBM in aligned chunks of 8
// (Win8).  The weight / bias sums stay in registers over the workgroup's tiles
// (one channel, a segment of its (b, tile) sequence) and are reduced in a fixed
// order into a per-workgroup partial [K + 1].
// ---------------------------------------------------------------------------
template <int DT, bool AL, int ACT, int KP>
__global__ __launch_bounds__(kConvThreads) void cconv_bwd_short_kernel(
    const typename Elem<DT>::T* __restrict__ gy, const typename Elem<DT>::T* __restrict__ x,
    const float* __restrict__ w, const float* __restrict__ bias, typename Elem<DT>::T* __restrict__ gx,
    float* __restrict__ part, int B, int C, int L, int K) {
  static_assert(KP == 4 || KP == 8, "cconv_bwd_short: taps padded to 4 or 8");
  static_assert(kConvPer == 8, "cconv_bwd_short: 8 outputs per thread");
  constexpr int NG = kConvPer + KP - 1;  // gpre positions per thread: [0, NG)
  constexpr int XB = (KP - 1 + 7) / 8;   // x chunks before the outputs: positions >= 1 - KP
  constexpr int XA = (NG + 7) / 8;       // x and gy chunks from the outputs on: positions < NG
  __shared__ float red[(KP + 1) * kConvThreads];
  const int c = int(blockIdx.x);
  const int ntiles = (L + kConvTile - 1) / kConvTile;
  const int g_begin = int(blockIdx.y) * kConvSegTiles;
  const int g_end = min(B * ntiles, g_begin + kConvSegTiles);
  const int t = int(threadIdx.x);
  float wk[KP], wr[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    const int sl = j - (KP - K);
    wk[j] = sl >= 0 ? w[int64_t(c) * K + (sl >= 0 ? sl : 0)] : 0.f;
    wr[j] = j < K ? w[int64_t(c) * K + (j < K ? K - 1 - j : 0)] : 0.f;
  }
  const float b0 = bias ? bias[c] : 0.f;
  float gwk[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) gwk[j] = 0.f;
  float gbs = 0.f;
  for (int g = g_begin; g < g_end; ++g) {
    const int b = g / ntiles, ti = g - b * ntiles;
    const int64_t row = int64_t(b) * C + c;
    const int base = ti * kConvTile + kConvPer * t;
    const RowBuf<DT, false> xb(x + row * L, L), gb(gy + row * L, L);
    Win8<DT, AL> xc[XB + XA], gc[XA];
#pragma unroll
    for (int i = 0; i < XB + XA; ++i) xc[i].load(xb, base + 8 * (i - XB));
#pragma unroll
    for (int i = 0; i < XA; ++i) gc[i].load(gb, base + 8 * i);
    // x at position base + p for p in [-8 XB, 8 XA), gy at base + p for p in [0, 8 XA)
    auto xat = [&](int p) { return xc[(p + 8 * XB) >> 3].at((p + 8 * XB) & 7); };
    auto gat = [&](int p) { return gc[p >> 3].at(p & 7); };
    float gp[NG];  // gpre at base + e
#pragma unroll
    for (int e = 0; e < NG; ++e) {
      float pre = b0;
#pragma unroll
      for (int j = 0; j < KP; ++j) pre = fmaf(wk[j], xat(e - KP + 1 + j), pre);
      gp[e] = (ACT == NSQ_ACT_SILU) ? gat(e) * dsilu(pre) : gat(e);
    }
    float out[kConvPer];
#pragma unroll
    for (int e = 0; e < kConvPer; ++e) {
      float a = 0.f;
#pragma unroll
      for (int sidx = 0; sidx < KP; ++sidx) a = fmaf(wr[sidx], gp[e + sidx], a);
      out[e] = a;
      gbs += gp[e];  // positions >= L have gy = 0, so gpre = 0
#pragma unroll
      for (int j = 0; j < KP; ++j) gwk[j] = fmaf(gp[e], xat(e - KP + 1 + j), gwk[j]);
    }
    const RowBuf<DT, AL> ob(gx + row * L, L);
#pragma unroll
    for (int e = 0; e < kConvPer; e += 2) ob.store_pair(base + e, make_float2(out[e], out[e + 1]));
  }
#pragma unroll
  for (int j = 0; j < KP; ++j) red[j * kConvThreads + t] = gwk[j];
  red[KP * kConvThreads + t] = gbs;
  __syncthreads();
  if (t <= KP) {
    float sacc = 0.f;
    for (int i = 0; i < kConvThreads; ++i) sacc += red[t * kConvThreads + i];
    // left-padded tap t -> weight index t - (KP - K); slot KP -> the bias
    const int nparts = int(gridDim.y);
    float* pw = part + (int64_t(c) * nparts + blockIdx.y) * (K + 1);
    if (t == KP)
      pw[K] = sacc;
    else if (t >= KP - K)
      pw[t - (KP - K)] = sacc;
  }
}

template <int DT>
static void launch_bwd_short(const void* gy, const void* x, const float* w, const float* bias, void* gx, float* gw,
                             float* gb, int act, int B, int C, int L, int K, float* ws, hipStream_t st) {
  using ET = typename Elem<DT>::T;
  const int64_t nparts = cconv_wgrad_parts(B, L);
  dim3 grid(C, unsigned(nparts));
  const bool al = rows16<DT>(L, x, gy, gx);
  auto go = [&](auto al_c, auto act_c) {
    constexpr bool A = decltype(al_c)::value;
    constexpr int F = decltype(act_c)::value;
    if (K <= 4)
      hipLaunchKernelGGL((cconv_bwd_short_kernel<DT, A, F, 4>), grid, dim3(kConvThreads), 0, st, (const ET*)gy,
                         (const ET*)x, w, bias, (ET*)gx, ws, B, C, L, K);
    else if constexpr (A)
      hipLaunchKernelGGL((cconv_bwd_short_kernel<DT, A, F, 8>), grid, dim3(kConvThreads), 0, st, (const ET*)gy,
                         (const ET*)x, w, bias, (ET*)gx, ws, B, C, L, K);
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  using SILU = std::integral_constant<int, NSQ_ACT_SILU>;
  using IDN = std::integral_constant<int, NSQ_ACT_IDENTITY>;
  if (al)
    act == NSQ_ACT_SILU ? go(T_{}, SILU{}) : go(T_{}, IDN{});
  else
    act == NSQ_ACT_SILU ? go(F_{}, SILU{}) : go(F_{}, IDN{});
  hipLaunchKernelGGL(cconv_wgrad_reduce_kernel, dim3(C), dim3(kConvThreads + 64), 0, st, (const float*)ws,
                     int(nparts), K, gw, gb);
}

template <int DT>
static void launch_fwd(const void* x, const float* w, const float* bias, void* y, int act, int B, int C, int L, int K,
                       hipStream_t st) {
  using ET = typename Elem<DT>::T;
  const bool al = rows16<DT>(L, x, y, nullptr);
  if (!short_fwd<DT>(K, act, int64_t(B) * C * L, al)) return launch_fwd_mma<DT>(x, w, bias, y, act, B, C, L, K, st);
  dim3 grid(B * C, unsigned(ceil_div(L, kConvTile)));
  auto go = [&](auto al_c, auto act_c) {
    constexpr bool A = decltype(al_c)::value;
    constexpr int F = decltype(act_c)::value;
    if (K <= 4)
      hipLaunchKernelGGL((cconv_fwd_short_kernel<DT, A, F, 4>), grid, dim3(kConvThreads), 0, st, (const ET*)x, w,
                         bias, (ET*)y, C, L, K);
    else if constexpr (A || (DT != NSQ_DTYPE_F32 && F == NSQ_ACT_IDENTITY)) {
      if (K <= 8)
        hipLaunchKernelGGL((cconv_fwd_short_kernel<DT, A, F, 8>), grid, dim3(kConvThreads), 0, st, (const ET*)x, w,
                           bias, (ET*)y, C, L, K);
      else if constexpr (A)
        hipLaunchKernelGGL((cconv_fwd_short_kernel<DT, A, F, 16>), grid, dim3(kConvThreads), 0, st, (const ET*)x, w,
                           bias, (ET*)y, C, L, K);
    }
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  using SILU = std::integral_constant<int, NSQ_ACT_SILU>;
  using IDN = std::integral_constant<int, NSQ_ACT_IDENTITY>;
  if (al)
    act == NSQ_ACT_SILU ? go(T_{}, SILU{}) : go(T_{}, IDN{});
  else
    act == NSQ_ACT_SILU ? go(F_{}, SILU{}) : go(F_{}, IDN{});
}

template <int DT>
static void launch_bwd(const void* gy, const void* x, const float* w, const float* bias, void* gx, float* gw,
                       float* gb, int act, int B, int C, int L, int K, float* ws, hipStream_t st) {
  if (short_bwd<DT>(K, int64_t(B) * C * L, rows16<DT>(L, x, gy, gx)))
    return launch_bwd_short<DT>(gy, x, w, bias, gx, gw, gb, act, B, C, L, K, ws, st);
  launch_bwd_mma<DT>(gy, x, w, bias, gx, gw, gb, act, B, C, L, K, ws, st);
}

static int validate_cconv(const void* a, const void* b, const float* w, int dtype, int act, int64_t B, int64_t C,
                          int64_t L, int64_t K) {
  NSQ_CHECK_ARG(a && b && w, "causal_conv1d: null tensor pointer");
  NSQ_CHECK_ARG(valid_dtype(dtype), "causal_conv1d: unsupported dtype code %d", dtype);
  NSQ_CHECK_ARG(act == NSQ_ACT_IDENTITY || act == NSQ_ACT_SILU, "causal_conv1d: activation code %d not in {0, 1}", act);
  NSQ_CHECK_ARG(B >= 1 && C >= 1 && L >= 1, "causal_conv1d: sizes must be positive");
  NSQ_CHECK_ARG(K >= 1 && K <= kConvMaxK, "causal_conv1d: kernel size %lld outside [1, %d]", (long long)K, kConvMaxK);
  NSQ_CHECK_ARG(B * C <= 0x7fffffff && L < (int64_t(1) << 28), "causal_conv1d: tensor too large (rows are staged through 32-bit byte offsets: L < 2^28)");
  return NSQ_OK;
}

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch[kMaxScratchDevices] = {nullptr};
}  // namespace

// Device address of the current GPU's scratch, looked up on the first call
// made with that device current and kept for later calls.  nullptr on failure
// (error recorded).
static float* noalloc_scratch() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices) {
    set_error("causal_conv1d_bwd_noalloc: no current HIP device (or device index >= %d)", kMaxScratchDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("causal_conv1d_bwd_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                hipGetErrorString(e));
      return nullptr;
    }
    g_scratch[dev] = static_cast<float*>(p);
  }
  return g_scratch[dev];
}

// What the noalloc entry point counts against its scratch, which fixes the shapes it takes: partials of one run per
// kConvSegTiles tiles, and for silu above 16 taps an fp32 row set [B, C, L] that no kernel needs any more (the entry
// point's shapes stay what they were).  Never less than the backward uses where that fits (at most max(C, 4096 + C)
// partial rows).
static size_t noalloc_bytes(int64_t B, int64_t C, int64_t L, int64_t K, int act) {
  const int64_t pre = act == NSQ_ACT_SILU && K > 16 ? B * C * L : 0;
  const size_t was = size_t(pre + C * cconv_wgrad_parts(B, L) * (K + 1)) * sizeof(float);
  const size_t now = nsq_causal_conv1d_bwd_workspace_bytes(B, C, L, K, act);
  return was > now ? was : now;
}

template <class... A>
static void launch_bwd_dtype(int dtype, A... a) {
  switch (dtype) {
    case NSQ_DTYPE_F32: launch_bwd<NSQ_DTYPE_F32>(a...); break;
    case NSQ_DTYPE_BF16: launch_bwd<NSQ_DTYPE_BF16>(a...); break;
    default: launch_bwd<NSQ_DTYPE_F16>(a...); break;
  }
}

}  // namespace nsq

using namespace nsq;

extern "C" {

size_t nsq_causal_conv1d_bwd_workspace_bytes(int64_t B, int64_t C, int64_t L, int64_t K, int activation) {
  (void)activation;
  // the weight / bias gradient partials [C][parts][K + 1]
  if (K < 1 || K > kConvMaxK || B < 1 || C < 1 || L < 1) return 0;
  const int64_t few = cconv_wgrad_parts(B, L), runs = mma_runs(B, C, L), parts = few > runs ? few : runs;
  return size_t(C * parts * (K + 1)) * sizeof(float);
}

int nsq_causal_conv1d_fwd(const void* x, const float* weight, const float* bias, void* y, int dtype, int activation,
                          int64_t B, int64_t C, int64_t L, int64_t K, void* stream) {
  clear_error();
  int rc = validate_cconv(x, y, weight, dtype, activation, B, C, L, K);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case NSQ_DTYPE_F32: launch_fwd<NSQ_DTYPE_F32>(x, weight, bias, y, activation, int(B), int(C), int(L), int(K), st); break;
    case NSQ_DTYPE_BF16: launch_fwd<NSQ_DTYPE_BF16>(x, weight, bias, y, activation, int(B), int(C), int(L), int(K), st); break;
    default: launch_fwd<NSQ_DTYPE_F16>(x, weight, bias, y, activation, int(B), int(C), int(L), int(K), st); break;
  }
  NSQ_CHECK_LAUNCH();
  return NSQ_OK;
}

int nsq_causal_conv1d_bwd(const void* gy, const void* x, const float* weight, const float* bias, void* gx,
                          float* gweight, float* gbias, int dtype, int activation, int64_t B, int64_t C, int64_t L,
                          int64_t K, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  int rc = validate_cconv(gy, x, weight, dtype, activation, B, C, L, K);
  if (rc) return rc;
  NSQ_CHECK_ARG(gx && gweight, "causal_conv1d_bwd: null gradient output pointer");
  const size_t need = nsq_causal_conv1d_bwd_workspace_bytes(B, C, L, K, activation);
  NSQ_CHECK_ARG(need == 0 || (workspace && workspace_bytes >= need),
                "causal_conv1d_bwd: workspace of %zu bytes required, got %zu", need, workspace_bytes);
  launch_bwd_dtype(dtype, gy, x, weight, bias, gx, gweight, gbias, activation, int(B), int(C), int(L), int(K),
                   (float*)workspace, (hipStream_t)stream);
  NSQ_CHECK_LAUNCH();
  return NSQ_OK;
}

// The partials are written in full by one kernel before the next reads them,
// so the buffer needs no clearing between calls.
int nsq_causal_conv1d_bwd_noalloc(const void* gy, const void* x, const float* weight, const float* bias, void* gx,
                                  float* gweight, float* gbias, int dtype, int activation, int64_t B, int64_t C,
                                  int64_t L, int64_t K, void* stream) {
  clear_error();
  int rc = validate_cconv(gy, x, weight, dtype, activation, B, C, L, K);
  if (rc) return rc;
  NSQ_CHECK_ARG(gx && gweight, "causal_conv1d_bwd_noalloc: null gradient output pointer");
  const size_t need = noalloc_bytes(B, C, L, K, activation);
  if (need > kNoAllocScratchBytes) {
    set_error("causal_conv1d_bwd_noalloc: B=%lld C=%lld L=%lld K=%lld needs %zu bytes of scratch, more than the "
              "fixed %zu-byte device buffer; call nsq_causal_conv1d_bwd with a workspace instead",
              (long long)B, (long long)C, (long long)L, (long long)K, need, kNoAllocScratchBytes);
    return NSQ_ERR_UNSUPPORTED;
  }
  float* ws = nullptr;
  if (need) {
    ws = noalloc_scratch();
    if (!ws) return NSQ_ERR_HIP;
  }
  launch_bwd_dtype(dtype, gy, x, weight, bias, gx, gweight, gbias, activation, int(B), int(C), int(L), int(K), ws,
                   (hipStream_t)stream);
  NSQ_CHECK_LAUNCH();
  return NSQ_OK;
}

}  // extern "C"
