// Launches of the small-plane 2D convolution (fftconv2d_plane.h); one unit per
// dtype instantiates them (fftconv2d_plane_{f32,bf16,f16}.hip).
#pragma once

#include "fftconv_nd_plan.h"
#include "fftconv2d_plane.h"

namespace nsq {

// gk[i] = sum of the nz shares in order; gs[h] = channel h's value at the shift (lag 0).
static __global__ __launch_bounds__(256) void plane2_reduce_kernel(const float* __restrict__ part, int nz, int64_t n,
                                                                   int size, int lag0, float* __restrict__ gk,
                                                                   float* __restrict__ gs) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  float a = part[i];
  for (int z = 1; z < nz; ++z) a += part[z * n + i];
  gk[i] = a;
  if (gs && i % size == lag0) gs[i / size] = a;
}

template <class F>
inline void with_plane2(const Plane2Size& z, F&& f) {
  with_log<4, 7>(z.lF0, [&](auto A) {
    with_log<3, 6>(z.lM, [&](auto B) {
      constexpr int LA = decltype(A)::value, LB = decltype(B)::value;
      if constexpr (LA + LB >= 9 && LA + LB <= 13) f(Plane2<LA, LB>{});
    });
  });
}

template <class K>
inline void plane2_allow_lds(K* kernel, size_t bytes) {
  if (bytes > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(bytes));
}

// Workgroups a channel's batch is split over.  They run in rounds of as many as the GPU holds at once, and a round takes
// a workgroup's own transforms (`fixed`: the filter's, its gradient's) and those of its images (`each`): the split with
// the least rounds x transforms, the smallest of them.  (4096 waves, whatever their rounds, left 8 of 520 workgroups to
// a second round at B=28 H=130 39 x 25, K = 77 x 25: gated forward + backward 425 us in bf16.)
template <class K>
inline int64_t plane2_split(K* kernel, int threads, size_t lds, const NdPlan& p, int64_t most, int fixed, int each) {
  int per_cu = 1;
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), threads, lds);
  const int64_t slots = int64_t(256) * (per_cu < 1 ? 1 : per_cu);
  const int64_t B = p.B, H = p.H;
  int64_t best = 1, cost = 0;
  for (int64_t per = B; per >= 1;) {  // share sizes, downwards: one for each number of shares where B allows
    const int64_t nz = ceil_div(B, per);
    if (nz > most) break;
    const int64_t c = ceil_div(H * nz, slots) * (fixed + each * per);
    if (per == B || c < cost) {
      best = nz;
      cost = c;
    }
    const int64_t next = ceil_div(B, nz + 1);
    per = next < per ? next : per - 1;
  }
  return best;
}

inline Plane2Geom plane2_geom(const NdPlan& p, int dtype, std::initializer_list<const void*> images) {
  const uintptr_t access = dtype == NSQ_DTYPE_F32 ? 16 : 8;
  bool vec = int64_t(p.S[0]) * p.S[2] % 4 == 0;
  for (const void* q : images) vec = vec && reinterpret_cast<uintptr_t>(q) % access == 0;
  return Plane2Geom{int(p.B), int(p.H), p.S[0], p.S[2], p.K[0], p.K[2], p.c[0], p.c[2], int(p.kb != 1), 1, int(vec)};
}

template <int DT>
void plane2_fwd(const NdPlan& p, const Plane2Size& z, const void* x, const float* k, const void* s, void* y,
                const GatedIO* gate, const float2* tw, hipStream_t st) {
  using ET = typename Elem<DT>::T;
  with_plane2(z, [&](auto pl) {
    using P = decltype(pl);
    auto go = [&](auto gated) {
      constexpr bool G = decltype(gated)::value;
      const GatedIO ga = G ? *gate : GatedIO{};
      Plane2Geom g = plane2_geom(p, DT, {x, y, ga.kg, ga.v, ga.y1out});
      const size_t lds = plane2_lds<P, DT>(g);
      auto* kern = &plane2_fwd_kernel<DT, P, G>;
      plane2_allow_lds(kern, lds);
      if (p.kb == 1) g.per_wg = int(ceil_div(p.B, plane2_split(kern, P::T, lds, p, plane2_max_split(p, z), 1, 2)));
      hipLaunchKernelGGL(kern, dim3(unsigned(p.H * ceil_div(p.B, g.per_wg))), dim3(P::T), lds, st,
                         (const ET*)x, k, (const ET*)s, (ET*)y, g, ga, tw);
    };
    gate ? go(std::true_type{}) : go(std::false_type{});
  });
}

template <int DT>
void plane2_bwd(const NdPlan& p, const Plane2Size& z, const void* gy, const void* x, const float* k, const void* s,
                void* gx, float* gk, float* gs, float* ws, const GatedIO* gate, const float2* tw, hipStream_t st) {
  using ET = typename Elem<DT>::T;
  with_plane2(z, [&](auto pl) {
    using P = decltype(pl);
    auto go = [&](auto gated) {
      constexpr bool G = decltype(gated)::value;
      const GatedIO ga = G ? *gate : GatedIO{};
      Plane2Geom g = plane2_geom(p, DT, {gy, x, gx, ga.kg, ga.v, ga.y1, ga.dv, ga.dkg});
      const size_t lds = plane2_lds<P, DT>(g);
      auto* kern = &plane2_bwd_kernel<DT, P, G>;
      plane2_allow_lds(kern, lds);
      if (p.kb == 1) g.per_wg = int(ceil_div(p.B, plane2_split(kern, P::T, lds, p, plane2_max_split(p, z), 2, 3)));
      const int nz = int(ceil_div(p.B, g.per_wg));
      float* part = p.kb == 1 && nz > 1 ? ws : nullptr;
      hipLaunchKernelGGL(kern, dim3(unsigned(p.H * nz)), dim3(P::T), lds, st, (const ET*)gy, (const ET*)x, k,
                         (const ET*)s, (ET*)gx, gk, gs, part, g, ga, tw);
      if (part) {
        const int size = p.K[0] * p.K[2];
        const int64_t n = p.H * size;
        hipLaunchKernelGGL(plane2_reduce_kernel, dim3(unsigned(ceil_div(n, 256))), dim3(256), 0, st,
                           (const float*)part, nz, n, size, p.c[0] * p.K[2] + p.c[2], gk, gs);
      }
    };
    gate ? go(std::true_type{}) : go(std::false_type{});
  });
}

#define NSQ_PLANE2_INSTANCES(DT)                                                                                    \
  template void plane2_fwd<DT>(const NdPlan&, const Plane2Size&, const void*, const float*, const void*, void*,     \
                               const GatedIO*, const float2*, hipStream_t);                                        \
  template void plane2_bwd<DT>(const NdPlan&, const Plane2Size&, const void*, const void*, const float*,            \
                               const void*, void*, float*, float*, float*, const GatedIO*, const float2*,          \
                               hipStream_t);

}  // namespace nsq
