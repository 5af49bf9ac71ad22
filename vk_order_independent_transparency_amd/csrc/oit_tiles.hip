// oit_tiles.hip - pass 1 of the tile path (runs per tile) and the dispatch of
// its composites, which are compiled one layer count at a time
// (oit_tiles_k.hip).
#include "oit_frame.hpp"

namespace oit {

namespace {

// Pass 1 over one source stream: fragments first .. first + 64 kU - 1.
template <int kU>
__device__ __forceinline__ void link_wave(const FragView& f, uint32_t T, uint32_t spp, uint32_t tile0,
                                          const uint64_t* opq, const TileBuf& tb, uint64_t first) {
  const uint32_t lane = lane_id();
  uint32_t t[kU];
  float dv[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const uint64_t i = first + (uint64_t)u * 64u + lane;
    const bool in = i < f.count;
    t[u] = in ? ld_stream(&f.target[i]) : kEmpty;
    dv[u] = (opq && in) ? ld_stream(&f.depth[i]) : 0.f;
  }
  bool lead[kU];
  uint32_t len[kU], pos[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    if (t[u] >= T) t[u] = kEmpty;
    if (opq && t[u] != kEmpty && !opaque_visible(opq, T, 1u, t[u], depth_key(dv[u]), 1u)) t[u] = kEmpty;
    const uint32_t tile = t[u] == kEmpty ? kEmpty : tile0 + (pm_index(t[u], T, spp) >> 6);
    const uint32_t before = __shfl_up(tile, 1u);
    const bool start = lane == 0u || before != tile;
    const uint64_t above = (__ballot(start) >> lane) >> 1;
    len[u] = above ? (uint32_t)__builtin_ctzll(above) + 1u : 64u - lane;
    lead[u] = start && tile != kEmpty;
    t[u] = tile;
    pos[u] = 0u;
    asm volatile("" : "+v"(pos[u]));  // the zeros are written before any atomic goes out
  }
#pragma unroll
  for (int u = 0; u < kU; ++u)
    if (lead[u]) pos[u] = atomicAdd(&tb.cnt[t[u]], 1u);
  returns_done();
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    if (lead[u]) {
      const uint32_t id = f.id_base + (uint32_t)(first + (uint64_t)u * 64u + lane);
      const uint64_t at = (uint64_t)t[u] * kTileRuns;
      if (pos[u] < kTileRuns) {
        tb.run[at + pos[u]] = ((uint64_t)id << 32) | len[u];
      } else {
        const uint32_t prev = __hip_atomic_exchange(&tb.more[at + pos[u] % kTileRuns], id + 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        tb.link[id] = ((uint64_t)len[u] << 32) | prev;
      }
    }
  }
}

__device__ __forceinline__ void reset_ctl(const TileBuf& tb) {
  if (blockIdx.x == 0)
    for (uint32_t i = threadIdx.x; i < kTileCtlWords; i += blockDim.x) tb.ctl[i] = 0u;
}

template <int kU>
__global__ __launch_bounds__(kBlock) void k_tile_link(Common c, FragView f, TileBuf tb) {
  reset_ctl(tb);
  const uint64_t first = ((uint64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * (64u * kU);
  link_wave<kU>(f, c.T, c.spp, 0u, c.opq_z, tb, first);
}

__global__ __launch_bounds__(64) void k_set_segs(SegArgs a, TileSeg* dst) {
  if (threadIdx.x < a.n) dst[threadIdx.x] = a.s[threadIdx.x];
}

}  // namespace

hipError_t launch_tile_link(const Common& c, const FragView& f, const TileBuf& tb, hipStream_t s) {
  if (f.count == 0) return hipSuccess;
  constexpr int kU = 4;
  const dim3 g((uint32_t)(((uint64_t)f.count + kBlock * kU - 1) / (kBlock * kU))), b(kBlock);
  hipLaunchKernelGGL((k_tile_link<kU>), g, b, 0, s, c, f, tb);
  return hipGetLastError();
}

hipError_t launch_set_segs(const TileSeg* segs, uint32_t n, TileSeg* dst, hipStream_t s) {
  for (uint32_t i = 0; i < n; i += kSegArgs) {
    SegArgs a;
    a.n = n - i < kSegArgs ? n - i : kSegArgs;
    for (uint32_t j = 0; j < a.n; ++j) a.s[j] = segs[i + j];
    hipLaunchKernelGGL(k_set_segs, dim3(1), dim3(64), 0, s, a, dst + i);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_tile_resolve(const TileBuf& tb, const TileSrc& src, const TileDst& dst, uint32_t K, int mode,
                               bool tail, hipStream_t s) {
  switch (K) {
    case 1: return tile_resolve_k<1>(tb, src, dst, mode, tail, s);
    case 2: return tile_resolve_k<2>(tb, src, dst, mode, tail, s);
    case 4: return tile_resolve_k<4>(tb, src, dst, mode, tail, s);
    case 8: return tile_resolve_k<8>(tb, src, dst, mode, tail, s);
    case 16: return tile_resolve_k<16>(tb, src, dst, mode, tail, s);
    case 32: return tile_resolve_k<32>(tb, src, dst, mode, tail, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace oit
