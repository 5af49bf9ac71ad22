// oit_tiles.hip - pass 1 of the tile path (runs per tile) and the dispatch of
// its composites, which are compiled one layer count at a time
// (oit_tiles_k.hip).
#include "oit_tiles.hpp"

namespace oit {

namespace {

// Runs with gaps, for a chunk of many runs whose targets are all valid: a
// lane joins the nearest earlier lane of its tile at most kGap lanes before
// it, and a run goes from a chain's first lane to its last, over the lanes of
// other tiles in between, which the composite drops. A rasteriser that walks
// triangles in 2x2 quads alternates between two rows, so that a chunk is two
// runs so and up to 32 without (1920x1080 in quads, 12.7 M fragments: Loop64
// K = 8 502 us without, 276 with, 310 with an atomic per fragment; K = 16 518,
// 290, 247; Loop32 588, 336, 358). The gap is as long as what a quad of four
// front and four back fragments needs. Chunks of few runs, as raster order
// leaves them, are not looked through, and the code is kept small: unrolled
// over lanes and chunks it took them 23.5 us instead of 22.
constexpr int kManyStarts = 15;  // runs of a chunk past which gaps are looked for: spheres of a pixel or two make up to 14
constexpr uint32_t kGap = 8;    // (join_gaps' shifts go by it)
constexpr int kGapTiles = 16;
// A chunk that is still of more than kDirectRuns runs puts them on the tiles'
// lists, list by lane, without drawing a place: one atomic a run instead of
// two, and no scattered record (1920x1080 shuffled, 12.7 M runs: 1.39 ms for
// this pass with places, the Loop64 frame 3.08 ms; 2.70 so. 256x256, 338
// thousand: 186 and 134 us). Whoever finds a list empty marks the tile. Not in
// a batch, whose binning goes by the run counts.
constexpr int kDirectRuns = 32;
__device__ __forceinline__ void join_gaps(uint32_t tile, bool& lead, uint32_t& run) {
  // the lanes of the lane's tile, for the first kGapTiles tiles of the chunk
  uint64_t mine = 0ull, left = __ballot(tile != kEmpty);
#pragma unroll 1
  for (int n = 0; left != 0ull && n < kGapTiles; ++n) {
    const uint64_t same = __ballot(tile == (uint32_t)__builtin_amdgcn_readlane(tile, __builtin_ctzll(left)));
    if ((same >> lane_id()) & 1u) mine = same;
    left &= ~same;
  }
  if (mine == 0ull) return;
  const uint32_t lane = lane_id();
  lead = lane == 0u || (mine << (64u - lane)) >> (64u - kGap) == 0ull;
  // from the lane on: every member and the kGap - 1 lanes after it; the next
  // gap of that ends the chain
  const uint64_t from = mine >> lane;
  uint64_t reach = from | from << 1;
  reach |= reach << 2;
  reach |= reach << 4;
  const uint64_t chain = ~reach ? from & ((1ull << __builtin_ctzll(~reach)) - 1ull) : from;
  run = pack_run(64u - (uint32_t)__builtin_clzll(chain), (uint32_t)__builtin_popcountll(chain));
}

// One of a tile's runs of which another `place` came before: into the tile's
// own slots, or onto its lists.
__device__ __forceinline__ void put_run(const TileBuf& tb, uint32_t tile, uint32_t place, uint32_t id, uint32_t word) {
  const uint64_t at = (uint64_t)tile * kTileRuns;
  if (place < kTileRuns) {
    tb.run[at + place] = ((uint64_t)id << 32) | word;
  } else {
    const uint32_t prev = __hip_atomic_exchange(&tb.more[at + place % kTileRuns], id + 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    tb.link[id] = ((uint64_t)word << 32) | prev;
  }
}

// The run that starts at the lane, of a chunk whose runs start at `starts`.
__device__ __forceinline__ uint32_t run_from(uint64_t starts) {
  const uint64_t above = (starts >> lane_id()) >> 1;
  const uint32_t len = above ? (uint32_t)__builtin_ctzll(above) + 1u : 64u - lane_id();
  return pack_run(len, len);
}

// A chunk of many runs, from its targets on (a wave comes here with all of
// its chunks, one by one: little code beside the path that raster order takes).
template <bool kDirect>
__device__ __forceinline__ void link_scattered(const FragView& f, uint32_t T, uint32_t spp, uint32_t tile0,
                                               const TileBuf& tb, uint64_t first) {
  const uint64_t i = first + lane_id();
  const bool in = i < f.count;
  const uint32_t t = in ? f.target[i] : kEmpty;
  const uint32_t tile = t < T ? tile0 + (pm_index(t, T, spp) >> 6) : kEmpty;
  const uint32_t before = __shfl_up(tile, 1u);
  const bool start = lane_id() == 0u || before != tile;
  bool lead = start && tile != kEmpty;
  uint32_t run = run_from(__ballot(start));
  // (a fragment without a valid target inside a run could pass for one of its tile's)
  if (__ballot(in && tile == kEmpty) == 0ull) join_gaps(tile, lead, run);
  const uint32_t id = f.id_base + (uint32_t)i;
  if (kDirect && __builtin_popcountll(__ballot(lead)) > kDirectRuns) {
    if (!lead) return;
    const uint32_t prev = __hip_atomic_exchange(&tb.more[(uint64_t)tile * kTileRuns + lane_id()], id + 1u,
                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    tb.link[id] = ((uint64_t)run << 32) | prev;
    if (prev == 0u) atomicOr(&tb.cnt[tile], kTileUncounted);
  } else if (lead) {
    put_run(tb, tile, atomicAdd(&tb.cnt[tile], 1u) & ~kTileUncounted, id, run);
  }
}

// Pass 1 over one source stream: fragments first .. first + 64 kU - 1.
// Fragments behind the opaque pass stay in their runs (pass 2 tests them):
// where a surface runs between the front and the back of a sphere, every
// second fragment is behind it, and the runs would be of one fragment
// (808x402, 24 opaque spheres: 30 us for this pass, 10 so).
template <int kU, bool kDirect>
__device__ __forceinline__ void link_wave(const FragView& f, uint32_t T, uint32_t spp, uint32_t tile0,
                                          const TileBuf& tb, uint64_t first) {
  const uint32_t lane = lane_id();
  uint32_t t[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const uint64_t i = first + (uint64_t)u * 64u + lane;
    const bool in = i < f.count;
    t[u] = in ? ld_stream(&f.target[i]) : kEmpty;
  }
  bool lead[kU];
  uint64_t starts[kU];
  uint32_t pos[kU];
  int most = 0;  // runs of a chunk
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    if (t[u] >= T) t[u] = kEmpty;
    const uint32_t tile = t[u] == kEmpty ? kEmpty : tile0 + (pm_index(t[u], T, spp) >> 6);
    const uint32_t before = __shfl_up(tile, 1u);
    const bool start = lane == 0u || before != tile;
    starts[u] = __ballot(start);
    const int runs = __builtin_popcountll(starts[u]);
    most = most > runs ? most : runs;
    lead[u] = start && tile != kEmpty;
    t[u] = tile;
    pos[u] = 0u;
    asm volatile("" : "+v"(pos[u]));  // the zeros are written before any atomic goes out
  }
  if (most > kManyStarts) {  // (wave-uniform)
#pragma unroll 1
    for (int u = 0; u < kU; ++u) link_scattered<kDirect>(f, T, spp, tile0, tb, first + (uint64_t)u * 64u);
    return;
  }
#pragma unroll
  for (int u = 0; u < kU; ++u)
    if (lead[u]) pos[u] = atomicAdd(&tb.cnt[t[u]], 1u);
  returns_done();
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    if (lead[u])
      put_run(tb, t[u], kDirect ? pos[u] & ~kTileUncounted : pos[u],
              f.id_base + (uint32_t)(first + (uint64_t)u * 64u + lane), run_from(starts[u]));
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
  link_wave<kU, true>(f, c.T, c.spp, 0u, tb, first);
}

template <int kU>
__global__ __launch_bounds__(kBlock) void k_tile_link_batch(BatchArgs b, TileBuf tb) {
  reset_ctl(tb);
  if (blockIdx.x == 0)
    for (uint32_t i = kTileTickets + threadIdx.x; i < kTileCtlBatch; i += kBlock) tb.ctl[i] = 0u;
  const uint32_t unit = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6));
  if (unit >= b.units) return;
  const uint64_t g = (uint64_t)unit * (64u * kU);
  const BatchFrameDev fr = b.frames[find_frame<false>(b.frames, b.f0, b.f1, g)];
  FragView f;
  f.target = fr.target;
  f.depth = fr.depth;
  f.rgba = fr.rgba;
  f.count = fr.count;
  f.id_base = fr.frag_base;
  link_wave<kU, false>(f, fr.T, 1u, fr.target_base / 64u, tb, g - fr.frag_base);
}

// The queued tiles of a batch group (more fragments than a wave's LDS holds):
// each tile's fragments into its targets' buckets, one behind the other and
// each in id order, by a counting sort. A block's waves take a share of the
// tile's sorted runs each, count per target, and place their fragments behind
// the earlier shares'; a fragment's place among its batch's is its rank among
// the lanes of its target. Against a wave per tile that reads the tile once
// for every 696 fragments' worth of targets, the 24-frame mix (205 M
// fragments, about 120 M of them in such tiles) went from 10.3 to 5.4 ms, with
// rows of 16 targets (below) and one queue atomic for 64 tiles to 4.3, with
// tickets to 3.9: blocks that stepped through the queue were at work half of
// the time, some tiles holding 36 thousand fragments. Bound by its scattered
// 8-byte stores and about 230 vector instructions per 64 fragments.
// Leaves each target's number and place in `run` and
// the tile's base in the first two words of `more`.
constexpr uint32_t kBinThreads = 256;
constexpr uint32_t kBinWaves = kBinThreads / 64u;

struct BinWave {
  uint32_t bits[128];
  uint32_t delta[64];
  uint32_t at[64];  // per target: the share's fragments, then its next place
};

// Calls body(ids, act) for kU batches of 64 fragments of the runs r0 .. r1 - 1
// at a time, in order. An inactive lane's id is a fragment of the runs.
template <int kU, typename F>
__device__ __forceinline__ void each_batch(BinWave& w, const uint64_t* run, uint32_t r0, uint32_t r1, F&& body) {
  const uint32_t lane = lane_id();
  for (uint32_t r = r0; r < r1; r += 64u) {
    const bool on = r + lane < r1;
    const uint64_t rec = on ? run[r + lane] : 0ull;
    const uint32_t start = (uint32_t)(rec >> 32), len = run_len((uint32_t)rec);
    const uint32_t incl = wave_scan_u32(len);
    const uint32_t size = __builtin_amdgcn_readlane(incl, 63);  // 64 runs of at most 64 each
    const uint32_t id0 = rfl(start);
    clear_marks(w);
    mark_run(w, on, incl - len);
    w.delta[lane] = start - (incl - len);
    wave_lds_sync();
    const uint32_t lo_bits = w.bits[2u * lane], hi_bits = w.bits[2u * lane + 1u];
    const uint32_t n_starts = (uint32_t)__builtin_popcount(lo_bits) + (uint32_t)__builtin_popcount(hi_bits);
    const uint32_t below = wave_scan_u32(n_starts) - n_starts;
    for (uint32_t b = 0; b * 64u < size; b += kU) {
      uint32_t id[kU];
      bool act[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t bb = b + (uint32_t)u, pos = bb * 64u + lane;
        const uint32_t k = __builtin_amdgcn_mbcnt_hi(
            __builtin_amdgcn_readlane(hi_bits, bb & 63u),
            __builtin_amdgcn_mbcnt_lo(__builtin_amdgcn_readlane(lo_bits, bb & 63u),
                                      __builtin_amdgcn_readlane(below, bb & 63u)));
        act[u] = pos < size;
        id[u] = act[u] ? w.delta[k & 63u] + pos : id0;
      }
      body(id, act);
    }
    wave_lds_sync();
  }
}

struct BinArgs {
  TileBuf tb;
  const BatchFrameDev* frames;
  uint32_t f0, f1, split;
  const CodecTables* tab;
};

__global__ __launch_bounds__(kBinThreads, 8) void k_tile_bin(BinArgs g) {
  __shared__ uint64_t s_run[kBinRuns];
  __shared__ BinWave s_w[kBinWaves];
  __shared__ uint64_t s_base;
  __shared__ uint32_t s_next;
  const uint32_t lane = lane_id(), wave = rfl(threadIdx.x >> 6);
  const uint32_t n_tiles = rfl(ld_relaxed(&g.tb.ctl[g.tb.ctl_index]));
  BinWave& w = s_w[wave];
  const uint32_t turn = blockIdx.x % kTicketLanes;
  for (uint32_t q = blockIdx.x; q < n_tiles;) {
    uint32_t ticket = 0;
    if (threadIdx.x == 0) ticket = draw_ticket(g.tb, g.tb.ticket0 + turn * 16u);
    const uint32_t entry = rfl(g.tb.deep[g.tb.deep_base + q]);
    const uint32_t tile = g.split ? g.tb.tile_first + (entry & 0xFFFFu) : entry;
    const uint32_t m = rfl(g.tb.cnt[tile]);
    // Left to the deep composite, which like this kernel and the binned
    // composite tells such a tile by its run count: the entry is read by every
    // wave of the block and by later kernels, so nothing is written to it. (The
    // count is the same in every thread: cleared by the composites alone.)
    if (m > kBinRuns) {
      if (threadIdx.x == 0) {
        atomicAdd(&g.tb.ctl[g.tb.ctl_index + 1u], 1u);
        s_next = gridDim.x + turn + kTicketLanes * ticket;
      }
      __syncthreads();
      q = rfl(s_next);
      __syncthreads();
      continue;
    }
    const auto fr = (FramePtr)g.frames;
    const uint32_t f = rfl(find_frame<true>(g.frames, g.f0, g.f1, (uint64_t)tile * kTileTargets));
    const uint32_t id_base = fr[f].frag_base;
    const uint32_t base_target = tile * kTileTargets - fr[f].target_base;  // the tile's first target
    const auto* const target = (const __attribute__((address_space(1))) uint32_t*)fr[f].target;
    const auto* const depth = (const __attribute__((address_space(1))) float*)fr[f].depth;
    const float4* const rgba = fr[f].rgba;
    // the runs, in ascending order of their first ids
    if (wave == 0u) {
      uint32_t got = 0;
      each_run(g.tb, tile, m, [&](uint32_t start, uint32_t len, bool on) {
        const uint64_t mask = __ballot(on);
        if (on) s_run[got + lanes_below(mask)] = ((uint64_t)start << 32) | len;
        got += (uint32_t)__builtin_popcountll(mask);
      });
    }
    w.at[lane] = 0u;
    if (threadIdx.x == 0) s_next = gridDim.x + turn + kTicketLanes * ticket;
    __syncthreads();
    if (m <= kBinThreads) {
      const uint64_t mine = threadIdx.x < m ? s_run[threadIdx.x] : 0ull;
      uint32_t rank = 0;
      for (uint32_t j = 0; j < m; ++j) rank += (uint32_t)(s_run[j] >> 32) < (uint32_t)(mine >> 32) ? 1u : 0u;
      __syncthreads();
      if (threadIdx.x < m) s_run[rank] = mine;
    } else {
      uint32_t size = 2u * kBinThreads;
      while (size < m) size <<= 1;
      for (uint32_t i = m + threadIdx.x; i < size; i += kBinThreads) s_run[i] = kEmpty64;
      for (uint32_t k = 2; k <= size; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
          __syncthreads();
          for (uint32_t i = threadIdx.x; i < size; i += kBinThreads) {
            const uint32_t x = i ^ j;
            if (x > i) {
              const uint64_t a = s_run[i], b = s_run[x];
              if (((i & k) == 0u) == (a > b)) {
                s_run[i] = b;
                s_run[x] = a;
              }
            }
          }
        }
      }
    }
    __syncthreads();
    const uint32_t r0 = m * wave / kBinWaves, r1 = m * (wave + 1u) / kBinWaves;
    constexpr int kC = 8;
    each_batch<kC>(w, s_run, r0, r1, [&](const uint32_t (&id)[kC], const bool (&act)[kC]) {
      uint32_t t[kC];
#pragma unroll
      for (int u = 0; u < kC; ++u) t[u] = target[id[u] - id_base];
#pragma unroll
      for (int u = 0; u < kC; ++u) {
        const uint32_t loc = t[u] - base_target;
        if (act[u] && loc < kTileTargets) atomicAdd(&w.at[loc], 1u);  // (not another tile's, in a gap)
      }
    });
    __syncthreads();
    if (wave == 0u) {
      uint32_t n[kBinWaves], sum = 0;
#pragma unroll
      for (uint32_t v = 0; v < kBinWaves; ++v) {
        n[v] = s_w[v].at[lane];
        sum += n[v];
      }
      // 16 neighbouring targets share rows of 16 entries, a cache line, where
      // that takes at most half as much again as their entries: neighbours
      // are written and read together
      uint32_t top = sum, all = sum;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)top, o);
        top = top > other ? top : other;
        all += (uint32_t)__shfl_xor((int)all, o);
      }
      const bool rows = 32u * top <= 3u * all;
      const uint32_t space = rows ? 16u * top : all;
      const uint32_t incl = wave_scan_u32((lane & 15u) == 0u ? space : 0u);
      const uint32_t before = wave_scan_u32(sum) - sum;
      const uint32_t group0 = (uint32_t)__shfl((int)before, (int)(lane & 48u));
      uint32_t at = (incl - space) + (rows ? lane & 15u : before - group0);
      if (rows) at |= kBinRow;
      const uint32_t step = bin_step(at);
      // the tiles' fragments are disjoint: all of them fit
      if (lane == 63u) {
        const uint64_t base = atomicAdd((unsigned long long*)&g.tb.ctl[kTileBucket], (unsigned long long)incl);
        g.tb.more[(uint64_t)tile * kTileRuns] = (uint32_t)base;
        g.tb.more[(uint64_t)tile * kTileRuns + 1u] = (uint32_t)(base >> 32);
        s_base = base;
      }
      g.tb.run[(uint64_t)tile * kTileRuns + lane] = ((uint64_t)sum << 32) | at;
#pragma unroll
      for (uint32_t v = 0; v < kBinWaves; ++v) {
        s_w[v].at[lane] = at;
        at += n[v] * step;
      }
    }
    __syncthreads();
    const uint64_t base = s_base;
    auto* const out = (__attribute__((address_space(1))) uint64_t*)g.tb.bucket + (((uint64_t)rfl((uint32_t)(base >> 32)) << 32) | rfl((uint32_t)base));
    constexpr int kU = 4;
    each_batch<kU>(w, s_run, r0, r1, [&](const uint32_t (&id)[kU], const bool (&act)[kU]) {
      uint32_t t[kU];
      float dv[kU];
      float4 cv[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t i = id[u] - id_base;
        t[u] = target[i];
        dv[u] = depth[i];
        cv[u] = ld_global_stream(&rgba[i]);
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t off = t[u] - base_target, loc = off & 63u;
        const bool on = act[u] && off < kTileTargets;
        const uint64_t cd = ((uint64_t)depth_key(dv[u]) << 32) | encode_color_quick(cv[u], g.tab);
        uint64_t same = __ballot(on);
#pragma unroll
        for (uint32_t b = 0; b < 6u; ++b) {
          const bool bit = (loc >> b) & 1u;
          const uint64_t set = __ballot(bit);
          same &= bit ? set : ~set;
        }
        wave_lds_sync();
        const uint32_t at = w.at[loc];
        const uint32_t n = (uint32_t)__builtin_popcountll(same), rank = lanes_below(same);
        wave_lds_sync();
        if (on) {
          const uint32_t step = bin_step(at);
          out[bin_at(at) + rank * step] = cd;
          if (rank + 1u == n) w.at[loc] = at + n * step;
        }
      }
    });
    q = rfl(s_next);
    __syncthreads();
  }
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

hipError_t launch_tile_link_batch(const BatchArgs& a, const TileBuf& tb, hipStream_t s) {
  const uint32_t blocks = (a.units + kBlock / 64 - 1u) / (kBlock / 64);
  hipLaunchKernelGGL((k_tile_link_batch<8>), dim3(blocks ? blocks : 1u), dim3(kBlock), 0, s, a, tb);
  return hipGetLastError();
}

hipError_t launch_tile_bin(const BatchArgs& a, const TileBuf& tb, uint32_t tiles, uint32_t split, hipStream_t s) {
  const BinArgs args{tb, a.frames, a.f0, a.f1, split, a.tab};
  constexpr uint32_t kResident = kComputeUnits * (2048u / kBinThreads);
  const uint32_t blocks = tiles < kResident ? (tiles + kTicketLanes - 1u) / kTicketLanes * kTicketLanes : kResident;
  hipLaunchKernelGGL(k_tile_bin, dim3(blocks), dim3(kBinThreads), 0, s, args);
  return hipGetLastError();
}

hipError_t launch_tile_batch(const BatchArgs& a, const TileBuf& tb, uint32_t K, bool tail, hipStream_t s) {
  if (a.tiles == 0) return hipSuccess;
  switch (K) {
    case 1: return tile_batch_k<1>(a, tb, tail, s);
    case 2: return tile_batch_k<2>(a, tb, tail, s);
    case 4: return tile_batch_k<4>(a, tb, tail, s);
    case 8: return tile_batch_k<8>(a, tb, tail, s);
    case 16: return tile_batch_k<16>(a, tb, tail, s);
    case 32: return tile_batch_k<32>(a, tb, tail, s);
    default: return hipErrorInvalidValue;
  }
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
