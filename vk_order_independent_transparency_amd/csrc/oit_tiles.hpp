// oit_tiles.hpp - the tile path: a frame's fragments are not linked or stored
// per target but listed per tile of 64 targets, as runs of consecutive
// fragments, and one wave composites a tile from LDS.
//
// Why: the per-target structures (lists, slots) cost a memory-side atomic or
// a scattered read-modify-write per fragment or per pair of fragments and
// then a composite bound by dependent loads. A rasterised fragment stream is
// coherent: consecutive fragments fall on consecutive targets, so 64 of them
// touch one or two tiles of 64 consecutive targets (one or two atomics), and
// the composite reads whole runs with coalesced loads, builds the targets'
// lists in LDS and sorts them in registers.
//
// Pass 1 (k_tile_link, per append): each wave cuts its 64-fragment chunks
// into runs of one tile (with short gaps where there are many, join_gaps) and
// publishes every run (first id, length, the tile's own fragments among
// those) with one returning add on the tile's run count: the first kTileRuns
// runs go to the tile's own slots, later ones onto kTileRuns unordered lists
// of the tile (run number mod kTileRuns), so that a wave walks them side by
// side. Chunks without any order put their runs on the lists directly.
// Pass 2 (k_tile_resolve): one wave per tile sorts the runs by first id,
// takes their fragments 64 at a time, pushes (key, colour) onto the targets'
// lists in LDS in ascending id, and each lane then walks its own target's
// list, newest fragment first (the walk order of the reference's lists,
// oitLinkedList.frag.glsl:72,116-143).
// Tiles with over 1024 runs, or of many runs that would be read more often
// than pays, go to a queue that k_tile_deep takes: the same, in groups of
// fragments from the newest to the oldest, with the front K kept in
// registers. A batch's queue is taken by k_tile_bin (oit_tiles.hip) and
// k_tile_binned: per target in order in memory, then a lane per target. The line between them is what a wave's LDS holds: 696
// fragments; read in parts beyond it, the batch took 10.3 ms against 3.6.
//
// Measured (composite alone): 1920x1080 Loop64 K = 8, 12.7 M fragments, 147
// us, where counting, storing, classifying and compositing per target took
// 290; 1600x900 Loop32 K = 16, 8.8 M, 175 us against 290. While resident, the
// waves keep the vector units about 80 % busy; the rest is uneven tiles.
//
// The result is a function of the frame's fragments and their ids alone, so
// every algorithm whose stored set does not depend on arrival is composited
// here with its own order and tail rule (TileMode).
#pragma once

#include <cstddef>

#include "oit_frame.hpp"

namespace oit {

namespace {

constexpr uint32_t kTileTargets = 64;

// A run's word: ids it goes over (1 .. 64) and how many of them are the
// tile's own.
__device__ __forceinline__ uint32_t pack_run(uint32_t len, uint32_t own) { return len | own << 8; }
__device__ __forceinline__ uint32_t run_len(uint32_t w) { return w & 255u; }
__device__ __forceinline__ uint32_t run_own(uint32_t w) { return w >> 8; }

// Per-wave LDS of a group of fragments: entries in ascending id, 1 ..
// kEntries, linked per target. A list value is the entry's LDS address, so a
// walk needs no address arithmetic. Entry 0 ends every list: its key is above
// every depth key, it is its own successor and its colour is transparent, so
// walks and blends need no test for a list's end either. kId: the entries
// hold their fragments' ids too (Loop32's tail, the debug outputs).
struct TileEntry {
  uint32_t key;
  uint32_t next;
  uint32_t col;
};
struct alignas(16) TileEntryId {
  uint32_t key;
  uint32_t next;
  uint32_t col;
  uint32_t id;
};
template <bool kId>
struct EntryOf {
  using T = TileEntry;
};
template <>
struct EntryOf<true> {
  using T = TileEntryId;
};
// Aligned for the 64-bit runs that are sorted in the entries' space: a block
// holds several of these one behind the other.
template <int C, bool kId>
struct alignas(16) TileLds {
  static constexpr uint32_t kEntries = C;
  static constexpr bool kHasId = kId;
  static constexpr uint32_t kSize = sizeof(typename EntryOf<kId>::T);
  typename EntryOf<kId>::T e[C + 1];
  uint32_t head[64];
  uint32_t count[64];
  uint32_t bits[128];  // run starts over the runs' positions (kMaxPositions)
  uint32_t delta[64];  // per run: first id minus first position
};
constexpr uint32_t kMaxPositions = 4096;  // fragments of a tile's runs, as far as `bits` goes

using LdsWord = __attribute__((address_space(3))) uint32_t;
using LdsEntry = __attribute__((address_space(3))) TileEntry;
using LdsEntryId = __attribute__((address_space(3))) TileEntryId;
__device__ __forceinline__ const LdsEntry& entry_at(uint32_t v) { return *(const LdsEntry*)v; }
__device__ __forceinline__ uint32_t entry_id(uint32_t v) { return ((const LdsEntryId*)v)->id; }
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// Loads from the frame's arrays as global memory: through a pointer that the
// compiler cannot place they would be flat loads, which also wait for LDS.
template <typename T>
__device__ __forceinline__ T ld_global_stream(const T* p) {
  return __builtin_nontemporal_load((const __attribute__((address_space(1))) T*)p);
}
typedef float Float4a __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 ld_global_stream(const float4* p) {
  const Float4a v = __builtin_nontemporal_load((const __attribute__((address_space(1))) Float4a*)p);
  return make_float4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ uint32_t rfl(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Inclusive prefix sum over the wave's lanes, and the largest value, by DPP
// row shifts and broadcasts (lanes without a source add 0).
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, kRows, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v) {
  v += dpp_or_zero<0x111, 0xf>(v);
  v += dpp_or_zero<0x112, 0xf>(v);
  v += dpp_or_zero<0x114, 0xf>(v);
  v += dpp_or_zero<0x118, 0xf>(v);
  v += dpp_or_zero<0x142, 0xa>(v);  // lane 15 to the second row, lane 47 to the fourth
  v += dpp_or_zero<0x143, 0xc>(v);  // lane 31 to the upper half
  return v;
}
__device__ __forceinline__ uint32_t wave_top_u32(uint32_t v) {
  auto top = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
  v = top(v, dpp_or_zero<0x111, 0xf>(v));
  v = top(v, dpp_or_zero<0x112, 0xf>(v));
  v = top(v, dpp_or_zero<0x114, 0xf>(v));
  v = top(v, dpp_or_zero<0x118, 0xf>(v));
  v = top(v, dpp_or_zero<0x142, 0xa>(v));
  v = top(v, dpp_or_zero<0x143, 0xc>(v));
  return __builtin_amdgcn_readlane(v, 63);
}

// ---------------------------------------------------------------------------
// Sorting in registers. A sort key is (depth key << 30) | entry: 62 bits, as
// a double non-negative, finite and in the order of the integer (subnormals
// included: 64-bit subnormals are not flushed), so one compare-exchange is
// v_min_f64 + v_max_f64 where an unsigned 64-bit one is a compare and four
// selects, six where a colour moves along.
// ---------------------------------------------------------------------------

__device__ __forceinline__ double min_raw(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_raw(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double pack2(uint32_t hi, uint32_t lo) { return __hiloint2double((int)hi, (int)lo); }
__device__ __forceinline__ uint32_t hi32(double d) { return (uint32_t)__double2hiint(d); }
__device__ __forceinline__ uint32_t lo32(double d) { return (uint32_t)__double2loint(d); }

// Batcher's merge exchange for any N (inputs past the used ones hold the
// sentinel, so a network of N >= the largest list sorts every lane's).
template <int N>
struct Net {
  int a[N * 8] = {};
  int b[N * 8] = {};
  int n = 0;
  constexpr Net() {
    int t = 0;
    while ((1 << t) < N) ++t;
    for (int p = t > 0 ? 1 << (t - 1) : 0; p > 0; p >>= 1) {
      int q = 1 << (t - 1), r = 0, d = p;
      while (true) {
        for (int i = 0; i + d < N; ++i) {
          if ((i & p) == r) {
            a[n] = i;
            b[n] = i + d;
            ++n;
          }
        }
        if (q == p) break;
        d = q - p;
        q >>= 1;
        r = p;
      }
    }
  }
};

template <int N>
__device__ __forceinline__ void sort_net(double (&v)[N]) {
  if constexpr (N > 1) {
    constexpr Net<N> net;
#pragma unroll
    for (int i = 0; i < net.n; ++i) {
      const double x = v[net.a[i]], y = v[net.b[i]];
      v[net.a[i]] = min_raw(x, y);
      v[net.b[i]] = max_raw(x, y);
    }
  }
}

// The same network on list values, descending.
template <int N>
__device__ __forceinline__ void sort_newest_first(uint32_t (&v)[N]) {
  if constexpr (N > 1) {
    constexpr Net<N> net;
#pragma unroll
    for (int i = 0; i < net.n; ++i) {
      const uint32_t x = v[net.a[i]], y = v[net.b[i]];
      v[net.a[i]] = x > y ? x : y;
      v[net.b[i]] = x > y ? y : x;
    }
  }
}

// Bubbles x into the sorted v; returns the value pushed out. Each step writes
// v[j] in place, so that a loop around it needs no copies of v.
template <int K>
__device__ __forceinline__ double insert_sorted(double (&v)[K], double x) {
#pragma unroll
  for (int j = 0; j < K; ++j) {
    double up;
    asm("v_max_f64 %1, %0, %2\n\tv_min_f64 %0, %0, %2" : "+v"(v[j]), "=&v"(up) : "v"(x));
    x = up;
  }
  return x;
}

// ---------------------------------------------------------------------------
// Fragments by id
// ---------------------------------------------------------------------------

// kMany: the frame may have several segments. A kernel of its own: the
// search's loads would make every fragment load wait for the one before.
template <bool kMany>
__device__ __forceinline__ TileSeg seg_of(const TileSrc& s, uint32_t id) {
  TileSeg r;
  r.target = s.one.target;
  r.depth = s.one.depth;
  r.rgba = s.one.rgba;
  r.id_base = s.one.id_base;
  if constexpr (kMany) {
    if (s.nseg > 1u) {
      const auto* t = (const __attribute__((address_space(1))) TileSeg*)s.segs;
      uint32_t lo = 0, hi = s.nseg;  // last segment whose first id is <= id
      while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (t[mid].id_base <= id) lo = mid;
        else hi = mid;
      }
      r.target = t[lo].target;
      r.depth = t[lo].depth;
      r.rgba = t[lo].rgba;
      r.id_base = t[lo].id_base;
    }
  }
  return r;
}

// Marks where runs start: bit p of w.bits for every run after the first whose
// first position is p + 1, so that a position's run is the number of bits
// below it. clear_marks() first, then each lane's run.
template <typename Lds>
__device__ __forceinline__ void clear_marks(Lds& w) {
  w.bits[lane_id()] = 0u;
  w.bits[lane_id() + 64u] = 0u;
  wave_lds_sync();
}
template <typename Lds>
__device__ __forceinline__ void mark_run(Lds& w, bool on, uint32_t off) {
  if (on && off > 0u) atomicOr(&w.bits[(off - 1u) >> 5], 1u << ((off - 1u) & 31u));
}

// Loads the fragments of some runs into w and links them per target,
// ascending: those of the targets whose index in the tile shifted by `shift`
// is `part`. The runs have `size` positions in all (at most kMaxPositions),
// their starts marked in w.bits and the words at LDS address `deltas` giving
// each one's first id minus first position; id0 is a fragment of theirs.
// `base` is the list index of the tile's first target: fragments of other
// tiles, in a run's gaps, are in no part.
// Returns false (wave-uniform) where the fragments are more than `cap`.
template <bool kMany, typename Lds>
__device__ __forceinline__ bool build_lists(Lds& w, const TileSrc& src, const CodecTables* tab, uint32_t deltas,
                                            uint32_t id0, uint32_t size, uint32_t shift, uint32_t part, uint32_t cap,
                                            uint32_t base, uint32_t target, bool in) {
  constexpr int kU = 3;  // 64-fragment batches in flight together
  const uint32_t lane = lane_id();
  const uint32_t nb = (size + 63u) >> 6;
  const uint32_t end = lds_address(&w.e[0]);
  // the lane's target's opaque depth: fragments behind it are not listed
  const bool opaque = src.opq != nullptr;
  uint32_t front = kEmpty;
  if (opaque && in) front = *((const __attribute__((address_space(1))) uint32_t*)src.opq + 2u * (uint64_t)target + 1u);
  w.head[lane] = end;
  w.count[lane] = 0u;
  if (lane == 0u) {
    w.e[0].key = kEmpty;
    w.e[0].next = end;
    w.e[0].col = 0u;
  }
  wave_lds_sync();
  // lane i: the run starts in positions 64 i .. 64 i + 63, and those below
  const uint32_t lo_bits = w.bits[2u * lane], hi_bits = w.bits[2u * lane + 1u];
  const uint32_t n_starts = (uint32_t)__builtin_popcount(lo_bits) + (uint32_t)__builtin_popcount(hi_bits);
  const uint32_t below = wave_scan_u32(n_starts) - n_starts;
  uint32_t used = 0;  // entries so far
  // the fields of kU batches; the next kU are loaded while these are listed
  struct Fields {
    uint32_t id, loc;
    float4 cv;
    float dv;
    bool act;
  };
  auto load = [&](uint32_t b, Fields (&f)[kU]) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint32_t bb = b + (uint32_t)u;
      const uint32_t pos = bb * 64u + lane;
      const uint32_t k = __builtin_amdgcn_mbcnt_hi(
          __builtin_amdgcn_readlane(hi_bits, bb & 63u),
          __builtin_amdgcn_mbcnt_lo(__builtin_amdgcn_readlane(lo_bits, bb & 63u),
                                    __builtin_amdgcn_readlane(below, bb & 63u)));
      f[u].act = pos < size;
      // lanes past the last fragment read the first one's fields: every lane
      // loads, so no load waits behind a branch
      const uint32_t at = *(const LdsWord*)(deltas + 4u * (f[u].act ? k : 0u)) + pos;
      f[u].id = f[u].act ? at : id0;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const TileSeg s = seg_of<kMany>(src, f[u].id);
      const uint32_t i = f[u].id - s.id_base;
      f[u].loc = ld_global_stream(&s.target[i]);
      f[u].dv = ld_global_stream(&s.depth[i]);
      f[u].cv = ld_global_stream(&s.rgba[i]);
    }
  };
  Fields ahead[kU];
  load(0u, ahead);
  for (uint32_t b = 0; b < nb; b += kU) {
    uint32_t id[kU], loc[kU], key[kU], col[kU];
    bool act[kU];
    float4 cv[kU];
    float dv[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      id[u] = ahead[u].id;
      loc[u] = ahead[u].loc;
      act[u] = ahead[u].act;
      dv[u] = ahead[u].dv;
      cv[u] = ahead[u].cv;
    }
    if (b + kU < nb) load(b + kU, ahead);
    // onto the targets' lists, batch after batch
    uint32_t v[kU], old[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      v[u] = end;
      old[u] = 0u;
      if (b + (uint32_t)u >= nb) {  // wave-uniform: nothing in this batch
        act[u] = false;
        continue;
      }
      loc[u] = pm_index(loc[u], src.T, src.spp) - base;
      key[u] = depth_key(dv[u]);
      col[u] = encode_color_quick(cv[u], tab);
      act[u] = act[u] && (loc[u] >> shift) == part;
      if (opaque) {
        const uint32_t z = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(loc[u] << 2), (int)front);
        act[u] = act[u] && key[u] < z;
      }
      const uint64_t on = __ballot(act[u]);
      v[u] = end + (used + lanes_below(on) + 1u) * Lds::kSize;
      used += (uint32_t)__builtin_popcountll(on);
      if (used > cap) return false;
      if (act[u]) {
        old[u] = atomicMax(&w.head[loc[u]], v[u]);
        atomicAdd(&w.count[loc[u]], 1u);
      }
    }
    bool any = false;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (act[u]) {
        if constexpr (Lds::kHasId) {
          LdsEntryId* const e = (LdsEntryId*)v[u];
          e->key = key[u];
          e->next = old[u];
          e->col = col[u];
          e->id = id[u];
        } else {
          LdsEntry* const e = (LdsEntry*)v[u];
          e->key = key[u];
          e->next = old[u];
          e->col = col[u];
        }
      }
      any = any || old[u] > v[u];
    }
    // lanes of one target in one instruction may meet in any order: one that
    // found a larger value at the head is inserted behind it, one at a time
    if (__ballot(any) != 0ull) {
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        uint64_t m = __ballot(old[u] > v[u]);
        while (m) {
          wave_lds_sync();
          if (lane == (uint32_t)__builtin_ctzll(m)) {
            uint32_t q = w.head[loc[u]];
            uint32_t nx = entry_at(q).next;
            while (nx > v[u]) {
              q = nx;
              nx = entry_at(q).next;
            }
            ((LdsEntry*)v[u])->next = nx;
            ((LdsEntry*)q)->next = v[u];
          }
          m &= m - 1u;
          wave_lds_sync();
        }
      }
    }
  }
  wave_lds_sync();
  return true;
}

// Sort key of an entry: equal depths put the earlier fragment (the lower list
// value) first, for Loop32 the later one (its colour is the one kept).
constexpr uint32_t kLowMask = 0x3FFFFFFFu;
template <int kMode>
__device__ __forceinline__ double sort_key(uint32_t key, uint32_t v) {
  return pack2(key >> 2, (key << 30) | (kMode == kTileLoop32 ? kLowMask - v : v));
}
template <int kMode>
__device__ __forceinline__ uint32_t key_value(double k) {  // the list value in a sort key
  const uint32_t low = lo32(k) & kLowMask;
  return kMode == kTileLoop32 ? kLowMask - low : low;
}
__device__ __forceinline__ uint32_t key_depth(double k) { return (hi32(k) << 2) | (lo32(k) >> 30); }

// The end of a wave's share of a tile, all of it (split 0) or one of 1 <<
// split parts. The last share to end returns the tile's run structures to
// their clear values for the next frame, or, where a share could not be taken
// (`deferred`), queues the tile for the deep composite, which writes all of
// it, counts the tails of those shares and then clears. Queue entry: the
// tile; with shares (at most kSharedTiles tiles) the deferred ones << 16 too.
// `queue` (a batch, where many tiles are queued) collects a wave's entries:
// one atomic on the queue's length for 64 of them. (An atomic each, on one
// address, took as long as the composite.)
struct TileQueue {
  uint32_t n = 0, entry = 0;
  __device__ __forceinline__ void flush(const TileBuf& tb) {
    if (n == 0u) return;
    uint32_t at = 0;
    if (lane_id() == 0u) at = atomicAdd(&tb.ctl[tb.ctl_index], n);
    at = rfl(at);
    if (lane_id() < n) tb.deep[tb.deep_base + at + lane_id()] = entry;
    n = 0u;
  }
  __device__ __forceinline__ void push(const TileBuf& tb, uint32_t e) {
    if (lane_id() == n) entry = e;
    if (++n == 64u) flush(tb);
  }
};

__device__ __forceinline__ void end_share(const TileBuf& tb, uint32_t tile, uint32_t m, uint32_t first, uint32_t split,
                                          bool deferred, TileQueue* queue) {
  uint32_t entry = tile;
  if (split > 0u) {
    entry -= tb.tile_first;
    uint32_t sum = 0;
    if (lane_id() == 0u) {
      const uint32_t mine = 1u + (deferred ? 256u << (first >> (6u - split)) : 0u);
      sum = mine + atomicAdd(&tb.ctl[tb.share0 + entry], mine);
    }
    sum = rfl(sum);
    if ((sum & 255u) != (1u << split)) return;
    if (lane_id() == 0u) tb.ctl[tb.share0 + entry] = 0u;
    deferred = sum > 255u;
    entry |= (sum >> 8) << 16;
  }
  if (deferred) {
    if (queue) queue->push(tb, entry);
    else if (lane_id() == 0u) tb.deep[tb.deep_base + atomicAdd(&tb.ctl[tb.ctl_index], 1u)] = entry;
  } else {
    if (lane_id() == 0u) tb.cnt[tile] = 0u;
    if (m > kTileRuns) tb.more[(uint64_t)tile * kTileRuns + lane_id()] = 0u;
  }
}

// What one wave knows about its tile.
struct TileLane {
  uint32_t tile;
  uint32_t t;     // target
  uint32_t end;   // list value of the end entry
  uint32_t head;  // list value of the newest entry
  uint32_t cnt;   // fragments of the target
  uint32_t most;  // largest cnt of the tile (wave-uniform)
  uint32_t tails; // colour-pass tail fragments
  bool in;        // the target exists
};

// Full colour of a fragment (Loop32's tail, oitLoop.frag.glsl:114-118).
template <bool kMany>
__device__ __forceinline__ float4 full_colour(const TileSrc& src, uint32_t id) {
  const TileSeg s = seg_of<kMany>(src, id);
  const Float4a v = *(const __attribute__((address_space(1))) Float4a*)&s.rgba[id - s.id_base];
  return make_float4(v.x, v.y, v.z, v.w);
}

// Loop64 orders equal depths by packed colour, then id. Where a target has
// some (rare), its values are sorted by (colour, list value) and then again
// by depth, each carrying its place in the first order above its list value.
template <int N>
__device__ __forceinline__ void order_ties(uint32_t end, double (&v)[N]) {
  constexpr uint32_t kBits = 16;  // LDS addresses
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t p = key_value<kTileLoop64>(v[k]);
    v[k] = sort_key<kTileLoop64>(p != end ? (uint32_t)entry_at(p).col : kEmpty, p);
  }
  sort_net<N>(v);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t p = key_value<kTileLoop64>(v[k]);
    v[k] = sort_key<kTileLoop64>(entry_at(p).key, ((uint32_t)k << kBits) | p);
  }
  sort_net<N>(v);
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = pack2(hi32(v[k]), lo32(v[k]) & (0xC0000000u | ((1u << kBits) - 1u)));
}

// Adds the wave's tail fragments to the frame's count.
__device__ __forceinline__ void count_tails(const TileBuf& tb, uint32_t tile, uint32_t tails) {
  const uint32_t sum = __builtin_amdgcn_readlane(wave_scan_u32(tails), 63);
  if (lane_id() == 0u && sum) atomicAdd(&tb.ctl[kTileTails + (tile & (kTileTailWords - 1u))], sum);
}

// Composite of the targets whose fragments are linked in LDS, none of whose targets
// holds more than N fragments, or (kLast) any number: the newest N in
// registers, sorted; older ones bubbled in. Returns false, with nothing
// written, where equal depths need exact_composite.
template <int N, int K, int kMode, bool kTail, bool kGeneral, bool kLast>
__device__ __forceinline__ bool tile_composite(TileLane& L, const TileSrc& src, const TileDst& dst,
                                               const float* s_dec, const float* s_alpha) {
  constexpr int F = N < K ? N : K;  // front values in v
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  const uint32_t end = L.end;
  double v[N];
  uint32_t p = L.head;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const uint32_t key = entry_at(p).key, next = entry_at(p).next;
    v[k] = sort_key<kMode>(key, p);
    p = next;
  }
  sort_net<N>(v);
  float4 under = zero;  // the Linked List's composite tail
  bool deferred = false;
  if constexpr (kLast) {
    if (L.most > (uint32_t)N) {
      double lost = sort_key<kMode>(kEmpty, end);  // the nearest value pushed out
      while (__ballot(p != end) != 0ull) {
        const uint32_t key = entry_at(p).key, next = entry_at(p).next;
        const double x = insert_sorted<N>(v, sort_key<kMode>(key, p));
        p = next;
        // a finished list pushes out the end entry: above every key, and its colour is transparent
        if constexpr (kMode == kTileList && kTail)
          under = over(under, decode_premult_lds(entry_at(key_value<kMode>(x)).col, s_dec, s_alpha));
        if constexpr (kMode == kTileLoop64) lost = min_raw(lost, x);
      }
      // Loop64: equal depths on both sides of the K-th may have to change places
      if constexpr (kMode == kTileLoop64) deferred = L.cnt > (uint32_t)N && key_depth(lost) == key_depth(v[K - 1]);
    }
  }
  if constexpr (kMode == kTileLoop64 || kMode == kTileLoop32) {
    bool tie = false;  // two entries of one depth
#pragma unroll
    for (int k = 1; k < N; ++k) tie = tie || (key_depth(v[k]) == key_depth(v[k - 1]) && key_depth(v[k]) != kEmpty);
    // Loop32 keeps K distinct depths: with more than K fragments a duplicate makes room for another
    deferred = deferred || (tie && L.cnt > (uint32_t)(kMode == kTileLoop32 ? K : N));
    if (__ballot(deferred) != 0ull) return false;
    if constexpr (kMode == kTileLoop64 && N > 1) {
      if (__ballot(tie) != 0ull) {
        // fragments of one colour too (the two sides of a sphere where they
        // meet) stay in id order: nothing to do
        bool mixed = false;
        uint32_t before = entry_at(key_value<kMode>(v[0])).col;
#pragma unroll
        for (int k = 1; k < N; ++k) {
          const uint32_t c = entry_at(key_value<kMode>(v[k])).col;
          mixed = mixed || (key_depth(v[k]) == key_depth(v[k - 1]) && c != before && key_depth(v[k]) != kEmpty);
          before = c;
        }
        if (__ballot(mixed) != 0ull) order_ties<N>(end, v);
      }
    }
  }
  float4 col = zero;
  uint32_t layers = 0;  // Loop32
#pragma unroll
  for (int k = 0; k < F; ++k) {
    const uint32_t e = key_value<kMode>(v[k]);
    const uint32_t c = entry_at(e).col;
    if constexpr (kMode == kTileLoop32) {
      // one layer per depth; the end entry follows the last
      const bool on = e != end && (k == 0 || key_depth(v[k]) != key_depth(v[k > 0 ? k - 1 : 0]));
      if (on) {
        col = over(col, decode_premult_lds(c, s_dec, s_alpha));
        if constexpr (kGeneral) {
          if (dst.fk_key) dst.fk_key[(uint64_t)L.t * K + layers] = key_depth(v[k]);
          if (dst.fk_val) dst.fk_val[(uint64_t)L.t * K + layers] = c;
        }
        ++layers;
      }
    } else {
      col = over(col, decode_premult_lds(c, s_dec, s_alpha));
    }
  }
  float4 d = dst.background;
  if (dst.rgba && L.in) d = dst.rgba[L.t];
  if constexpr (kTail && kMode != kTileList && (N > K || kLast)) {
    // the colour pass's tail: every fragment behind the front K, newest
    // first over the colour buffer (the ROP's primitive order)
    if (L.most > (uint32_t)K) {
      float4 acc = zero;
      uint32_t behind = 0;
      if (N > K && L.most <= (uint32_t)N) {  // all of it in registers: back into id order
        constexpr int E = N > K ? N - K : 1;
        uint32_t q[E];
#pragma unroll
        for (int k = 0; k < E; ++k) q[k] = key_value<kMode>(v[N > K ? K + k : 0]);
        sort_newest_first<E>(q);
#pragma unroll
        for (int k = 0; k < E; ++k) {
          if (__ballot(q[k] != end) != 0ull) {
            if constexpr (kMode == kTileLoop32) {
              if (q[k] != end) {
                acc = over(acc, full_colour<kGeneral>(src, entry_id(q[k])));
                ++behind;
              }
            } else {
              acc = over(acc, decode_premult_lds(entry_at(q[k]).col, s_dec, s_alpha));
              behind += q[k] != end ? 1u : 0u;
            }
          }
        }
      } else if constexpr (kLast) {
        const bool deep = L.cnt > (uint32_t)K;
        const double kth = v[K - 1];
        const uint32_t kth_value = key_value<kMode>(kth), kth_col = entry_at(kth_value).col;
        uint32_t equal = 0;  // Loop64: fragments of the K-th's depth
        uint32_t q = deep ? L.head : end;
        while (__ballot(q != end) != 0ull) {
          if (q != end) {
            const uint32_t key = entry_at(q).key;
            bool tail = key > key_depth(kth);
            if constexpr (kMode == kTileLoop64) {
              if (key == key_depth(kth)) {
                const uint32_t c = entry_at(q).col;
                tail = c > kth_col || (c == kth_col && q > kth_value);
                ++equal;
              }
            }
            if (tail) {
              if constexpr (kMode == kTileLoop32) acc = over(acc, full_colour<kGeneral>(src, entry_id(q)));
              else acc = over(acc, decode_premult_lds(entry_at(q).col, s_dec, s_alpha));
              ++behind;
            }
            q = entry_at(q).next;
          }
        }
        // Loop64: where that depth goes on behind the N, its colours decide
        if constexpr (kMode == kTileLoop64) {
          uint32_t kept = 0;
#pragma unroll
          for (int k = 0; k < K; ++k) kept += key_depth(v[k]) == key_depth(kth) ? 1u : 0u;
          if (__ballot(deep && key_depth(v[N - 1]) == key_depth(kth) && equal > kept) != 0ull) return false;
        }
      }
      d = over(acc, d);
      uint32_t tails = behind;
      if constexpr (kMode == kTileLoop64) {  // those equal to the K-th key (itself at least) are counted too
        if (L.cnt > (uint32_t)K) {
          const uint32_t ck = entry_at(key_value<kMode>(v[F - 1])).col;
#pragma unroll
          for (int k = 0; k < F; ++k)
            if (key_depth(v[k]) == key_depth(v[F - 1]) && entry_at(key_value<kMode>(v[k])).col == ck) ++tails;
        }
      }
      L.tails += tails;
    }
  }
  if (L.in) {
    if constexpr (kMode == kTileList) col = over(col, under);
    dst.out[L.t] = over(col, d);
    if constexpr (kGeneral) {
      const uint32_t n = L.cnt < (uint32_t)K ? L.cnt : (uint32_t)K;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        uint32_t key = kEmpty, val = kEmpty;
        if (k < F && (uint32_t)k < n && kMode != kTileLoop32) {
          const uint32_t e = key_value<kMode>(v[k < F ? k : 0]);
          key = key_depth(v[k < F ? k : 0]);
          val = entry_at(e).col;
        }
        if (kMode != kTileLoop32 || (uint32_t)k >= layers) {
          if (dst.fk_key) dst.fk_key[(uint64_t)L.t * K + k] = key;
          if (dst.fk_val) dst.fk_val[(uint64_t)L.t * K + k] = val;
        }
      }
      if (dst.counts) dst.counts[L.t] = kMode == kTileLoop32 ? layers : n;
    }
  }
  return true;
}

// Composite of the targets linked in LDS by 64-bit integer keys with the
// colours moved along, for the rare tiles where equal depths decide what is
// kept: Loop64 by (depth, colour), Loop32 dropping a depth that it already
// holds (its newest fragment is met first).
template <int K, int kMode, bool kTail, bool kGeneral>
__device__ __forceinline__ void exact_composite(TileLane& L, const TileSrc& src, const TileDst& dst,
                                                const float* s_dec, const float* s_alpha) {
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  const uint32_t end = L.end;
  auto full_key = [&](uint32_t key, uint32_t p) {  // Loop64; a list value orders as the ids do
    return ((uint64_t)key << 32) | (kMode == kTileLoop64 ? (uint32_t)entry_at(p).col : p);
  };
  FrontK<K> f;
  f.init();
  uint32_t held = 0;
  for (uint32_t p = L.head; __ballot(p != end) != 0ull;) {
    const bool on = p != end;
    const uint32_t key = entry_at(p).key, c = entry_at(p).col;
    bool put = on;
    if constexpr (kMode == kTileLoop32) {
#pragma unroll
      for (int k = 0; k < K; ++k) put = put && (f.sk[k] == kEmpty64 || (uint32_t)(f.sk[k] >> 32) != key);
    }
    uint64_t ev;
    uint32_t evc;
    f.insert(put ? full_key(key, p) : kEmpty64, c, ev, evc);
    p = entry_at(p).next;
    held += put ? 1u : 0u;
  }
  const uint32_t n = held < (uint32_t)K ? held : (uint32_t)K;
  const bool deep = held > (uint32_t)K;
  float4 col = zero;
#pragma unroll
  for (int k = 0; k < K; ++k)
    if ((uint32_t)k < n) col = over(col, decode_premult_lds(f.col[k], s_dec, s_alpha));
  float4 d = dst.background;
  if (dst.rgba && L.in) d = dst.rgba[L.t];
  if constexpr (kTail) {
    if (__ballot(deep) != 0ull) {
      const uint64_t kth = f.sk[K - 1];
      float4 acc = zero;
      uint32_t behind = 0, keep = 0;  // keep: fragments equal to Loop64's K-th key that are in the tail, the newest
      for (int pass = 0; pass < 2; ++pass) {
        acc = zero;
        behind = 0;
        uint32_t left = keep;
        for (uint32_t q = deep ? L.head : end; __ballot(q != end) != 0ull;) {
          const uint32_t key = entry_at(q).key;
          const uint64_t x = full_key(key, q);
          bool tail = q != end && (kMode == kTileLoop32 ? key > (uint32_t)(kth >> 32) : x > kth);
          if (kMode == kTileLoop64 && q != end && x == kth && left > 0u) {
            tail = true;
            --left;
          }
          if (tail) {
            if constexpr (kMode == kTileLoop32) acc = over(acc, full_colour<kGeneral>(src, entry_id(q)));
            else acc = over(acc, decode_premult_lds(entry_at(q).col, s_dec, s_alpha));
            ++behind;
          }
          q = entry_at(q).next;
        }
        if constexpr (kMode != kTileLoop64) break;
        if (pass == 1 || __ballot(deep && behind < L.cnt - (uint32_t)K) == 0ull) break;
        keep = deep ? L.cnt - (uint32_t)K - behind : 0u;
      }
      if (deep) d = over(acc, d);
      L.tails += behind;
      if constexpr (kMode == kTileLoop64) {
        if (deep) {
#pragma unroll
          for (int k = 0; k < K; ++k) L.tails += f.sk[k] == kth ? 1u : 0u;
        }
      }
    }
  }
  if (!L.in) return;
  dst.out[L.t] = over(col, d);
  if constexpr (kGeneral) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const bool on = (uint32_t)k < n;
      if (dst.fk_key) dst.fk_key[(uint64_t)L.t * K + k] = on ? (uint32_t)(f.sk[k] >> 32) : kEmpty;
      if (dst.fk_val) dst.fk_val[(uint64_t)L.t * K + k] = on ? f.col[k] : kEmpty;
    }
    if (dst.counts) dst.counts[L.t] = n;
  }
}

// Calls f(first id, word, valid) for up to 64 of the tile's runs at a time,
// every lane of the wave taking part: the slots', and where m is past those
// (or marked kTileUncounted, which is past any) the lists' to their ends.
template <typename F>
__device__ __forceinline__ void each_run(const TileBuf& tb, uint32_t tile, uint32_t m, F&& f) {
  const uint32_t lane = lane_id();
  {
    const bool on = lane < kTileRuns && lane < (m & ~kTileUncounted);
    const uint64_t rec = on ? tb.run[(uint64_t)tile * kTileRuns + lane] : 0ull;
    f((uint32_t)(rec >> 32), (uint32_t)rec, on);
  }
  uint32_t v = m > kTileRuns ? tb.more[(uint64_t)tile * kTileRuns + lane] : 0u;
  while (__ballot(v != 0u) != 0ull) {
    const bool on = v != 0u;
    const uint64_t l = on ? tb.link[v - 1u] : 0ull;
    f(v - 1u, (uint32_t)(l >> 32), on);
    v = on ? (uint32_t)l : 0u;
  }
}

// Sorts run[0 .. got) ascending, got <= 64 R, by one wave: R runs a lane in
// registers, sorted in the lane and then merged over 2, 4 .. 64 lanes, each
// merge by a step against the mirrored lane and halving steps after it
// (Batcher's bitonic merge with all of its exchanges ascending). A run's 48
// bits (first id, own, length) are a double in the integers' order, as the
// sort keys are. Bound by its 21 exchanges between lanes of R values each; in
// LDS, 512 runs took 45 steps of four exchanges, one waiting for the other
// (1920x1080 shuffled, about 400 runs a tile: Loop64 4.30 ms so, 3.10 in
// registers; 256x256: 464 and 272 us). A function of its own: inlined, its
// registers and code cost the composite of the common tiles two per cent
// (1368x978, Loop64 K = 16: 44.5 us, 43.7 so).
template <int R>
__device__ __attribute__((noinline)) void sort_runs(uint64_t* run, uint32_t got) {
  const uint32_t lane = lane_id();
  double v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t i = lane * R + (uint32_t)r;
    const uint64_t x = i < got ? run[i] : 0ull;
    const uint32_t first = (uint32_t)(x >> 32);
    v[r] = i < got ? pack2(first >> 16, first << 16 | (uint32_t)x) : pack2(0x3FFFFFFFu, 0u);
  }
  wave_lds_sync();
  sort_net<R>(v);
  auto swap_with = [&](uint32_t mask, uint32_t bit, bool mirror) {
    const int from = (int)((lane ^ mask) << 2);
    auto other = [&](double x) {
      return pack2((uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)hi32(x)),
                   (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)lo32(x)));
    };
    const bool low = (lane & bit) == 0u;
#pragma unroll
    for (int r = 0; r < R / 2; ++r) {
      const int q = R - 1 - r;
      const double x = other(v[r]), y = other(v[q]);
      const double a = mirror ? y : x, b = mirror ? x : y;
      v[r] = (a < v[r]) == low ? a : v[r];
      v[q] = (b < v[q]) == low ? b : v[q];
    }
  };
#pragma unroll 1
  for (uint32_t w = 2; w <= 64u; w <<= 1) {
    swap_with(w - 1u, w >> 1, true);
#pragma unroll 1
    for (uint32_t h = w >> 2; h > 0u; h >>= 1) swap_with(h, h, false);
#pragma unroll
    for (int j = R / 2; j > 0; j >>= 1) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if ((r & j) == 0) {
          const double x = v[r], y = v[r + j];
          v[r] = min_raw(x, y);
          v[r + j] = max_raw(x, y);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t i = lane * R + (uint32_t)r;
    if (i < got)
      run[i] = ((uint64_t)(hi32(v[r]) << 16 | lo32(v[r]) >> 16) << 32) | (lo32(v[r]) & 0xFFFFu);
  }
  wave_lds_sync();
}

// The runs of the tile whose first id is in [lo, hi), sorted, into run[], and
// how many they are; where that is over kMost, nothing is in order.
template <uint32_t kMost>
__device__ __forceinline__ uint32_t load_runs(uint64_t* run, const TileBuf& tb, uint32_t tile, uint32_t m, uint64_t lo,
                                              uint64_t hi) {
  uint32_t got = 0;  // wave-uniform
  each_run(tb, tile, m, [&](uint32_t start, uint32_t len, bool on) {
    on = on && start >= lo && start < hi;
    const uint64_t mask = __ballot(on);
    const uint32_t at = got + lanes_below(mask);
    if (on && at < kMost) run[at] = ((uint64_t)start << 32) | len;
    got += (uint32_t)__builtin_popcountll(mask);
  });
  wave_lds_sync();
  if (got > kMost) return got;
  if (got <= 256u) sort_runs<4>(run, got);
  else if (kMost <= 512u || got <= 512u) sort_runs<8>(run, got);
  else sort_runs<(int)(kMost / 64u)>(run, got);
  return got;
}

// What a wave loads of a tile ahead of its turn: the run count and the lanes'
// runs.
constexpr uint32_t kAheadRuns = 32;
constexpr uint32_t kManyRuns = 1024;  // runs that a wave sorts
struct TileAhead {
  uint32_t m;
  uint64_t rec;
};
__device__ __forceinline__ TileAhead load_ahead(const TileBuf& tb, uint32_t tile, uint32_t tiles) {
  const uint32_t at = tile < tiles ? tile : tiles - 1u;  // past the last: loaded for nothing
  TileAhead a;
  a.m = *(const __attribute__((address_space(1))) uint32_t*)&tb.cnt[at];
  a.rec = *(const __attribute__((address_space(1))) uint64_t*)&tb.run[(uint64_t)at * kTileRuns +
                                                                      (lane_id() & (kAheadRuns - 1u))];
  return a;
}

// The composite of one tile by one wave (split 0), or of the 64 >> split
// targets from `first` on: see the head of the file.
template <int K, int kMode, bool kTail, bool kGeneral, typename Lds>
__device__ __forceinline__ void tile_wave(uint32_t tile, uint32_t first, uint32_t split, const TileAhead& ahead, const TileBuf& tb, const TileSrc& src,
                                          const TileDst& dst, Lds& w, const float* s_dec, const float* s_alpha,
                                          TileQueue* queue) {
  const uint32_t lane = lane_id();
  const uint32_t base = (tile - dst.tile0) * kTileTargets, a = base + lane;  // list indices in the frame
  const bool in = a < dst.T;
  TileLane L;
  L.tile = tile;
  L.t = in ? pm_target(a, dst.T, dst.spp) : 0u;
  L.end = lds_address(&w.e[0]);
  L.tails = 0u;
  const uint32_t m = rfl(ahead.m);
  const uint32_t last = first + (64u >> split);
  if (m == 0u) {
    if (in && lane >= first && lane < last) {
      float4 d = dst.background;
      if (dst.rgba) d = dst.rgba[L.t];
      dst.out[L.t] = over(make_float4(0.f, 0.f, 0.f, 0.f), d);
      if constexpr (kGeneral) {
        for (int k = 0; k < K; ++k) {
          if (dst.fk_key) dst.fk_key[(uint64_t)L.t * K + k] = kEmpty;
          if (dst.fk_val) dst.fk_val[(uint64_t)L.t * K + k] = kEmpty;
        }
        if (dst.counts) dst.counts[L.t] = 0u;
      }
    }
    return;
  }
  // positions of the runs, and the tile's own fragments among them (or, where
  // those are no more than cap, any number between)
  uint32_t size, frags, id0, deltas = lds_address(w.delta), cap = Lds::kEntries;
  if (__builtin_expect(m <= 64u, 1)) {  // (spills go to the other tiles' code: Loop64 K = 8 150 us, 147 so)
    uint32_t start = kEmpty, len = 0u;
    uint64_t rec = ahead.rec;
    if (m > kAheadRuns && lane >= kAheadRuns && lane < m) rec = tb.run[(uint64_t)tile * kTileRuns + lane];
    if (lane < m) {
      start = (uint32_t)(rec >> 32);
      len = (uint32_t)rec;
    }
    const uint32_t own = run_own(len);
    len = run_len(len);
    if constexpr (kMode == kTileList) {
      if ((__builtin_amdgcn_readlane(wave_scan_u32(len), 63) >> split) > cap &&
          (__builtin_amdgcn_readlane(wave_scan_u32(own), 63) >> split) > cap) {  // binned instead
        end_share(tb, tile, m, first, split, true, queue);
        return;
      }
    }
    // the runs in ascending order of their first ids
    uint32_t rank = 0;
    for (uint32_t j = 0; j < m; ++j) rank += __builtin_amdgcn_readlane(start, j) < start ? 1u : 0u;
    const int to = (int)((lane < m ? rank : lane) << 2);
    start = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)start);
    len = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)len);
    const uint32_t incl = wave_scan_u32(len);
    size = frags = __builtin_amdgcn_readlane(incl, 63);
    if (size > cap) frags = __builtin_amdgcn_readlane(wave_scan_u32(own), 63);  // (where it decides)
    id0 = rfl(start);
    clear_marks(w);
    if (size <= kMaxPositions) mark_run(w, lane < m, incl - len);  // 64 runs of at most 64: always
    w.delta[lane] = start - (incl - len);
  } else if constexpr (kMode == kTileList) {
    end_share(tb, tile, m, first, split, true, queue);
    return;
  } else {
    // many runs: gathered and sorted in the entries' space, of which their
    // deltas then take the end, 4 bytes a run
    if (m > kManyRuns && !(m & kTileUncounted)) {
      end_share(tb, tile, m, first, split, true, queue);
      return;
    }
    uint64_t* const run = reinterpret_cast<uint64_t*>(&w.e[0]);
    const uint32_t got = load_runs<kManyRuns>(run, tb, tile, m, 0u, 1ull << 32);
    if (got > kManyRuns) {
      end_share(tb, tile, m, first, split, true, queue);
      return;
    }
    cap = Lds::kEntries - (got * (uint32_t)sizeof(uint32_t) + Lds::kSize - 1u) / Lds::kSize;
    uint32_t* const delta = reinterpret_cast<uint32_t*>(&w.e[cap + 1u]);
    deltas = lds_address(delta);
    id0 = rfl((uint32_t)(run[0] >> 32));
    size = frags = 0;
#pragma unroll 1
    for (uint32_t c = 0; c < got; c += 64u) {
      const uint32_t word = c + lane < got ? (uint32_t)run[c + lane] : 0u;
      size += __builtin_amdgcn_readlane(wave_scan_u32(run_len(word)), 63);
      frags += __builtin_amdgcn_readlane(wave_scan_u32(run_own(word)), 63);
    }
    // Many passes over all of these runs are slower than the deep composite's
    // groups, each fragment once for the front K and once for the tail
    // (512x512, 2000 spheres, three in ten clustered, a tile for two waves:
    // Loop64 K = 8 1.60 ms with up to 4096 positions here, 1.03 with up to four
    // times what the LDS holds, 0.92 with three times; Loop32 2.10, 1.02 at
    // four; 1920x1080 in blocks of 8x8 pixels, a tile for a wave: Loop32 0.31
    // at three times, 0.37 at two). Where four or eight waves share a tile
    // there are few tiles, and one wave's groups are the longer way (181x89,
    // 718 spheres: Loop64 K = 8 61 us so, 118 with groups).
    const uint32_t most = split + (kMode == kTileLoop32 ? 3u : 2u);
    if (size > kMaxPositions || (split < 2u && frags > most * cap)) {
      end_share(tb, tile, m, first, split, true, queue);
      return;
    }
    clear_marks(w);
    // from the last runs down: the deltas lie over the last ones. They take 4
    // bytes a run at the end of a space for 8, so that a delta is behind every
    // run of the batches before its own
    static_assert(Lds::kEntries * Lds::kSize >= kManyRuns * sizeof(uint64_t), "the runs fit the entries' space");
    uint32_t at_end = size;
#pragma unroll 1
    for (uint32_t c = (got - 1u) & ~63u;; c -= 64u) {
      const bool on = c + lane < got;
      const uint64_t rec = on ? run[c + lane] : 0ull;
      const uint32_t len = run_len((uint32_t)rec), incl = wave_scan_u32(len);
      at_end -= __builtin_amdgcn_readlane(incl, 63);
      const uint32_t off = at_end + incl - len;
      mark_run(w, on, off);
      if (on) delta[c + lane] = (uint32_t)(rec >> 32) - off;
      if (c == 0u) break;
    }
  }
  wave_lds_sync();
  // more fragments than the LDS holds: 1 << shift of the tile's targets at a
  // time, each part reading all of the runs and keeping its own fragments; a
  // part that is still too large is halved
  uint32_t shift = 6u - split;
  if constexpr (kMode != kTileList) {
    while (shift > 0u && (frags >> (6u - shift)) > cap) --shift;
  }
  for (uint32_t t0 = first; t0 < last;) {
    const uint32_t part = t0 >> shift;
    if (!build_lists<kGeneral>(w, src, dst.tab, deltas, id0, size, shift, part, cap, base, L.t, in)) {
      wave_lds_sync();
      if (shift == 0u || kMode == kTileList) {  // one target's fragments
        end_share(tb, tile, m, first, split, true, queue);
        return;
      }
      --shift;
      continue;
    }
    t0 += 1u << shift;
    L.in = in && (lane >> shift) == part;
    L.head = w.head[lane];
    L.cnt = w.count[lane];
    L.most = wave_top_u32(L.cnt);
    // sizes of the sorted part; with a tail in id order, K + 8 values hold
    // nearly every tile's tails too
    constexpr int R = (kTail && kMode != kTileList && K <= 16) ? K + 8 : K;
    bool done;
#define OIT_TILE_SIZE(n) \
  tile_composite<(n < R ? n : R), K, kMode, kTail, kGeneral, (n >= R)>(L, src, dst, s_dec, s_alpha)
    if (L.most <= 4u || R <= 4) done = OIT_TILE_SIZE(4);
    else if (L.most <= 8u || R <= 8) done = OIT_TILE_SIZE(8);
    else if (L.most <= 12u || R <= 12) done = OIT_TILE_SIZE(12);
    else if (L.most <= 16u || R <= 16) done = OIT_TILE_SIZE(16);
    else if (kMode == kTileLoop64 && R > 20 && L.most <= 20u) done = OIT_TILE_SIZE(20);  // (24 spill)
    else if (L.most <= 24u || R <= 24) done = OIT_TILE_SIZE(24);
    else done = OIT_TILE_SIZE(32);
#undef OIT_TILE_SIZE
    if constexpr (kMode == kTileLoop64 || kMode == kTileLoop32) {
      if (__builtin_expect(!done, 0)) exact_composite<K, kMode, kTail, kGeneral>(L, src, dst, s_dec, s_alpha);
    }
    wave_lds_sync();
  }
  if constexpr (kTail && kMode != kTileList) {
    if (__ballot(L.tails != 0u) != 0ull) count_tails(tb, tile, L.tails);
  }
  end_share(tb, tile, m, first, split, false, queue);
}

// ---------------------------------------------------------------------------
// Deep tiles: more runs or fragments than the one-group composite takes
// ---------------------------------------------------------------------------

constexpr uint32_t kDeepRuns = 1024;  // runs sorted in LDS at once
constexpr int kDeepEntries = 512;     // fragments of a group

template <int K>
struct DeepLds {
  TileLds<kDeepEntries, true> g;
  uint32_t carry[K * 64];   // the front K's colours between groups, [k][lane]
  uint64_t run[kDeepRuns];  // first id << 32 | length, ascending
  uint32_t delta[kDeepEntries];  // per run of a group
};

// Calls body(last) for the tile's fragments group by group, the newest
// first: w.g holds the group's entries (ascending) and the targets' lists.
// `keep`: the tile has one group and its lists are still in w.g.
template <typename Lds, typename F>
__device__ __forceinline__ uint32_t each_group(Lds& w, const TileBuf& tb, const TileSrc& src, const TileDst& dst,
                                               uint32_t tile, uint32_t m, bool keep, F&& body) {
  const uint32_t list_index = (tile - dst.tile0) * kTileTargets + lane_id();
  const bool in = list_index < dst.T;
  const uint32_t t = in ? pm_target(list_index, dst.T, dst.spp) : 0u;
  const uint32_t lane = lane_id();
  if (keep) {
    body(true);
    return 1u;
  }
  uint32_t groups = 0;
  const uint64_t begin = src.one.id_base;
  uint64_t hi = begin + src.frags;
  while (hi > begin) {
    uint64_t lo = begin;
    if (m > kTileRuns) {  // (the lists may hold uncounted runs)
      // a window of at most kDeepRuns runs below hi: first ids differ, so a
      // span of kDeepRuns ids is one; from there to a fuller one, every other
      // step to where an even spread would have three quarters of kDeepRuns
      // (halving alone walked the lists up to thirty times for each window:
      // 1920x1080 shuffled, 21.7 M fragments, Loop64 6.59 ms, 5.44 so)
      auto count = [&](uint64_t from) {
        uint32_t c = 0;
        each_run(tb, tile, m, [&](uint32_t start, uint32_t, bool on) {
          c += (uint32_t)__builtin_popcountll(__ballot(on && start >= from && start < hi));
        });
        return c;
      };
      uint64_t bad = begin;
      uint32_t c_bad = count(bad);
      if (c_bad > kDeepRuns) {
        uint64_t ok = hi - kDeepRuns;  // > bad: more runs than that are between bad and hi
        uint32_t c_ok = 0;
        for (bool spread = true; ok - bad > 1u && c_ok < kDeepRuns / 2u; spread = !spread) {
          uint64_t mid = bad + (ok - bad) / 2u;
          if (spread) {
            const uint64_t at = hi - (hi - bad) * (kDeepRuns / 4u * 3u) / c_bad;
            if (at > bad && at < ok) mid = at;
          }
          const uint32_t c = count(mid);
          if (c > kDeepRuns) {
            bad = mid;
            c_bad = c;
          } else {
            ok = mid;
            c_ok = c;
          }
        }
        lo = ok;
      }
    }
    uint32_t e = load_runs<kDeepRuns>(w.run, tb, tile, m, lo, hi);
    while (e > 0u) {
      // as many of the newest runs as one group holds
      uint32_t r = 0, N = 0;
      while (r < e) {
        const uint32_t left = e - r, len = lane < left ? run_len((uint32_t)w.run[left - 1u - lane]) : 0u;
        const uint32_t sum = N + wave_scan_u32(len);
        const uint32_t k = (uint32_t)__builtin_popcountll(__ballot(lane < left && sum <= (uint32_t)kDeepEntries));
        if (k > 0u) N = __builtin_amdgcn_readlane(sum, k - 1u);
        r += k;
        if (k < 64u) break;
      }
      if (r == 0u) break;  // no run is longer than a group
      const uint32_t first = e - r;
      clear_marks(w.g);
      for (uint32_t c = 0, off = 0; c < r; c += 64u) {
        const bool on = c + lane < r;
        const uint64_t rec = on ? w.run[first + c + lane] : 0ull;
        const uint32_t len = run_len((uint32_t)rec), incl = wave_scan_u32(len), at = off + incl - len;
        mark_run(w.g, on, at);
        if (on) w.delta[c + lane] = (uint32_t)(rec >> 32) - at;
        off += __builtin_amdgcn_readlane(incl, 63);
      }
      const uint32_t id0 = rfl((uint32_t)(w.run[first] >> 32));
      wave_lds_sync();
      (void)build_lists<true>(w.g, src, dst.tab, lds_address(w.delta), id0, N, 6u, 0u, kDeepEntries,
                                         (tile - dst.tile0) * kTileTargets, t, in);
      body(first == 0u && lo == begin);
      ++groups;
      wave_lds_sync();
      e = first;
    }
    hi = lo;
  }
  return groups;
}

// What the deep composites write for a target.
template <int K, int kMode>
struct DeepOut {
  float4 col, under, tail;  // front K, the list composite's tail, the colour pass's tail
  bool deep;                // has a colour-pass tail
  uint32_t tails, n, cnt;
};

// Composite with the front K as sorted doubles. An entry's list value orders
// equal depths within a group; between groups the kept entries' colours move
// to `carry` and their list values past every entry's (they are newer than
// all that follows, so they come after at equal depths; first, in Loop32's
// order). Returns false where equal depths at the K-th need exact_deep.
template <int K, int kMode, bool kTail>
__device__ __forceinline__ bool sorted_deep(uint32_t tile, uint32_t m, const TileBuf& tb, const TileSrc& src,
                                            const TileDst& dst, DeepLds<K>& w, const float* s_dec,
                                            const float* s_alpha, DeepOut<K, kMode>& o) {
  constexpr uint32_t kCarry = 1u << 20;  // list values of carried entries: past every LDS address
  const uint32_t end = lds_address(&w.g.e[0]);
  const uint32_t lane = lane_id();
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  auto colour_of = [&](double x) {
    const uint32_t p = key_value<kMode>(x);
    if (p >= kCarry) return w.carry[(p - kCarry) * 64u + lane];
    return (uint32_t)entry_at(p).col;
  };
  double v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = sort_key<kMode>(kEmpty, end);
  double lost = sort_key<kMode>(kEmpty, end);
  uint32_t cnt = 0;
  o.under = zero;
  const uint32_t groups = each_group(w, tb, src, dst, tile, m, false, [&](bool last) {
    uint32_t p = w.g.head[lane];
    cnt += w.g.count[lane];
    while (__ballot(p != end) != 0ull) {
      const double x = sort_key<kMode>(entry_at(p).key, p);
      p = entry_at(p).next;
      double ev = x;
      if (__ballot(x < v[K - 1]) != 0ull) ev = insert_sorted<K>(v, x);
      // a value pushed out is an entry once the target has K (the end entry's colour is transparent)
      if constexpr (kMode == kTileList) {
        if constexpr (kTail) o.under = over(o.under, decode_premult_lds(colour_of(ev), s_dec, s_alpha));
      } else {
        lost = min_raw(lost, ev);
      }
    }
    if (!last) {
      uint32_t c[K];
#pragma unroll
      for (int k = 0; k < K; ++k) c[k] = colour_of(v[k]);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const uint32_t at = (uint32_t)(kMode == kTileLoop32 ? K - 1 - k : k);
        w.carry[at * 64u + lane] = c[k];
        if (key_value<kMode>(v[k]) != end) v[k] = sort_key<kMode>(key_depth(v[k]), kCarry + at);
      }
    }
  });
  o.cnt = cnt;
  o.n = cnt < (uint32_t)K ? cnt : (uint32_t)K;
  o.deep = cnt > (uint32_t)K;
  if constexpr (kMode != kTileList) {
    bool tie = o.deep && key_depth(lost) == key_depth(v[K - 1]);
#pragma unroll
    for (int k = 1; k < K; ++k) tie = tie || (key_depth(v[k]) == key_depth(v[k - 1]) && key_depth(v[k]) != kEmpty);
    if (__ballot(tie) != 0ull) return false;
  }
  o.col = zero;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t c = colour_of(v[k]);
    o.col = over(o.col, decode_premult_lds(c, s_dec, s_alpha));
  }
  o.tails = 0;
  o.tail = zero;
  if constexpr (kTail && kMode != kTileList) {
    if (__ballot(o.deep) != 0ull) {
      const uint32_t kth = key_depth(v[K - 1]);  // no tail entry has its depth
      float4 acc = zero;
      uint32_t behind = 0;
      (void)each_group(w, tb, src, dst, tile, m, groups == 1u, [&](bool) {
        uint32_t q = o.deep ? w.g.head[lane] : end;
        while (__ballot(q != end) != 0ull) {
          if (q != end) {
            if (entry_at(q).key > kth) {
              if constexpr (kMode == kTileLoop32) acc = over(acc, full_colour<true>(src, entry_id(q)));
              else acc = over(acc, decode_premult_lds(entry_at(q).col, s_dec, s_alpha));
              ++behind;
            }
            q = entry_at(q).next;
          }
        }
      });
      o.tail = acc;
      o.tails = behind + ((kMode == kTileLoop64 && o.deep) ? 1u : 0u);  // Loop64 counts the K-th key's own too
    }
  }
  return true;
}

// The same for Loop64 and Loop32 by 64-bit integer keys with the colours moved
// along: Loop64 by (depth, colour), Loop32 by (depth, id) and dropping a depth
// that it already holds (its newest fragment is met first).
template <int K, int kMode, bool kTail>
__device__ __forceinline__ void exact_deep(uint32_t tile, uint32_t m, uint32_t t, bool in, const TileBuf& tb,
                                           const TileSrc& src, const TileDst& dst, DeepLds<K>& w, const float* s_dec,
                                           const float* s_alpha, DeepOut<K, kMode>& o) {
  const uint32_t lane = lane_id();
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  auto full_key = [&](uint32_t key, uint32_t p) {
    return ((uint64_t)key << 32) | (kMode == kTileLoop64 ? (uint32_t)entry_at(p).col : entry_id(p));
  };
  const uint32_t end = lds_address(&w.g.e[0]);
  FrontK<K> f;
  f.init();
  uint32_t cnt = 0, held = 0;
  const uint32_t groups = each_group(w, tb, src, dst, tile, m, false, [&](bool) {
    uint32_t p = w.g.head[lane];
    cnt += w.g.count[lane];
    while (__ballot(p != end) != 0ull) {
      const bool on = p != end;
      const uint32_t key = entry_at(p).key, c = entry_at(p).col;
      uint64_t x = on ? full_key(key, p) : kEmpty64;
      bool put = on;
      if constexpr (kMode == kTileLoop32) {
#pragma unroll
        for (int k = 0; k < K; ++k) put = put && (f.sk[k] == kEmpty64 || (uint32_t)(f.sk[k] >> 32) != key);
      }
      if (!put) x = kEmpty64;
      p = entry_at(p).next;
      uint64_t ev = x;
      uint32_t evc = c;
      f.insert(x, c, ev, evc);
      held += put ? 1u : 0u;
    }
  });
  o.cnt = cnt;
  o.n = held < (uint32_t)K ? held : (uint32_t)K;
  o.deep = held > (uint32_t)K;
  o.col = zero;
#pragma unroll
  for (int k = 0; k < K; ++k)
    if ((uint32_t)k < o.n) o.col = over(o.col, decode_premult_lds(f.col[k], s_dec, s_alpha));
  o.tail = zero;
  o.tails = 0;
  if constexpr (kTail) {
    if (__ballot(o.deep) != 0ull) {
      const uint64_t kth = f.sk[K - 1];
      float4 acc = zero;
      uint32_t behind = 0, keep = 0;  // keep: fragments equal to Loop64's K-th key that are in the tail, the newest
      for (int pass = 0; pass < 2; ++pass) {
        acc = zero;
        behind = 0;
        uint32_t left = keep;
        (void)each_group(w, tb, src, dst, tile, m, groups == 1u, [&](bool) {
          uint32_t q = o.deep ? w.g.head[lane] : end;
          while (__ballot(q != end) != 0ull) {
            if (q != end) {
              const uint32_t key = entry_at(q).key;
              const uint64_t x = full_key(key, q);
              bool tail = kMode == kTileLoop32 ? key > (uint32_t)(kth >> 32) : x > kth;
              if (kMode == kTileLoop64 && x == kth && left > 0u) {
                tail = true;
                --left;
              }
              if (tail) {
                if constexpr (kMode == kTileLoop32) acc = over(acc, full_colour<true>(src, entry_id(q)));
                else acc = over(acc, decode_premult_lds(entry_at(q).col, s_dec, s_alpha));
                ++behind;
              }
              q = entry_at(q).next;
            }
          }
        });
        if constexpr (kMode != kTileLoop64) break;
        if (pass == 1 || __ballot(o.deep && behind < cnt - (uint32_t)K) == 0ull) break;
        keep = o.deep ? cnt - (uint32_t)K - behind : 0u;
      }
      o.tail = acc;
      o.tails = behind;
      if constexpr (kMode == kTileLoop64) {
        if (o.deep) {
#pragma unroll
          for (int k = 0; k < K; ++k) o.tails += f.sk[k] == kth ? 1u : 0u;
        }
      }
    }
  }
  if (in && (dst.fk_key || dst.fk_val)) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const bool on = (uint32_t)k < o.n;
      if (dst.fk_key) dst.fk_key[(uint64_t)t * K + k] = on ? (uint32_t)(f.sk[k] >> 32) : kEmpty;
      if (dst.fk_val)
        dst.fk_val[(uint64_t)t * K + k] = on ? f.col[k] : kEmpty;
    }
  }
}

template <int K, int kMode, bool kTail>
__device__ __forceinline__ void deep_wave(uint32_t tile, uint32_t shares, uint32_t split, const TileBuf& tb, const TileSrc& src, const TileDst& dst,
                                          DeepLds<K>& w, const float* s_dec, const float* s_alpha) {
  const uint32_t lane = lane_id();
  const uint32_t a = (tile - dst.tile0) * kTileTargets + lane;
  const bool in = a < dst.T;
  const uint32_t t = in ? pm_target(a, dst.T, dst.spp) : 0u;
  const uint32_t m = rfl(tb.cnt[tile]);
  DeepOut<K, kMode> o;
  if constexpr (kMode == kTileList) {
    (void)sorted_deep<K, kMode, kTail>(tile, m, tb, src, dst, w, s_dec, s_alpha, o);
  } else {
    // the debug outputs, too, are the integer form's
    bool done = false;
    if (!(dst.fk_key || dst.fk_val)) done = sorted_deep<K, kMode, kTail>(tile, m, tb, src, dst, w, s_dec, s_alpha, o);
    if (!done) exact_deep<K, kMode, kTail>(tile, m, t, in, tb, src, dst, w, s_dec, s_alpha, o);
  }
  float4 d = dst.background;
  if (dst.rgba && in) d = dst.rgba[t];
  if constexpr (kTail && kMode != kTileList) {
    if (o.deep) d = over(o.tail, d);
    count_tails(tb, tile, (shares >> (lane >> (6u - split))) & 1u ? o.tails : 0u);
  }
  if (lane == 0u) tb.cnt[tile] = 0u;
  if (m > kTileRuns) tb.more[(uint64_t)tile * kTileRuns + lane] = 0u;
  if (!in) return;
  if constexpr (kMode == kTileList) o.col = over(o.col, o.under);
  dst.out[t] = over(o.col, d);
  if (dst.counts) dst.counts[t] = o.n;
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

constexpr uint32_t kComputeUnits = 256;

// Fragments that a wave's LDS holds, and the waves per SIMD that the launch
// bound asks for.
// (12 or 16 bytes each: about the same LDS.)
constexpr int tile_entries(bool id) { return id ? 520 : 696; }
template <bool kId>
constexpr bool tile_lds_ok() {
  using Lds = TileLds<tile_entries(kId), kId>;
  // four blocks of four waves, with the decode tables, in a compute unit's 160 KB
  return alignof(Lds) % alignof(uint64_t) == 0 && offsetof(Lds, e) == 0 &&
         4u * (4u * sizeof(Lds) + 2048u) <= 160u * 1024u;
}
static_assert(tile_lds_ok<false>() && tile_lds_ok<true>(), "alignment and size of a wave's LDS");
template <int K>
constexpr int tile_waves() { return K >= 32 ? 3 : 4; }

// Draws a ticket (one lane). The address is hidden: for a wave-uniform one the
// compiler combines the wave's lanes and waits for the result at once.
__device__ __forceinline__ uint32_t draw_ticket(const TileBuf& tb, uint32_t counter) {
  uint32_t at = counter;
  asm volatile("" : "+v"(at));
  return atomicAdd(&tb.ctl[at], 1u);
}

// The composites' arguments. They are read from the kernel arguments where
// they are used: `fresh_args` hides the address from the compiler once per
// tile, or it would keep all of them (some 90 scalar registers) in registers
// across the tiles and spill.
struct TileArgs {
  TileBuf tb;
  TileSrc src;
  TileDst dst;
  uint32_t tiles;
  uint32_t split;  // 1 << split waves share a tile
};
using ArgsPtr = const __attribute__((address_space(4))) TileArgs*;
__device__ __forceinline__ const TileArgs& fresh_args() {
  auto p = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const TileArgs*)p;
}

template <int K, int kMode, bool kTail, bool kGeneral>
__global__ __launch_bounds__(kBlock, tile_waves<K>()) void k_tile_resolve(TileArgs args) {
  constexpr bool kId = kGeneral || kMode == kTileLoop32;
  __shared__ float s_dec[256];
  __shared__ float s_alpha[256];
  __shared__ TileLds<tile_entries(kId), kId> s_w[kBlock / 64];
  stage_decode(s_dec, s_alpha, args.dst.tab);
  __syncthreads();
  // resident waves that step through the tiles: a block's LDS is not held by
  // its slowest wave, and the tables are staged once
  const uint32_t wave = rfl(threadIdx.x >> 6);
  const uint32_t stride = gridDim.x * (kBlock / 64);
  const uint32_t tiles = args.tiles, split = args.split, items = tiles << split;
  uint32_t item = blockIdx.x * (kBlock / 64) + wave;
  if (item >= items) return;
  TileAhead now = load_ahead(args.tb, item >> split, tiles);
  for (; item < items; item += stride) {
    const TileArgs& g = fresh_args();
    const TileAhead next = load_ahead(g.tb, (item + stride) >> split, tiles);
    const uint32_t first = (item & ((1u << split) - 1u)) << (6u - split);
    tile_wave<K, kMode, kTail, kGeneral>(item >> split, first, split, now, g.tb, g.src, g.dst, s_w[wave],
                                                  s_dec, s_alpha, nullptr);
    now = next;
  }
}

template <int K, int kMode, bool kTail>
__global__ __launch_bounds__(64) void k_tile_deep(TileArgs args) {
  const uint32_t n = rfl(ld_relaxed(&args.tb.ctl[args.tb.ctl_index]));
  if (blockIdx.x >= n) return;
  __shared__ float s_dec[256];
  __shared__ float s_alpha[256];
  __shared__ DeepLds<K> w;
  for (uint32_t k = threadIdx.x; k < 256u; k += 64u) {
    s_dec[k] = args.dst.tab->dec[k];
    s_alpha[k] = args.dst.tab->alpha[k];
  }
  __syncthreads();
  for (;;) {  // tickets: deep tiles differ much in depth
    const TileArgs& g = fresh_args();
    uint32_t q = 0;
    if (threadIdx.x == 0) q = atomicAdd(&g.tb.ctl[g.tb.ctl_index + 1u], 1u);
    q = rfl(q);
    if (q >= n) break;
    const uint32_t entry = rfl(g.tb.deep[g.tb.deep_base + q]);
    const uint32_t tile = g.split ? g.tb.tile_first + (entry & 0xFFFFu) : entry;
    const uint32_t shares = g.split ? entry >> 16 : 1u;
    deep_wave<K, kMode, kTail>(tile, shares, g.split, g.tb, g.src, g.dst, w, s_dec, s_alpha);
    wave_lds_sync();
  }
}

// A batch's queued tiles of more runs are left to the deep composite, a wave
// each: a clustered 512x512 frame has tiles of 1100 to 1400 (nine frames, 16 M
// fragments: 1.80 ms with 1024, 1.16 with 2048, 1.55 with lists).
constexpr uint32_t kBinRuns = 2048;

// A batch group's frames: the same composite, each tile with its frame's
// arrays and size.
struct TileBatchArgs {
  TileBuf tb;
  const BatchFrameDev* frames;
  uint32_t f0, f1;
  uint32_t tile0, tiles, split;
  const CodecTables* tab;
};
using BatchArgsPtr = const __attribute__((address_space(4))) TileBatchArgs*;
__device__ __forceinline__ const TileBatchArgs& fresh_batch_args() {
  auto p = (BatchArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const TileBatchArgs*)p;
}
using FramePtr = const __attribute__((address_space(4))) BatchFrameDev*;
// The frame of a tile, from the frame of an earlier one on.
__device__ __forceinline__ uint32_t next_frame(FramePtr fr, uint32_t f, uint32_t f1, uint32_t tile) {
  while (f + 1u < f1 && fr[f + 1u].target_base <= (uint64_t)tile * kTileTargets) ++f;
  return f;
}
__device__ __forceinline__ void frame_views(FramePtr fr, uint32_t f, const CodecTables* tab, TileSrc& src,
                                            TileDst& dst) {
  src.one.target = fr[f].target;
  src.one.depth = fr[f].depth;
  src.one.rgba = fr[f].rgba;
  src.one.id_base = fr[f].frag_base;
  src.frags = fr[f].count;
  src.T = dst.T = fr[f].T;
  dst.tile0 = fr[f].target_base / kTileTargets;
  dst.out = fr[f].out;
  dst.background = make_float4(fr[f].background.x, fr[f].background.y, fr[f].background.z, fr[f].background.w);
  dst.tab = tab;
}

template <int K, bool kTail>
__global__ __launch_bounds__(kBlock, tile_waves<K>()) void k_tile_batch(TileBatchArgs args) {
  __shared__ float s_dec[256];
  __shared__ float s_alpha[256];
  __shared__ TileLds<tile_entries(false), false> s_w[kBlock / 64];
  stage_decode(s_dec, s_alpha, args.tab);
  __syncthreads();
  const uint32_t wave = rfl(threadIdx.x >> 6);
  const uint32_t stride = gridDim.x * (kBlock / 64);
  const uint32_t end = args.tile0 + args.tiles, split = args.split;
  uint32_t item = (args.tile0 << split) + blockIdx.x * (kBlock / 64) + wave;
  const uint32_t items = end << split;
  if (item >= items) return;
  TileAhead now = load_ahead(args.tb, item >> split, end);
  uint32_t f = args.f0;
  TileQueue queue;
  for (; item < items; item += stride) {
    const TileBatchArgs& g = fresh_batch_args();
    const TileAhead next = load_ahead(g.tb, (item + stride) >> split, end);
    const auto fr = (FramePtr)g.frames;
    f = rfl(next_frame(fr, f, g.f1, item >> split));
    TileSrc src;
    TileDst dst;
    frame_views(fr, f, g.tab, src, dst);
    const uint32_t first = (item & ((1u << split) - 1u)) << (6u - split);
    tile_wave<K, kTileList, kTail, false>(item >> split, first, split, now, g.tb, src, dst, s_w[wave], s_dec,
                                                 s_alpha, &queue);
    now = next;
  }
  queue.flush(args.tb);
}

// Sorted register array of K packed keys for a list walk (newest element
// first), with the colours in an LDS column per lane: key = (depth key << 30)
// | order << 6 | slot, where order falls with every element walked, so that
// equal depths put the smaller id first, and slot is the element's place in
// the lane's column of K + 1. An insert writes its colour to the free slot
// and bubbles the key in; the slot of the key pushed out is the next free
// one.
template <int K>
struct FrontS {
  double v[K];
  uint32_t free;  // the lane's free slot
  uint32_t* col;  // the lane's column, slots kBlock words apart
  __device__ __forceinline__ void init(uint32_t* column) {
    uint32_t high = 0x3FFFFFFFu, low = 0xFFFFFFC0u;
    asm volatile("" : "+v"(high), "+v"(low));  // or the sentinels are kept in registers across the tiles
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = pack2(high, low + (uint32_t)(k + 1));
    free = 0u;
    col = column;
  }
  // `step` is the element's place in the walk (below 2^24).
  static __device__ __forceinline__ double key_of(uint64_t cd, uint32_t step, uint32_t slot) {
    const uint32_t key = (uint32_t)(cd >> 32);
    return pack2(key >> 2, (key << 30) | ((0xFFFFFFu - step) << 6) | slot);
  }
  // Returns the colour pushed out; a lane that is not `on` puts in a sentinel.
  // The first step + 1 places can be occupied; those behind hold sentinels,
  // one of which is pushed out (step is wave-uniform).
  __device__ __forceinline__ uint32_t insert(uint64_t cd, uint32_t step, bool on) {
    const double key = key_of(cd, step, free);
    double x = pack2(on ? hi32(key) : 0x3FFFFFFFu, on ? lo32(key) : 0xFFFFFFC0u | free);
    col[free * kBlock] = (uint32_t)cd;
#pragma unroll
    for (int b = 0; b < K; b += 4) {
      if ((uint32_t)b <= step) {
#pragma unroll
        for (int j = b; j < b + 4 && j < K; ++j) {
          double up;
          asm("v_max_f64 %1, %0, %2\n\tv_min_f64 %0, %0, %2" : "+v"(v[j]), "=&v"(up) : "v"(x));
          x = up;
        }
      }
    }
    free = lo32(x) & 63u;
    return col[free * kBlock];
  }
  __device__ __forceinline__ uint32_t colour(int k) const { return col[(lo32(v[k]) & 63u) * kBlock]; }
};

// A binned target: its first place behind the tile's base and, in the high
// bit, whether its entries lie 16 apart (a row of 16 targets) or follow each
// other.
constexpr uint32_t kBinRow = 1u << 31;
__device__ __forceinline__ uint32_t bin_step(uint32_t at) { return at & kBinRow ? 16u : 1u; }
__device__ __forceinline__ uint32_t bin_at(uint32_t at) { return at & ~kBinRow; }

// The binned tiles' composite (k_tile_bin has put their fragments in order):
// a wave per tile, a lane per target, each its bucket from the newest on.
// Bound by the latency of one lane's list; four entries are loaded ahead, and
// a trip of four that are behind the K in every lane only blends them (the
// 24-frame mix's K = 8 frames, clusters of up to 560 layers: 570 us one by one, 412 so).
template <int K, bool kTail>
__global__ __launch_bounds__(kBlock, K <= 8 ? 8 : (K <= 16 ? 6 : 4)) void k_tile_binned(TileBatchArgs args) {
  const uint32_t n_tiles = rfl(ld_relaxed(&args.tb.ctl[args.tb.ctl_index]));
  if (blockIdx.x / kTicketLanes * (kBlock / 64) * kTicketLanes >= n_tiles) return;
  __shared__ float s_dec[256];
  __shared__ float s_alpha[256];
  __shared__ uint32_t s_col[(K + 1) * kBlock];
  stage_decode(s_dec, s_alpha, args.tab);
  __syncthreads();
  const uint32_t lane = lane_id();
  const uint32_t turn = blockIdx.x % kTicketLanes;
  constexpr uint32_t kWaves = kBlock / 64;
  for (uint32_t q = (blockIdx.x / kTicketLanes * kWaves + rfl(threadIdx.x >> 6)) * kTicketLanes + turn; q < n_tiles;) {
    const TileBatchArgs& g = fresh_batch_args();
    uint32_t ticket = 0;
    if (lane == 0u) ticket = draw_ticket(g.tb, g.tb.ticket0 + (kTicketLanes + turn) * 16u);
    const uint32_t entry = rfl(g.tb.deep[g.tb.deep_base + q]);
    const uint32_t tile = g.split ? g.tb.tile_first + (entry & 0xFFFFu) : entry;
    if (rfl(g.tb.cnt[tile]) > kBinRuns) {  // the deep composite's
      q = turn + gridDim.x * kWaves + kTicketLanes * rfl(ticket);
      continue;
    }
    const auto fr = (FramePtr)g.frames;
    TileSrc src;
    TileDst dst;
    frame_views(fr, rfl(find_frame<true>(g.frames, g.f0, g.f1, (uint64_t)tile * kTileTargets)), g.tab, src, dst);
    const auto* const bucket = (const __attribute__((address_space(1))) uint64_t*)g.tb.bucket;
    const uint64_t rec = g.tb.run[(uint64_t)tile * kTileRuns + lane];
    const uint32_t* const more = &g.tb.more[(uint64_t)tile * kTileRuns];
    const uint64_t base = ((uint64_t)more[1] << 32) | more[0];
    const uint32_t n = (uint32_t)(rec >> 32), most = wave_top_u32(n);
    const uint32_t step = bin_step((uint32_t)rec), newest = bin_at((uint32_t)rec) + (n - 1u) * step;
    const auto* const entry_of = bucket + base;
    FrontS<K> a;
    a.init(s_col + threadIdx.x);
    float4 tailc = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr uint32_t kU = 4;  // entries of a trip; the next trip's are on their way
    uint64_t ahead[kU];
#pragma unroll
    for (uint32_t u = 0; u < kU; ++u) ahead[u] = entry_of[u < n ? newest - u * step : 0u];
#pragma nounroll
    for (uint32_t s = 0; s < most; s += kU) {
      uint64_t cd[kU];
#pragma unroll
      for (uint32_t u = 0; u < kU; ++u) cd[u] = ahead[u];
#pragma unroll
      for (uint32_t u = 0; u < kU; ++u) ahead[u] = entry_of[s + kU + u < n ? newest - (s + kU + u) * step : 0u];
      // most trips of a long list are behind the K in every lane
      uint64_t front = s < (uint32_t)K ? 1ull : 0ull;
#pragma unroll
      for (uint32_t u = 0; u < kU; ++u)
        front |= __ballot(s + u < n) & __ballot(a.key_of(cd[u], s + u, 0u) < a.v[K - 1]);
      uint32_t behind[kU];  // what falls behind; 0 leaves the tail as it is
#pragma unroll
      for (uint32_t u = 0; u < kU; ++u) behind[u] = (uint32_t)cd[u];
      if (front != 0ull) {
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) behind[u] = a.insert(cd[u], s + u, s + u < n);
      }
      if (kTail) {
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
          const bool tail = s + u >= (uint32_t)K && s + u < n;
          tailc = over(tailc, decode_premult_lds(tail ? behind[u] : 0u, s_dec, s_alpha));
        }
      }
    }
    float4 col = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
      if ((k & 3) == 0) asm volatile("" ::: "memory");  // colours in fours: fewer registers
      if ((uint32_t)k < most && (uint32_t)k < n) col = over(col, decode_premult_lds(a.colour(k), s_dec, s_alpha));
    }
    const uint32_t t = (tile - dst.tile0) * kTileTargets + lane;
    if (t < dst.T) dst.out[t] = over(over(col, tailc), dst.background);
    if (lane == 0u) g.tb.cnt[tile] = 0u;
    g.tb.more[(uint64_t)tile * kTileRuns + lane] = 0u;
    q = turn + gridDim.x * kWaves + kTicketLanes * rfl(ticket);
  }
}

template <int K, bool kTail>
__global__ __launch_bounds__(64) void k_tile_batch_deep(TileBatchArgs args) {
  if (rfl(ld_relaxed(&args.tb.ctl[args.tb.ctl_index + 1u])) == 0u) return;  // none left over
  const uint32_t n = rfl(ld_relaxed(&args.tb.ctl[args.tb.ctl_index]));
  __shared__ float s_dec[256];
  __shared__ float s_alpha[256];
  __shared__ DeepLds<K> w;
  for (uint32_t k = threadIdx.x; k < 256u; k += 64u) {
    s_dec[k] = args.tab->dec[k];
    s_alpha[k] = args.tab->alpha[k];
  }
  __syncthreads();
  for (uint32_t q = blockIdx.x; q < n; q += gridDim.x) {
    const TileBatchArgs& g = fresh_batch_args();
    const uint32_t entry = rfl(g.tb.deep[g.tb.deep_base + q]);
    const uint32_t tile = g.split ? g.tb.tile_first + (entry & 0xFFFFu) : entry;
    if (rfl(g.tb.cnt[tile]) <= kBinRuns) continue;  // composited: its count is 0
    const auto fr = (FramePtr)g.frames;
    TileSrc src;
    TileDst dst;
    frame_views(fr, rfl(find_frame<true>(g.frames, g.f0, g.f1, (uint64_t)tile * kTileTargets)), g.tab, src, dst);
    deep_wave<K, kTileList, kTail>(tile, 1u, 0u, g.tb, src, dst, w, s_dec, s_alpha);
    wave_lds_sync();
  }
}

// Waves that share a tile, 1 << split, of `slots` resident waves: the least of
// rounds x cost, where a wave pays for the fragments it reads (all of the
// tile's, once for every part that fits its LDS, and about 200 fragments'
// time besides) and for those it lists and sorts (its share). Few tiles get
// up to eight waves each (a 145x103 frame of 130 thousand fragments, 234
// tiles: 80 us with a wave each, one tile after another's latency, 22 with
// eight); and so do tiles a little more numerous than the waves, or larger
// than one part (808x402, 3.5 M fragments, 5076 tiles: 136 us with a wave
// each, in two rounds of two parts, 123 with two; beyond two rounds it gained nothing:
// 1600x900 Loop32 175 us with a wave a tile, 230 with two).
inline uint32_t tile_split(uint32_t tiles, uint32_t slots, uint64_t frags, uint32_t cap) {
  if (tiles > kSharedTiles || tiles > 2u * slots) return 0;
  const uint64_t n = tiles ? frags / tiles : 0u;
  uint32_t best = 0;
  uint64_t least = ~0ull;
  for (uint32_t split = 0; split <= 3u; ++split) {
    const uint64_t rounds = (((uint64_t)tiles << split) + slots - 1u) / slots;
    const uint64_t parts = ((n + n / 4u) >> split) / cap + 1u;  // a quarter more: tiles differ
    const uint64_t cost = rounds * (parts * (n + 200u) + (n >> split));
    if (cost < least) {
      least = cost;
      best = split;
    }
  }
  return best;
}
constexpr uint32_t kListedFragments = 300;  // a tile of a batch group, whose fragments are not counted apart

template <int K>
struct TileBatch {
  template <bool kTail>
  static hipError_t go(const BatchArgs& a, const TileBuf& tb, hipStream_t s) {
    const uint32_t tiles = a.tiles * (kBlock / kTileTargets);
    const uint32_t split = tile_split(tiles, kComputeUnits * (uint32_t)tile_waves<K>() * (kBlock / 64),
                                      (uint64_t)tiles * kListedFragments, tile_entries(false));
    const TileBatchArgs args{tb, a.frames, a.f0, a.f1, a.tile0 * (kBlock / kTileTargets), tiles, split, a.tab};
    const uint32_t want = ((tiles << split) + kBlock / 64 - 1u) / (kBlock / 64);
    const uint32_t fit = kComputeUnits * (uint32_t)tile_waves<K>();
    hipLaunchKernelGGL((k_tile_batch<K, kTail>), dim3(want < fit ? want : fit), dim3(kBlock), 0, s, args);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = launch_tile_bin(a, tb, tiles, split, s);
    if (e != hipSuccess) return e;
    const uint32_t need = (tiles + kBlock / 64 - 1u) / (kBlock / 64);
    const uint32_t most = kComputeUnits * (K >= 32 ? 4u : 8u);
    const uint32_t blocks = need < most ? (need + kTicketLanes - 1u) / kTicketLanes * kTicketLanes : most;
    hipLaunchKernelGGL((k_tile_binned<K, kTail>), dim3(blocks), dim3(kBlock), 0, s, args);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL((k_tile_batch_deep<K, kTail>), dim3(tiles < kComputeUnits ? tiles : kComputeUnits), dim3(64), 0, s,
                       args);
    return hipGetLastError();
  }
};

template <int K>
struct TileResolve {
  template <int kMode, bool kTail>
  static hipError_t go(const TileBuf& tb, const TileSrc& src, const TileDst& dst, hipStream_t s) {
    const uint32_t tiles = (dst.T + kTileTargets - 1u) / kTileTargets;
    const uint32_t fit = kComputeUnits * (uint32_t)tile_waves<K>();  // blocks resident at once
    const uint32_t split = tile_split(tiles, fit * (kBlock / 64), src.frags, tile_entries(kMode == kTileLoop32));
    const uint32_t want = ((tiles << split) + kBlock / 64 - 1u) / (kBlock / 64);
    // three rounds of resident blocks: tiles differ in depth, and the blocks
    // of the later rounds go where the earlier ones have ended (1600x900 Loop32
    // K = 16: 247 us with one round, 204 with three; 1920x1080 Loop64: 155, 159)
    const uint32_t most = 3u * fit;
    const dim3 g(want < most ? want : most), b(kBlock);
    // kGeneral: several segments, or the debug outputs
    const bool dbg = dst.fk_key || dst.fk_val || dst.counts || src.nseg > 1u;
    const TileArgs args{tb, src, dst, tiles, split};
    if (dbg) hipLaunchKernelGGL((k_tile_resolve<K, kMode, kTail, true>), g, b, 0, s, args);
    else hipLaunchKernelGGL((k_tile_resolve<K, kMode, kTail, false>), g, b, 0, s, args);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || src.frags == 0u) return e;
    const uint32_t blocks = tiles < kDeepBlocks ? tiles : kDeepBlocks;
    hipLaunchKernelGGL((k_tile_deep<K, kMode, kTail>), dim3(blocks), dim3(64), 0, s, args);
    return hipGetLastError();
  }
  template <int kMode>
  static hipError_t tail_or_not(const TileBuf& tb, const TileSrc& src, const TileDst& dst, bool tail, hipStream_t s) {
    return tail ? go<kMode, true>(tb, src, dst, s) : go<kMode, false>(tb, src, dst, s);
  }
  static hipError_t run(const TileBuf& tb, const TileSrc& src, const TileDst& dst, int mode, bool tail,
                        hipStream_t s) {
    switch (mode) {
      case kTileLoop64: return tail_or_not<kTileLoop64>(tb, src, dst, tail, s);
      case kTileLoop32: return tail_or_not<kTileLoop32>(tb, src, dst, tail, s);
      default: return hipErrorInvalidValue;
    }
  }
};

}  // namespace

}  // namespace oit
