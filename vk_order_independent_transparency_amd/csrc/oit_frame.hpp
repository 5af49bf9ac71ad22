// oit_frame.hpp - device-side pieces shared by the kernel translation units:
// wave runs, colour-pass tail lists, the sorted front-K arrays, target
// orders, the opaque test, codec staging, the dispatch on the layer count.
#pragma once

#include "oit_kernels.hpp"

namespace oit {

namespace {

constexpr uint32_t kBlock = 256;

inline uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

// A run of consecutive lanes that carry the same target. Fragment ids grow
// with the lane, so a run is a block of consecutive ids of one target, and
// no fragment outside the wave can have an id inside it.
struct Run {
  uint32_t lane;
  uint32_t start_lane;
  uint32_t end_lane;
  bool start;
  bool end;
};

// Must be reached by all 64 lanes (callers keep every lane alive and give
// lanes without a fragment a target of kEmpty).
__device__ __forceinline__ Run same_target_run(uint32_t t) {
  Run r;
  r.lane = lane_id();
  const uint32_t tp = __shfl_up(t, 1u);
  const uint32_t tn = __shfl_down(t, 1u);
  r.start = (r.lane == 0) || (tp != t);
  r.end = (r.lane == 63) || (tn != t);
  const uint64_t starts = __ballot(r.start);
  const uint64_t ends = __ballot(r.end);
  const uint64_t le = (2ull << r.lane) - 1ull;  // lanes <= this lane
  r.start_lane = 63u - (uint32_t)__builtin_clzll(starts & le);
  r.end_lane = r.lane + (uint32_t)__builtin_ctzll(ends >> r.lane);
  return r;
}

// Colour-pass tail list value of frame-local fragment lid: ((lid + 1) << 1)
// | boundary flag, so that 0 can terminate the lists; its link word is
// next[lid]. Values order as ids do.
__device__ __forceinline__ uint32_t tail_value(uint32_t lid, uint32_t flag) { return ((lid + 1u) << 1) | flag; }
__device__ __forceinline__ uint32_t tail_index(uint32_t v) { return (v >> 1) - 1u; }
// values below this have link words in arrays of `cap` fragments
__device__ __forceinline__ uint32_t tail_value_cap(uint32_t cap) { return (cap + 1u) << 1; }

// Colour-pass tail lists, phase 1: a tail fragment `lid` stores its
// premultiplied colour at index lid, and its record (target << 32) | tail
// value goes to the frame's tail queue. The queue is cut into regions of
// 1024 fragment ids, each with its own counter, and a record goes to the
// region of its fragment's id: a fragment enters the tail once, so region
// r's entries fit in rec[r * 1024 ..]. The lanes of one region share one
// returning atomic, so a wave waits for one round trip however many tail
// fragments it finds. The queue holds only tail fragments, so the link pass
// reads nothing of the others. Called by every active lane of the wave that
// may hold a tail fragment.
__device__ __forceinline__ void tail_queue_push(bool tail, uint32_t t, uint32_t lid, uint32_t flag, float4 payload,
                                                const TailBuf& tb, uint32_t mask) {
  tail = tail && lid < tb.cap && tb.qn != nullptr;
  if (tail) {
    tb.rgba[lid] = payload;
    if (tb.mask) tb.mask[lid] = mask;
  }
  const uint32_t r = lid >> kTailRegionShift;
  const uint32_t lane = lane_id();
  // group the lanes by region (cross-lane work only), then one atomic per
  // group, all of them in flight together
  uint64_t rem = __ballot(tail);
  uint32_t my_leader = 0;
  uint64_t my_group = 0;
  while (rem) {
    const uint32_t leader = (uint32_t)__builtin_ctzll(rem);
    const uint32_t rl = __builtin_amdgcn_readlane(r, leader);
    const uint64_t m = __ballot(tail && r == rl);
    if ((m >> lane) & 1ull) {
      my_leader = leader;
      my_group = m;
    }
    rem &= ~m;
  }
  uint32_t q = 0;
  if (tail && lane == my_leader) q = atomicAdd(&tb.qn[r], (uint32_t)__builtin_popcountll(my_group));
  q = __shfl(q, (int)my_leader);
  if (tail)
    tb.rec[((uint64_t)r << kTailRegionShift) + q + lanes_below(my_group)] = ((uint64_t)t << 32) | tail_value(lid, flag);
}

// Sorted register array of K (sort key, colour) pairs, ascending; inserting x
// returns the element pushed out of the back (x itself if it does not fit):
// insertionSortTail, oitCompositeDefines.glsl:116-139, unrolled into selects.
template <int K>
struct FrontK {
  uint64_t sk[K];
  uint32_t col[K];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      sk[k] = kEmpty64;
      col[k] = 0u;
    }
  }
  __device__ __forceinline__ void insert(uint64_t x, uint32_t xc, uint64_t& ev, uint32_t& evc) {
    const bool fits = x < sk[K - 1];
    ev = fits ? sk[K - 1] : x;
    evc = fits ? col[K - 1] : xc;
#pragma unroll
    for (int j = K - 1; j > 0; --j) {
      const bool before = x < sk[j - 1];
      const bool here = x < sk[j];
      sk[j] = before ? sk[j - 1] : (here ? x : sk[j]);
      col[j] = before ? col[j - 1] : (here ? xc : col[j]);
    }
    const bool first = x < sk[0];
    sk[0] = first ? x : sk[0];
    col[0] = first ? xc : col[0];
  }
  // The same insert when at most w - 1 slots can be occupied (w is wave
  // uniform): slots at and beyond w hold the +inf sentinel before and after
  // the insert, so whole blocks of four slots at or beyond w are skipped
  // with one scalar branch each (executing more slots is also exact).
  __device__ __forceinline__ void insert_bounded(uint64_t x, uint32_t xc, uint64_t& ev, uint32_t& evc, int w) {
    const bool fits = x < sk[K - 1];
    ev = fits ? sk[K - 1] : x;
    evc = fits ? col[K - 1] : xc;
#pragma unroll
    for (int b = ((K - 1) / 4) * 4; b >= 0; b -= 4) {
      if (b < w) {
#pragma unroll
        for (int j = (b + 3 < K - 1 ? b + 3 : K - 1); j >= b && j > 0; --j) {
          const bool before = x < sk[j - 1];
          const bool here = x < sk[j];
          sk[j] = before ? sk[j - 1] : (here ? x : sk[j]);
          col[j] = before ? col[j - 1] : (here ? xc : col[j]);
        }
      }
    }
    const bool first = x < sk[0];
    sk[0] = first ? x : sk[0];
    col[0] = first ? xc : col[0];
  }
};

// FrontK with a third payload moved alongside (the ordered interlock's sample
// masks under coverage shading); the same bounded insert.
template <int K>
struct FrontKM {
  uint64_t sk[K];
  uint32_t col[K];
  uint32_t msk[K];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      sk[k] = kEmpty64;
      col[k] = 0u;
      msk[k] = 0u;
    }
  }
  __device__ __forceinline__ void insert_bounded(uint64_t x, uint32_t xc, uint32_t xm, uint64_t& ev, uint32_t& evc,
                                                 int w) {
    const bool fits = x < sk[K - 1];
    ev = fits ? sk[K - 1] : x;
    evc = fits ? col[K - 1] : xc;
#pragma unroll
    for (int b = ((K - 1) / 4) * 4; b >= 0; b -= 4) {
      if (b < w) {
#pragma unroll
        for (int j = (b + 3 < K - 1 ? b + 3 : K - 1); j >= b && j > 0; --j) {
          const bool before = x < sk[j - 1];
          const bool here = x < sk[j];
          sk[j] = before ? sk[j - 1] : (here ? x : sk[j]);
          col[j] = before ? col[j - 1] : (here ? xc : col[j]);
          msk[j] = before ? msk[j - 1] : (here ? xm : msk[j]);
        }
      }
    }
    const bool first = x < sk[0];
    sk[0] = first ? x : sk[0];
    col[0] = first ? xc : col[0];
    msk[0] = first ? xm : msk[0];
  }
};

// Sorted register array of K sort keys only (depth key << 32 | node index),
// ascending: the colours are reloaded by node index after the walk, which
// keeps one third fewer registers live during the latency-bound walk.
template <int K>
struct FrontKeys {
  uint64_t sk[K];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int k = 0; k < K; ++k) sk[k] = kEmpty64;
  }
  // insertionSortTail with a wave-uniform bound w on the occupied slots + 1
  __device__ __forceinline__ uint64_t insert_bounded(uint64_t x, int w) {
    const uint64_t ev = x < sk[K - 1] ? sk[K - 1] : x;
#pragma unroll
    for (int b = ((K - 1) / 4) * 4; b >= 0; b -= 4) {
      if (b < w) {
#pragma unroll
        for (int j = (b + 3 < K - 1 ? b + 3 : K - 1); j >= b && j > 0; --j) {
          const bool before = x < sk[j - 1];
          const bool here = x < sk[j];
          sk[j] = before ? sk[j - 1] : (here ? x : sk[j]);
        }
      }
    }
    sk[0] = x < sk[0] ? x : sk[0];
    return ev;
  }
};

// Largest value of v over the active lanes, as a wave-uniform (scalar) value.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t w = __shfl_xor(v, o);
    v = w > v ? w : v;
  }
  return __builtin_amdgcn_readfirstlane(v);
}

// Front-to-back blend of the first n sorted packed colours
// (oitLinkedList.frag.glsl:162-166, oitSimple.frag.glsl:161-165).
template <int K>
__device__ __forceinline__ float4 blend_front(const FrontK<K>& a, uint32_t n, const CodecTables* tab) {
  float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int k = 0; k < K; ++k)
    if ((uint32_t)k < n) c = over(c, decode_premult(a.col[k], tab));
  return c;
}

// Tail values held in registers per walk of an unordered tail list, and
// the walks a fold takes before it sorts a longer list instead. At 1080p
// with K = 8 the longest tail is 14 (1 % of the tails need a second walk);
// a window of 16 cost the K = 8 composites two to three waves per SIMD.
constexpr int kTailWindow = 8;
constexpr uint32_t kTailWalks = 4;

// One walk of an unordered tail list: the kTailWindow largest values below
// `bound`, in descending order (0 = none), by an insertion network in
// registers; returns how many values of the list lie below `bound`. A walk
// longer than the arrays hold (a cycle) reports kErrWalk and sets `bad`.
__device__ __forceinline__ uint32_t tail_window(const TailBuf& tb, uint32_t head, uint32_t vcap, uint32_t bound,
                                                uint32_t (&w)[kTailWindow], bool& bad) {
#pragma unroll
  for (int k = 0; k < kTailWindow; ++k) w[k] = 0u;
  uint32_t n = 0, hops = 0;
  uint32_t v = head;
  while (v != 0u && v < vcap) {  // a link outside the arrays ends the walk
    if (++hops > tb.cap) {
      report_error(tb.err, kErrWalk);
      bad = true;
      break;
    }
    const uint32_t nx = tb.next[tail_index(v)];
    if (v < bound) {
      ++n;
      uint32_t x = v;
#pragma unroll
      for (int k = 0; k < kTailWindow; ++k) {
        const uint32_t hi = w[k] > x ? w[k] : x;
        x = w[k] > x ? x : w[k];
        w[k] = hi;
      }
    }
    v = nx;
  }
  return n;
}

// A tail list longer than kTailWindow * kTailWalks, sorted into descending
// order in place: a bottom-up merge sort of the singly linked list (runs of
// 1, 2, 4, ... merged pass by pass, each pass relinking every node once),
// O(n log n) link reads instead of one walk per window. The list is the
// composite lane's own and acyclic (tail_window walked it to its end first);
// a link at or above vcap ends it. Returns the new head.
__device__ __forceinline__ uint32_t tail_sort_desc(const TailBuf& tb, uint32_t head, uint32_t vcap) {
  auto nxt = [&](uint32_t v) -> uint32_t {
    const uint32_t x = tb.next[tail_index(v)];
    return x < vcap ? x : 0u;
  };
  for (uint32_t run = 1;; run <<= 1) {
    uint32_t p = head, out = 0u, last = 0u, merges = 0u;
    while (p != 0u) {
      ++merges;
      uint32_t q = p, np = 0u;
      while (np < run && q != 0u) {
        ++np;
        q = nxt(q);
      }
      uint32_t nq = run;
      while (np > 0u || (nq > 0u && q != 0u)) {
        uint32_t e;
        if (np == 0u || (nq > 0u && q != 0u && q > p)) {  // descending: the larger value first
          e = q;
          q = nxt(q);
          --nq;
        } else {
          e = p;
          p = nxt(p);
          --np;
        }
        if (last == 0u) out = e;
        else tb.next[tail_index(last)] = e;
        last = e;
      }
      p = q;
    }
    if (last != 0u) tb.next[tail_index(last)] = 0u;
    head = out;
    if (merges <= 1u) return head;
  }
}

// Colour buffer after the colour pass: the tail fragments of target t over
// the background in id order (the ROP's primitive order, main.cpp:548-558),
// folded newest first: acc = t_n over ... over t_1, then acc over the
// background. The list is unordered, so each walk takes the next
// kTailWindow values in descending order (one walk for most targets, up to
// kTailWalks) and loads their colours four at a time; a longer tail is
// sorted in place and folded in one walk.
// tail_fold with the list's head value already loaded (a composite issues
// that load with its own first loads instead of after them).
__device__ __forceinline__ float4 tail_fold_from(const TailBuf& tb, uint32_t head, float4 bg) {
  const uint32_t vcap = tail_value_cap(tb.cap);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (head == 0u || head >= vcap) return over(acc, bg);
  uint32_t bound = 0xFFFFFFFFu;
  bool bad = false;
  for (bool first = true;; first = false) {
    uint32_t w[kTailWindow];
    const uint32_t n = tail_window(tb, head, vcap, bound, w, bad);
    if (first && !bad && n > (uint32_t)kTailWindow * kTailWalks) {  // a long tail: sorted, then one walk
      for (uint32_t v = tail_sort_desc(tb, head, vcap); v != 0u && v < vcap;) {
        const uint32_t id = tail_index(v);
        const uint32_t nx = tb.next[id];
        acc = over(acc, tb.rgba[id]);
        v = nx;
      }
      break;
    }
#pragma unroll
    for (int g = 0; g < kTailWindow; g += 4) {
      if (w[g] == 0u) break;
      float4 c[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) c[j] = w[g + j] ? tb.rgba[tail_index(w[g + j])] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t v = w[g + j];
        if (v != 0u) acc = over(acc, c[j]);
      }
    }
    if (bad || n <= (uint32_t)kTailWindow) break;
    bound = w[kTailWindow - 1];
  }
  return over(acc, bg);
}

__device__ __forceinline__ float4 tail_fold(const TailBuf& tb, uint32_t t, float4 bg) {
  return tail_fold_from(tb, tb.head[t], bg);
}

// Sample shading with spp samples per pixel lays targets out sample-major
// (sample * pixels + pixel). pm_index(t) is target t's place in pixel-major
// order (pixel * spp + sample) and pm_target(a) its inverse. The stream gives
// a fragment's covered samples consecutive ids, so structures indexed
// pixel-major (the WBOIT accumulators) take one wave's atomics on one run of
// entries, and composites that walk targets in pixel-major order give a
// pixel's samples neighbouring lanes, whose list nodes share cache lines.
// spp is 1, 2, 4 or 8: shifts and compares, no divisions.
__device__ __forceinline__ uint32_t pm_index(uint32_t t, uint32_t T, uint32_t spp) {
  if (spp <= 1u) return t;
  const uint32_t sh = (uint32_t)__builtin_ctz(spp);
  const uint32_t px = T >> sh;
  uint32_t smp = 0;
  for (uint32_t k = 1; k < spp; ++k) smp += t >= k * px ? 1u : 0u;
  return ((t - smp * px) << sh) | smp;
}
__device__ __forceinline__ uint32_t pm_target(uint32_t a, uint32_t T, uint32_t spp) {
  if (spp <= 1u) return a;
  const uint32_t sh = (uint32_t)__builtin_ctz(spp);
  return (a & (spp - 1u)) * (T >> sh) + (a >> sh);
}

// Colour buffer of target t before the colour-pass tail: the colour of the
// frame's opaque pass, else the clear colour.
__device__ __forceinline__ float4 dest_of(const Common& c, uint32_t t) {
  return c.opq_rgba ? c.opq_rgba[t] : c.background;
}

constexpr uint32_t kMaxCoverage = 8;  // samples of a coverage mask

// Early depth test of a transparent fragment against the frame's opaque pass
// (early_fragment_tests with post_depth_coverage, oitColorDepthDefines.glsl:
// 24-37; VK_COMPARE_OP_LESS without depth write, main.cpp:526-528,541-543):
// the samples of mask m whose opaque depth key is larger than key (one test
// at target t unless coverage shading). Zero: the fragment does not exist.
__device__ __forceinline__ uint32_t opaque_visible(const uint64_t* z, uint32_t T, uint32_t cov, uint32_t t,
                                                   uint32_t key, uint32_t m) {
  if (!z) return m;
  if (cov > 1u) {
    // every plane's key in one round trip, whether the sample is covered or not
    // (1920x1080, 4 samples: frame 446 -> 436 us against a test after each load)
    const uint32_t* const keys = reinterpret_cast<const uint32_t*>(z) + 1;
    uint32_t k[kMaxCoverage];
#pragma unroll
    for (uint32_t s = 0; s < kMaxCoverage; ++s) k[s] = s < cov ? keys[2u * ((uint64_t)s * T + t)] : 0u;
    uint32_t r = 0u;
#pragma unroll
    for (uint32_t s = 0; s < kMaxCoverage; ++s) r |= key < k[s] ? 1u << s : 0u;
    return r & m;
  }
  return key < (uint32_t)(z[t] >> 32) ? m : 0u;
}

// Coverage shading: the ROP blends each tail fragment into the samples of
// its mask; per sample the newest-first fold over the sample's colour (the
// opaque pass's, else the clear colour), then the sum over samples in order
// divided by their count (the MSAA resolve). Without an opaque pass a target
// without tail fragments keeps the clear colour.
__device__ __forceinline__ float4 tail_fold_cov(const TailBuf& tb, uint32_t t, const Common& c) {
  const uint32_t S = c.cov;
  const uint32_t vcap = tail_value_cap(tb.cap);
  const uint32_t head = tb.head ? tb.head[t] : 0u;
  const bool empty = head == 0u || head >= vcap;
  if (empty && !c.opq_rgba) return c.background;
  float4 acc[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) acc[s] = make_float4(0.f, 0.f, 0.f, 0.f);
  uint32_t bound = 0xFFFFFFFFu;
  bool bad = false;
  while (!empty) {  // windows of the unordered list, newest first (tail_fold_from)
    uint32_t w[kTailWindow];
    const uint32_t n = tail_window(tb, head, vcap, bound, w, bad);
    if (bound == 0xFFFFFFFFu && !bad && n > (uint32_t)kTailWindow * kTailWalks) {  // a long tail: sorted, one walk
      for (uint32_t v = tail_sort_desc(tb, head, vcap); v != 0u && v < vcap;) {
        const uint32_t id = tail_index(v);
        const uint32_t nx = tb.next[id];
        const uint32_t m = tb.mask[id];
        const float4 col = tb.rgba[id];
#pragma unroll
        for (int s = 0; s < 8; ++s)
          if ((uint32_t)s < S && ((m >> s) & 1u)) acc[s] = over(acc[s], col);
        v = nx;
      }
      break;
    }
#pragma unroll
    for (int g = 0; g < kTailWindow; g += 4) {
      if (w[g] == 0u) break;
      float4 col[4];
      uint32_t msk[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool h = w[g + j] != 0u;
        col[j] = h ? tb.rgba[tail_index(w[g + j])] : make_float4(0.f, 0.f, 0.f, 0.f);
        msk[j] = h ? tb.mask[tail_index(w[g + j])] : 0u;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int s = 0; s < 8; ++s)
          if ((uint32_t)s < S && ((msk[j] >> s) & 1u)) acc[s] = over(acc[s], col[j]);
    }
    if (bad || n <= (uint32_t)kTailWindow) break;
    bound = w[kTailWindow - 1];
  }
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    if ((uint32_t)s < S) {
      const float4 cb = over(acc[s], c.opq_rgba ? c.opq_rgba[(uint64_t)s * c.T + t] : c.background);
      sum = make_float4(sum.x + cb.x, sum.y + cb.y, sum.z + cb.z, sum.w + cb.w);
    }
  }
  const float fs = (float)S;
  return make_float4(sum.x / fs, sum.y / fs, sum.z / fs, sum.w / fs);
}

// Coverage-shaded front blend (oitLinkedList.frag.glsl:147-160,
// oitSimple.frag.glsl:142-159): per sample, front to back over the sorted
// layers whose mask holds it; the sample colours summed in order and divided
// by the sample count.
template <int K>
__device__ __forceinline__ float4 blend_front_cov(const uint32_t* cols, const uint32_t* masks, uint32_t n, uint32_t S,
                                                  const float* s_dec, const float* s_alpha) {
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t s = 0; s < S; ++s) {
    float4 sc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < K; ++k)
      if ((uint32_t)k < n && ((masks[k] >> s) & 1u)) sc = over(sc, decode_premult_lds(cols[k], s_dec, s_alpha));
    sum = make_float4(sum.x + sc.x, sum.y + sc.y, sum.z + sc.z, sum.w + sc.w);
  }
  const float fs = (float)S;
  return make_float4(sum.x / fs, sum.y / fs, sum.z / fs, sum.w / fs);
}

template <int K>
__device__ __forceinline__ void write_debug(const ResolveOut& o, uint32_t t, const FrontK<K>& a, uint32_t n,
                                            uint32_t count, bool ids_from_nodes, bool vals_are_colors) {
  if (o.fk_key) {
#pragma unroll
    for (int k = 0; k < K; ++k) o.fk_key[(uint64_t)t * K + k] = (uint32_t)k < n ? (uint32_t)(a.sk[k] >> 32) : kEmpty;
  }
  if (o.fk_val) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      uint32_t v = kEmpty;
      if ((uint32_t)k < n) {
        v = vals_are_colors ? a.col[k] : (uint32_t)a.sk[k];
        if (ids_from_nodes) v -= 1u;  // node n holds fragment id n - 1
      }
      o.fk_val[(uint64_t)t * K + k] = v;
    }
  }
  if (o.counts) o.counts[t] = count;
}

// Codec thresholds staged in LDS for the block.
__device__ __forceinline__ void stage_thresholds(float* s_thr, const CodecTables* tab) {
  for (uint32_t k = threadIdx.x; k < 257u; k += kBlock) s_thr[k] = tab->thr[k];
  __syncthreads();
}

__device__ __forceinline__ void stage_decode(float* s_dec, float* s_alpha, const CodecTables* tab) {
  for (uint32_t k = threadIdx.x; k < 256u; k += kBlock) {
    s_dec[k] = tab->dec[k];
    s_alpha[k] = tab->alpha[k];
  }
}

// Last frame in [lo, hi) whose base is <= key (bases ascend); key is wave
// uniform, so the probes are scalar loads.
template <bool kTargets>
__device__ __forceinline__ uint32_t find_frame(const BatchFrameDev* fr, uint32_t lo, uint32_t hi, uint64_t key) {
  while (hi - lo > 1u) {
    const uint32_t mid = (lo + hi) >> 1;
    const uint64_t base = kTargets ? (uint64_t)fr[mid].target_base : (uint64_t)fr[mid].frag_base;
    if (base <= key) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Orders LDS ops of one wave: every lane's earlier LDS access has completed
// and none is moved across (the wave's lanes exchange data through LDS).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <template <int> class F, typename... A>
hipError_t dispatch_k(uint32_t K, A&&... args) {
  switch (K) {
    case 1: return F<1>::run(args...);
    case 2: return F<2>::run(args...);
    case 4: return F<4>::run(args...);
    case 8: return F<8>::run(args...);
    case 16: return F<16>::run(args...);
    case 32: return F<32>::run(args...);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

}  // namespace oit
