// compact.hip -- level-step kernels of the compact databases (gfx950, wave64).
//
// A database is compact when every graph has at most 64 vertices, its label
// alphabets are small (NEL * (NVL + 1) <= 63) and a graph's vertices fit 255
// groups (below): transactions, molecules, random graphs of the common
// sizes.  The kernels of kernels.hip mine the others, and all databases under
// the entry point that allocates nothing.
//
// Layout.  A vertex is one 8-byte *group* (g the graph's first group, u the
// vertex's local id: group g + u): four 12-bit items (neighbour 6 bits, label
// pair edge label * NVL + neighbour label 6 bits) and, in bits 48-55, the place
// (relative to g) of a further group when the vertex has more than four
// neighbours.  One gather per rightmost-path source fetches all of the common
// vertices' neighbours; nothing depends on an offset read first.  (With a
// 4-byte offset and 4-byte entries a row's sources touched 4-5 lines of 128
// bytes per segment, in two dependent steps.)
//
// Rows are {8 g, tuple} of 1 + TW words (tuple bytes past the pattern's
// vertices repeat vertex 0's, so that the visited set is an OR over all bytes),
// pattern-major; a chunk is a run of whole segments (rows of one graph) of ONE
// pattern, so everything about the pattern is wave-uniform: the sources are
// walked in a scalar loop, and the label rules of a source (order rule,
// minimum label, 2-edge path masks) are a 64-bit mask over label pairs.  An
// item is tested with two shifts: its label pair against the mask, its
// neighbour against the row's visited set.
//
// Per block of up to 64 rows and per source, the passing items are counted,
// ranked over the wave and appended to the chunk's dense list
//   source << 25 | item << 13 | row of the chunk
// (4 bytes a candidate; backward targets are sources 64 on, with the edge
// label in the label pair's place; source 127 moves the row base on by
// kMarkRows).  Counts live in LDS records indexed by the key itself (K <=
// 4032; no hashing, no overflow).  A key names its source, and within a source
// the list is in row order, so every key's entries are in row order: k_cwrite
// can place the children's rows graph-contiguously in list order.
//
// What bounds k_clevel: the gathers.  64 rows lie in some 40 graphs, so a load
// of one group a lane touches about as many lines; a block's 20 vector memory
// instructions touch 300 lines in all, of which 170 miss the 32 KB L1 that 28
// waves share and are asked of L2.  The address units are 80-85 %
// busy and L1 waits on pending lines for 75 % of the time (100,000
// transactions: 2.85 ms for the levels of 8-byte tuples, 2.3 ms with the loads
// alone); neither more waves, loads further ahead nor lines kept in an XCD's
// L2 change it.  Vector issue comes next (850 instructions a block) and is
// hidden behind it.  Items at bit offsets that one shift reaches and 16-byte
// counter records took all levels of that case from 5.15 ms to 4.75, the
// sibling rules (k_cchildren), which leave fewer candidates to list, to 4.2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"
#include "wave.hpp"

namespace gm {
namespace {

constexpr uint32_t kNone32 = 0xFFFFFFFFu;
constexpr uint32_t kMarkSource = 127u;
constexpr uint32_t kBackSource = 64u;  // source number of backward target 0
constexpr int kMarkRows = 4096;        // (rows of a block stay below kMarkRows + 64 < 2^13)

// (lambdas used several times must not become calls: a call needs scratch)
#define GM_INLINE __attribute__((always_inline))

// wave-uniform read-only data through the scalar cache
typedef const uint32_t __attribute__((address_space(4))) *ConstWords;
template <class T>
__device__ __forceinline__ T cload(ConstWords c) {
  uint32_t w[sizeof(T) / 4];
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) w[i] = c[i];
  T t;
  __builtin_memcpy(&t, w, sizeof(t));
  return t;
}
template <class T>
__device__ __forceinline__ T cload(const void *p) {
  return cload<T>((ConstWords)(uintptr_t)p);
}

// A kernel argument read where it is used (from the argument segment,
// through the scalar cache) instead of held in scalar registers from the
// kernel's start on: k_clevel uses some thirty of them, most of them once.
#define GM_ARG(field) arg_at<decltype(StepArgs::field), offsetof(StepArgs, field)>()
template <class T, size_t kOffset>
__device__ __forceinline__ T arg_at() {
  ConstWords c = (ConstWords)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(c));
  return cload<T>(c + kOffset / 4);
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// lanes below this one in a ballot
__device__ __forceinline__ uint32_t below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Pointers read from the argument segment are generic; these make the
// accesses global ones (a flat access also waits on the LDS counter).
#define GM_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ GM_GLOBAL T *as_global(T *p) {
  return (GM_GLOBAL T *)(uintptr_t)p;
}

template <int TW>
struct CRow {
  uint32_t x[1 + TW];
};

// The graph vertex at pattern vertex i (wave-uniform), in byte 0 (image) or in
// all four (image4): one byte permute of the two words that can hold it; past
// eight vertices the words are picked by masks (selects would become an
// indexed array in scratch).
template <int TW>
__device__ __forceinline__ uint32_t image_of(const CRow<TW> &t, int i, uint32_t sel) {
  uint32_t lo = t.x[1], hi = TW > 1 ? t.x[TW > 1 ? 2 : 1] : 0u;
  if constexpr (TW > 2) {
    lo = hi = 0;
#pragma unroll
    for (int q = 0; q < TW; q += 2) {
      const uint32_t m = 0u - (uint32_t)((i >> 3) == q / 2);
      lo |= t.x[1 + q] & m;
      if (q + 1 < TW) hi |= t.x[q + 1 < TW ? 2 + q : 1] & m;
    }
  }
  return __builtin_amdgcn_perm(hi, lo, sel);
}
template <int TW>
__device__ __forceinline__ uint32_t image(const CRow<TW> &t, int i) {
  return image_of<TW>(t, i, 0x0C0C0C00u | (uint32_t)(i & 7));
}
template <int TW>
__device__ __forceinline__ uint32_t image4(const CRow<TW> &t, int i) {
  return image_of<TW>(t, i, 0x01010101u * (uint32_t)(i & 7));
}

// A group: items at bits 0, 12, 24 and 36 (unused ones all ones), the next
// group's place at bits 48-55.
typedef unsigned long long Group;
__device__ __forceinline__ uint32_t next_of(Group g) { return (uint32_t)(g >> 32) >> 16; }
__device__ __forceinline__ uint32_t item(Group g, int i) { return (uint32_t)(g >> (12 * i)) & 0xFFFu; }
// the items' neighbours, a byte each
__device__ __forceinline__ uint32_t neighbours(Group g) {
  return item(g, 0) % 64 | (item(g, 1) % 64) << 8 | (item(g, 2) % 64) << 16 | (item(g, 3) % 64) << 24;
}
// 0x80 in the lowest byte of x that is zero, if any (and perhaps above it)
__device__ __forceinline__ uint32_t zero_bytes(uint32_t x) { return (x - 0x01010101u) & ~x & 0x80808080u; }

// Inclusive sum over the wave in data-parallel primitives (six adds; the
// shuffle scan goes through LDS).
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t dpp_from(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kCtrl, kRows, 0xF, kRows == 0xF);
}
__device__ __forceinline__ uint32_t wave_incl(uint32_t x) {
  x += dpp_from<0x111, 0xF>(x);  // row_shr:1
  x += dpp_from<0x112, 0xF>(x);  // row_shr:2
  x += dpp_from<0x114, 0xF>(x);  // row_shr:4
  x += dpp_from<0x118, 0xF>(x);  // row_shr:8
  x += dpp_from<0x142, 0xA>(x);  // row_bcast:15 to rows 1 and 3
  x += dpp_from<0x143, 0xC>(x);  // row_bcast:31 to rows 2 and 3
  // (kept whole: taken apart by a caller's difference, the partial sums keep
  // the adds from becoming single add-with-shift instructions)
  asm("" : "+v"(x));
  return x;
}

// A key's counts in the chunk: the block's segments that hold it (by head
// lane), its support (bit 31: the mask's bit 0 is a carried segment, counted
// already) and its embeddings.
struct alignas(16) KeyCount {
  unsigned long long mask;
  uint32_t sup, emb;
};

// The chunk's candidate list: extents of entries, the first at
// chunk * page, further ones from the pool (64 slices with a cursor each on a
// line of its own).  An extent starts with {entries, next extent or kNone32};
// extents are named in units of kListUnit entries.
struct ListOut {
  GM_GLOBAL uint32_t *ext;
  uint32_t used, cap;
  bool off;  // the pool ran out: the stage runs again with a larger one
};

template <bool ROOT, int TW, bool M32>
__global__ void __launch_bounds__(64, (M32 ? (TW <= 8 ? 7 : 6) : TW <= 3 ? 6 : 5)) k_clevel(StepArgs) {
  extern __shared__ __attribute__((aligned(16))) uint32_t dyn[];
  const int K = (int)GM_ARG(K);
  KeyCount *const kc = reinterpret_cast<KeyCount *>(dyn);
  __shared__ uint32_t stage[64];  // a source's items on their way to the list
  const int lane = threadIdx.x;
  const uint32_t gci = blockIdx.x;
  if (gci < (uint32_t)kSpread) stamp_start(GM_ARG(spread), gci);

  // the chunk: pattern p, nominal rows [nom0, nom1) of the pattern's pend
  // (relative to its first row: a pattern has fewer than 2^32), moved
  // forward to segment starts
  constexpr int RW = 1 + TW;
  int p;
  uint32_t nom0, pend;
  uint64_t first;
  const char *meta = nullptr;
  CMetaHead H = {};
  uint32_t nom;
  if constexpr (ROOT) {
    nom = (uint32_t)GM_ARG(nom);
    const uint4 ct = cload<uint4>(GM_ARG(rtab) + GM_ARG(tab0) + gci);
    p = (int)ct.x;
    first = ct.z;
    pend = ct.w;
    nom0 = ct.y * nom;
  } else {
    const uint2 ct = cload<uint2>(GM_ARG(ctab) + GM_ARG(tab0) + gci);
    p = uniform((int)ct.x);
    meta = reinterpret_cast<const char *>(GM_ARG(meta)) + (int64_t)p * GM_ARG(meta_stride);
    H = cload<CMetaHead>(meta);
    first = H.row0;
    pend = (uint32_t)H.nrows;
    nom = H.nom;
    nom0 = (uint32_t)uniform((int)ct.y) * nom;
  }
  const uint32_t nom1 = pend - nom0 <= nom ? pend : nom0 + nom;
  GM_GLOBAL const uint32_t *const rows = as_global(GM_ARG(crow) + first * RW);
  uint32_t b = nom0;
  bool empty = !ROOT && (H.flags & kPatDead);
  if (!empty && nom0 > 0) {
    for (uint64_t base = nom0;; base += 64) {
      if (base >= nom1) {
        empty = true;
        break;
      }
      const uint64_t r = base + (uint32_t)lane;
      const bool f = r < pend && rows[r * RW] != rows[(r - 1) * RW];
      const uint64_t m = __ballot(f);
      if (m) {
        b = (uint32_t)base + (uint32_t)__ffsll((long long)m) - 1u;
        empty = b >= nom1;
        break;
      }
    }
  }
  if (empty) {
    if (lane == 0) GM_ARG(cchunks)[gci] = CChunk{0, 0, 0u};
    return;
  }
  const uint32_t start = b;
  for (int i = lane; i < K; i += 64) kc[i] = KeyCount{0, 0, 0};
  wave_sync();

  const uint32_t page = GM_ARG(page);
  ListOut L{as_global(GM_ARG(clist)) + (uint64_t)gci * page, 2u, page, false};
  // room for n entries in one extent: their place in it
  auto reserve = [&](uint32_t n) GM_INLINE -> uint32_t {
    if (L.used + n > L.cap) {
      const uint32_t units = (max(page, n + 2u) + kListUnit - 1) / kListUnit;
      uint32_t at = kNone32;
      if (lane == 0 && !L.off) {
        unsigned long long *const spread = GM_ARG(spread);
        const uint32_t sub_size = GM_ARG(pool_sub), pool0 = GM_ARG(pool0);
        for (uint32_t t = 0; t < (uint32_t)kSpread && at == kNone32; ++t) {
          const uint32_t sub = (gci + t) & (kSpread - 1);
          const unsigned long long o = atomicAdd(&spread[sub * kSpreadStride + kSpreadPool], (unsigned long long)units);
          if (o + units <= (unsigned long long)sub_size) at = pool0 + sub * sub_size + (uint32_t)o;
        }
        L.ext[0] = L.used - 2u;
        L.ext[1] = at;
        if (at == kNone32) atomicOr(GM_ARG(error_flag), kErrListPool);
      }
      at = (uint32_t)uniform((int)at);
      L.off = L.off || at == kNone32;
      if (!L.off) L.ext = as_global(GM_ARG(clist)) + (uint64_t)at * kListUnit;
      L.used = 2u;
      L.cap = L.off ? kNone32 - 1u : units * kListUnit;
    }
    const uint32_t pos = L.used;
    L.used += n;
    return pos;
  };

  uint32_t n_pruned = 0;
  unsigned long long listed = 0;
  bool carry = false;   // the block's first rows may go on with the last block's segment
  uint32_t carry_g = 0;  // of this graph
  uint32_t rowbase = 0;  // rows of the chunk before the list's current row base
  for (;;) {
    const int ws = (int)min(64u, pend - b);
    CRow<TW> t;
    {
      GM_GLOBAL const uint32_t *src = rows + ((uint64_t)b + (uint32_t)min(lane, ws - 1)) * RW;
#pragma unroll
      for (int q = 0; q < RW; ++q) t.x[q] = src[q];
    }
    const uint32_t g = t.x[0];
    const uint32_t pg = __shfl_up(g, 1, 64);
    const uint64_t diff = __ballot(lane < ws && (lane == 0 ? !carry || g != carry_g : pg != g));
    if (carry && (diff & 1ull)) {  // it ended with the last block: its keys' marks are done with
      for (int i = lane; i < K; i += 64) {
        kc[i].sup &= 0x7FFFFFFFu;
        kc[i].mask = 0;
      }
      wave_sync();
    }
    // the block: up to the first segment start at or past nom1 (none of the
    // window's rows when a carried segment ended with the last block there),
    // to the pattern's end, or to the window's last segment start (its segment may
    // go on); a window that is one segment is taken whole and carried on
    int nb;
    bool last = true, carry_out = false;
    {
      uint64_t after = 0;
      if (nom1 < pend && (nom1 <= b || nom1 - b < 64)) after = diff & (nom1 <= b ? ~0ull : ~0ull << (nom1 - b));
      const uint64_t later = diff & ~1ull;
      if (after) {
        nb = __ffsll((long long)after) - 1;
      } else if (pend - b == (uint32_t)ws) {
        nb = ws;
      } else {
        last = false;
        if (later) {
          nb = 63 - __clzll((long long)later);
        } else {
          nb = 64;
          carry_out = true;
        }
      }
    }
    const bool live = lane < nb;
    const uint64_t starts = nb == 64 ? diff : diff & ((1ull << nb) - 1ull);
    const uint32_t head = (uint32_t)head_lane(starts, lane);
    const uint32_t who = (uint32_t)lane << 12 | head << 18;
    while (b - start - rowbase >= (uint32_t)kMarkRows) {
      const uint32_t pos = reserve(1);
      if (lane == 0 && !L.off) L.ext[pos] = kMarkSource << 25;
      rowbase += kMarkRows;
    }
    const uint32_t row0 = b - start - rowbase, rowrel = row0 + (uint32_t)lane;

    // the row's visited vertices (all of them for lanes past the block, whose
    // items then never pass)
    unsigned long long used = 0;
    if constexpr (ROOT) {
      used = 1ull << (t.x[1] & 63u);
    } else {
#pragma unroll
      for (int i = 0; i < 4 * TW; ++i)
        used |= 1ull << ((t.x[1 + i / 4] >> ((i & 3) * 8)) & 63u);
    }
    if (!live) used = ~0ull;

    GM_GLOBAL const char *const vgrp = (GM_GLOBAL const char *)as_global(GM_ARG(vgrp));
    auto load_group = [&](uint32_t u) GM_INLINE -> Group { return *(GM_GLOBAL const Group *)(vgrp + (g + u * 8u)); };
    const int nsrc = ROOT ? 1 : H.nsrc;
    const char *srcs = meta + sizeof(CMetaHead);
    // (lanes past the block load too: their rows are the window's)
    auto load_src = [&](int j) GM_INLINE -> Group {
      if constexpr (ROOT) return load_group(t.x[1] & 63u);
      return load_group(image<TW>(t, cload<int>(srcs + j * (int)sizeof(CSource) + 16)));
    };
    auto load_next = [&](Group q) GM_INLINE -> Group {
      Group o = kEmptyGroup;
      if (next_of(q)) o = load_group(next_of(q));
      return o;
    };
    // a lane's items past its first two groups, one group at a time
    auto walk_on = [&](Group o, auto &&fn) GM_INLINE {
      uint32_t nx = next_of(o);
      while (nx) {
        const Group c = load_group(nx);
#pragma unroll
        for (int i = 0; i < 4; ++i) fn(item(c, i));
        nx = next_of(c);
      }
    };
    // count key for the segment of head lane h, list the entry at byte `at`
    // of the extent
    auto emit = [&](uint32_t at, uint32_t key, uint32_t entry, uint32_t h) GM_INLINE {
      if (!L.off) *(GM_GLOBAL uint32_t *)((GM_GLOBAL char *)L.ext + at) = entry;
      atomicOr(&kc[key].mask, 1ull << h);
      atomicAdd(&kc[key].emb, 1u);
    };

    Group P = load_src(0), Pn = nsrc > 1 ? load_src(1) : kEmptyGroup;
    Group O = load_next(P);
    for (int j = 0; j < nsrc; ++j) {
      // the groups of the next two sources are in flight while this one's
      // items are tested
      const Group Pnn = j + 2 < nsrc ? load_src(j + 2) : kEmptyGroup;
      const Group On = j + 1 < nsrc ? load_next(Pn) : kEmptyGroup;
      const bool more = __ballot(next_of(P) != 0) != 0;          // some vertex has more than four neighbours
      const bool deep = more && __ballot(next_of(O) != 0) != 0;  // more than eight

      // backward: from the rightmost vertex (source 0) to the images of the
      // path vertices that the pattern lists, a byte compare each against all
      // neighbours
      if constexpr (!ROOT) {
        if (j == 0 && H.nback) {
          const char *backs = srcs + nsrc * (int)sizeof(CSource);
          const uint32_t np = neighbours(P), no = neighbours(O);
          for (int q = 0; q < H.nback; ++q) {
            const int f = cload<int>(backs + q * (int)sizeof(CSource) + 16);
            const uint32_t v4 = image4<TW>(t, f);
            const uint32_t zp = zero_bytes(np ^ v4), zo = more ? zero_bytes(no ^ v4) : 0u;
            if (!deep && !__ballot((zp | zo) != 0)) continue;
            const CSource bk = cload<CSource>(backs + q * (int)sizeof(CSource));
            uint32_t lab = 63;
            if (zp | zo) lab = item(zp ? P : O, __builtin_ctz(zp ? zp : zo) >> 3) >> 6;
            if (deep) walk_on(O, [&](uint32_t x) GM_INLINE { lab = (x & 63u) == (v4 & 63u) ? min(lab, x >> 6) : lab; });
            const bool ok = live && ((bk.rule >> lab) & 1ull), kept = ok && ((bk.keep >> lab) & 1ull);
            n_pruned += ok && !kept ? 1u : 0u;
            const uint64_t m = __ballot(kept);
            if (m) {
              const uint32_t pos = reserve((uint32_t)__popcll(m)) + below(m);
              listed += (unsigned long long)__popcll(m);
              const uint32_t el = (lab * GM_ARG(inv_nvl)) >> 16;
              if (kept) emit(pos * 4u, (uint32_t)bk.kbase + el, (kBackSource + (uint32_t)q) << 25 | el << 19 | rowrel, head);
            }
          }
        }
      }

      // forward to unvisited neighbours whose label pair the source's rule
      // lets through
      typedef typename std::conditional<M32, uint32_t, unsigned long long>::type Mask;
      Mask rule, keep;
      uint32_t kbase, source = (uint32_t)j << 25;
      if constexpr (ROOT) {
        // from a vertex to neighbours of its label or a larger one; the
        // source's number is the label
        const uint32_t lu = (t.x[1] >> 8) & 0xFFu;
        const unsigned long long nl = ((1ull << GM_ARG(NVL)) - 1ull) & (~0ull << lu);
        rule = keep = (Mask)(nl * GM_ARG(lab_rep));
        kbase = lu * (uint32_t)GM_ARG(AR);
        source = lu << 25;
      } else {
        const CSource sc = cload<CSource>(srcs + j * (int)sizeof(CSource));
        rule = (Mask)sc.rule;
        keep = (Mask)sc.keep;
        kbase = (uint32_t)sc.kbase;
      }
      auto label_bit = [&](Mask x, uint32_t it) GM_INLINE -> uint32_t { return (uint32_t)(x >> (it >> 6 & (M32 ? 31u : 63u))); };
      auto bit = [&](Mask x, uint32_t it) GM_INLINE -> uint32_t { return label_bit(x, it) & ~(uint32_t)(used >> (it & 63u)) & 1u; };
      const Mask cut = (Mask)(rule & ~keep);
      uint32_t p[8], c = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = bit(keep, item(P, i));
      c = p[0] + p[1] + p[2] + p[3];
      if (cut) {
#pragma unroll
        for (int i = 0; i < 4; ++i) n_pruned += bit(cut, item(P, i));
      }
      if (more) {
#pragma unroll
        for (int i = 0; i < 4; ++i) p[4 + i] = bit(keep, item(O, i));
        c += p[4] + p[5] + p[6] + p[7];
        if (cut) {
#pragma unroll
          for (int i = 0; i < 4; ++i) n_pruned += bit(cut, item(O, i));
        }
      }
      if (deep)
        walk_on(O, [&](uint32_t x) GM_INLINE {
          n_pruned += bit(cut, x);
          c += bit(keep, x);
        });
      const uint32_t incl = wave_incl(c), total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      if (total) {
        listed += total;
        const uint32_t pos = reserve(total);
        uint32_t at = incl - c;
        if (!ROOT && total <= 64 && !deep) {
          // Through LDS, so that the list store and the two counter updates
          // are one instruction each for the whole source: a lane's items one
          // at a time were three to four of each, a sixth of the lanes busy.
          // (The root writes directly, 134 us against 145 this way for a batch
          // of 64 databases: its entries' sources and keys differ by lane.)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (p[i]) stage[at] = item(P, i) | who;
            at += p[i];
          }
          if (more) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              if (p[4 + i]) stage[at] = item(O, i) | who;
              at += p[4 + i];
            }
          }
          wave_sync();
          const uint32_t x = stage[lane], r = x >> 12 & 63u;  // (lanes past the items: stale, unused)
          if ((uint32_t)lane < total)
            emit((pos + (uint32_t)lane) * 4u, kbase + (x >> 6 & 63u), source | (x & 0xFFFu) << 13 | (row0 + r), x >> 18);
          wave_sync();
        } else {
          at = (at + pos) * 4u;
          const uint32_t tag = source | rowrel;
          auto put = [&](uint32_t x, uint32_t ok) GM_INLINE {
            if (ok) emit(at, kbase + (x >> 6), tag | x << 13, head);
            at += 4u * ok;
          };
          uint32_t m = 0;
#pragma unroll
          for (int i = 0; i < 8; ++i) m |= p[i] << i;
          while (m) {
            const int i = __builtin_ctz(m);
            m &= m - 1;
            put(item(i & 4 ? O : P, i & 3), 1u);
          }
          if (deep) walk_on(O, [&](uint32_t x) GM_INLINE { put(x, bit(keep, x)); });
        }
      }
      P = Pn;
      O = On;
      Pn = Pnn;
    }
    wave_sync();
    // support: one per segment of the block that holds the key, less a
    // segment carried in; a carried-out segment keeps its bit (head lane 0)
    // and is marked as counted in bit 31
    for (int i = lane; i < K; i += 64) {
      const unsigned long long m = kc[i].mask;
      if (m) {
        const uint32_t sv = kc[i].sup;
        const uint32_t kp = carry_out ? (uint32_t)(m & 1ull) : 0u;
        kc[i].sup = ((sv & 0x7FFFFFFFu) + (uint32_t)__popcll(m) - (sv >> 31)) | (kp << 31);
        kc[i].mask = kp;
      }
    }
    wave_sync();
    if (last) break;
    b += (uint32_t)nb;
    carry = carry_out;
    carry_g = (uint32_t)uniform((int)g);  // (a carried block is one segment)
  }
  // close the list, commit the counts to the chunk's replica and keep the
  // chunk's {key, first} records behind the list: the embeddings that the
  // replica had before are the place of the chunk's rows among the key's.
  // (The write took them from a cursor by an atomic of its own per chunk and
  // child, a million at a root level of 2.6 million rows: 69 us of the write,
  // now 28; 34 and 15 for 50,000 molecules, 138 and 90 on their small levels.)
  uint32_t nrec = 0;
  for (int i0 = 0; i0 < K; i0 += 64) nrec += (uint32_t)__popcll(__ballot(i0 + lane < K && kc[min(i0 + lane, K - 1)].emb != 0));
  GM_GLOBAL uint32_t *const ext0 = L.ext;
  const uint32_t n0 = L.used - 2u;
  uint32_t at = 0;
  if (nrec) {
    at = reserve(2u * nrec);
    const uint32_t n = L.ext == ext0 ? n0 : 0u;  // a new extent for the records closed the old one
    if (lane == 0 && !L.off) {
      L.ext[0] = n;
      L.ext[1] = kNone32;
    }
  }
  unsigned long long *const acc = GM_ARG(acc) + (int64_t)(gci & (uint32_t)(GM_ARG(rep) - 1)) * GM_ARG(nkeys) +
                                  (int64_t)(p - GM_ARG(p_base)) * K;
  uint32_t w = at;
  for (int i0 = 0; i0 < K; i0 += 64) {
    const int i = i0 + lane;
    const uint32_t e = i < K ? kc[i].emb : 0u;
    const uint64_t m = __ballot(e != 0);
    if (e) {
      const unsigned long long before =
          atomicAdd(&acc[i], ((unsigned long long)kc[i].sup << kSupShift) | (unsigned long long)e);
      if (!L.off) {
        const uint32_t q = w + 2u * below(m);
        L.ext[q] = (uint32_t)i;
        L.ext[q + 1] = (uint32_t)before;  // (a pattern of 2^32 embeddings and more is refused)
      }
    }
    w += 2u * (uint32_t)__popcll(m);
  }
  const unsigned long long w_pruned = wave_sum((unsigned long long)n_pruned);
  if (lane == 0) {
    GM_ARG(cchunks)[gci] = CChunk{(int64_t)(first + start), (uint64_t)(L.ext - as_global(GM_ARG(clist))) + at, L.off ? 0u : nrec};
    unsigned long long *const spread = GM_ARG(spread), *const line = spread + (gci & (kSpread - 1)) * kSpreadStride;
    if (listed + w_pruned) atomicAdd(&line[kSpreadCand], listed + w_pruned);
    if (w_pruned) atomicAdd(&line[kSpreadPruned], w_pruned);
    atomicMax(&line[kSpreadFill], (unsigned long long)nrec);
    stamp_end(spread, gci);
  }
}

// ------------------------------------------------------------------ WRITE
// One wave per chunk: the records name the chunk's keys; those that became
// children get a small index and a run of the child's rows (the replica's
// first row and the record's place in it), then the list is taken 64 entries at a time:
// an entry's child index comes from an LDS map of its key, its position is
// the child's run plus its rank among the window's entries of the same child
// (one ballot per index bit: a chunk's pattern has one to a few children),
// and the parent's row is read with the new vertex put in.  Chunks without
// children read no list.
constexpr int kWinUnroll = 2;  // windows whose loads are issued together

template <bool ROOT, int TW>
__global__ void __launch_bounds__(64, (TW <= 4 ? 8 : 5)) k_cwrite(StepArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t dyn[];
  const int K = (int)a.K;
  unsigned long long *const cbase = reinterpret_cast<unsigned long long *>(dyn);
  uint32_t *const crun = dyn + 2 * K;
  uint32_t *const skey = dyn + 3 * K;  // first key of every source number
  uint16_t *const cmap = reinterpret_cast<uint16_t *>(skey + 128);
  const int lane = threadIdx.x;
  const uint32_t gci = blockIdx.x;
  const CChunk c = cload<CChunk>(a.cchunks + gci);
  if (c.nrec == 0) return;
  const int p = ROOT ? (int)cload<uint4>(a.rtab + a.tab0 + gci).x : (int)cload<uint2>(a.ctab + a.tab0 + gci).x;
  for (int i = lane; i < K; i += 64) cmap[i] = 0;
  wave_sync();
  const int64_t kb = (int64_t)(p - a.p_base) * K;
  const int64_t rsel = (int64_t)(gci & (uint32_t)(a.rep - 1));
  int nchild = 0;
  for (uint32_t i0 = 0; i0 < c.nrec; i0 += 64) {
    const uint32_t i = i0 + lane;
    int32_t ch = -1;
    uint32_t key = 0, first = 0;
    if (i < c.nrec) {
      key = a.clist[c.rec + 2u * i];
      first = a.clist[c.rec + 2u * i + 1u];
      const int32_t v = a.sup[kb + key];
      ch = v < 0 ? -v - 1 : -1;
    }
    const uint64_t m = __ballot(ch >= 0);
    if (ch >= 0) {
      const int ix = nchild + (int)below(m);
      cmap[key] = (uint16_t)(ix + 1);
      cbase[ix] = a.cursor[(int64_t)ch * a.rep + rsel] + first;
      crun[ix] = 0;
    }
    nchild += __popcll(m);
  }
  if (nchild == 0) return;
  const int bits = nchild > 1 ? 32 - __clz(nchild - 1) : 0;
  constexpr int RW = 1 + TW;
  const int CW = a.CS >> 2;
  int nvp = 1;
  if constexpr (ROOT) {
    skey[lane] = (uint32_t)(lane * a.AR);
  } else {
    const char *meta = reinterpret_cast<const char *>(a.meta) + (int64_t)p * a.meta_stride;
    const CMetaHead H = cload<CMetaHead>(meta);
    const CSource *src = reinterpret_cast<const CSource *>(meta + sizeof(CMetaHead));
    nvp = H.nv;
    if (lane < H.nsrc) skey[lane] = (uint32_t)src[lane].kbase;
    if (lane < H.nback) skey[kBackSource + lane] = (uint32_t)src[H.nsrc + lane].kbase;
  }
  wave_sync();
  unsigned long long written = 0;
  uint32_t rowbase = 0;
  for (const uint32_t *ext = a.clist + (uint64_t)gci * a.page;;) {
    const uint32_t n = (uint32_t)uniform((int)ext[0]), next = (uint32_t)uniform((int)ext[1]);
    const uint32_t *list = ext + 2;
    for (uint32_t j0 = 0; j0 < n; j0 += 64 * kWinUnroll) {
      uint32_t e[kWinUnroll];
      int ix[kWinUnroll];
      CRow<TW> t[kWinUnroll];
#pragma unroll
      for (int u = 0; u < kWinUnroll; ++u) {
        const uint32_t j = j0 + u * 64 + lane;
        e[u] = j < n ? list[j] : kNone32;
      }
#pragma unroll
      for (int u = 0; u < kWinUnroll; ++u) {
        const uint32_t sid = e[u] >> 25;
        // entries past the end read as marks too, at the lanes behind all others
        const uint64_t marks = __ballot(sid == kMarkSource);
        uint32_t row = rowbase + (e[u] & 0x1FFFu);
        if (marks) {
          row += (uint32_t)kMarkRows * below(marks);
          rowbase += (uint32_t)kMarkRows * (uint32_t)__popcll(__ballot(sid == kMarkSource && e[u] != kNone32));
        }
        ix[u] = sid != kMarkSource ? (int)cmap[skey[sid] + (e[u] >> 19 & 63u)] - 1 : -1;
        if (ix[u] >= 0) {
          const uint32_t *src = a.crow + (c.start + (int64_t)row) * RW;
          __builtin_memcpy(&t[u], src, sizeof(t[u]));
        }
      }
#pragma unroll
      for (int u = 0; u < kWinUnroll; ++u) {
        const bool sel = ix[u] >= 0;
        const uint64_t active = __ballot(sel);
        if (!active) continue;
        written += (unsigned long long)__popcll(active);
        const uint32_t h = sel ? (uint32_t)ix[u] : 0u;
        uint64_t peers = active;
        for (int bit = 0; bit < bits; ++bit) {
          const bool hb = (h >> bit) & 1u;
          const uint64_t m = __ballot(sel && hb);
          peers &= hb ? m : ~m;
        }
        const uint32_t rank = below(peers);
        const uint32_t run = sel ? crun[h] : 0u;
        wave_sync();
        if (sel && rank == 0) crun[h] = run + (uint32_t)__popcll(peers);
        wave_sync();
        if (sel) {
          const unsigned long long pos = cbase[h] + (unsigned long long)run + rank;
          const uint32_t w = (e[u] >> 13) & 63u;
          const bool forward = e[u] >> 25 < kBackSource;
          if ((int64_t)pos < a.ccap) {
            uint32_t out[2 + TW];
            out[0] = t[u].x[0];
            const uint32_t v0 = t[u].x[1] & 0xFFu;
            const uint32_t fill = v0 * 0x01010101u;  // past the pattern's vertices: vertex 0 again
            if constexpr (ROOT) {
              out[1] = (fill & 0xFFFF00FFu) | w << 8;
              out[2] = fill;
            } else {
              const uint32_t put = w << ((nvp & 3) * 8), clear = ~(0xFFu << ((nvp & 3) * 8));
#pragma unroll
              for (int q = 0; q <= TW; ++q) {
                const uint32_t word = q < TW ? t[u].x[q < TW ? 1 + q : 1] : fill;
                out[1 + q] = forward && (nvp >> 2) == q ? (word & clear) | put : word;
              }
            }
            uint32_t *dst = a.crow_out + pos * (unsigned long long)(1 + CW);
            if (CW == 1) {
              __builtin_memcpy(dst, out, 8);
            } else if (TW >= 1 && CW == 2) {
              __builtin_memcpy(dst, out, 12);
            } else {
#pragma unroll
              for (int q = 0; q < 2 + TW; ++q)
                if (q <= CW) dst[q] = out[q];
              for (int q = 2 + TW; q <= CW; ++q) dst[q] = fill;
            }
          }
        }
      }
    }
    if (next == kNone32) break;
    ext = a.clist + (uint64_t)next * kListUnit;
  }
  if (lane == 0 && written)
    atomicAdd(&a.spread[(gci & (kSpread - 1)) * kSpreadStride + kSpreadWritten], written);
}

// ------------------------------------------------------------- CHILDREN
// After the children were chosen (see k_cursors): every (child, replica)'s
// cursor starts at its first row, and the children's chunk table is filled
// ({child, chunk of the child}).  `rep` lanes take one frequent key; t is the
// lane's index over all of them.
// With kByRecord the bases are the host's, in its mapped memory, per record and
// not per child: they are read beside the ids, a trip over the bus less.
template <bool kByRecord>
__device__ __forceinline__ void cursors_of(const StepArgs &a, int64_t t, const int32_t *fchild,
                                           const unsigned long long *row_base, const uint32_t *chunk_base, int64_t F) {
  const int64_t i = t / a.rep;
  const int r = (int)(t % a.rep);
  const bool ok = i < F;
  int64_t key = 0, at = 0;
  int32_t ch = -1;
  unsigned long long rows = 0, row0 = 0;
  uint32_t chunk0 = 0;
  if (ok) {
    ch = fchild[i];
    if (kByRecord && row_base) {  // (none: no child is written)
      row0 = row_base[i];
      chunk0 = chunk_base[i];
    }
    key = (int64_t)a.freq[4 * i];
    at = (int64_t)r * a.nkeys + key;
    rows = a.acc[at] & ((1ull << kSupShift) - 1);
  }
  unsigned long long sr = rows;  // inclusive scan over the key's replicas
  for (int o = 1; o < a.rep; o <<= 1) {
    const unsigned long long y = __shfl_up(sr, o, 64);
    if (r >= o) sr += y;
  }
  if (!ok) return;
  a.acc[at] = 0;
  if (ch < 0) return;
  if (r == 0) a.sup[key] = -(ch + 1);
  if (!kByRecord) {
    row0 = row_base[ch];
    chunk0 = chunk_base[ch];
  }
  a.cursor[(int64_t)ch * a.rep + r] = row0 + (sr - rows);
  const unsigned long long all = a.freq[4 * i + 2];
  const uint32_t n =
      chunk_count((uint32_t)all, chunk_nominal((uint32_t)a.child_blocks, (uint32_t)all, (uint32_t)a.freq[4 * i + 1]));
  uint2 *tab = a.child_tab + chunk0;
  for (uint32_t k = (uint32_t)r; k < n; k += (uint32_t)a.rep) tab[k] = make_uint2((uint32_t)ch, k);
}

__global__ void __launch_bounds__(256) k_ccursors(StepArgs a, const int32_t *fchild, const unsigned long long *row_base,
                                                  const uint32_t *chunk_base, int64_t F) {
  if (blockIdx.x == 0) clear_counters(a);
  cursors_of<true>(a, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, fchild, row_base, chunk_base, F);
}

// The children, chosen on the device: a tile of 1,024 records per workgroup,
// which adds up the records before its tile itself (a pass over at most a few
// ten thousand of them, cheaper than a launch for their sums).  The last
// tile's workgroup has the totals.  When the host chose, it read the list,
// numbered the children and sent ids, bases and metadata back: 100-350 us
// between k_reduce_list and the next k_clevel on the 100,000-transaction
// levels of 5,000-11,000 records; the host now waits for four words.
constexpr int kSelThreads = 1024;

struct SelSums {
  unsigned long long rows, dropped;
  uint32_t n, chunks, undecided;
  __device__ __forceinline__ void add(const SelSums &x) {
    rows += x.rows;
    dropped += x.dropped;
    n += x.n;
    chunks += x.chunks;
    undecided += x.undecided;
  }
};

struct SelRec {
  unsigned long long w, rows;
};
__device__ __forceinline__ SelRec sel_load(const StepArgs &a, uint32_t i) {
  return SelRec{a.freq[4ull * i + 1], a.freq[4ull * i + 2]};
}
template <bool ROOT>
__device__ __forceinline__ SelSums sel_of(const StepArgs &a, const SelRec &r) {
  const unsigned long long w = r.w, rows = r.rows;
  const uint32_t answer = (uint32_t)(w >> 32) & 0xFFu;  // k_canon_level's, + 1
  const bool sel = ROOT || answer == kCanonMin + 1;
  SelSums s;
  s.n = sel ? 1u : 0u;
  s.rows = sel ? rows : 0ull;
  s.dropped = sel ? 0ull : rows;
  uint32_t chunks = ROOT ? kChunksMany : (uint32_t)(w >> 40);  // k_canon_level's
  if (chunks == kChunksMany && sel)
    chunks = chunk_count((uint32_t)rows, chunk_nominal((uint32_t)a.child_blocks, (uint32_t)rows, (uint32_t)w));
  s.chunks = sel ? chunks : 0u;
  // (2^32 rows and more: for the host, which refuses them)
  s.undecided = (!ROOT && answer != kCanonMin + 1 && answer != kCanonNotMin + 1) || (sel && rows >> 32) ? 1u : 0u;
  return s;
}

__device__ __forceinline__ SelSums wave_total(const SelSums &x) {
  return SelSums{wave_sum(x.rows), wave_sum(x.dropped), wave_sum(x.n), wave_sum(x.chunks), wave_sum(x.undecided)};
}

template <bool ROOT>
__global__ void __launch_bounds__(kSelThreads) k_cselect(StepArgs a, CSelect c) {
  constexpr int kWaves = kSelThreads / 64;
  __shared__ SelSums s_before[kWaves], s_own[kWaves];
  const uint32_t F = min(*a.freq_count, a.freq_cap);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t tiles = F > 0 ? (F + kSelThreads - 1) / kSelThreads : 1u;
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    SelSums b{0, 0, 0, 0, 0};  // the lane's share of the records before the tile
    uint32_t q0 = 0;
    for (; q0 + 4 <= tile; q0 += 4) {  // four records' loads in flight
      SelRec r[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) r[u] = sel_load(a, (q0 + (uint32_t)u) * kSelThreads + threadIdx.x);
#pragma unroll
      for (int u = 0; u < 4; ++u) b.add(sel_of<ROOT>(a, r[u]));
    }
    for (; q0 < tile; ++q0) b.add(sel_of<ROOT>(a, sel_load(a, q0 * kSelThreads + threadIdx.x)));
    const uint32_t i = tile * kSelThreads + threadIdx.x;
    const SelSums x = i < F ? sel_of<ROOT>(a, sel_load(a, i)) : SelSums{0, 0, 0, 0, 0};
    // the wave's own sums: counts by ballot, the others with their scans
    unsigned long long tr;
    const unsigned long long er = wave_exclusive_scan<unsigned long long>(x.rows, tr);
    const uint64_t chosen = __ballot(x.n != 0);
    const uint32_t en = below(chosen), ic = wave_incl(x.chunks), ec = ic - x.chunks;
    const SelSums wx{tr, wave_sum(x.dropped), (uint32_t)__popcll(chosen), (uint32_t)__builtin_amdgcn_readlane((int)ic, 63),
                     (uint32_t)__popcll(__ballot(x.undecided != 0))};
    if (tile > 0) {
      const SelSums wb = wave_total(b);
      if (lane == 0) s_before[wave] = wb;
    }
    if (lane == 0) s_own[wave] = wx;
    __syncthreads();
    SelSums base{0, 0, 0, 0, 0};  // everything before this wave's records
#pragma unroll 4
    for (int q = 0; q < wave; ++q) base.add(s_own[q]);
    if (tile > 0) {
#pragma unroll 4
      for (int q = 0; q < kWaves; ++q) base.add(s_before[q]);
    }
    if (tile == tiles - 1 && wave == kWaves - 1) {  // base and this wave's own: the totals
      unsigned long long nv = 2;
      if (!ROOT) {
        nv = a.spread[lane * kSpreadStride + kSpreadNv];
        for (int o = 32; o > 0; o >>= 1) nv = max(nv, __shfl_xor(nv, o, 64));
      }
      if (lane == 0) {
        a.down[kTotChildren] = (unsigned long long)(base.n + wx.n) | (unsigned long long)(base.undecided + wx.undecided) << 32;
        a.down[kTotRows] = base.rows + wx.rows;
        a.down[kTotChunks] = (unsigned long long)(base.chunks + wx.chunks) | nv << 32;
        a.down[kTotDropped] = base.dropped + wx.dropped;
      }
    }
    if (i < F) c.fchild[i] = x.n ? (int32_t)(base.n + en) : -1;
    if (x.n) {
      const uint32_t ch = base.n + en;
      c.crec[ch] = i;
      c.row_base[ch] = base.rows + er;
      c.chunk_base[ch] = base.chunks + ec;
    }
    __syncthreads();
  }
}

// A frequent key as the tuple it adds to pattern p of nv vertices.
struct NewTuple {
  int from, to, el, tl;  // tl: the to vertex's label; root: of vertex 1
  int fl;                // root: of vertex 0
  bool forward;
};
template <bool ROOT>
__device__ __forceinline__ NewTuple tuple_of(const StepArgs &a, uint32_t x, int nv) {
  NewTuple t{0, 1, 0, 0, 0, true};
  const uint32_t NEL = (uint32_t)a.NEL, NVL = (uint32_t)a.NVL, SB = (uint32_t)a.S * NEL;
  if (ROOT || x >= SB) {
    const uint32_t y = ROOT ? x : x - SB, y1 = y / NVL;
    t.tl = (int)(y - y1 * NVL);
    const uint32_t f = y1 / NEL;
    t.el = (int)(y1 - f * NEL);
    if (ROOT) {
      t.fl = (int)f;
    } else {
      t.from = (int)f;
      t.to = nv;
    }
  } else {
    t.forward = false;
    t.from = nv - 1;
    t.to = (int)(x / NEL);
    t.el = (int)(x - (uint32_t)t.to * NEL);
  }
  return t;
}

// The 2-edge children's arms: (0,1,a,e1,b) then (1,2,b,e2,c) is the path with
// centre b, or (0,2,a,e2,c) with centre a.
__global__ void __launch_bounds__(256) k_ct2(StepArgs a, CMetaArgs m) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= m.C) return;
  const uint32_t key = (uint32_t)a.freq[4ull * m.crec[c]], p = key / (uint32_t)a.K;
  const CMetaHead H = *reinterpret_cast<const CMetaHead *>(reinterpret_cast<const char *>(a.meta) + (int64_t)p * a.meta_stride);
  const NewTuple t = tuple_of<false>(a, key - p * (uint32_t)a.K, H.nv);
  const uint32_t w = m.pcode[p];
  const int l0 = m.pvlab[(int64_t)p * a.S], l1 = m.pvlab[(int64_t)p * a.S + 1], e1 = (int)(w >> 16 & 0xFF);
  const bool at1 = t.from == 1;
  const int centre = at1 ? l1 : l0, arm1 = e1 * a.NVL + (at1 ? l0 : l1), arm2 = t.el * a.NVL + t.tl;
  unsigned long long *row = m.t2 + ((int64_t)H.job * a.NVL + centre) * a.AR;
  atomicOr(&row[arm1], 1ull << arm2);
  atomicOr(&row[arm2], 1ull << arm1);
}

// Cursors and chunk table (the first blocks), then the children's metadata,
// one wave per child: the child's code is its parent's plus the new tuple; the
// rightmost path follows the forward tuples from the last vertex to the root;
// a path vertex's rule (CSource) is a lane's.  The same facts as the host's
// make_cmeta.
struct ChildLds {
  unsigned long long vm[kCompactV];  // arms that go with every pattern edge at a vertex (path rule)
  unsigned long long fm[kCompactV];  // label pairs the parent extends by to a frequent pattern (sibling rule)
  unsigned long long bwd;            // vertices the rightmost one has an edge to
  uint32_t code[64];
  uint8_t lab[kCompactV], found[kCompactV], path[kCompactV];  // label; its forward tuple; rightmost path's tuples
};

template <bool ROOT>
__global__ void __launch_bounds__(256) k_cchildren(StepArgs a, CSelect c, CMetaArgs m, int64_t F, int64_t cursor_blocks) {
  __shared__ ChildLds lds[4];
  if ((int64_t)blockIdx.x < cursor_blocks) {
    if (blockIdx.x == 0) clear_counters(a);
    cursors_of<false>(a, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, c.fchild, c.row_base, c.chunk_base, F);
    return;
  }
  const int lane = threadIdx.x & 63;
  ChildLds &L = lds[threadIdx.x >> 6];
  const int64_t ci = ((int64_t)blockIdx.x - cursor_blocks) * 4 + (threadIdx.x >> 6);
  if (ci >= m.C) return;
  const unsigned long long *f = a.freq + 4ull * m.crec[ci];
  const uint32_t key = (uint32_t)f[0], p = key / (uint32_t)a.K;  // below 2^26: one piece
  int job = (int)p, nv = 2;
  if constexpr (!ROOT) {
    const CMetaHead H = *reinterpret_cast<const CMetaHead *>(reinterpret_cast<const char *>(a.meta) + (int64_t)p * a.meta_stride);
    job = H.job;
    nv = H.nv;
  }
  NewTuple t = tuple_of<ROOT>(a, key - p * (uint32_t)a.K, nv);
  const int cnv = !ROOT && t.forward ? nv + 1 : nv, n = m.len + 1;  // the child's vertices and tuples (n <= 64)
  // labels and code
  if (lane < a.CS) {
    int l = 0;
    if (lane < cnv) {
      if (ROOT)
        l = lane == 0 ? t.fl : t.tl;
      else
        l = lane < nv ? (int)m.pvlab[(int64_t)p * a.S + lane] : t.tl;
    }
    L.lab[lane] = (uint8_t)l;
    m.vlab[ci * a.CS + lane] = (uint8_t)l;
  }
  L.vm[lane] = ~0ull;
  if (lane == 0) L.bwd = 0;
  wave_sync();
  if (lane < n) {
    const int tl = ROOT || t.forward ? t.tl : (int)L.lab[t.to];
    const uint32_t w = lane < m.len ? m.pcode[(int64_t)p * m.len + lane]
                                    : (uint32_t)t.from | (uint32_t)t.to << 8 | (uint32_t)t.el << 16 | (uint32_t)tl << 24;
    L.code[lane] = w;
    m.code[ci * n + lane] = w;
    if (lane == 0) m.key[ci] = key;
    const int u = (int)(w & 0xFF), v = (int)(w >> 8 & 0xFF);
    if (u < v) L.found[v] = (uint8_t)lane;
    else if (u == cnv - 1) atomicOr(&L.bwd, 1ull << v);
    if (m.masks) {
      const int e = (int)(w >> 16 & 0xFF) * a.NVL;
      const unsigned long long *tj = m.t2 + (int64_t)job * a.NVL * a.AR;
      atomicAnd(&L.vm[u], tj[L.lab[u] * a.AR + e + L.lab[v]]);
      atomicAnd(&L.vm[v], tj[L.lab[v] * a.AR + e + L.lab[u]]);
    }
  }
  wave_sync();
  int nrm = 0;
  for (int v = cnv - 1; v > 0;) {
    const int k = L.found[v];
    if (lane == 0) L.path[nrm] = (uint8_t)k;
    ++nrm;
    v = (int)(L.code[k] & 0xFF);
  }
  wave_sync();
  // Sibling rule: an extension of the child at a vertex that the parent has on
  // its rightmost path was one of the parent's too (the same path edge there,
  // or an order rule that only got stricter), and its pattern contains the
  // parent's: it must have been frequent.  (The root's children: the edge must
  // be a frequent one.)
  L.fm[lane] = m.siblings && (ROOT || !t.forward || lane < nv) ? 0ull : ~0ull;
  wave_sync();
  auto frequent = [&](int64_t k) GM_INLINE -> bool {
    const int32_t s = a.sup[k];  // (negative: chosen, its id)
    return s < 0 || (s > 0 && s >= (a.minsup_job ? a.minsup_job[job] : a.minsup_one));
  };
  if (m.siblings) {
    // a lane per (vertex, label pair): the rightmost vertex, then the path's
    const int pairs = (nrm + 1) * a.AR;
    for (int x = lane; x < pairs; x += 64) {
      const int q = x / a.AR, b = x - q * a.AR, v = q ? (int)(L.code[L.path[q - 1]] & 0xFFu) : cnv - 1;
      bool ok = false;
      if constexpr (ROOT) {
        const int el = b / a.NVL, l = b - el * a.NVL, lv = L.lab[v];
        ok = frequent((int64_t)p * a.K + (min(lv, l) * a.NEL + el) * a.NVL + max(lv, l));
      } else if (v < nv) {
        ok = frequent((int64_t)p * a.K + a.S * a.NEL + v * a.AR + b);
      }
      if (ok) atomicOr(&L.fm[v], 1ull << b);
    }
  }
  wave_sync();
  // The same at a new vertex, by another pattern of the level: when the parent
  // is G + g and the child's new edge n starts at a vertex of G, G + n is in
  // the child too; if it is a pattern of this level (its code is minimal), what
  // it extends its last vertex by must have been frequent.
  int64_t cousin = -1;
  if constexpr (!ROOT) {
    if (m.pkey && t.forward) {
      const uint32_t pk = m.pkey[p], g = pk / m.pK;
      const int nvg = pk - g * m.pK >= (uint32_t)(m.pS * a.NEL) ? nv - 1 : nv;  // G's vertices
      if (t.from < nvg) {
        const int32_t r = m.psup[(int64_t)g * m.pK + m.pS * a.NEL + (t.from * a.NEL + t.el) * a.NVL + t.tl];
        if (r < 0) cousin = (int64_t)(-(r + 1)) * a.K;
      }
      if (cousin >= 0) {
        const uint64_t ok = __ballot(lane < a.AR && frequent(cousin + a.S * a.NEL + nvg * a.AR + lane));
        if (lane == 0) L.fm[cnv - 1] = ok;
      }
      wave_sync();
    }
  }
  // lane q: the rightmost path's edge q and its from vertex f
  const uint32_t w = lane < nrm ? L.code[L.path[lane]] : 0u;
  const int fv = (int)(w & 0xFF), e1 = (int)(w >> 16 & 0xFF), l1 = lane < nrm ? (int)L.lab[w >> 8 & 0xFF] : 0;
  const int lf = (int)L.lab[fv], rv = cnv - 1, minlabel = (int)L.lab[0], maxlabel = (int)L.lab[rv];
  const unsigned long long all = (1ull << a.NVL) - 1ull;
  auto from_label = [&](int x) GM_INLINE -> unsigned long long { return all & (~0ull << x); };
  // forward from f: (e, l) with l >= minlabel and (e1 < e or (e1 == e and l1 <= l))
  unsigned long long fr = 0, br = 0;
  if (lane < nrm) {
    if (e1 + 1 < a.NEL) fr = (from_label(minlabel) * a.lab_rep) & (~0ull << ((e1 + 1) * a.NVL));
    fr |= from_label(max(minlabel, l1)) << (e1 * a.NVL);
    // backward to f: (e, label of f) with e1 < e or (e1 == e and l1 <= maxlabel)
    const int e0 = l1 <= maxlabel ? e1 : e1 + 1;
    if (lane > 0 && !((L.bwd >> fv) & 1ull) && e0 < a.NEL) br = (a.lab_rep & (~0ull << (e0 * a.NVL))) << lf;
  }
  const uint64_t mf = __ballot(fr != 0), mb = __ballot(br != 0);
  const unsigned long long own = from_label(minlabel) * a.lab_rep;
  const int has_own = own || mb ? 1 : 0, nsrc = has_own + __popcll(mf), nback = __popcll(mb);
  const int SB = a.CS * a.NEL;
  char *out = m.meta + ci * m.meta_stride;
  CSource *src = reinterpret_cast<CSource *>(out + sizeof(CMetaHead));
  if (lane == 0) {
    CMetaHead h;
    h.job = job;
    h.nv = (uint8_t)cnv;
    h.nsrc = (uint8_t)nsrc;
    h.nback = (uint8_t)nback;
    h.flags = 0;
    h.row0 = c.row_base[ci];
    h.nrows = f[2];
    h.nom = chunk_nominal((uint32_t)a.child_blocks, (uint32_t)f[2], (uint32_t)f[1]);
    h.pad = 0;
    *reinterpret_cast<CMetaHead *>(out) = h;
    if (has_own) src[0] = CSource{own, own & L.vm[rv] & L.fm[rv], rv, SB + rv * a.AR};
  }
  if (fr) src[has_own + (int)below(mf)] = CSource{fr, fr & L.vm[fv] & L.fm[fv], fv, SB + fv * a.AR};
  if (br) {
    // a new arm at both ends: (e, label of f) at the rightmost vertex, (e, its label) at f
    const unsigned long long both = (L.vm[rv] >> lf) & (L.vm[fv] >> maxlabel) & a.lab_rep;
    unsigned long long keep = m.masks ? br & (both << lf) : br;
    if (!ROOT && m.siblings && (!t.forward || cousin >= 0)) {
      const int64_t at = t.forward ? cousin : (int64_t)p * a.K;
      for (int el = 0; el < a.NEL; ++el)
        if (!frequent(at + fv * a.NEL + el)) keep &= ~(1ull << (el * a.NVL + lf));
    }
    src[nsrc + (int)below(mb)] = CSource{br, keep, fv, fv * a.NEL};
  }
}

// A compact database of selected graphs gathered from a resident one: one
// workgroup per selected graph t copies its groups (their links are relative)
// and its root rows, rebased to the new first group dgb[t].
__global__ void __launch_bounds__(64) k_cgather(CGatherArgs g) {
  const int64_t t = blockIdx.x;
  const int32_t src = g.sel[t];
  const uint32_t b0 = g.ggb[src], nb = g.ggb[src + 1] - b0, d0 = g.dgb[t];
  const int32_t v0 = g.gvbase[src], nv = g.gvbase[src + 1] - v0, dv = g.dvb[t];
  for (uint32_t i = threadIdx.x; i < nb; i += blockDim.x) g.out_vgrp[d0 + i] = g.vgrp[b0 + i];
  for (int32_t i = threadIdx.x; i < nv; i += blockDim.x)
    g.out_rrows[dv + i] = make_uint2(d0 * 8u, g.rrows[v0 + i].y);
}

template <bool ROOT, int TW>
hipError_t level_of(const StepArgs &a, hipStream_t s) {
  const size_t lds = clevel_lds_bytes(a.K);
  if (a.AR <= 31)  // label pairs fit a 32-bit mask (bit 31 is the empty item's)
    hipLaunchKernelGGL((k_clevel<ROOT, TW, true>), dim3((unsigned)a.n_chunks), dim3(64), lds, s, a);
  else
    hipLaunchKernelGGL((k_clevel<ROOT, TW, false>), dim3((unsigned)a.n_chunks), dim3(64), lds, s, a);
  return hipGetLastError();
}

template <bool ROOT, int TW>
hipError_t write_of(const StepArgs &a, hipStream_t s) {
  hipLaunchKernelGGL((k_cwrite<ROOT, TW>), dim3((unsigned)a.n_chunks), dim3(64), (size_t)a.K * 14 + 512 + 16, s, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_clevel(const StepArgs &a, bool root, hipStream_t s) {
  if (a.n_chunks <= 0) return hipSuccess;
  if (root) return level_of<true, 1>(a, s);
  switch (a.S >> 2) {
    case 1: return level_of<false, 1>(a, s);
    case 2: return level_of<false, 2>(a, s);
    case 3: return level_of<false, 3>(a, s);
    case 4: return level_of<false, 4>(a, s);
    case 5: return level_of<false, 5>(a, s);
    case 6: return level_of<false, 6>(a, s);
    case 7: return level_of<false, 7>(a, s);
    case 8: return level_of<false, 8>(a, s);
    case 16: return level_of<false, 16>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_cwrite(const StepArgs &a, bool root, hipStream_t s) {
  if (a.n_chunks <= 0) return hipSuccess;
  if (root) return write_of<true, 1>(a, s);
  switch (a.S >> 2) {
    case 1: return write_of<false, 1>(a, s);
    case 2: return write_of<false, 2>(a, s);
    case 3: return write_of<false, 3>(a, s);
    case 4: return write_of<false, 4>(a, s);
    case 5: return write_of<false, 5>(a, s);
    case 6: return write_of<false, 6>(a, s);
    case 7: return write_of<false, 7>(a, s);
    case 8: return write_of<false, 8>(a, s);
    case 16: return write_of<false, 16>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_ccursors(const StepArgs &a, const int32_t *fchild, const unsigned long long *row_base,
                           const uint32_t *chunk_base, int64_t F, hipStream_t s) {
  if (F <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_ccursors, dim3((unsigned)((F * a.rep + 255) / 256)), dim3(256), 0, s, a, fchild, row_base,
                     chunk_base, F);
  return hipGetLastError();
}

hipError_t launch_cselect(const StepArgs &a, const CSelect &c, bool root, uint32_t expect, hipStream_t s) {
  // a workgroup per tile of the records expected, any number covers them
  const unsigned g = std::max(1u, std::min(256u, (expect + kSelThreads - 1) / kSelThreads));
  if (root)
    hipLaunchKernelGGL(k_cselect<true>, dim3(g), dim3(kSelThreads), 0, s, a, c);
  else
    hipLaunchKernelGGL(k_cselect<false>, dim3(g), dim3(kSelThreads), 0, s, a, c);
  return hipGetLastError();
}

hipError_t launch_cchildren(const StepArgs &a, const CSelect &c, const CMetaArgs &m, bool root, int64_t F, hipStream_t s) {
  if (F <= 0) return hipSuccess;
  if (m.C > 0 && m.len + 1 > 64) return hipErrorInvalidValue;
  const int64_t cb = (F * a.rep + 255) / 256;
  const unsigned g = (unsigned)(cb + (m.C + 3) / 4);
  if (root)
    hipLaunchKernelGGL(k_cchildren<true>, dim3(g), dim3(256), 0, s, a, c, m, F, cb);
  else
    hipLaunchKernelGGL(k_cchildren<false>, dim3(g), dim3(256), 0, s, a, c, m, F, cb);
  return hipGetLastError();
}

hipError_t launch_ct2(const StepArgs &a, const CMetaArgs &m, hipStream_t s) {
  if (m.C <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_ct2, dim3((unsigned)((m.C + 255) / 256)), dim3(256), 0, s, a, m);
  return hipGetLastError();
}

hipError_t launch_cgather(const CGatherArgs &g, hipStream_t s) {
  if (g.n_sel <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_cgather, dim3((unsigned)g.n_sel), dim3(64), 0, s, g);
  return hipGetLastError();
}

}  // namespace gm
