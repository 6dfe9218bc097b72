// canon.hip -- minimum DFS code check on the device (gfx950, wave64).
//
// One 64-lane wave decides for one DFS code C of n edges whether C is the
// code that gSpan's greedy is_min grows on C's own pattern graph
// (src/gspan/ismin.cpp:36-140; src/globals/dfs_ismin.cpp:23-160), with the
// same steps as the host check in canonical.cpp:
//   1. the root tuple is the smallest (fromlabel, elabel, tolabel) over the
//      directed pattern edges with fromlabel <= tolabel (not compared with
//      C[0]);
//   2. with the embeddings of the code grown so far, the next tuple is the
//      backward edge from the rightmost vertex to the rightmost-path vertex
//      nearest the root that an embedding reaches (smallest elabel, under
//      get_backward's order rule, graph_types.cpp:389-413); else the
//      smallest (elabel, tolabel) forward edge from the rightmost vertex
//      (graph_types.cpp:337-355); else from the deepest rightmost-path
//      vertex that has one (graph_types.cpp:305-323);
//   3. the first tuple that differs from C answers "not minimal"; reaching
//      the end answers "minimal".
// The pattern graph (an edge-id matrix and neighbour masks) and two
// embedding lists (vertex map, used-edge and used-vertex masks) live in
// LDS; the lanes take the embeddings, and each step's smallest tuple is a
// wave-wide minimum.  A code beyond the LDS capacity (more than kCanonE
// edges, kCanonV - 1 vertices, kCanonCap embeddings, or a repeated edge)
// is left undecided (kCanonHost) for the host check.  Explicit codes (any
// labels) take canon_core; a level's own codes, with dense labels, canon_level.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kernels.hpp"
#include "wave.hpp"

namespace gm {
namespace {

constexpr int kCV = kCanonV;
constexpr int kCE = kCanonE;
constexpr int kCap = kCanonCap;
constexpr unsigned long long kNone = ~0ull;
constexpr uint32_t kNoKey = ~0u;

struct Emb {
  unsigned long long used, vused;  // pattern edges / vertices matched
  uint8_t map[kCV];                // code vertex -> pattern vertex
};
static_assert(sizeof(Emb) == 16 + kCV && kCV % 8 == 0, "Emb layout");

struct CanonLds {
  unsigned long long nb[kCV];  // neighbour mask per pattern vertex
  int32_t lab[kCV];            // vertex labels
  int32_t wel[kCE], wtl[kCE];  // C: edge label, to label per tuple
  uint8_t wfrom[kCE], wto[kCE];
  uint8_t rm[kCE];             // rightmost path of the code grown so far, last forward tuple first
  alignas(4) int8_t eid[kCV * kCV];  // tuple index of the edge between two vertices, -1: none
  int32_t nrm;
  Emb emb[2][kCap];
};

// word copy of an embedding (a struct copy goes through private memory)
__device__ __forceinline__ void copy_emb(Emb &dst, const Emb &src) {
  const unsigned long long *s = reinterpret_cast<const unsigned long long *>(&src);
  unsigned long long *d = reinterpret_cast<unsigned long long *>(&dst);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(Emb) / 8); ++k) d[k] = s[k];
}

// (a, b) as one unsigned key with the order of the signed pair
__device__ __forceinline__ unsigned long long pair_key(int32_t a, int32_t b) {
  return ((unsigned long long)((uint32_t)a ^ 0x80000000u) << 32) | (unsigned long long)((uint32_t)b ^ 0x80000000u);
}
__device__ __forceinline__ int32_t key_hi(unsigned long long k) { return (int32_t)((uint32_t)(k >> 32) ^ 0x80000000u); }
__device__ __forceinline__ int32_t key_lo(unsigned long long k) { return (int32_t)((uint32_t)k ^ 0x80000000u); }

__device__ __forceinline__ unsigned long long wave_min64(unsigned long long v) {
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long t = __shfl_xor(v, o, 64);
    v = t < v ? t : v;
  }
  return v;
}

__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

__device__ __forceinline__ uint64_t below(int lane) { return (1ull << lane) - 1ull; }

// The grown code's tuple i: tuple 0 is the chosen root (0, 1, el0); the
// later ones equal C's (the check stops at the first difference).
struct Grown {
  int32_t el0;
  __device__ __forceinline__ int from(const CanonLds &L, int i) const { return i ? L.wfrom[i] : 0; }
  __device__ __forceinline__ int to(const CanonLds &L, int i) const { return i ? L.wto[i] : 1; }
  __device__ __forceinline__ int32_t el(const CanonLds &L, int i) const { return i ? L.wel[i] : el0; }
};

// The check of C (wfrom/wto/wel/wtl for n tuples, lab for nv vertices, set
// by the caller).  Every lane returns the same answer.
__device__ __forceinline__ int canon_core(CanonLds &L, int n, int nv, int lane) {
  if (n <= 1) return kCanonMin;
  if (n > kCE || nv > kCV - 1) return kCanonHost;
  {
    uint32_t *e32 = reinterpret_cast<uint32_t *>(L.eid);
    for (int i = lane; i < kCV * kCV / 4; i += 64) e32[i] = 0xFFFFFFFFu;
  }
  for (int v = lane; v < kCV; v += 64) L.nb[v] = 0;
  __syncthreads();
  // the pattern graph, one tuple per lane; a tuple outside nv vertices or a
  // repeated vertex pair leaves the code to the host
  int bad = 0;
  for (int i = lane; i < n; i += 64) {
    const int a = L.wfrom[i], b = L.wto[i];
    if (a >= nv || b >= nv || a == b) {
      bad = 1;
      continue;
    }
    L.eid[a * kCV + b] = (int8_t)i;
    L.eid[b * kCV + a] = (int8_t)i;
    atomicOr(&L.nb[a], 1ull << b);
    atomicOr(&L.nb[b], 1ull << a);
  }
  __syncthreads();
  for (int i = lane; i < n; i += 64) {
    const int a = L.wfrom[i], b = L.wto[i];
    if (a < nv && b < nv && a != b && (L.eid[a * kCV + b] != i || L.eid[b * kCV + a] != i)) bad = 1;
  }
  if (__ballot(bad != 0)) return kCanonHost;

  // 1. root tuple: smallest (fromlabel, elabel), then smallest tolabel
  unsigned long long k1 = kNone;
  for (int d = lane; d < 2 * n; d += 64) {
    const int i = d >> 1;
    const int u = (d & 1) ? L.wto[i] : L.wfrom[i], v = (d & 1) ? L.wfrom[i] : L.wto[i];
    if (L.lab[u] <= L.lab[v]) {
      const unsigned long long k = pair_key(L.lab[u], L.wel[i]);
      k1 = k < k1 ? k : k1;
    }
  }
  k1 = wave_min64(k1);
  const int32_t bfl = key_hi(k1), bel = key_lo(k1);
  unsigned long long k2 = kNone;
  for (int d = lane; d < 2 * n; d += 64) {
    const int i = d >> 1;
    const int u = (d & 1) ? L.wto[i] : L.wfrom[i], v = (d & 1) ? L.wfrom[i] : L.wto[i];
    if (L.lab[u] == bfl && L.wel[i] == bel && L.lab[u] <= L.lab[v]) {
      const unsigned long long k = pair_key(L.lab[v], 0);
      k2 = k < k2 ? k : k2;
    }
  }
  k2 = wave_min64(k2);
  const int32_t btl = key_hi(k2);
  int ncur = 0;
  for (int base = 0; base < 2 * n; base += 64) {
    const int d = base + lane;
    bool hit = false;
    int u = 0, v = 0, i = 0;
    if (d < 2 * n) {
      i = d >> 1;
      u = (d & 1) ? L.wto[i] : L.wfrom[i];
      v = (d & 1) ? L.wfrom[i] : L.wto[i];
      hit = L.lab[u] == bfl && L.wel[i] == bel && L.lab[v] == btl;
    }
    const unsigned long long m = __ballot(hit);
    if (ncur + __popcll(m) > kCap) return kCanonHost;
    if (hit) {
      Emb &e = L.emb[0][ncur + __popcll(m & below(lane))];
      e.used = 1ull << i;
      e.vused = (1ull << u) | (1ull << v);
      e.map[0] = (uint8_t)u;
      e.map[1] = (uint8_t)v;
    }
    ncur += __popcll(m);
  }
  const Grown g{bel};
  const int32_t minlabel = bfl;
  int cur = 0;

  for (int mpos = 1; mpos < n; ++mpos) {
    __syncthreads();
    if (lane == 0) {  // rightmost path of tuples [0, mpos) (dfs_code.cpp:75-90)
      int nrm = 0, old_from = -1;
      for (int i = mpos - 1; i >= 0; --i) {
        const int f = g.from(L, i), t = g.to(L, i);
        if (f < t && (nrm == 0 || old_from == t)) {
          L.rm[nrm++] = (uint8_t)i;
          old_from = f;
        }
      }
      L.nrm = nrm;
    }
    __syncthreads();
    const int nrm = L.nrm;
    const int maxtoc = g.to(L, L.rm[0]);
    if (maxtoc + 1 >= kCV) return kCanonHost;
    const Emb *E = L.emb[cur];
    Emb *X = L.emb[cur ^ 1];

    // backward edges from the rightmost vertex: the path vertex nearest the
    // root that any embedding reaches, then the smallest edge label -- one
    // minimum of (nrm - path index, elabel) over every embedding's first hit
    // from the root end
    unsigned long long bk = kNone;
    for (int j = lane; j < ncur; j += 64) {
      const int r = E[j].map[maxtoc];
      for (int ii = nrm - 1; ii >= 1; --ii) {
        const int e1 = L.rm[ii];
        const int id = L.eid[r * kCV + E[j].map[g.from(L, e1)]];
        if (id < 0 || ((E[j].used >> id) & 1ull)) continue;
        const int32_t le = L.wel[id], e1el = g.el(L, e1);
        if (e1el < le || (e1el == le && L.lab[E[j].map[g.to(L, e1)]] <= L.lab[r])) {
          const unsigned long long k = pair_key(nrm - ii, le);
          bk = k < bk ? k : bk;
          break;
        }
      }
    }
    bk = wave_min64(bk);
    if (bk != kNone) {
      const int ii = nrm - key_hi(bk);
      const int32_t bl = key_lo(bk);
      const int e1 = L.rm[ii];
      const int e1f = g.from(L, e1), e1t = g.to(L, e1);
      const int32_t e1el = g.el(L, e1);
      if (!(L.wfrom[mpos] == maxtoc && L.wto[mpos] == e1f && L.wel[mpos] == bl)) return kCanonNotMin;
      int nn = 0;
      for (int base = 0; base < ncur; base += 64) {
        const int j = base + lane;
        bool hit = false;
        int id = 0;
        if (j < ncur) {
          const int r = E[j].map[maxtoc], target = E[j].map[e1f];
          id = L.eid[r * kCV + target];
          if (id >= 0 && !((E[j].used >> id) & 1ull)) {
            const int32_t le = L.wel[id];
            hit = le == bl && (e1el < le || (e1el == le && L.lab[E[j].map[e1t]] <= L.lab[r]));
          }
        }
        const unsigned long long m = __ballot(hit);
        if (hit) {
          Emb &x = X[nn + __popcll(m & below(lane))];
          copy_emb(x, E[j]);
          x.used |= 1ull << id;
        }
        nn += __popcll(m);
      }
      ncur = nn;
      cur ^= 1;
      continue;
    }

    // forward edges: from the rightmost vertex (source level -1), else from
    // the deepest rightmost-path vertex that has one (level = path index);
    // first the smallest level any embedding has, then the smallest
    // (elabel, tolabel) at that level.  cand(j, lvl, w) is the rule.
    auto fwd_ok = [&](int j, int lvl, int w, int32_t &le, int32_t &tl) -> bool {
      tl = L.lab[w];
      if (minlabel > tl) return false;
      if (lvl < 0) {
        le = L.wel[L.eid[E[j].map[maxtoc] * kCV + w]];
        return true;
      }
      const int e = L.rm[lvl];
      const int u = E[j].map[g.from(L, e)], x = E[j].map[g.to(L, e)];
      if (w == x) return false;
      le = L.wel[L.eid[u * kCV + w]];
      const int32_t eel = g.el(L, e);
      return eel < le || (eel == le && L.lab[x] <= tl);
    };
    auto src_of = [&](int j, int lvl) -> int { return lvl < 0 ? E[j].map[maxtoc] : E[j].map[g.from(L, L.rm[lvl])]; };
    int lv_lane = 1 << 30;
    for (int j = lane; j < ncur; j += 64) {
      for (int lvl = -1; lvl < nrm && lvl < lv_lane; ++lvl) {
        unsigned long long c = L.nb[src_of(j, lvl)] & ~E[j].vused;
        bool any = false;
        while (c && !any) {
          const int w = __ffsll((long long)c) - 1;
          c &= c - 1;
          int32_t le, tl;
          any = fwd_ok(j, lvl, w, le, tl);
        }
        if (any) lv_lane = lvl;
      }
    }
    int lvl = lv_lane;
    for (int o = 32; o > 0; o >>= 1) lvl = min(lvl, __shfl_xor(lvl, o, 64));
    if (lvl >= nrm) return kCanonMin;  // nothing left to grow: the pattern is covered
    unsigned long long fk = kNone;
    for (int j = lane; j < ncur; j += 64) {
      unsigned long long c = L.nb[src_of(j, lvl)] & ~E[j].vused;
      while (c) {
        const int w = __ffsll((long long)c) - 1;
        c &= c - 1;
        int32_t le, tl;
        if (fwd_ok(j, lvl, w, le, tl)) {
          const unsigned long long k = pair_key(le, tl);
          fk = k < fk ? k : fk;
        }
      }
    }
    fk = wave_min64(fk);
    const int newfrom = lvl < 0 ? maxtoc : g.from(L, L.rm[lvl]);
    const int32_t bel2 = key_hi(fk), btl2 = key_lo(fk);
    if (!(L.wfrom[mpos] == newfrom && L.wto[mpos] == maxtoc + 1 && L.wel[mpos] == bel2 && L.wtl[mpos] == btl2))
      return kCanonNotMin;
    // every embedding's images of the new edge: count, scan, write
    int nn = 0;
    for (int base = 0; base < ncur; base += 64) {
      const int j = base + lane;
      unsigned long long hits = 0;
      if (j < ncur) {
        unsigned long long c = L.nb[src_of(j, lvl)] & ~E[j].vused;
        while (c) {
          const int w = __ffsll((long long)c) - 1;
          c &= c - 1;
          int32_t le, tl;
          if (fwd_ok(j, lvl, w, le, tl) && le == bel2 && tl == btl2) hits |= 1ull << w;
        }
      }
      const int cnt = __popcll(hits);
      const int incl = wave_incl_scan(cnt, lane);
      const int total = __shfl(incl, 63, 64);
      if (nn + total > kCap) return kCanonHost;
      int pos = nn + incl - cnt;
      if (j < ncur) {
        const int u = src_of(j, lvl);
        while (hits) {
          const int w = __ffsll((long long)hits) - 1;
          hits &= hits - 1;
          Emb &y = X[pos++];
          copy_emb(y, E[j]);
          y.map[maxtoc + 1] = (uint8_t)w;
          y.used |= 1ull << L.eid[u * kCV + w];
          y.vused |= 1ull << w;
        }
      }
      nn += total;
    }
    ncur = nn;
    cur ^= 1;
  }
  return kCanonMin;
}

// The same check for a level's own codes: dense labels (a byte each), LDS laid
// out for the level's length, so that 32 waves fit a CU from 6 edges down (16
// with the fixed layout above), every embedding and path vertex of a step at
// once, a lane per pair, and the step's smallest tuple as one 32-bit minimum
// (path place | edge label | vertex label) in data-parallel primitives.  What
// bounds it is a code's chain of LDS reads.  With a lane per embedding walking
// the path, 64-bit minima through LDS and one lane finding the rightmost path
// again for every tuple, a level of 23,000 2-edge codes took 73 us and the
// twelve levels of 100,000 transactions 550 us; now 46 and 288 us.
//
// Sizes for codes of n edges: VS bytes of vertex map (the code's vertices and
// the next one, whole words of 8).
struct LevelLds {
  int vs, eb;       // vertex places, bytes of an embedding {used, vused, map}
  size_t emb, nb, w, rm, lab, eid, bytes;
};
__host__ __device__ inline LevelLds level_lds(int n) {
  LevelLds l;
  l.vs = ((n + 2 < kCV ? n + 2 : kCV) + 7) & ~7;
  l.eb = 16 + l.vs;
  l.emb = 0;
  l.nb = l.emb + 2 * (size_t)kCap * l.eb;
  l.w = l.nb + 8 * (size_t)l.vs;
  l.rm = l.w + 4 * (size_t)n;
  l.lab = l.rm + 4 * (size_t)n;
  l.eid = l.lab + (size_t)l.vs;
  l.eid = (l.eid + 7) & ~size_t(7);
  l.bytes = l.eid + (size_t)l.vs * l.vs;
  return l;
}

__device__ __forceinline__ uint32_t wave_min32(uint32_t x) {
  auto step = [&](uint32_t y) __attribute__((always_inline)) { x = y < x ? y : x; };
  step((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)x, 0x111, 0xF, 0xF, false));  // row_shr:1
  step((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)x, 0x112, 0xF, 0xF, false));
  step((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)x, 0x114, 0xF, 0xF, false));
  step((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)x, 0x118, 0xF, 0xF, false));
  step((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)x, 0x142, 0xA, 0xF, false));  // row_bcast:15
  step((uint32_t)__builtin_amdgcn_update_dpp(-1, (int)x, 0x143, 0xC, 0xF, false));  // row_bcast:31
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// w: n tuples from | to << 8 | elabel << 16 | tolabel << 24, lab: nv labels.
__device__ __forceinline__ int canon_level(char *lds, const LevelLds &l, int n, int nv, int lane) {
  if (n <= 1) return kCanonMin;
  if (n > kCE || nv > kCV - 1) return kCanonHost;
  unsigned long long *const nb = reinterpret_cast<unsigned long long *>(lds + l.nb);
  const uint32_t *const w = reinterpret_cast<const uint32_t *>(lds + l.w);
  uint32_t *const rm = reinterpret_cast<uint32_t *>(lds + l.rm);  // rightmost path, last forward tuple first
  const uint8_t *const lab = reinterpret_cast<const uint8_t *>(lds + l.lab);
  int8_t *const eid = reinterpret_cast<int8_t *>(lds + l.eid);
  const int vs = l.vs;
  struct Ref {
    char *p;
    __device__ __forceinline__ unsigned long long &used() const { return reinterpret_cast<unsigned long long *>(p)[0]; }
    __device__ __forceinline__ unsigned long long &vused() const { return reinterpret_cast<unsigned long long *>(p)[1]; }
    __device__ __forceinline__ uint8_t &map(int i) const { return reinterpret_cast<uint8_t *>(p + 16)[i]; }
  };
  int cur = 0;
  auto emb = [&](int half, int j) { return Ref{lds + l.emb + (half * kCap + j) * l.eb}; };

  for (int i = lane; i < vs * vs / 8; i += 64) reinterpret_cast<unsigned long long *>(eid)[i] = ~0ull;
  for (int v = lane; v < vs; v += 64) nb[v] = 0;
  wave_sync();
  // the pattern graph, one tuple per lane; a tuple outside nv vertices or a
  // repeated vertex pair leaves the code to the host
  bool bad = false;
  const uint32_t own = lane < n ? w[lane] : 0u;
  const int oa = (int)(own & 0xFFu), ob = (int)(own >> 8 & 0xFFu);
  if (lane < n) {
    bad = oa >= nv || ob >= nv || oa == ob;
    if (!bad) {
      eid[oa * vs + ob] = (int8_t)lane;
      eid[ob * vs + oa] = (int8_t)lane;
      atomicOr(&nb[oa], 1ull << ob);
      atomicOr(&nb[ob], 1ull << oa);
    }
  }
  wave_sync();
  if (lane < n && !bad) bad = eid[oa * vs + ob] != lane || eid[ob * vs + oa] != lane;
  if (__ballot(bad)) return kCanonHost;

  // 1. root tuple: the smallest (fromlabel, elabel, tolabel), and its images
  uint32_t rk = kNoKey;
  const uint32_t oel = own >> 16 & 0xFFu;
  uint32_t la = 0, lb = 0;
  if (lane < n) {
    la = lab[oa];
    lb = lab[ob];
    rk = min(la, lb) << 16 | oel << 8 | max(la, lb);
  }
  rk = wave_min32(rk);
  const uint32_t minlabel = rk >> 16, rel = rk >> 8 & 0xFFu, rtl = rk & 0xFFu;
  int ncur = 0;
  {
    const bool e = lane < n && oel == rel, h0 = e && la == minlabel && lb == rtl, h1 = e && lb == minlabel && la == rtl;
    const uint64_t m0 = __ballot(h0), m1 = __ballot(h1);
    ncur = __popcll(m0) + __popcll(m1);
    if (ncur > kCap) return kCanonHost;
    const int p0 = __popcll(m0 & below(lane)) + __popcll(m1 & below(lane));
    auto put = [&](int pos, int u, int v) {
      const Ref x = emb(0, pos);
      x.used() = 1ull << lane;
      x.vused() = 1ull << u | 1ull << v;
      x.map(0) = (uint8_t)u;
      x.map(1) = (uint8_t)v;
    };
    if (h0) put(p0, oa, ob);
    if (h1) put(p0 + (h0 ? 1 : 0), ob, oa);
  }
  if (lane == 0) rm[0] = 0u | 1u << 8 | rel << 16;
  int nrm = 1, maxtoc = 1;

  for (int mpos = 1; mpos < n; ++mpos) {
    wave_sync();
    const uint32_t cw = (uint32_t)__builtin_amdgcn_readfirstlane((int)w[mpos]);
    const bool last = mpos == n - 1;
    // backward edges from the rightmost vertex: the path vertex nearest the
    // root that any embedding reaches, then the smallest edge label
    auto back = [&](const Ref &E, uint32_t path, int &id, uint32_t &le) {
      const int r = E.map(maxtoc);
      id = eid[r * vs + E.map((int)(path & 0xFFu))];
      if (id < 0 || ((E.used() >> id) & 1ull)) return false;
      le = w[id] >> 16 & 0xFFu;
      const uint32_t pel = path >> 16 & 0xFFu;
      return pel < le || (pel == le && lab[E.map((int)(path >> 8 & 0xFFu))] <= lab[r]);
    };
    uint32_t key = kNoKey;
    if (nrm > 1) {
      const int d = nrm - 1, pairs = ncur * d;
      const uint32_t inv = (1u << 20) / (uint32_t)d + 1u;  // exact quotients: at most 64 x 40 pairs
      for (int q = lane; q < pairs; q += 64) {
        const int j = (int)((uint32_t)q * inv >> 20), ii = 1 + q - j * d;
        int id;
        uint32_t le = 0;
        if (back(emb(cur, j), rm[ii], id, le)) key = min(key, (uint32_t)(nrm - ii) << 8 | le);
      }
      key = wave_min32(key);
    }
    if (key != kNoKey) {
      const uint32_t path = (uint32_t)__builtin_amdgcn_readfirstlane((int)rm[nrm - (int)(key >> 8)]);
      const uint32_t bl = key & 0xFFu;
      if ((cw & 0xFFFFFFu) != ((uint32_t)maxtoc | (path & 0xFFu) << 8 | bl << 16)) return kCanonNotMin;
      if (last) return kCanonMin;
      // the embeddings with that edge, moved up in place (at most 64: a lane
      // each, read before any is written)
      int id = 0;
      uint32_t le = 0;
      const bool hit = lane < ncur && back(emb(cur, lane), path, id, le) && le == bl;
      const uint64_t m = __ballot(hit);
      const Ref x = emb(cur, __popcll(m & below(lane))), e = emb(cur, lane);
      for (int k = 0; k < l.eb / 8; ++k) {
        unsigned long long v = 0;
        if (hit) v = reinterpret_cast<unsigned long long *>(e.p)[k];
        if (k == 0) v |= 1ull << id;
        wave_sync();
        if (hit) reinterpret_cast<unsigned long long *>(x.p)[k] = v;
        wave_sync();
      }
      ncur = __popcll(m);
      continue;
    }

    // forward edges: from the rightmost vertex (place 0), else from the
    // deepest path vertex that has one (place 1 + path index); then the
    // smallest (elabel, tolabel)
    auto source = [&](const Ref &E, int place) { return (int)E.map(place ? (int)(rm[place - 1] & 0xFFu) : maxtoc); };
    // the labels of the edge to v, if the rules let it through
    auto forward = [&](const Ref &E, int place, int u, int v, uint32_t &lw) {
      const uint32_t tl = lab[v], le = w[eid[u * vs + v]] >> 16 & 0xFFu;
      lw = le << 8 | tl;
      if (minlabel > tl) return false;
      if (place == 0) return true;
      const uint32_t path = rm[place - 1], pel = path >> 16 & 0xFFu;
      const int x = E.map((int)(path >> 8 & 0xFFu));
      return v != x && (pel < le || (pel == le && lab[x] <= tl));
    };
    {
      const int d = nrm + 1, pairs = ncur * d;
      const uint32_t inv = (1u << 20) / (uint32_t)d + 1u;
      for (int q = lane; q < pairs; q += 64) {
        const int j = (int)((uint32_t)q * inv >> 20), place = q - j * d;
        const Ref E = emb(cur, j);
        const int u = source(E, place);
        for (unsigned long long c = nb[u] & ~E.vused(); c; c &= c - 1) {
          uint32_t lw;
          if (forward(E, place, u, __ffsll((long long)c) - 1, lw)) key = min(key, (uint32_t)place << 16 | lw);
        }
      }
      key = wave_min32(key);
    }
    if (key == kNoKey) return kCanonMin;  // nothing left to grow: the pattern is covered
    const int place = (int)(key >> 16);
    const uint32_t path0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)rm[place ? place - 1 : 0]);
    const uint32_t from = place ? path0 & 0xFFu : (uint32_t)maxtoc;
    if (cw != (from | (uint32_t)(maxtoc + 1) << 8 | (key >> 8 & 0xFFu) << 16 | key << 24)) return kCanonNotMin;
    if (last) return kCanonMin;
    // every embedding's images of the new edge: count, scan, write
    unsigned long long hits = 0;
    int u = 0;
    const Ref E = emb(cur, lane);
    if (lane < ncur) {
      u = source(E, place);
      for (unsigned long long c = nb[u] & ~E.vused(); c; c &= c - 1) {
        const int v = __ffsll((long long)c) - 1;
        uint32_t lw;
        if (forward(E, place, u, v, lw) && lw == (key & 0xFFFFu)) hits |= 1ull << v;
      }
    }
    const int cnt = __popcll(hits);
    const int incl = wave_incl_scan(cnt, lane);
    const int total = __builtin_amdgcn_readlane(incl, 63);
    if (total > kCap) return kCanonHost;
    for (int pos = incl - cnt; hits; hits &= hits - 1, ++pos) {
      const int v = __ffsll((long long)hits) - 1;
      const Ref y = emb(cur ^ 1, pos);
      for (int k = 2; k < l.eb / 8; ++k)
        reinterpret_cast<unsigned long long *>(y.p)[k] = reinterpret_cast<const unsigned long long *>(E.p)[k];
      y.used() = E.used() | 1ull << eid[u * vs + v];
      y.vused() = E.vused() | 1ull << v;
      y.map(maxtoc + 1) = (uint8_t)v;
    }
    ncur = total;
    cur ^= 1;
    // the new edge, then the path from its source on
    const int kept = nrm - place;
    const uint32_t moved = lane < kept ? rm[place + lane] : 0u;
    wave_sync();
    if (lane < kept) rm[1 + lane] = moved;
    if (lane == 0) rm[0] = cw & 0xFFFFFFu;
    nrm = 1 + kept;
    ++maxtoc;
  }
  return kCanonMin;
}

// Frequent keys of a later level: key -> (parent, new tuple) -> C.  The
// answer + 1 goes to bits 32-39 of the record's support word, and when the
// children are chosen on the device (c.spread) their chunks, which take two
// divisions, to bits 40-63 (all ones: too many for them).
__global__ void __launch_bounds__(64) k_canon_level(CanonArgs c) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x;
  const uint32_t nf = min(*c.freq_count, c.freq_cap);
  const int len = c.len;
  const LevelLds l = level_lds(min(len + 1, kCE));
  uint32_t *const w = reinterpret_cast<uint32_t *>(lds + l.w);
  uint8_t *const lab = reinterpret_cast<uint8_t *>(lds + l.lab);
  const uint32_t SB = (uint32_t)(c.S * c.NEL);
  for (uint32_t slot = blockIdx.x; slot < nf; slot += gridDim.x) {
    unsigned long long *f = c.freq + 4ull * slot;
    const uint32_t key = (uint32_t)f[0], pk = key / (uint32_t)c.K, x = key - pk * (uint32_t)c.K;
    const unsigned long long sup = f[1], rows = f[2];
    const int64_t p = (int64_t)pk + c.p_base;
    const int nvp = meta_at(c.meta, c.meta_stride, p)->nv;
    const bool forward = x >= SB;
    const int nv = nvp + (forward ? 1 : 0);
    int res = kCanonHost;
    if (len + 1 <= kCE && nv <= kCV - 1) {
      wave_sync();  // the previous key's LDS is no longer read
      for (int t = lane; t < len; t += 64) w[t] = c.pcode[p * len + t];
      for (int v = lane; v < nvp; v += 64) lab[v] = c.pvlab[p * c.S + v];
      if (lane == 0) {
        if (!forward) {  // rightmost -> to
          const uint32_t to = x / (uint32_t)c.NEL;
          w[len] = (uint32_t)(nvp - 1) | to << 8 | (x - to * (uint32_t)c.NEL) << 16 | (uint32_t)c.pvlab[p * c.S + to] << 24;
        } else {  // from -> new vertex nvp
          const uint32_t y = x - SB, y1 = y / (uint32_t)c.NVL, tl = y - y1 * (uint32_t)c.NVL, from = y1 / (uint32_t)c.NEL;
          w[len] = from | (uint32_t)nvp << 8 | (y1 - from * (uint32_t)c.NEL) << 16 | tl << 24;
          lab[nvp] = (uint8_t)tl;
        }
      }
      wave_sync();
      res = canon_level(lds, l, len + 1, nv, lane);
    }
    // answer + 1, so that a record the kernel did not reach reads as 0
    if (lane == 0) {
      unsigned long long v = (sup & 0xFFFFFFFFull) | ((unsigned long long)(res + 1) << 32);
      if (c.spread) {
        const uint32_t chunks = chunk_count((uint32_t)rows, chunk_nominal((uint32_t)c.child_blocks, (uint32_t)rows, (uint32_t)sup));
        v |= (unsigned long long)min(chunks, kChunksMany) << 40;
        if (res != kCanonNotMin)
          atomicMax(&c.spread[(slot & (kSpread - 1)) * kSpreadStride + kSpreadNv], (unsigned long long)nv);
      }
      f[1] = v;
      if (c.down && slot < c.down_cap) c.down[4ull * slot + 1] = v;
    }
  }
}

// Explicit codes: n codes of len tuples (from, to, fromlabel, elabel,
// tolabel); vertex labels as the code carries them (-1: none, 0 default),
// later tuples overriding earlier ones (DFSCode::toGraph,
// src/globals/dfs_code.cpp:245-265).
__global__ void __launch_bounds__(64) k_canon_list(CanonArgs c) {
  __shared__ CanonLds L;
  const int lane = threadIdx.x;
  const int len = c.len;
  for (int64_t q = blockIdx.x; q < c.n; q += gridDim.x) {
    const int32_t *code = c.codes + q * (int64_t)len * 5;
    __syncthreads();
    int nv = 0, bad = 0;
    for (int t = 0; t < len; ++t) {  // uniform loads
      const int a = code[5 * t], b = code[5 * t + 1];
      if (a < 0 || b < 0 || a == b) bad = 1;
      nv = max(nv, max(a, b) + 1);
    }
    if (bad) {
      if (lane == 0) c.out[q] = kCanonBad;
      continue;
    }
    if (len > kCE || nv > kCV - 1) {
      if (lane == 0) c.out[q] = kCanonHost;
      continue;
    }
    for (int t = lane; t < len; t += 64) {
      L.wfrom[t] = (uint8_t)code[5 * t];
      L.wto[t] = (uint8_t)code[5 * t + 1];
      L.wel[t] = code[5 * t + 3];
      L.wtl[t] = code[5 * t + 4];
    }
    if (lane == 0) {
      for (int v = 0; v < nv; ++v) L.lab[v] = 0;
      for (int t = 0; t < len; ++t) {
        if (code[5 * t + 2] != -1) L.lab[code[5 * t]] = code[5 * t + 2];
        if (code[5 * t + 4] != -1) L.lab[code[5 * t + 1]] = code[5 * t + 4];
      }
    }
    __syncthreads();
    const int res = canon_core(L, len, nv, lane);
    if (lane == 0) c.out[q] = (uint8_t)res;
  }
}

}  // namespace

hipError_t launch_canon_level(const CanonArgs &c, int grid, hipStream_t s) {
  if (grid <= 0) return hipSuccess;
  const size_t lds = level_lds(std::min(c.len + 1, kCE)).bytes;
  hipLaunchKernelGGL(k_canon_level, dim3(grid), dim3(64), lds, s, c);
  return hipGetLastError();
}

hipError_t launch_canon_list(const CanonArgs &c, hipStream_t s) {
  if (c.n <= 0) return hipSuccess;
  const unsigned grid = (unsigned)(c.n < 16384 ? c.n : 16384);
  hipLaunchKernelGGL(k_canon_list, dim3(grid), dim3(64), 0, s, c);
  return hipGetLastError();
}

}  // namespace gm
