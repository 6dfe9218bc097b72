// kernels.hpp -- launch interface of the level-step kernels (kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device.hpp"

namespace gm {

// Rows per chunk (nominal): one wave of k_level / k_write owns a chunk,
// whose bounds are moved forward to the next segment start.  Large levels
// take kChunkRows; smaller ones shorter chunks (down to one block of 64
// rows), so that a level has enough waves to fill the device.
constexpr int kChunkRows = 256;
constexpr int kMinChunkRows = 64;
constexpr int64_t kLevelWaves = 16384;  // waves a level step aims for
// Compact levels: blocks of 64 rows in a chunk, up to four while at least
// kCompactWaves chunks (16 a CU) are left.  A chunk's ends cost: its keys'
// counters cleared, committed and recorded, its children's cursors.  (Aiming
// for 16,384 chunks: 0.58 against 0.43 ms for one query on 50,000 molecules,
// 2.57 against 2.41 ms to mine them; 2,048: 0.78 against 0.74 for 10,000
// transactions.
// Up to eight blocks: 7.49 against 7.33 ms for 100,000 transactions, sixteen
// 8.19.)
constexpr int kCompactBlocks = 4;
constexpr int64_t kCompactWaves = 4096;
inline int compact_blocks(int64_t rows, int most = kCompactBlocks) {
  int blocks = most;
  while (blocks > 1 && rows / (62 * blocks) < kCompactWaves) blocks /= 2;
  return blocks;
}
// Statistics counters that every wave bumps are spread over kSpread cache
// lines: atomics on one address serialise across the device.
constexpr int kSpread = 64;
constexpr int kSpreadStride = 16;  // 64-bit words per line
constexpr int kSpreadCand = 0;     // extension candidates enumerated (listed + pruned)
constexpr int kSpreadFill = 1;     // largest count-table fill of a chunk (atomicMax)
constexpr int kSpreadPool = 2;     // compact levels: list entries taken from the slice's pool
constexpr int kSpreadPruned = 3;   // candidates dropped by the 2-edge path rule
constexpr int kSpreadStart = 4;    // ~(earliest start) of the extension + support stage (atomicMax)
constexpr int kSpreadEnd = 5;      // latest end of the stage (atomicMax); device wall clock
constexpr int kSpreadWritten = 6;  // child rows written by k_write
constexpr int kSpreadFailed = 7;   // chunks recounted by k_level_fix
constexpr int kSpreadNv = 8;       // most vertices of a child that k_canon_level let through (atomicMax)
// the counter block: 8 words (frequent keys, failed chunks, error bits), then the spread lines
constexpr int kCounterWords = 8 + kSpread * kSpreadStride;
// words of the block that k_cselect fills: children | undecided records << 32,
// their rows, their chunks | most vertices << 32, the dropped records' rows
constexpr int kTotChildren = 2, kTotRows = 3, kTotChunks = 4, kTotDropped = 5;

// One chunk of a level's rows: [start, end) after alignment to segment
// starts (a segment is the rows of one pattern in one graph; at the root,
// the vertices of one graph).
struct alignas(16) ChunkInfo {
  int64_t start, end;
  uint32_t flags;  // kChunkFailed
  uint32_t nkeys;  // (key, embeddings, item sum) records the chunk left for k_write
  int32_t p_lo;    // their keys are (pattern - p_lo) * K + key
  uint32_t pad;
};
// A chunk of a compact level: its first row and its {key, first place}
// records, nrec of them at entry rec of the list buffer.
struct alignas(16) CChunk {
  int64_t start;
  uint64_t rec;
  uint32_t nrec;
};
constexpr uint32_t kListUnit = 16;  // list extents start at multiples of this many entries (64 bytes)
constexpr int kErrListPool = 16;  // error bit: a compact level's list pool ran out (the stage runs again)
constexpr uint32_t kChunkFailed = 1;  // the LDS count table overflowed; k_level_fix counted it

// Everything the level-step kernels read or write.  Plain device pointers.
struct StepArgs {
  // database (device.hpp layout)
  const int32_t *gvbase;
  const int32_t *vadj;
  const uint32_t *adj;
  const uint8_t *vlab;
  const int32_t *gjob;
  const int32_t *vgraph;  // graph of each vertex
  // rows of this launch: [row_lo, row_hi); later levels: pattern-major rows
  // (pid, rgraph, vt) whose list regions hold rbound entries from rlist;
  // root level: the database's vertices (lists at their adjacency offsets)
  int64_t row_lo, row_hi;
  const int32_t *pid;
  const int32_t *rgraph;
  const uint8_t *vt;
  const uint32_t *rbound;
  const unsigned long long *rlist;
  int32_t S;  // tuple stride in bytes
  const PatMeta *meta;  // meta_stride bytes per pattern (the wide layout when S = 64; compact levels: CMetaHead)
  int32_t meta_stride;
  // path pruning masks (2 * mask_stride words per pattern; 0: none):
  // fwd[0] new arms at the rightmost vertex, fwd[1 + i] at rm[i].from
  // (bit elabel * NVL + label), bwd[1 + i] backward edges to rm[i].from (bit
  // elabel); a clear bit marks an extension with an infrequent 2-edge path
  const unsigned long long *pmask;
  int32_t mask_stride;
  int64_t K;              // keys per pattern (root: keys per job)
  int32_t p_lo, p_hi;     // patterns (root: jobs) of this launch; (p - p_lo) * K < 2^32
  int32_t p_base;         // first pattern of the level piece: counter keys are (p - p_base) * K + key
  int32_t NEL, NVL;
  // chunks of this launch: chunk i at chunks[chunk0 + i], n_chunks of them,
  // chunk_rows nominal rows each
  ChunkInfo *chunks;
  int64_t chunk0, n_chunks;
  int32_t chunk_rows;
  // candidate lists: {code, child item count}; row r's list at
  // row_list(r), rccnt[r] entries
  uint2 *cand;
  uint16_t *rccnt;
  // rep replicas (a power of two) of the packed counters acc[p * K + key] =
  // support << 40 | embeddings and of the item sums accb[p * K + key];
  // chunk i counts into replica i mod rep, replica r at offset r * nkeys
  unsigned long long *acc, *accb;
  int32_t rep;
  int32_t table_bits;  // per-wave LDS count table of k_level
  // per chunk, chunk_key_cap records {(pattern - p_lo) * K + key,
  // embeddings, item sum}: the chunk's candidates per key, so that k_write
  // reserves the children's rows without counting them again
  uint4 *chunk_keys;
  int32_t chunk_key_cap;
  uint32_t *fail_list, *fail_count;  // chunks whose count table overflowed
  unsigned long long *spread;
  int32_t *error_flag;
  // k_reduce: supports (>= 0), then child ids (-(child + 1)) once chosen
  int32_t *sup;
  int64_t nkeys;
  const int32_t *minsup_job;  // per job; null: every job's is minsup_one
  int32_t minsup_one;
  unsigned long long *freq;  // (key, support, embeddings, item sum) of frequent keys, in key order
  uint32_t *freq_count;
  uint32_t freq_cap;
  uint32_t *tile_count;  // k_reduce: frequent keys per tile of tile_keys keys
  int64_t tile_keys;
  // the counter block (kCounterWords words, freq right behind it) and its
  // mapped host copy, which k_reduce_list fills with the counters and the
  // first down_cap records (null: no mapped copy)
  const unsigned long long *counters;
  unsigned long long *down;
  uint32_t down_cap;
  // k_write: child rows; cur_rows / cur_list[c * rep + r] are the first row
  // and the first list entry of child c for the chunks of replica r, and
  // cursor[c * rep + r] = rows << 32 | list entries reserved so far
  unsigned long long *cur_rows, *cur_list, *cursor;
  int32_t *cpid;
  int32_t *crgraph;
  uint8_t *cvt;
  uint32_t *cbound;
  unsigned long long *crlist;
  int32_t CS;  // child tuple stride
  int64_t ccap;
  // ---- compact levels (compact.hip)
  const unsigned long long *vgrp;
  const uint32_t *crow;   // the rows (root: rrows)
  uint32_t *crow_out;     // the children's rows
  const uint4 *rtab;      // root chunks
  const uint2 *ctab;      // later levels' chunks: {pattern, chunk of the pattern}
  int64_t tab0;           // first chunk of the piece in its table
  int32_t nom;            // nominal rows of a root chunk (later levels': in their metadata)
  CChunk *cchunks;
  uint32_t *clist;        // chunk c's first extent at c * page; then 64 pool slices of pool_sub units from unit pool0
  uint32_t page, pool0, pool_sub;
  int32_t AR;             // label pairs: NEL * NVL
  uint32_t inv_nvl;       // (x * inv_nvl) >> 16 = x / NVL for x < 64
  unsigned long long lab_rep;  // bit el * NVL for every edge label
  uint2 *child_tab;       // the children's chunk table
  int32_t child_blocks;   // blocks of a child's chunk (chunk_nominal)
};
// The children's metadata built on the device (k_cchildren), from the level's
// codes and labels: len tuples and S labels a pattern (root: none).
struct CMetaArgs {
  const uint32_t *pcode;
  const uint8_t *pvlab;
  int32_t len;
  const uint32_t *crec;  // child -> record of the frequent list
  int64_t C;
  // path rule: arms t2[(job * NVL + centre) * AR + arm]; null: none
  unsigned long long *t2;
  int32_t masks;         // the table is complete: the sources' keep masks follow it
  int32_t siblings;      // and they follow the parents' frequent extensions
  // the level's patterns as the level before chose them: their keys there and
  // its support table (chosen keys: -(pattern + 1)); null: not known
  const uint32_t *pkey;
  const int32_t *psup;
  uint32_t pK;
  int32_t pS;
  uint32_t *key;         // out: the children's keys
  char *meta;            // out: meta_stride bytes a child
  int32_t meta_stride;
  uint32_t *code;        // out: len + 1 tuples a child
  uint8_t *vlab;         // out: CS labels a child
};
// Compact levels: dynamic LDS of k_clevel, and the launches (see the general
// ones below).
inline size_t clevel_lds_bytes(int64_t K) { return (size_t)16 * (size_t)K; }
hipError_t launch_clevel(const StepArgs &a, bool root, hipStream_t s);
hipError_t launch_cwrite(const StepArgs &a, bool root, hipStream_t s);
hipError_t launch_ccursors(const StepArgs &a, const int32_t *fchild, const unsigned long long *row_base,
                           const uint32_t *chunk_base, int64_t F, hipStream_t s);
// Choose the children on the device: the frequent records whose code is
// minimal (root: all), in key order; their ids, first rows and first chunks,
// and the totals for the host (kTot* words of a.down).
struct CSelect {
  int32_t *fchild;                // per record
  uint32_t *crec;                 // per child
  unsigned long long *row_base;   // per child
  uint32_t *chunk_base;           // per child
};
hipError_t launch_cselect(const StepArgs &a, const CSelect &c, bool root, uint32_t expect, hipStream_t s);
// k_ccursors and the children's metadata (m.C of them) in one launch.
hipError_t launch_cchildren(const StepArgs &a, const CSelect &c, const CMetaArgs &m, bool root, int64_t F, hipStream_t s);
// The arms of the 2-edge children (m.t2, cleared by the caller).
hipError_t launch_ct2(const StepArgs &a, const CMetaArgs &m, hipStream_t s);
struct CGatherArgs {
  const unsigned long long *vgrp;
  const uint2 *rrows;
  const uint32_t *ggb;
  const int32_t *gvbase;
  const int32_t *sel, *dvb;
  const uint32_t *dgb;
  int64_t n_sel;
  unsigned long long *out_vgrp;
  uint2 *out_rrows;
};
hipError_t launch_cgather(const CGatherArgs &g, hipStream_t s);

// Dynamic LDS of k_level for table_bits, and the per-chunk key records its
// table leaves at most.
size_t level_lds_bytes(int table_bits);
int level_chunk_keys(int table_bits);
hipError_t launch_level(const StepArgs &a, bool root, hipStream_t s);
// Recount the chunks k_level listed as failed (persistent grid; cheap when
// none failed).
hipError_t launch_level_fix(const StepArgs &a, bool root, hipStream_t s);
// The level's supports and its frequent-key list in key order: a pass that
// counts the frequent keys of each tile of a.tile_keys keys (and clears the
// other keys' replicas), and a pass that writes each tile's records behind
// those of the tiles before it.  At most kReduceTiles tiles (the second pass
// adds their counts up), each a whole number of the workgroup's steps.
constexpr int64_t kReduceTiles = 1024;
constexpr int kReduceSplitRep = 8;  // replicas from which four lane groups share a key's
// Keys and counters up to which one workgroup reduces a level (k_reduce_small):
// 4-5 us below the line against 9 and a launch for k_reduce and k_reduce_list;
// past it, at 3,240 keys of 8 replicas or 8,000 of 2, 11 us against 7-9, and at
// 130,000 counters 16 against 9.
constexpr int64_t kSmallKeys = 2048, kSmallCounters = 16384;
inline bool reduce_small(int64_t nkeys, int rep) { return nkeys <= kSmallKeys && nkeys * rep <= kSmallCounters; }
inline int64_t reduce_tile_keys(int64_t nkeys, int rep) {
  const int64_t step = rep >= kReduceSplitRep ? 64 : 256;
  const int64_t steps = (nkeys + step * kReduceTiles - 1) / (step * kReduceTiles);
  return step * (steps > 0 ? steps : 1);
}
__host__ __device__ inline int64_t reduce_tiles(const StepArgs &a) { return (a.nkeys + a.tile_keys - 1) / a.tile_keys; }
hipError_t launch_reduce(const StepArgs &a, bool root, hipStream_t s);
// Children of every chunk in chunks[0, n_chunks) (the whole level).
hipError_t launch_write(const StepArgs &a, bool root, hipStream_t s);
// Copy `bytes` (a multiple of 8) between device memory and mapped pinned
// host memory with a kernel on stream s.
hipError_t launch_copy8(void *dst, const void *src, size_t bytes, hipStream_t s);
// For the F frequent keys (the keys of the frequent list a.freq, in its
// order): sup[key] = -(fchild[i] + 1) for the chosen ones (fchild >= 0),
// their (child, replica) cursors from row_base / list_base[child] and the
// replicas' counts; the keys' replicas and the level's counters are cleared.
hipError_t launch_cursors(const StepArgs &a, const int32_t *fchild, const unsigned long long *row_base,
                          const unsigned long long *list_base, int64_t F, hipStream_t s);
// Gather selected graphs of a resident packed database into a new one
// (k_gather_graphs): per selected graph t, its source graph, first vertex
// and first adjacency entry in the output, and its job.
struct GatherArgs {
  const int32_t *gvbase, *vadj;
  const uint32_t *adj;
  const uint8_t *vlab;
  const int32_t *sel, *dvb, *dab, *djob;
  int64_t n_sel;
  int32_t *out_gvbase, *out_vadj, *out_gjob, *out_vgraph;
  uint32_t *out_adj;
  uint8_t *out_vlab;
};
hipError_t launch_gather_graphs(const GatherArgs &g, hipStream_t s);
// Zero `bytes` (a multiple of 8) of device memory with a kernel.
hipError_t launch_fill8(void *dst, size_t bytes, hipStream_t s);
// The static workspace of the entry point that allocates nothing: a
// file-scope device array of kStaticScratchBytes in kernels.hip; *ptr gets
// its address on the current device (looked up once per device).
constexpr size_t kStaticScratchBytes = 64ull << 20;
hipError_t static_scratch(void **ptr, size_t *bytes);
// Minimum DFS code check on the device (canon.hip): one wave per code, the
// pattern graph and the embedding lists in LDS.  Codes beyond these sizes are
// left to the host check (kCanonHost).
constexpr int kCanonV = 40;     // pattern vertices (+1 for the grown code's next vertex)
constexpr int kCanonE = 64;     // pattern edges (64-bit used-edge masks)
constexpr int kCanonCap = 64;   // embeddings of the grown code held at once
constexpr int kCanonNotMin = 0, kCanonMin = 1, kCanonHost = 2, kCanonBad = 3;
constexpr uint32_t kChunksMany = 0xFFFFFFu;
struct CanonArgs {
  // a later level's frequent records (key, support, embeddings, item sum):
  // the answer + 1 for record i goes to bits 32-39 of its support word (and
  // with spread its chunks, at most kChunksMany, to bits 40-63)
  unsigned long long *freq;
  const uint32_t *freq_count;
  uint32_t freq_cap;
  // mapped host copy of the first down_cap records' support words (record i
  // at down[4 * i + 1]); null: none
  unsigned long long *down;
  uint32_t down_cap;
  // the level's patterns: nv from meta, len tuples each packed from | to << 8
  // | elabel << 16 | tolabel << 24 (dense labels), S vertex labels each
  // (S: the level's tuple stride; meta_bytes(S) bytes of metadata each)
  const PatMeta *meta;
  int32_t meta_stride;
  int32_t p_base;  // record keys are (pattern - p_base) * K + key
  const uint32_t *pcode;
  const uint8_t *pvlab;
  int32_t len;
  int64_t K;
  int32_t S, NEL, NVL;
  // children chosen on the device: kSpreadNv lines and blocks of a child's chunk; null: not
  unsigned long long *spread;
  int32_t child_blocks;
  // explicit codes: n codes of len (from, to, fromlabel, elabel, tolabel)
  // tuples; out[i] gets the answer (kCanonBad: a malformed tuple)
  const int32_t *codes;
  int64_t n;
  uint8_t *out;
};
// grid: waves over the frequent records (any count covers them)
hipError_t launch_canon_level(const CanonArgs &c, int grid, hipStream_t s);
hipError_t launch_canon_list(const CanonArgs &c, hipStream_t s);
// Zero the per-level counters (frequent-key count, failure list, spread
// statistics but the written-row slots).
hipError_t launch_clear_counters(const StepArgs &a, hipStream_t s);

}  // namespace gm
