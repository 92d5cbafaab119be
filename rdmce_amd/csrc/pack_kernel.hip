// Packed search for gfx950: many small roots per wavefront, one tree node
// per lane.
//
// The one-wave-per-root kernel (mce_kernel.hip, the reference's layout:
// BkPivotBitBalance.cuh:510-608) spends a whole wave on one tree node at a
// time, so a node of a root with |P0| <= 64 costs hundreds of wave
// instructions for a few words of set work.  Here a wave keeps up to
// pk_slots subproblems resident in its LDS and a stack of tree-node records
// in HBM; every pass of its loop hands up to 64 pending tasks to the 64
// lanes, and each lane computes one tree node on its own:
//
//   task    (record, candidate t of the record's V): the child of t as the
//           sequential search makes it, P' = (P \ {v in V : v < t}) & N(t),
//           XP' = (XP | {v in V : v < t}) & N(t), XX' = XX & cols(t)
//           (BkPivotBitBalance.cuh:40-70: the k-th candidate of a published
//           level, which is what the reference's thieves materialise),
//           followed by aggressive node generation (:351-382);
//   node    a leaf is counted when XP' and XX' are empty; otherwise the
//           pivot is the (|P' \ N(u)|, lowest row) argmin over the rows u
//           of P' | XP' | XX' (:229-257), and a node whose P' an excluded
//           row covers is pruned; a branching node pushes its record, whose
//           candidates V = P' \ N(pivot) become |V| tasks.
//
// Every child is a function of its parent record and its candidate alone,
// so the order in which lanes take tasks never changes the search tree:
// node counts, cliques, hash and histogram equal the one-wave-per-root
// kernel's and the oracle's.  Dispatch takes tasks from the top of the stack
// (the newest records), which keeps the stack near depth x 64 records;
// beyond pk_thr records only the top record is expanded (plain depth-first
// order), which bounds it by pk_thr + 64 (64 NW + 3) records.
//
// A subproblem occupies an LDS slot from its build until its last record is
// consumed:  rows of P0 and of X0' over P0 (NW words), the columns of the X0'
// block for each P0 vertex (NX words: XX' = XX & cols(t) is one load), and
// the label hashes of P0.  Roots with |P0| > 64 NW or |X0'| > 64 NX are
// appended to a.wide for the next launch of the run.  When a.wide_h is set,
// the vertex bitmap of a run that met such roots is copied to a.pk_pool
// (while it has room) and the next launch derives each of them from that
// copy (a.pk_whandle) instead of building it again.  A derived root with
// too many X0' rows whose top node one of them prunes (it covers P0) is
// settled there, as one tree node, and goes nowhere.
//
// Sharing: a wave that runs out of roots and records asks for work (its bit in
// pk_idle); every kPackPoll passes a working wave looks for such waves and
// mails one of them half of its run's unbuilt roots or, when its run has none
// to spare, every other record among the lowest of its stack (the shallowest,
// so the largest subtrees) with a copy of their subproblem - or the upper half
// of a single record's candidates.  The records given away stay in the stack
// as empty ones.  This is the reference's root-down exposure
// (BkPivotBitBalance.cuh:87-138) with the giver doing the copying: a taker
// reads only its own mail, so a few thousand waiting waves poll a few thousand
// lines.  What it measured, all launches: R-MAT 14, edge factor 14 (108M
// nodes, most below a few roots) 110 ms without sharing, 49 ms giving the lower
// half of the stack (the giver was left with little and asked next), 12.5 ms
// giving every other record; a 200k-vertex community graph 31, 28 and 24 ms.
// It is off where no root can reach the sharing bound (|P0| is at most the
// largest out-degree).
#include "mce_common.hpp"

extern __shared__ uint64_t lds_dyn[];

namespace rdmce {
namespace {

// Passes between looks for idle waves (a power of two; a pass takes 10 - 20
// us), and pending tasks from which on a wave gives some away.  R-MAT 14 /
// community graph, ms: looks every 4 passes 12.7 / 27.1, 8 12.5 / 24.0, 16
// 13.7 / 23.8 (each gift copies a subproblem, and the taker starts with part
// of a pass).
#ifdef RDMCE_PACK_EAGER_GIFTS  // test builds: gifts on small graphs, counted by kind in the results' sharing fields
constexpr uint32_t kPackPoll = 1, kPackSpare = 2;
#else
constexpr uint32_t kPackPoll = 8;
constexpr uint32_t kPackSpare = 32;
#endif

template <int NW, int NX>
struct PackCfg {
  static constexpr uint32_t RS = pack_rec_words(NW, NX);
  static constexpr uint32_t SW = pack_slot_words(NW, NX);
  static constexpr uint32_t HS = pack_hist_words(NW);
  // record fields (each a column of pk_cap words in the wave's stack):
  // P XP V (NW each), XX (NX), key, meta, R (NW, read and written only for
  // clique lists).  meta = end << 40 | first << 32 | slot << 16 | |R|, where the record's remaining candidates are the members of V in
  // [first, end).
  static constexpr uint32_t oP = 0, oX = NW, oV = 2 * NW, oXX = 3 * NW, oKey = 3 * NW + NX, oMeta = 3 * NW + NX + 1,
                            oR = 3 * NW + NX + 2;
  // slot word offsets
  static constexpr uint32_t sProw = 0, sXrow = 64 * NW * NW, sXcol = sXrow + 64 * NX * NW, sG = sXcol + 64 * NW * NX;
};

// Bits [64 q, 64 q + 64) of the range [first, end) that a record's meta names.
__device__ __forceinline__ uint64_t range_word(uint64_t meta, uint32_t q) {
  const uint32_t first = (uint32_t)(meta >> 32) & 0xFF, end = (uint32_t)(meta >> 40) & 0xFF, lo = 64u * q;
  return low_mask(end > lo ? end - lo : 0u) & ~low_mask(first > lo ? first - lo : 0u);
}

// Position of the k-th (0-based) set bit of w; k < popcount(w).
__device__ __forceinline__ uint32_t select64(uint64_t w, uint32_t k) {
  uint32_t pos = 0, c;
  c = (uint32_t)__popcll(w & 0xFFFFFFFFull);
  if (k >= c) { k -= c; w >>= 32; pos = 32; }
  c = (uint32_t)__popcll(w & 0xFFFFull);
  if (k >= c) { k -= c; w >>= 16; pos += 16; }
  c = (uint32_t)__popcll(w & 0xFFull);
  if (k >= c) { k -= c; w >>= 8; pos += 8; }
  c = (uint32_t)__popcll(w & 0xFull);
  if (k >= c) { k -= c; w >>= 4; pos += 4; }
  c = (uint32_t)__popcll(w & 0x3ull);
  if (k >= c) { k -= c; w >>= 2; pos += 2; }
  if (k >= (uint32_t)(w & 1)) pos += 1;
  return pos;
}

// Mail words are written and read at the coherence point of the XCDs' L2s
// (relaxed device-scope accesses).  Plain accesses with a release by the giver
// and an acquire by the taker write back and invalidate a whole L2 for each
// gift: R-MAT 14 spent three quarters of its wave time waiting, with more
// gifts making it slower.
__device__ __forceinline__ void st_mail(uint64_t *p, uint64_t v) {
  __hip_atomic_store((unsigned long long *)p, (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t ld_mail(const uint64_t *p) { return ld_relaxed((unsigned long long *)p); }
// Waits until this wave's mail stores have reached that point.  (A fence of
// workgroup scope does not wait for global stores, one of device scope writes
// back the L2.)
__device__ __forceinline__ void mail_stored() {
#ifdef __AMDGCN__
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
  wave_fence();
}

// The per-wave LDS areas (word offsets from lds_dyn).
struct PackLds {
  ldsu64 *hist;     // kLdsHist clique sizes (outside batches)
  lds64 *map;       // 64 u32: dispatch map
  lds64 *meta;      // kPackMetaWords x S
  lds64 *bhist;     // batches: HS x S per-slot clique sizes
  lds64 *slots;     // SW x S
};

// Slot bookkeeping, kPackMetaWords arrays of S words.
enum PackMeta { mCanon, mKey, mPX, mBase, mV, mNodes, mRefs, mCount, mHash };

template <int NW, int NX>
struct PackWave {
  using C = PackCfg<NW, NX>;
  const KArgs &a;
  PackLds L;
  uint32_t S;
  uint32_t me;

  __device__ __forceinline__ lds64 *m(PackMeta f, uint32_t s) const { return L.meta + (uint32_t)f * S + s; }
  __device__ __forceinline__ lds64 *slot(uint32_t s) const { return L.slots + s * C::SW; }
};

// Counts one maximal clique of slot s (size, key = sum of label hashes),
// with R's members given by rb (bits over P0).  Per lane.
template <int NW, int NX, bool LISTS>
__device__ __forceinline__ void pk_emit(const PackWave<NW, NX> &w, uint32_t s, uint32_t size, uint64_t key,
                                        const uint64_t (&rb)[NW], uint64_t &cnt, uint64_t &hsh) {
  using C = PackCfg<NW, NX>;
  const KArgs &a = w.a;
  const uint64_t h = splitmix64_mix(key);
  if (a.root_graph) {
    __hip_atomic_fetch_add(w.m(mCount, s), (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(w.m(mHash, s), h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(w.L.bhist + s * C::HS + size, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  } else {
    cnt++;
    hsh += h;
    if (size < kLdsHist) {
      __hip_atomic_fetch_add(w.L.hist + size, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else if (size < a.hist_len) {
      atomicAdd(&a.hist[size], 1ull);
    } else {
      atomicAdd(&a.hist[a.hist_len - 1], 1ull);
      atomicOr(a.err, kErrHistOverflow);
    }
  }
  if (LISTS && a.list) {
    // entry: size, the root's vertices, then R's members in P0 order
    const unsigned long long pos = atomicAdd(a.list_cursor, (unsigned long long)(size + 1));
    if (pos + size + 1 > a.list_cap) {
      atomicOr(a.err, kErrListFull);
    } else {
      uint32_t *dst = a.list + pos;
      const uint64_t bg = *w.m(mBase, s), vv = *w.m(mV, s);
      const uint32_t *pl = a.pk_plist + ((uint64_t)w.me * w.S + s) * kPackMaxP;
      dst[0] = size;
      dst[1] = a.labels[(uint32_t)vv];
      uint32_t k = 1;
      if ((uint32_t)bg == 2) dst[++k] = a.labels[(uint32_t)(vv >> 32)];
      for (int q = 0; q < NW; ++q)
        for (uint64_t r = rb[q]; r; r &= r - 1) dst[++k] = a.labels[pl[q * 64 + __builtin_ctzll(r)]];
    }
  }
}

// The columns of slot s's X0' block from its rows (in place): bit x of column
// j is bit j of row x.  Lane l holds row 64 b + l of block b; one ballot per
// P0 vertex and block.
template <int NW, int NX>
__device__ __forceinline__ void pk_columns(const PackWave<NW, NX> &w, uint32_t s, uint32_t p, uint32_t xq) {
  using C = PackCfg<NW, NX>;
  const uint32_t l = cold_lane();
  lds64 *sl = w.slot(s);
  wave_fence();
#pragma unroll
  for (int b = 0; b < NX; ++b) {
    uint64_t row[NW];
#pragma unroll
    for (int q = 0; q < NW; ++q) row[q] = (64u * b + l < xq) ? (uint64_t)sl[C::sXrow + (64u * b + l) * NW + q] : 0ull;
#pragma unroll
    for (int q = 0; q < NW; ++q) {
      uint64_t mine = 0;
      const uint32_t n = p > 64u * q ? (p - 64u * q < 64 ? p - 64u * q : 64u) : 0u;
      for (uint32_t j = 0; j < n; ++j) {
        const uint64_t col = __ballot((row[q] >> j) & 1);
        if (l == j) mine = col;
      }
      if (64u * q + l < p) sl[C::sXcol + (64u * q + l) * NX + b] = mine;
    }
  }
}

// The top node of slot s's root (R = {}, P = P0, XP = {}, XX = X0'), a row per
// lane: its pivot is the (|P0 \ N(u)|, row) argmin over all rows.  Returns
// false when an X0' row covers P0 (pruned: no maximal clique below), else the
// candidates V = P0 \ N(pivot).  As a task like the others, a top node kept one
// lane busy with up to 64 NW + 64 NX rows while the rest of its pass had a
// few each.
template <int NW, int NX>
__device__ __forceinline__ bool pk_top(const PackWave<NW, NX> &w, uint32_t s, uint32_t p, uint32_t xq,
                                       uint64_t (&V)[NW]) {
  const uint32_t l = cold_lane();
  const lds64 *sl = w.slot(s);
  uint32_t best = ~0u;
#pragma unroll
  for (int r = 0; r < NW + NX; ++r) {
    const uint32_t row = 64u * r + l;  // (P0 rows first, then 64 NW + x)
    if (r < NW ? row < p : row - 64u * NW < xq) {
      uint32_t c = p;
#pragma unroll
      for (int q = 0; q < NW; ++q) c -= (uint32_t)__popcll((uint64_t)sl[row * NW + q]);
      const uint32_t k = (c << 16) | row;
      best = k < best ? k : best;
    }
  }
  best = wave_min_u32(best);
#pragma unroll
  for (int q = 0; q < NW; ++q)
    V[q] = low_mask(p > 64u * q ? p - 64u * q : 0u) & ~bcast64((uint64_t)sl[(best & 0xFFFF) * NW + q]);
  return (best >> 16) != 0;
}

// Bookkeeping of slot s once its rows, columns, label hashes (and clique-list
// ids) are in place; its top node is counted.
template <int NW, int NX>
__device__ __forceinline__ void pk_seal(const PackWave<NW, NX> &w, uint32_t s, uint64_t p, uint64_t xq, uint64_t canon,
                                        uint64_t base_key, uint32_t base_size, uint32_t graph, uint32_t v0,
                                        uint32_t v1) {
  using C = PackCfg<NW, NX>;
  const KArgs &a = cold_args(w.a);
  const uint32_t l = cold_lane();
  if (l == 0) {
    *w.m(mCanon, s) = canon;
    *w.m(mKey, s) = base_key;
    *w.m(mPX, s) = p | (xq << 32);
    *w.m(mBase, s) = (uint64_t)base_size | ((uint64_t)graph << 32);
    *w.m(mV, s) = (uint64_t)v0 | ((uint64_t)v1 << 32);
    *w.m(mNodes, s) = 1;
    *w.m(mRefs, s) = 1;  // the top node's record, pushed next
    *w.m(mCount, s) = 0;
    *w.m(mHash, s) = 0;
  }
  if (a.root_graph)
    for (uint32_t i = l; i < C::HS; i += 64) w.L.bhist[s * C::HS + i] = 0;
  wave_fence();
}

// Counts the root's own vertex set {v0, v1} (or {v0}) as a maximal clique:
// a root whose candidate and excluded sets are both empty.  Lane 0.
template <int NW, int NX>
__device__ __forceinline__ void pk_emit_base(const PackWave<NW, NX> &w, uint64_t base_key, uint32_t base_size,
                                             uint32_t graph, uint32_t v0, uint32_t v1, uint64_t &cnt, uint64_t &hsh) {
  const KArgs &a = w.a;
  if (lane() != 0) return;
  const uint64_t h = splitmix64_mix(base_key);
  if (a.root_graph) {
    atomicAdd(&a.g_count[graph], 1ull);
    atomicAdd(&a.g_hash[graph], h);
    atomicAdd(&a.g_hist[(uint64_t)graph * a.g_hist_stride + base_size], 1ull);
  } else {
    cnt++;
    hsh += h;
    __hip_atomic_fetch_add(w.L.hist + base_size, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  if (a.list) {
    const unsigned long long pos = atomicAdd(a.list_cursor, (unsigned long long)(base_size + 1));
    if (pos + base_size + 1 > a.list_cap) {
      atomicOr(a.err, kErrListFull);
    } else {
      a.list[pos] = base_size;
      a.list[pos + 1] = a.labels[v0];
      if (base_size == 2) a.list[pos + 2] = a.labels[v1];
    }
  }
}

// Builds root `canon` into slot s (the whole wave).  Returns 1 when the root
// occupies the slot (V: its top node's candidates), 0 when it needs no search
// (its 2-clique, if maximal, is counted here), 2 when it is too wide for this
// variant (the caller hands it to the next launch), 3 when its top node is
// pruned by an X0' row covering P0.  1 and 3: the caller counts the top node,
// px = |P0| | |X0'| << 32.
template <int NW, int NX>
__device__ __forceinline__ uint32_t pk_build(const PackWave<NW, NX> &w, uint8_t *scratch, uint32_t s, uint64_t canon,
                                             Acc &acc, uint64_t &cnt, uint64_t &hsh, uint64_t (&V)[NW], uint64_t &px) {
  using C = PackCfg<NW, NX>;
  const KArgs &a = cold_args(w.a);
  const uint32_t l = cold_lane();
  Sub sub;
  sub.canon = canon;
  sub.graph = a.root_graph ? bcast32(a.root_graph[canon]) : 0;
  uint32_t *Pl = (uint32_t *)scratch;
  const uint64_t ccap = a.slot_bytes / 4;
  uint64_t p = 0, x = 0;
  const uint32_t above = root_lists(a, canon, Pl, ccap, sub, p, x, acc);
  if (p == 0) {
    if (x == 0) pk_emit_base(w, sub.base_key, sub.base_size, sub.graph, sub.v0, sub.v1, cnt, hsh);
    return 0;
  }
  if (p > 64u * NW || p + x > ccap) {
    return 2;
  }
  wave_fence();
  const uint32_t *P = Pl;
  uint32_t *X = Pl + p;
  const uint64_t xq = compact_x(a, P, p, X, x, above);
  wave_fence();
  if (xq > 64u * NX) {
    return 2;
  }
  const uint64_t rows = p + xq;
  // the bitmap tiers' accounting: both lists and a W x rows_pad bitmap
  acc.build += 4 * (p + x) + 8ull * ((p + 63) / 64) * align_up(rows, 64);
  lds64 *sl = w.slot(s);
  for (uint32_t i = l; i < C::sXcol; i += 64) sl[i] = 0;  // P0 rows and X0' rows
  for (uint32_t i = l; i < p; i += 64) sl[C::sG + i] = a.label_hash[P[i]];
  if (a.list) {
    uint32_t *pl = a.pk_plist + ((uint64_t)w.me * w.S + s) * kPackMaxP;
    for (uint32_t i = l; i < p; i += 64) pl[i] = P[i];
  }
  wave_fence();
  acc.scan += match_rows(
      a, P, p, X, rows, above,
      [&](uint64_t i, uint32_t j) {
        or64_lds(sl + C::sProw + i * NW + (j >> 6), 1ull << (j & 63));
        or64_lds(sl + C::sProw + (uint64_t)j * NW + (i >> 6), 1ull << (i & 63));
      },
      [&](uint64_t i, uint32_t wd, uint64_t bits) { or64_lds(sl + C::sXrow + (i - p) * NW + wd, bits); });
  wave_fence();
  px = p | (xq << 32);
  if (!pk_top<NW, NX>(w, s, (uint32_t)p, (uint32_t)xq, V)) return 3;
  pk_columns<NW, NX>(w, s, (uint32_t)p, (uint32_t)xq);
  pk_seal<NW, NX>(w, s, p, xq, canon, sub.base_key, sub.base_size, sub.graph, sub.v0, sub.v1);
  return 1;
}

// ---------------------------------------------------------------------------
// Edge roots derived from their first vertex's bitmap.
//
// Every edge root (v0, u_k) with u_k the k-th vertex of U = N+(v0) is a
// restriction of the vertex root v0 (BkPivotBitBalance.cuh:414-427 builds it
// as the LEVEL_1 root): P0 = {u_j : j > k, u_j ~ u_k}, X0 = {x ~ v0 : x < v0,
// x ~ u_k} then {u_j : j < k, u_j ~ u_k} (ascending vertex order), and X0'
// keeps the rows of X0 with a neighbour in P0.  A wave that takes a run of
// edge roots of one v0 therefore builds the vertex root's bitmap once, in its
// scratch region (rows U then X0v' = the x ~ v0 below v0 with a neighbour in
// U, word-major), and derives each edge root from it by bit extraction:
// rows of the edge root are the vertex rows restricted to P0's columns and
// compressed to P0's indices.  The subproblem (rows, order, label hashes) is
// exactly the one pk_build makes, so the search tree is unchanged.
// ---------------------------------------------------------------------------
constexpr uint32_t kGroupMaxW = 16;  // |U| <= 1024
constexpr uint32_t kPoolHdr = 8;     // kept vertex bitmap: v0 d0 W0 xq0 rp o0 rfirst lh0, then T, cm and lh

struct PkGroup {
  uint32_t v0, d0, W0, xq0, rp;
  uint64_t o0;          // U = col[o0, o0 + d0)
  uint64_t rfirst;      // canonical id of the edge root (v0, U[0])
  const uint64_t *T;    // W0 x rp words: rows 0..d0-1 (U), d0..d0+xq0-1 (X0v')
  const uint64_t *cm;   // W0 words: OR of the X0v' rows (U vertices with a neighbour below v0)
  uint64_t *wide;       // the run's roots too wide for this variant, kept until the run ends
  const uint64_t *lh;   // d0 words: splitmix64(label) of each member of U
  uint64_t lh0;         // splitmix64(label(v0))
};

// Builds the bitmap of vertex root v0 into `scratch` (the whole wave), with
// room for `run` wide root ids after it; `claim` is an LDS word for handing
// out rows.  Returns false when it does not fit (the caller then builds each
// edge root on its own).
__device__ __forceinline__ bool pk_group_build(const KArgs &a0, uint8_t *scratch, uint32_t v0, uint64_t run, PkGroup &G,
                                               Acc &acc, ldsu32 *claim) {
  const KArgs &a = cold_args(a0);
  const uint32_t l = cold_lane();
  const uint64_t b0 = bcast64(a.rowoff[v0]), e0 = bcast64(a.rowoff[(uint64_t)v0 + 1]), o0 = bcast64(a.outoff[v0]);
  const uint64_t d0 = e0 - o0, x0 = o0 - b0;
  const uint64_t W0 = (d0 + 63) / 64;
  if (W0 == 0 || W0 > kGroupMaxW) return false;
  const uint64_t rpa = align_up(d0 + x0, 64), nbx = (x0 + 63) / 64;
  const uint64_t cm_off = align_up(8 * W0 * rpa, 256);
  const uint64_t wide_off = cm_off + align_up(8 * W0, 256);
  const uint64_t lh_off = wide_off + align_up(8 * run, 256);
  const uint64_t mask_off = lh_off + align_up(8 * d0, 256);
  if (mask_off + 8 * nbx > a.slot_bytes) return false;
  const uint32_t *U = a.col + o0;
  uint64_t *T = (uint64_t *)scratch;
  uint64_t *cm = (uint64_t *)(scratch + cm_off);
  uint64_t *kept = (uint64_t *)(scratch + mask_off);  // a bit per lower neighbour: its row is not empty
  for (uint64_t i = l; i < W0 * rpa; i += 64) T[i] = 0;
  wave_fence();
  // Rows of every lower neighbour, then those that are not empty moved
  // together.  Bound by the chain of loads into the adjacency lists: looking
  // for each lower neighbour's first one in U beforehand, to build kept rows
  // only, went through the lists twice (R-MAT 24, 1.02e10 cliques: 1,953 ms
  // against 1,886; R-MAT 18, roots of core <= 120: 3.99 against 3.88).
  acc.scan += match_rows(
      a, U, d0, a.col + b0, d0 + x0, v0,
      [&](uint64_t i, uint32_t j) {
        or64(&T[(uint64_t)(j >> 6) * rpa + i], 1ull << (j & 63));
        or64(&T[(uint64_t)(i >> 6) * rpa + j], 1ull << (i & 63));
      },
      [&](uint64_t i, uint32_t wd, uint64_t bits) { or64(&T[(uint64_t)wd * rpa + i], bits); }, claim);
  wave_fence();
  uint64_t xq0 = 0;
  for (uint64_t b = 0; b < nbx; ++b) {
    uint64_t any = 0;
    for (uint64_t z = 0; z < W0; ++z)
      if (64 * b + l < x0) any |= T[z * rpa + d0 + 64 * b + l];
    const uint64_t m = __ballot(any != 0);
    if (l == 0) kept[b] = m;
    xq0 += (uint64_t)__popcll(m);
  }
  wave_fence();
  // Column by column, downwards in memory: no word is written before it is read.
  const uint64_t rows = d0 + xq0, rp = align_up(rows, 64);
  for (uint64_t z = 0; z < W0; ++z) {
    if (z && rp != rpa)
      for (uint64_t i = l; i < d0; i += 64) T[z * rp + i] = T[z * rpa + i];
    uint64_t o = 0, at = z * rp + d0;
    for (uint64_t b = 0; b < nbx; ++b) {
      const uint64_t m = bcast64(kept[b]);
      if (m == 0) continue;
      const uint64_t v = (m >> l) & 1 ? T[z * rpa + d0 + 64 * b + l] : 0ull;
      o |= v;
      wave_fence();
      if ((m >> l) & 1) T[at + rank_below(m)] = v;
      at += (uint64_t)__popcll(m);
    }
    const uint64_t ow = ((uint64_t)wave_or_u32((uint32_t)(o >> 32)) << 32) | wave_or_u32((uint32_t)o);
    if (l == 0) cm[z] = ow;
    wave_fence();
  }
  acc.build += 4 * (e0 - b0) + 4 * (d0 + x0) + 8 * W0 * rp;
  G.v0 = v0;
  G.d0 = (uint32_t)d0;
  G.W0 = (uint32_t)W0;
  G.xq0 = (uint32_t)xq0;
  G.rp = (uint32_t)rp;
  G.o0 = o0;
  G.rfirst = bcast64(a.rfirst[v0]);
  G.T = T;
  G.cm = cm;
  G.wide = (uint64_t *)(scratch + wide_off);
  uint64_t *lh = (uint64_t *)(scratch + lh_off);
  for (uint64_t j = l; j < d0; j += 64) lh[j] = a.label_hash[a.col[o0 + j]];
  wave_fence();
  G.lh = lh;
  G.lh0 = bcast64(a.label_hash[v0]);
  return true;
}

// Derives edge root `canon` = (v0, u_k) of group G into slot s (the whole
// wave).  Returns as pk_build does.
template <int NW, int NX>
__device__ __forceinline__ uint32_t pk_derive(const PackWave<NW, NX> &w, const PkGroup &G, uint32_t s, uint64_t canon,
                                              Acc &acc, uint64_t &cnt, uint64_t &hsh, uint64_t (&V)[NW], uint64_t &px) {
  using C = PackCfg<NW, NX>;
  const KArgs &a = cold_args(w.a);
  const uint32_t l = cold_lane();
  const uint32_t k = (uint32_t)(canon - G.rfirst);
  const uint32_t uk = a.list ? bcast32(a.col[G.o0 + k]) : 0u;  // the root's v1 (clique lists only)
  const uint32_t graph = a.root_graph ? bcast32(a.root_graph[canon]) : 0;
  const uint64_t base_key = G.lh0 + bcast64(G.lh[k]);
  // Row k of U, split at k: P0 above it, the U part of X0 below it (one
  // word per lane).
  const uint32_t q = l;
  const uint64_t ak = q < G.W0 ? G.T[(uint64_t)q * G.rp + k] : 0ull;
  const uint32_t kq = k >> 6, kb = k & 63;
  const uint64_t above = q > kq ? ~0ull : (q == kq ? (kb == 63 ? 0ull : ~0ull << (kb + 1)) : 0ull);
  const uint64_t below = q < kq ? ~0ull : (q == kq ? low_mask(kb) : 0ull);
  const uint64_t pk = ak & above, xu = ak & below;
  const uint32_t p = __builtin_amdgcn_readlane(wave_scan_add_u32((uint32_t)__popcll(pk)), 63);
  uint64_t words_read = G.W0;
  if (p == 0) {
    const bool xlow = (readlane64(q < G.W0 ? G.cm[q] : 0ull, kq) >> kb) & 1;
    if (!xlow && __ballot(xu != 0) == 0) pk_emit_base(w, base_key, 2, graph, G.v0, uk, cnt, hsh);
    acc.build += 8 * (words_read + 1);
    return 0;
  }
  if (p > 64u * NW) {
    return 2;
  }
  // Candidate X0 rows, 64 a block: the rows x of X0v' adjacent to u_k (blocks
  // [0, nbx)), then the U rows j < k adjacent to u_k (a block per word of xu) -
  // ascending vertex order.
  const uint32_t nbx = (G.xq0 + 63) / 64, nb = nbx + kq + 1;
  auto candidate = [&](uint32_t b, uint32_t &row) -> bool {
    if (b < nbx) {
      row = G.d0 + 64 * b + l;
      return 64 * b + l < G.xq0 && ((G.T[(uint64_t)kq * G.rp + row] >> kb) & 1);
    }
    row = 64 * (b - nbx) + l;
    return (readlane64(xu, b - nbx) >> l) & 1;
  };
  // X0' keeps the rows with a neighbour in P0.  Row numbers go to lists in the
  // slot's column area (rewritten below): X0' rows, then P0 rows.  A row that
  // covers P0 prunes the root's top node: the root is done, whatever its width.
  lds64 *sl = w.slot(s);
  ldsu32 *xl = (ldsu32 *)(sl + C::sXcol), *pl = xl + 64 * NX;
  uint32_t xq = 0;
  bool cov = false;
  for (uint32_t b = 0; b < nb; ++b) {
    uint32_t row;
    const bool cand = candidate(b, row);
    if (__ballot(cand) == 0) continue;
    uint64_t hit = 0, miss = 0;
    for (uint32_t z = kq; z < G.W0; ++z) {  // (P0 lies above u_k)
      const uint64_t mz = readlane64(pk, z);
      if (mz && cand) {
        const uint64_t t = G.T[(uint64_t)z * G.rp + row];
        hit |= t & mz;
        miss |= mz & ~t;
      }
    }
    cov |= cand && miss == 0;
    const uint64_t m = __ballot(hit != 0);
    const uint32_t at = xq + rank_below(m);
    if (hit != 0 && at < 64u * NX) xl[at] = row;
    xq += (uint32_t)__popcll(m);
  }
  const uint32_t nxu = __builtin_amdgcn_readlane(wave_scan_add_u32((uint32_t)__popcll(xu)), 63);
  words_read += (uint64_t)nbx * 64 + (uint64_t)nxu * G.W0;
  px = (uint64_t)p | ((uint64_t)xq << 32);
  if (__ballot(cov) != 0) {
    acc.build += 8 * words_read;
    return 3;
  }
  if (xq > 64u * NX) return 2;
  for (uint32_t z = kq, before = 0; z < G.W0; ++z) {
    const uint64_t mz = readlane64(pk, z);
    if ((mz >> l) & 1) pl[before + rank_below(mz)] = 64 * z + l;
    before += (uint32_t)__popcll(mz);
  }
  wave_fence();
  uint32_t prow[NW], xrow[NX];
#pragma unroll
  for (int r = 0; r < NW; ++r) prow[r] = 64u * r + l < p ? (uint32_t)pl[64 * r + l] : 0u;
#pragma unroll
  for (int r = 0; r < NX; ++r) xrow[r] = 64u * r + l < xq ? (uint32_t)xl[64 * r + l] : 0u;
  wave_fence();  // the lists are read before the column area is rewritten
  // Every row restricted to P0's columns and compressed to P0's indices: the
  // columns in order, one at a time, the same for every lane; a column's bit
  // is shifted into the top of a 32-bit word (2 instructions per row block
  // and column), and its ballot over the X0' rows is that column of the X0'
  // block.  (Compressing each row on its own and transposing the block after
  // took 16 instructions per column and 5 per column of all 64 NW.)
  uint32_t pc[NW] = {}, xc[NX] = {};       // words being filled
  uint32_t po[NW][2 * NW] = {}, xo[NX][2 * NW] = {};
  uint64_t col[NW][NX] = {};               // lane l: column 64 q + l
  uint32_t c = 0;
  auto put = [&](uint32_t done) {          // word done / 32 - 1 is full, or the last one
    const uint32_t sh = (32 - (done & 31)) & 31, w = (done - 1) / 32;
#pragma unroll
    for (uint32_t o = 0; o < 2 * NW; ++o) {  // (selects: an indexed array would go to scratch)
#pragma unroll
      for (int r = 0; r < NW; ++r) po[r][o] = o == w ? pc[r] >> sh : po[r][o];
#pragma unroll
      for (int r = 0; r < NX; ++r) xo[r][o] = o == w ? xc[r] >> sh : xo[r][o];
    }
  };
  for (uint32_t z = kq; z < G.W0; ++z) {
    const uint64_t mz = readlane64(pk, z);
    if (mz == 0) continue;
    uint64_t pw[NW], xw[NX];
#pragma unroll
    for (int r = 0; r < NW; ++r) pw[r] = 64u * r + l < p ? G.T[(uint64_t)z * G.rp + prow[r]] : 0ull;
#pragma unroll
    for (int r = 0; r < NX; ++r) xw[r] = 64u * r + l < xq ? G.T[(uint64_t)z * G.rp + xrow[r]] : 0ull;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t ph[NW], xh[NX];
#pragma unroll
      for (int r = 0; r < NW; ++r) ph[r] = (uint32_t)(pw[r] >> (32 * h));
#pragma unroll
      for (int r = 0; r < NX; ++r) xh[r] = (uint32_t)(xw[r] >> (32 * h));
      for (uint32_t m = (uint32_t)(mz >> (32 * h)); m; m &= m - 1) {
        const uint32_t b = (uint32_t)__builtin_ctzll((uint64_t)m);
#pragma unroll
        for (int r = 0; r < NW; ++r) pc[r] = ((ph[r] >> b) << 31) | (pc[r] >> 1);
#pragma unroll
        for (int r = 0; r < NX; ++r) {
          const uint32_t t = xh[r] >> b;
          xc[r] = (t << 31) | (xc[r] >> 1);
          const uint64_t cb = __ballot(t & 1);
#pragma unroll
          for (int q = 0; q < NW; ++q)
            if (c == 64u * q + l) col[q][r] = cb;
        }
        if ((++c & 31) == 0) put(c);
      }
    }
  }
  if (c & 31) put(c);
#pragma unroll
  for (int r = 0; r < NW; ++r) {
    const uint32_t t = 64u * r + l;
    if (t < p) {
#pragma unroll
      for (int o = 0; o < NW; ++o) sl[C::sProw + t * NW + o] = (uint64_t)po[r][2 * o] | ((uint64_t)po[r][2 * o + 1] << 32);
#pragma unroll
      for (int b = 0; b < NX; ++b) sl[C::sXcol + t * NX + b] = col[r][b];
      sl[C::sG + t] = G.lh[prow[r]];
      if (a.list) a.pk_plist[((uint64_t)w.me * w.S + s) * kPackMaxP + t] = a.col[G.o0 + prow[r]];
    }
  }
#pragma unroll
  for (int r = 0; r < NX; ++r) {
    const uint32_t t = 64u * r + l;
    if (t < xq) {
#pragma unroll
      for (int o = 0; o < NW; ++o) sl[C::sXrow + t * NW + o] = (uint64_t)xo[r][2 * o] | ((uint64_t)xo[r][2 * o + 1] << 32);
    }
  }
  words_read += (uint64_t)(p + xq) * G.W0;
  acc.build += 8 * words_read + 8ull * NW * (p + xq);
  wave_fence();
  pk_top<NW, NX>(w, s, p, xq, V);
  pk_seal<NW, NX>(w, s, p, xq, canon, base_key, 2, graph, G.v0, uk);
  return 1;
}

// Moves what slot s (uniform) accumulated - batches: count, hash, clique
// sizes; root statistics: its node count - to the results, a word per lane.
// (One lane per finished slot, going through its sizes one by one, took 67 LDS
// round trips a root: 400 small graphs in one replay 7.9 ms against 7.7.)
template <int NW, int NX>
__device__ __forceinline__ void pk_finish(const PackWave<NW, NX> &w, uint32_t s) {
  using C = PackCfg<NW, NX>;
  const KArgs &a = cold_args(w.a);
  const uint32_t l = cold_lane();
  if (a.root_nodes && l == 0) atomicAdd(&a.root_nodes[*w.m(mCanon, s)], (unsigned long long)*w.m(mNodes, s));
  if (a.root_graph) {
    const uint32_t g = bcast32((uint32_t)(*w.m(mBase, s) >> 32));
    if (l < 2) {
      const uint64_t v = *w.m(l ? mHash : mCount, s);
      if (v) atomicAdd(l ? &a.g_hash[g] : &a.g_count[g], (unsigned long long)v);
    }
    for (uint32_t i = l; i < C::HS; i += 64) {
      const uint64_t v = w.L.bhist[s * C::HS + i];
      if (v) {
        if (i < a.g_hist_stride) atomicAdd(&a.g_hist[(uint64_t)g * a.g_hist_stride + i], (unsigned long long)v);
        else atomicOr(a.err, kErrHistOverflow);
      }
    }
  }
}

template <int NW, int NX, bool LISTS>
__device__ __forceinline__ void pack_main(const KArgs &a) {
  using C = PackCfg<NW, NX>;
  const uint32_t l = lane();
  const uint32_t S = a.pk_slots;
  lds64 *base = (lds64 *)lds_dyn;
  PackWave<NW, NX> w{a, {}, S, (uint32_t)blockIdx.x};
  w.L.hist = (ldsu64 *)base;
  w.L.map = base + kLdsHist;
  w.L.meta = w.L.map + 32;
  w.L.bhist = w.L.meta + kPackMetaWords * S;
  w.L.slots = w.L.bhist + (a.root_graph ? C::HS * S : 0);
  const uint64_t n_dispatch = dispatch_count(a);
  if (n_dispatch == 0) return;
  for (uint32_t i = l; i < kLdsHist; i += 64) w.L.hist[i] = 0;
  wave_fence();
  uint32_t shard = w.me % kShards;
  uint8_t *scratch = a.slots + (uint64_t)w.me * a.slot_bytes;
  // The wave's record stack, field-major: field f of record r is
  // stk[f * cap + r], so lanes touching neighbouring records touch
  // neighbouring words.
  uint64_t *stk = a.pk_stack + (uint64_t)w.me * a.pk_cap * C::RS;
  const uint64_t cap = a.pk_cap;
  constexpr bool lists = LISTS;  // clique lists: R is kept in the records
  auto fld = [stk, cap](uint32_t f, uint32_t r) -> uint64_t & { return stk[(uint64_t)f * cap + r]; };
  ldsu32 *map32 = (ldsu32 *)w.L.map;
  Acc acc{};
  uint64_t cnt = 0, hsh = 0, words = 0, nodes = 0;  // per lane
  uint32_t top = 0;                                  // records in the stack
  uint64_t pending = 0;                              // candidates (tasks) in the stack
  uint32_t busy = 0;                                 // occupied slots
  const uint32_t full = S >= 32 ? ~0u : ((1u << S) - 1);
  bool roots_left = true;
  // Dispatch: runs of consecutive dispatch entries (edge roots of one v0,
  // a.pk_gstart) or single entries; a run of two or more edge roots shares
  // the vertex bitmap of its v0 (pk_group_build).
  uint64_t gcur = 0, gend = 0;
  bool grouped = false;
  uint32_t nwide = 0;  // wide roots of the current grouped run, in G.wide
  PkGroup G{};
  bool new_run = false;  // [gcur, gend) has been taken and its vertex bitmap is to be built
  // Sharing: this wave's mail and its parts.
  const bool sharing = a.pk_share != 0;
  uint32_t tick = 0, given = 0;  // records below `given` are empty (given away)
  constexpr uint32_t oMeta0 = kMailHdr, oSlot = kMailHdr + 16, oIds = oSlot + C::SW, oRecs = oIds + kPackMaxP / 2;
  uint64_t *mail = a.pk_mail + (uint64_t)w.me * kPackMailWords;
  // Gives an idle wave, if there is one, part of this wave's work.
  auto give = [&]() {
    const KArgs &a = cold_args(w.a);
    const uint32_t l = cold_lane();
    // The last unbuilt root goes before records of a deep stack do: records
    // that were given away stay in it as empty ones, and a root built on top of
    // those would need its own 64 records per level beyond pk_thr.
    const bool range = gend - gcur >= (top > a.pk_thr ? 1u : 2u);
    uint64_t dm = 0, sel_m = 0;
    uint32_t ci = 0, s0 = 0, cands = 0, mid = 0;
    bool split = false, take = false;
    if (!range) {
      if (pending < kPackSpare) return;
      // lane l looks at record given + l
      const uint32_t nl = top - given < 64 ? top - given : 64;
      uint64_t rem[NW];
#pragma unroll
      for (int q = 0; q < NW; ++q) rem[q] = 0;
      if (l < nl) {
        dm = fld(C::oMeta, given + l);
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          rem[q] = fld(C::oV + q, given + l) & range_word(dm, q);
          ci += (uint32_t)__popcll(rem[q]);
        }
      }
      const uint64_t nz = __ballot(ci != 0);
      if (nz == 0) {
        given += nl;
        return;
      }
      const uint32_t f = (uint32_t)__builtin_ctzll(nz);
      s0 = __builtin_amdgcn_readlane((uint32_t)(dm >> 16) & 0xFF, f);
      const uint64_t same = __ballot(ci != 0 && ((uint32_t)(dm >> 16) & 0xFF) == s0);
      const uint32_t cf = __builtin_amdgcn_readlane(ci, f);
      if (same & (same - 1)) {  // every other record
        take = ((same >> l) & 1) && (rank_below(same) & 1);
      } else {                  // a single record: the upper half of its candidates
        take = l == f;
        split = cf > 1;
        uint32_t kk = ci / 2, base = 0;
#pragma unroll
        for (int q = 0; q < NW - 1; ++q) {
          const uint32_t cq = (uint32_t)__popcll(rem[q]);
          if (base == (uint32_t)q * 64 && kk >= cq) {
            kk -= cq;
            base = (uint32_t)(q + 1) * 64;
          }
        }
        uint64_t rw = rem[0];
#pragma unroll
        for (int q = 1; q < NW; ++q)
          if (base == (uint32_t)q * 64) rw = rem[q];
        mid = base + (split && take ? select64(rw, kk) : 0u);
      }
      sel_m = __ballot(take);
      cands = split ? cf - cf / 2
                    : __builtin_amdgcn_readlane(wave_scan_add_u32(take ? ci : 0u), 63);
    }
    // claim an idle wave
    const int to = find_wave(a.pk_idle, a.pk_nwaves, w.me);
    if (to < 0) return;
    const uint64_t tb = 1ull << (to & 63);
    bool mine = false;
    if (l == 0) mine = (atomicAnd(&a.pk_idle[to >> 6], (unsigned long long)~tb) & tb) != 0;
    if (!bcast32(mine)) return;
    uint64_t *out = a.pk_mail + (uint64_t)to * kPackMailWords;
    uint64_t flag;
    if (range) {  // the upper half of the run's unbuilt roots
      const uint64_t at = gend - gcur > 1 ? gcur + (gend - gcur + 1) / 2 : gcur;
      if (l == 0) {
        st_mail(out + 1, at);
        st_mail(out + 2, gend);
      }
      gend = at;
      flag = 2;
    } else {
      const lds64 *sl = w.slot(s0);
      const uint32_t n = (uint32_t)__popcll(sel_m), rk = rank_below(sel_m);
      for (uint32_t i = l; i < C::SW; i += 64) st_mail(out + oSlot + i, sl[i]);
      if (l < kPackMetaWords) {
        uint64_t v = w.L.meta[l * S + s0];
        v = l == mRefs ? (uint64_t)n : (l == mNodes || l == mCount || l == mHash ? 0ull : v);
        st_mail(out + oMeta0 + l, v);
      }
      if (lists) {
        const uint64_t *ids = (const uint64_t *)(a.pk_plist + ((uint64_t)w.me * S + s0) * kPackMaxP);
        for (uint32_t i = l; i < kPackMaxP / 2; i += 64) st_mail(out + oIds + i, ids[i]);
      }
      if (take) {
        for (uint32_t f = 0; f < (lists ? C::RS : C::RS - NW); ++f)
          if (f != C::oMeta) st_mail(out + oRecs + f * 64 + rk, fld(f, given + l));
        uint64_t tm = dm & ~(0xFFull << 16);  // the taker's slot 0
        if (split) tm = (tm & ~(0xFFull << 32)) | ((uint64_t)mid << 32);
        st_mail(out + oRecs + C::oMeta * 64 + rk, tm);
        fld(C::oMeta, given + l) = split ? (dm & ~(0xFFull << 40)) | ((uint64_t)mid << 40) : dm & 0xFFFFFFFFull;
      }
      pending -= cands;
      const uint64_t empty = __ballot(given + l < top && (ci == 0 || (take && !split)));
      given += ~empty ? (uint32_t)__builtin_ctzll(~empty) : 64u;
      flag = 1 | ((uint64_t)n << 8) | ((uint64_t)cands << 32);
    }
#ifdef RDMCE_PACK_EAGER_GIFTS
    acc.published += range;
    acc.owner += split;
#endif
    state_add(a, (uint32_t)to, kWorking - kLooking);
    mail_stored();  // the mail is there before its flag
    if (l == 0) st_mail(out, flag);
  };
  // Waits for work from another wave; false when there is none to come.
  auto wait_mail = [&]() -> bool {
    const KArgs &a = cold_args(w.a);
    const uint32_t l = cold_lane();
    const uint64_t bit = 1ull << (w.me & 63);
    if (l == 0) st_mail(mail, 0);
    mail_stored();
    if (l == 0) atomicOr(&a.pk_idle[w.me >> 6], (unsigned long long)bit);
    state_add(a, w.me, kLooking - kWorking);
    uint64_t flag = 0;
    bool asked = true;
    for (uint32_t n = 1, k = 0;; n = n < 8 ? n * 2 : 8, ++k) {
      unsigned long long v = 0;
      if (l == 0) v = ld_mail(mail);
      flag = bcast64(v);
      if (flag) break;
      if (asked && (k & 3) == 0 && !any_working(a, w.me)) {
        // withdraw; a wave that has cleared the bit already will send
        bool had = false;
        if (l == 0) had = (atomicAnd(&a.pk_idle[w.me >> 6], (unsigned long long)~bit) & bit) != 0;
        if (bcast32(had)) return false;
        asked = false;
      }
      if (l == 0) nap(n);
    }
    wave_fence();
    ++acc.shared;
    if ((flag & 0xFF) == 2) {
      gcur = bcast64(ld_mail(mail + 1));
      gend = bcast64(ld_mail(mail + 2));
      new_run = true;
      return true;
    }
    const uint32_t n = (uint32_t)(flag >> 8) & 0xFF;
    lds64 *sl = w.slot(0);
    for (uint32_t i = l; i < C::SW; i += 64) sl[i] = ld_mail(mail + oSlot + i);
    if (l < kPackMetaWords) w.L.meta[l * S] = ld_mail(mail + oMeta0 + l);
    if (a.root_graph)
      for (uint32_t i = l; i < C::HS; i += 64) w.L.bhist[i] = 0;
    if (lists) {
      uint64_t *ids = (uint64_t *)(a.pk_plist + (uint64_t)w.me * S * kPackMaxP);
      for (uint32_t i = l; i < kPackMaxP / 2; i += 64) ids[i] = ld_mail(mail + oIds + i);
    }
    if (l < n)
      for (uint32_t f = 0; f < (lists ? C::RS : C::RS - NW); ++f) fld(f, l) = ld_mail(mail + oRecs + f * 64 + l);
    wave_fence();
    top = n;
    given = 0;
    pending = flag >> 32;
    busy = 1;
    return true;
  };
  if (sharing) state_add(a, w.me, kWorking);
  for (;;) {
    const KArgs &a = cold_args(w.a);
    const uint32_t l = cold_lane();
    // Refill: build roots into free slots while fewer than 64 tasks wait.
    while ((roots_left || gcur != gend || nwide) && pending < 64 && busy != full) {
      if (gcur == gend) {
        if (nwide) {  // the finished run's wide roots go out with a copy of its vertex bitmap
          wave_fence();
          const uint64_t tw = (uint64_t)G.W0 * G.rp, need = kPoolHdr + tw + G.W0 + G.d0;
          unsigned long long at = 0, hp = 0;
          if (l == 0) {
            at = atomicAdd(a.n_wide, (unsigned long long)nwide);
            hp = atomicAdd(a.pk_pool_used, (unsigned long long)need);
          }
          at = bcast64(at);
          hp = bcast64(hp);
          const bool kept = hp + need <= a.pk_pool_words;
          if (kept) {
            uint64_t *dst = a.pk_pool + hp;
            if (l < kPoolHdr) {
              const uint64_t hv[kPoolHdr] = {G.v0, G.d0, G.W0, G.xq0, G.rp, G.o0, G.rfirst, G.lh0};
              uint64_t v = 0;
#pragma unroll
              for (uint32_t f = 0; f < kPoolHdr; ++f) v = f == l ? hv[f] : v;
              dst[l] = v;
            }
            for (uint64_t i = l; i < tw; i += 64) dst[kPoolHdr + i] = G.T[i];
            for (uint64_t i = l; i < G.W0; i += 64) dst[kPoolHdr + tw + i] = G.cm[i];
            for (uint64_t i = l; i < G.d0; i += 64) dst[kPoolHdr + tw + G.W0 + i] = G.lh[i];
            acc.build += 8 * need;
          }
          for (uint32_t i = l; i < nwide; i += 64) {
            a.wide[at + i] = G.wide[i];
            a.wide_h[at + i] = kept ? hp : ~0ull;
          }
          nwide = 0;
        }
        if (!roots_left) break;
        uint64_t gi = 0;
        const Claim claim = next_entry(a, a.pk_gstart ? a.pk_ngroups : n_dispatch, shard, gi);
        if (claim == kHop) continue;
        if (claim == kNone) {
          roots_left = false;
          break;
        }
        gcur = a.pk_gstart ? bcast64(a.pk_gstart[gi]) : gi;
        gend = a.pk_gstart ? bcast64(a.pk_gstart[gi + 1]) : gi + 1;
        new_run = true;
      }
      if (new_run) {
        new_run = false;
        grouped = false;
        if (gend - gcur >= 2 && a.root_mode == 2) {
          const uint64_t c0 = bcast64(a.perm ? a.perm[gcur] : (a.reverse ? n_dispatch - 1 - gcur : gcur));
          grouped = pk_group_build(a, scratch, bcast32((uint32_t)(a.roots[c0] >> 32)), a.wide_h ? gend - gcur : 0, G, acc,
                                   map32);
        }
      }
#ifdef RDMCE_PACK_EAGER_GIFTS  // test builds: the stack's bound counts on this
      if (top > a.pk_thr + 64 && l == 0) atomicOr(a.err, kErrPackStack);
#endif
      const uint64_t i = gcur++;
      const uint64_t canon = bcast64(a.perm ? a.perm[i] : (a.reverse ? n_dispatch - 1 - i : i));
      if (a.eager && bcast32(a.eager[i])) {  // split before launch: to the one-root-per-wave kernel
        if (l == 0) a.heavy[atomicAdd(a.n_heavy, 1ull)] = canon;
        continue;
      }
      const uint32_t s = (uint32_t)__builtin_ctzll((uint64_t)(~busy & full));
      bool derive = grouped;
      const uint64_t hk = a.pk_whandle ? bcast64(a.pk_whandle[i]) : ~0ull;
      if (hk != ~0ull) {  // the vertex bitmap an earlier launch kept for this root
        const uint64_t *hdr = a.pk_pool + hk;
        const uint64_t hv = hdr[l & (kPoolHdr - 1)];
        G.v0 = __builtin_amdgcn_readlane((uint32_t)hv, 0);
        G.d0 = __builtin_amdgcn_readlane((uint32_t)hv, 1);
        G.W0 = __builtin_amdgcn_readlane((uint32_t)hv, 2);
        G.xq0 = __builtin_amdgcn_readlane((uint32_t)hv, 3);
        G.rp = __builtin_amdgcn_readlane((uint32_t)hv, 4);
        G.o0 = readlane64(hv, 5);
        G.rfirst = readlane64(hv, 6);
        G.lh0 = readlane64(hv, 7);
        G.T = hdr + kPoolHdr;
        G.cm = G.T + (uint64_t)G.W0 * G.rp;
        G.lh = G.cm + G.W0;
        derive = true;
      }
      uint64_t topV[NW], px = 0;
      const uint32_t built = derive ? pk_derive<NW, NX>(w, G, s, canon, acc, cnt, hsh, topV, px)
                                    : pk_build<NW, NX>(w, scratch, s, canon, acc, cnt, hsh, topV, px);
      if (built & 1) {  // the top node: every row scanned, and the pivot's read unless it is pruned
        const uint32_t p = (uint32_t)px, Wr = (p + 63) / 64;
        acc.nodes += 1;
        acc.words += (uint64_t)(p + (uint32_t)(px >> 32) + (built == 1)) * Wr;
        if (built == 3 && a.root_nodes && l == 0) atomicAdd(&a.root_nodes[canon], 1ull);
      }
      if (built == 2) {  // too wide for this variant: to the next launch
        if (grouped && a.wide_h) {
          if (l == 0) G.wide[nwide] = canon;
          ++nwide;
        } else if (l == 0) {
          const unsigned long long at = atomicAdd(a.n_wide, 1ull);
          a.wide[at] = canon;
          if (a.wide_h) a.wide_h[at] = hk;
        }
      }
      if (built == 1) {  // the top node's record: lane f writes field f
        uint64_t v = 0;
        const uint32_t p = (uint32_t)px, xq = (uint32_t)(px >> 32);
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          v = l == C::oP + q ? low_mask(p > 64u * q ? p - 64u * q : 0u) : v;
          v = l == C::oV + q ? topV[q] : v;
          pending += (uint32_t)__popcll(topV[q]);
        }
#pragma unroll
        for (int j = 0; j < NX; ++j) v = l == C::oXX + j ? low_mask(xq > 64u * j ? xq - 64u * j : 0u) : v;
        v = l == C::oKey ? *w.m(mKey, s) : v;
        v = l == C::oMeta ? ((uint64_t)(64 * NW) << 40) | ((uint64_t)s << 16) : v;
        if (l < C::RS) fld(l, top) = v;
        wave_fence();
        ++top;
        busy |= 1u << s;
      }
    }
    if (__builtin_expect_with_probability(top == 0, 0, 0.999)) {  // no records and no roots left (see the refill condition)
      if (!sharing || !wait_mail()) break;
      continue;
    }

    // A look for idle waves, used at the end of the pass.
    const unsigned long long seen = sharing && (++tick & (kPackPoll - 1)) == 0 ? state_poll(a) : 0ull;

    // Dispatch up to 64 tasks from the top of the stack: look-lane i sees
    // record top-1-i; task lane l takes candidate k of look-record ri.
    const uint32_t nlook = top < 64 ? top : 64;
    uint32_t ci = 0;
    uint64_t lrem[NW], lmeta = 0;
#pragma unroll
    for (int q = 0; q < NW; ++q) lrem[q] = 0;
    if (l < nlook) {
      const uint32_t r = top - 1 - l;
      lmeta = fld(C::oMeta, r);
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        lrem[q] = fld(C::oV + q, r) & range_word(lmeta, q);
        ci += (uint32_t)__popcll(lrem[q]);
      }
    }
    const uint32_t lslot = (uint32_t)(lmeta >> 16) & 0xFF;
    const uint32_t incl = wave_scan_add_u32(ci), excl = incl - ci;
    uint32_t T = __builtin_amdgcn_readlane(incl, 63);  // tasks in the top 64 records: min(pending, 64) or more
    T = T < 64 ? T : 64u;
    if (top > a.pk_thr) {  // deep stack: expand the top record only
      const uint32_t c0 = __builtin_amdgcn_readlane(ci, 0);
      T = T < c0 ? T : c0;
    }
    const bool lfull = l < nlook && incl <= T;
    const bool lpart = l < nlook && excl < T && incl > T;
    const uint32_t nfull = (uint32_t)__popcll(__ballot(lfull));
    map32[l] = 0;
    wave_fence();
    if (l < nlook && ci && excl < T) map32[excl] = ((l + 1) << 8) | excl;
    wave_fence();
    const uint32_t mv = wave_scan_max_u32(l < T ? map32[l] : 0u);
    const bool act = l < T;
    const uint32_t ri = act ? (mv >> 8) - 1 : 0u, k = act ? l - (mv & 0xFF) : 0u;

    // The task's parent record.
    uint64_t R[NW], P[NW], XP[NW], V[NW], XX[NX], key = 0;
    uint32_t meta = 0, t = 0;
#pragma unroll
    for (int q = 0; q < NW; ++q) R[q] = P[q] = XP[q] = V[q] = 0;
#pragma unroll
    for (int j = 0; j < NX; ++j) XX[j] = 0;
    if (act) {
      const uint32_t r = top - 1 - ri;
      const uint64_t m64 = fld(C::oMeta, r);
      uint64_t rem[NW];
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        if (lists) R[q] = fld(C::oR + q, r);
        P[q] = fld(C::oP + q, r);
        XP[q] = fld(C::oX + q, r);
        V[q] = fld(C::oV + q, r);
        rem[q] = V[q] & range_word(m64, q);
      }
#pragma unroll
      for (int j = 0; j < NX; ++j) XX[j] = fld(C::oXX + j, r);
      key = fld(C::oKey, r);
      meta = (uint32_t)m64;
      // t = the k-th remaining candidate
      uint32_t kk = k, base = 0;
#pragma unroll
      for (int q = 0; q < NW - 1; ++q) {
        const uint32_t cq = (uint32_t)__popcll(rem[q]);
        if (base == (uint32_t)q * 64 && kk >= cq) {
          kk -= cq;
          base = (uint32_t)(q + 1) * 64;
        }
      }
      uint64_t rw = rem[0];
#pragma unroll
      for (int q = 1; q < NW; ++q)
        if (base == (uint32_t)q * 64) rw = rem[q];
      t = base + select64(rw, kk);
    }
    // A child's P | XP lies within its parent's P | XP: when no parent of
    // this pass reaches the last word, the tasks skip that word of every row
    // they scan.
    const bool wlast = NW == 1 || __ballot(act && (P[NW - 1] | XP[NW - 1]) != 0) != 0;
    wave_fence();  // every parent is read before records are rewritten below
    if (lpart) {   // the partly taken record keeps its candidates from the (T - excl)-th on
      uint32_t kk = T - excl, base = 0;
#pragma unroll
      for (int q = 0; q < NW - 1; ++q) {
        const uint32_t cq = (uint32_t)__popcll(lrem[q]);
        if (base == (uint32_t)q * 64 && kk >= cq) {
          kk -= cq;
          base = (uint32_t)(q + 1) * 64;
        }
      }
      uint64_t rw = lrem[0];
#pragma unroll
      for (int q = 1; q < NW; ++q)
        if (base == (uint32_t)q * 64) rw = lrem[q];
      const uint32_t first = base + select64(rw, kk);
      fld(C::oMeta, top - 1 - l) = (lmeta & ~(0xFFull << 32)) | ((uint64_t)first << 32);
    }
    if (lfull) __hip_atomic_fetch_sub(w.m(mRefs, lslot), (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    top -= nfull;
    given = given < top ? given : top;

    // The task: one tree node per lane.
    const uint32_t s = (meta >> 16) & 0xFF;
    bool branch = false;
    if (act) {
      const lds64 *sl = w.slot(s);
      const uint64_t px = *w.m(mPX, s);
      const uint32_t p = (uint32_t)px;
      const uint32_t Wr = (p + 63) / 64;  // the root's own width (accounting as the other kernel)
      uint32_t rsize, xpop = 0;  // xpop: rows of the parent's XX
      {
        // Child of candidate t: the parent's candidates below t have moved
        // from P to XP, as when the sequential search reaches t.
        const uint32_t jt = t >> 6, bt = t & 63;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          const uint64_t below = (uint32_t)q < jt ? V[q] : ((uint32_t)q == jt ? V[q] & low_mask(bt) : 0ull);
          const uint64_t rt = sl[C::sProw + t * NW + q];
          P[q] = P[q] & ~below & rt;
          XP[q] = (XP[q] | below) & rt;
          R[q] |= (uint32_t)q == jt ? 1ull << bt : 0ull;
        }
#pragma unroll
        for (int j = 0; j < NX; ++j) {
          xpop += (uint32_t)__popcll(XX[j]);
          XX[j] &= sl[C::sXcol + t * NX + j];
        }
        key += sl[C::sG + t];
        rsize = (meta & 0xFFFF) + 1;
        words += Wr;
      }
      // Row scans: the rows of P0 and X0' follow each other in the slot, so row
      // r (P0 rows first, then 64 NW + x) is at r * NW.  Two rows a pass, both
      // loads in flight before either is used; a lane goes on to its next word
      // when one is used up, so that a pass of the wave is lost only to the
      // lane with the most rows, not once per word.
      auto row_pair = [&](uint64_t &m, uint32_t wb, uint64_t &b0, uint64_t &b1, uint32_t &i0, uint32_t &i1,
                          uint64_t (&r0)[NW], uint64_t (&r1)[NW], uint32_t &c0, uint32_t &c1) {
        b0 = m & (~m + 1);
        m ^= b0;
        b1 = m & (~m + 1);
        m ^= b1;
        i0 = wb + (uint32_t)__builtin_ctzll(b0);
        i1 = b1 ? wb + (uint32_t)__builtin_ctzll(b1) : i0;
#pragma unroll
        for (int z = 0; z < NW; ++z) {
          r0[z] = z + 1 < NW || wlast ? (uint64_t)sl[i0 * NW + z] : 0ull;
          r1[z] = z + 1 < NW || wlast ? (uint64_t)sl[i1 * NW + z] : 0ull;
        }
        c0 = c1 = 0;
#pragma unroll
        for (int z = 0; z < NW; ++z) {
          if (z + 1 < NW || wlast) {
            c0 += (uint32_t)__popcll(P[z] & ~r0[z]);
            c1 += (uint32_t)__popcll(P[z] & ~r1[z]);
          }
        }
      };
      // P' against itself: aggressive node generation moves every vertex
      // adjacent to all of P' \ {itself} (it misses one: itself) to R, and the
      // others' counts are those of the pivot choice - the moved vertices are
      // adjacent to all of them, so P' without them gives the same counts.
      uint32_t psz = 0, best = ~0u;
#pragma unroll
      for (int q = 0; q < NW; ++q) psz += (uint32_t)__popcll(P[q]);
      bool anym = false;
      if (psz == 1) {
        uint32_t i = 0;
#pragma unroll
        for (int q = NW - 1; q >= 0; --q)
          if (P[q]) i = 64u * q + (uint32_t)__builtin_ctzll(P[q]);
        best = (1u << 16) | i;
      } else if (psz > 1) {
        uint64_t mk[NW], xacc[NW], nx[NW];
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          mk[q] = 0;
          xacc[q] = ~0ull;
          nx[q] = P[q];
        }
        uint32_t wb = 0;
        for (;;) {
          uint64_t left = 0;
#pragma unroll
          for (int q = 0; q < NW; ++q) left |= nx[q];
          if (left == 0) break;
          if (NW > 1 && nx[0] == 0) {
#pragma unroll
            for (int q = 0; q + 1 < NW; ++q) nx[q] = nx[q + 1];
            nx[NW - 1] = 0;
            wb += 64;
          }
          uint64_t b0, b1, r0[NW], r1[NW];
          uint32_t i0, i1, c0, c1;
          row_pair(nx[0], wb, b0, b1, i0, i1, r0, r1, c0, c1);
          const bool mv0 = c0 == 1, mv1 = c1 == 1 && b1;
          if (mv0 || mv1) {
#pragma unroll
            for (int q = 0; q < NW; ++q)
              mk[q] |= wb == 64u * q ? (mv0 ? b0 : 0ull) | (mv1 ? b1 : 0ull) : 0ull;
#pragma unroll
            for (int z = 0; z < NW; ++z)
              if (z + 1 < NW || wlast) xacc[z] &= (mv0 ? r0[z] : ~0ull) & (mv1 ? r1[z] : ~0ull);
          }
          const uint32_t k0 = mv0 ? ~0u : (c0 << 16) | i0, k1 = mv1 ? ~0u : (c1 << 16) | i1;
          best = k0 < best ? k0 : best;
          best = k1 < best && b1 ? k1 : best;
        }
        words += (uint64_t)psz * Wr;
        uint32_t nm = 0;
#pragma unroll
        for (int q = 0; q < NW; ++q) nm += (uint32_t)__popcll(mk[q]);
        if (nm) {
          anym = true;
#pragma unroll
          for (int q = 0; q < NW; ++q) {
            R[q] |= mk[q];
            P[q] &= ~mk[q];
            XP[q] &= xacc[q];
            for (uint64_t m = mk[q]; m; m &= m - 1) {
              const uint32_t i = 64u * q + (uint32_t)__builtin_ctzll(m);
#pragma unroll
              for (int j = 0; j < NX; ++j) XX[j] &= sl[C::sXcol + i * NX + j];
              key += sl[C::sG + i];
            }
          }
          rsize += nm;
          words += (uint64_t)nm * Wr;
          psz -= nm;
        }
      }
      words += (uint64_t)xpop * (anym ? Wr + 1 : 1);
      // Evaluate the node.
      uint32_t cw = 0, xw = 0;
      uint64_t xany = 0;
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        cw += (uint32_t)__popcll(P[q] | XP[q]);
        xany |= XP[q];
      }
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        xw += (uint32_t)__popcll(XX[j]);
        xany |= XX[j];
      }
      ++nodes;
      if (a.root_nodes) __hip_atomic_fetch_add(w.m(mNodes, s), (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (psz == 0) {
        if (xany == 0) pk_emit<NW, NX, LISTS>(w, s, (uint32_t)*w.m(mBase, s) + rsize, key, R, cnt, hsh);
      } else {
        words += (uint64_t)(cw + xw) * Wr;
        // pivot: (|P' \ N(u)|, row) argmin over P' (above), then XP' and XX';
        // an excluded row that covers P' ends the scan (the minimum does not
        // depend on the order rows are visited in).
        uint64_t nx[NW + NX];
#pragma unroll
        for (int q = 0; q < NW; ++q) nx[q] = XP[q];
#pragma unroll
        for (int j = 0; j < NX; ++j) nx[NW + j] = XX[j];
        uint32_t wb = 0;
        bool zero = false;
        for (;;) {
          uint64_t left = 0;
#pragma unroll
          for (int q = 0; q < NW + NX; ++q) left |= nx[q];
          if (left == 0 || zero) break;
          if (nx[0] == 0) {
#pragma unroll
            for (int q = 0; q + 1 < NW + NX; ++q) nx[q] = nx[q + 1];
            nx[NW + NX - 1] = 0;
            wb += 64;
          }
          if (nx[0]) {
            uint64_t b0, b1, r0[NW], r1[NW];
            uint32_t i0, i1, c0, c1;
            row_pair(nx[0], wb, b0, b1, i0, i1, r0, r1, c0, c1);
            const uint32_t k0 = (c0 << 16) | i0, k1 = (c1 << 16) | i1;
            best = k0 < best ? k0 : best;
            best = k1 < best ? k1 : best;
            zero = c0 == 0 || c1 == 0;
          }
        }
        if (!zero) {  // else an excluded row covers P': no maximal clique below
          words += Wr;
          const lds64 *pr = sl + (best & 0xFFFF) * NW;
#pragma unroll
          for (int q = 0; q < NW; ++q) V[q] = P[q] & ~(uint64_t)pr[q];
          branch = true;
        }
      }
      meta = (meta & 0x00FF0000u) | rsize;
    }

    // Push the branching nodes' records (the children of the deepest
    // records highest) and account.
    uint64_t bm = __ballot(branch);
    if (top + (uint32_t)__popcll(bm) > a.pk_cap) {  // unreachable by the bound above; never write past the arena
      if (l == 0) atomicOr(a.err, kErrPackStack);
      bm = 0;
      branch = false;
    }
    const uint32_t npush = (uint32_t)__popcll(bm);
    uint32_t vc = 0;
    if (branch) {
      const uint32_t r = top + npush - 1 - rank_below(bm);
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        if (lists) fld(C::oR + q, r) = R[q];
        fld(C::oP + q, r) = P[q];
        fld(C::oX + q, r) = XP[q];
        fld(C::oV + q, r) = V[q];
        vc += (uint32_t)__popcll(V[q]);
      }
#pragma unroll
      for (int j = 0; j < NX; ++j) fld(C::oXX + j, r) = XX[j];
      fld(C::oKey, r) = key;
      fld(C::oMeta, r) = (uint64_t)meta | ((uint64_t)(64 * NW) << 40);  // every candidate remains
      __hip_atomic_fetch_add(w.m(mRefs, s), (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    const uint32_t vsum = __builtin_amdgcn_readlane(wave_scan_add_u32(vc), 63);
    top += npush;
    pending = pending - T + vsum;
    wave_fence();
    // Slots whose last record is consumed are done.
    const bool done = l < S && ((busy >> l) & 1) && *w.m(mRefs, l) == 0;
    const uint64_t dm = __ballot(done);
    if (a.root_nodes || a.root_graph)
      for (uint64_t d = dm; d; d &= d - 1) pk_finish<NW, NX>(w, (uint32_t)__builtin_ctzll(d));
    busy &= ~(uint32_t)dm;
    if (__builtin_expect_with_probability(__ballot((seen >> 32) != 0) != 0, 0, 0.999)) {
      // Of the working waves about one per idle one tries: when all tried,
      // they queued on the few idle waves' words.
      const uint32_t looking = __builtin_amdgcn_readlane(wave_scan_add_u32((uint32_t)(seen >> 32)), 63);
      const uint32_t working = __builtin_amdgcn_readlane(wave_scan_add_u32((uint32_t)seen), 63);
      const uint32_t h = (uint32_t)splitmix64_mix(((uint64_t)w.me << 32) | tick);
      if ((uint32_t)(((uint64_t)h * working) >> 32) < looking) give();
    }
  }

  // Exit: the wave's sums.
  acc.count = wave_sum64(cnt);
  acc.hash = wave_sum64(hsh);
  acc.words += wave_sum64(words);
  acc.nodes += wave_sum64(nodes);
  acc.build += 4 * wave_sum64(acc.scan);
  wave_fence();
  flush_sums(a, w.me, acc, w.L.hist);
}

// One kernel per variant and occupancy target (WPE waves per SIMD: the
// register budget 512 / WPE VGPRs).
template <int NW, int NX, int WPE, bool LISTS>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, 8))) void pack_kernel(KArgs a) {
  pack_main<NW, NX, LISTS>(a);
}

template <int NW, int NX>
hipError_t launch_variant(const KArgs &a, uint32_t waves, uint32_t wpc, size_t lds, hipStream_t stream) {
  // Runs that write clique lists carry R in every record: one instantiation
  // (4 waves per SIMD) for them, so the others hold no R at all.
  if (a.list)
    hipLaunchKernelGGL((pack_kernel<NW, NX, 4, true>), dim3(waves), dim3(64), lds, stream, a);
  else if (wpc <= 16)
    hipLaunchKernelGGL((pack_kernel<NW, NX, (NW == 1 ? 4 : 3), false>), dim3(waves), dim3(64), lds, stream, a);
  else if (wpc <= 20)
    hipLaunchKernelGGL((pack_kernel<NW, NX, 5, false>), dim3(waves), dim3(64), lds, stream, a);
  else if (wpc <= 24)
    hipLaunchKernelGGL((pack_kernel<NW, NX, 6, false>), dim3(waves), dim3(64), lds, stream, a);
  else
    hipLaunchKernelGGL((pack_kernel<NW, NX, 8, false>), dim3(waves), dim3(64), lds, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pack(const KArgs &a, int variant, uint32_t waves, uint32_t waves_per_cu, hipStream_t stream) {
  const bool batch = a.root_graph != nullptr;
  if (variant == 0) return launch_variant<1, 1>(a, waves, waves_per_cu, pack_lds_bytes(1, 1, a.pk_slots, batch), stream);
  if (variant == 1)
    return launch_variant<2, 2>(a, waves, waves_per_cu, pack_lds_bytes(2, 2, a.pk_slots, batch), stream);
  const size_t lds = pack_lds_bytes(2, 4, a.pk_slots, batch);
  if (a.list)
    hipLaunchKernelGGL((pack_kernel<2, 4, 3, true>), dim3(waves), dim3(64), lds, stream, a);
  else
    hipLaunchKernelGGL((pack_kernel<2, 4, 3, false>), dim3(waves), dim3(64), lds, stream, a);
  return hipGetLastError();
}

}  // namespace rdmce
