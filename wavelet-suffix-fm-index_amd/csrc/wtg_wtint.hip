// wtg_wtint.hip -- sdsl::wt_int<> on the GPU: construction
// (wt_int/wt_int_par.hpp:368-406: tree bits, rank_support_v, select_support_mcl
// for 1 and 0 over the concatenated tree) and batched queries, one lane per
// query (rank :553-577, access :519-541, inverse_select :588-611,
// select :622-660).  Queries are chains of dependent random accesses, so the
// kernels keep many independent waves in flight rather than using LDS.
#include "wtg_internal.hpp"
#include "wtg_order.hpp"
#include <cstring>

struct wtg_wtint {
  uint64_t n = 0, sigma = 0, nbits = 0;
  uint32_t L = 0;
  uint64_t* words = nullptr;
  uint64_t* dir = nullptr;
  wtg_select s1{}, s0{};
};

struct WtQ {
  const uint64_t* words;
  const uint64_t* D;
  SelQ s1, s0;
  uint64_t n, W;
  uint32_t L;
  uint32_t apart;  // q_apart
};

// Every level of a walk looks up two to four positions whose loads do not
// depend on each other: all are issued before the first is used (one round trip
// to memory per level; with a rank after the other there were as many as
// lookups).  10^6 queries each on a 20-level tree of 2^24 symbols: rank 593 ->
// 540 us, access 850 -> 554, select 953 -> 897, lex_count 1030 -> 843,
// range_count 2157 -> 1540: 128-byte lines from behind the L2 at 7.4 TB/s, the same in
// every one of them.  Ordered batches below.
// APART (q_apart): a lookup's word once its entry is there, and only then the next lookup.
template <bool APART, uint32_t N>
__device__ __forceinline__ void wt_fetch(const WtQ& w, const uint64_t (&at)[N], RankAt (&f)[N]) {
#pragma unroll
  for (uint32_t k = 0; k < N; k++) {
    rank9_entry(f[k], w.D, at[k]);
    if constexpr (APART) asm volatile("" : "+v"(f[k].base));  // waits for the entry
    rank9_word(f[k], w.words, w.W);
  }
}

// A batch's columns as they came and, where it was to be put in order, in order,
// with the places the queries had; asis: it was in order, the others were not written.
struct QBatch {
  QCols came, put;
  const uint32_t *place, *asis;
};
// the query of this thread: where its columns are (p) and its answer goes (q); not
// in the batch past its end.  The grid of a batch to be put in order is a multiple of the XCDs.
struct QSlot {
  uint64_t p, q;
  bool put, in;
};
__device__ __forceinline__ QSlot q_slot(const QBatch& b, uint64_t nq) {
  QSlot s;
  s.put = b.place && *b.asis == 0;
  const uint32_t blk = s.put ? (blockIdx.x % QO_XCDS) * (gridDim.x / QO_XCDS) + blockIdx.x / QO_XCDS : blockIdx.x;
  s.p = (uint64_t)blk * blockDim.x + threadIdx.x;
  s.in = s.p < nq;
  s.q = s.in && s.put ? b.place[s.p] : s.p;
  return s;
}
__device__ __forceinline__ uint64_t q_col(const QBatch& b, const QSlot& s, uint32_t c) {
  return (s.put ? b.put.c[c] : b.came.c[c])[s.p];
}

// the walk of c from the root: i becomes rank(i, c), the result the number of values
// below c in [0, i) (wt_int/wt_int_par.hpp:553-577, :753-780)
template <bool APART>
__device__ __forceinline__ uint64_t rank_walk(const WtQ& w, uint64_t& i, uint64_t c) {
  uint64_t offset = 0, mask = 1ull << (w.L - 1), node_size = w.n, res = 0;
  for (uint32_t k = 0; k < w.L && i; k++) {
    RankAt f[3];
    wt_fetch<APART>(w, {offset, offset + i, offset + node_size}, f);
    const uint64_t o = rank9_of(f[0]), oi = rank9_of(f[1]) - o, oe = rank9_of(f[2]) - o;
    if (c & mask) { offset += node_size - oe; node_size = oe; res += i - oi; i = oi; }
    else { node_size -= oe; i -= oi; }
    offset += w.n;
    mask >>= 1;
  }
  return res;
}

__global__ void k_wtint_rank(WtQ w, QBatch b, uint64_t nq, uint64_t* __restrict__ out) {
  const QSlot slot = q_slot(b, nq);
  if (!slot.in) return;
  const uint64_t q = slot.q;
  uint64_t i = q_col(b, slot, 0);
  const uint64_t c = q_col(b, slot, 1);
  if (i > w.n) { out[q] = WTG_NONE; return; }
  if (w.L < 64 && (1ull << w.L) <= c) { out[q] = 0; return; }
  if (w.apart && !slot.put) rank_walk<true>(w, i, c);
  else rank_walk<false>(w, i, c);
  out[q] = i;
}

// lex_count traversal (wt_int/wt_int_par.hpp:712-741): rank(i,c) and the number
// of values below / above c in [i, j)
struct LexWalk {
  uint64_t c, i, j, offset, size, smaller, greater;
  bool out;  // c is no symbol: nothing to walk
};
__device__ __forceinline__ LexWalk lex_begin(const WtQ& w, uint64_t i, uint64_t j, uint64_t c) {
  LexWalk x{c, i, j, 0, w.n, 0, 0, w.L < 64 && (1ull << w.L) <= c};
  if (x.out) { x.i = 0; x.smaller = j - i; }
  return x;
}
struct LexAt {
  RankAt f[4];
};
template <bool APART>
__device__ __forceinline__ void lex_fetch(const WtQ& w, const LexWalk& x, LexAt& a) {
  wt_fetch<APART>(w, {x.offset, x.offset + x.i, x.offset + x.j, x.offset + x.size}, a.f);
}
__device__ __forceinline__ void lex_step(const WtQ& w, LexWalk& x, const LexAt& a, uint64_t mask) {
  const uint64_t o = rank9_of(a.f[0]), oi = rank9_of(a.f[1]) - o, oj = rank9_of(a.f[2]) - o, oe = rank9_of(a.f[3]) - o;
  if (x.c & mask) {
    x.offset += x.size - oe;
    x.size = oe;
    x.smaller += (x.j - x.i) - (oj - oi);
    x.i = oi;
    x.j = oj;
  } else {
    x.size -= oe;
    x.greater += oj - oi;
    x.i -= oi;
    x.j -= oj;
  }
  x.offset += w.n;
}
template <bool APART>
__device__ __forceinline__ void lex_walk(const WtQ& w, LexWalk& x) {
  uint64_t mask = 1ull << (w.L - 1);
  for (uint32_t k = 0; k < w.L; k++, mask >>= 1) {
    LexAt a;
    lex_fetch<APART>(w, x, a);
    lex_step(w, x, a, mask);
  }
}
__device__ __forceinline__ void wtint_lex(const WtQ& w, bool apart, uint64_t i, uint64_t j, uint64_t c, uint64_t& rk,
                                          uint64_t& sm, uint64_t& gr) {
  LexWalk x = lex_begin(w, i, j, c);
  if (!x.out) {
    if (apart) lex_walk<true>(w, x);
    else lex_walk<false>(w, x);
  }
  rk = x.i;
  sm = x.smaller;
  gr = x.greater;
}

__global__ void k_wtint_lex_count(WtQ w, QBatch b, uint64_t nq, uint64_t* __restrict__ out_rank,
                                  uint64_t* __restrict__ out_smaller, uint64_t* __restrict__ out_greater) {
  const QSlot slot = q_slot(b, nq);
  if (!slot.in) return;
  const uint64_t q = slot.q, i = q_col(b, slot, 0), j = q_col(b, slot, 1), c = q_col(b, slot, 2);
  uint64_t rk = WTG_NONE, sm = WTG_NONE, gr = WTG_NONE;
  if (i <= j && j <= w.n) wtint_lex(w, w.apart && !slot.put, i, j, c, rk, sm, gr);
  out_rank[q] = rk;
  out_smaller[q] = sm;
  out_greater[q] = gr;
}

// lex_smaller_count (wt_int/wt_int_par.hpp:753-780): rank(i,c) and the number of
// values below c in [0, i)
__global__ void k_wtint_lex_smaller(WtQ w, QBatch b, uint64_t nq, uint64_t* __restrict__ out_rank,
                                    uint64_t* __restrict__ out_smaller) {
  const QSlot slot = q_slot(b, nq);
  if (!slot.in) return;
  const uint64_t q = slot.q;
  uint64_t i = q_col(b, slot, 0);
  const uint64_t c = q_col(b, slot, 1);
  if (i > w.n) { out_rank[q] = out_smaller[q] = WTG_NONE; return; }
  if (w.L < 64 && (1ull << w.L) <= c) { out_rank[q] = 0; out_smaller[q] = i; return; }
  const uint64_t res = w.apart && !slot.put ? rank_walk<true>(w, i, c) : rank_walk<false>(w, i, c);
  out_rank[q] = i;
  out_smaller[q] = res;
}

// range_search_2d count (wt_int/wt_int_par.hpp:801-870, report = false): the
// positions in [lb, rb] with values in [vlb, vrb], as the difference of two
// lex_count "smaller" counts over [lb, rb + 1).  The reference clamps vrb to 2^L
// and its leaf test does not compare vlb, so vlb = 2^L counts the value 2^L - 1:
// vlb is clamped to 2^L - 1 the same way.
template <bool APART>
__global__ void k_wtint_range_count(WtQ w, QBatch b, uint64_t nq, uint64_t* __restrict__ out) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  const uint64_t lb = b.came.c[0][q], rb = b.came.c[1][q];
  uint64_t vlb = b.came.c[2][q], vrb = b.came.c[3][q];
  if (rb >= w.n) { out[q] = WTG_NONE; return; }
  const uint64_t top = w.L < 64 ? (1ull << w.L) : ~0ull;
  if (vrb > top) vrb = top;
  if (vlb > vrb || lb > rb) { out[q] = 0; return; }
  if (w.L < 64 && vlb > top - 1) vlb = top - 1;
  // both walks level by level together (every value is <= vrb: the upper one has no steps)
  LexWalk lo = lex_begin(w, lb, rb + 1, vlb), hi = lex_begin(w, lb, rb + 1, vlb);
  const bool all = w.L < 64 ? vrb >= top - 1 : vrb == ~0ull;
  if (all) hi.smaller = rb + 1 - lb;
  else hi.c = vrb + 1;
  uint64_t mask = 1ull << (w.L - 1);
  for (uint32_t k = 0; k < w.L; k++, mask >>= 1) {
    LexAt al, ah{};
    lex_fetch<APART>(w, lo, al);
    if (!all) lex_fetch<APART>(w, hi, ah);
    lex_step(w, lo, al, mask);
    if (!all) lex_step(w, hi, ah, mask);
  }
  out[q] = hi.smaller - lo.smaller;
}

// The same in two walks for an ordered batch (each ordered by its own bound):
// the lower one leaves its count or a mark, the upper one takes it from there.
constexpr uint64_t WT_RANGE_EMPTY = WTG_NONE - 1;
template <bool UPPER>
__global__ void k_wtint_range_half(WtQ w, QBatch b, uint64_t nq, uint64_t* __restrict__ out) {
  const QSlot slot = q_slot(b, nq);
  if (!slot.in) return;
  const uint64_t q = slot.q, lb = q_col(b, slot, 0), rb = q_col(b, slot, 1);
  const uint64_t top = w.L < 64 ? (1ull << w.L) : ~0ull;
  uint64_t v = q_col(b, slot, 2), rk, below, gr;
  const bool apart = w.apart && !slot.put;
  if (UPPER) {
    const uint64_t low = out[q];
    if (low == WTG_NONE) return;
    if (low == WT_RANGE_EMPTY) { out[q] = 0; return; }
    if (v >= top - (w.L < 64 ? 1 : 0)) below = rb + 1 - lb;  // every value is <= v
    else wtint_lex(w, apart, lb, rb + 1, v + 1, rk, below, gr);
    out[q] = below - low;
  } else {
    uint64_t vrb = q_col(b, slot, 3);
    if (rb >= w.n) { out[q] = WTG_NONE; return; }
    if (vrb > top) vrb = top;
    if (v > vrb || lb > rb) { out[q] = WT_RANGE_EMPTY; return; }
    if (w.L < 64 && v > top - 1) v = top - 1;
    wtint_lex(w, apart, lb, rb + 1, v, rk, below, gr);
    out[q] = below;
  }
}

__global__ void k_wtint_access(WtQ w, QBatch b, uint64_t nq, uint64_t* __restrict__ out_sym,
                               uint64_t* __restrict__ out_rank) {
  const QSlot slot = q_slot(b, nq);
  if (!slot.in) return;
  const uint64_t q = slot.q;
  uint64_t i = q_col(b, slot, 0);
  if (i >= w.n) {
    out_sym[q] = WTG_NONE;
    if (out_rank) out_rank[q] = WTG_NONE;
    return;
  }
  uint64_t offset = 0, res = 0, node_size = w.n;
  for (uint32_t k = 0; k < w.L; k++) {
    res <<= 1;
    RankAt f[3];
    wt_fetch<false>(w, {offset, offset + i, offset + node_size}, f);
    const uint64_t o = rank9_of(f[0]), oi = rank9_of(f[1]) - o, oe = rank9_of(f[2]) - o;
    if ((f[1].word >> ((offset + i) & 63)) & 1ull) { offset += node_size - oe; node_size = oe; i = oi; res |= 1; }
    else { node_size -= oe; i -= oi; }
    offset += w.n;
  }
  out_sym[q] = res;
  if (out_rank) out_rank[q] = i;
}

template <uint32_t MAXL>  // the tree's levels are at most MAXL
__global__ void k_wtint_select(WtQ w, QBatch b, uint64_t nq, uint64_t* __restrict__ out) {
  const QSlot slot = q_slot(b, nq);
  if (!slot.in) return;
  const uint64_t q = slot.q;
  uint64_t i = q_col(b, slot, 0);
  const uint64_t c = q_col(b, slot, 1);
  uint64_t path_off[MAXL + 1], path_rank[MAXL + 1];
  uint64_t offset = 0, mask = 1ull << (w.L - 1), node_size = w.n;
  path_off[0] = path_rank[0] = 0;
  for (uint32_t k = 0; k < w.L && node_size; k++) {
    RankAt f[2];
    wt_fetch<false>(w, {offset, offset + node_size}, f);
    const uint64_t o = rank9_of(f[0]), oe = rank9_of(f[1]) - o;
    path_rank[k] = o;
    if (c & mask) { offset += node_size - oe; node_size = oe; }
    else node_size -= oe;
    offset += w.n;
    path_off[k + 1] = offset;
    mask >>= 1;
  }
  if (i == 0 || node_size == 0 || node_size < i || (w.L < 64 && (c >> w.L) != 0)) {
    out[q] = WTG_NONE;  // the reference throws std::logic_error here
    return;
  }
  mask = 1;
  for (uint32_t k = w.L; k > 0; k--) {
    offset = path_off[k - 1];
    const uint64_t o = path_rank[k - 1];
    if (c & mask) i = select_plain(w.s1, o + i) - offset + 1;
    else i = select_plain(w.s0, offset - o + i) - offset + 1;
    mask <<= 1;
  }
  out[q] = i - 1;
}

// Whether a batch of nq symbol queries that is walked as it came takes one lookup's
// entry and word after the other.  With all of a level in flight at once a large batch on levels larger
// than an L2 asks for lines again that are on their way: 2^18 lex_counts on 2^27 bits in
// 4 levels take 2.6 M lines from behind the L2s, and 1.3 M so.
// us at once -> apart, rank / lex_count:
//   2^27 bits, 4 levels: 2^17 25 -> 27, 34 -> 32; 2^18 38 -> 31, 59 -> 40; 2^20 113 -> 104, 199 -> 187
//              8 levels: 2^17 31 -> 34, 46 -> 42; 2^18 53 -> 40, 82 -> 58; 2^20 189 -> 176, 307 -> 313
//   2^26 bits, 8 levels: 2^17 28 -> 31, 38 -> 38; 2^18 42 -> 37, 63 -> 53; 2^20 136 -> 129, 209 -> 214
//   2^20 bits, 10 levels: 2^12 17 -> 20, 19 -> 21; 2^18 27 -> 27, 34 -> 34; 2^20 66 -> 71, 90 -> 101
static bool q_apart(const wtg_wtint* wt, uint64_t nq) { return wt->nbits >= 1ull << 26 && nq >= 1ull << 18; }

static WtQ make_q(const wtg_wtint* wt, uint64_t nq) {
  WtQ w{};
  w.words = wt->words;
  w.D = wt->dir;
  const uint64_t W = (wt->nbits + 63) / 64;
  w.s1 = SelQ{wt->s1.superblock, wt->s1.mini, wt->s1.long_index, wt->s1.long_pool, wt->words, W, 1};
  w.s0 = SelQ{wt->s0.superblock, wt->s0.mini, wt->s0.long_index, wt->s0.long_pool, wt->words, W, 0};
  w.n = wt->n;
  w.W = W;
  w.L = wt->L;
  w.apart = q_apart(wt, nq);
  return w;
}

extern "C" int wtg_wtint_build(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n,
                               uint32_t max_level, wtg_wtint** out) {
  WTG_REQUIRE(ctx && out && (n == 0 || d_sym), "wtg_wtint_build: null argument");
  WTG_REQUIRE(sym_bytes == 1 || sym_bytes == 2 || sym_bytes == 4 || sym_bytes == 8, "bad sym_bytes");
  WTG_TRY(wtg_set_device(ctx));
  *out = nullptr;
  wtg_wtint* wt = new wtg_wtint();
  wt->n = n;
  int rc = WTG_OK;
  uint32_t L = max_level;
  if (n == 0) {  // wt_int_par.hpp:373-374: empty tree
    wt->L = max_level;
    *out = wt;
    return WTG_OK;
  }
  if (L == 0) {  // :384-392: max_level = hi(max(1, max value)) + 1
    uint64_t mx = 0;
    if ((rc = wtg_max_value(ctx, d_sym, sym_bytes, n, &mx)) != WTG_OK) { delete wt; return rc; }
    if (mx < 1) mx = 1;
    L = (uint32_t)wtg_hi_host(mx) + 1;
  }
  wt->L = L;
  wt->nbits = n * L;
  const uint64_t nw = wtg_levels_words(n, L);
  unsigned long long* d_distinct = (unsigned long long*)((char*)ctx->d_small + 128);
  if ((rc = wtg_malloc(ctx, (void**)&wt->words, nw * 8)) != WTG_OK) goto fail;
  if ((rc = wtg_malloc(ctx, (void**)&wt->dir, wtg_rank9_words(wt->nbits) * 8)) != WTG_OK) goto fail;
  if ((rc = wtg_levels_build_async(ctx, d_sym, sym_bytes, n, L, wt->words, nullptr, 0, d_distinct)) != WTG_OK)
    goto fail;
  // the distinct count rides the stream into pinned memory; the support build
  // right behind the tree reads its count of ones with a sync, after which the
  // count is there (no sync of its own, no idle gap between tree and supports)
  if (hipMemcpyAsync(ctx->h_stage + WTG_STAGE_AUX, d_distinct, 8, hipMemcpyDeviceToHost, ctx->stream) !=
      hipSuccess) {
    wtg_set_error("wtg_wtint_build: copy failed");
    rc = WTG_ERR_HIP;
    goto fail;
  }
  if ((rc = wtg_rank_select_run(ctx, wt->words, wt->nbits, wt->dir, true, &wt->s1, &wt->s0)) != WTG_OK)
    goto fail;
  if ((rc = wtg_finish(ctx)) != WTG_OK) goto fail;
  if (hipStreamSynchronize(ctx->stream) != hipSuccess) {  // (a no-op wait: the supports synced)
    wtg_set_error("wtg_wtint_build: sync failed");
    rc = WTG_ERR_HIP;
    goto fail;
  }
  wt->sigma = *reinterpret_cast<volatile unsigned long long*>(ctx->h_stage + WTG_STAGE_AUX);
  *out = wt;
  return WTG_OK;
fail:
  wtg_wtint_destroy(ctx, wt);
  return rc;
}

extern "C" int wtg_wtint_from_tree(wtg_ctx* ctx, const uint64_t* d_tree, uint64_t n, uint32_t levels,
                                   uint64_t sigma, wtg_wtint** out) {
  WTG_REQUIRE(ctx && out && (n == 0 || d_tree), "wtg_wtint_from_tree: null argument");
  WTG_REQUIRE(levels <= 64, "wtg_wtint_from_tree: levels > 64");
  WTG_TRY(wtg_set_device(ctx));
  *out = nullptr;
  wtg_wtint* wt = new wtg_wtint();
  wt->n = n;
  wt->L = levels;
  wt->sigma = sigma;
  if (n == 0 || levels == 0) {
    *out = wt;
    return WTG_OK;
  }
  wt->nbits = n * levels;
  const uint64_t nw = wtg_levels_words(n, levels);
  int rc = WTG_OK;
  if ((rc = wtg_malloc(ctx, (void**)&wt->words, (nw + 1) * 8)) != WTG_OK) goto fail;
  if ((rc = wtg_malloc(ctx, (void**)&wt->dir, wtg_rank9_words(wt->nbits) * 8)) != WTG_OK) goto fail;
  if ((rc = wtg_fill_u64(ctx, wt->words + nw, 1, 0)) != WTG_OK) goto fail;
  if (hipMemcpyAsync(wt->words, d_tree, nw * 8, hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess) {
    wtg_set_error("wtg_wtint_from_tree: copy failed");
    rc = WTG_ERR_HIP;
    goto fail;
  }
  if ((rc = wtg_rank_select_run(ctx, wt->words, wt->nbits, wt->dir, true, &wt->s1, &wt->s0)) != WTG_OK)
    goto fail;
  if ((rc = wtg_finish(ctx)) != WTG_OK) goto fail;
  *out = wt;
  return WTG_OK;
fail:
  wtg_wtint_destroy(ctx, wt);
  return rc;
}

extern "C" int wtg_wtint_destroy(wtg_ctx* ctx, wtg_wtint* wt) {
  if (!wt) return WTG_OK;
  WTG_REQUIRE(ctx, "null ctx");
  wtg_free(ctx, wt->words);
  wtg_free(ctx, wt->dir);
  wtg_select_free(ctx, &wt->s1);
  wtg_select_free(ctx, &wt->s0);
  delete wt;
  return WTG_OK;
}

extern "C" int wtg_wtint_info(const wtg_wtint* wt, uint64_t* n, uint32_t* levels, uint64_t* sigma,
                              const uint64_t** d_words, const uint64_t** d_dir) {
  WTG_REQUIRE(wt, "null wt");
  if (n) *n = wt->n;
  if (levels) *levels = wt->L;
  if (sigma) *sigma = wt->sigma;
  if (d_words) *d_words = wt->words;
  if (d_dir) *d_dir = wt->dir;
  return WTG_OK;
}
extern "C" const wtg_select* wtg_wtint_select1(const wtg_wtint* wt) { return wt ? &wt->s1 : nullptr; }
extern "C" const wtg_select* wtg_wtint_select0(const wtg_wtint* wt) { return wt ? &wt->s0 : nullptr; }

static int q_check(wtg_ctx* ctx, const wtg_wtint* wt, uint64_t nq, const void* a, const void* b) {
  WTG_REQUIRE(ctx && wt && (nq == 0 || (a && b)), "null argument");
  if (wt->n == 0 && nq) {
    wtg_set_error("query on an empty wt_int");
    return WTG_ERR_ARG;
  }
  return WTG_OK;
}

// Whether ordering a batch pays: level bits too many for an XCD's L2 beside the
// directory, and queries enough for the three passes before the walk (17 to 30 us; 9 us
// where the sample shows a batch in order).  By symbol it needs symbols enough, too: on
// few levels the queries share the lines as they come.
// us as it came -> ordered, uniform symbols / a few of them common:
//   rank        2^24 bits, 16 levels, 2^18: 70 -> 58 / 64 -> 60;   2^19: 134 -> 80 / 119 -> 84
//               2^26 bits, 12 levels, 2^18: 70 -> 58 / 61 -> 64;   2^19: 129 -> 80 / 110 -> 94
//               2^27 bits, 10 levels, 2^18:  55 -> 60 / 48 -> 67;  2^19: 111 -> 83 / 97 -> 103
//               2^27 bits,  8 levels, 2^19:  87 -> 81 / 83 -> 105; 2^20: 183 -> 126 / 176 -> 178
//                           4 levels, 2^20: 103 -> 111 / 104 -> 133
//               2^28.3 bits, 20 levels, 2^17: 78 -> 61 / 70 -> 62; 2^18: 147 -> 82 / 139 -> 92; 2^20: 592 -> 210 / 578 -> 274
//   select      2^26 bits, 16 levels, 2^18: 128 -> 101 / 114 -> 112; 2^20: 452 -> 241 / 374 -> 256
//               2^27 bits,  8 levels, 2^18:  53 -> 66 / 51 -> 70;  2^19: 86 -> 86 / 77 -> 92; 2^25: 2^19 85 -> 87 / 591 -> 414
//   lex_count   2^26 bits, 12 levels, 2^18: 95 -> 75 / 87 -> 84;   2^27, 8, 2^20: 313 -> 202 / 313 -> 302
//   range_count (two walks, each with its own order)
//               2^26 bits, 12 levels, 2^18: 155 -> 138 / 140 -> 154; 16 levels: 197 -> 148 / 188 -> 161
//   access (by position)
//               2^24 bits, 16 levels, 2^19: 132 -> 139 / 118 -> 116; 2^20: 257 -> 246 / 226 -> 196
//               2^26 bits, 20 levels, 2^18: 111 -> 117 / 96 -> 94;   2^19: 214 -> 204 / 187 -> 154
//               2^27 bits,  4 levels, 2^18:  36 -> 44 / 37 -> 43;    2^19:  61 -> 55 / 61 -> 54
//               2^27 bits,  8 levels, 2^18:  54 -> 53 / 52 -> 49;    2^20: 191 -> 114 / 188 -> 92
static bool order_pays_position(const wtg_wtint* wt, uint64_t nq) {
  return wt->nbits >= 1ull << 24 && nq >= (wt->nbits >= 1ull << 27 && wt->L >= 8 ? 1ull << 18 : 1ull << 19);
}
static bool order_pays_symbol(const wtg_wtint* wt, uint64_t nq, uint32_t walks = 1) {
  if (wt->nbits < 1ull << 24 || wt->L < 8) return false;
  if (wt->L < 10) return nq >= 15ull << 16;
  return nq >= (wt->L >= 12 && wt->nbits >= 1ull << 26 && (walks == 1 || wt->L >= 16) ? 1ull << 18 : 1ull << 19);
}
static bool order_pays_select(const wtg_wtint* wt, uint64_t nq) {
  return order_pays_symbol(wt, nq) || (wt->nbits >= 1ull << 24 && wt->L >= 8 && nq >= 1ull << 19);
}

// A batch in chunks: walk(batch, queries, answers' offset, grid) launches the kernel
// that answers one chunk.
template <uint32_t NC, class F>
static int q_ordered(wtg_ctx* ctx, char* scratch, const QCols& in, uint32_t key, uint64_t nq, F&& walk) {
  const QOrder o = order_layout(scratch, QO_CHUNK, QO_COLS);
  const uint64_t step = wtg_ceil_div(nq, wtg_ceil_div(nq, QO_CHUNK));  // chunks of one size
  for (uint64_t at = 0; at < nq; at += step) {
    const uint64_t m = nq - at < step ? nq - at : step;
    QCols part{};
    for (uint32_t c = 0; c < NC; c++) part.c[c] = in.c[c] + at;
    order_chunk<NC>(ctx, part, KeyCol{part.c[key]}, m, o);
    QBatch b{part, {}, o.q, o.asis};
    for (uint32_t c = 0; c < NC; c++) b.put.c[c] = o.col[c];
    walk(b, m, at, dim3((unsigned)(wtg_ceil_div(m, 256 * QO_XCDS) * QO_XCDS)));
  }
  WTG_LAUNCH_CHECK();
  return WTG_OK;
}

// The batch as it came, or ordered by column `key` where that pays.
template <uint32_t NC, class F>
static int q_batch(wtg_ctx* ctx, const QCols& in, uint32_t key, bool pays, uint64_t nq, F&& walk) {
  WTG_TRY(wtg_set_device(ctx));
  char* scratch = pays ? (char*)wtg_query_scratch(ctx, QO_BYTES) : nullptr;
  if (scratch) {
    WTG_TRY(q_ordered<NC>(ctx, scratch, in, key, nq, walk));
  } else {
    walk(QBatch{in, {}, nullptr, nullptr}, nq, (uint64_t)0, dim3((unsigned)wtg_ceil_div(nq, 256)));
    WTG_LAUNCH_CHECK();
  }
  return wtg_finish(ctx);
}

extern "C" int wtg_wtint_rank_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_i,
                                    const uint64_t* d_c, uint64_t nq, uint64_t* d_out) {
  WTG_TRY(q_check(ctx, wt, nq, d_i, d_out));
  WTG_REQUIRE(nq == 0 || d_c, "null d_c");
  if (!nq) return WTG_OK;
  return q_batch<2>(ctx, QCols{{d_i, d_c}}, 1, order_pays_symbol(wt, nq), nq,
                    [&](const QBatch& b, uint64_t m, uint64_t at, dim3 grid) {
    WTG_LAUNCH(ctx, "wtint_rank", k_wtint_rank, grid, dim3(256), 0, make_q(wt, nq), b, m, d_out + at);
  });
}
static int access_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_i, uint64_t nq, uint64_t* d_sym,
                        uint64_t* d_rank) {
  return q_batch<1>(ctx, QCols{{d_i}}, 0, order_pays_position(wt, nq), nq,
                    [&](const QBatch& b, uint64_t m, uint64_t at, dim3 grid) {
    WTG_LAUNCH(ctx, "wtint_access", k_wtint_access, grid, dim3(256), 0, make_q(wt, nq), b, m, d_sym + at,
               d_rank ? d_rank + at : nullptr);
  });
}
extern "C" int wtg_wtint_access_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_i,
                                      uint64_t nq, uint64_t* d_out) {
  WTG_TRY(q_check(ctx, wt, nq, d_i, d_out));
  if (!nq) return WTG_OK;
  return access_batch(ctx, wt, d_i, nq, d_out, nullptr);
}
extern "C" int wtg_wtint_inverse_select_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_i,
                                              uint64_t nq, uint64_t* d_rank, uint64_t* d_sym) {
  WTG_TRY(q_check(ctx, wt, nq, d_i, d_sym));
  WTG_REQUIRE(nq == 0 || d_rank, "null d_rank");
  if (!nq) return WTG_OK;
  return access_batch(ctx, wt, d_i, nq, d_sym, d_rank);
}
extern "C" int wtg_wtint_lex_count_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_i,
                                         const uint64_t* d_j, const uint64_t* d_c, uint64_t nq, uint64_t* d_rank,
                                         uint64_t* d_smaller, uint64_t* d_greater) {
  WTG_TRY(q_check(ctx, wt, nq, d_i, d_rank));
  WTG_REQUIRE(nq == 0 || (d_j && d_c && d_smaller && d_greater), "null argument");
  if (!nq) return WTG_OK;
  return q_batch<3>(ctx, QCols{{d_i, d_j, d_c}}, 2, order_pays_symbol(wt, nq), nq,
                    [&](const QBatch& b, uint64_t m, uint64_t at, dim3 grid) {
    WTG_LAUNCH(ctx, "wtint_lex_count", k_wtint_lex_count, grid, dim3(256), 0, make_q(wt, nq), b, m, d_rank + at,
               d_smaller + at, d_greater + at);
  });
}
extern "C" int wtg_wtint_lex_smaller_count_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_i,
                                                 const uint64_t* d_c, uint64_t nq, uint64_t* d_rank,
                                                 uint64_t* d_smaller) {
  WTG_TRY(q_check(ctx, wt, nq, d_i, d_rank));
  WTG_REQUIRE(nq == 0 || (d_c && d_smaller), "null argument");
  if (!nq) return WTG_OK;
  return q_batch<2>(ctx, QCols{{d_i, d_c}}, 1, order_pays_symbol(wt, nq), nq,
                    [&](const QBatch& b, uint64_t m, uint64_t at, dim3 grid) {
    WTG_LAUNCH(ctx, "wtint_lex_smaller", k_wtint_lex_smaller, grid, dim3(256), 0, make_q(wt, nq), b, m, d_rank + at,
               d_smaller + at);
  });
}
extern "C" int wtg_wtint_range_count_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_lb,
                                           const uint64_t* d_rb, const uint64_t* d_vlb, const uint64_t* d_vrb,
                                           uint64_t nq, uint64_t* d_out) {
  WTG_TRY(q_check(ctx, wt, nq, d_lb, d_out));
  WTG_REQUIRE(nq == 0 || (d_rb && d_vlb && d_vrb), "null argument");
  if (!nq) return WTG_OK;
  WTG_TRY(wtg_set_device(ctx));
  // the second walk reads the batch after the first has written: not over its own answers
  bool apart = true;
  for (const uint64_t* x : {d_lb, d_rb, d_vlb, d_vrb}) apart = apart && (x + nq <= d_out || d_out + nq <= x);
  char* scratch = apart && order_pays_symbol(wt, nq, 2) ? (char*)wtg_query_scratch(ctx, QO_BYTES) : nullptr;
  if (scratch) {
    WTG_TRY(q_ordered<4>(ctx, scratch, QCols{{d_lb, d_rb, d_vlb, d_vrb}}, 2, nq,
                         [&](const QBatch& b, uint64_t m, uint64_t at, dim3 grid) {
      WTG_LAUNCH(ctx, "wtint_range_lower", k_wtint_range_half<false>, grid, dim3(256), 0, make_q(wt, nq), b, m,
                 d_out + at);
    }));
    WTG_TRY(q_ordered<3>(ctx, scratch, QCols{{d_lb, d_rb, d_vrb}}, 2, nq,
                         [&](const QBatch& b, uint64_t m, uint64_t at, dim3 grid) {
      WTG_LAUNCH(ctx, "wtint_range_upper", k_wtint_range_half<true>, grid, dim3(256), 0, make_q(wt, nq), b, m,
                 d_out + at);
    }));
  } else {
    const dim3 grid((unsigned)wtg_ceil_div(nq, 256));
    const QBatch b{{{d_lb, d_rb, d_vlb, d_vrb}}, {}, nullptr, nullptr};
    if (q_apart(wt, nq))
      WTG_LAUNCH(ctx, "wtint_range_count", k_wtint_range_count<true>, grid, dim3(256), 0, make_q(wt, nq), b, nq, d_out);
    else
      WTG_LAUNCH(ctx, "wtint_range_count", k_wtint_range_count<false>, grid, dim3(256), 0, make_q(wt, nq), b, nq, d_out);
    WTG_LAUNCH_CHECK();
  }
  return wtg_finish(ctx);
}
extern "C" int wtg_wtint_select_batch(wtg_ctx* ctx, const wtg_wtint* wt, const uint64_t* d_i,
                                      const uint64_t* d_c, uint64_t nq, uint64_t* d_out) {
  WTG_TRY(q_check(ctx, wt, nq, d_i, d_out));
  WTG_REQUIRE(nq == 0 || d_c, "null d_c");
  if (!nq) return WTG_OK;
  return q_batch<2>(ctx, QCols{{d_i, d_c}}, 1, order_pays_select(wt, nq), nq,
                    [&](const QBatch& b, uint64_t m, uint64_t at, dim3 grid) {
    if (wt->L <= 24)
      WTG_LAUNCH(ctx, "wtint_select", k_wtint_select<24>, grid, dim3(256), 0, make_q(wt, nq), b, m, d_out + at);
    else
      WTG_LAUNCH(ctx, "wtint_select", k_wtint_select<64>, grid, dim3(256), 0, make_q(wt, nq), b, m, d_out + at);
  });
}
