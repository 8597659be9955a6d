// wtg_internal.hpp -- context, error plumbing and gfx950 device helpers shared
// by the wavelet-tree / rank / select kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>
#include <vector>
#include <map>
#include "wtg.h"

// ------------------------------------------------------------------ errors
void wtg_set_error(const std::string& msg);
#define WTG_CHECK_HIP(expr)                                                      \
  do {                                                                           \
    hipError_t _e = (expr);                                                      \
    if (_e != hipSuccess) {                                                      \
      wtg_set_error(std::string(#expr) + ": " + hipGetErrorString(_e));          \
      return WTG_ERR_HIP;                                                        \
    }                                                                            \
  } while (0)
#define WTG_REQUIRE(cond, msg)                                                   \
  do {                                                                           \
    if (!(cond)) { wtg_set_error(msg); return WTG_ERR_ARG; }                     \
  } while (0)
#define WTG_TRY(expr)                                                            \
  do { int _rc = (expr); if (_rc != WTG_OK) return _rc; } while (0)

// ---------------------------------------------------------------- context
struct wtg_kstat { double ms = 0; uint64_t launches = 0; };
struct wtg_kpending { std::string name; hipEvent_t a, b; };

struct wtg_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  int blocking = 1;
  int level_method = 0;  // 0: multi-level direct passes, 1: level-by-level split
  // growable workspace (device); regions carved per call
  void* ws = nullptr;
  size_t ws_bytes = 0;
  // error flags, one word per WTG_FLAG bit, in the pinned staging area: kernels
  // store to them (wtg_raise), so a call's last step is the stream's
  // synchronization alone, with no copy queued for it.  Each has a word in device
  // memory before it, so that a kernel in which every wave finds an error stores once.
  uint32_t* d_flag = nullptr;  // the words in device memory, then where the others are (in d_small)
  void* d_small = nullptr;     // 512 device bytes: a call's counters, from 256 on d_flag
  uint8_t* d_stage = nullptr;  // h_stage as the device sees it
  // pinned host staging for small transfers (async copies need no bounce
  // buffer): [0, 256) the error flags, [WTG_STAGE_D2H, +16 KiB) device-to-host
  // reads (each followed by a stream sync before use), [WTG_STAGE_H2D, +32 KiB)
  // host-to-device tables (h2d_ev marks the last such copy)
  uint8_t* h_stage = nullptr;
  hipEvent_t h2d_ev = nullptr;
  // where large query batches are put in order (wtg_query_scratch)
  void* qscratch = nullptr;
  // scratch of calls that wait for their own work (wtg_scratch_use)
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  bool scratch_used = false;  // by the call that is running: not to be given back
  // stream timer
  hipEvent_t t0 = nullptr, t1 = nullptr;
  // per-kernel timing
  bool pooled = false;   // wtg_malloc / wtg_free use the stream-ordered pool
  bool ktime = false;
  std::string kfilter;   // time only launches whose name starts with this (empty: all)
  std::vector<wtg_kpending> kpending;
  std::vector<hipEvent_t> kpool;
  std::map<std::string, wtg_kstat> kstats;
};

// workspace of at least `bytes`, 256-byte aligned regions carved by the caller
int wtg_ws_reserve(wtg_ctx* ctx, size_t bytes);
// ctx->scratch of at least `bytes` while this lives (null: 0, or no memory for it), for calls
// that cannot be captured: growing it, or giving it back (wtg_ctx_trim, or an
// allocation that finds no memory), moves nothing that a recorded graph reads.
struct wtg_scratch_use {
  wtg_ctx* const ctx;
  char* mem = nullptr;
  wtg_scratch_use(wtg_ctx* c, size_t bytes);
  ~wtg_scratch_use() { if (mem) ctx->scratch_used = false; }
  wtg_scratch_use(const wtg_scratch_use&) = delete;
  wtg_scratch_use& operator=(const wtg_scratch_use&) = delete;
};
// A block of `bytes` (the same in every call) for a batch of queries, allocated at
// the first use, and given back by wtg_ctx_trim, by an allocation that finds no memory, or
// with the context.  Null while the stream is being captured (a graph may be replayed
// beside the context's other work) or when there is no memory: the caller then answers
// the batch as it came.
void* wtg_query_scratch(wtg_ctx* ctx, size_t bytes);
constexpr size_t WTG_STAGE_AUX = 256;  // [256, 4096): reads collected by a later sync of the call
constexpr size_t WTG_STAGE_D2H = 4096, WTG_STAGE_D2H_MAX = 16384;
constexpr size_t WTG_STAGE_H2D = 32768, WTG_STAGE_H2D_MAX = 32768;
constexpr size_t WTG_STAGE_BYTES = WTG_STAGE_H2D + WTG_STAGE_H2D_MAX;
// copy device bytes to host dst through the pinned staging area (one stream sync)
int wtg_stage_d2h(wtg_ctx* ctx, void* dst, const void* d_src, size_t bytes);
// stream-ordered host-to-device copy of a small table through the staging area
// (waits for the previous such copy before reusing the buffer)
int wtg_stage_h2d(wtg_ctx* ctx, void* d_dst, const void* src, size_t bytes);
// bits of the device error flags (word k of ctx->d_flag: bit k), decoded by wtg_ctx_sync
constexpr uint32_t WTG_FLAG_WORDS = 4;
constexpr uint32_t WTG_FLAG_HOST = 4;  // word of d_flag where the address of the pinned words begins
constexpr uint32_t WTG_FLAG_WAIT = 1u;      // a bounded look-back wait expired
constexpr uint32_t WTG_FLAG_BADSYM = 2u;    // input symbol >= 2^levels / tables inconsistent with the keys
constexpr uint32_t WTG_FLAG_SA_RANKS = 4u;  // suffix ranks inconsistent
constexpr uint32_t WTG_FLAG_BAD_SA = 8u;    // a suffix array entry outside [0, n)

// called at the end of every public entry point: sync if blocking, check flag
int wtg_finish(wtg_ctx* ctx);
// error path of an entry point that stops early: wait for the stream and clear
// the device flag, so a flag raised by this call does not fail the next one
// (the error already set is kept)
void wtg_abandon(wtg_ctx* ctx);
int wtg_set_device(wtg_ctx* ctx);

// kernel launch with optional per-kernel event timing
struct wtg_kscope {
  wtg_ctx* ctx; const char* name; hipEvent_t a = nullptr, b = nullptr;
  wtg_kscope(wtg_ctx* c, const char* n);
  ~wtg_kscope();
};
#define WTG_LAUNCH(ctx, name, kernel, grid, block, shmem, ...)                   \
  do {                                                                           \
    wtg_kscope _ks((ctx), (name));                                               \
    hipLaunchKernelGGL(kernel, (grid), (block), (shmem), (ctx)->stream,          \
                       __VA_ARGS__);                                             \
  } while (0)
#define WTG_LAUNCH_CHECK()                                                       \
  WTG_CHECK_HIP(hipGetLastError())

int wtg_fill_u64(wtg_ctx* ctx, void* d, uint64_t n_u64, uint64_t value);
// internal entry points shared between translation units
int wtg_levels_build_async(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n,
                           uint32_t levels, uint64_t* d_words, wtg_node* d_nodes,
                           uint64_t node_slots, unsigned long long* d_distinct);
// level pipeline over levels [start, levels) of keys already grouped by their
// top `start` bits (counts in d_cnt_start[2^start]); level k at bit (k-start)*n
// (d_ones_start: the first level's ones per node when the caller has them)
int wtg_levels_build_from(wtg_ctx* ctx, const void* d_keys, int key_bytes, uint64_t n, uint32_t levels,
                          uint32_t start, const uint32_t* d_cnt_start, uint64_t* d_words,
                          const uint32_t* d_ones_start = nullptr);
size_t wtg_levels_ws_bytes(uint64_t n, uint32_t levels, int key_bytes);
int wtg_rank_select_run(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, uint64_t* d_dir,
                        bool build, wtg_select* sel1, wtg_select* sel0);
// The same in two halves, for callers that fold the long-superblock counts'
// host read into a read of their own: begin enqueues everything up to the two
// counts (at pend->d_nl; the workspace must stay untouched until end), end
// allocates and fills the long pools.  known_ones (build only): the number of
// ones when the caller knows it, which saves a host read.
// For many vectors at once (one host read per half for all of them): give
// each its own workspace (ws_ext, wtg_rank_select_ws_bytes) and an arena for
// the select content, and pass known_ones = WTG_ONES_DEFER: begin then stops
// after the rank pass, with the number of ones at ws_ext + WTG_RS_ONES_OFF
// (uint64), and wtg_rank_select_count, given that number, enqueues the rest up
// to the long counts (uint32 per structure, bit t at ws_ext + WTG_RS_NL_OFF + 4t).
constexpr uint64_t WTG_ONES_UNKNOWN = ~0ull;
constexpr uint64_t WTG_ONES_DEFER = ~0ull - 1;
constexpr size_t WTG_RS_ONES_OFF = 64, WTG_RS_NL_OFF = 192;
// bump allocation from one device block; what it holds is freed with the
// block, never by wtg_select_free
struct wtg_arena {
  char* base;
  size_t size, used;
};
struct wtg_rs_pending {
  bool active;
  const uint64_t* d_words;
  uint64_t nbits;
  const uint32_t* d_nl;
  wtg_select* outs[2];
  const uint64_t* sbend[2];
  const unsigned long long* last[2];
  const char* fin[2];
  wtg_arena* ar;
  bool want[2];
};
int wtg_rank_select_begin(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, uint64_t* d_dir, bool build,
                          wtg_select* sel1, wtg_select* sel0, uint64_t known_ones, wtg_rs_pending* pend,
                          char* ws_ext = nullptr, wtg_arena* ar = nullptr);
int wtg_rank_select_count(wtg_ctx* ctx, wtg_rs_pending* pend, uint64_t ones);
int wtg_rank_select_end(wtg_ctx* ctx, const wtg_rs_pending* pend, const uint32_t nl[2]);
// The three halves for select1 of many vectors whose sizes are alike
// (wtg_rank_select_many_fits), each kernel launched once for all of them; the
// counts are where begin leaves them.  dev: 3 * nvec * WTG_RS_MANY_BYTES of device
// memory for the argument tables, the object alive until the stream has been waited
// for after end.
constexpr size_t WTG_RS_MANY_BYTES = 256;
struct wtg_rs_many {
  std::vector<char> host[3];
  char* dev = nullptr;
};
bool wtg_rank_select_many_fits(uint32_t nvec, const uint64_t* nbits);
int wtg_rank_select_begin_many(wtg_ctx* ctx, uint32_t nvec, const uint64_t* const* d_words, const uint64_t* nbits,
                               uint64_t* const* dirs, wtg_select* sel1, wtg_rs_pending* pend, char* ws, size_t stride,
                               wtg_arena* ar, wtg_rs_many* many);
int wtg_rank_select_count_many(wtg_ctx* ctx, uint32_t nvec, wtg_rs_pending* pend, const uint64_t* ones,
                               wtg_rs_many* many);
int wtg_rank_select_end_many(wtg_ctx* ctx, uint32_t nvec, const wtg_rs_pending* pend, const uint64_t* nl, wtg_arena* ar,
                             wtg_rs_many* many);
size_t wtg_rank_select_ws_bytes(uint64_t nbits);
// arena bytes of one select structure: before the count (by nbits), after it
// (by the number of ones), and its long pool (by the long count)
size_t wtg_select_arena_worst(uint64_t nbits);
size_t wtg_select_arena_count(uint64_t ones);
size_t wtg_select_arena_pool(uint32_t n_long);
// multi-level direct build (up to 8 levels per pass; n >= 1, L <= 24, n < 2^32)
// and whether it is on (WTG_LEVEL_SPLIT=1 selects the level-by-level split)
int wtg_mld_enabled();
int wtg_mld_build_from(wtg_ctx* ctx, const void* d_keys, int key_bytes, uint64_t n, uint32_t L, uint32_t s0,
                       const uint32_t* d_cnt0, const uint64_t* d_src_off, uint64_t* d_words);
size_t wtg_mld_ws_bytes(uint64_t n, uint32_t L, uint32_t s0);
// 1..64 levels without node records: multi-level passes while the nodes hold
// many keys, then the small nodes' remaining levels tile by tile
int wtg_mld_build_sparse(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n, uint32_t L, uint64_t* d_words,
                         unsigned long long* d_distinct);
// 25..64 levels one split per level, nodes numbered by rank within the level (wtg_deep.hip)
int wtg_deep_build(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n, uint32_t L, uint64_t* d_words,
                   unsigned long long* d_distinct);
int wtg_mld_build(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n, uint32_t L, uint64_t* d_words,
                  wtg_node* d_nodes, uint64_t node_slots, unsigned long long* d_distinct);
// resolves the per-device address of the allocation-free rank9 scratch (wtg_ctx_create)
int wtg_noalloc_init_device(int device);
int wtg_max_value(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n, uint64_t* out);
int wtg_fill_bytes_zero(wtg_ctx* ctx, void* d, uint64_t bytes);

static inline size_t wtg_align256(size_t x) { return (x + 255) & ~size_t(255); }
static inline uint64_t wtg_ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }
static inline int wtg_log2up_host(uint64_t x) {
  int a = 0; if (x == 0) return 0; uint64_t b = x - 1; while (b) { b >>= 1; a++; } return a;
}
static inline int wtg_hi_host(uint64_t x) { int r = 0; if (!x) return 0; while (x >>= 1) r++; return r; }

// ------------------------------------------------------------- device side
#define WTG_WAVE 64
#define WTG_SPIN_LIMIT (1u << 26)   // bounded waits: iterations before giving up

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }
__device__ __forceinline__ uint32_t mbcnt64(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// raise an error flag: one lane of the wave, and of the waves the first, stores to
// pinned host memory (a plain store: atomic read-modify-write operations do not reach
// it).  The others mostly see the word that a wave before them left in their L2 (an older 0
// costs one exchange more).
__device__ __forceinline__ void wtg_raise(uint32_t* err, uint32_t flag) {
  if (mbcnt64(__builtin_amdgcn_read_exec()) != 0) return;
  const uint32_t k = (uint32_t)__builtin_ctz(flag);
  if (__hip_atomic_load(err + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0) return;
  const bool first = atomicExch(err + k, 1u) == 0;
  __hip_atomic_store(err + k, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (!first) return;
  uint32_t* const host = *reinterpret_cast<uint32_t* const*>(err + WTG_FLAG_HOST);
  __hip_atomic_store(host + k, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ uint64_t wave_ballot(bool p) { return __ballot(p); }
__device__ __forceinline__ uint32_t popc64(uint64_t x) { return (uint32_t)__popcll(x); }

template <typename U>
__device__ __forceinline__ U wave_sum(U v) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) v += __shfl_xor(v, d);
  return v;
}

// Inclusive scans over the 64 lanes with DPP moves (no LDS round trip): row_shr
// 1, 2, 4, 8 scan each 16-lane row (lanes with no source in the row take the
// identity), then row_bcast 15 combines row 0's last lane into row 1 and row 2's
// into row 3, and row_bcast 31 the last lane of rows 0-1 into rows 2-3.
template <int CTRL, int RM>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t ident, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)ident, (int)v, CTRL, RM, 0xf, false);
}
template <int CTRL, int RM>
__device__ __forceinline__ double dpp_f64(double ident, double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v), o = (uint64_t)__double_as_longlong(ident);
  const uint32_t lo = dpp_u32<CTRL, RM>((uint32_t)o, (uint32_t)u);
  const uint32_t hi = dpp_u32<CTRL, RM>((uint32_t)(o >> 32), (uint32_t)(u >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
#define WTG_DPP_SCAN_STEPS(STEP) STEP(0x111, 0xf) STEP(0x112, 0xf) STEP(0x114, 0xf) STEP(0x118, 0xf) \
  STEP(0x142, 0xa) STEP(0x143, 0xc)
__device__ __forceinline__ uint32_t wave_incl_sum_dpp(uint32_t v) {
#define WTG_STEP(C, R) v += dpp_u32<C, R>(0u, v);
  WTG_DPP_SCAN_STEPS(WTG_STEP)
#undef WTG_STEP
  return v;
}
__device__ __forceinline__ int32_t wave_incl_max_dpp(int32_t v) {
#define WTG_STEP(C, R) { const int32_t t = (int32_t)dpp_u32<C, R>(0x80000000u, (uint32_t)v); v = t > v ? t : v; }
  WTG_DPP_SCAN_STEPS(WTG_STEP)
#undef WTG_STEP
  return v;
}
// inclusive scan over the 64 lanes, Hillis-Steele with shuffles
template <typename U>
__device__ __forceinline__ U wave_incl_scan_shfl(U v) {
  const int l = lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    U t = __shfl_up(v, d);
    if (l >= d) v += t;
  }
  return v;
}
// inclusive scan over the 64 lanes: 32-bit values by DPP moves, wider ones by
// shuffles
template <typename U>
__device__ __forceinline__ U wave_incl_scan(U v) {
  if constexpr (sizeof(U) == 4) {
    return (U)wave_incl_sum_dpp((uint32_t)v);
  } else {
    return wave_incl_scan_shfl(v);
  }
}
// running max of a and min of b over the lanes (no NaNs, no -0: max and min
// are exact and equal the sequential walk's); a lane with no source in a step
// reads its own value (the instructions themselves: __builtin_fmax quiets its
// operands first)
__device__ __forceinline__ void wave_incl_maxmin_f64_dpp(double& a, double& b) {
#define WTG_STEP(C, R) { const double ta = dpp_f64<C, R>(a, a), tb = dpp_f64<C, R>(b, b); \
    asm("v_max_f64 %0, %1, %2" : "=v"(a) : "v"(ta), "v"(a)); \
    asm("v_min_f64 %0, %1, %2" : "=v"(b) : "v"(tb), "v"(b)); }
  WTG_DPP_SCAN_STEPS(WTG_STEP)
#undef WTG_STEP
}

// position (0..63) of the k-th (0-based) set bit of x; x must have > k ones
__device__ __forceinline__ uint32_t select_in_word(uint64_t x, uint32_t k) {
  uint32_t pos = 0;
  uint32_t c = __popc((uint32_t)x);
  if (k >= c) { k -= c; pos += 32; x >>= 32; }
  c = __popc((uint32_t)x & 0xFFFFu);
  if (k >= c) { k -= c; pos += 16; x >>= 16; }
  c = __popc((uint32_t)x & 0xFFu);
  if (k >= c) { k -= c; pos += 8; x >>= 8; }
  c = __popc((uint32_t)x & 0xFu);
  if (k >= c) { k -= c; pos += 4; x >>= 4; }
  c = __popc((uint32_t)x & 0x3u);
  if (k >= c) { k -= c; pos += 2; x >>= 2; }
  c = (uint32_t)(x & 1u);
  if (k >= c) { pos += 1; }
  return pos;
}

// position (0..63) of the k-th set bit of hi:lo, halving the window: k - c wraps
// past k where the bit is below the middle
__device__ __forceinline__ uint32_t select_halves(uint32_t lo, uint32_t hi, uint32_t k) {
  uint32_t c = (uint32_t)__popc(lo), pos = 0;
  uint32_t w = lo;
  if (k >= c) { w = hi; pos = 32; }
  k = min(k, k - c);
#pragma unroll
  for (uint32_t s = 16; s > 0; s >>= 1) {
    c = (uint32_t)__popc(__builtin_amdgcn_ubfe(w, pos, s));  // (offset taken modulo 32)
    pos += k >= c ? s : 0u;
    k = min(k, k - c);
  }
  return pos;
}

// ---------------------------------------------------- decoupled look-back
// status word = flag<<62 | value; flag 1 = tile aggregate, 2 = inclusive prefix.
#define LB_AGG 1ull
#define LB_PRE 2ull
#define LB_VMASK ((1ull << 62) - 1)

__device__ __forceinline__ void lb_store(uint64_t* p, uint64_t flag, uint64_t v) {
  __hip_atomic_store(p, (flag << 62) | (v & LB_VMASK), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t lb_load(uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Publishes the aggregate of `tile` (one lane).  Tile 0 publishes its
// inclusive prefix directly.
__device__ __forceinline__ void lb_publish(uint64_t* states, uint64_t tile, uint64_t agg) {
  lb_store(&states[tile], tile == 0 ? LB_PRE : LB_AGG, agg);
}

// Called by ONE full wave (all 64 lanes) after lb_publish: walks back over the
// predecessors, publishes the inclusive prefix and returns the exclusive
// prefix (same in all lanes).  Every wait is bounded: on expiry the device
// error flag is raised and the partial sum is used, so the kernel always drains.
__device__ __forceinline__ uint64_t lb_wait(uint64_t* states, uint64_t tile, uint64_t agg,
                                            uint32_t* err) {
  const int l = lane_id();
  if (tile == 0) return 0;
  uint64_t excl = 0;
  int64_t base = (int64_t)tile - 1;
  uint32_t spins = 0;
  while (true) {
    int64_t j = base - l;
    uint64_t s = (j >= 0) ? lb_load(&states[j]) : (LB_PRE << 62);
    while (true) {
      bool notready = (s >> 62) == 0;
      if (wave_ballot(notready) == 0) break;
      if (++spins > WTG_SPIN_LIMIT) {
        if (l == 0) wtg_raise(err, WTG_FLAG_WAIT);
        s = (LB_PRE << 62);  // give up: treat as prefix 0 (results invalid, flag raised)
        break;
      }
      __builtin_amdgcn_s_sleep(1);
      if (notready) s = lb_load(&states[j]);
    }
    uint64_t pm = wave_ballot((s >> 62) == LB_PRE);
    uint32_t first = pm ? (uint32_t)__builtin_ctzll(pm) : 64u;
    uint64_t v = ((uint32_t)l <= first) ? (s & LB_VMASK) : 0ull;
    excl += wave_sum(v);
    if (pm) break;
    base -= 64;
  }
  if (l == 0) lb_store(&states[tile], LB_PRE, excl + agg);
  return excl;
}

// publish + wait in one call (one full wave)
__device__ __forceinline__ uint64_t lb_exclusive(uint64_t* states, uint64_t tile, uint64_t agg,
                                                 uint32_t* err) {
  if (lane_id() == 0) lb_publish(states, tile, agg);
  return lb_wait(states, tile, agg, err);
}

// ------------------------------------------------------ block scan helper
// exclusive scan of one u32 per thread over a 256-thread block (the wave scans
// by shuffles or, DPP, by DPP moves)
template <bool DPP = false>
__device__ __forceinline__ uint32_t block_excl_scan_u32(uint32_t v, uint32_t* s_wave,
                                                        uint32_t& total) {
  const int w = threadIdx.x >> 6, l = lane_id();
  uint32_t incl = DPP ? wave_incl_sum_dpp(v) : wave_incl_scan_shfl(v);
  if (l == 63) s_wave[w] = incl;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint32_t t = s_wave[k];
    if (k < w) off += t;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return incl - v + off;
}

// ------------------------------------------- exclusive scan of a u32 array
// out[0..n] (out[n] = total); 256 threads x 16 items per tile; OUT = uint32_t
// or uint64_t (the running sum is 64-bit either way)
template <typename OUT>
__global__ __launch_bounds__(256) void k_scan_u32(const uint32_t* __restrict__ in,
                                                  OUT* __restrict__ out, uint64_t n,
                                                  uint64_t* states, uint32_t* counter,
                                                  uint32_t* err) {
  __shared__ uint32_t s_wave[4];
  __shared__ uint32_t s_tile;
  __shared__ uint64_t s_pre;
  if (threadIdx.x == 0) s_tile = atomicAdd(counter, 1u);
  __syncthreads();
  const uint64_t tile = s_tile;
  const uint64_t base = tile * 4096 + (uint64_t)threadIdx.x * 16;
  uint32_t v[16];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < 16; k++) {
    v[k] = (base + k < n) ? in[base + k] : 0u;
    sum += v[k];
  }
  uint32_t tot;
  uint32_t ex = block_excl_scan_u32(sum, s_wave, tot);
  if (threadIdx.x < 64) {
    uint64_t pre = lb_exclusive(states, tile, tot, err);
    if (threadIdx.x == 0) s_pre = pre;
  }
  __syncthreads();
  uint64_t run = s_pre + ex;
#pragma unroll
  for (int k = 0; k < 16; k++) {
    if (base + k < n) out[base + k] = (OUT)run;
    run += v[k];
  }
  if (base < n && base + 16 >= n) out[n] = (OUT)run;
  if (n == 0 && tile == 0 && threadIdx.x == 0) out[0] = 0;
}


// ------------------------------------------------ rank / select device side
// rank_support_v<1,1>::rank (rank/rank_support_v_par.hpp:131-142)
__device__ __forceinline__ uint64_t rank9_dev(const uint64_t* __restrict__ D,
                                              const uint64_t* __restrict__ words, uint64_t i) {
  const uint64_t b = i >> 9;
  uint64_t r = D[2 * b] + ((D[2 * b + 1] >> (63 - 9 * ((i & 511) >> 6))) & 0x1FF);
  if (i & 63) r += popc64(words[i >> 6] & ((1ull << (i & 63)) - 1));
  return r;
}
// The same in two steps, so that several lookups' loads are in flight together:
// the directory entry in one 16-byte load and the word, read without a test of
// i (W: the vector's words, at least one; the last word stands in for the one
// past it, of which no bit is counted), then the rank.
typedef uint32_t wtg_u4_a8 __attribute__((ext_vector_type(4), aligned(8)));
struct RankAt {
  uint64_t i, base, sub, word;
};
__device__ __forceinline__ void rank9_entry(RankAt& a, const uint64_t* __restrict__ D, uint64_t i) {
  const wtg_u4_a8 d = *reinterpret_cast<const wtg_u4_a8*>(D + 2 * (i >> 9));
  a.i = i;
  a.base = (uint64_t)d.x | (uint64_t)d.y << 32;
  a.sub = (uint64_t)d.z | (uint64_t)d.w << 32;
}
__device__ __forceinline__ void rank9_word(RankAt& a, const uint64_t* __restrict__ words, uint64_t W) {
  const uint64_t k = a.i >> 6;
  a.word = words[k < W ? k : W - 1];
}
__device__ __forceinline__ RankAt rank9_fetch(const uint64_t* __restrict__ D, const uint64_t* __restrict__ words,
                                              uint64_t W, uint64_t i) {
  RankAt a;
  rank9_entry(a, D, i);
  rank9_word(a, words, W);
  return a;
}
__device__ __forceinline__ uint64_t rank9_of(const RankAt& a) {
  const uint32_t lo = (uint32_t)a.i;
  return a.base + ((a.sub >> (63 - 9 * ((lo >> 6) & 7))) & 0x1FF) + popc64(a.word & ((1ull << (lo & 63)) - 1));
}

struct SelQ {
  const uint64_t* superblock;
  const uint32_t* mini;
  const int64_t* long_index;
  const uint64_t* long_pool;
  const uint64_t* words;
  uint64_t W;
  int bit;
};

__device__ __forceinline__ uint64_t select_plain(const SelQ& s, uint64_t i) {
  // select/select_support_mcl_par.hpp:564-611
  i -= 1;
  const uint64_t sb = i >> 12, off = i & 0xFFF;
  // (all three loads at once: the long superblocks are the rare ones)
  const int64_t li = s.long_index[sb];
  const uint64_t start = s.superblock[sb];
  const uint32_t mini = s.mini[sb * 64 + (off >> 6)];
  if (li >= 0) return s.long_pool[(uint64_t)li * 4096 + off];
  const uint64_t base = start + mini;
  uint32_t r = (uint32_t)(off & 63);
  if (r == 0) return base;
  uint64_t wp = (base + 1) >> 6;
  const uint64_t flip = s.bit ? 0ull : ~0ull;
  uint64_t keep = ~0ull << ((base + 1) & 63);
  // four words a step, all loaded before one is looked at: samples are 64 ones
  // apart, so at the density of a tree's levels one step has the bit
  for (; wp < s.W; wp += 4) {
    uint64_t x[4];
    if (wp + 4 <= s.W) {
      const wtg_u4_a8 a = *reinterpret_cast<const wtg_u4_a8*>(s.words + wp);
      const wtg_u4_a8 b = *reinterpret_cast<const wtg_u4_a8*>(s.words + wp + 2);
      x[0] = (uint64_t)a.x | (uint64_t)a.y << 32;
      x[1] = (uint64_t)a.z | (uint64_t)a.w << 32;
      x[2] = (uint64_t)b.x | (uint64_t)b.y << 32;
      x[3] = (uint64_t)b.z | (uint64_t)b.w << 32;
#pragma unroll
      for (int k = 0; k < 4; k++) x[k] ^= flip;
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) x[k] = wp + k < s.W ? s.words[wp + k] ^ flip : 0ull;
    }
    x[0] &= keep;
    keep = ~0ull;
    const uint32_t c0 = popc64(x[0]), c1 = c0 + popc64(x[1]), c2 = c1 + popc64(x[2]), c3 = c2 + popc64(x[3]);
    if (c3 >= r) {
      const int k = (c0 < r) + (c1 < r) + (c2 < r);
      const uint32_t before = k == 0 ? 0u : k == 1 ? c0 : k == 2 ? c1 : c2;
      const uint64_t y = k == 0 ? x[0] : k == 1 ? x[1] : k == 2 ? x[2] : x[3];
      return ((wp + k) << 6) + select_halves((uint32_t)y, (uint32_t)(y >> 32), r - 1 - before);
    }
    r -= c3;
  }
  return WTG_NONE;
}

