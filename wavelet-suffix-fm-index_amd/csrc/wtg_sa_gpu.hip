// wtg_sa_gpu.hip -- suffix array of a byte text on the GPU by prefix doubling
// (the reference calls divsufsort, fm-index/par/WT.C:35-36; any exact suffix
// sorter gives the same array).  The sigma distinct byte values are coded
// 1..sigma in byte order in c = bits(sigma) bits, 0 past the text end (so a
// suffix that ends sorts before its extensions); round 0 sorts all suffixes by
// their first q = floor(63 / c) bytes (7 for 256 values, 21 for DNA).  A
// suffix's rank is the position of its group's first suffix in the sorted
// order (32 bits).  The suffixes still in groups of two or more form a list in
// that order, (suffix, group rank) each.  A later round h = q, 2q, 4q, ... reads
// every listed suffix's rank h bytes on (+ 1; 0 past the end) and orders each
// group by it (k_sa_refine): groups that fit a block in LDS by counting the smaller and
// equal ranks, or by a sort where a group is larger than SA_COUNT, and groups larger
// than a block's by a radix sort of (group rank, rank h bytes on) over all of them.  New rank = group rank + the smaller ones.  A suffix alone in its new
// group keeps its final rank (the ranks stay consistent, as in Larsson-Sadakane
// doubling), its sa entry is written and it leaves the list; the end is an empty
// list.
#include "wtg_internal.hpp"
#include <rocprim/device/device_radix_sort.hpp>

namespace {

// byte values present in the text: present[b] = 1
__global__ __launch_bounds__(256) void k_sa_present(const uint8_t* __restrict__ t, uint64_t n,
                                                    uint32_t* __restrict__ present) {
  __shared__ uint32_t s[256];
  s[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t base = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 16;
#pragma unroll
  for (int j = 0; j < 16; j++)
    if (base + j < n) s[t[base + j]] = 1u;
  __syncthreads();
  if (s[threadIdx.x]) present[threadIdx.x] = 1u;
}

// round-0 key of suffix i: its first q bytes, each as code[byte] (1..sigma, in
// byte order) in c bits, 0 past the text end; q*c <= 63, so q <= 63.  The
// block's 256 + 63 codes are staged in LDS.
__global__ __launch_bounds__(256) void k_sa_init(const uint8_t* __restrict__ t, uint64_t n,
                                                 const uint16_t* __restrict__ code, uint32_t c, uint32_t q,
                                                 uint64_t* __restrict__ key, uint32_t* __restrict__ idx) {
  __shared__ uint16_t s_code[256];
  __shared__ uint16_t s_win[256 + 64];
  s_code[threadIdx.x] = code[threadIdx.x];
  __syncthreads();
  const uint64_t b0 = (uint64_t)blockIdx.x * 256;
  for (uint32_t j = threadIdx.x; j < 256 + 64; j += 256) {
    const uint64_t p = b0 + j;
    s_win[j] = p < n ? s_code[t[p]] : (uint16_t)0;
  }
  __syncthreads();
  const uint64_t i = b0 + threadIdx.x;
  if (i >= n) return;
  uint64_t k = 0;
  for (uint32_t j = 0; j < q; j++) k = (k << c) | (uint64_t)s_win[threadIdx.x + j];
  key[i] = k;
  idx[i] = (uint32_t)i;
}

constexpr uint32_t SA_TILE = 4096;  // sorted positions per block (1024 per wave)

// Run starts after a sort: position p starts a run of equal keys (b), of equal
// group parts key >> sh (a); p is kept unless it is a run of its own.
struct SaHeads {
  bool a, b, keep;
};
__device__ __forceinline__ SaHeads sa_heads(const uint64_t* __restrict__ key, uint64_t p, uint64_t m, uint64_t k,
                                            uint32_t sh) {
  SaHeads r{false, false, false};
  if (p >= m) return r;
  const uint64_t before = p ? key[p - 1] : 0;
  r.b = p == 0 || before != k;
  r.a = p == 0 || (before >> sh) != (k >> sh);
  r.keep = !(r.b && (p + 1 == m || key[p + 1] != k));
  return r;
}

// per tile of sorted positions: its last run start (tb), last group start (ta,
// unless whole) and kept positions (tc)
__global__ __launch_bounds__(256) void k_sa_tiles(const uint64_t* __restrict__ key, uint64_t m, int whole, uint32_t sh,
                                                  uint32_t* __restrict__ ta, uint32_t* __restrict__ tb,
                                                  uint32_t* __restrict__ tc) {
  __shared__ uint32_t s_a[4], s_b[4], s_c[4];
  const uint32_t w = threadIdx.x >> 6;
  const uint64_t base = (uint64_t)blockIdx.x * SA_TILE + threadIdx.x;
  uint32_t a = 0, b = 0, c = 0;
#pragma unroll
  for (uint32_t j = 0; j < SA_TILE / 256; j++) {
    const uint64_t p = base + j * 256;
    const SaHeads h = sa_heads(key, p, m, p < m ? key[p] : 0, sh);
    if (h.b) b = (uint32_t)p;
    if (h.a) a = (uint32_t)p;
    c += h.keep;
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t x = (uint32_t)__shfl_xor((int)a, d), y = (uint32_t)__shfl_xor((int)b, d);
    a = x > a ? x : a;
    b = y > b ? y : b;
  }
  c = wave_sum(c);
  if (lane_id() == 0) { s_a[w] = a; s_b[w] = b; s_c[w] = c; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; k++) {
      a = s_a[k] > a ? s_a[k] : a;
      b = s_b[k] > b ? s_b[k] : b;
      c += s_c[k];
    }
    if (!whole) ta[blockIdx.x] = a;
    tb[blockIdx.x] = b;
    tc[blockIdx.x] = c;
  }
}

// over the tiles, in place (one block): exclusive maximum of ta (unless whole)
// and tb, exclusive sum of tc, whose total goes to *kept
__global__ __launch_bounds__(256) void k_sa_tile_prefix(uint32_t* __restrict__ ta, uint32_t* __restrict__ tb,
                                                        uint32_t* __restrict__ tc, uint64_t ntiles, int whole,
                                                        uint32_t* __restrict__ kept) {
  __shared__ uint32_t s_w[3][4];
  uint32_t ca = 0, cb = 0, cc = 0;  // carries (every thread keeps them)
  const int lane = lane_id(), w = threadIdx.x >> 6;
  for (uint64_t c0 = 0; c0 < ntiles; c0 += 256) {
    const uint64_t i = c0 + threadIdx.x;
    const bool in = i < ntiles;
    const uint32_t a = in && !whole ? ta[i] : 0u, b = in ? tb[i] : 0u, c = in ? tc[i] : 0u;
    uint32_t xa = a, xb = b, xc = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t ya = (uint32_t)__shfl_up((int)xa, d), yb = (uint32_t)__shfl_up((int)xb, d),
                     yc = (uint32_t)__shfl_up((int)xc, d);
      if (lane >= d) {
        xa = ya > xa ? ya : xa;
        xb = yb > xb ? yb : xb;
        xc += yc;
      }
    }
    if (lane == 63) { s_w[0][w] = xa; s_w[1][w] = xb; s_w[2][w] = xc; }
    __syncthreads();
    uint32_t ea = (uint32_t)__shfl_up((int)xa, 1), eb = (uint32_t)__shfl_up((int)xb, 1), ec = xc - c;
    if (lane == 0) ea = eb = 0;
    ea = ea > ca ? ea : ca;
    eb = eb > cb ? eb : cb;
    ec += cc;
    for (int k = 0; k < 4; k++) {
      const uint32_t qa = s_w[0][k], qb = s_w[1][k], qc = s_w[2][k];
      if (k < w) {
        ea = qa > ea ? qa : ea;
        eb = qb > eb ? qb : eb;
        ec += qc;
      }
      ca = qa > ca ? qa : ca;
      cb = qb > cb ? qb : cb;
      cc += qc;
    }
    if (in) {
      if (!whole) ta[i] = ea;
      tb[i] = eb;
      tc[i] = ec;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *kept = cc;
}

// After a sort of (group rank << sh | key) pairs (whole: one group of rank 0):
// the rank of sorted position p is its group's plus the distance of its run's
// start from its group's.  A run of one has its final rank: its sa entry is
// written.  The others go to the list, in order, from `list0` on.  A wave takes
// 1024 consecutive positions, a chunk of 64 at a time: run starts and kept
// positions are ballots, so nothing but the keys is read twice.
__global__ __launch_bounds__(256) void k_sa_apply(const uint64_t* __restrict__ key, const uint32_t* __restrict__ val,
                                                  uint64_t m, uint64_t n, int whole, uint32_t sh,
                                                  const uint32_t* __restrict__ ta, const uint32_t* __restrict__ tb,
                                                  const uint32_t* __restrict__ tc, uint32_t* __restrict__ rank,
                                                  int64_t* __restrict__ sa, uint32_t* __restrict__ idx,
                                                  uint32_t* __restrict__ grp, uint32_t list0,
                                                  uint32_t* __restrict__ err) {
  constexpr uint32_t J = SA_TILE / 256;
  __shared__ uint32_t s_a[4], s_b[4], s_c[4];
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (uint32_t)lane_id();
  const uint64_t p0 = (uint64_t)blockIdx.x * SA_TILE + w * (SA_TILE / 4);
  uint64_t kv[J], ma[J], mb[J], mk[J];
  uint32_t la = 0, lb = 0, lc = 0;  // the wave's last starts, kept positions
#pragma unroll
  for (uint32_t j = 0; j < J; j++) {
    const uint64_t p = p0 + j * 64 + lane;
    kv[j] = p < m ? key[p] : 0;
  }
#pragma unroll
  for (uint32_t j = 0; j < J; j++) {
    const uint64_t p = p0 + j * 64 + lane;
    const SaHeads h = sa_heads(key, p, m, kv[j], sh);
    ma[j] = wave_ballot(h.a);
    mb[j] = wave_ballot(h.b);
    mk[j] = wave_ballot(h.keep);
    if (ma[j]) la = (uint32_t)(p0 + j * 64) + 63u - (uint32_t)__builtin_clzll(ma[j]);
    if (mb[j]) lb = (uint32_t)(p0 + j * 64) + 63u - (uint32_t)__builtin_clzll(mb[j]);
    lc += popc64(mk[j]);
  }
  if (lane == 0) { s_a[w] = la; s_b[w] = lb; s_c[w] = lc; }
  __syncthreads();
  uint32_t ca = whole ? 0u : ta[blockIdx.x], cb = tb[blockIdx.x], cc = list0 + tc[blockIdx.x];
  for (uint32_t k = 0; k < w; k++) {
    ca = s_a[k] > ca ? s_a[k] : ca;
    cb = s_b[k] > cb ? s_b[k] : cb;
    cc += s_c[k];
  }
  const uint64_t upto = ~0ull >> (63 - lane);
#pragma unroll
  for (uint32_t j = 0; j < J; j++) {
    const uint32_t c0 = (uint32_t)(p0 + j * 64);
    const uint64_t p = p0 + j * 64 + lane;
    const uint64_t fa = ma[j] & upto, fb = mb[j] & upto;
    const uint32_t first = whole ? 0u : fa ? c0 + 63u - (uint32_t)__builtin_clzll(fa) : ca;
    const uint32_t head = fb ? c0 + 63u - (uint32_t)__builtin_clzll(fb) : cb;
    if (p < m) {
      const uint32_t g = whole ? 0u : (uint32_t)(kv[j] >> sh);
      const uint32_t r = g + (head - first), i = val[p];
      if (whole || r != g) rank[i] = r;  // (a group's first run keeps its rank)
      if (mk[j] >> lane & 1u) {
        const uint32_t q = cc + mbcnt64(mk[j]);
        idx[q] = i;
        grp[q] = r;
      } else if (r < n) {
        sa[r] = (int64_t)i;
      } else {
        wtg_raise(err, WTG_FLAG_SA_RANKS);  // ranks inconsistent: not expected
      }
    }
    if (ma[j]) ca = c0 + 63u - (uint32_t)__builtin_clzll(ma[j]);
    if (mb[j]) cb = c0 + 63u - (uint32_t)__builtin_clzll(mb[j]);
    cc += popc64(mk[j]);
  }
}

// the listed suffixes' ranks h bytes on (+ 1; 0 past the end), before any rank
// of this round changes; also clears the round's two counters
__global__ __launch_bounds__(256) void k_sa_gather(const uint32_t* __restrict__ idx, uint64_t m, uint64_t n, uint64_t h,
                                                   const uint32_t* __restrict__ rank, uint32_t* __restrict__ key2,
                                                   uint32_t* __restrict__ counts) {
  const uint64_t k = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (k < 2) counts[k] = 0;
  if (k >= m) return;
  const uint64_t i = (uint64_t)idx[k] + h;
  key2[k] = i < n ? rank[i] + 1 : 0u;
}

constexpr uint32_t SA_CAP = 2048, SA_W = 1536;
// Groups longer than this are sorted, not counted.  Copies of one text with 0.01% of
// the bytes changed: 1000 copies of 32 KB 68.0 -> 24.3 ms (39.4 with a radix sort of the
// list each round), 300 of 32 KB 9.6 -> 4.8 (15.5), 100 of 320 KB 17.9 -> 16.0 (39.5).
// From 24 to 96 it makes no difference; with 160 the last one takes 19.9 ms.
constexpr uint32_t SA_COUNT = 64;

// Bitonic sort of a block's SA_CAP distinct keys, thread t's being 8 t .. 8 t + 7
// before and after: partners less than 8 apart are in the thread's registers, less than
// 512 apart in the wave, the three other steps go through s_x[SA_CAP].
__device__ __forceinline__ void sa_block_sort(uint64_t (&x)[8], uint64_t* s_x) {
  const uint32_t t = threadIdx.x;
  const auto inside = [&](uint32_t s, bool up) {  // partners s < 8 apart
#pragma unroll
    for (uint32_t r = 0; r < 8; r++)
      if ((r & s) == 0) {
        const uint64_t a = x[r], b = x[r | s];
        const bool keep = (a < b) == up;
        x[r] = keep ? a : b;
        x[r | s] = keep ? b : a;
      }
  };
  const auto take = [&](uint32_t r, uint64_t y, bool lower) { x[r] = (y < x[r]) == lower ? y : x[r]; };
#pragma unroll
  for (uint32_t r = 0; r < 8; r += 2) {  // runs of 2, up and down in turn
    const uint64_t a = x[r], b = x[r + 1];
    const bool keep = (a < b) == ((r & 2) == 0);
    x[r] = keep ? a : b;
    x[r + 1] = keep ? b : a;
  }
#pragma unroll
  for (uint32_t s = 2; s > 0; s >>= 1)  // runs of 4
#pragma unroll
    for (uint32_t r = 0; r < 8; r++)
      if ((r & s) == 0) {
        const uint64_t a = x[r], b = x[r | s];
        const bool keep = (a < b) == ((r & 4) == 0);
        x[r] = keep ? a : b;
        x[r | s] = keep ? b : a;
      }
  for (uint32_t k = 1; k <= SA_CAP / 8; k <<= 1) {  // runs of 8 k
    const bool up = (t & k) == 0;
    for (uint32_t s = k >> 1; s >= 64; s >>= 1) {  // threads of another wave
      __syncthreads();
#pragma unroll
      for (uint32_t r = 0; r < 8; r++) s_x[r * 256 + t] = x[r];
      __syncthreads();
#pragma unroll
      for (uint32_t r = 0; r < 8; r++) take(r, s_x[r * 256 + (t ^ s)], ((t & s) == 0) == up);
    }
    for (uint32_t s = k >> 1 < 32 ? k >> 1 : 32; s > 0; s >>= 1) {
#pragma unroll
      for (uint32_t r = 0; r < 8; r++)
        take(r, (uint64_t)__shfl_xor((unsigned long long)x[r], (int)s), ((t & s) == 0) == up);
    }
    inside(4, up);
    inside(2, up);
    inside(1, up);
  }
}

// One round over the list: a block takes the groups that start in its window of
// SA_W list positions and end within SA_CAP of the window's start (as long as a
// group has at most SA_CAP - SA_W suffixes it does).  For each suffix it counts
// the group's smaller, equal and earlier equal ranks h bytes on, which gives the
// new rank, the new place in the group, and whether it is alone.  Suffixes of
// larger groups go to (bkey, bval) for a sort.  The blocks' outputs follow one
// another in any order: groups stay whole, and nothing else is read from the
// order of the list.
// Counting reads a group's ranks once for each of its suffixes.  A block with a
// group of more than SA_COUNT sorts its suffixes by (group, rank h bytes on) instead.
// Six waves a SIMD: the sort's registers would leave four (20 copies of 1.6 MB 13.1
// against 12.7 ms).
// Groups are mostly small, and one pass over a round's list takes the place of a
// radix sort's seven passes plus run marking, scan and compaction: 2^25 DNA bytes
// with copied segments, all rounds after the first
// 7.2 -> 1.0 ms.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_sa_refine(const uint32_t* __restrict__ idx, const uint32_t* __restrict__ grp,
                                                   const uint32_t* __restrict__ key2, uint64_t m, uint64_t n,
                                                   uint32_t sh, uint32_t* __restrict__ rank, int64_t* __restrict__ sa,
                                                   uint32_t* __restrict__ idx2, uint32_t* __restrict__ grp2,
                                                   uint32_t* __restrict__ counts, uint64_t* __restrict__ bkey,
                                                   uint32_t* __restrict__ bval, uint32_t* __restrict__ err) {
  constexpr uint32_t M = SA_CAP / 256, NONE = 0xFFFFFFFFu;
  __shared__ uint64_t s_x[SA_CAP];  // the list's groups and ranks, or the keys of a sort
  __shared__ uint32_t s_i[SA_CAP];
  __shared__ uint64_t s_h[SA_CAP / 64], s_kp[SA_CAP / 64];
  uint32_t* const s_g = reinterpret_cast<uint32_t*>(s_x);
  uint32_t* const s_k = s_g + SA_CAP;
  __shared__ uint32_t s_base, s_bbase;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (uint32_t)lane_id();
  const uint64_t lo = (uint64_t)blockIdx.x * SA_W;
  const uint32_t have = m - lo < SA_CAP ? (uint32_t)(m - lo) : SA_CAP;  // list positions in reach
  const bool more = m - lo > SA_CAP;                                    // the list goes on past them
  const uint32_t width = have < SA_W ? have : SA_W;
  uint32_t g[M], kk[M], ii[M];
#pragma unroll
  for (uint32_t j = 0; j < M; j++) {
    const uint32_t p = (w + 4 * j) * 64 + lane;
    g[j] = kk[j] = ii[j] = 0;
    bool head = false;
    if (p < have) {
      g[j] = grp[lo + p];
      kk[j] = key2[lo + p];
      ii[j] = idx[lo + p];
      head = lo + p == 0 || grp[lo + p - 1] != g[j];
      s_g[p] = g[j];
      s_k[p] = kk[j];
    }
    const uint64_t hm = wave_ballot(head);
    if (lane == 0) s_h[w + 4 * j] = hm;
  }
  __syncthreads();
  // f: the first group start in the window; e: the end of the last group that
  // is this block's (both block-uniform)
  uint32_t f = SA_CAP, last = 0, next = more ? SA_CAP + 1 : have;  // last start in the window, the start after it
  {
    const uint64_t hv = lane < SA_CAP / 64 ? s_h[lane] : 0ull;
    const uint64_t in = lane < SA_W / 64 ? hv : 0ull, out = hv & ~in;
    const uint64_t bi = wave_ballot(in != 0), bo = wave_ballot(out != 0);
    if (bi) {
      const uint32_t c0 = (uint32_t)__builtin_ctzll(bi), c1 = 63u - (uint32_t)__builtin_clzll(bi);
      f = c0 * 64 + (uint32_t)__builtin_ctzll(s_h[c0]);
      last = c1 * 64 + 63u - (uint32_t)__builtin_clzll(s_h[c1]);
    }
    if (bo) {
      const uint32_t c0 = (uint32_t)__builtin_ctzll(bo);
      next = c0 * 64 + (uint32_t)__builtin_ctzll(s_h[c0]);
    } else if (more && grp[lo + SA_CAP] != s_g[SA_CAP - 1]) {
      next = SA_CAP;
    }
  }
  const uint32_t e = f == SA_CAP ? 0u : next <= SA_CAP ? next : last;
  // positions of the window before f belong to a group of an earlier window: a
  // large one if it started before the previous window, or ends past its reach
  bool pre = false;
  if (lo > 0 && f > 0) {
    const uint32_t end = f < SA_CAP ? f : (next <= SA_CAP ? next : SA_CAP + 1);
    pre = end > SA_CAP - SA_W || (lo > SA_W && grp[lo - SA_W - 1] == s_g[0]);
  }
  uint32_t np[M], ng[M];  // new place and rank (NONE: leaves the list, or not this block's)
  uint32_t span[M];       // its group's start | end << 16 (0: not this block's)
  uint32_t nbig = 0, most = 0;
  uint64_t bigm[M];
  const uint64_t upto = ~0ull >> (63 - lane);
#pragma unroll
  for (uint32_t j = 0; j < M; j++) {
    const uint32_t c = w + 4 * j, p = c * 64 + lane;
    const bool big = p < width && ((p < f && pre) || (f < SA_CAP && p >= f && p >= e));
    bigm[j] = wave_ballot(big);
    nbig += popc64(bigm[j]);
    np[j] = ng[j] = NONE;
    span[j] = 0;
    if (p >= f && p < e) {
      uint32_t q = c;
      uint64_t h = s_h[q] & upto;
      while (h == 0) h = s_h[--q];  // (f starts a group at or before p)
      const uint32_t S = q * 64 + 63u - (uint32_t)__builtin_clzll(h);
      uint32_t E = e;
      q = c;
      h = s_h[q] & ~upto;
      while (h == 0 && ++q < SA_CAP / 64) h = s_h[q];
      if (h) E = q * 64 + (uint32_t)__builtin_ctzll(h);
      span[j] = S | E << 16;
      most = max(most, E - S);
    }
  }
  // the suffix of place j is the less-th of its group, before it eqb of eq like it
  const auto placed = [&](uint32_t j, uint32_t less, bool alone, uint32_t place) {
    const uint32_t r = g[j] + less;
    if (less) rank[ii[j]] = r;
    if (alone) {
      if (r < n) sa[r] = (int64_t)ii[j];
      else wtg_raise(err, WTG_FLAG_SA_RANKS);  // ranks inconsistent: not expected
    } else {
      ng[j] = r;
    }
    np[j] = place;
  };
  if (__syncthreads_or(most > SA_COUNT)) {
    // sorted by group (its start), rank h bytes on, place: what lies before the
    // block's groups and behind them stays there
#pragma unroll
    for (uint32_t j = 0; j < M; j++) {
      const uint32_t p = (w + 4 * j) * 64 + lane;
      const uint64_t S = span[j] ? span[j] & 0xFFFFu : p < f ? 0u : SA_CAP - 1;  // (no group of two starts there)
      s_x[p] = S << 43 | (uint64_t)(span[j] ? kk[j] : p < f ? 0u : ~0u) << 11 | p;
    }
    __syncthreads();
    uint64_t x[8];
#pragma unroll
    for (uint32_t r = 0; r < 8; r++) x[r] = s_x[threadIdx.x * 8 + r];
    sa_block_sort(x, s_x);
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < 8; r++) s_x[threadIdx.x * 8 + r] = x[r];
    __syncthreads();
    // starts of equal keys, and from them what each suffix's own thread has to know
#pragma unroll
    for (uint32_t j = 0; j < M; j++) {
      const uint32_t c = w + 4 * j, p = c * 64 + lane;
      const uint64_t hm = wave_ballot(p == 0 || s_x[p] >> 11 != s_x[p ? p - 1 : 0] >> 11);
      if (lane == 0) s_kp[c] = hm;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < M; j++) {
      const uint32_t c = w + 4 * j, p = c * 64 + lane;
      uint32_t q = c;
      uint64_t h = s_kp[q] & upto;
      while (h == 0) h = s_kp[--q];  // (place 0 is a start)
      const uint32_t head = q * 64 + 63u - (uint32_t)__builtin_clzll(h);
      const bool ends = p + 1 >= e || (s_kp[(p + 1) >> 6] >> ((p + 1) & 63) & 1u);
      s_i[(uint32_t)s_x[p] & (SA_CAP - 1)] = p | head << 11 | (uint32_t)(head == p && ends) << 22;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < M; j++)
      if (span[j]) {
        const uint32_t v = s_i[(w + 4 * j) * 64 + lane];
        placed(j, (v >> 11 & (SA_CAP - 1)) - (span[j] & 0xFFFFu), v >> 22, v & (SA_CAP - 1));
      }
  } else {
#pragma unroll
    for (uint32_t j = 0; j < M; j++)
      if (span[j]) {
        const uint32_t p = (w + 4 * j) * 64 + lane, S = span[j] & 0xFFFFu, E = span[j] >> 16;
        uint32_t less = 0, eq = 0, eqb = 0;
        for (uint32_t t = S; t < E; t++) {
          const uint32_t kt = s_k[t];
          less += kt < kk[j];
          const uint32_t same = kt == kk[j];
          eq += same;
          eqb += t < p ? same : 0u;
        }
        placed(j, less, eq == 1, S + less + eqb);
      }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < M; j++) {  // into the new order
    if (np[j] != NONE) {
      s_g[np[j]] = ng[j];
      s_i[np[j]] = ii[j];
    }
  }
  if (lane == 0) s_k[w] = nbig;
  __syncthreads();
  uint64_t km[M];
#pragma unroll
  for (uint32_t j = 0; j < M; j++) {
    const uint32_t c = w + 4 * j, p = c * 64 + lane;
    km[j] = wave_ballot(p >= f && p < e && s_g[p] != NONE);
    if (lane == 0) s_kp[c] = km[j];
  }
  __syncthreads();
  const uint32_t kc = lane < SA_CAP / 64 ? popc64(s_kp[lane]) : 0u;
  const uint32_t incl = wave_incl_sum_dpp(kc);
  const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
  if (threadIdx.x == 0) {
    s_base = total ? atomicAdd(&counts[0], total) : 0u;
    const uint32_t nb = s_k[0] + s_k[1] + s_k[2] + s_k[3];
    s_bbase = nb ? atomicAdd(&counts[1], nb) : 0u;
  }
  __syncthreads();
  uint32_t bat = s_bbase;
  for (uint32_t k = 0; k < w; k++) bat += s_k[k];
#pragma unroll
  for (uint32_t j = 0; j < M; j++) {
    const uint32_t c = w + 4 * j, p = c * 64 + lane;
    const uint32_t ex = (uint32_t)__builtin_amdgcn_readlane((int)(incl - kc), (int)c);
    if (km[j] >> lane & 1u) {
      const uint32_t q = s_base + ex + mbcnt64(km[j]);
      idx2[q] = s_i[p];
      grp2[q] = s_g[p];
    }
    if (bigm[j] >> lane & 1u) {
      const uint32_t q = bat + mbcnt64(bigm[j]);
      bkey[q] = (uint64_t)g[j] << sh | kk[j];
      bval[q] = ii[j];
    }
    bat += popc64(bigm[j]);
  }
}

// bwt[i] = t[sa[i]-1], or t[n-1] where sa[i] = 0 (fm-index/par/WT.C:38-41)
__global__ void k_bwt(const uint8_t* __restrict__ t, const int64_t* __restrict__ sa, uint64_t n,
                      uint8_t* __restrict__ bwt, uint32_t* __restrict__ err) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t p = sa[i];
  if (p < 0 || (uint64_t)p >= n) {  // not a suffix array of this text
    wtg_raise(err, WTG_FLAG_BAD_SA);
    bwt[i] = 0;
    return;
  }
  bwt[i] = p ? t[p - 1] : t[n - 1];
}

}  // namespace

extern "C" int wtg_bwt_from_sa_gpu(wtg_ctx* ctx, const uint8_t* d_text, const int64_t* d_sa, uint64_t n,
                                   uint8_t* d_bwt) {
  WTG_REQUIRE(ctx && (n == 0 || (d_text && d_sa && d_bwt)), "wtg_bwt_from_sa_gpu: null argument");
  if (n == 0) return WTG_OK;
  WTG_TRY(wtg_set_device(ctx));
  WTG_LAUNCH(ctx, "bwt", k_bwt, dim3((unsigned)wtg_ceil_div(n, 256)), dim3(256), 0, d_text, d_sa, n, d_bwt,
             ctx->d_flag);
  WTG_LAUNCH_CHECK();
  return wtg_finish(ctx);
}

// a failed launch releases the buffers (goto out) instead of returning
#define SA_LAUNCH_CHECK()                                                  \
  do {                                                                     \
    const hipError_t _e = hipGetLastError();                               \
    if (_e != hipSuccess) {                                                \
      wtg_set_error(hipGetErrorString(_e));                                \
      rc = WTG_ERR_HIP;                                                    \
      goto out;                                                            \
    }                                                                      \
  } while (0)

extern "C" int wtg_suffix_array_gpu(wtg_ctx* ctx, const uint8_t* d_text, uint64_t n, int64_t* d_sa) {
  WTG_REQUIRE(ctx && (n == 0 || (d_text && d_sa)), "wtg_suffix_array_gpu: null argument");
  WTG_REQUIRE(n < (1ull << 31), "wtg_suffix_array_gpu: n >= 2^31");
  if (n == 0) return WTG_OK;
  WTG_TRY(wtg_set_device(ctx));
  const uint64_t tiles = wtg_ceil_div(n, SA_TILE);
  uint64_t *k0 = nullptr, *k1 = nullptr;
  uint32_t *v0 = nullptr, *v1 = nullptr;
  size_t tmp_bytes = 0;
  for (unsigned eb : {63u, 64u}) {  // temporary storage for the widest sort
    size_t b = 0;
    if (rocprim::radix_sort_pairs(nullptr, b, k0, k1, v0, v1, (uint32_t)n, 0, eb, ctx->stream) != hipSuccess) {
      wtg_set_error("wtg_suffix_array_gpu: sort size query failed");
      return WTG_ERR_HIP;
    }
    tmp_bytes = b > tmp_bytes ? b : tmp_bytes;
  }
  // All buffers in one block: the context's scratch, or for a large text (it would
  // stay that large), and where there is no memory for it outside the pool, an
  // allocation of this call.  From the pool, thirteen allocations of 4 to 8 n bytes
  // cost 2.5 to 50 ms a call and one for all of them 50 ms between calls that allocate too
  // (n = 2^25: the pool unmaps and maps what does not fit its free blocks).
  size_t o = 0;
  const auto take = [&](size_t bytes) { const size_t at = o; o = wtg_align256(o + bytes); return at; };
  const size_t o_k0 = take(n * 8), o_k1 = take(n * 8), o_v0 = take(n * 4), o_v1 = take(n * 4), o_rank = take(n * 4);
  const size_t o_i0 = take(n * 4), o_i1 = take(n * 4), o_g0 = take(n * 4), o_g1 = take(n * 4), o_key2 = take(n * 4);
  const size_t o_tab = take((3 * tiles + 4) * 4), o_pres = take(256 * 4 + 256 * 2), o_tmp = take(tmp_bytes);
  constexpr size_t SA_KEEP_MAX = 8ull << 30;
  char* mem = nullptr;
  int rc = WTG_OK;
  const wtg_scratch_use kept(ctx, o <= SA_KEEP_MAX ? o : 0);
  if (kept.mem) mem = kept.mem;
  else WTG_TRY(wtg_malloc(ctx, (void**)&mem, o));
  k0 = (uint64_t*)(mem + o_k0);
  k1 = (uint64_t*)(mem + o_k1);
  v0 = (uint32_t*)(mem + o_v0);
  v1 = (uint32_t*)(mem + o_v1);
  uint32_t* const rank = (uint32_t*)(mem + o_rank);
  uint32_t* const idx[2] = {(uint32_t*)(mem + o_i0), (uint32_t*)(mem + o_i1)};
  uint32_t* const grp[2] = {(uint32_t*)(mem + o_g0), (uint32_t*)(mem + o_g1)};
  uint32_t* const key2 = (uint32_t*)(mem + o_key2);
  uint32_t* const tab = (uint32_t*)(mem + o_tab);
  uint32_t* const present = (uint32_t*)(mem + o_pres);
  void* const tmp = mem + o_tmp;
  {
    // tile tables, then the kept count, then the round's two counters
    uint32_t *ta = tab, *tb = tab + tiles, *tc = tab + 2 * tiles, *kept = tab + 3 * tiles, *counts = kept + 1;
    uint32_t nbits = 1;
    while (nbits < 32 && (1ull << nbits) <= n) nbits++;
    // round 0 codes the sigma distinct bytes as 1..sigma in c bits (order kept),
    // so it sorts by q = floor(63 / c) bytes: 7 for 256 values, 21 for DNA
    uint16_t* d_code = (uint16_t*)(present + 256);  // codes up to 256: 16 bits
    uint32_t h_present[256];
    uint16_t h_code[256];
    if ((rc = wtg_fill_bytes_zero(ctx, present, 256 * 4)) != WTG_OK) goto out;
    WTG_LAUNCH(ctx, "sa_present", k_sa_present, dim3((unsigned)wtg_ceil_div(n, 4096)), dim3(256), 0, d_text, n,
               present);
    SA_LAUNCH_CHECK();
    if ((rc = wtg_stage_d2h(ctx, h_present, present, sizeof(h_present))) != WTG_OK) goto out;
    uint32_t sigma = 0;
    for (int b = 0; b < 256; b++) h_code[b] = h_present[b] ? (uint16_t)++sigma : 0;
    uint32_t cbits = 1;
    while ((1u << cbits) <= sigma) cbits++;
    const uint32_t q = 63 / cbits;
    if ((rc = wtg_stage_h2d(ctx, d_code, h_code, sizeof(h_code))) != WTG_OK) goto out;
    // sorts the m pairs (k0, v0) by their low end_bit bits, then ranks, sa entries
    // and the list from list0 on; *left: the list's length after it
    const auto sorted_round = [&](uint64_t m, unsigned end_bit, int whole, int b, uint32_t list0, uint64_t* left) -> int {
      const unsigned grid = (unsigned)wtg_ceil_div(m, SA_TILE);
      if (rocprim::radix_sort_pairs(tmp, tmp_bytes, k0, k1, v0, v1, (uint32_t)m, 0, end_bit, ctx->stream) !=
          hipSuccess) {
        wtg_set_error("wtg_suffix_array_gpu: sort failed");
        return WTG_ERR_HIP;
      }
      WTG_LAUNCH(ctx, "sa_tiles", k_sa_tiles, dim3(grid), dim3(256), 0, k1, m, whole, nbits, ta, tb, tc);
      WTG_LAUNCH_CHECK();
      WTG_LAUNCH(ctx, "sa_tile_prefix", k_sa_tile_prefix, dim3(1), dim3(256), 0, ta, tb, tc, (uint64_t)grid, whole,
                 kept);
      WTG_LAUNCH_CHECK();
      WTG_LAUNCH(ctx, "sa_apply", k_sa_apply, dim3(grid), dim3(256), 0, k1, v1, m, n, whole, nbits, ta, tb, tc, rank,
                 d_sa, idx[b], grp[b], list0, ctx->d_flag);
      WTG_LAUNCH_CHECK();
      uint32_t k = 0;
      WTG_TRY(wtg_stage_d2h(ctx, &k, kept, 4));
      *left = list0 + (uint64_t)k;
      return WTG_OK;
    };
    WTG_LAUNCH(ctx, "sa_init", k_sa_init, dim3((unsigned)wtg_ceil_div(n, 256)), dim3(256), 0, d_text, n, d_code, cbits,
               q, k0, v0);
    SA_LAUNCH_CHECK();
    uint64_t m = 0, h = q;
    int b = 0;
    if ((rc = sorted_round(n, q * cbits, 1, b, 0, &m)) != WTG_OK) goto out;
    for (; m > 0; h *= 2, b ^= 1) {
      if (m > n || h >= 2 * n) {
        wtg_set_error("wtg_suffix_array_gpu: ranks did not separate");
        rc = WTG_ERR_DEVICE;
        goto out;
      }
      WTG_LAUNCH(ctx, "sa_gather", k_sa_gather, dim3((unsigned)wtg_ceil_div(m, 256)), dim3(256), 0, idx[b], m, n, h,
                 rank, key2, counts);
      SA_LAUNCH_CHECK();
      WTG_LAUNCH(ctx, "sa_refine", k_sa_refine, dim3((unsigned)wtg_ceil_div(m, SA_W)), dim3(256), 0, idx[b], grp[b],
                 key2, m, n, nbits, rank, d_sa, idx[b ^ 1], grp[b ^ 1], counts, k0, v0, ctx->d_flag);
      SA_LAUNCH_CHECK();
      uint32_t c[2];
      if ((rc = wtg_stage_d2h(ctx, c, counts, 8)) != WTG_OK) goto out;
      m = c[0];
      if (c[1] && (rc = sorted_round(c[1], 2 * nbits, 0, b ^ 1, c[0], &m)) != WTG_OK) goto out;
    }
  }
  rc = wtg_finish(ctx);
out:
  if (rc != WTG_OK) wtg_abandon(ctx);
  if (mem != kept.mem) wtg_free(ctx, mem);
  return rc;
}
#undef SA_LAUNCH_CHECK
