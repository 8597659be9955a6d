// wtg_mld.hip -- multi-level direct construction of the level-wise wavelet
// tree: up to 8 levels per pass over the keys.
//
// Reference semantics (wavelet/levelWT/WT.C:43-227 == serialWT/WT.C:32-103):
// level l holds P_l = the stable sort of the symbols by their top l bits
// (x >> (L-l)); the bit at global position l*n + i is bit L-1-l of P_l[i].
//
// Levels are built in groups [s, s+g), g <= 8.  The keys of a group are in
// P_s order (the input order for s = 0), so the level-s nodes are contiguous
// segments.  For a key x at position i of P_s, with d = the g bits after its
// top s bits (x >> (L-s-g)) & (2^g-1), and for each level l = s + j:
//     pos_l(i) = NodeStart_l(x >> (L-l)) + #{i' < i in P_s : same top l bits}
// because P_l is the stable sort of P_s by the top l bits.  NodeStart_l(p) =
// #keys with smaller top l bits = Cum[p << (s+g-l)], Cum being the exclusive
// prefix of the histogram of the top s+g bits.  The count of equal-prefix keys
// before i splits into the tiles of i's segment before i's tile (the "carry",
// kept per d, a range of d for coarser levels) and the rank inside the tile.
//
// Tiles are segment-aligned (each covers <= 2^tl keys of one level-s node),
// so every key of a tile shares the top s bits and a tile's ranks are those of
// its own local subtree over the next g levels.  Per group:
//   k_mld_count   per tile, the key count of each leaf d (few leaves in
//                 registers, more by LDS atomics);
//   k_mld_scan1/2 column-wise exclusive prefix of those counts over the tiles
//                 (carry(t, d) = P[t][d] - P[first tile of t's segment][d]);
//   k_mld_hist    the histogram of the top s+g bits from that prefix, then
//                 k_scan_u32 -> Cum (the node starts of all g levels);
//   k_mld_emit    per tile, a level pipeline in LDS: at level s+j the tile's
//                 keys are stably sorted by their top j bits of d, so the
//                 wave ballots of the level bit over 64-key chunks are the
//                 tile's level bits in node order; a stable split of each node
//                 by that bit (chunk zero prefix + per-node table) gives the
//                 next order.  The staged bits go out as runs, one per node
//                 and level (interior words stored, edge words OR-ed), and the
//                 keys, now in leaf order, to their P_{s+g} positions (the
//                 next group's input);
//   k_mld_ntiles  the next group's tiles per level-(s+g) node.
// Key traffic per group: read twice (count, emit), written once (scatter).
#include "wtg_internal.hpp"
#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace {

constexpr uint32_t MLD_WT = 2048;           // keys per wave of the count pass
constexpr uint32_t MLD_GMAX = 8;            // levels per group
constexpr uint32_t MLD_T4K_N = 21, MLD_T4K_NODE = 15;  // 4096-key tiles: log2 of the least keys, and per node
constexpr uint32_t MLD_CPW = 8;             // 64-key chunks per wave of the emit pass
constexpr uint32_t LOC_CAP = 2048;          // keys of a k_mld_local block
constexpr uint32_t MLD_SR = 64;             // tiles per block of the carry scan

struct MldArgs {
  const void* keys;          // P_s order; group 0: the input symbols (key type K)
  uint64_t n;
  uint32_t L, s, g;
  uint32_t tl;               // log2 of the keys per tile
  uint32_t ntiles0;          // s == 0: ceil(n / 2^tl)
  uint32_t nseg;             // s > 0: segments (2^s, or the most the list below can hold)
  const uint32_t* tstart;    // s > 0: nseg + 1 entries, first tile of each segment
  const uint32_t* tseg;      // s > 0: the segment of each tile
  const uint32_t* cum_s;     // s > 0: 2^s + 1 entries, keys before each level-s node, or
  const uint32_t* seg_start; // null, or the segments are a list of level-s nodes: where each
  const uint32_t* seg_cnt;   // starts in P_s and its keys (cum_s then unused)
  uint32_t clear;            // 1: the count pass clears the group's level words
  const uint32_t* tcnt;      // [tile][2^g] leaf counts (written by k_mld_count)
  uint32_t* tcnt_w;
  const uint32_t* ploc;      // [tile][2^g] block-local exclusive prefix over tiles
  const uint32_t* bpre;      // [block][2^g] exclusive prefix of the block sums
  const uint32_t* cum;       // 2^(s+g) + 1 entries
  uint64_t* words;
  uint32_t lvl0;             // the first level of the build: level l's bits go to (l - lvl0) * n
  uint32_t check;            // 1: flag input keys with bits at or above chk_shift
  uint32_t chk_shift;
  const uint64_t* src_off;   // null, or (first group) where each level-s node's keys start in `keys`
  void* kout;                // P_{s+g} keys (emit with SCATTER): uint32, or uint64 (WIDE)
  uint32_t* err;
};

// tile t -> (segment, first key in P_s, keys, first tile of the segment)
__device__ __forceinline__ bool mld_tile(const MldArgs& a, uint32_t t, uint32_t& seg, uint64_t& base,
                                         uint32_t& len, uint32_t& first) {
  if (a.s == 0) {
    const uint64_t off = (uint64_t)t << a.tl;
    if (t >= a.ntiles0 || off >= a.n) return false;
    seg = 0;
    base = off;
    len = (uint32_t)(a.n - off < (1u << a.tl) ? a.n - off : 1u << a.tl);
    first = 0;
    return true;
  }
  if (t >= a.tstart[a.nseg]) return false;
  const uint32_t lo = a.tseg[t];  // the segment of tile t (k_mld_tseg)
  seg = lo;
  first = a.tstart[lo];
  const uint64_t off = (uint64_t)(t - first) << a.tl;
  const uint64_t st = a.seg_cnt ? a.seg_start[lo] : a.cum_s[lo];
  const uint64_t cnt = a.seg_cnt ? a.seg_cnt[lo] : a.cum_s[lo + 1] - (uint32_t)st;
  if (off >= cnt) return false;  // (cannot happen for consistent tables)
  base = st + off;
  len = (uint32_t)(cnt - off < (1u << a.tl) ? cnt - off : 1u << a.tl);
  return true;
}

// where tile keys start in a.keys: their P_s position, or, when the level-s
// nodes' keys lie apart (src_off), that node's source offset + the tile's
// offset inside the node
__device__ __forceinline__ uint64_t mld_src(const MldArgs& a, uint32_t seg, uint64_t base) {
  return a.src_off ? a.src_off[seg] + (base - a.cum_s[seg]) : base;
}

template <typename K>
__device__ __forceinline__ uint64_t mld_key(const void* keys, uint64_t i) {
  return (uint64_t)reinterpret_cast<const K*>(keys)[i];
}

// a 16-byte word as a native vector (loads through any address space)
typedef uint32_t mld_u4 __attribute__((ext_vector_type(4)));

// element e of a 16-byte word of K-sized keys (little endian)
template <typename K>
__device__ __forceinline__ uint64_t word_elem(const mld_u4& q, uint32_t e) {
  const uint32_t c[4] = {q.x, q.y, q.z, q.w};
  if constexpr (sizeof(K) == 8) {
    return (uint64_t)c[2 * e] | ((uint64_t)c[2 * e + 1] << 32);
  } else {
    constexpr uint32_t B = 8 * sizeof(K), PER = 32 / B;
    const uint32_t dw = c[e / PER];
    return B == 32 ? dw : (dw >> (B * (e % PER))) & ((1u << (B & 31)) - 1u);
  }
}

// the g-bit leaf of element e: bits [tsh, tsh + g) of the key (gw = bits of
// that field inside the key's width, for keys narrower than a dword)
template <typename K>
__device__ __forceinline__ uint32_t word_leaf(const mld_u4& q, uint32_t e, uint32_t tsh, uint32_t gw, uint32_t gmask) {
  if constexpr (sizeof(K) == 8) {
    return (uint32_t)(word_elem<K>(q, e) >> tsh) & gmask;
  } else {
    constexpr uint32_t B = 8 * sizeof(K), PER = 32 / B;
    const uint32_t c[4] = {q.x, q.y, q.z, q.w};
    return __builtin_amdgcn_ubfe(c[e / PER], B * (e % PER) + tsh, gw);
  }
}

// leaf counts of the tiles, one wave per MLD_WT keys of a tile (the waves of a
// tile share its counters).  A wave's keys are read as the aligned 16-byte
// words that cover them, all loads in flight at once; counting needs no key
// order, so every element of every word is counted (LDS atomics; 64 words of one
// leaf add once) and the elements of the two edge words that lie outside the
// wave's range are taken back afterwards.  The aligned words never leave the
// pages of the range's own bytes.  Groups of at most 64 leaves have four copies
// of each counter, a lane's by its number, in neighbouring banks.
// Trees of at most SG leaves per tile (SG > 0) count in registers instead, a byte
// to a leaf, and add the lanes up at the end (a few leaves would otherwise put
// every lane's atomic on one of a few LDS words).
// Bound by vector instructions before (a test of every element of the words for one
// leaf, a ballot for each leaf): bytes, 2 levels, 171 M keys 154 us, now 86; 5
// levels, 148 M keys 112, now 80; 8 levels, 127 M keys 107, now 78 (the chain of
// tile, segment and key loads of each wave).
__device__ __forceinline__ void wave_sync_lds_mld() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// a device address as a global-memory pointer (global, not flat, loads)
typedef const __attribute__((address_space(1))) mld_u4* mld_gword;

template <typename K, uint32_t SG>
__global__ __launch_bounds__(256) void k_mld_count(MldArgs a) {
  constexpr uint32_t KW = sizeof(K), E = 16 / KW;
  constexpr uint32_t NW = (MLD_WT * KW / 16 + 1 + 63) / 64;  // words per lane (a range covers <= WT*KW/16 + 1)
  __shared__ uint32_t s_cnt_all[4][1u << MLD_GMAX];
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t G = 1u << a.g, lane = (uint32_t)lane_id();
  const uint32_t wl = a.tl - __builtin_ctz(MLD_WT);  // log2 of the waves per tile (0..2)
  const uint32_t t = (blockIdx.x * 4 + w) >> wl, sub = w & ((1u << wl) - 1);
  uint32_t* s_cnt = s_cnt_all[w >> wl];
  uint32_t seg, len = 0, first;
  uint64_t base = 0;
  const bool ok = mld_tile(a, t, seg, base, len, first);  // wave-uniform
  // this wave's keys: [base, base + len) from here on
  const uint32_t at = sub * MLD_WT;
  uintptr_t b0 = 0, b1 = 0, w0 = 0;
  uint32_t nw = 0;
  if (ok && at < len) {
    b0 = (uintptr_t)a.keys + (mld_src(a, seg, base) + at) * KW;
    len = len - at < MLD_WT ? len - at : MLD_WT;
    base += at;
    b1 = b0 + (uintptr_t)len * KW;
    w0 = b0 & ~(uintptr_t)15;
    nw = (uint32_t)((b1 - w0 + 15) >> 4);
  } else {
    len = 0;
  }
  mld_u4 v[NW];
  {
    const mld_gword wp = (mld_gword)w0;
#pragma unroll
    for (uint32_t m = 0; m < NW; m++) {
      const uint32_t k = m * 64 + lane;
      v[m] = k < nw ? wp[k] : mld_u4{0u, 0u, 0u, 0u};
    }
  }
  // clear the group's level words: a range clears, at each of the group's
  // levels, the words whose first bit falls on one of its positions (the
  // positions of a level-s node keep their range at every later level), so
  // every word is cleared once, by the group of its first bit's level, before
  // that group's emit ORs into it
  if (len && a.clear) {
    for (uint32_t j = 0; j < a.g; j++) {
      const uint64_t lb = (uint64_t)(a.s + j - a.lvl0) * a.n;
      const uint64_t wa = (lb + base + 63) >> 6, wb = (lb + base + len + 63) >> 6;
      for (uint64_t k = wa + lane; k < wb; k += 64) a.words[k] = 0ull;
    }
  }
  const uint32_t tsh = a.L - a.s - a.g;  // the leaf's first bit in the key
  constexpr uint32_t B = 8 * KW;
  const uint32_t gw = KW == 8 ? a.g : (tsh >= B ? 0u : (B - tsh < a.g ? B - tsh : a.g));
  const uint32_t gmask = G - 1;
  // the bad-key test over whole dwords: bits at or above chk_shift of a key
  uint32_t cm_lo = 0, cm_hi = 0;
  if (a.check) {
    const uint32_t c = a.chk_shift;
    if constexpr (KW == 8) {
      cm_lo = c >= 32 ? 0u : ~((1u << c) - 1u);
      cm_hi = c >= 32 ? ~((1u << (c - 32)) - 1u) : ~0u;
    } else {
      const uint32_t km = B == 32 ? ~0u : (1u << (B & 31)) - 1u;
      const uint32_t hm = c >= B ? 0u : km & ~((1u << c) - 1u);
      cm_lo = cm_hi = hm * (B == 8 ? 0x01010101u : B == 16 ? 0x00010001u : 1u);
    }
  }
  const uint32_t rl = a.g <= 6 ? 2 : 0;  // log2 of the copies of each counter
  if (sub == 0)
    for (uint32_t i = lane; i < G << rl; i += 64) s_cnt[i] = 0;
  if (wl) __syncthreads();
  else wave_sync_lds_mld();
  uint32_t acc_lo = 0, acc_hi = 0;  // OR of the interior words (edge words are tested per key below)
  bool bad = false;
  std::conditional_t<SG == 8, uint64_t, uint32_t> sc = 0;  // SG > 0: this lane's counts, a byte to a leaf
  static_assert(NW * E < 256, "a lane's keys in a byte");
  char* const my_cnt = reinterpret_cast<char*>(s_cnt + (lane & ((1u << rl) - 1)));
  const uint32_t fm = KW == 8 ? 0u : ((1u << gw) - 1u) << (tsh & 31) & (gw ? ~0u : 0u);
  const uint32_t fmr = B == 8 ? fm * 0x01010101u : B == 16 ? fm * 0x00010001u : fm;  // the leaf field of a dword's keys
#pragma unroll
  for (uint32_t m = 0; m < NW; m++) {
    if (m * 64 >= nw) break;  // wave-uniform
    const uint32_t k = m * 64 + lane;
    const bool act = k < nw;
    const uint32_t nact = popc64(wave_ballot(act));
    if (act && k > 0 && k + 1 < nw) {
      acc_lo |= v[m].x | v[m].z;
      acc_hi |= v[m].y | v[m].w;
    }
    if constexpr (SG > 0) {
      if (act) {
#pragma unroll
        for (uint32_t e = 0; e < E; e++)
          sc += (decltype(sc))1 << (8 * word_leaf<K>(v[m], e, tsh, gw, gmask));
      }
    } else {
      bool same;  // the leaf of every key of every lane's word is d0
      const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)word_leaf<K>(v[m], 0, tsh, gw, gmask));
      if constexpr (KW == 8) {
        same = wave_ballot(act && (word_leaf<K>(v[m], 0, tsh, gw, gmask) != d0 ||
                                   word_leaf<K>(v[m], 1, tsh, gw, gmask) != d0)) == 0;
      } else {
        const uint32_t x0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)v[m].x);  // lane 0 is active
        const uint32_t df = ((v[m].x ^ x0) | (v[m].y ^ x0) | (v[m].z ^ x0) | (v[m].w ^ x0)) & fmr;
        const uint32_t turned = (x0 >> (B & 31)) | (x0 << ((32 - B) & 31));
        same = ((x0 ^ turned) & fmr) == 0 && wave_ballot(act && df != 0) == 0;
      }
      if (same) {
        if (lane == 0) atomicAdd(&s_cnt[d0 << rl], nact * E);
      } else if (act) {
#pragma unroll
        for (uint32_t e = 0; e < E; e++)
          atomicAdd(reinterpret_cast<uint32_t*>(my_cnt + (word_leaf<K>(v[m], e, tsh, gw, gmask) << (rl + 2))), 1u);
      }
    }
  }
  if constexpr (SG > 0) {
#pragma unroll
    for (uint32_t h = 0; h < SG / 4; h++) {
      const uint32_t x = (uint32_t)(sc >> (16 * h) >> (16 * h));
      const uint32_t even = wave_incl_sum_dpp(x & 0xFF00FFu), odd = wave_incl_sum_dpp((x >> 8) & 0xFF00FFu);
      if (lane == 63 && nw) {
        const uint32_t c[4] = {even & 0xFFFFu, odd & 0xFFFFu, even >> 16, odd >> 16};
#pragma unroll
        for (uint32_t q = 0; q < 4; q++)
          if (4 * h + q < G) atomicAdd(&s_cnt[(4 * h + q) << rl], c[q]);
      }
    }
  }
  // edge words: elements outside [b0, b1) were counted above; the others
  // get the per-key bad-key test
  if (nw && lane < 2 && (lane == 0 || nw > 1)) {
    const uint32_t k = lane == 0 ? 0u : nw - 1;
    const mld_u4 q = ((mld_gword)w0)[k];
#pragma unroll
    for (uint32_t e = 0; e < E; e++) {
      const uintptr_t ea = w0 + 16 * (uintptr_t)k + e * KW;
      if (ea < b0 || ea >= b1) {
        atomicSub(&s_cnt[word_leaf<K>(q, e, tsh, gw, gmask) << rl], 1u);
      } else if (a.check && (word_elem<K>(q, e) >> a.chk_shift) != 0) {
        bad = true;
      }
    }
  }
  if (bad || ((acc_lo & cm_lo) | (acc_hi & cm_hi)) != 0) wtg_raise(a.err, WTG_FLAG_BADSYM);
  if (wl) __syncthreads();
  else wave_sync_lds_mld();
  if (ok)  // the waves of a tile write its counts in turns of 64 leaves
    for (uint32_t i = lane + 64 * sub; i < G; i += 64u << wl) {
      uint32_t c = 0;
      for (uint32_t r = 0; r < 1u << rl; r++) c += s_cnt[(i << rl) + r];
      a.tcnt_w[(uint64_t)t * G + i] = c;
    }
}

// buf[a + b] = x in LDS.  The element index is one add-and-shift (left to
// itself the compiler shifts every term of a + b before adding: five
// instructions per key and level instead of three)
__device__ __forceinline__ void lds_put(uint32_t a, uint32_t b, uint32_t* buf, uint32_t x) {
  typedef __attribute__((address_space(3))) uint32_t lds_u32;
  typedef __attribute__((address_space(3))) char lds_char;
  uint32_t off;
  asm("v_add_lshl_u32 %0, %1, %2, 2" : "=v"(off) : "v"(a), "v"(b));
  *(lds_u32*)((lds_char*)buf + off) = x;
}

// exclusive scan of one value per thread over the block's first 256 threads
// (the others hold 0 and take part in the barriers only)
template <bool DPP>
__device__ __forceinline__ uint32_t mld_scan256(uint32_t v, uint32_t* s_wave, uint32_t& total) {
  const uint32_t w = threadIdx.x >> 6, l = (uint32_t)lane_id();
  const uint32_t incl = DPP ? wave_incl_sum_dpp(v) : wave_incl_scan_shfl(v);
  if (l == 63 && w < 4) s_wave[w] = incl;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) {
    const uint32_t t = s_wave[k];
    if (k < w) off += t;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return incl - v + off;
}

// column-wise exclusive prefix of the leaf counts over the tiles, blocks of
// MLD_SR tiles: ploc = prefix inside the block, bsum = the block's totals.
// Thread (q, c) takes column c of MLD_SR/Q consecutive rows (Q = 256/G), all
// loaded before the scan.  Rows >= ntiles count 0 (row ntiles then holds the
// grand total).
__global__ __launch_bounds__(256) void k_mld_scan1(const uint32_t* __restrict__ tcnt, uint32_t* __restrict__ ploc,
                                                   uint32_t* __restrict__ bsum, const uint32_t* ntiles_dev,
                                                   uint32_t ntiles_host, uint32_t G, uint32_t nrows) {
  __shared__ uint32_t s_tot[256];
  const uint32_t nt = ntiles_dev ? *ntiles_dev : ntiles_host;
  const uint32_t Q = 256 / G < MLD_SR ? 256 / G : MLD_SR, c = threadIdx.x % G, q = threadIdx.x / G;
  const uint32_t per = q < Q ? MLD_SR / Q : 0u;  // rows of this thread (threads past Q*G idle)
  const uint64_t r0 = (uint64_t)blockIdx.x * MLD_SR + (uint64_t)q * per;
  uint32_t v[MLD_SR];
#pragma unroll
  for (uint32_t r = 0; r < MLD_SR; r++) {
    const uint64_t row = r0 + r;
    v[r] = (r < per && row < nt) ? tcnt[row * G + c] : 0u;
  }
  uint32_t acc = 0;
#pragma unroll
  for (uint32_t r = 0; r < MLD_SR; r++) {
    const uint32_t x = v[r];
    v[r] = acc;
    acc += x;
  }
  s_tot[threadIdx.x] = acc;
  __syncthreads();
  uint32_t pre = 0, tot = 0;
  for (uint32_t k = 0; k < Q; k++) {
    const uint32_t t = s_tot[k * G + c];
    if (k < q) pre += t;
    tot += t;
  }
#pragma unroll
  for (uint32_t r = 0; r < MLD_SR; r++) {
    const uint64_t row = r0 + r;
    if (r < per && row < nrows) ploc[row * G + c] = v[r] + pre;
  }
  if (q == 0) bsum[(uint64_t)blockIdx.x * G + c] = tot;
}

// The first group's tables from the block sums in one launch (one block; few
// block sums): their exclusive prefix per column as k_mld_scan2 makes it, the
// histogram (the column totals) and its exclusive prefix cum.  Four launches in
// one: 2^24 bytes, 8 levels, nodes and rank directory: 172 -> 168 us.
constexpr uint32_t MLD_ROOT_BLOCKS = 128;
__global__ __launch_bounds__(1024) void k_mld_root(const uint32_t* __restrict__ bsum, uint32_t* __restrict__ bpre,
                                                   uint32_t nblocks, uint32_t G, uint32_t* __restrict__ hist,
                                                   uint32_t* __restrict__ cum) {
  __shared__ uint32_t s_tot[1024], s_wave[4];
  const uint32_t c = threadIdx.x % G, q = threadIdx.x / G, Q = 1024 / G < 16 ? 1024 / G : 16;
  const uint32_t per = (nblocks + Q - 1) / Q, r0 = q * per, r1 = r0 + per < nblocks ? r0 + per : nblocks;  // (none past Q)
  uint32_t sum = 0;
  for (uint32_t r = r0; r < r1; r++) sum += bsum[(uint64_t)r * G + c];
  s_tot[threadIdx.x] = sum;
  __syncthreads();
  uint32_t run = 0, tot = 0;
  for (uint32_t k = 0; k < Q; k++) {
    const uint32_t t = s_tot[k * G + c];
    if (k < q) run += t;
    tot += t;
  }
  for (uint32_t r = r0; r < r1; r++) {
    const uint32_t v = bsum[(uint64_t)r * G + c];
    bpre[(uint64_t)r * G + c] = run;
    run += v;
  }
  uint32_t all;
  const uint32_t ex = mld_scan256<true>(threadIdx.x < G ? tot : 0u, s_wave, all);
  if (threadIdx.x < G) {
    hist[threadIdx.x] = tot;
    cum[threadIdx.x] = ex;
  }
  if (threadIdx.x == 0) cum[G] = all;
}

// exclusive prefix of the block sums per column: block c scans column c
__global__ __launch_bounds__(256) void k_mld_scan2(const uint32_t* __restrict__ bsum, uint32_t* __restrict__ bpre,
                                                   uint32_t nblocks, uint32_t G) {
  __shared__ uint32_t s_wave[4];
  const uint32_t c = blockIdx.x;
  uint32_t carry = 0;
  for (uint32_t b0 = 0; b0 < nblocks; b0 += 1024) {
    uint32_t v[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t b = b0 + threadIdx.x * 4 + k;
      v[k] = b < nblocks ? bsum[(uint64_t)b * G + c] : 0u;
      sum += v[k];
    }
    uint32_t tot;
    uint32_t ex = block_excl_scan_u32(sum, s_wave, tot) + carry;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t b = b0 + threadIdx.x * 4 + k;
      if (b < nblocks) bpre[(uint64_t)b * G + c] = ex;
      ex += v[k];
    }
    carry += tot;
  }
}

__device__ __forceinline__ uint32_t mld_prefix(const MldArgs& a, uint32_t row, uint32_t c) {
  const uint32_t G = 1u << a.g;
  return a.ploc[(uint64_t)row * G + c] + a.bpre[(uint64_t)(row / MLD_SR) * G + c];
}

// histogram of the top s+g bits: bin (seg << g) | d = keys of segment seg with
// leaf d = P[last tile + 1][d] - P[first tile][d]
__global__ __launch_bounds__(256) void k_mld_hist(MldArgs a, uint32_t* __restrict__ hist) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nbins = 1ull << (a.s + a.g);
  if (i >= nbins) return;
  const uint32_t seg = (uint32_t)(i >> a.g), d = (uint32_t)(i & ((1u << a.g) - 1));
  const uint32_t t0 = a.s == 0 ? 0u : a.tstart[seg];
  const uint32_t t1 = a.s == 0 ? a.ntiles0 : a.tstart[seg + 1];
  hist[i] = mld_prefix(a, t1, d) - mld_prefix(a, t0, d);
}

// tiles of each level-(s+g) node for the next group
__global__ __launch_bounds__(256) void k_mld_ntiles(const uint32_t* __restrict__ cum, uint64_t nseg,
                                                    uint32_t* __restrict__ nt, uint32_t tl) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nseg) return;
  nt[i] = (uint32_t)(((uint64_t)(cum[i + 1] - cum[i]) + (1u << tl) - 1) >> tl);
}

// tile -> segment map, one thread per tile: the last segment k with
// tstart[k] <= t (empty segments share their start with the next one)
__global__ __launch_bounds__(256) void k_mld_tseg(const uint32_t* __restrict__ tstart, uint64_t nseg,
                                                  uint32_t* __restrict__ tseg, uint64_t maxtiles) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= maxtiles || t >= tstart[nseg]) return;
  uint64_t lo = 0, hi = nseg;  // tstart[lo] <= t < tstart[hi]
  while (hi - lo > 1) {
    const uint64_t mid = (lo + hi) >> 1;
    if (tstart[mid] <= t) lo = mid; else hi = mid;
  }
  tseg[t] = (uint32_t)lo;
}

// 64 bits of an LDS bit array from bit position p (p + 64 < bits + 64 pad)
__device__ __forceinline__ uint64_t lds_bits64(const uint32_t* row, uint32_t p) {
  const uint32_t k = p >> 5, o = p & 31;
  const uint64_t lo = (uint64_t)row[k] | ((uint64_t)row[k + 1] << 32);
  const uint64_t hi = row[k + 2];
  return o ? (lo >> o) | (hi << (64 - o)) : lo;
}

// T keys per tile (mld_tile_log), T / 8 threads (8 chunks of 64 keys per wave).
// Bound by VALU issue (70% of the SIMDs' time in the 7-level pass over 2^28 uint32
// keys, 1.33 ms under the profiler, and 77% in the 6-level one), not by memory: 714 M
// instructions a 7-level pass while every wave kept the zero prefixes of its chunks
// in vector registers, 570 M with them on the scalar unit and in one LDS word a wave.
// WIDE (trees of more than 32 levels): the level loop moves the leaf d above
// the key's place in the tile instead of the key, and the scatter reads the
// 64-bit key again by that place
template <typename K, bool SCATTER, uint32_t T, bool WIDE>
__global__ __launch_bounds__(T / 8) __attribute__((amdgpu_waves_per_eu(8))) void k_mld_emit(MldArgs a) {
  constexpr uint32_t NT = T / 8, NWV = NT / 64;
  constexpr uint32_t BW = T / 32 + 2;  // staged bit words per level (+2 read-ahead pad)
  static_assert(NWV <= 8 && NT >= 256, "s_wz; 256 threads build the tables");
  // block scans by DPP moves in the bits-only pass, by shuffles in the pass
  // with key output (measured: the DPP form made the key-output pass 9%
  // slower and the bits-only pass faster: C2 5.68 -> 5.59 ms, C4 9.22 -> 8.96 ms)
  constexpr bool MLD_SCAN_DPP = !SCATTER;
  // LDS of the level pipeline: keys, tile prefix and staged bits (20 KiB at
  // 2048-key tiles, 31 KiB at 4096)
  __shared__ __align__(16) uint32_t s_k[T];      // the tile's keys in its level order
  __shared__ __align__(16) char s_rt[7424];      // the runs' tables (after the levels)
  static_assert(T <= 65535, "tile positions fit 16 bits");
  __shared__ uint16_t s_tpre[(1u << MLD_GMAX) + 1];   // exclusive prefix over d of the tile's counts
  __shared__ __align__(8) uint32_t s_bits[MLD_GMAX][BW];  // level bits in the tile's level order
  static_assert(BW % 2 == 0, "64-bit rows");
  __shared__ __align__(4) uint16_t s_xy[2u << MLD_GMAX];  // node tables of the levels (see below)
  __shared__ uint32_t s_lvl0[MLD_GMAX];
  __shared__ uint32_t s_wave[4];
  __shared__ uint32_t s_wz[MLD_GMAX][8];              // per level and wave: zeros in the waves before it
  uint32_t seg, len, first;
  uint64_t base;
  const uint32_t t = blockIdx.x;
  if (!mld_tile(a, t, seg, base, len, first)) return;
  const uint64_t src = mld_src(a, seg, base);
  const uint32_t g = a.g, G = 1u << g, lane = (uint32_t)lane_id();
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t sh = WIDE ? 16u : a.L - a.s - g;  // the leaf's first bit in what the level loop moves
  if (threadIdx.x < 8 * MLD_GMAX) s_wz[threadIdx.x >> 3][threadIdx.x & 7] = 0;
  // the tile's leaf counts and their exclusive prefix over d
  uint32_t xk[MLD_CPW];  // the wave's chunks, one key per lane
  {
    const uint32_t d = threadIdx.x;
    const uint32_t tv = d < G ? a.tcnt[(uint64_t)t * G + d] : 0u;
    // the tile's keys go straight to registers (level s needs no LDS copy);
    // all loads are in flight together with the tables above (unconditional:
    // positions past the tile load the tile's first key, replaced below)
    K kr[MLD_CPW];
#pragma unroll
    for (uint32_t m = 0; m < MLD_CPW; m++) {
      const uint32_t p = (w * MLD_CPW + m) * 64 + lane;
      kr[m] = reinterpret_cast<const K*>(a.keys)[src + (p < len ? p : 0u)];
    }
    uint32_t tot;
    const uint32_t te = mld_scan256<MLD_SCAN_DPP>(tv, s_wave, tot);
    if (d < G) s_tpre[d] = (uint16_t)te;
    if (d == 0) s_tpre[G] = (uint16_t)tot;
    // positions past the tile hold the pad key ~0: a one at every level, in
    // the last node, so each split leaves it where it is (behind the real keys)
#pragma unroll
    for (uint32_t m = 0; m < MLD_CPW; m++) {
      const uint32_t p = (w * MLD_CPW + m) * 64 + lane;
      if constexpr (WIDE) xk[m] = p < len ? ((uint32_t)((uint64_t)kr[m] >> (a.L - a.s - g)) & (G - 1)) << 16 | p : ~0u;
      else xk[m] = p < len ? (uint32_t)kr[m] : ~0u;
    }
  }
  __syncthreads();
  // node tables of all levels, from the tile's leaf counts alone: node q of
  // level s+j starts at S, with ZN keys with bit 0 (its first child) and ZS keys
  // with bit 0 in the nodes before it.  The split sends the node's k-th zero to
  // S + k and its k-th one to S + ZN + k: for a key at p with zc zeros before it
  // in the tile that is X + zc (zero) or Y + p - zc (one), with X = S - ZS and
  // Y = ZS + ZN.  Entry 2^(j+1) + 2q + b, i.e. by the key's top j + 1 bits below a
  // leading one, is X for b = 0 and Y + 1 for b = 1: with m = 0 or ~0 by the
  // key's bit both are (zc ^ m) + entry + (p & m)
  {
    const uint32_t r = threadIdx.x;
    const uint32_t j = 31 - __clz(r + 1);
    uint32_t S = 0, zn = 0;
    if (r < G - 1) {
      const uint32_t q = r + 1 - (1u << j), sgj = g - j;
      S = s_tpre[q << sgj];
      zn = s_tpre[(2 * q + 1) << (sgj - 1)] - S;
    }
    uint32_t tot;
    const uint32_t zx = mld_scan256<MLD_SCAN_DPP>(zn, s_wave, tot);  // over all entries; each level rebased below
    if (r < G - 1 && r + 1 == (1u << j)) s_lvl0[j] = zx;
    __syncthreads();
    if (r < G - 1) {
      const uint32_t zs = zx - s_lvl0[j];
      reinterpret_cast<uint32_t*>(s_xy)[r + 1] = (S - zs) | ((zs + zn + 1) << 16);
    }
  }
  __syncthreads();
  // the tile's own level pipeline: at level s+j the keys are stably sorted by
  // their top j bits of d (the tile's part of each level-(s+j) node is
  // contiguous); the ballots of the level bit in that order are the level's
  // bits, and a stable split of every node by that bit gives the next order.
  // A wave's chunks are consecutive, so the zeros before each of them are the
  // totals that the waves before it added to its word, and popcounts of ballots
  // on the scalar unit.  One buffer holds the keys: every wave has its own in registers
  // before the barrier, and writes them to their new places after it.
  const uint32_t nch = (len + 63) >> 6;
  const auto levels = [&](auto chunks) __attribute__((always_inline)) {
    constexpr uint32_t M = decltype(chunks)::value;  // chunks per wave
    uint64_t* const brow = reinterpret_cast<uint64_t*>(s_bits) + w * M + lane;  // (lane 0 stores)
    const uint32_t p0 = w * (M * 64) + lane;
    for (uint32_t j = 0; j < g; j++) {
      const uint32_t bp = sh + g - 1 - j;  // the key bit of level s+j
      // the wave's chunks, all loads first; the keys stay in registers until
      // the split below
      if (j > 0) {
#pragma unroll
        for (uint32_t m = 0; m < M; m++) xk[m] = s_k[p0 + m * 64];
      }
      uint32_t sg[M];  // 0 or ~0 by the level bit
      uint64_t om[M];
      uint32_t ones = 0;
#pragma unroll
      for (uint32_t m = 0; m < M; m++) {
        sg[m] = (uint32_t)__builtin_amdgcn_sbfe((int)xk[m], bp, 1);
        om[m] = wave_ballot(sg[m] != 0);
        ones += popc64(om[m]);
        if (lane == 0) brow[j * (BW / 2) + m] = om[m];
      }
      if (j + 1 == g && !SCATTER) break;  // the last level's order is not needed
      if (lane > w && lane < NWV) atomicAdd(&s_wz[j][lane], M * 64 - ones);
      // the table entries do not wait for the other waves' totals
      const uint16_t* nt = s_xy + (2u << j);
      uint32_t xy[M];
#pragma unroll
      for (uint32_t m = 0; m < M; m++) xy[m] = nt[__builtin_amdgcn_ubfe(xk[m], bp, j + 1)];
      __syncthreads();
      uint32_t zb = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_wz[j][w]);  // zeros before the wave's chunks
      // stable split of each node: its zeros first, then its ones.  Every
      // chunk of the tile takes part (chunks past the keys hold pad keys,
      // which stay in place)
#pragma unroll
      for (uint32_t m = 0; m < M; m++) {
        const uint64_t zm = ~om[m];
        const uint32_t zc =
            __builtin_amdgcn_mbcnt_hi((uint32_t)(zm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)zm, zb));
        lds_put((zc ^ sg[m]) + xy[m], (p0 + m * 64) & sg[m], s_k, xk[m]);
        zb += popc64(zm);
      }
      __syncthreads();
    }
  };
  // the last tile of a segment is often short: up to a quarter of a tile takes
  // a quarter of the chunks
  if (nch > 2 * NWV) {
    levels(std::integral_constant<uint32_t, MLD_CPW>{});
  } else {
    // (chunks 2w, 2w + 1 now: the keys loaded above as chunks 8w .. 8w + 7)
#pragma unroll
    for (uint32_t m = 0; m < MLD_CPW; m++) s_k[(w * MLD_CPW + m) * 64 + lane] = xk[m];
    __syncthreads();
#pragma unroll
    for (uint32_t m = 0; m < 2; m++) xk[m] = s_k[(w * 2 + m) * 64 + lane];
    __syncthreads();
    levels(std::integral_constant<uint32_t, 2>{});
  }
  // each leaf's node start and carry (keys of the leaf in its segment's earlier
  // tiles), the carry's exclusive prefix over d: read here, not before the
  // level pipeline, whose registers they would take
  uint32_t cum_d = 0, cpre_d, ctot;
  {
    const uint32_t d = threadIdx.x;
    uint32_t cv = 0;
    if (d < G) {
      cv = mld_prefix(a, t, d) - mld_prefix(a, first, d);
      cum_d = a.cum[((uint64_t)seg << g) + d];
    }
    cpre_d = mld_scan256<MLD_SCAN_DPP>(cv, s_wave, ctot);  // (its barriers end the pipeline too)
  }
  // write the level bits: for level s+j the tile's keys of local node q form
  // one run at NodeStart + carry.  Thread r < G-1 describes run r = (j, q);
  // then the destination words of all runs are dealt out over the block.
  const uint64_t n = a.n;
  const uint32_t nruns = G - 1;  // (j, q) pairs with j < g
  // run tables, carry prefix and leaf bases
  char* rt = s_rt;
  uint64_t* s_rgs = reinterpret_cast<uint64_t*>(rt);               // per run: global start,
  uint32_t* s_rls = reinterpret_cast<uint32_t*>(rt + 2048);        // start in the staged bits,
  uint32_t* s_rcnt = reinterpret_cast<uint32_t*>(rt + 3072);       // length,
  uint32_t* s_rw = reinterpret_cast<uint32_t*>(rt + 4096);         // first destination word item
  uint32_t* s_cpre = reinterpret_cast<uint32_t*>(rt + 5248);       // carry prefix over d (G + 1)
  uint32_t* s_lb = reinterpret_cast<uint32_t*>(rt + 6400);         // leaf d's key at tile position i goes to s_lb[d] + i
  static_assert(6400 + 4 * (1u << MLD_GMAX) <= sizeof(s_rt), "tables fit");
  uint32_t* s_cum = s_lb;  // node starts first, leaf bases after the run tables are built
  if (threadIdx.x < G) {
    s_cpre[threadIdx.x] = cpre_d;
    s_cum[threadIdx.x] = cum_d;
  }
  if (threadIdx.x == 0) s_cpre[G] = ctot;
  __syncthreads();
  bool off = false;  // tables inconsistent with the keys: what they put out of range is not written
  {
    const uint32_t r = threadIdx.x;
    uint32_t nw = 0;
    if (r < nruns) {
      const uint32_t j = 31 - __clz(r + 1), q = r + 1 - (1u << j);
      const uint32_t lo = q << (g - j), hi = (q + 1) << (g - j);
      const uint32_t cnt = s_tpre[hi] - s_tpre[lo];
      const uint64_t lb = (uint64_t)(a.s + j - a.lvl0) * n;  // the level's first bit
      const uint64_t gs = lb + s_cum[lo] + (s_cpre[hi] - s_cpre[lo]);
      if (gs < lb || gs + cnt > lb + n) off = true;
      else if (cnt) nw = (uint32_t)(((gs + cnt - 1) >> 6) - (gs >> 6) + 1);
      s_rgs[r] = gs;
      s_rls[r] = s_tpre[lo];
      s_rcnt[r] = cnt;
    }
    uint32_t tot;
    const uint32_t ex = mld_scan256<MLD_SCAN_DPP>(nw, s_wave, tot);  // (its barriers order the s_cum reads above)
    if (r < nruns) s_rw[r] = ex;
    if (r == 0) s_rw[nruns] = tot;
    if (SCATTER && r < G) s_lb[r] = cum_d + (s_cpre[r + 1] - s_cpre[r]) - s_tpre[r];
    __syncthreads();
  }
  const uint32_t nwords = s_rw[nruns];
  for (uint32_t it = threadIdx.x; it < nwords; it += NT) {
    uint32_t lo = 0, hi = nruns;  // the last run whose first word item is <= it
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (s_rw[mid] <= it) lo = mid; else hi = mid;
    }
    const uint32_t r = lo, j = 31 - __clz(r + 1);
    const uint64_t gs = s_rgs[r], ge = gs + s_rcnt[r];
    const uint64_t wi = (gs >> 6) + (it - s_rw[r]);
    const uint64_t wb = wi << 6;
    const uint32_t b0 = gs > wb ? (uint32_t)(gs - wb) : 0u;
    const uint32_t b1 = ge < wb + 64 ? (uint32_t)(ge - wb) : 64u;
    uint64_t v = lds_bits64(s_bits[j], (uint32_t)(s_rls[r] + (wb + b0 - gs))) << b0;
    if (b1 < 64) v &= (1ull << b1) - 1;
    if (b0 == 0 && b1 == 64) a.words[wi] = v;
    else if (v) atomicOr((unsigned long long*)&a.words[wi], (unsigned long long)v);
  }
  if (SCATTER) {
    // keys in leaf order to their P_{s+g} positions
#pragma unroll
    for (uint32_t m = 0; m < MLD_CPW; m++) {
      const uint32_t i = (w * MLD_CPW + m) * 64 + lane;
      if (i < len) {
        const uint32_t x = s_k[i];
        const uint32_t dest = s_lb[(x >> sh) & (G - 1)] + i;
        if (dest >= n) off = true;
        else if constexpr (WIDE)
          reinterpret_cast<uint64_t*>(a.kout)[dest] = (uint64_t) reinterpret_cast<const K*>(a.keys)[src + (x & 0xFFFFu)];
        else reinterpret_cast<uint32_t*>(a.kout)[dest] = x;
      }
    }
  }
  if (off) wtg_raise(a.err, WTG_FLAG_BADSYM);
}

// WTnode record v from the histogram prefix of all L bits (node (l, p) holds
// the keys with top l bits p: start Cum[p << (L-l)], count up to the next)
__device__ __forceinline__ wtg_node mld_node(const uint32_t* cum, uint32_t L, uint64_t n, uint64_t v) {
  wtg_node r;
  r.bitmapPtr = 0; r.length = 0; r.parent = WTG_NONE; r.leftChild = WTG_NONE; r.rightChild = WTG_NONE;
  if (v < (1ull << L) - 1) {
    const uint32_t l = 63 - __clzll(v + 1);
    const uint64_t p = v + 1 - (1ull << l);
    const uint32_t sh = L - l;
    const uint64_t st = cum[p << sh], c = cum[(p + 1) << sh] - st;
    if (c > 0 || v == 0) {
      r.bitmapPtr = (uint64_t)l * n + st;
      r.length = c;
      r.parent = v ? (v - 1) / 2 : WTG_NONE;
      if (l + 1 < L) {
        const uint64_t m = cum[(2 * p + 1) << (sh - 1)];
        if (m > st) r.leftChild = 2 * v + 1;
        if (cum[(p + 1) << sh] > m) r.rightChild = 2 * v + 2;
      }
    }
  }
  return r;
}
__global__ void k_mld_nodes(const uint32_t* __restrict__ cum, uint32_t L, uint64_t n, wtg_node* __restrict__ nodes,
                            uint64_t slots) {
  const uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v < slots) nodes[v] = mld_node(cum, L, n, v);
}

// A whole tree of at most 8 levels over at most ONE_CAP keys in one block:
// counts, node tables, the level pipeline of k_mld_emit, then every output word
// once (a word may hold several levels' bits) and the node records.  Such a
// call is launches and waits only: 5003 bytes, 5 levels, with nodes: one launch of
// 11 us instead of eight and a copy, the call
// 45-60 -> 22 us.
constexpr uint32_t ONE_CAP = 8192;
template <typename K>
__global__ __launch_bounds__(1024) void k_mld_one(const K* __restrict__ keys, uint32_t n, uint32_t L,
                                                  uint64_t* __restrict__ words, wtg_node* __restrict__ nodes,
                                                  uint64_t slots, unsigned long long* __restrict__ distinct,
                                                  uint32_t* __restrict__ err) {
  constexpr uint32_t M = ONE_CAP / 1024, NWV = 16;
  __shared__ uint32_t s_k[ONE_CAP];
  __shared__ uint32_t s_cnt[256], s_pre[257], s_nxy[255], s_lvl0[MLD_GMAX], s_wave[4];
  __shared__ __align__(8) uint32_t s_bits[MLD_GMAX][ONE_CAP / 32 + 2];
  __shared__ uint16_t s_ex[NWV][ONE_CAP / 64];
  const uint32_t tid = threadIdx.x, lane = (uint32_t)lane_id(), G = 1u << L;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  if (tid < 256) s_cnt[tid] = 0;
  K kr[M];
#pragma unroll
  for (uint32_t m = 0; m < M; m++) {
    const uint32_t p = (w + NWV * m) * 64 + lane;
    kr[m] = p < n ? keys[p] : (K)0;
  }
  __syncthreads();
  // (positions past the keys hold a one at every level: they stay behind the keys)
  uint32_t x[M];
  bool bad = false;
#pragma unroll
  for (uint32_t m = 0; m < M; m++) {
    const uint32_t p = (w + NWV * m) * 64 + lane;
    const bool in = p < n;
    x[m] = in ? (uint32_t)kr[m] & (G - 1) : G - 1;
    bad |= in && ((uint64_t)kr[m] >> L) != 0;
    if (in) atomicAdd(&s_cnt[x[m]], 1u);
  }
  if (bad) wtg_raise(err, WTG_FLAG_BADSYM);
  __syncthreads();
  if (distinct) {
    const uint32_t k = (uint32_t)__syncthreads_count(tid < 256 && s_cnt[tid & 255] != 0);
    if (tid == 0) *distinct = k;
  }
  uint32_t tot;
  const uint32_t ex = mld_scan256<true>(tid < 256 ? s_cnt[tid] : 0u, s_wave, tot);
  if (tid < 256) s_pre[tid] = ex;
  if (tid == 0) s_pre[256] = tot;
  __syncthreads();
  {  // node tables as in k_mld_emit
    const uint32_t r = tid, j = 31 - __clz(r + 1);
    uint32_t S = 0, zn = 0;
    if (r < G - 1) {
      const uint32_t q = r + 1 - (1u << j), sgj = L - j;
      S = s_pre[q << sgj];
      zn = s_pre[(2 * q + 1) << (sgj - 1)] - S;
    }
    const uint32_t zx = mld_scan256<true>(r < G - 1 ? zn : 0u, s_wave, tot);
    if (r < G - 1 && r + 1 == (1u << j)) s_lvl0[j] = zx;
    __syncthreads();
    if (r < G - 1) {
      const uint32_t zs = zx - s_lvl0[j];
      s_nxy[r] = (S - zs) | ((zs + zn) << 16);
    }
  }
  __syncthreads();
  for (uint32_t j = 0; j < L; j++) {
    const uint32_t bp = L - 1 - j;
    uint64_t zm[M];
    if (j > 0) {
#pragma unroll
      for (uint32_t m = 0; m < M; m++) x[m] = s_k[(w + NWV * m) * 64 + lane];
    }
#pragma unroll
    for (uint32_t m = 0; m < M; m++) {
      const uint64_t ones = wave_ballot((x[m] >> bp) & 1u);
      zm[m] = ~ones;
      if (lane == 0) reinterpret_cast<uint64_t*>(s_bits[j])[w + NWV * m] = ones;
    }
    __syncthreads();
    if (j + 1 == L) break;
    const uint64_t* row = reinterpret_cast<const uint64_t*>(s_bits[j]);
    const uint32_t v0 = 64u - popc64(row[2 * lane]), v1 = 64u - popc64(row[2 * lane + 1]);
    const uint32_t incl = wave_incl_sum_dpp(v0 + v1);
    s_ex[w][2 * lane] = (uint16_t)(incl - v0 - v1);
    s_ex[w][2 * lane + 1] = (uint16_t)(incl - v1);
    wave_sync_lds_mld();
    const uint32_t* nt = s_nxy + (1u << j) - 1;
#pragma unroll
    for (uint32_t m = 0; m < M; m++) {
      const uint32_t c = w + NWV * m, p = c * 64 + lane;
      const uint32_t xy = nt[__builtin_amdgcn_ubfe(x[m], bp + 1, j)];
      const uint32_t zc = __builtin_amdgcn_mbcnt_hi((uint32_t)(zm[m] >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)zm[m], s_ex[w][c]));
      const bool zero = ((x[m] >> bp) & 1u) == 0;
      s_k[(zero ? (xy & 0xFFFFu) + zc : (xy >> 16) + p - zc) & (ONE_CAP - 1)] = x[m];
    }
    __syncthreads();
  }
  const uint32_t nbits = n * L;
  for (uint32_t b = tid * 64; b < nbits; b += 1024 * 64) {
    const uint32_t end = b + 64 < nbits ? b + 64 : nbits;
    uint64_t v = 0;
    for (uint32_t at = b; at < end;) {
      const uint32_t l = at / n, o = at - l * n;
      const uint32_t cnt = end - at < n - o ? end - at : n - o;
      const uint64_t bits = lds_bits64(s_bits[l], o) & (cnt < 64 ? (1ull << cnt) - 1 : ~0ull);
      v |= bits << (at - b);
      at += cnt;
    }
    words[b >> 6] = v;
  }
  if (nodes)
    for (uint64_t v = tid; v < slots; v += 1024) nodes[v] = mld_node(s_pre, L, n, v);
}

__global__ void k_mld_nonzero(const uint32_t* __restrict__ h, uint64_t n, unsigned long long* out) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  uint64_t c = 0;
  for (; i < n; i += stride) c += h[i] != 0;
  c = wave_sum(c);
  if (lane_id() == 0 && c) atomicAdd(out, (unsigned long long)c);
}

// where the dense groups of a tree with small nodes end: whole 8-level groups,
// and an average node of at most 128 keys (LOC_H leaves room for uneven ones;
// 6000011 keys, 40 levels: 695 us with 128, 699 with 256, 717 with 64)
uint32_t mld_split_level(uint64_t n) {
  if (n <= (1ull << 15)) return 8;
  uint32_t s = 16;
  while (s < 24 && (n >> (s + 7)) != 0) s++;
  return s;
}
// Up to 24 levels both ways work.  Dense groups alone start the last of three
// groups at level 2/3 L; from about 512 keys per node there down, their tiles
// are mostly padding (one node per tile): n = 2^24, 24 levels (256 keys)
// 1230 us against 577, n = 3000017, 20 levels (183 keys) 264 against 200; at
// 1024 keys they are the faster way (n = 2^24, 20 levels: 449 against 506).
bool mld_use_sparse(uint64_t n, uint32_t L) {
  if (n <= LOC_CAP) return L > MLD_GMAX;  // (k_mld_one otherwise)
  const uint32_t last = L - L / 3;  // where the last of three near-equal groups starts
  return L > 16 && (n >> last) < 512;
}

struct MldPlan {
  uint32_t ngroups, gs[4], gg[4], gt[4];
  uint64_t maxtiles, maxblocks, maxbins;
  size_t off_keys[2], off_tcnt, off_ploc, off_bsum, off_bpre, off_hist, off_cum[2], off_tst, off_nt, off_tseg,
      off_scst, off_ctr, total;
};

// log2 of the keys per tile of a group of g levels over n keys in 2^s nodes.
// The tables of a wide group (256 leaves, 255 runs, a partial word at each end
// of a run for 8 levels) cost a 2048-key tile about what its keys do, so groups
// of 7 and 8 levels take 4096-key tiles (512 threads): n = 2^24 bytes, 8 levels,
// emit 140 -> 95 us; wt_int of 2^28 keys as 7 + 7 + 6 levels 5.39 -> 5.31 ms.
// 8192 keys (1024 threads): 2% faster on the former, 4% slower on 1024 uneven
// sequences.  Narrower groups keep 2048 keys, whose blocks wait for half as many
// waves at each of the level barriers (5 levels 387 us against 416, 2 levels 217
// against 249), and so do small inputs and small nodes, where larger tiles would
// leave the chip or the tiles partly empty.
uint32_t mld_tile_log(uint64_t n, uint32_t s, uint32_t g) {
  return g + 1 >= MLD_GMAX && n >= (1ull << MLD_T4K_N) && (n >> s) >= (1ull << MLD_T4K_NODE) ? 12 : 11;
}

// (key_bytes: 0, or the caller reads the keys after the last group too, and
// writes both buffers)
MldPlan mld_plan(uint64_t n, uint32_t L, uint32_t s0, uint32_t key_bytes = 0) {
  MldPlan P{};
  // as few groups as MLD_GMAX allows, of near-equal widths (wider first): a
  // pass's per-tile work outside the level pipeline (tables, runs, partial
  // words) grows with its 2^g leaves.  n = 2^28 uint32, 20 levels as 7 + 7 + 6:
  // 5.65 ms for the wt_int build, 6.58 ms as 8 + 8 + 4; groups of at most 7, 6
  // or 5 levels (more passes over the keys): 5.70, 6.00, 5.99 ms
  uint32_t s = s0, left = (L - s0 + MLD_GMAX - 1) / MLD_GMAX;
  while (s < L) {
    const uint32_t g = (L - s + left - 1) / left;
    left--;
    P.gs[P.ngroups] = s;
    P.gg[P.ngroups] = g;
    P.gt[P.ngroups] = mld_tile_log(n, s, g);
    P.ngroups++;
    s += g;
  }
  // a group over level-s nodes has at most ceil(n/T) + min(n, 2^s) tiles
  P.maxtiles = wtg_ceil_div(n, MLD_WT) + std::min<uint64_t>(n, 1ull << P.gs[P.ngroups - 1]) + 1;
  P.maxblocks = wtg_ceil_div(P.maxtiles + 1, MLD_SR) + 1;
  P.maxbins = 1ull << L;
  size_t o = 0;
  for (int b = 0; b < 2; b++) {
    P.off_keys[b] = o;
    if (P.ngroups > 1 || key_bytes) o = wtg_align256(o + n * (key_bytes ? key_bytes : 4));
  }
  P.off_tcnt = o; o = wtg_align256(o + (P.maxtiles + 1) * 256 * 4);
  P.off_ploc = o; o = wtg_align256(o + (P.maxtiles + 1) * 256 * 4);
  P.off_bsum = o; o = wtg_align256(o + P.maxblocks * 256 * 4);
  P.off_bpre = o; o = wtg_align256(o + P.maxblocks * 256 * 4);
  P.off_hist = o; o = wtg_align256(o + P.maxbins * 4);
  for (int b = 0; b < 2; b++) { P.off_cum[b] = o; o = wtg_align256(o + (P.maxbins + 1) * 4); }
  P.off_tst = o; o = wtg_align256(o + (P.maxbins + 1) * 4);
  P.off_nt = o; o = wtg_align256(o + P.maxbins * 4);
  P.off_tseg = o; o = wtg_align256(o + P.maxtiles * 4);
  P.off_scst = o; o = wtg_align256(o + (wtg_ceil_div(P.maxbins + 1, 4096) + 2) * 8);
  P.off_ctr = o; o = wtg_align256(o + 256);  // right after the scan states: one fill clears both
  P.total = o;
  return P;
}

// the count and emit passes of a group over keys of type K (the input's, or
// KO of the passes before)
template <typename K>
void mld_count_launch(wtg_ctx* ctx, unsigned grid, const MldArgs& a) {
  const dim3 cg((unsigned)wtg_ceil_div(grid, (uint64_t)4 * MLD_WT >> a.tl));  // 4 waves of MLD_WT keys per block
  if (a.g <= 2) WTG_LAUNCH(ctx, "mld_count", (k_mld_count<K, 4>), cg, dim3(256), 0, a);
  else if (a.g == 3) WTG_LAUNCH(ctx, "mld_count", (k_mld_count<K, 8>), cg, dim3(256), 0, a);
  else WTG_LAUNCH(ctx, "mld_count", (k_mld_count<K, 0>), cg, dim3(256), 0, a);
}
template <typename K, bool WIDE>
void mld_emit_launch(wtg_ctx* ctx, bool scatter, unsigned grid, const MldArgs& a) {
  if (a.tl == 12) {
    if (scatter) WTG_LAUNCH(ctx, "mld_emit", (k_mld_emit<K, true, 4096, WIDE>), dim3(grid), dim3(512), 0, a);
    else WTG_LAUNCH(ctx, "mld_emit", (k_mld_emit<K, false, 4096, WIDE>), dim3(grid), dim3(512), 0, a);
  } else {
    if (scatter) WTG_LAUNCH(ctx, "mld_emit", (k_mld_emit<K, true, 2048, WIDE>), dim3(grid), dim3(256), 0, a);
    else WTG_LAUNCH(ctx, "mld_emit", (k_mld_emit<K, false, 2048, WIDE>), dim3(grid), dim3(256), 0, a);
  }
}

// Levels [s0, L) of the keys d_sym (in P_{s0} order: sorted by their top s0
// bits, d_cnt0 = the 2^s0 node sizes; s0 = 0: any order, d_cnt0 unused);
// level l's bits go to bit (l - s0) * n of d_words.
// P: the plan of levels [s0, Lend) (workspace reserved by the caller); where
// Lend < L the last group scatters its keys too (as KO, to key buffer
// (ngroups - 1) & 1).
template <typename K, typename KO>
int mld_dense_groups(wtg_ctx* ctx, const MldPlan& P, const K* d_sym, uint64_t n, uint32_t L, uint32_t Lend, uint32_t s0,
                     const uint32_t* d_cnt0, const uint64_t* d_src_off, uint64_t* d_words,
                     unsigned long long* d_distinct) {
  constexpr bool WIDE = sizeof(KO) == 8;
  char* ws = (char*)ctx->ws;
  uint32_t* tcnt = (uint32_t*)(ws + P.off_tcnt);
  uint32_t* ploc = (uint32_t*)(ws + P.off_ploc);
  uint32_t* bsum = (uint32_t*)(ws + P.off_bsum);
  uint32_t* bpre = (uint32_t*)(ws + P.off_bpre);
  uint32_t* hist = (uint32_t*)(ws + P.off_hist);
  uint32_t* cum[2] = {(uint32_t*)(ws + P.off_cum[0]), (uint32_t*)(ws + P.off_cum[1])};
  uint32_t* tst = (uint32_t*)(ws + P.off_tst);
  uint32_t* nt = (uint32_t*)(ws + P.off_nt);
  uint32_t* tseg = (uint32_t*)(ws + P.off_tseg);
  uint64_t* scst = (uint64_t*)(ws + P.off_scst);
  uint32_t* ctr = (uint32_t*)(ws + P.off_ctr);
  KO* kbuf[2] = {(KO*)(ws + P.off_keys[0]), (KO*)(ws + P.off_keys[1])};
  // (the level words are cleared by the leaf-count passes)
  if (d_distinct) WTG_TRY(wtg_fill_u64(ctx, d_distinct, 1, 0));
  const uint32_t ntiles0 = (uint32_t)wtg_ceil_div(n, 1u << P.gt[0]);
  const void* src = d_sym;
  const uint32_t* cum_prev = nullptr;
  if (s0 > 0) {
    // the level-s0 nodes: their starts (cum[1]; group 0 writes cum[0]), tiles
    // per node, first tiles and the tile -> node map
    const uint64_t nb0 = 1ull << s0, st0 = wtg_ceil_div(nb0, 4096);
    WTG_TRY(wtg_fill_bytes_zero(ctx, scst, (char*)ctr + 256 - (char*)scst));
    WTG_LAUNCH(ctx, "mld_cum", k_scan_u32<uint32_t>, dim3((unsigned)st0), dim3(256), 0, d_cnt0, cum[1], nb0, scst,
               ctr, ctx->d_flag);
    WTG_LAUNCH_CHECK();
    WTG_LAUNCH(ctx, "mld_ntiles", k_mld_ntiles, dim3((unsigned)wtg_ceil_div(nb0, 256)), dim3(256), 0, cum[1], nb0,
               nt, P.gt[0]);
    WTG_LAUNCH_CHECK();
    WTG_TRY(wtg_fill_bytes_zero(ctx, scst, (char*)ctr + 256 - (char*)scst));
    WTG_LAUNCH(ctx, "mld_tiles", k_scan_u32<uint32_t>, dim3((unsigned)st0), dim3(256), 0, nt, tst, nb0, scst, ctr,
               ctx->d_flag);
    WTG_LAUNCH_CHECK();
    const uint64_t nt0 = wtg_ceil_div(n, 1u << P.gt[0]) + std::min<uint64_t>(n, nb0);
    WTG_LAUNCH(ctx, "mld_tseg", k_mld_tseg, dim3((unsigned)wtg_ceil_div(nt0, 256)), dim3(256), 0, tst, nb0, tseg,
               (uint64_t)P.maxtiles);
    WTG_LAUNCH_CHECK();
    cum_prev = cum[1];
  }
  for (uint32_t gi = 0; gi < P.ngroups; gi++) {
    const uint32_t s = P.gs[gi], g = P.gg[gi], G = 1u << g, tl = P.gt[gi];
    const bool more = gi + 1 < P.ngroups, last = !more && Lend == L;
    MldArgs a{};
    a.keys = src;
    a.n = n;
    a.L = L;
    a.s = s;
    a.g = g;
    a.tl = tl;
    a.ntiles0 = ntiles0;
    a.nseg = 1u << s;
    a.clear = 1;
    a.tstart = s ? tst : nullptr;
    a.tseg = s ? tseg : nullptr;
    a.cum_s = s ? cum_prev : nullptr;
    a.tcnt = tcnt;
    a.tcnt_w = tcnt;
    a.ploc = ploc;
    a.bpre = bpre;
    a.cum = cum[gi & 1];
    a.words = d_words;
    a.lvl0 = s0;
    // the input: no bits at or above L - s0 below the top s0 (none above bit 63)
    a.check = gi == 0 && L < 64 ? 1u : 0u;
    a.chk_shift = d_src_off ? L - s0 : L;
    a.src_off = gi == 0 ? d_src_off : nullptr;
    a.kout = last ? nullptr : kbuf[gi & 1];
    a.err = ctx->d_flag;
    // grid: an upper bound of the tiles (blocks past the real count exit)
    const uint64_t grid = s == 0 ? ntiles0 : wtg_ceil_div(n, 1u << tl) + std::min<uint64_t>(n, 1ull << s);
    const uint32_t nrows = (uint32_t)grid + 1;
    const uint32_t nblocks = (uint32_t)wtg_ceil_div(nrows, MLD_SR);
    if (gi == 0) mld_count_launch<K>(ctx, (unsigned)grid, a);
    else mld_count_launch<KO>(ctx, (unsigned)grid, a);
    WTG_LAUNCH_CHECK();
    WTG_LAUNCH(ctx, "mld_scan", k_mld_scan1, dim3(nblocks), dim3(256), 0, tcnt, ploc, bsum,
               s ? (const uint32_t*)(tst + (1u << s)) : nullptr, ntiles0, G, nrows);
    WTG_LAUNCH_CHECK();
    const uint64_t nbins = 1ull << (s + g);
    const uint64_t stiles = wtg_ceil_div(nbins, 4096);
    if (s == 0 && nblocks <= MLD_ROOT_BLOCKS) {
      WTG_LAUNCH(ctx, "mld_scan", k_mld_root, dim3(1), dim3(1024), 0, bsum, bpre, nblocks, G, hist, cum[gi & 1]);
      WTG_LAUNCH_CHECK();
    } else {
      WTG_LAUNCH(ctx, "mld_scan", k_mld_scan2, dim3(G), dim3(256), 0, bsum, bpre, nblocks, G);
      WTG_LAUNCH_CHECK();
      WTG_LAUNCH(ctx, "mld_hist", k_mld_hist, dim3((unsigned)wtg_ceil_div(nbins, 256)), dim3(256), 0, a, hist);
      WTG_LAUNCH_CHECK();
      WTG_TRY(wtg_fill_bytes_zero(ctx, scst, (char*)ctr + 256 - (char*)scst));
      WTG_LAUNCH(ctx, "mld_cum", k_scan_u32<uint32_t>, dim3((unsigned)stiles), dim3(256), 0, hist, cum[gi & 1], nbins,
                 scst, ctr, ctx->d_flag);
      WTG_LAUNCH_CHECK();
    }
    if (last && d_distinct) {
      WTG_LAUNCH(ctx, "mld_distinct", k_mld_nonzero, dim3((unsigned)std::min<uint64_t>(wtg_ceil_div(nbins, 256), 1024)),
                 dim3(256), 0, hist, nbins, d_distinct);
      WTG_LAUNCH_CHECK();
    }
    // the level bits of the group (and the keys in P_{s+g} order)
    if (gi == 0) mld_emit_launch<K, WIDE>(ctx, !last, (unsigned)grid, a);
    else mld_emit_launch<KO, WIDE>(ctx, !last, (unsigned)grid, a);
    WTG_LAUNCH_CHECK();
    if (more) {
      // the next group's tiles per node of level s+g
      WTG_LAUNCH(ctx, "mld_ntiles", k_mld_ntiles, dim3((unsigned)wtg_ceil_div(nbins, 256)), dim3(256), 0,
                 cum[gi & 1], nbins, nt, P.gt[gi + 1]);
      WTG_LAUNCH_CHECK();
      WTG_TRY(wtg_fill_bytes_zero(ctx, scst, (char*)ctr + 256 - (char*)scst));
      WTG_LAUNCH(ctx, "mld_tiles", k_scan_u32<uint32_t>, dim3((unsigned)stiles), dim3(256), 0, nt, tst, nbins, scst,
                 ctr, ctx->d_flag);
      WTG_LAUNCH_CHECK();
      const uint64_t ntiles_next = wtg_ceil_div(n, 1u << P.gt[gi + 1]) + std::min<uint64_t>(n, nbins);
      WTG_LAUNCH(ctx, "mld_tseg", k_mld_tseg, dim3((unsigned)wtg_ceil_div(ntiles_next, 256)), dim3(256), 0, tst,
                 nbins, tseg, (uint64_t)P.maxtiles);
      WTG_LAUNCH_CHECK();
      src = kbuf[gi & 1];
      cum_prev = cum[gi & 1];
    }
  }
  return WTG_OK;
}

template <typename K>
int mld_build_t(wtg_ctx* ctx, const K* d_sym, uint64_t n, uint32_t L, uint32_t s0, const uint32_t* d_cnt0,
                const uint64_t* d_src_off, uint64_t* d_words, wtg_node* d_nodes, uint64_t node_slots,
                unsigned long long* d_distinct) {
  if (n <= ONE_CAP && L <= MLD_GMAX && s0 == 0) {
    WTG_LAUNCH(ctx, "mld_one", k_mld_one<K>, dim3(1), dim3(1024), 0, d_sym, (uint32_t)n, L, d_words, d_nodes,
               node_slots, d_distinct, ctx->d_flag);
    WTG_LAUNCH_CHECK();
    return WTG_OK;
  }
  const MldPlan P = mld_plan(n, L, s0);
  WTG_TRY(wtg_ws_reserve(ctx, P.total));
  WTG_TRY((mld_dense_groups<K, uint32_t>(ctx, P, d_sym, n, L, L, s0, d_cnt0, d_src_off, d_words, d_distinct)));
  if (d_nodes && node_slots && s0 == 0) {
    WTG_LAUNCH(ctx, "nodes", k_mld_nodes, dim3((unsigned)wtg_ceil_div(node_slots, 256)), dim3(256), 0,
               (const uint32_t*)((char*)ctx->ws + P.off_cum[(P.ngroups - 1) & 1]), L, n, d_nodes, node_slots);
    WTG_LAUNCH_CHECK();
  }
  return WTG_OK;
}


// ---------------------------------------------------- small nodes, all levels
// Small nodes need no tables: whatever the level, their keys stay inside their
// own range of positions, so a block that holds whole nodes in LDS builds all
// their remaining levels alone, and its bits are one run per level.  A block
// takes the nodes that start in a window of LOC_W positions and end within
// LOC_CAP of the window's start (all but the window's last node do, and that
// one does if it has at most LOC_H keys); the others are "large".
constexpr uint32_t LOC_H = 512, LOC_W = LOC_CAP - LOC_H;
// a node of c keys that starts `off` positions into its window
__device__ __forceinline__ bool loc_large(uint32_t off, uint32_t c) { return (uint64_t)off + c > LOC_CAP; }
constexpr uint32_t LOC_TW = (2048 + LOC_W - 1) / LOC_W;  // windows per 2048-key tile of a listed segment

struct LocArgs {
  const void* kin;            // keys in P_s order (mode 0: the input)
  uint64_t n;
  uint32_t L, s;              // levels s .. L-1
  uint32_t mode;              // 0: one block, the whole input (n <= LOC_CAP, s = 0);
                              // 1: windows of the nodes st[0..m) (st[m] = n);
                              // 2: LOC_TW windows per tile t of the list: its segment k's leaves
                              //    st[k m .. k m + m), which end with the segment
  const uint32_t* st;         // node starts, non-decreasing
  uint32_t m;
  uint32_t nseg;              // mode 2: the list
  const uint32_t* tstart;
  const uint32_t* tseg;
  const uint32_t* seg_start;
  const uint32_t* seg_cnt;
  uint64_t* words;            // level l's bits at bit l * n
  unsigned long long* distinct;  // nullable: += the nodes that level L would have
  uint32_t* err;
  const uint32_t* left;       // modes 1 and 2, nullable: the large nodes left,
  uint32_t* tell;             // for the host here (pinned)
};

// the first i in [0, m] with st[i] >= v, where st[m] stands for a value >= v
// (a whole wave; 64 probes a step)
__device__ __forceinline__ uint32_t wave_lower_bound(const uint32_t* __restrict__ st, uint32_t m, uint32_t v) {
  uint32_t lo = 0, hi = m;
  while (lo < hi) {
    const uint32_t step = (hi - lo + 63) >> 6;
    const uint32_t i = lo + (uint32_t)lane_id() * step;
    const uint32_t c = popc64(wave_ballot(i < hi && st[i] < v));
    if (c == 0) break;
    const uint32_t up = lo + c * step;
    lo = lo + (c - 1) * step + 1;
    if (up < hi) hi = up;
  }
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
}

// All levels s .. L-1 of at most LOC_CAP consecutive keys of P_s that are whole
// nodes.  Every key carries its node's range (S, E) in the tile; with O(p) the
// level's ones before p, a zero at p goes to p - (O(p) - O(S)), a one to
// E - (O(E) - O(p)), and its node's range is cut at mid = E - (O(E) - O(S)).
// O comes from the level's bits and their prefix per 32-bit word (one LDS read
// per lookup).  Once every node is a single key the order stands and only bits
// remain to be read.  Bound by VALU issue (~30 instructions per key and level
// while nodes have several keys); 6000011 uint64 keys, 40 levels: levels 16..39
// in 0.25 ms (2.35 ms level by level over the whole array).  R64: more than 32 levels remain (64-bit keys in LDS).
template <typename KIN, bool R64>
__global__ __launch_bounds__(256) void k_mld_local(LocArgs a) {
  using KT = typename std::conditional<R64, uint64_t, uint32_t>::type;
  constexpr uint32_t M = LOC_CAP / 256;  // 64-key chunks per wave
  __shared__ KT s_key[LOC_CAP];
  __shared__ uint32_t s_se[LOC_CAP];
  __shared__ __align__(8) uint32_t s_bits[8][LOC_CAP / 32 + 2];
  __shared__ uint2 s_ow[4][LOC_CAP / 32 + 1];  // per wave: the level's bits and the ones before each word
  __shared__ uint32_t s_flag[2];
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t lane = (uint32_t)lane_id();
  if (a.left && blockIdx.x == 0 && threadIdx.x == 0)
    __hip_atomic_store(a.tell, *a.left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  // the block's keys: [a0, a0 + len) of P_s
  uint32_t a0 = 0, len = 0;
  if (a.mode == 0) {
    len = (uint32_t)a.n;
  } else {
    uint64_t lo, end = a.n;        // the window's first position, where the last node ends
    uint32_t m = a.m, width = LOC_W;
    const uint32_t* st = a.st;
    if (a.mode == 1) {
      lo = (uint64_t)blockIdx.x * LOC_W;
    } else {
      const uint32_t t = blockIdx.x / LOC_TW, j = blockIdx.x % LOC_TW;
      if (t >= a.tstart[a.nseg]) return;
      const uint32_t k = a.tseg[t];
      lo = (uint64_t)a.seg_start[k] + ((uint64_t)(t - a.tstart[k]) << 11) + j * LOC_W;
      if (j + 1 == LOC_TW) width = 2048 - j * LOC_W;
      end = (uint64_t)a.seg_start[k] + a.seg_cnt[k];
      st += (uint64_t)k * m;
    }
    if (lo >= end) return;
    const uint32_t i0 = wave_lower_bound(st, m, (uint32_t)lo);
    const uint32_t i1 = lo + width < end ? wave_lower_bound(st, m, (uint32_t)lo + width) : m;
    a0 = i0 < m ? st[i0] : (uint32_t)end;
    uint32_t e0 = i1 < m ? st[i1] : (uint32_t)end;
    if (a0 >= e0) return;
    const uint32_t last = st[wave_lower_bound(st, m, e0) - 1];  // the last node that starts in the window
    if (loc_large(last - (uint32_t)lo, e0 - last)) e0 = last;
    if (a0 >= e0) return;
    len = e0 - a0;
    if (len > LOC_CAP) return;  // (cannot happen for consistent tables)
  }
  const uint32_t r = a.L - a.s;  // levels to build
  const KIN* kin = reinterpret_cast<const KIN*>(a.kin) + a0;
  if (a.mode == 0) {  // one block: its words are cleared here
    const uint64_t nw = (a.n * a.L + 63) >> 6;
    for (uint64_t k = threadIdx.x; k < nw; k += 256) a.words[k] = 0ull;
    __threadfence();
  }
  // keys, and each key's node: heads are the keys whose top s bits differ from
  // the key before (positions past the keys are heads)
  KT x[M];
  uint32_t se[M];
  uint64_t hm[M];
  bool bad = false;
#pragma unroll
  for (uint32_t m = 0; m < M; m++) {
    const uint32_t p = (w + 4 * m) * 64 + lane;
    uint64_t k = 0, q = 0;
    if (p < len) {
      k = (uint64_t)kin[p];
      q = p ? (uint64_t)kin[p - 1] : 0;
    }
    const bool head = p >= len || p == 0 || (a.s > 0 && (k >> r) != (q >> r));
    if (a.mode == 0 && a.L < 64 && (k >> a.L) != 0) bad = true;
    hm[m] = wave_ballot(head);
    if (lane == 0) reinterpret_cast<uint64_t*>(s_bits[0])[w + 4 * m] = hm[m];
    x[m] = (KT)k;
  }
  if (bad) wtg_raise(a.err, WTG_FLAG_BADSYM);
  if (threadIdx.x < 2) s_flag[threadIdx.x] = 0;
  __syncthreads();
  {
    const uint64_t* hd = reinterpret_cast<const uint64_t*>(s_bits[0]);
    const uint64_t upto = ~0ull >> (63 - lane);  // lanes 0 .. lane
#pragma unroll
    for (uint32_t m = 0; m < M; m++) {
      const uint32_t c0 = w + 4 * m;
      uint32_t c = c0;
      uint64_t f = hm[m] & upto;
      while (f == 0 && c > 0) f = hd[--c];
      const uint32_t S = c * 64 + (f ? 63u - (uint32_t)__builtin_clzll(f) : 0u);
      c = c0;
      f = hm[m] & ~upto;
      while (f == 0 && ++c < LOC_CAP / 64) f = hd[c];
      const uint32_t E = f ? c * 64 + (uint32_t)__builtin_ctzll(f) : LOC_CAP;
      se[m] = S | E << 16;
    }
  }
  __syncthreads();
  bool active = true;  // some node has several keys (block-uniform)
  uint32_t ndist = 0;
  const uint64_t n = a.n;
  for (uint32_t i = 0; i < r; i++) {
    const uint32_t bp = r - 1 - i, lv = i & 7;
    uint64_t om[M];
#pragma unroll
    for (uint32_t m = 0; m < M; m++) {
      om[m] = wave_ballot((x[m] >> bp) & 1u);
      if (lane == 0) reinterpret_cast<uint64_t*>(s_bits[lv])[w + 4 * m] = om[m];
    }
    const bool last = i + 1 == r;
    if (active && !(last && !a.distinct)) {
      __syncthreads();
      if (threadIdx.x == 0) s_flag[lv & 1 ? 0 : 1] = 0;  // the next level's
      const uint32_t b = s_bits[lv][lane];
      const uint32_t cnt = __popc(b), incl = wave_incl_sum_dpp(cnt);
      s_ow[w][lane] = make_uint2(b, incl - cnt);
      if (lane == 63) s_ow[w][64] = make_uint2(0u, incl);
      wave_sync_lds_mld();
      bool any = false;
#pragma unroll
      for (uint32_t m = 0; m < M; m++) {
        const uint32_t c = w + 4 * m, p = c * 64 + lane;
        const uint32_t S = se[m] & 0xFFFFu, E = se[m] >> 16;
        const uint2 ws = s_ow[w][S >> 5], we = s_ow[w][E >> 5];
        const uint32_t OS = ws.y + __popc(__builtin_amdgcn_ubfe(ws.x, 0u, S & 31));
        const uint32_t OE = we.y + __popc(__builtin_amdgcn_ubfe(we.x, 0u, E & 31));
        const uint32_t base = s_ow[w][2 * c].y;
        const uint32_t OP =
            __builtin_amdgcn_mbcnt_hi((uint32_t)(om[m] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)om[m], base));
        const bool one = (x[m] >> bp) & 1u;
        const uint32_t mid = E - (OE - OS);
        const uint32_t dest = one ? E - (OE - OP) : p - (OP - OS);
        const uint32_t s2 = one ? mid : S, e2 = one ? E : mid;
        if (last) {
          ndist += popc64(wave_ballot(p < len && dest == s2));
        } else {
          any |= e2 - s2 > 1;
          s_key[dest] = x[m];
          s_se[dest] = s2 | e2 << 16;
        }
      }
      if (!last) {
        if (wave_ballot(any) != 0 && lane == 0) s_flag[lv & 1] = 1;
        __syncthreads();
        active = s_flag[lv & 1] != 0;
#pragma unroll
        for (uint32_t m = 0; m < M; m++) {
          const uint32_t p = (w + 4 * m) * 64 + lane;
          x[m] = s_key[p];
          se[m] = s_se[p];
        }
      }
    } else if (last && a.distinct && w == 0) {
      ndist = len;  // every key its own node
    }
    if (lv == 7 || last) {
      // the staged levels' bits: one run per level at l * n + a0
      __syncthreads();
      constexpr uint32_t RW = LOC_CAP / 64 + 1;  // words a run can touch
      for (uint32_t it = threadIdx.x; it < (lv + 1) * RW; it += 256) {
        const uint32_t k = it / RW;
        const uint64_t gs = (uint64_t)(a.s + i - lv + k) * n + a0, ge = gs + len;
        const uint64_t wi = (gs >> 6) + it % RW, wb = wi << 6;
        if (wb >= ge) continue;
        const uint32_t b0 = gs > wb ? (uint32_t)(gs - wb) : 0u;
        const uint32_t b1 = ge < wb + 64 ? (uint32_t)(ge - wb) : 64u;
        uint64_t v = lds_bits64(s_bits[k], (uint32_t)(wb + b0 - gs)) << b0;
        if (b1 < 64) v &= (1ull << b1) - 1;
        if (b0 == 0 && b1 == 64) a.words[wi] = v;
        else if (v) atomicOr((unsigned long long*)&a.words[wi], (unsigned long long)v);
      }
      __syncthreads();
    }
  }
  if (a.distinct && lane == 0 && ndist) atomicAdd(a.distinct, (unsigned long long)ndist);
}

// the large level-S nodes, as a list (in any order: the
// order of the segments changes no output)
__global__ __launch_bounds__(256) void k_mld_big(const uint32_t* __restrict__ cum, uint32_t nn, uint32_t* __restrict__ bs,
                                                 uint32_t* __restrict__ bc, uint32_t* __restrict__ nb, uint32_t cap,
                                                 uint32_t* __restrict__ err) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nn) return;
  const uint32_t st = cum[i], c = cum[i + 1] - st;
  if (!loc_large(st % LOC_W, c)) return;
  const uint32_t k = atomicAdd(nb, 1u);
  if (k >= cap) { wtg_raise(err, WTG_FLAG_BADSYM); return; }  // (cannot happen: the sizes sum to n)
  bs[k] = st;
  bc[k] = c;
}

// tiles of each listed segment (0 past the list)
__global__ __launch_bounds__(256) void k_mld_list_tiles(const uint32_t* __restrict__ bc, const uint32_t* __restrict__ nb,
                                                        uint32_t cap, uint32_t* __restrict__ nt, uint32_t tl) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= cap) return;
  nt[i] = i < *nb ? (uint32_t)(((uint64_t)bc[i] + (1u << tl) - 1) >> tl) : 0u;
}

// The tiles of a list of at most LIST_ONE segments in one launch: their count per
// segment (none past the list), first tiles and the tile -> segment map, for which four
// launches (k_mld_list_tiles, a fill, a scan, k_mld_tseg) take the other lists.
constexpr uint32_t LIST_ONE = 1024;
__global__ __launch_bounds__(LIST_ONE) void k_mld_list(const uint32_t* __restrict__ bc, const uint32_t* __restrict__ nb,
                                                       uint32_t cap, uint32_t tl, uint32_t* __restrict__ tst,
                                                       uint32_t* __restrict__ tseg, uint64_t maxtiles) {
  __shared__ uint32_t s_st[LIST_ONE + 1], s_w[LIST_ONE / 64];
  const uint32_t t = threadIdx.x, w = t >> 6;
  const uint32_t n = t < cap && t < *nb ? (uint32_t)(((uint64_t)bc[t] + (1u << tl) - 1) >> tl) : 0u;
  const uint32_t incl = wave_incl_sum_dpp(n);
  if ((t & 63) == 63) s_w[w] = incl;
  __syncthreads();
  uint32_t st = incl - n;
  for (uint32_t k = 0; k < w; k++) st += s_w[k];
  s_st[t] = st;
  if (t == LIST_ONE - 1) s_st[LIST_ONE] = st + n;
  __syncthreads();
  if (t < cap) tst[t] = st;
  const uint32_t total = s_st[cap];
  if (t == 0) tst[cap] = total;
  for (uint32_t k = t; k < total && k < maxtiles; k += LIST_ONE) {
    uint32_t lo = 0, hi = cap;  // s_st[lo] <= k < s_st[hi]
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (s_st[mid] <= k) lo = mid; else hi = mid;
    }
    tseg[k] = lo;
  }
}

// per listed segment (a block each): its leaves' starts, the large leaves as
// the next list, or (last group) its distinct leaves
__global__ __launch_bounds__(256) void k_mld_leaf(MldArgs a, uint32_t* __restrict__ lst, const uint32_t* __restrict__ nb,
                                                  uint32_t* __restrict__ bs2, uint32_t* __restrict__ bc2,
                                                  uint32_t* __restrict__ nb2, uint32_t cap,
                                                  unsigned long long* distinct) {
  __shared__ uint32_t s_wave[4];
  const uint32_t k = blockIdx.x, d = threadIdx.x, G = 1u << a.g;
  if (k >= *nb) return;
  uint32_t c = 0;
  if (d < G) c = mld_prefix(a, a.tstart[k + 1], d) - mld_prefix(a, a.tstart[k], d);
  uint32_t tot;
  const uint32_t st = a.seg_start[k] + mld_scan256<true>(c, s_wave, tot);
  if (d < G) lst[(uint64_t)k * G + d] = st;
  const uint32_t in_tile = (st - a.seg_start[k]) & 2047;
  if (nb2 && c && loc_large(in_tile % LOC_W, c)) {
    const uint32_t q = atomicAdd(nb2, 1u);
    if (q >= cap) { wtg_raise(a.err, WTG_FLAG_BADSYM); return; }
    bs2[q] = st;
    bc2[q] = c;
  }
  if (distinct) {
    const uint32_t q = popc64(wave_ballot(c != 0));
    if (lane_id() == 0 && q) atomicAdd(distinct, (unsigned long long)q);
  }
}

template <typename KIN>
void mld_local_launch(wtg_ctx* ctx, unsigned grid, const LocArgs& a) {
  if (a.L - a.s > 32) WTG_LAUNCH(ctx, "mld_local", (k_mld_local<KIN, true>), dim3(grid), dim3(256), 0, a);
  else WTG_LAUNCH(ctx, "mld_local", (k_mld_local<KIN, false>), dim3(grid), dim3(256), 0, a);
}

// Levels 0 .. L-1 of an input whose nodes get small before the last level:
// dense groups (tables over all 2^l prefixes) down to level S, where an average
// node is small, then the small nodes' remaining levels in one pass
// (k_mld_local).  Nodes that are still large there (skewed inputs) go on as a
// list of segments, up to 8 levels per round, each round handing its small
// leaves to the same kernel; a large node has more than LOC_H keys, so at most
// n / LOC_H of them exist at any level, and tables and work stay linear in n
// whatever the values.
template <typename K, typename KO>
int mld_sparse_t(wtg_ctx* ctx, const K* d_sym, uint64_t n, uint32_t L, uint64_t* d_words,
                 unsigned long long* d_distinct) {
  constexpr bool WIDE = sizeof(KO) == 8;
  if (d_distinct) WTG_TRY(wtg_fill_u64(ctx, d_distinct, 1, 0));
  LocArgs q{};
  q.n = n;
  q.L = L;
  q.words = d_words;
  q.distinct = d_distinct;
  q.err = ctx->d_flag;
  if (n <= LOC_CAP) {
    q.kin = d_sym;
    mld_local_launch<K>(ctx, 1, q);
    WTG_LAUNCH_CHECK();
    return WTG_OK;
  }
  const uint32_t S = std::min(mld_split_level(n), L - 1);
  const MldPlan P = mld_plan(n, S, 0, sizeof(KO));
  const uint32_t cap = (uint32_t)(n / LOC_H) + 1;  // listed segments
  const uint64_t maxt = wtg_ceil_div(n, MLD_WT) + cap + 1, maxb = wtg_ceil_div(maxt + 1, MLD_SR) + 1;
  // the list rounds' tables, after the dense ones (whose keys stay in use)
  size_t o = P.total;
  const size_t o_tcnt = o; o = wtg_align256(o + (maxt + 1) * 256 * 4);
  const size_t o_ploc = o; o = wtg_align256(o + (maxt + 1) * 256 * 4);
  const size_t o_bsum = o; o = wtg_align256(o + maxb * 256 * 4);
  const size_t o_bpre = o; o = wtg_align256(o + maxb * 256 * 4);
  const size_t o_lst = o; o = wtg_align256(o + (size_t)cap * 256 * 4);
  const size_t o_nt = o; o = wtg_align256(o + (size_t)cap * 4);
  const size_t o_tst = o; o = wtg_align256(o + ((size_t)cap + 1) * 4);
  const size_t o_tseg = o; o = wtg_align256(o + maxt * 4);
  size_t o_bs[2], o_bc[2];
  for (int b = 0; b < 2; b++) {
    o_bs[b] = o; o = wtg_align256(o + (size_t)cap * 4);
    o_bc[b] = o; o = wtg_align256(o + (size_t)cap * 4);
  }
  const size_t o_scst = o; o = wtg_align256(o + (wtg_ceil_div(cap, 4096) + 2) * 8);
  const size_t o_ctr = o; o = wtg_align256(o + 256);
  const size_t o_nb = o; o = wtg_align256(o + 256);
  WTG_TRY(wtg_ws_reserve(ctx, o));
  char* ws = (char*)ctx->ws;
  KO* kbuf[2] = {(KO*)(ws + P.off_keys[0]), (KO*)(ws + P.off_keys[1])};
  uint32_t* nb = (uint32_t*)(ws + o_nb);  // list lengths, 8 bytes apart
  // the words of levels S .. L-1 (level S's first word may end level S-1, whose group clears it)
  const uint64_t wt = (S * n + 63) >> 6;
  WTG_TRY(wtg_fill_bytes_zero(ctx, d_words + wt, (wtg_levels_words(n, L) - wt) * 8));
  WTG_TRY((mld_dense_groups<K, KO>(ctx, P, d_sym, n, L, S, 0, nullptr, nullptr, d_words, nullptr)));
  const uint32_t* cum = (const uint32_t*)(ws + P.off_cum[(P.ngroups - 1) & 1]);
  uint32_t kb = (P.ngroups - 1) & 1;  // the buffer that holds P_s
  WTG_TRY(wtg_fill_u64(ctx, nb, 1, 0));
  WTG_LAUNCH(ctx, "mld_big", k_mld_big, dim3((unsigned)wtg_ceil_div(1ull << S, 256)), dim3(256), 0, cum, 1u << S,
             (uint32_t*)(ws + o_bs[0]), (uint32_t*)(ws + o_bc[0]), nb, cap, ctx->d_flag);
  WTG_LAUNCH_CHECK();
  q.kin = kbuf[kb];
  q.s = S;
  q.mode = 1;
  q.st = cum;
  // how many large nodes are left: read back where the call waits in any case (in
  // a blocking context, or for the distinct count, and not while the stream is
  // being captured), so that no empty round is launched.  Otherwise the call only
  // enqueues: every round, for the longest list there can be (6000011 keys, 40
  // levels: 530 us on the stream against 410 read back with no large node, 565
  // against 580 with half of the keys in three values).
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  WTG_CHECK_HIP(hipStreamIsCapturing(ctx->stream, &cs));
  const bool ask = (ctx->blocking || d_distinct) && cs == hipStreamCaptureStatusNone;
  // (the small nodes' kernel stores it to pinned memory: a read is a wait, without a copy)
  q.m = 1u << S;
  q.left = ask ? nb : nullptr;
  q.tell = (uint32_t*)(ctx->d_stage + WTG_STAGE_AUX + 64);
  mld_local_launch<KO>(ctx, (unsigned)wtg_ceil_div(n, LOC_W), q);
  WTG_LAUNCH_CHECK();
  uint32_t cur = 0;
  for (uint32_t s = S; s < L;) {
    uint32_t hb = cap;
    if (ask) {
      WTG_CHECK_HIP(hipStreamSynchronize(ctx->stream));
      hb = *reinterpret_cast<volatile uint32_t*>(ctx->h_stage + WTG_STAGE_AUX + 64);
      if (hb > cap) hb = cap;  // (flagged on the device)
      if (hb == 0) break;
    }
    const uint32_t g = (L - s + (L - s + MLD_GMAX - 1) / MLD_GMAX - 1) / ((L - s + MLD_GMAX - 1) / MLD_GMAX);
    const bool last = s + g == L;
    const uint32_t* bs = (const uint32_t*)(ws + o_bs[cur]);
    const uint32_t* bc = (const uint32_t*)(ws + o_bc[cur]);
    uint32_t* tst = (uint32_t*)(ws + o_tst);
    uint32_t* tcnt = (uint32_t*)(ws + o_tcnt);
    uint32_t* ploc = (uint32_t*)(ws + o_ploc);
    uint32_t* bsum = (uint32_t*)(ws + o_bsum);
    uint32_t* bpre = (uint32_t*)(ws + o_bpre);
    uint32_t* lst = (uint32_t*)(ws + o_lst);
    uint64_t* scst = (uint64_t*)(ws + o_scst);
    uint32_t* ctr = (uint32_t*)(ws + o_ctr);
    const unsigned sgrid = (unsigned)wtg_ceil_div(hb, 256), stiles = (unsigned)wtg_ceil_div(hb, 4096);
    const uint64_t grid = wtg_ceil_div(n, MLD_WT) + hb;  // at least the tiles of hb segments of n keys at most
    const uint32_t nrows = (uint32_t)grid + 1, nblocks = (uint32_t)wtg_ceil_div(nrows, MLD_SR);
    MldArgs a{};
    a.keys = kbuf[kb];
    a.n = n;
    a.L = L;
    a.s = s;
    a.g = g;
    a.tl = 11;
    a.nseg = hb;
    a.tstart = tst;
    a.tseg = (const uint32_t*)(ws + o_tseg);
    a.seg_start = bs;
    a.seg_cnt = bc;
    a.tcnt = a.tcnt_w = tcnt;
    a.ploc = ploc;
    a.bpre = bpre;
    a.cum = lst;
    a.words = d_words;
    a.kout = last ? nullptr : kbuf[kb ^ 1];
    a.err = ctx->d_flag;
    if (hb <= LIST_ONE) {
      WTG_LAUNCH(ctx, "mld_tiles", k_mld_list, dim3(1), dim3(LIST_ONE), 0, bc, nb + 2 * cur, hb, 11u, tst,
                 (uint32_t*)(ws + o_tseg), maxt);
      WTG_LAUNCH_CHECK();
    } else {
      WTG_LAUNCH(ctx, "mld_ntiles", k_mld_list_tiles, dim3(sgrid), dim3(256), 0, bc, nb + 2 * cur, hb,
                 (uint32_t*)(ws + o_nt), 11u);
      WTG_LAUNCH_CHECK();
      WTG_TRY(wtg_fill_bytes_zero(ctx, scst, (char*)ctr + 256 - (char*)scst));
      WTG_LAUNCH(ctx, "mld_tiles", k_scan_u32<uint32_t>, dim3(stiles), dim3(256), 0, (uint32_t*)(ws + o_nt), tst,
                 (uint64_t)hb, scst, ctr, ctx->d_flag);
      WTG_LAUNCH_CHECK();
      WTG_LAUNCH(ctx, "mld_tseg", k_mld_tseg, dim3((unsigned)wtg_ceil_div(grid, 256)), dim3(256), 0, tst, (uint64_t)hb,
                 (uint32_t*)(ws + o_tseg), maxt);
      WTG_LAUNCH_CHECK();
    }
    mld_count_launch<KO>(ctx, (unsigned)grid, a);
    WTG_LAUNCH_CHECK();
    WTG_LAUNCH(ctx, "mld_scan", k_mld_scan1, dim3(nblocks), dim3(256), 0, tcnt, ploc, bsum,
               (const uint32_t*)(tst + hb), 0u, 1u << g, nrows);
    WTG_LAUNCH_CHECK();
    WTG_LAUNCH(ctx, "mld_scan", k_mld_scan2, dim3(1u << g), dim3(256), 0, bsum, bpre, nblocks, 1u << g);
    WTG_LAUNCH_CHECK();
    if (!last) WTG_TRY(wtg_fill_u64(ctx, nb + 2 * (cur ^ 1), 1, 0));
    WTG_LAUNCH(ctx, "mld_leaf", k_mld_leaf, dim3(hb), dim3(256), 0, a, lst, nb + 2 * cur, (uint32_t*)(ws + o_bs[cur ^ 1]),
               (uint32_t*)(ws + o_bc[cur ^ 1]), last ? nullptr : nb + 2 * (cur ^ 1), cap, last ? d_distinct : nullptr);
    WTG_LAUNCH_CHECK();
    mld_emit_launch<KO, WIDE>(ctx, !last, (unsigned)grid, a);
    WTG_LAUNCH_CHECK();
    s += g;
    kb ^= 1;
    cur ^= 1;
    if (last) break;
    q.kin = kbuf[kb];
    q.s = s;
    q.mode = 2;
    q.st = lst;
    q.m = 1u << g;
    q.nseg = hb;
    q.tstart = tst;
    q.tseg = a.tseg;
    q.seg_start = bs;
    q.seg_cnt = bc;
    q.left = ask ? nb + 2 * cur : nullptr;
    mld_local_launch<KO>(ctx, (unsigned)(grid * LOC_TW), q);
    WTG_LAUNCH_CHECK();
  }
  return WTG_OK;
}

}  // namespace

// 1: build with the multi-level direct passes; 0: the level-by-level split pipeline
int wtg_mld_enabled() {
  static int on = -1;
  if (on < 0) {
    const char* e = std::getenv("WTG_LEVEL_SPLIT");
    on = (e && e[0] == '1') ? 0 : 1;
  }
  return on;
}

static int mld_dispatch(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n, uint32_t L, uint32_t s0,
                        const uint32_t* d_cnt0, const uint64_t* d_src_off, uint64_t* d_words, wtg_node* d_nodes,
                        uint64_t node_slots, unsigned long long* d_distinct) {
  switch (sym_bytes) {
    case 1: return mld_build_t<uint8_t>(ctx, (const uint8_t*)d_sym, n, L, s0, d_cnt0, d_src_off, d_words, d_nodes,
                                        node_slots, d_distinct);
    case 2: return mld_build_t<uint16_t>(ctx, (const uint16_t*)d_sym, n, L, s0, d_cnt0, d_src_off, d_words, d_nodes,
                                         node_slots, d_distinct);
    case 4: return mld_build_t<uint32_t>(ctx, (const uint32_t*)d_sym, n, L, s0, d_cnt0, d_src_off, d_words, d_nodes,
                                         node_slots, d_distinct);
    default: return mld_build_t<uint64_t>(ctx, (const uint64_t*)d_sym, n, L, s0, d_cnt0, d_src_off, d_words,
                                          d_nodes, node_slots, d_distinct);
  }
}

template <typename K>
static int mld_sparse_dispatch(wtg_ctx* ctx, const void* d_sym, uint64_t n, uint32_t L, uint64_t* d_words,
                               unsigned long long* d_distinct) {
  return L > 32 ? mld_sparse_t<K, uint64_t>(ctx, (const K*)d_sym, n, L, d_words, d_distinct)
                : mld_sparse_t<K, uint32_t>(ctx, (const K*)d_sym, n, L, d_words, d_distinct);
}

// n >= 1, 1 <= L <= 64, n < 2^32; no node records
int wtg_mld_build_sparse(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n, uint32_t L, uint64_t* d_words,
                         unsigned long long* d_distinct) {
  switch (sym_bytes) {
    case 1: return mld_sparse_dispatch<uint8_t>(ctx, d_sym, n, L, d_words, d_distinct);
    case 2: return mld_sparse_dispatch<uint16_t>(ctx, d_sym, n, L, d_words, d_distinct);
    case 4: return mld_sparse_dispatch<uint32_t>(ctx, d_sym, n, L, d_words, d_distinct);
    default: return mld_sparse_dispatch<uint64_t>(ctx, d_sym, n, L, d_words, d_distinct);
  }
}

// n >= 1, 1 <= L <= 24, n < 2^32
int wtg_mld_build(wtg_ctx* ctx, const void* d_sym, int sym_bytes, uint64_t n, uint32_t L, uint64_t* d_words,
                  wtg_node* d_nodes, uint64_t node_slots, unsigned long long* d_distinct) {
  if (!d_nodes && mld_use_sparse(n, L)) return wtg_mld_build_sparse(ctx, d_sym, sym_bytes, n, L, d_words, d_distinct);
  return mld_dispatch(ctx, d_sym, sym_bytes, n, L, 0, nullptr, nullptr, d_words, d_nodes, node_slots, d_distinct);
}

// levels [s0, L) of keys already sorted by their top s0 bits (d_cnt0: the 2^s0
// node sizes), level l at bit (l - s0) * n of d_words; 0 <= s0 < L <= 24.
// d_src_off (nullable, s0 > 0): node v's keys are d_keys[d_src_off[v] ..] and
// hold only their low L - s0 bits (the node gives the top s0)
int wtg_mld_build_from(wtg_ctx* ctx, const void* d_keys, int key_bytes, uint64_t n, uint32_t L, uint32_t s0,
                       const uint32_t* d_cnt0, const uint64_t* d_src_off, uint64_t* d_words) {
  return mld_dispatch(ctx, d_keys, key_bytes, n, L, s0, d_cnt0, s0 ? d_src_off : nullptr, d_words, nullptr, 0,
                      nullptr);
}

size_t wtg_mld_ws_bytes(uint64_t n, uint32_t L, uint32_t s0) { return mld_plan(n, L, s0).total; }
