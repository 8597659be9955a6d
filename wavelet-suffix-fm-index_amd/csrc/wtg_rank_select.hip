// wtg_rank_select.hip -- (b) rank_support_v<1,1> directory and (b') the
// select_support_mcl<b,1> samples, built in one pass over the bit words.
//
// Directory (rank/rank_support_v_par.hpp:78-113): entry b covers words
// [8b, 8b+8): D[2b] = ones in words [0,8b); D[2b+1] = sum_j c_j << (63-9j) for
// j = 1..min(7, m-1), plus c_m << (63-9m) when the entry has m < 8 words.
//
// Select content (select/select_support_mcl_par.hpp:227-276 / :483-561): for
// superblock k of 4096 arguments, a = pos(4096k), e = pos(min(4096k+4095,m-1));
// e-a > logn^4 -> "long" (all 4096 positions) else "mini" (pos(4096k+64t)-a).
//
// Two passes over the words: ones per 512-word tile (k_rank_tile_sums) and,
// after their exclusive scan, one lane per directory entry (k_rank_entries):
// the lane's 8 word counts give the entry's 9-bit fields, a DPP scan of the
// entry totals its prefix, and the samples of the argument ranks j%64==0 (at
// most one per word and bit value) are found and written slot by slot: the low
// 32 bits of pos(j) straight into slot j/64 of the final mini
// array (mini offsets are < logn^4 < 2^32, so subtracting the low 32 bits of
// the superblock start later gives the exact offset), and the superblock
// starts/ends.  A second kernel classifies long/mini superblocks and rebases
// the mini offsets; a third fills the rare long superblocks.
#include "wtg_internal.hpp"
#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#define FLAG_LOOKBACK 1u

struct SelOut {
  uint32_t* mini;        // worst-case sized: ceil(nbits/4096)*64 entries
  uint64_t* sbstart;     // ceil(nbits/4096)+1
  uint64_t* sbend;       // ceil(nbits/4096)+1
  unsigned long long* last;  // 1 + position of the last argument (0 = none)
};

struct RankSelArgs {
  const uint64_t* words;
  uint64_t nbits;
  uint64_t W;            // words
  uint64_t S;            // capacity>>9 (entries 0..S)
  uint64_t* D;           // out (BUILD) or in (FROM_D)
  uint64_t* states;
  uint32_t* counter;
  uint32_t* err;
  const uint64_t* tpre;  // BUILD: ones before each tile (exclusive scan of k_rank_tile_sums)
  unsigned long long* ones_total;  // out: total ones
  SelOut sel[2];         // [0] = select0, [1] = select1
  int want[2];
};

// ones per tile of 512 words (64 directory entries), one wave per tile,
// lane-consecutive loads
constexpr int RS_TILE_WORDS = 512;
__device__ __forceinline__ void rank_tile_sums(const uint64_t* __restrict__ words, uint64_t W, uint64_t ntiles,
                                               uint32_t* __restrict__ tsum, bool aligned) {
  const uint64_t waves = (uint64_t)gridDim.x * 4;
  for (uint64_t t = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6); t < ntiles; t += waves) {
    const uint64_t q0 = t * (RS_TILE_WORDS / 2) + lane_id();  // 16-byte pairs of words
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < RS_TILE_WORDS / 128; k++) {
      const uint64_t wi = 2 * (q0 + (uint64_t)k * 64);
      if (aligned && wi + 2 <= W) {
        const uint4 v = reinterpret_cast<const uint4*>(words)[wi >> 1];
        c += popc64(((uint64_t)v.y << 32) | v.x) + popc64(((uint64_t)v.w << 32) | v.z);
      } else {
        c += (wi < W ? popc64(words[wi]) : 0u) + (wi + 1 < W ? popc64(words[wi + 1]) : 0u);
      }
    }
    c = wave_sum(c);
    if (lane_id() == 0) tsum[t] = c;
  }
}
__global__ __launch_bounds__(256) void k_rank_tile_sums(const uint64_t* __restrict__ words, uint64_t W,
                                                        uint64_t ntiles, uint32_t* __restrict__ tsum, bool aligned) {
  rank_tile_sums(words, W, ntiles, tsum, aligned);
}

__device__ __forceinline__ void rs_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// inclusive scan over the 64 lanes: DPP shifts inside each row of 16, then the
// row totals read back as scalars
__device__ __forceinline__ uint32_t wave_incl_scan_dpp(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);  // row_shr:8
  const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
  const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
  const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
  const uint32_t row = (uint32_t)lane_id() >> 4;
  return v + (row == 0 ? 0u : row == 1 ? r0 : row == 2 ? r0 + r1 : r0 + r1 + r2);
}

// Directory entries and select samples: one lane per directory entry (8
// words), one wave per tile of 512 words.  The lane's word counts give the
// entry's 9-bit fields directly; one DPP scan of the entry totals gives each
// entry's prefix inside the tile.  Select samples (argument ranks that are
// multiples of 64): a word holds at most one per bit value, and a tile's are
// consecutive slots, 512 of both values together.  Each word that holds one
// writes its number to the slot's place in LDS; then the lanes take the slots in
// order, 64 at a time, every lane with work, and the samples leave as whole
// lines.  n = 2^28, 20 levels (5.37 Gbit): 461 us with the owner of each word
// selecting (half of the lanes idle) and storing, 298 us so; the directory
// alone takes 140.  A lane going through its entry's samples in a loop: 530 us
// (one chain of dependent steps), 700 us two of each value at a time.
constexpr uint32_t RS_SLOTS = RS_TILE_WORDS + 1, RS_ENDS = 9;  // a tile's samples, superblock ends of one value, at most
struct TileSel {       // one bit value's arguments in a tile
  uint64_t t0;         // the vector's arguments before the tile
  uint16_t* slot;      // the word of each sample (LDS)
  uint16_t* end;       // the word of each superblock end (LDS)
};
// word number `widx` of the tile holds c arguments, r of the tile's before it
__device__ __forceinline__ void word_marks(const TileSel& s, uint32_t widx, uint32_t r, uint32_t c) {
  const uint32_t q = ((uint32_t)s.t0 & 4095u) + r;       // rank, from the superblock of the tile's first argument
  const uint32_t d = (0u - q) & 63u;
  if (d < c) s.slot[((q + 63) >> 6) - ((((uint32_t)s.t0 & 4095u) + 63) >> 6)] = (uint16_t)widx;
  const uint32_t de = 4095u - (q & 4095u);
  if (de < c) s.end[q >> 12] = (uint16_t)widx;
}
__device__ __forceinline__ uint32_t rs_at(uint32_t widx) {  // a word's place in LDS (spread over the banks)
  return widx ^ ((widx >> 5) & 7);
}

__device__ __forceinline__ void rank_entries(const RankSelArgs& a, uint64_t ntiles, bool write_dir, bool aligned) {
  __shared__ uint64_t s_x[4][RS_TILE_WORDS];
  __shared__ uint16_t s_f[4][RS_TILE_WORDS];          // ones of the tile before each word
  __shared__ uint16_t s_slot[4][2][RS_SLOTS + 1], s_end[4][2][RS_ENDS + 1];
  const uint64_t t = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= ntiles) return;
  const int lane = lane_id();
  const uint64_t e = t * 64 + (uint64_t)lane;  // directory entry
  const uint64_t w0 = e * 8;
  uint64_t x[8];
  if (aligned && w0 + 8 <= a.W) {
    const uint4* q = reinterpret_cast<const uint4*>(a.words + w0);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint4 v = q[k];
      x[2 * k] = ((uint64_t)v.y << 32) | v.x;
      x[2 * k + 1] = ((uint64_t)v.w << 32) | v.z;
    }
  } else {
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = w0 + k < a.W ? a.words[w0 + k] : 0ull;
  }
  uint32_t f[9];  // f[j] = ones in words [w0, w0 + j)
  f[0] = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) f[k + 1] = f[k] + popc64(x[k]);
  const uint32_t incl = wave_incl_scan_dpp(f[8]);
  const uint64_t tp0 = a.tpre[t], tp1 = a.tpre[t + 1], T = a.tpre[ntiles];
  const uint32_t tin = incl - f[8];   // ones of the tile before word w0
  const uint64_t pre = tp0 + tin;
  if (write_dir && e <= a.S) {
    const uint64_t m = a.W > w0 ? (a.W - w0 < 8 ? a.W - w0 : 8) : 0;  // words of the entry
    uint64_t F = 0;
#pragma unroll
    for (int j = 1; j < 8; j++)
      if ((uint64_t)j <= m) F |= (uint64_t)f[j] << (63 - 9 * j);
    a.D[2 * e] = pre;
    a.D[2 * e + 1] = F;
  }
  if (t == 0 && lane == 0) *a.ones_total = T;
  if (!a.want[0] && !a.want[1]) return;
  const uint64_t tb = t * RS_TILE_WORDS * 64;  // the tile's first bit
  const uint64_t v0 = tb < a.nbits ? tb : a.nbits;
  const uint64_t v1 = tb + RS_TILE_WORDS * 64 < a.nbits ? tb + RS_TILE_WORDS * 64 : a.nbits;
  const uint32_t wv = threadIdx.x >> 6;
  const TileSel g1{tp0, s_slot[wv][1], s_end[wv][1]}, g0{v0 - tp0, s_slot[wv][0], s_end[wv][0]};
#pragma unroll
  for (uint32_t k = 0; k < 8; k++) {
    const uint32_t widx = (uint32_t)lane * 8 + k, r = tin + f[k], c = f[k + 1] - f[k];
    s_x[wv][rs_at(widx)] = x[k];
    s_f[wv][widx] = (uint16_t)r;
    if (a.want[1]) word_marks(g1, widx, r, c);
    if (a.want[0]) {
      const uint64_t lo = (w0 + k) * 64;
      const uint32_t z = lo + 64 <= a.nbits ? 64 - c
                         : lo >= a.nbits   ? 0u
                                           : popc64(~x[k] & ((1ull << (a.nbits - lo)) - 1));
      word_marks(g0, widx, widx * 64 - r, z);
    }
  }
  rs_wave_sync();
  // position in the tile of argument rank j of the vector, in word widx
  const auto position = [&](uint32_t b, uint64_t j, uint64_t t0, uint32_t widx) {
    const uint64_t xw = s_x[wv][rs_at(widx)];
    const uint32_t fw = s_f[wv][widx], flip = b ? 0u : ~0u;
    const uint32_t before = b ? fw : widx * 64 - fw;
    return widx * 64 + select_halves((uint32_t)xw ^ flip, (uint32_t)(xw >> 32) ^ flip, (uint32_t)(j - t0) - before);
  };
  // (a tile's argument count wraps only where set bits past the vector's end
  // outnumber its last zeros)
#pragma unroll
  for (uint32_t b = 0; b < 2; b++) {
    if (!a.want[b]) continue;
    const uint64_t t0 = b ? tp0 : v0 - tp0, t1 = b ? tp1 : v1 - tp1;
    const uint64_t first = (t0 + 63) >> 6, end = (t1 + 63) >> 6;
    const uint32_t n = end <= first ? 0u : end - first < RS_SLOTS ? (uint32_t)(end - first) : RS_SLOTS;
#pragma unroll 2
    for (uint32_t i = (uint32_t)lane; i < n; i += 64) {
      const uint64_t slot = first + i;
      const uint64_t pos = tb + position(b, slot * 64, t0, s_slot[wv][b][i]);
      a.sel[b].mini[slot] = (uint32_t)pos;
      if ((slot & 63) == 0) a.sel[b].sbstart[slot >> 6] = pos;
    }
    const uint64_t eb = t0 >> 12, ee = t1 >> 12;  // superblocks that end in the tile
    const uint32_t ne = ee <= eb ? 0u : ee - eb < RS_ENDS ? (uint32_t)(ee - eb) : RS_ENDS;
    if ((uint32_t)lane < ne)
      a.sel[b].sbend[eb + lane] = tb + position(b, (eb + lane) * 4096 + 4095, t0, s_end[wv][b][lane]);
  }
  // last argument position (+1): only the tile holding the last one (the last
  // zero) writes it, a plain store; the scanned tile counts identify that tile
  const bool has_last1 = tp0 < T && tp1 == T;
  const bool has_last0 = v0 - tp0 < a.nbits - T && v1 - tp1 == a.nbits - T;
  if (has_last1 || has_last0) {
    uint64_t last1 = 0, last0 = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const uint64_t lo = (w0 + k) * 64;
      if (lo < a.nbits) {
        const uint64_t z = ~x[k] & (a.nbits - lo >= 64 ? ~0ull : (1ull << (a.nbits - lo)) - 1);
        if (x[k]) last1 = lo + (63 - __clzll(x[k])) + 1;
        if (z) last0 = lo + (63 - __clzll(z)) + 1;
      }
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint64_t o1 = (uint64_t)__shfl_xor((unsigned long long)last1, d);
      const uint64_t o0 = (uint64_t)__shfl_xor((unsigned long long)last0, d);
      last1 = o1 > last1 ? o1 : last1;
      last0 = o0 > last0 ? o0 : last0;
    }
    if (lane == 0) {
      if (a.want[1] && has_last1) *a.sel[1].last = last1;
      if (a.want[0] && has_last0) *a.sel[0].last = last0;
    }
  }
}
__global__ __launch_bounds__(256) void k_rank_entries(RankSelArgs a, uint64_t ntiles, bool write_dir, bool aligned) {
  rank_entries(a, ntiles, write_dir, aligned);
}

// ----------------------------------------------------- select assembly
struct AsmArgs {
  uint32_t* mini;
  uint8_t* mini_width;
  uint8_t* long_width;
  uint32_t* long_flag;
  const uint64_t* sbstart;
  const uint64_t* sbend;
  const unsigned long long* last;
  uint64_t m;          // arguments
  uint64_t sb;
  uint32_t logn4;
};

__device__ __forceinline__ uint32_t hi_dev(uint64_t x) { return x ? 63 - __clzll(x) : 0; }

// thread per 4 mini slots (one 16-byte load and store): rebase the samples of
// mini superblocks to their start, clear those of long superblocks; the first
// thread of a superblock writes its widths and long flag
__device__ __forceinline__ void select_assemble(const AsmArgs& a) {
  const uint64_t idx4 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx4 >= a.sb * 16) return;
  const uint64_t k = idx4 >> 4;  // superblock (64 slots = 16 threads)
  const uint64_t st = a.sbstart[k];
  const uint64_t en = (k + 1 < a.sb) ? a.sbend[k] : (uint64_t)(*a.last) - 1;
  const bool lng = (en - st) > (uint64_t)a.logn4;
  const uint64_t nsamp = (a.m + 63) / 64;
  const uint64_t i0 = idx4 * 4;
  uint4 v = reinterpret_cast<const uint4*>(a.mini)[idx4];
  const uint32_t s32 = (uint32_t)st;
  v.x = (!lng && i0 + 0 < nsamp) ? v.x - s32 : 0u;
  v.y = (!lng && i0 + 1 < nsamp) ? v.y - s32 : 0u;
  v.z = (!lng && i0 + 2 < nsamp) ? v.z - s32 : 0u;
  v.w = (!lng && i0 + 3 < nsamp) ? v.w - s32 : 0u;
  reinterpret_cast<uint4*>(a.mini)[idx4] = v;
  if ((idx4 & 15) == 0) {
    a.mini_width[k] = lng ? 0 : (uint8_t)(hi_dev(en - st) + 1);
    a.long_width[k] = lng ? (uint8_t)(hi_dev(en) + 1) : 0;
    a.long_flag[k] = lng ? 1u : 0u;
  }
}
__global__ __launch_bounds__(256) void k_select_assemble(AsmArgs a) { select_assemble(a); }

// also lists the long superblocks (list[ex[k]] = k) and copies their count
// ex[sb] to *nl_out
__device__ __forceinline__ void long_index(const uint32_t* __restrict__ flag, const uint32_t* __restrict__ ex,
                                           int64_t* __restrict__ li, uint64_t sb, uint32_t* __restrict__ list,
                                           uint32_t* __restrict__ nl_out) {
  const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < sb) {
    li[k] = flag[k] ? (int64_t)ex[k] : -1;
    if (flag[k]) list[ex[k]] = (uint32_t)k;
  }
  if (k == 0) *nl_out = ex[sb];
}
__global__ void k_long_index(const uint32_t* __restrict__ flag, const uint32_t* __restrict__ ex,
                             int64_t* __restrict__ li, uint64_t sb, uint32_t* __restrict__ list,
                             uint32_t* __restrict__ nl_out) {
  long_index(flag, ex, li, sb, list, nl_out);
}

// one block of LF_THREADS per long superblock (list[blockIdx.x]): enumerate the
// arguments in [a, e], one word per thread per round (a long superblock can
// hold dense stretches, and each thread walks its word's set bits serially)
constexpr int LF_THREADS = 1024;
__device__ __forceinline__ void long_fill(const uint64_t* __restrict__ words, uint64_t nbits, int bit,
                                          const uint64_t* __restrict__ sbstart, const uint64_t* __restrict__ sbend,
                                          const unsigned long long* last, const uint32_t* __restrict__ list,
                                          uint64_t sb, uint64_t* __restrict__ pool) {
  constexpr int NWV = LF_THREADS / 64;
  __shared__ uint32_t s_wave[NWV];
  const uint64_t k = list[blockIdx.x];
  const uint64_t st = sbstart[k];
  const uint64_t en = (k + 1 < sb) ? sbend[k] : (uint64_t)(*last) - 1;
  uint64_t* out = pool + (uint64_t)blockIdx.x * 4096;
  uint32_t run = 0;
  const uint64_t w0 = st >> 6, w1 = en >> 6;
  for (uint64_t base = w0; base <= w1; base += LF_THREADS) {
    const uint64_t wi = base + threadIdx.x;
    uint64_t x = 0;
    if (wi <= w1) {
      x = bit ? words[wi] : ~words[wi];
      const uint64_t lo = wi * 64;
      if (lo < st) x &= ~0ull << (st - lo);
      if (lo + 63 > en) x &= (en - lo == 63) ? ~0ull : ((1ull << (en - lo + 1)) - 1);
      if (lo + 64 > nbits) x &= (nbits > lo) ? ((nbits - lo >= 64) ? ~0ull : ((1ull << (nbits - lo)) - 1)) : 0ull;
    }
    const uint32_t c = popc64(x);
    const int w = threadIdx.x >> 6, l = lane_id();
    const uint32_t incl = wave_incl_scan(c);
    if (l == 63) s_wave[w] = incl;
    __syncthreads();
    uint32_t off = 0, tt = 0;
#pragma unroll
    for (int q = 0; q < NWV; q++) { const uint32_t t = s_wave[q]; if (q < w) off += t; tt += t; }
    __syncthreads();
    uint32_t r = run + incl - c + off;
    while (x) {
      if (r < 4096) out[r] = wi * 64 + (uint64_t)__builtin_ctzll(x);
      r++;
      x &= x - 1;
    }
    run += tt;
  }
}
__global__ __launch_bounds__(LF_THREADS) void k_long_fill(const uint64_t* __restrict__ words, uint64_t nbits,
                                                          int bit, const uint64_t* __restrict__ sbstart,
                                                          const uint64_t* __restrict__ sbend,
                                                          const unsigned long long* last,
                                                          const uint32_t* __restrict__ list, uint64_t sb,
                                                          uint64_t* __restrict__ pool) {
  long_fill(words, nbits, bit, sbstart, sbend, last, list, sb, pool);
}

// ------------------------------------------- the same for many vectors
// Vector blockIdx.y of each launch; its arguments are in a table.  16 vectors of
// 2^25 bits, directory and select1: 16 x 9 launches of 2 to 7 us each made building
// and asking them 3.25 ms, these seven 2.54 (sums 14 us, scan 5, entries 22,
// assembly, its scan and the index 5 each).
struct RsVec {
  RankSelArgs a;
  uint64_t wtiles;
  uint32_t* tsum;
  uint64_t* tpre;
  uint64_t* ctr;  // the counter block (32 words)
  bool aligned;
};
struct RsFin {
  AsmArgs a;
  uint32_t *ex, *list, *nl;
  int64_t* li;
};
struct RsLong {
  const uint64_t* words;
  uint64_t nbits;
  const uint64_t *sbstart, *sbend;
  const unsigned long long* last;
  const uint32_t* list;
  uint64_t sb;
  uint64_t* pool;
  uint32_t nl;
  int bit;
};
__global__ __launch_bounds__(256) void k_rank_tile_sums_many(const RsVec* __restrict__ v) {
  const RsVec r = v[blockIdx.y];
  if (blockIdx.x == 0 && threadIdx.x < 32) r.ctr[threadIdx.x] = 0;
  rank_tile_sums(r.a.words, r.a.W, r.wtiles, r.tsum, r.aligned);
}
// exclusive prefix of in[0, n) with the sum at out[n]: one block, 4096 at a time
template <typename OUT>
__device__ __forceinline__ void scan_by_block(const uint32_t* __restrict__ in, OUT* __restrict__ out, uint64_t n) {
  __shared__ uint32_t s_wave[4];
  OUT run = 0;
  for (uint64_t at = 0; at < n; at += 4096) {
    const uint64_t b = at + (uint64_t)threadIdx.x * 16;
    uint32_t x[16], c = 0, total;
#pragma unroll
    for (int k = 0; k < 16; k++) {
      x[k] = b + k < n ? in[b + k] : 0u;
      c += x[k];
    }
    OUT o = run + block_excl_scan_u32<true>(c, s_wave, total);
#pragma unroll
    for (int k = 0; k < 16; k++) {
      if (b + k < n) out[b + k] = o;
      o += x[k];
    }
    run += total;
  }
  if (threadIdx.x == 0) out[n] = run;
}
__global__ __launch_bounds__(256) void k_rank_scan_many(const RsVec* __restrict__ v) {
  scan_by_block(v[blockIdx.y].tsum, v[blockIdx.y].tpre, v[blockIdx.y].wtiles);
}
__global__ __launch_bounds__(256) void k_rank_entries_many(const RsVec* __restrict__ v) {
  const RsVec r = v[blockIdx.y];
  rank_entries(r.a, r.wtiles, true, r.aligned);
}
__global__ __launch_bounds__(256) void k_select_assemble_many(const RsFin* __restrict__ f) {
  const AsmArgs a = f[blockIdx.y].a;
  select_assemble(a);
}
__global__ __launch_bounds__(256) void k_select_scan_many(const RsFin* __restrict__ f) {
  scan_by_block(f[blockIdx.y].a.long_flag, f[blockIdx.y].ex, f[blockIdx.y].a.sb);
}
__global__ __launch_bounds__(256) void k_long_index_many(const RsFin* __restrict__ f) {
  const RsFin r = f[blockIdx.y];
  long_index(r.a.long_flag, r.ex, r.li, r.a.sb, r.list, r.nl);
}
__global__ __launch_bounds__(LF_THREADS) void k_long_fill_many(const RsLong* __restrict__ v) {
  const RsLong r = v[blockIdx.y];
  if (blockIdx.x >= r.nl) return;
  long_fill(r.words, r.nbits, r.bit, r.sbstart, r.sbend, r.last, r.list, r.sb, r.pool);
}

// ------------------------------------------------------------- queries
// rank1(i), or rank0(i) = i - rank1(i) for BIT = 0, from the rank1 directory
template <int BIT>
__global__ void k_rank9_query(const uint64_t* __restrict__ words, const uint64_t* __restrict__ D,
                              uint64_t nbits, const uint64_t* __restrict__ idx, uint64_t nq,
                              uint64_t* __restrict__ out) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  const uint64_t i = idx[q];
  if (i > nbits) { out[q] = WTG_NONE; return; }
  if (nbits == 0) { out[q] = 0; return; }
  const uint64_t r = rank9_of(rank9_fetch(D, words, (nbits + 63) >> 6, i));
  out[q] = BIT ? r : i - r;
}

__global__ void k_select_query(SelQ s, const uint64_t* __restrict__ iv, uint64_t nq, uint64_t m,
                               uint64_t* __restrict__ out) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  const uint64_t i = iv[q];
  out[q] = (i >= 1 && i <= m) ? select_plain(s, i) : WTG_NONE;
}

// ================================================================== host
extern "C" uint64_t wtg_rank9_words(uint64_t nbits) {
  if (nbits == 0) return 2;
  const uint64_t cap = (nbits + 63) / 64 * 64;
  return ((cap >> 9) + 1) * 2;
}

namespace {
struct SelTmp {
  uint64_t* sbend = nullptr;
  unsigned long long* last = nullptr;
};

// device memory of a select structure: its own allocation, or the next
// 256-byte-aligned piece of the arena
int sel_take(wtg_ctx* ctx, wtg_arena* ar, void** p, uint64_t bytes) {
  if (!ar) return wtg_malloc(ctx, p, bytes);
  const size_t a = wtg_align256(bytes);
  WTG_REQUIRE(ar->used + a <= ar->size, "select arena exhausted");
  *p = ar->base + ar->used;
  ar->used += a;
  return WTG_OK;
}

int sel_alloc_worst(wtg_ctx* ctx, uint64_t nbits, int bit, wtg_select* s, wtg_arena* ar) {
  std::memset(s, 0, sizeof(*s));
  s->nbits = nbits;
  s->bit = bit;
  const uint64_t sbmax = wtg_ceil_div(nbits, 4096) + 1;
  WTG_TRY(sel_take(ctx, ar, (void**)&s->mini, sbmax * 64 * 4));
  WTG_TRY(sel_take(ctx, ar, (void**)&s->superblock, sbmax * 8));
  return WTG_OK;
}

// scratch of one select structure's finish: long flags, their exclusive scan,
// the scan's tile states and counter, and the list of long superblocks
struct FinScratch {
  uint32_t* flag;
  uint32_t* ex;
  uint64_t* st;
  uint32_t* ctr;
  uint32_t* list;
};
FinScratch fin_scratch(char* scratch, uint64_t sb) {
  FinScratch f;
  f.flag = (uint32_t*)scratch;
  f.ex = (uint32_t*)(scratch + wtg_align256(sb * 4));
  f.st = (uint64_t*)(scratch + wtg_align256(sb * 4) + wtg_align256((sb + 1) * 4));
  f.ctr = (uint32_t*)((char*)f.st + wtg_align256((wtg_ceil_div(sb, 4096) + 1) * 8));
  f.list = (uint32_t*)((char*)f.ctr + 256);
  return f;
}

// finish one select structure once the arguments are counted, in two halves
// so that both structures share one host read of their long-superblock
// counts: sel_count stages the widths, the long flags and their scan, and
// writes the number of long superblocks to *d_nl; sel_fill allocates and
// fills the long pool once that number is on the host
// (many: its arguments go there instead of to launches)
int sel_count(wtg_ctx* ctx, uint64_t nbits, wtg_select* s, uint64_t m, const uint64_t* sbend,
              const unsigned long long* last, char* scratch, uint32_t* d_nl, wtg_arena* ar,
              std::vector<RsFin>* many = nullptr) {
  const uint64_t cap = (nbits + 63) / 64 * 64;
  s->arg_cnt = m;
  s->logn = (uint32_t)wtg_hi_host(cap) + 1;
  s->logn4 = (s->logn * s->logn) * (s->logn * s->logn);
  s->sb = wtg_ceil_div(m, 4096);
  s->n_long = 0;
  const uint64_t sb = s->sb;
  WTG_TRY(sel_take(ctx, ar, (void**)&s->mini_width, sb ? sb : 1));
  WTG_TRY(sel_take(ctx, ar, (void**)&s->long_width, sb ? sb : 1));
  WTG_TRY(sel_take(ctx, ar, (void**)&s->long_index, (sb ? sb : 1) * 8));
  if (sb == 0) return many ? WTG_OK : wtg_fill_bytes_zero(ctx, d_nl, 4);  // (many: cleared with the counters)
  const FinScratch f = fin_scratch(scratch, sb);
  uint32_t* flag = f.flag;
  uint32_t* ex = f.ex;
  uint64_t* st = f.st;
  uint32_t* ctr = f.ctr;
  if (!many) WTG_TRY(wtg_fill_bytes_zero(ctx, st, (char*)ctr + 256 - (char*)st));
  AsmArgs aa{};
  aa.mini = s->mini; aa.mini_width = s->mini_width; aa.long_width = s->long_width;
  aa.long_flag = flag; aa.sbstart = s->superblock; aa.sbend = sbend; aa.last = last;
  aa.m = m; aa.sb = sb; aa.logn4 = s->logn4;
  if (many) {
    many->push_back(RsFin{aa, ex, f.list, d_nl, s->long_index});
    return WTG_OK;
  }
  WTG_LAUNCH(ctx, "select_assemble", k_select_assemble, dim3((unsigned)wtg_ceil_div(sb * 16, 256)),
             dim3(256), 0, aa);
  WTG_LAUNCH_CHECK();
  WTG_LAUNCH(ctx, "select_scan", k_scan_u32<uint32_t>, dim3((unsigned)wtg_ceil_div(sb, 4096)), dim3(256), 0,
             flag, ex, sb, st, ctr, ctx->d_flag);
  WTG_LAUNCH_CHECK();
  WTG_LAUNCH(ctx, "select_longidx", k_long_index, dim3((unsigned)wtg_ceil_div(sb, 256)), dim3(256), 0,
             flag, ex, s->long_index, sb, f.list, d_nl);
  WTG_LAUNCH_CHECK();
  return WTG_OK;
}

int sel_fill(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, wtg_select* s, uint32_t nl,
             const uint64_t* sbend, const unsigned long long* last, const char* scratch, wtg_arena* ar,
             std::vector<RsLong>* many = nullptr) {
  const uint64_t sb = s->sb;
  s->n_long = nl;
  if (sb == 0 || nl == 0) return WTG_OK;
  const FinScratch f = fin_scratch(const_cast<char*>(scratch), sb);
  WTG_TRY(sel_take(ctx, ar, (void**)&s->long_pool, (uint64_t)nl * 4096 * 8));
  if (many) {
    many->push_back(RsLong{d_words, nbits, s->superblock, sbend, last, f.list, sb, s->long_pool, nl, s->bit});
    return WTG_OK;
  }
  WTG_TRY(wtg_fill_u64(ctx, s->long_pool, (uint64_t)nl * 4096, 0));
  WTG_LAUNCH(ctx, "select_longfill", k_long_fill, dim3(nl), dim3(LF_THREADS), 0, d_words, nbits, s->bit,
             s->superblock, sbend, last, f.list, sb, s->long_pool);
  WTG_LAUNCH_CHECK();
  return WTG_OK;
}

// workspace: counter | ones_total | last[2] | long counts[2] (256 bytes, first)
// | states | tile sums | tile prefixes | scan states | sbend[2] | finish scratch[2]
struct RsLayout {
  uint64_t W, S, tiles, wtiles, stiles, sbmax;
  size_t o_ctr, o_states, o_tsum, o_tpre, o_scst, o_end0, o_end1, fin_bytes, o_fin, total;
};
RsLayout rs_layout(uint64_t nbits) {
  RsLayout L{};
  const uint64_t cap = (nbits + 63) / 64 * 64;
  L.W = cap >> 6;
  L.S = cap >> 9;
  L.tiles = wtg_ceil_div(L.S + 1, 256);
  L.sbmax = wtg_ceil_div(nbits, 4096) + 1;
  // word tiles: every entry 0..S has its first word 8b inside them
  L.wtiles = wtg_ceil_div(8 * (L.S + 1), RS_TILE_WORDS);
  L.stiles = wtg_ceil_div(L.wtiles, 4096);
  size_t o = 0;
  L.o_ctr = o; o = wtg_align256(o + 256);
  L.o_states = o; o = wtg_align256(o + (L.tiles + 1) * 8);
  L.o_tsum = o; o = wtg_align256(o + (L.wtiles + 1) * 4);
  L.o_tpre = o; o = wtg_align256(o + (L.wtiles + 1) * 8);
  L.o_scst = o; o = wtg_align256(o + (L.stiles + 1) * 8);
  L.o_end0 = o; o = wtg_align256(o + L.sbmax * 8);
  L.o_end1 = o; o = wtg_align256(o + L.sbmax * 8);
  L.fin_bytes = wtg_align256(4 * wtg_align256((L.sbmax + 1) * 8) + 4096);
  L.o_fin = o; o = wtg_align256(o + 2 * L.fin_bytes);
  L.total = o;
  return L;
}
static_assert(WTG_RS_ONES_OFF == 64 && WTG_RS_NL_OFF == 192, "counter block layout");

}  // namespace

size_t wtg_rank_select_ws_bytes(uint64_t nbits) { return rs_layout(nbits).total; }
size_t wtg_select_arena_worst(uint64_t nbits) {
  const uint64_t sbmax = wtg_ceil_div(nbits, 4096) + 1;
  return wtg_align256(sbmax * 64 * 4) + wtg_align256(sbmax * 8);
}
size_t wtg_select_arena_count(uint64_t ones) {
  const uint64_t sb = std::max<uint64_t>(wtg_ceil_div(ones, 4096), 1);
  return 2 * wtg_align256(sb) + wtg_align256(sb * 8);
}
size_t wtg_select_arena_pool(uint32_t n_long) { return wtg_align256((uint64_t)n_long * 4096 * 8); }

int wtg_rank_select_begin(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, uint64_t* d_dir, bool build,
                          wtg_select* sel1, wtg_select* sel0, uint64_t known_ones, wtg_rs_pending* pend,
                          char* ws_ext, wtg_arena* ar) {
  *pend = wtg_rs_pending{};
  const RsLayout L = rs_layout(nbits);
  const uint64_t W = L.W, S = L.S, wtiles = L.wtiles, stiles = L.stiles;
  const size_t o_ctr = L.o_ctr, o_states = L.o_states, o_tsum = L.o_tsum, o_tpre = L.o_tpre;
  const size_t o_scst = L.o_scst, o_end0 = L.o_end0, o_end1 = L.o_end1, o_fin = L.o_fin;
  const size_t fin_bytes = L.fin_bytes;
  if (!ws_ext) WTG_TRY(wtg_ws_reserve(ctx, L.total));
  char* ws = ws_ext ? ws_ext : (char*)ctx->ws;
  WTG_TRY(wtg_fill_bytes_zero(ctx, ws, o_end0));
  uint32_t* ctr = (uint32_t*)(ws + o_ctr);
  unsigned long long* ones_total = (unsigned long long*)(ws + o_ctr + WTG_RS_ONES_OFF);
  unsigned long long* last = (unsigned long long*)(ws + o_ctr + 128);  // [0]=zeros, [1]=ones
  wtg_select* outs[2] = {sel0, sel1};
  RankSelArgs ra{};
  ra.words = d_words; ra.nbits = nbits; ra.W = W; ra.S = S; ra.D = d_dir;
  ra.states = (uint64_t*)(ws + o_states); ra.counter = ctr; ra.err = ctx->d_flag;
  ra.ones_total = ones_total;
  for (int t = 0; t < 2; t++) {
    ra.want[t] = outs[t] != nullptr && nbits > 0;
    if (ra.want[t]) {
      WTG_TRY(sel_alloc_worst(ctx, nbits, t, outs[t], ar));
      ra.sel[t].mini = outs[t]->mini;
      ra.sel[t].sbstart = outs[t]->superblock;
      ra.sel[t].sbend = (uint64_t*)(ws + (t ? o_end1 : o_end0));
      ra.sel[t].last = last + t;
    } else if (outs[t]) {
      std::memset(outs[t], 0, sizeof(wtg_select));
      outs[t]->bit = t;
    }
  }
  if (nbits == 0) {
    if (build) WTG_TRY(wtg_fill_u64(ctx, d_dir, 2, 0));
    for (int t = 0; t < 2; t++)
      if (outs[t]) {
        WTG_TRY(sel_take(ctx, ar, (void**)&outs[t]->mini_width, 1));
        WTG_TRY(sel_take(ctx, ar, (void**)&outs[t]->long_width, 1));
        WTG_TRY(sel_take(ctx, ar, (void**)&outs[t]->long_index, 8));
        outs[t]->logn = 1;
        outs[t]->logn4 = 1;
      }
    return WTG_OK;
  }
  {
    // ones per 512-word tile, their exclusive scan, then one pass writing the
    // directory entries and the select samples (a wave per tile)
    ra.tpre = (const uint64_t*)(ws + o_tpre);
    const unsigned g4 = (unsigned)wtg_ceil_div(wtiles, 4);
    WTG_LAUNCH(ctx, "rank_sums", k_rank_tile_sums, dim3(g4), dim3(256), 0, d_words, W, wtiles,
               (uint32_t*)(ws + o_tsum), ((uintptr_t)d_words & 15) == 0);
    WTG_LAUNCH_CHECK();
    WTG_LAUNCH(ctx, "rank_scan", k_scan_u32<uint64_t>, dim3((unsigned)stiles), dim3(256), 0,
               (const uint32_t*)(ws + o_tsum), (uint64_t*)(ws + o_tpre), wtiles, (uint64_t*)(ws + o_scst), ctr + 1,
               ctx->d_flag);
    WTG_LAUNCH_CHECK();
    WTG_LAUNCH(ctx, "rank_select", k_rank_entries, dim3(g4), dim3(256), 0, ra, wtiles, build,
               ((uintptr_t)d_words & 15) == 0);
  }
  WTG_LAUNCH_CHECK();
  if (!ra.want[0] && !ra.want[1]) return WTG_OK;  // rank9 alone: no count of ones needed
  pend->active = true;
  pend->d_words = d_words;
  pend->nbits = nbits;
  pend->d_nl = (const uint32_t*)(ws + o_ctr + WTG_RS_NL_OFF);
  pend->ar = ar;
  for (int t = 0; t < 2; t++) {
    pend->want[t] = ra.want[t];
    pend->outs[t] = ra.want[t] ? outs[t] : nullptr;
    pend->sbend[t] = ra.sel[t].sbend;
    pend->last[t] = last + t;
    pend->fin[t] = ws + o_fin + t * fin_bytes;
  }
  WTG_REQUIRE(known_ones != WTG_ONES_DEFER || (build && ws_ext), "rank/select: a deferred count needs its own workspace");
  if (known_ones == WTG_ONES_DEFER) return WTG_OK;
  uint64_t m1 = 0;
  if (build && known_ones != WTG_ONES_UNKNOWN) {
    m1 = known_ones;
  } else if (build) {
    unsigned long long t = 0;
    WTG_TRY(wtg_stage_d2h(ctx, &t, ones_total, 8));
    m1 = t;
  } else {
    // ones = D[2S] + ones in the last entry
    uint64_t e[2];
    WTG_CHECK_HIP(hipMemcpyAsync(e, d_dir + 2 * S, 16, hipMemcpyDeviceToHost, ctx->stream));
    std::vector<uint64_t> tailw(8, 0);
    const uint64_t wb = 8 * S;
    const uint64_t nt = W > wb ? W - wb : 0;
    if (nt) WTG_CHECK_HIP(hipMemcpyAsync(tailw.data(), d_words + wb, nt * 8, hipMemcpyDeviceToHost, ctx->stream));
    WTG_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    m1 = e[0];
    for (uint64_t k = 0; k < nt; k++) m1 += __builtin_popcountll(tailw[k]);
  }
  return wtg_rank_select_count(ctx, pend, m1);
}

int wtg_rank_select_count(wtg_ctx* ctx, wtg_rs_pending* pend, uint64_t ones) {
  if (!pend->active) return WTG_OK;
  const uint64_t m[2] = {pend->nbits - ones, ones};
  uint32_t* d_nl = const_cast<uint32_t*>(pend->d_nl);
  for (int t = 0; t < 2; t++)
    if (pend->want[t])
      WTG_TRY(sel_count(ctx, pend->nbits, pend->outs[t], m[t], pend->sbend[t], pend->last[t],
                        const_cast<char*>(pend->fin[t]), d_nl + t, pend->ar));
  return WTG_OK;
}

int wtg_rank_select_end(wtg_ctx* ctx, const wtg_rs_pending* pend, const uint32_t nl[2]) {
  if (!pend->active) return WTG_OK;
  for (int t = 0; t < 2; t++)
    if (pend->outs[t])
      WTG_TRY(sel_fill(ctx, pend->d_words, pend->nbits, pend->outs[t], nl[t], pend->sbend[t], pend->last[t],
                       pend->fin[t], pend->ar));
  return WTG_OK;
}

// a host table to its place in device memory (kept in `host` until the caller's
// next wait)
template <typename T>
static int many_upload(wtg_ctx* ctx, const std::vector<T>& v, std::vector<char>& host, char* dev) {
  static_assert(sizeof(T) <= WTG_RS_MANY_BYTES, "table entries");
  host.assign((const char*)v.data(), (const char*)(v.data() + v.size()));
  WTG_CHECK_HIP(hipMemcpyAsync(dev, host.data(), host.size(), hipMemcpyHostToDevice, ctx->stream));
  return WTG_OK;
}

// Many vectors in one launch of each kernel pay where none is much larger than
// the others (the grid is as wide as the largest for each) and one block scans a
// vector's tiles; nbits >= 1 each.
bool wtg_rank_select_many_fits(uint32_t nvec, const uint64_t* nbits) {
  uint64_t sum = 0, most = 0;
  for (uint32_t b = 0; b < nvec; b++) {
    const uint64_t t = rs_layout(nbits[b]).wtiles;
    sum += t;
    most = std::max(most, t);
  }
  return nvec >= 2 && most <= 65536 && most * nvec <= 8 * sum;
}

int wtg_rank_select_begin_many(wtg_ctx* ctx, uint32_t nvec, const uint64_t* const* d_words, const uint64_t* nbits,
                               uint64_t* const* dirs, wtg_select* sel1, wtg_rs_pending* pend, char* ws, size_t stride,
                               wtg_arena* ar, wtg_rs_many* many) {
  std::vector<RsVec> t(nvec);
  uint64_t most = 1;
  for (uint32_t b = 0; b < nvec; b++) {
    const RsLayout L = rs_layout(nbits[b]);
    char* w = ws + stride * b;
    unsigned long long* last = (unsigned long long*)(w + L.o_ctr + 128);
    WTG_TRY(sel_alloc_worst(ctx, nbits[b], 1, &sel1[b], ar));
    RsVec& r = t[b];
    r = RsVec{};
    r.a.words = d_words[b]; r.a.nbits = nbits[b]; r.a.W = L.W; r.a.S = L.S; r.a.D = dirs[b];
    r.a.err = ctx->d_flag;
    r.a.tpre = (const uint64_t*)(w + L.o_tpre);
    r.a.ones_total = (unsigned long long*)(w + L.o_ctr + WTG_RS_ONES_OFF);
    r.a.want[1] = 1;
    r.a.sel[1] = SelOut{sel1[b].mini, sel1[b].superblock, (uint64_t*)(w + L.o_end1), last + 1};
    r.wtiles = L.wtiles;
    r.tsum = (uint32_t*)(w + L.o_tsum);
    r.tpre = (uint64_t*)(w + L.o_tpre);
    r.ctr = (uint64_t*)(w + L.o_ctr);
    r.aligned = ((uintptr_t)d_words[b] & 15) == 0;
    most = std::max(most, L.wtiles);
    wtg_rs_pending& p = pend[b];
    p = wtg_rs_pending{};
    p.active = true;
    p.d_words = d_words[b];
    p.nbits = nbits[b];
    p.d_nl = (const uint32_t*)(w + L.o_ctr + WTG_RS_NL_OFF);
    p.ar = ar;
    p.want[1] = true;
    p.outs[1] = &sel1[b];
    p.sbend[1] = r.a.sel[1].sbend;
    p.last[1] = last + 1;
    p.fin[1] = w + L.o_fin + L.fin_bytes;
  }
  WTG_TRY(many_upload(ctx, t, many->host[0], many->dev));
  const RsVec* d = (const RsVec*)many->dev;
  const dim3 g((unsigned)wtg_ceil_div(most, 4), nvec);
  WTG_LAUNCH(ctx, "rank_sums", k_rank_tile_sums_many, g, dim3(256), 0, d);
  WTG_LAUNCH(ctx, "rank_scan", k_rank_scan_many, dim3(1, nvec), dim3(256), 0, d);
  WTG_LAUNCH(ctx, "rank_select", k_rank_entries_many, g, dim3(256), 0, d);
  WTG_LAUNCH_CHECK();
  return WTG_OK;
}

int wtg_rank_select_count_many(wtg_ctx* ctx, uint32_t nvec, wtg_rs_pending* pend, const uint64_t* ones,
                               wtg_rs_many* many) {
  std::vector<RsFin> t;
  for (uint32_t b = 0; b < nvec; b++)
    WTG_TRY(sel_count(ctx, pend[b].nbits, pend[b].outs[1], ones[b], pend[b].sbend[1], pend[b].last[1],
                      const_cast<char*>(pend[b].fin[1]), const_cast<uint32_t*>(pend[b].d_nl) + 1, pend[b].ar, &t));
  if (t.empty()) return WTG_OK;
  uint64_t sb = 1;
  for (const RsFin& f : t) sb = std::max(sb, f.a.sb);
  char* dev = many->dev + nvec * WTG_RS_MANY_BYTES;
  WTG_TRY(many_upload(ctx, t, many->host[1], dev));
  const RsFin* d = (const RsFin*)dev;
  const unsigned nv = (unsigned)t.size();
  WTG_LAUNCH(ctx, "select_assemble", k_select_assemble_many, dim3((unsigned)wtg_ceil_div(sb * 16, 256), nv), dim3(256),
             0, d);
  WTG_LAUNCH(ctx, "select_scan", k_select_scan_many, dim3(1, nv), dim3(256), 0, d);
  WTG_LAUNCH(ctx, "select_longidx", k_long_index_many, dim3((unsigned)wtg_ceil_div(sb, 256), nv), dim3(256), 0, d);
  WTG_LAUNCH_CHECK();
  return WTG_OK;
}

int wtg_rank_select_end_many(wtg_ctx* ctx, uint32_t nvec, const wtg_rs_pending* pend, const uint64_t* nl, wtg_arena* ar,
                             wtg_rs_many* many) {
  std::vector<RsLong> t;
  for (uint32_t b = 0; b < nvec; b++)
    WTG_TRY(sel_fill(ctx, pend[b].d_words, pend[b].nbits, pend[b].outs[1], (uint32_t)nl[b], pend[b].sbend[1],
                     pend[b].last[1], pend[b].fin[1], ar, &t));
  if (t.empty()) return WTG_OK;
  uint32_t most = 1;
  for (const RsLong& r : t) most = std::max(most, r.nl);
  WTG_TRY(wtg_fill_u64(ctx, ar->base, ar->used / 8, 0));
  char* dev = many->dev + 2 * nvec * WTG_RS_MANY_BYTES;
  WTG_TRY(many_upload(ctx, t, many->host[2], dev));
  WTG_LAUNCH(ctx, "select_longfill", k_long_fill_many, dim3(most, (unsigned)t.size()), dim3(LF_THREADS), 0,
             (const RsLong*)dev);
  WTG_LAUNCH_CHECK();
  return WTG_OK;
}

int wtg_rank_select_run(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, uint64_t* d_dir, bool build,
                        wtg_select* sel1, wtg_select* sel0) {
  wtg_rs_pending pend;
  WTG_TRY(wtg_rank_select_begin(ctx, d_words, nbits, d_dir, build, sel1, sel0, WTG_ONES_UNKNOWN, &pend));
  if (!pend.active) return WTG_OK;
  uint32_t nl[2] = {0, 0};
  WTG_TRY(wtg_stage_d2h(ctx, nl, pend.d_nl, 8));
  return wtg_rank_select_end(ctx, &pend, nl);
}

extern "C" int wtg_rank9_build(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, uint64_t* d_dir) {
  WTG_REQUIRE(ctx && d_dir && (nbits == 0 || d_words), "wtg_rank9_build: null argument");
  WTG_TRY(wtg_set_device(ctx));
  WTG_TRY(wtg_rank_select_run(ctx, d_words, nbits, d_dir, true, nullptr, nullptr));
  return wtg_finish(ctx);
}

extern "C" int wtg_rank9_select_build(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits,
                                      uint64_t* d_dir, wtg_select* sel1, wtg_select* sel0) {
  WTG_REQUIRE(ctx && d_dir && (nbits == 0 || d_words), "wtg_rank9_select_build: null argument");
  WTG_TRY(wtg_set_device(ctx));
  WTG_TRY(wtg_rank_select_run(ctx, d_words, nbits, d_dir, true, sel1, sel0));
  return wtg_finish(ctx);
}

extern "C" int wtg_select_build(wtg_ctx* ctx, const uint64_t* d_words, const uint64_t* d_dir,
                                uint64_t nbits, int bit, wtg_select* out) {
  WTG_REQUIRE(ctx && out && d_dir && (nbits == 0 || d_words), "wtg_select_build: null argument");
  WTG_REQUIRE(bit == 0 || bit == 1, "bit must be 0 or 1");
  WTG_TRY(wtg_set_device(ctx));
  WTG_TRY(wtg_rank_select_run(ctx, d_words, nbits, (uint64_t*)d_dir, false, bit ? out : nullptr,
                          bit ? nullptr : out));
  return wtg_finish(ctx);
}

namespace {
// argument words of the two-bit patterns `10` (pattern 10) and `01` (pattern 1):
// bit i = (bit i-1, bit i) == the pattern; the previous word's top bit is the
// carry, and before the vector sits the bit that rules out position 0
__global__ __launch_bounds__(256) void k_pattern_words(const uint64_t* __restrict__ w, uint64_t W, uint32_t pattern,
                                                       uint64_t tail_mask, uint64_t* __restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < W; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t x = w[i];
    const uint64_t c = i ? w[i - 1] >> 63 : (pattern == 10 ? 0ull : 1ull);
    const uint64_t prev = (x << 1) | c;
    uint64_t r = pattern == 10 ? prev & ~x : ~prev & x;
    if (i + 1 == W) r &= tail_mask;
    out[i] = r;
  }
}
}  // namespace

extern "C" int wtg_pattern_words(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, uint32_t pattern, int clip,
                                 uint64_t* d_out) {
  WTG_REQUIRE(ctx && (nbits == 0 || (d_words && d_out)), "wtg_pattern_words: null argument");
  WTG_REQUIRE(pattern == 10 || pattern == 1, "wtg_pattern_words: pattern must be 10 or 1 (01)");
  if (nbits == 0) return WTG_OK;
  WTG_TRY(wtg_set_device(ctx));
  const uint64_t W = (nbits + 63) / 64;
  const uint64_t tail = (clip && (nbits & 63)) ? (1ull << (nbits & 63)) - 1 : ~0ull;
  const unsigned g = (unsigned)std::min<uint64_t>(wtg_ceil_div(W, 256), 65536);
  WTG_LAUNCH(ctx, "pattern_words", k_pattern_words, dim3(g), dim3(256), 0, d_words, W, pattern, tail, d_out);
  WTG_LAUNCH_CHECK();
  return wtg_finish(ctx);
}

extern "C" int wtg_select_free(wtg_ctx* ctx, wtg_select* s) {
  WTG_REQUIRE(ctx && s, "null argument");
  wtg_free(ctx, s->superblock);
  wtg_free(ctx, s->mini);
  wtg_free(ctx, s->mini_width);
  wtg_free(ctx, s->long_index);
  wtg_free(ctx, s->long_width);
  wtg_free(ctx, s->long_pool);
  std::memset(s, 0, sizeof(*s));
  return WTG_OK;
}

extern "C" int wtg_rank9_batch(wtg_ctx* ctx, const uint64_t* d_words, const uint64_t* d_dir,
                               uint64_t nbits, const uint64_t* d_idx, uint64_t nq, uint64_t* d_out) {
  return wtg_rank9_batch_bit(ctx, d_words, d_dir, nbits, 1, d_idx, nq, d_out);
}

extern "C" int wtg_rank9_batch_bit(wtg_ctx* ctx, const uint64_t* d_words, const uint64_t* d_dir, uint64_t nbits,
                                   int bit, const uint64_t* d_idx, uint64_t nq, uint64_t* d_out) {
  WTG_REQUIRE(ctx && d_dir && (nq == 0 || (d_idx && d_out)), "wtg_rank9_batch: null argument");
  WTG_REQUIRE(bit == 0 || bit == 1, "wtg_rank9_batch_bit: bit must be 0 or 1");
  if (nq == 0) return WTG_OK;
  WTG_TRY(wtg_set_device(ctx));
  const dim3 g((unsigned)wtg_ceil_div(nq, 256));
  if (bit)
    WTG_LAUNCH(ctx, "rank9_query", k_rank9_query<1>, g, dim3(256), 0, d_words, d_dir, nbits, d_idx, nq, d_out);
  else
    WTG_LAUNCH(ctx, "rank9_query", k_rank9_query<0>, g, dim3(256), 0, d_words, d_dir, nbits, d_idx, nq, d_out);
  WTG_LAUNCH_CHECK();
  return wtg_finish(ctx);
}

extern "C" int wtg_select_batch(wtg_ctx* ctx, const wtg_select* s, const uint64_t* d_words,
                                const uint64_t* d_i, uint64_t nq, uint64_t* d_out) {
  WTG_REQUIRE(ctx && s && (nq == 0 || (d_i && d_out)), "wtg_select_batch: null argument");
  if (nq == 0) return WTG_OK;
  WTG_TRY(wtg_set_device(ctx));
  SelQ q{s->superblock, s->mini, s->long_index, s->long_pool, d_words,
         (s->nbits + 63) / 64, s->bit};
  WTG_LAUNCH(ctx, "select_query", k_select_query, dim3((unsigned)wtg_ceil_div(nq, 256)), dim3(256), 0,
             q, d_i, nq, s->arg_cnt, d_out);
  WTG_LAUNCH_CHECK();
  return wtg_finish(ctx);
}

// ------------------------------------------------- allocation-free rank9 build
// wtg_rank9_build_noalloc runs the kernels of wtg_rank9_build (tile sums, their
// exclusive scan, the directory pass) with their scratch in one file-scope
// device array instead of the context's workspace, so the call makes no device
// allocation.  Layout for a vector of at most WTG_RANK9_NOALLOC_MAX_BITS bits:
// [scan counter + ones total: 256 B][scan look-back states][tile sums][tile prefixes].
namespace {
constexpr uint64_t na_words(uint64_t nbits) { return (nbits + 63) / 64; }
constexpr uint64_t na_wtiles(uint64_t nbits) {
  return (8 * ((na_words(nbits) * 64 >> 9) + 1) + RS_TILE_WORDS - 1) / RS_TILE_WORDS;
}
constexpr uint64_t na_stiles(uint64_t nbits) { return (na_wtiles(nbits) + 4095) / 4096; }
constexpr uint64_t na_al(uint64_t x) { return (x + 255) & ~uint64_t(255); }
constexpr uint64_t NA_O_STATES = 256;
constexpr uint64_t na_o_tsum(uint64_t nbits) { return NA_O_STATES + na_al((na_stiles(nbits) + 1) * 8); }
constexpr uint64_t na_o_tpre(uint64_t nbits) { return na_o_tsum(nbits) + na_al((na_wtiles(nbits) + 1) * 4); }
constexpr uint64_t na_bytes(uint64_t nbits) { return na_o_tpre(nbits) + na_al((na_wtiles(nbits) + 1) * 8); }
constexpr uint64_t NA_SCRATCH_BYTES = na_bytes(WTG_RANK9_NOALLOC_MAX_BITS);
static_assert(NA_SCRATCH_BYTES <= (13ull << 20), "scratch of the allocation-free rank9 build is 13 MiB at most");
}  // namespace

static __device__ __align__(256) uint8_t scratch[NA_SCRATCH_BYTES];

// device addresses of `scratch`, one per device (each device holds its own copy)
static std::mutex g_na_mu;
static std::map<int, uint8_t*> g_na_ptr;

// Called by wtg_ctx_create with `device` current: resolves the device address
// of `scratch` once per device.
int wtg_noalloc_init_device(int device) {
  std::lock_guard<std::mutex> lk(g_na_mu);
  if (g_na_ptr.count(device)) return WTG_OK;
  void* ptr = nullptr;
  WTG_CHECK_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  if (!ptr) {
    wtg_set_error("hipGetSymbolAddress(scratch) returned a null address");
    return WTG_ERR_HIP;
  }
  g_na_ptr[device] = (uint8_t*)ptr;
  return WTG_OK;
}

__global__ void k_na_zero(uint64_t* __restrict__ d, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = 0;
}

extern "C" int wtg_rank9_build_noalloc(wtg_ctx* ctx, const uint64_t* d_words, uint64_t nbits, uint64_t* d_dir) {
  WTG_REQUIRE(ctx && d_dir && (nbits == 0 || d_words), "wtg_rank9_build_noalloc: null argument");
  if (nbits > WTG_RANK9_NOALLOC_MAX_BITS) {
    wtg_set_error("wtg_rank9_build_noalloc: nbits above WTG_RANK9_NOALLOC_MAX_BITS (2^35); use wtg_rank9_build");
    return WTG_ERR_UNSUPPORTED;
  }
  WTG_TRY(wtg_set_device(ctx));
  uint8_t* ws = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_na_mu);
    auto it = g_na_ptr.find(ctx->device);
    if (it != g_na_ptr.end()) ws = it->second;
  }
  if (!ws) {
    wtg_set_error("wtg_rank9_build_noalloc: scratch address of this device not resolved (context not created)");
    return WTG_ERR_HIP;
  }
  if (nbits == 0) {
    hipLaunchKernelGGL(k_na_zero, dim3(1), dim3(64), 0, ctx->stream, d_dir, (uint64_t)2);
    WTG_LAUNCH_CHECK();
    return wtg_finish(ctx);
  }
  const uint64_t cap = (nbits + 63) / 64 * 64;
  const uint64_t W = cap >> 6, S = cap >> 9;
  const uint64_t wtiles = na_wtiles(nbits), stiles = na_stiles(nbits);
  uint32_t* ctr = (uint32_t*)ws;
  unsigned long long* ones_total = (unsigned long long*)(ws + 64);
  uint64_t* scst = (uint64_t*)(ws + NA_O_STATES);
  uint32_t* tsum = (uint32_t*)(ws + na_o_tsum(nbits));
  uint64_t* tpre = (uint64_t*)(ws + na_o_tpre(nbits));
  // the scan's counter and look-back states start at zero (the previous call's
  // values stay in the array)
  const uint64_t nz = na_o_tsum(nbits) / 8;
  hipLaunchKernelGGL(k_na_zero, dim3((unsigned)wtg_ceil_div(nz, 256)), dim3(256), 0, ctx->stream, (uint64_t*)ws, nz);
  WTG_LAUNCH_CHECK();
  const bool aligned = ((uintptr_t)d_words & 15) == 0;
  const unsigned g4 = (unsigned)wtg_ceil_div(wtiles, 4);
  hipLaunchKernelGGL(k_rank_tile_sums, dim3(g4), dim3(256), 0, ctx->stream, d_words, W, wtiles, tsum, aligned);
  WTG_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_scan_u32<uint64_t>, dim3((unsigned)stiles), dim3(256), 0, ctx->stream,
                     (const uint32_t*)tsum, tpre, wtiles, scst, ctr, ctx->d_flag);
  WTG_LAUNCH_CHECK();
  RankSelArgs ra{};
  ra.words = d_words; ra.nbits = nbits; ra.W = W; ra.S = S; ra.D = d_dir;
  ra.err = ctx->d_flag; ra.tpre = tpre; ra.ones_total = ones_total;
  ra.want[0] = ra.want[1] = 0;
  hipLaunchKernelGGL(k_rank_entries, dim3(g4), dim3(256), 0, ctx->stream, ra, wtiles, true, aligned);
  WTG_LAUNCH_CHECK();
  return wtg_finish(ctx);
}
