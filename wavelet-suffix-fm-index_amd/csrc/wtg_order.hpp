// wtg_order.hpp -- a large batch of queries in the order of one of its columns.
//
// The walks of a large batch are bound by 128-byte lines from behind the L2s:
// 10^6 random queries touch most of a level that is several times an XCD's 4 MiB.
// Such a batch is first split into 256 parts by symbol (by position where the
// symbol is not known), at 255 of a sample of its own keys, so the parts are
// even whatever the keys are; the walk then takes the parts in order, each XCD
// an eighth of them, and an XCD's queries in flight share a small part of every
// level.  Answers are written where the query stood.  A batch whose sample is in
// order is walked as it came.  What it measured stands with the rules of its users
// (the order_pays functions).
#pragma once
#include "wtg_internal.hpp"

namespace {

constexpr uint32_t QO_BINS = 256, QO_SAMPLE = 1024, QO_XCDS = 8;
constexpr uint32_t QO_THREADS = 512, QO_PER = 8, QO_TILE = QO_THREADS * QO_PER;
constexpr uint32_t QO_RUNS = 16;
constexpr uint64_t QO_CHUNK = 1ull << 20;  // queries ordered at a time: the scratch is 36 bytes for each
constexpr uint32_t QO_COLS = 4;
struct QCols {
  const uint64_t* c[QO_COLS];
};
struct KeyCol {  // the key of a query: an element of a column
  const uint64_t* k;
  __device__ __forceinline__ uint64_t operator()(uint64_t i) const { return k[i]; }
};
struct QOrder {
  uint64_t* col[QO_COLS];  // the columns, in order
  uint32_t* q;             // where the query stood
  uint64_t* split;         // [QO_BINS - 1] first key of bins 1..
  uint32_t* tot;           // [QO_BINS] queries of each bin
  uint32_t* cur;           // [QO_BINS] of which placed
  uint32_t* asis;          // 1: the sample is in order, nothing else is filled in
};
constexpr size_t QO_BYTES = QO_CHUNK * (QO_COLS * 8 + 4) + QO_BINS * 16;

__device__ __forceinline__ uint32_t qo_bin(const uint64_t* s_split, uint64_t key) {
  uint32_t b = 0;  // splitters <= key
#pragma unroll
  for (uint32_t h = QO_BINS / 2; h > 0; h >>= 1)
    if (s_split[b + h - 1] <= key) b += h;
  return b;
}

// The splitters: every fourth of 1024 keys of the batch.  A block places 16 of
// them, 16 threads to a key, each counting the smaller ones among 64 (44 -> 5 us
// with one block and a thread for each key).  The batch is in order, up or down, if its
// sample is but for as many places as runs of a sixteenth of it would leave.
template <class KEY>
__global__ __launch_bounds__(256) void k_order_split(KEY key, uint64_t nq, QOrder o) {
  __shared__ uint64_t s_key[QO_SAMPLE + 16];
  const uint32_t t = threadIdx.x;
#pragma unroll
  for (uint32_t k = t; k < QO_SAMPLE; k += 256) s_key[k + (k >> 6)] = key((k * nq) / QO_SAMPLE);
  if (blockIdx.x == 0) o.tot[t] = o.cur[t] = 0;
  __syncthreads();
  if (blockIdx.x == 0) {
    uint32_t ups = 0, downs = 0;
    for (uint32_t k = t; k < QO_SAMPLE; k += 256) {
      const uint64_t a = s_key[k + (k >> 6)], b = k + 1 < QO_SAMPLE ? s_key[k + 1 + ((k + 1) >> 6)] : a;
      ups += a < b;
      downs += a > b;
    }
    ups = wave_sum(ups);
    downs = wave_sum(downs);
    __shared__ uint32_t s_run[2];
    if (t < 2) s_run[t] = 0;
    __syncthreads();
    if (lane_id() == 0) {
      atomicAdd(&s_run[0], ups);
      atomicAdd(&s_run[1], downs);
    }
    __syncthreads();
    if (t == 0) *o.asis = min(s_run[0], s_run[1]) < QO_RUNS;
  }
  const uint32_t mine = blockIdx.x * 16 + (t >> 4), part = (t & 15) * 64;
  const uint64_t v = s_key[mine + (mine >> 6)];
  uint32_t r = 0;
#pragma unroll 8
  for (uint32_t k = part; k < part + 64; k++) {
    const uint64_t x = s_key[k + (part >> 6)];
    r += x < v || (x == v && k < mine);
  }
#pragma unroll
  for (uint32_t d = 1; d < 16; d <<= 1) r += __shfl_xor(r, d, 64);
  constexpr uint32_t E = QO_SAMPLE / QO_BINS;
  if ((t & 15) == 0 && r % E == 0 && r) o.split[r / E - 1] = v;
}

template <class KEY>
__device__ __forceinline__ void qo_bins(const uint64_t* s_split, const KEY& key, uint64_t base, uint64_t nq,
                                        uint32_t (&bin)[QO_PER]) {
  uint64_t v[QO_PER];
#pragma unroll
  for (uint32_t k = 0; k < QO_PER; k++) v[k] = base + k * QO_THREADS < nq ? key(base + k * QO_THREADS) : 0ull;
#pragma unroll
  for (uint32_t k = 0; k < QO_PER; k++) bin[k] = qo_bin(s_split, v[k]);
}

template <class KEY>
__global__ __launch_bounds__(QO_THREADS) void k_order_count(KEY key, uint64_t nq, QOrder o) {
  __shared__ uint64_t s_split[QO_BINS];
  __shared__ uint32_t s_cnt[QO_BINS];
  if (*o.asis) return;
  const uint32_t t = threadIdx.x;
  if (t < QO_BINS) {
    s_split[t] = t < QO_BINS - 1 ? o.split[t] : ~0ull;
    s_cnt[t] = 0;
  }
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * QO_TILE + t;
  uint32_t bin[QO_PER];
  qo_bins(s_split, key, base, nq, bin);
#pragma unroll
  for (uint32_t k = 0; k < QO_PER; k++)
    if (base + k * QO_THREADS < nq) atomicAdd(&s_cnt[bin[k]], 1u);
  __syncthreads();
  if (t < QO_BINS && s_cnt[t]) atomicAdd(&o.tot[t], s_cnt[t]);
}

// A tile's queries by bin in LDS, a column at a time, so that neighbouring threads
// store to one run of a bin (16 queries, one line, in an even tile; stored where
// they were found 25-87 us, so 14-25 for one to four columns of 10^6).
// (the order inside a bin is the one the blocks arrive in: no answer depends on it)
template <uint32_t NC, class KEY>
__global__ __launch_bounds__(QO_THREADS) void k_order_put(QCols in, KEY key, uint64_t nq, QOrder o) {
  __shared__ uint64_t s_split[QO_BINS];
  __shared__ uint32_t s_cnt[QO_BINS], s_first[QO_BINS], s_tot[2][QO_BINS / 64];
  __shared__ uint32_t s_to[QO_TILE];
  __shared__ uint64_t s_buf[QO_TILE];
  if (*o.asis) return;
  const uint32_t t = threadIdx.x;
  uint32_t tot = 0, incl = 0;
  if (t < QO_BINS) {
    s_split[t] = t < QO_BINS - 1 ? o.split[t] : ~0ull;
    s_cnt[t] = 0;
    tot = o.tot[t];
    incl = wave_incl_sum_dpp(tot);
    if ((t & 63) == 63) s_tot[0][t >> 6] = incl;
  }
  __syncthreads();
  const uint64_t tile = (uint64_t)blockIdx.x * QO_TILE, base = tile + t;
  uint32_t bin[QO_PER], at[QO_PER];
  qo_bins(s_split, key, base, nq, bin);
#pragma unroll
  for (uint32_t k = 0; k < QO_PER; k++) at[k] = base + k * QO_THREADS < nq ? atomicAdd(&s_cnt[bin[k]], 1u) : 0u;
  __syncthreads();
  uint32_t cnt = 0, here = 0;
  if (t < QO_BINS) {
    cnt = s_cnt[t];
    here = wave_incl_sum_dpp(cnt);
    if ((t & 63) == 63) s_tot[1][t >> 6] = here;
  }
  __syncthreads();
  if (t < QO_BINS) {
    uint32_t to = incl - tot;
    here -= cnt;
    for (uint32_t w = 0; w < (t >> 6); w++) {
      to += s_tot[0][w];
      here += s_tot[1][w];
    }
    s_first[t] = here;                                            // in the tile
    s_cnt[t] = cnt ? to + atomicAdd(&o.cur[t], cnt) - here : 0u;  // from there to the ordered batch
  }
  __syncthreads();
  const uint32_t m = (uint32_t)(nq - tile < QO_TILE ? nq - tile : QO_TILE);
  uint32_t* s_q = reinterpret_cast<uint32_t*>(s_buf);
#pragma unroll
  for (uint32_t k = 0; k < QO_PER; k++)
    if (t + k * QO_THREADS < m) {
      at[k] += s_first[bin[k]];
      s_to[at[k]] = at[k] + s_cnt[bin[k]];
      s_q[at[k]] = (uint32_t)tile + t + k * QO_THREADS;
    }
  __syncthreads();
  for (uint32_t k = t; k < m; k += QO_THREADS) o.q[s_to[k]] = s_q[k];
#pragma unroll
  for (uint32_t c = 0; c < NC; c++) {
    uint64_t v[QO_PER];
#pragma unroll
    for (uint32_t k = 0; k < QO_PER; k++) v[k] = t + k * QO_THREADS < m ? in.c[c][base + k * QO_THREADS] : 0ull;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < QO_PER; k++)
      if (t + k * QO_THREADS < m) s_buf[at[k]] = v[k];
    __syncthreads();
    for (uint32_t k = t; k < m; k += QO_THREADS) o.col[c][s_to[k]] = s_buf[k];
  }
}

// scratch: `cols` columns of `cap` queries, their places, the tables
QOrder order_layout(char* scratch, uint64_t cap, uint32_t cols) {
  QOrder o{};
  for (uint32_t c = 0; c < cols; c++) o.col[c] = (uint64_t*)scratch + c * cap;
  o.split = (uint64_t*)scratch + cols * cap;
  o.asis = (uint32_t*)(o.split + QO_BINS - 1);
  o.tot = (uint32_t*)(o.split + QO_BINS);
  o.cur = o.tot + QO_BINS;
  o.q = o.cur + QO_BINS;
  return o;
}
template <uint32_t NC, class KEY>
void order_chunk(wtg_ctx* ctx, const QCols& in, const KEY& key, uint64_t m, const QOrder& o) {
  const dim3 g((unsigned)wtg_ceil_div(m, QO_TILE)), b(QO_THREADS);
  WTG_LAUNCH(ctx, "order_split", k_order_split<KEY>, dim3(QO_SAMPLE / 16), dim3(256), 0, key, m, o);
  WTG_LAUNCH(ctx, "order_count", k_order_count<KEY>, g, b, 0, key, m, o);
  WTG_LAUNCH(ctx, "order_put", (k_order_put<NC, KEY>), g, b, 0, in, key, m, o);
}

}  // namespace
