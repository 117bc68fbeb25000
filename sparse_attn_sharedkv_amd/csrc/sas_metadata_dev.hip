// On-device scheduler: the algorithm of sas_metadata_build (sas_metadata.cpp),
// run by one workgroup on the GPU from device-resident sequence lengths, with
// the same output word for word. A call then needs no host synchronisation:
// the lengths never leave the GPU, and a caller can capture scheduler,
// attention and merge in one HIP graph.
//
// Work split: the per-batch prefix, slot numbers and merge-row numbers are
// block-wide scans; block counts and per-core costs are one item / core per
// thread. The greedy fills are what the time goes into (one after another they
// are a serial walk over the items): a fill walks runs of equal items, not
// items, so its length is about the cores plus the runs; the budget search
// evaluates every candidate it may need in one walk, a budget per lane (the
// doubling search, the first levels of the bisection tree that follows it, and
// the fill of whole items), then one thread replays the host's exact path
// through the results; every lane leaves checkpoints of its walk, from which the
// chosen fill's cursors are recorded by as many lanes at once; and costs below
// 2^20 blocks are walked in floats (a step is a serial chain of about 20 operations
// and costs some 300 clocks, so the chain's length is what counts). FA and FD rows
// are written one core per thread. Measured on MI355X (rebuild, us; before: a
// walk over the items in 64 bits, four to five walks one after another):
//   64 x 1 rows, 128 heads, top-k 2048   141 -> 38      23 sequences, 640 ragged rows  281 -> 56
//   8192 prefill rows, window          3354 -> 128     2000 x 1 ragged rows           924 -> 238
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <type_traits>

#include "../../include/sas_mi355x.h"
#include "sas_items.h"

namespace sas {
void set_error(const std::string& msg);
}

namespace sasdev {

constexpr int NT = 1024;            // threads of the scheduling workgroup
constexpr int NWAVE = NT / 64;
constexpr int BWAVES = 3;           // waves evaluating budgets
constexpr int BLANES = 64 * BWAVES;
constexpr int BLEVELS = 7;          // bisection levels of a round: 127 lanes
constexpr int WHOLE_LANE = 63;      // of the first round: the fill of whole items
constexpr int NCK = 24;             // checkpoints of a walk
constexpr int64_t NO_SPLIT = INT64_MAX / 4;
constexpr int64_t SPLIT_PENALTY = 3;  // same rule and constant as the host scheduler

struct Cursor {
  int32_t i;  // item index
  int32_t j;  // first block not yet assigned inside item i
};

// The items as runs of consecutive items of equal block count: run k holds items
// start[k] .. start[k + 1] - 1, each of nblk[start[k]] blocks.
struct Runs {
  const uint16_t* start;  // [num + 1]
  const int32_t* nblk;    // per item
  int num;
};

// Every lane's state each `stride` steps of a walk (the wave's steps, so a state's
// run is the same in every lane of it): what recording a fill restarts from.
struct Checkpoints {
  uint32_t at[NCK][BLANES];  // items left in the run | cores << 16
  int32_t room[NCK][BLANES];
  uint16_t run[NCK][BWAVES];
  uint16_t num[BWAVES];
};

// Costs below SMALL are walked in floats, which hold them and their sums and
// differences exactly: a step is a serial chain, and the float forms of its two
// floored quotients are the shortest.
constexpr int64_t SMALL = 1 << 20;
// 1 / d, at most 2^-20.4 of it too small: x * inv_of(d) for 0 <= x < SMALL is then
// never above the quotient and less than one below it
__device__ inline float inv_of(float d) { return __builtin_amdgcn_rcpf(d) * (1.0f - 0x1p-21f); }
__device__ inline float floor_div(float x, float d, float inv) {
  const float q = __builtin_floorf(x * inv);
  return __builtin_fmaf(-q, d, x) >= d ? q + 1.0f : q;
}
__device__ inline int64_t inv_of(int64_t) { return 0; }
__device__ inline int64_t floor_div(int64_t x, int64_t d, int64_t) { return x / d; }
__device__ inline float less(float x, float k, float d) { return __builtin_fmaf(-k, d, x); }
__device__ inline int64_t less(int64_t x, int64_t k, int64_t d) { return x - k * d; }

// One lane's greedy fill (sas_metadata.cpp), run by run, under its own budget b and
// shortest piece ms. `room` is what the open core's budget has left, -1 when no
// core is open. A step: items that fit the open core go into it together; the item
// after them closes it, taking `room` less the item cost of its blocks when both
// parts keep >= ms; the rest L goes to fresh cores: ks of them take
// T = max(b - c, ms) blocks and close, while at least T + ms blocks are left, and
// one takes the remainder, staying open when it fits the budget (ks is 0 when the
// first one does) and closing otherwise. The step is select-only: with a budget
// per lane some lane takes each side of every condition, and branches would only
// add their latency to a serial walk.
template <typename V>
struct Filler {
  V c, ms, bc, T, t_inv;
  V room = -1, cores = 0, left = 0;

  __device__ Filler(V c_, V b, V ms_) : c(c_), ms(ms_), bc(b - c_), T(bc > ms_ ? bc : ms_) {
    t_inv = inv_of(T);
  }
  // FIT: whole items may fit an open core (need <= b); BIG: an item may need
  // several fresh ones (nb > b - c). on_act(L0, ks, L): the step closes a core.
  template <bool FIT, bool BIG, typename F>
  __device__ inline void step(V nb, V need, V need_inv, F&& on_act) {
    if constexpr (FIT) {
      const V fit = floor_div(room > 0 ? room : (V)0, need, need_inv);
      const V t = fit < left ? fit : left;
      room = less(room, t, need);
      left -= t;
    }
    const bool act = left > 0;
    const V r = room - c, x = nb - r;
    const V L0 = (r < x ? r : x) >= ms ? x : nb;
    V ks = 0, L = L0;
    if constexpr (BIG) {
      ks = floor_div(L0 > ms ? L0 - ms : (V)0, T, t_inv);
      L = less(L0, ks, T);
    }
    on_act(act, L0, ks, L);
    const V rest = bc - L;
    cores += act ? ks + 1 : (V)0;
    left -= act ? (V)1 : (V)0;
    room = act ? (BIG && rest < 0 ? (V)-1 : rest) : room;
  }
};

// The number of cores of the lane's fill, counted until it exceeds `stop_after`.
template <typename V>
__device__ int greedy_fill(const Runs& rn, int64_t c, int64_t b, int64_t ms, int stop_after,
                           Checkpoints& ck, int stride) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  Filler<V> f((V)c, (V)b, (V)ms);
  const V stop = (V)stop_after;
  int nck = 0, due = 0;
  auto none = [](bool, V, V, V) {};
  for (int k0 = 0; k0 < rn.num; k0 += 64) {
    const int kk = k0 + lane < rn.num ? k0 + lane : rn.num - 1;
    const int my_start = rn.start[kk], my_end = rn.start[kk + 1];
    const int my_nb = rn.nblk[my_start];
    const int lim = rn.num - k0 < 64 ? rn.num - k0 : 64;
    for (int k = 0; k < lim; ++k) {
      const V nb = (V)__builtin_amdgcn_readlane(my_nb, k);
      const V need = f.c + nb;
      const V need_inv = inv_of(need);
      f.left = f.cores > stop ? (V)0
                              : (V)(__builtin_amdgcn_readlane(my_end, k) -
                                    __builtin_amdgcn_readlane(my_start, k));
      const bool fit = __ballot(nb <= f.bc) != 0, big = __ballot(nb > f.bc) != 0;
      auto walk = [&](auto with_fit, auto with_big) {
        while (__ballot(f.left > 0) != 0) {
          if (due-- == 0) {
            // (64-bit walks restart from their beginning)
            if (nck < (__is_same(V, float) ? NCK : 1)) {
              ck.at[nck][threadIdx.x] =
                  (uint32_t)(int)f.left | ((uint32_t)(f.cores > stop ? stop + 1 : f.cores) << 16);
              ck.room[nck][threadIdx.x] = (int32_t)f.room;
              if (lane == 0) ck.run[nck][wid] = (uint16_t)(k0 + k);
              ++nck;
            }
            due = stride - 1;
          }
          f.template step<decltype(with_fit)::value, decltype(with_big)::value>(nb, need, need_inv,
                                                                                none);
          f.left = f.cores > stop ? (V)0 : f.left;
        }
      };
      if (!big) walk(std::true_type{}, std::false_type{});
      else if (!fit) walk(std::false_type{}, std::true_type{});
      else walk(std::true_type{}, std::true_type{});
    }
  }
  if (lane == 0) ck.num[wid] = (uint16_t)nck;
  return f.cores > stop ? stop_after + 1 : (int)f.cores;
}

// The end cursors of the fill that lane `who` of the workgroup counted (at most
// SAS_AIC_CORE_NUM cores): lane l of a wave walks from checkpoint l to the next.
template <typename V>
__device__ void record_fill(const Runs& rn, int64_t c, int64_t b, int64_t ms, int who,
                            const Checkpoints& ck, Cursor* ends) {
  const int lane = threadIdx.x & 63, nck = ck.num[who >> 6];
  if (lane >= nck) return;
  Filler<V> f((V)c, (V)b, (V)ms);
  auto item_at = [&](int l) {  // the next item of checkpoint l
    return rn.start[ck.run[l][who >> 6] + 1] - (int)(ck.at[l][who] & 0xFFFFu);
  };
  const int n = rn.start[rn.num];
  const int until = lane + 1 < nck ? item_at(lane + 1) : n;
  int k = ck.run[lane][who >> 6];
  f.left = (V)(int)(ck.at[lane][who] & 0xFFFFu);
  f.cores = (V)(int)(ck.at[lane][who] >> 16);
  f.room = (V)ck.room[lane][who];
  int end = rn.start[k + 1];
  auto record = [&](V core, int i, V j) {
    if (core <= (V)SAS_AIC_CORE_NUM) ends[(int)core - 1] = Cursor{i, (int32_t)j};
  };
  while (end - (int)f.left < until) {
    if (f.left == 0) {
      ++k;
      f.left = (V)(rn.start[k + 1] - end);
      end = rn.start[k + 1];
    }
    const V nb = (V)rn.nblk[rn.start[k]], need = f.c + nb;
    f.template step<true, true>(nb, need, inv_of(need), [&](bool act, V L0, V ks, V L) {
      if (!act) return;
      const int i = end - (int)f.left;
      if (f.room >= 0) record(f.cores, i, nb - L0);
      for (V q = 1; q <= ks && f.cores + q <= (V)SAS_AIC_CORE_NUM; q += 1)
        record(f.cores + q, i, nb - L0 + q * f.T);
      if (L > f.bc) record(f.cores + 1 + ks, i + 1, 0);
    });
  }
  if (lane == nck - 1 && f.room >= 0) record(f.cores, n, 0);
}

// [lo, hi] of node `node` (heap order, 1 = root) of the bisection tree over
// [lo0, hi0]; false when the path to it ends before.
__device__ inline bool bisect_node(int node, int64_t lo0, int64_t hi0, int64_t* lo, int64_t* hi) {
  int64_t l = lo0, h = hi0;
  for (int d = 30 - __clz(node); d >= 0; --d) {
    if (l >= h) return false;
    const int64_t mid = l + (h - l) / 2;
    if ((node >> d) & 1) l = mid + 1; else h = mid;
  }
  *lo = l;
  *hi = h;
  return l < h;
}

// cost of core c's range [s, e) (sas_metadata.cpp: makespan, one term)
__device__ int64_t core_cost(const int32_t* nblk, int n, int64_t c_item, Cursor s, Cursor e) {
  int64_t cost = 0;
  for (int i = s.i; i < n && (i < e.i || (i == e.i && e.j > 0)); ++i) {
    const int64_t lo = i == s.i ? s.j : 0;
    const int64_t hi = i == e.i ? e.j : nblk[i];
    cost += c_item + (hi - lo);
  }
  return cost;
}

// Exclusive prefix sum of one value per thread over the workgroup (wave scans
// with shuffles, then the sixteen wave totals); *total gets the sum. Two
// barriers; `wsum` is reusable once every thread has returned.
__device__ int64_t block_excl_scan(int64_t v, int64_t* wsum, int64_t* total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int64_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int64_t y = __shfl_up(x, off);
    if (lane >= off) x += y;
  }
  if (lane == 63) wsum[wid] = x;
  __syncthreads();
  if (wid == 0) {
    int64_t t = lane < NWAVE ? wsum[lane] : 0;
#pragma unroll
    for (int off = 1; off < NWAVE; off <<= 1) {
      const int64_t y = __shfl_up(t, off);
      if (lane >= off) t += y;
    }
    if (lane < NWAVE) wsum[NWAVE + lane] = t;  // inclusive wave prefixes
  }
  __syncthreads();
  *total = wsum[2 * NWAVE - 1];
  return (wid > 0 ? wsum[NWAVE + wid - 1] : 0) + x - v;
}

struct Params {
  int32_t* meta;
  const int32_t* act_q;         // [batch] query rows, or null: every batch has uniform_q
  const int32_t* cu_q;          // or [batch + 1] cumulative query rows
  const int32_t* seqused_kv;    // [batch]
  int32_t batch, uniform_q, num_heads, m_base, ori_win_left, scenario, cmp_ratio, cmp_topk;
  int32_t num_cores, s2_base, min_split_blocks, fd_head_chunk;
  int32_t reuse;  // nonzero: a buffer already holding this schedule's key is kept
};

constexpr int BPT = (SAS_DEV_SCHED_MAX_BATCH + NT - 1) / NT;  // batches per thread in the prefix

__global__ __launch_bounds__(NT) void sched_kernel(const Params p) {
  __shared__ int32_t nblk[SAS_DEV_SCHED_MAX_ITEMS];
  __shared__ int32_t istart[SAS_DEV_SCHED_MAX_BATCH + 1];  // first item of each batch
  __shared__ uint16_t run_start[SAS_DEV_SCHED_MAX_ITEMS + 1];
  __shared__ Checkpoints ck;
  __shared__ Cursor ends[SAS_AIC_CORE_NUM];
  __shared__ int16_t ncores[BLANES];  // of the last walk, lane by lane
  __shared__ int64_t wsum[2 * NWAVE];
  __shared__ int64_t s_lo, s_hi, s_total, s_longest, s_span;
  __shared__ int s_err, s_ncore, s_nwhole, s_miss, s_ks, s_win;

  const int tid = threadIdx.x;
  const int wid = tid >> 6;
  int32_t* meta = p.meta;
  int32_t* const cfg = meta + SAS_CFG_OFFSET;
  int32_t* const key = meta + SAS_META_KEY_OFFSET;
  if (tid == 0) {
    s_miss = 0;
    s_err = 0;
    s_total = 0;
    s_longest = 0;
    s_span = 0;
  }
  __syncthreads();

  const int batch = p.batch;
  const int hblocks = (p.num_heads + p.m_base - 1) / p.m_base;
  auto rows_of = [&](int b) {
    return p.cu_q ? p.cu_q[b + 1] - p.cu_q[b] : p.act_q ? p.act_q[b] : p.uniform_q;
  };
  // ---- first item of every batch: thread t owns batches BPT t .. BPT t + BPT - 1 ----
  {
    int64_t cnt[BPT];
    int64_t mine = 0;
#pragma unroll
    for (int e = 0; e < BPT; ++e) {
      const int b = BPT * tid + e;
      cnt[e] = 0;
      if (b < batch) {
        const int aq = rows_of(b), ak = p.seqused_kv[b];
        if (aq < 0 || ak < 0) atomicOr(&s_err, 1);
        cnt[e] = (int64_t)(aq > 0 ? aq : 0) * hblocks;
      }
      mine += cnt[e];
    }
    int64_t total_items;
    int64_t at = block_excl_scan(mine, wsum, &total_items);
#pragma unroll
    for (int e = 0; e < BPT; ++e) {
      const int b = BPT * tid + e;
      if (b < batch) istart[b] = (int32_t)(at < SAS_DEV_SCHED_MAX_ITEMS ? at : SAS_DEV_SCHED_MAX_ITEMS);
      at += cnt[e];
    }
    if (tid == 0) {
      if (total_items > SAS_DEV_SCHED_MAX_ITEMS) atomicOr(&s_err, 2);
      istart[batch] = (int32_t)(total_items < SAS_DEV_SCHED_MAX_ITEMS ? total_items
                                                                      : SAS_DEV_SCHED_MAX_ITEMS);
    }
  }
  __syncthreads();
  if (s_err) {
    if (tid == 0) {
      cfg[0] = 0;  // no magic: refused
      cfg[1] = (s_err & 1) ? -1 : -2;
      key[0] = 0;
    }
    return;
  }
  const int n = istart[batch];
  const int64_t c_item = 1 + ((p.num_heads < p.m_base ? p.num_heads : p.m_base) + 31) / 32;
  auto batch_of = [&](int i) {  // last b with istart[b] <= i
    int lo = 0, hi = batch;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (istart[mid] <= i) lo = mid; else hi = mid;
    }
    return lo;
  };

  // ---- block count of every item (golden item geometry, sas_items.h) ----
  int64_t my_total = 0, my_longest = 0;
  for (int i = tid; i < n; i += NT) {
    const int b = batch_of(i);
    const int s = (i - istart[b]) / hblocks;
    const sas::ItemGeom g = sas::item_geom(rows_of(b), p.seqused_kv[b], s, p.ori_win_left,
                                           p.scenario, p.cmp_ratio, p.cmp_topk);
    const int64_t len = (int64_t)g.n_win + g.n_cmp;
    const int32_t nb = len < (1ll << 31)  // 32-bit division unless it could overflow
                           ? (int32_t)((uint32_t)(len + p.s2_base - 1) / (uint32_t)p.s2_base)
                           : (int32_t)((len + p.s2_base - 1) / p.s2_base);
    nblk[i] = nb;
    my_total += c_item + nb;
    my_longest = my_longest > c_item + nb ? my_longest : c_item + nb;
  }
  // wave sums first: one LDS atomic per wave
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    my_total += __shfl_xor(my_total, off);
    const int64_t o = __shfl_xor(my_longest, off);
    my_longest = my_longest > o ? my_longest : o;
  }
  if ((tid & 63) == 0) {
    atomicAdd((unsigned long long*)&s_total, (unsigned long long)my_total);
    atomicMax((unsigned long long*)&s_longest, (unsigned long long)my_longest);
  }
  __syncthreads();

  // ---- the buffer already holds the schedule of these inputs: keep it ----
  // Only for a buffer its owner declares persistent (p.reuse): one that nothing
  // but this scheduler writes between calls, such as a captured graph's static
  // buffer. A freshly allocated buffer may hold a stale key and config row over
  // rows that something else has since overwritten, so it is always rebuilt.
  const int keyw = 16 + batch + n;  // key words
  const bool keyable = keyw <= SAS_CFG_OFFSET - SAS_META_KEY_OFFSET;
  auto key_word = [&](int w) -> int32_t {
    if (w >= 16 + batch) return nblk[w - 16 - batch];
    if (w >= 16) return rows_of(w - 16);
    const int32_t hdr[16] = {(int32_t)SAS_KEY_MAGIC, n, batch, p.num_heads, p.m_base,
                             p.ori_win_left, p.scenario, p.cmp_ratio, p.cmp_topk, p.num_cores,
                             p.s2_base, p.min_split_blocks, p.fd_head_chunk, 0, 0, 0};
    return hdr[w];
  };
  if (keyable && p.reuse) {
    bool miss = tid == 0 && cfg[0] != SAS_META_MAGIC;
    for (int w = tid; w < keyw; w += NT) miss = miss || key[w] != key_word(w);
    if (miss) s_miss = 1;
    __syncthreads();
    if (!s_miss) return;
  }
  // ---- rebuild: clear everything (vector stores; no memset node when captured) ----
  for (int k = tid; k < SAS_META_SIZE; k += NT) meta[k] = 0;  // rows, key region, config
  __syncthreads();

  int ncore = 1;
  if (n > 0) {
    // ---- runs of equal items: thread t looks at items per t .. per (t + 1) - 1 ----
    const int per = (n + NT - 1) / NT;
    const int i_lo = per * tid < n ? per * tid : n, i_hi = i_lo + per < n ? i_lo + per : n;
    auto starts_run = [&](int i) { return i == 0 || nblk[i] != nblk[i - 1]; };
    int mine = 0;
    for (int i = i_lo; i < i_hi; ++i) mine += starts_run(i);
    int64_t num_runs;
    int at = (int)block_excl_scan(mine, wsum, &num_runs);
    for (int i = i_lo; i < i_hi; ++i)
      if (starts_run(i)) run_start[at++] = (uint16_t)i;
    if (tid == 0) run_start[num_runs] = (uint16_t)n;
    __syncthreads();
    const Runs runs = {run_start, nblk, (int)num_runs};
    // (a budget never exceeds the total of all costs)
    const bool small = s_total < SMALL && p.min_split_blocks < SMALL;
    // One lane's walk has at most a step per run and per core, and the stride spreads the
    // checkpoints over as many; a wave walks each run until its slowest lane is through,
    // so its walk may be longer, and what follows the last checkpoint is recorded from there
    const int steps = runs.num + p.num_cores + 1;
    const int stride = steps > 16 * NCK ? (steps + NCK - 1) / NCK : 16;
    auto clamp_ms = [&](int64_t ms) { return small && ms > SMALL ? SMALL : ms; };
    auto fill = [&](int64_t b, int64_t ms) -> int {
      if (small) return greedy_fill<float>(runs, c_item, b, clamp_ms(ms), p.num_cores, ck, stride);
      return greedy_fill<int64_t>(runs, c_item, b, ms, p.num_cores, ck, stride);
    };
    auto record = [&](int64_t b, int64_t ms, int who) {
      if (small) record_fill<float>(runs, c_item, b, clamp_ms(ms), who, ck, ends);
      else record_fill<int64_t>(runs, c_item, b, ms, who, ck, ends);
    };
    // thread 0: the host's path through evaluated bisection nodes (node 1 is lane
    // `lane0`); s_win is the lane that counted the fill at s_hi
    auto replay = [&](int64_t lo, int64_t hi, int lane0) {
      for (int d = 0, nd = 1; d < BLEVELS && lo < hi; ++d) {
        const int64_t mid = lo + (hi - lo) / 2;
        if (ncores[lane0 + nd - 1] <= p.num_cores) {
          hi = mid;
          s_win = lane0 + nd - 1;
          nd = 2 * nd;
        } else {
          lo = mid + 1;
          nd = 2 * nd + 1;
        }
      }
      s_lo = lo;
      s_hi = hi;
    };

    // ---- smallest budget whose fill fits num_cores (the host's search) ----
    // Doubling search: lane k < 63 of wave 0 evaluates h_k = min(total, h_0 2^k),
    // the last lane the fill of whole items. It mostly ends at h_1, so the waves
    // beside it evaluate the first levels of the bisection of [h_0 + 1, h_1].
    const int64_t h0 = (s_total + p.num_cores - 1) / p.num_cores > 1
                           ? (s_total + p.num_cores - 1) / p.num_cores : 1;
    const int64_t h1 = 2 * h0 < s_total ? 2 * h0 : s_total;
    if (wid < BWAVES) {
      int64_t b = h0, ms = p.min_split_blocks, nlo = 0, nhi = 0;
      if (tid == WHOLE_LANE) {
        b = s_longest;
        ms = NO_SPLIT;
      } else if (wid == 0) {
        for (int k = 0; k < tid && b < s_total; ++k) b = 2 * b < s_total ? 2 * b : s_total;
      } else if (h0 < s_total && tid - 63 < (1 << BLEVELS) &&
                 bisect_node(tid - 63, h0 + 1, h1, &nlo, &nhi)) {
        b = nlo + (nhi - nlo) / 2;
      }
      const int cores = fill(b, ms);
      ncores[tid] = (int16_t)cores;
      if (wid == 0) {
        const bool stop = tid != WHOLE_LANE && (b >= s_total || cores <= p.num_cores);
        const int ks = __ffsll((long long)__ballot(stop)) - 1;  // lane 62 has reached total
        const int64_t hi = __shfl(b, ks);
        const int64_t prev = __shfl(b, ks > 0 ? ks - 1 : 0);
        if (tid == 0) {
          s_lo = ks > 0 ? prev + 1 : 1;
          s_hi = hi;
          s_win = s_ks = ks;
        }
        if (tid == WHOLE_LANE) s_nwhole = cores;
      }
    }
    __syncthreads();
    if (tid == 0 && s_ks == 1) replay(h0 + 1, h1, 64);
    __syncthreads();
    // what is left of [lo, hi], BLEVELS levels a round; then, if the chosen budget
    // was not counted in the last walk, one more walk at it
    const bool more = s_lo < s_hi;
    while (s_lo < s_hi) {
      const int64_t lo = s_lo, hi = s_hi;
      if (wid < BWAVES) {
        int64_t nlo = 0, nhi = 0, b = hi;
        if (tid + 1 < (1 << BLEVELS) && bisect_node(tid + 1, lo, hi, &nlo, &nhi))
          b = nlo + (nhi - nlo) / 2;
        ncores[tid] = (int16_t)fill(b, p.min_split_blocks);
      }
      __syncthreads();
      if (tid == 0) {
        s_win = -1;
        replay(lo, hi, 0);
      }
      __syncthreads();
    }
    // ---- the fill at the chosen budget ----
    // (a walk of its own only when the last one did not count it)
    auto walk_and_record = [&](int64_t b, int64_t ms, int who) {
      if (wid == 0) {
        if (who < 0) ncores[tid] = (int16_t)fill(b, ms);
        record(b, ms, who < 0 ? 0 : who);
        if (tid == 0) s_ncore = ncores[who < 0 ? 0 : who];
      }
      __syncthreads();
    };
    walk_and_record(s_lo, p.min_split_blocks, s_win);
    ncore = s_ncore;
    int64_t my_span = 0;
    for (int c = tid; c < ncore && ncore <= SAS_AIC_CORE_NUM; c += NT) {
      const Cursor s = c == 0 ? Cursor{0, 0} : ends[c - 1];
      const int64_t cost = core_cost(nblk, n, c_item, s, ends[c]);
      my_span = my_span > cost ? my_span : cost;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int64_t o = __shfl_xor(my_span, off);
      my_span = my_span > o ? my_span : o;
    }
    if ((tid & 63) == 0) atomicMax((unsigned long long*)&s_span, (unsigned long long)my_span);
    __syncthreads();
    if (s_longest <= s_span + SPLIT_PENALTY && s_nwhole <= p.num_cores)
      walk_and_record(s_longest, NO_SPLIT, more || s_win < 0 ? -1 : WHOLE_LANE);
    ncore = s_ncore;
    if (ncore > p.num_cores) {
      if (tid == 0) cfg[1] = -3;  // over capacity
      return;
    }
  } else if (tid == 0) {
    ends[0] = Cursor{0, 0};
  }
  __syncthreads();

  // ---- FA rows (one core per thread) and partial slots ----
  // A piece is partial iff it is the first piece of a core that starts inside
  // an item or the last one of a core that ends inside one; the host numbers
  // them in core order, first before last. An item is split iff it owns such
  // a piece, and its first piece is the "last" partial piece of some core.
  auto put_cursor = [&](int32_t* row, Cursor c) {
    if (c.i < n) {
      const int b = batch_of(c.i);
      row[0] = b;
      row[1] = c.i - istart[b];  // m = query row * head blocks + head block
      row[2] = c.j;
    } else {
      row[0] = batch;
      row[1] = 0;
      row[2] = 0;
    }
  };
  const int c = tid;  // ncore <= SAS_AIC_CORE_NUM < NT
  Cursor cs{0, 0}, ce{0, 0};
  bool first_partial = false, last_partial = false;
  if (c < ncore) {
    cs = c == 0 ? Cursor{0, 0} : ends[c - 1];
    ce = ends[c];
    first_partial = cs.j > 0 && cs.i < n;
    last_partial = ce.j > 0 && ce.i < n && !(first_partial && ce.i == cs.i);
  }
  int64_t slots_total, split_total;
  const int64_t slot_base =
      block_excl_scan((first_partial ? 1 : 0) + (last_partial ? 1 : 0), wsum, &slots_total);
  __syncthreads();  // wsum reused
  const int64_t split_before = block_excl_scan(last_partial ? 1 : 0, wsum, &split_total);
  if (c < ncore) {
    int32_t* row = meta + c * SAS_FA_METADATA_SIZE;
    row[0] = 1;
    if (c == 0) {
      row[1] = row[2] = row[3] = 0;  // core 0 starts at the origin (metadata.py:985-987)
    } else {
      put_cursor(row + 1, cs);
    }
    put_cursor(row + 4, ce);
    row[7] = (int32_t)slot_base;
  }
  // ---- FD rows: the split items in order, each in head chunks ----
  const int mb_heads = p.num_heads < p.m_base ? p.num_heads : p.m_base;
  int chunk = p.fd_head_chunk < mb_heads ? p.fd_head_chunk : mb_heads;
  if (chunk < 1) chunk = 1;
  while (split_total * ((mb_heads + chunk - 1) / chunk) > SAS_AIV_CORE_NUM && chunk < mb_heads)
    chunk = 2 * chunk < mb_heads ? 2 * chunk : mb_heads;
  const int per_item = (mb_heads + chunk - 1) / chunk;
  const int64_t nfd = split_total * per_item;
  if (nfd > SAS_AIV_CORE_NUM) {
    if (tid == 0) cfg[1] = -3;
    return;
  }
  if (last_partial) {
    const int i = ce.i;
    int c2 = c + 1;  // cores wholly inside item i, then the one with its last piece
    while (ends[c2].i == i && ends[c2].j > 0) ++c2;
    const int32_t first_slot = (int32_t)slot_base + (first_partial ? 1 : 0);
    const int b = batch_of(i);
    int k = (int)split_before * per_item;
    for (int h0 = 0; h0 < mb_heads; h0 += chunk, ++k) {
      int32_t* row = meta + SAS_FD_OFFSET + k * SAS_FD_METADATA_SIZE;
      row[0] = 1;
      row[1] = b;
      row[2] = i - istart[b];
      row[3] = first_slot;
      row[4] = c2 - c + 1;
      row[5] = h0;
      row[6] = chunk < mb_heads - h0 ? chunk : mb_heads - h0;
    }
  }
  if (keyable)
    for (int w = tid; w < keyw; w += NT) key[w] = key_word(w);
  if (tid == 0) {
    cfg[1] = p.s2_base;
    cfg[2] = ncore;
    cfg[3] = (int32_t)nfd;
    cfg[4] = (int32_t)slots_total;
    cfg[5] = p.num_heads;
    cfg[6] = p.m_base;
    cfg[7] = n;
    cfg[0] = SAS_META_MAGIC;
  }
}

}  // namespace sasdev

static int build_device(int32_t* meta, int batch, const int32_t* act_q, const int32_t* cu_q,
                        int uniform_q, const int32_t* seqused_kv, int num_heads, int m_base,
                        int ori_win_left, int scenario, int cmp_ratio, int cmp_topk, int num_cores,
                        int s2_base, int min_split_blocks, int fd_head_chunk, int reuse,
                        void* stream) {
  if (!meta || batch < 0 || batch > SAS_DEV_SCHED_MAX_BATCH || (batch > 0 && !seqused_kv) ||
      (!act_q && !cu_q && uniform_q < 0)) {
    sas::set_error("sas_metadata_build_device: null pointer or batch out of range");
    return SAS_E_INVALID;
  }
  if (num_heads < 1 || num_heads > 4096 || m_base < 1 || m_base > 4096 || scenario < 1 ||
      scenario > 3 || (scenario >= 2 && cmp_ratio < 1) || cmp_topk < 0 || num_cores < 1 ||
      num_cores > SAS_AIC_CORE_NUM || s2_base < 32 || s2_base % 32 != 0 ||
      min_split_blocks < 1 || fd_head_chunk < 1 || ori_win_left < -1) {
    sas::set_error("sas_metadata_build_device: argument out of range");
    return SAS_E_INVALID;
  }
  sasdev::Params p;
  p.meta = meta;
  p.act_q = act_q;
  p.cu_q = cu_q;
  p.seqused_kv = seqused_kv;
  p.batch = batch;
  p.uniform_q = uniform_q;
  p.num_heads = num_heads;
  p.m_base = m_base;
  p.ori_win_left = ori_win_left;
  p.scenario = scenario;
  p.cmp_ratio = cmp_ratio;
  p.cmp_topk = cmp_topk;
  p.num_cores = num_cores;
  p.s2_base = s2_base;
  p.min_split_blocks = min_split_blocks;
  p.fd_head_chunk = fd_head_chunk;
  p.reuse = reuse != 0;
  hipLaunchKernelGGL(sasdev::sched_kernel, dim3(1), dim3(sasdev::NT), 0, (hipStream_t)stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    sas::set_error(std::string("sas_metadata_build_device: ") + hipGetErrorString(e));
    return SAS_E_HIP;
  }
  return SAS_OK;
}

extern "C" int sas_metadata_build_device(int32_t* meta, int batch, const int32_t* act_q,
                                         int uniform_q, const int32_t* seqused_kv, int num_heads,
                                         int m_base, int ori_win_left, int scenario, int cmp_ratio,
                                         int cmp_topk, int num_cores, int s2_base,
                                         int min_split_blocks, int fd_head_chunk, int reuse,
                                         void* stream) {
  return build_device(meta, batch, act_q, nullptr, uniform_q, seqused_kv, num_heads, m_base,
                      ori_win_left, scenario, cmp_ratio, cmp_topk, num_cores, s2_base,
                      min_split_blocks, fd_head_chunk, reuse, stream);
}

extern "C" int sas_metadata_build_device_cu(int32_t* meta, int batch, const int32_t* cu_q,
                                            const int32_t* seqused_kv, int num_heads, int m_base,
                                            int ori_win_left, int scenario, int cmp_ratio,
                                            int cmp_topk, int num_cores, int s2_base,
                                            int min_split_blocks, int fd_head_chunk, int reuse,
                                            void* stream) {
  return build_device(meta, batch, nullptr, cu_q, -1, seqused_kv, num_heads, m_base, ori_win_left,
                      scenario, cmp_ratio, cmp_topk, num_cores, s2_base, min_split_blocks,
                      fd_head_chunk, reuse, stream);
}
