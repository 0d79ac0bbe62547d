// Routing refresh for gfx950: one workgroup per (batch, head).
//
// Restates tao_stream.py:310-357 with _topk_oldest (:50-53):
//   h    = r(softmax_D(raw_q))                 (anchor query row)
//   hv_p = r(h * pw[p])                        (page weights of the epoch)
//   page mass = r(sum_D hv_p) over completed pages; stable top-`coarse`
//   pages (descending, lowest index wins ties), re-sorted ascending;
//   candidates = 8 fines of each chosen page + every pending fine;
//   mass_j = r(sum_D r(hv_page(j) * sw_j)); stable top-M candidates kept in
//   score order.
// Every fp32 sum uses the butterfly order of the oracle (wave_fold_sum: DPP
// on the bit-reversed channel layout), so selected ids are bit-identical to
// the oracle's. Selection: 64-bit keys (monotone bf16 score
// << 32 | ~index) ranked by counting (<= 512 keys) or an LDS bitonic network.
// Eight waves issue the loads of eight rows each before reducing them, so a
// refresh costs a few memory latencies rather than one per row.
#include "route_lds.h"
#include "tao_launch.h"
#include "tao_common.h"

namespace tao {
namespace {

constexpr int kMaxSort = 2048;   // pages or candidates per head

template <int D>
struct RouteSmem {
  float h[D];
  unsigned long long keys[kMaxSort];
  int cand_id[kMaxSort];
  int cand_page[kMaxSort];
  int chosen[kMaxSort / 8];
};

TAO_DEV unsigned long long score_key(float score_bf, int index) {
  bf16_t bits = f2bf(score_bf);
  if (bits == 0x8000) bits = 0;      // -0 ties with +0, as in torch's sort
  const uint32_t hi = bf16_order_key(bits);
  return ((unsigned long long)hi << 32) | (unsigned long long)(0xFFFFFFFFu - (uint32_t)index);
}

TAO_DEV int key_index(unsigned long long key) {
  return (int)(0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFull));
}

constexpr int kRouteThreads = 512;   // 8 waves
constexpr int kWaves = kRouteThreads / 64;
constexpr int kBatch = 8;            // rows whose loads one wave issues together
constexpr int kRefreshThreads = 1024;   // the refresh: 16 waves per (batch, head)
constexpr int kRefreshWaves = kRefreshThreads / 64;
constexpr int kRefreshRowsPerWave = 5;   // staged rows one refresh wave reduces together
constexpr int kRankMax = 512;        // rank-count selection up to this many keys

// Masses of up to kBatch rows per wave: every lane loads its two (or one)
// channels of all rows first, then each row is reduced in butterfly order:
// r(sum_D r(h * pw[page]) [* sw[id]]).
// Segment-weight rows: fines below `split` read the state's final weights,
// later (pending) fines read the epoch's pool rows.
struct SwRows {
  const bf16_t* lo; const bf16_t* hi; int split;
  TAO_DEV const bf16_t* row(int id, int D) const {
    return id < split ? lo + (size_t)id * D : hi + (size_t)(id - split) * D;
  }
};

template <int D>
TAO_DEV void wave_masses(const float* h, const bf16_t* pw, const SwRows* sw,
                         const int* pages, const int* ids, int count, int lane,
                         float* out) {
  constexpr int PER = D / 64;
  const int e0 = fold_lane(lane);      // channels e0 + 64 k (bit-reversed layout)
  bf16_t pv[kBatch][PER], sv[kBatch][PER];
#pragma unroll
  for (int r = 0; r < kBatch; ++r) {
    if (r < count) {
      const bf16_t* srow = sw ? sw->row(ids[r], D) : nullptr;
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        pv[r][k] = pw[(size_t)pages[r] * D + e0 + 64 * k];
        sv[r][k] = sw ? srow[e0 + 64 * k] : (bf16_t)0;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kBatch; ++r) {
    if (r < count) {
      float v[PER];
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const float hv = rbf(h[e0 + 64 * k] * bf2f(pv[r][k]));
        v[k] = sw ? rbf(hv * bf2f(sv[r][k])) : hv;
      }
      float s = v[0];
#pragma unroll
      for (int k = 1; k < PER; ++k) s += v[k];
      out[r] = rbf(wave_fold_sum(s));
    }
  }
}

// h = r(softmax_D(raw_q row)) of one query by one wave: fp32 exp correctly
// rounded, butterfly sum (tao_stream.py:253-254).
template <int D>
TAO_DEV void query_weights(const bf16_t* rq, int lane, float* h) {
  constexpr int PER = D / 64;
  const int e0 = fold_lane(lane);      // channels e0 + 64 k (bit-reversed layout)
  float x[PER], e[PER];
  float mx = -__builtin_inff();
#pragma unroll
  for (int k = 0; k < PER; ++k) { x[k] = bf2f(rq[e0 + 64 * k]); mx = fmaxf(mx, x[k]); }
  mx = wave_fold_max(mx);
#pragma unroll
  for (int k = 0; k < PER; ++k) e[k] = exp_cr(x[k] - mx);
  float s = e[0];
#pragma unroll
  for (int k = 1; k < PER; ++k) s += e[k];
  s = wave_fold_sum(s);
#pragma unroll
  for (int k = 0; k < PER; ++k) h[e0 + 64 * k] = rbf(e[k] / s);
}

// Number of keys larger than `mine` among keys[0, n) (keys are unique).
TAO_DEV int key_rank(const unsigned long long* keys, int n, unsigned long long mine) {
  int r = 0;
  int j = 0;
  for (; j + 8 <= n; j += 8) {
    unsigned long long k8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) k8[i] = keys[j + i];
#pragma unroll
    for (int i = 0; i < 8; ++i) r += k8[i] > mine;
  }
  for (; j < n; ++j) r += keys[j] > mine;
  return r;
}

// Stable descending selection of the top `count` keys (unique 64-bit keys:
// score << 32 | ~index) by a workgroup of NT threads. Writes the selected
// keys, best first, to dst.
template <int NT>
TAO_DEV void select_top_n(unsigned long long* keys, int n, int count, unsigned long long* dst) {
  if (n <= 2 * NT / 8) {
    // T lanes per key (8 for n <= NT / 8, else 4): lane part p counts the
    // larger keys among keys p, p + T, ... (four reads in flight at a time;
    // 0 is below every key); DPP adds the T parts.
    const int T = n <= NT / 8 ? 8 : 4;
    const int i = threadIdx.x / T, part = threadIdx.x % T;
    const unsigned long long mine = keys[min(i, n - 1)];
    int cnt = 0;
    for (int j0 = part; j0 < n; j0 += 4 * T) {
      unsigned long long k4[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) k4[u] = j0 + u * T < n ? keys[j0 + u * T] : 0ull;
#pragma unroll
      for (int u = 0; u < 4; ++u) cnt += k4[u] > mine;
    }
    cnt += __builtin_amdgcn_update_dpp(0, cnt, 0xB1, 0xF, 0xF, false);
    cnt += __builtin_amdgcn_update_dpp(0, cnt, 0x4E, 0xF, 0xF, false);
    if (T == 8) cnt += __builtin_amdgcn_update_dpp(0, cnt, 0x141, 0xF, 0xF, false);
    if (i < n && part == 0 && cnt < count) dst[cnt] = mine;
    __syncthreads();
    return;
  }
  if (n <= kRankMax) {
    for (int i = threadIdx.x; i < n; i += NT) {
      const unsigned long long mine = keys[i];
      const int rank = key_rank(keys, n, mine);
      if (rank < count) dst[rank] = mine;
    }
    __syncthreads();
    return;
  }
  int np = 1;
  while (np < n) np <<= 1;
  for (int i = n + threadIdx.x; i < np; i += NT) keys[i] = 0ull;
  __syncthreads();
  for (int k = 2; k <= np; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < np; i += NT) {
        const int ixj = i ^ j;
        if (ixj > i) {
          const unsigned long long a = keys[i], b = keys[ixj];
          const bool desc = (i & k) == 0;
          if (desc ? (a < b) : (a > b)) { keys[i] = b; keys[ixj] = a; }
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < count; i += NT) dst[i] = keys[i];
  __syncthreads();
}

TAO_DEV void select_top(unsigned long long* keys, int n, int count, unsigned long long* dst) {
  select_top_n<kRouteThreads>(keys, n, count, dst);
}

template <int D>
__global__ __launch_bounds__(kRouteThreads) void route_kernel(RouteParams p) {
  __shared__ RouteSmem<D> sm;
  __shared__ unsigned long long top[kMaxSort];
  if (gate_closed(p.gate)) return;   // uniform: every thread reads one header word
  constexpr int PER = D / 64;
  const int BH = p.B * p.H;
  const int bh = blockIdx.x % BH;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Turn description (single-turn mode: the state's current epoch).
  long long anchor = 0;
  int K = p.completed, pending = p.pending, coarse = p.coarse, selected = p.selected;
  int write_state = 1;
  int32_t* sel_out = p.sel + (size_t)bh * p.sel_cap;
  const bf16_t* pw = p.pw + (size_t)bh * p.page_cap * D;
  SwRows swr{p.sw + (size_t)bh * p.fine_cap * D, nullptr, 0x7FFFFFFF};
  if (p.turns) {
    const int64_t* t = p.turns + 8 * (blockIdx.x / BH);
    anchor = t[0];
    const int erel = (int)t[1];
    K = (int)t[2]; pending = (int)t[3]; coarse = (int)t[4]; selected = (int)t[5];
    sel_out = p.sel_pool + ((size_t)t[6] * BH + bh) * p.sel_cap;
    write_state = (int)t[7];
    pw = p.pw_pool + ((size_t)erel * BH + bh) * p.pool_pcap * D;
    swr.hi = p.psw_pool + ((size_t)erel * BH + bh) * 8 * D;
    swr.split = K * p.group;
  }

  if (wave == 0) query_weights<D>(p.rq + b * p.rq_sb + anchor * p.rq_st + h * p.rq_sh, lane, sm.h);
  __syncthreads();

  // ---- coarse pages: stable top-`coarse` by page mass, then ascending.
  if (coarse > 0) {
    for (int base = wave * kBatch; base < K; base += kWaves * kBatch) {
      int pages[kBatch];
      float mass[kBatch];
      const int count = min(kBatch, K - base);
#pragma unroll
      for (int r = 0; r < kBatch; ++r) pages[r] = base + min(r, count - 1);
      wave_masses<D>(sm.h, pw, nullptr, pages, pages, count, lane, mass);
      if (lane < count) {
        float mine = mass[0];
#pragma unroll
        for (int r = 1; r < kBatch; ++r) if (lane == r) mine = mass[r];
        sm.keys[base + lane] = score_key(mine, base + lane);
      }
    }
    __syncthreads();
    select_top(sm.keys, K, coarse, top);
    if (tid < coarse) {
      const int mine = key_index(top[tid]);
      int rank = 0;
      for (int j = 0; j < coarse; ++j) rank += key_index(top[j]) < mine;
      sm.chosen[rank] = mine;
    }
    __syncthreads();
  }

  // ---- candidates: 8 fines of each chosen page, then the pending fines.
  const int group = p.group;
  const int E = group * coarse + pending;
  for (int j = tid; j < E; j += kRouteThreads) {
    int page, id;
    if (j < group * coarse) {
      page = sm.chosen[j / group];
      id = page * group + j % group;
    } else {
      page = K;
      id = K * group + (j - group * coarse);
    }
    sm.cand_page[j] = page;
    sm.cand_id[j] = id;
  }
  __syncthreads();
  for (int base = wave * kBatch; base < E; base += kWaves * kBatch) {
    int pages[kBatch], ids[kBatch];
    float mass[kBatch];
    const int count = min(kBatch, E - base);
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      const int j = base + min(r, count - 1);
      pages[r] = sm.cand_page[j];
      ids[r] = sm.cand_id[j];
    }
    wave_masses<D>(sm.h, pw, &swr, pages, ids, count, lane, mass);
    if (lane < count) {
      float mine = mass[0];
#pragma unroll
      for (int r = 1; r < kBatch; ++r) if (lane == r) mine = mass[r];
      sm.keys[base + lane] = score_key(mine, base + lane);
    }
  }
  __syncthreads();
  select_top(sm.keys, E, selected, top);
  for (int m = tid; m < selected; m += kRouteThreads) {
    const int id = sm.cand_id[key_index(top[m])];
    sel_out[m] = id;
    if (write_state && p.turns) p.sel[(size_t)bh * p.sel_cap + m] = id;
  }
  if (write_state)
    for (int i = tid; i < coarse; i += kRouteThreads)
      p.chosen[(size_t)bh * p.chosen_cap + i] = sm.chosen[i];
  if (write_state && bh == 0 && tid == 0) p.header[1] = selected;
}

// ---------------------------------------------------------------------------
// Single-turn refresh of a stream (the decode driver's route turns) with its
// rows staged in LDS: the same arithmetic, candidate order, butterfly sums
// and stable selections as route_kernel, but every row is fetched with
// coalesced 16-byte loads into LDS, so a refresh costs two memory round
// trips: (1) the page weights of the completed and pending pages, the
// pending fines' segment weights and the anchor query; (2) the segment
// weights of the chosen pages' fines. Serves states with at most
// kRefreshPages pages and kRefreshRows candidates; route_kernel serves the
// rest.
constexpr int kRefreshPages = 128;
constexpr int kRefreshRows = 128;

template <int D>
struct RefreshSmem {
  bf16_t pw[kRefreshPages][D];         // page weights, completed then pending page
  bf16_t sw[kRefreshRows][D];          // segment weights of the candidates, in order
  float h[D];
  unsigned long long keys[kRefreshRows];
  unsigned long long top[kRefreshRows];
  int chosen[kRefreshRows / 8 + 1];
};

// Masses of kBatch staged rows on one wave (bit-reversed channel layout,
// the butterfly sum of wave_masses): r(sum_D r(h * pw_row) [* sw_row]).
// The rows' reductions are independent and unrolled, so their latencies
// overlap. Rows past `count` (wave-uniform) give 0 and are not used; this
// wave's lane r < count receives row r's mass.
template <int D, int NB>
TAO_DEV float staged_masses(const float* h, const bf16_t* const* pw_rows,
                            const bf16_t* const* sw_rows, int count, int lane) {
  constexpr int PER = D / 64;
  const int e0 = fold_lane(lane);
  float hq[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) hq[k] = h[e0 + 64 * k];
  // Rows past `count` repeat the last row (callers clamp), so every read is
  // unconditional and the reads of all rows are in flight together.
  bf16_t pv[NB][PER], sv[NB][PER];
#pragma unroll
  for (int r = 0; r < NB; ++r)
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      pv[r][k] = pw_rows[r][e0 + 64 * k];
      sv[r][k] = sw_rows ? sw_rows[r][e0 + 64 * k] : (bf16_t)0;
    }
  float part[NB];
#pragma unroll
  for (int r = 0; r < NB; ++r) {
    float v[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const float hv = rbf(hq[k] * bf2f(pv[r][k]));
      v[k] = sw_rows ? rbf(hv * bf2f(sv[r][k])) : hv;
    }
    float s = v[0];
#pragma unroll
    for (int k = 1; k < PER; ++k) s += v[k];
    part[r] = s;
  }
  wave_fold_sum_n<NB>(part);
  float mine = 0.0f;
#pragma unroll
  for (int r = 0; r < NB; ++r)
    if (lane == r) mine = rbf(part[r]);
  (void)count;
  return mine;
}

// The refresh's selection for (batch, head) bh by a workgroup of NT
// threads: the route of RouteParams' single turn, left in LDS (sm.top: the
// selected candidates' keys, best first; sm.chosen: the chosen pages,
// ascending; sm.pw / sm.sw: the page weights and the candidates' segment
// weights). Each mass is a butterfly sum inside one wave, so the result does
// not depend on NT. With `write_out` the selection is also stored in the
// state (sel, chosen; header[1] by head 0).
template <int D, int NT>
TAO_DEV void refresh_select(const RouteParams& p, int bh, RefreshSmem<D>& sm, bool write_out) {
  constexpr int C16 = D / 8;            // 16-byte chunks per row
  constexpr int NW = NT / 64;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int K = p.completed, pending = p.pending, coarse = p.coarse, selected = p.selected;
  constexpr int group = 8;          // coarse_group (checked at launch)
  const int P = K + (pending > 0 ? 1 : 0);
  const int E = group * coarse + pending;
  const bf16_t* pw = p.pw + (size_t)bh * p.page_cap * D;
  const bf16_t* sw = p.sw + (size_t)bh * p.fine_cap * D;
  // ---- round trip 1: page weights, pending segment weights, anchor query
  // (every load issued before any store to LDS)
  constexpr int PW_PT = (kRefreshPages * C16 + NT - 1) / NT;
  constexpr int SW_PT = (kRefreshRows * C16 + NT - 1) / NT;
  constexpr int PD_PT = (8 * C16 + NT - 1) / NT;   // pending fines: fewer than 8 rows
  // Loads are unconditional (indices clamped to a valid row) so the
  // scheduler can issue them all before the guarded LDS stores.
  uint4 pwv[PW_PT], pdv[PD_PT];
#pragma unroll
  for (int k = 0; k < PW_PT; ++k) {
    const int ic = min(tid + k * NT, P * C16 - 1);
    pwv[k] = *(const uint4*)(pw + (size_t)(ic / C16) * D + (ic % C16) * 8);
  }
  if (pending > 0) {
#pragma unroll
    for (int k = 0; k < PD_PT; ++k) {
      const int ic = min(tid + k * NT, pending * C16 - 1);
      pdv[k] = *(const uint4*)(sw + (size_t)(K * group + ic / C16) * D + (ic % C16) * 8);
    }
  }
#pragma unroll
  for (int k = 0; k < PW_PT; ++k) {
    const int i = tid + k * NT;
    if (i < P * C16) *(uint4*)&sm.pw[i / C16][(i % C16) * 8] = pwv[k];
  }
  if (pending > 0) {
#pragma unroll
    for (int k = 0; k < PD_PT; ++k) {
      const int i = tid + k * NT;
      if (i < pending * C16) *(uint4*)&sm.sw[group * coarse + i / C16][(i % C16) * 8] = pdv[k];
    }
  }
  if (wave == 0) query_weights<D>(p.rq + b * p.rq_sb + h * p.rq_sh, lane, sm.h);
  __syncthreads();
  // ---- coarse pages: stable top-`coarse` by page mass, then ascending
  if (coarse > 0) {
    for (int base = wave * kRefreshRowsPerWave; base < K; base += NW * kRefreshRowsPerWave) {
      const int count = min(kRefreshRowsPerWave, K - base);
      const bf16_t* rows[kRefreshRowsPerWave];
#pragma unroll
      for (int r = 0; r < kRefreshRowsPerWave; ++r) rows[r] = sm.pw[base + min(r, count - 1)];
      const float mass = staged_masses<D, kRefreshRowsPerWave>(sm.h, rows, nullptr, count, lane);
      if (lane < count) sm.keys[base + lane] = score_key(mass, base + lane);
    }
    __syncthreads();
    select_top_n<NT>(sm.keys, K, coarse, sm.top);
    if (tid < coarse) {
      const int mine = key_index(sm.top[tid]);
      int rank = 0;
      for (int j = 0; j < coarse; ++j) rank += key_index(sm.top[j]) < mine;
      sm.chosen[rank] = mine;
    }
    __syncthreads();
    // ---- round trip 2: segment weights of the chosen pages' fines
    uint4 swv[SW_PT];
#pragma unroll
    for (int k = 0; k < SW_PT; ++k) {
      const int ic = min(tid + k * NT, group * coarse * C16 - 1);
      const int row = ic / C16;
      const int id = sm.chosen[row / group] * group + row % group;
      swv[k] = *(const uint4*)(sw + (size_t)id * D + (ic % C16) * 8);
    }
#pragma unroll
    for (int k = 0; k < SW_PT; ++k) {
      const int i = tid + k * NT;
      if (i < group * coarse * C16) *(uint4*)&sm.sw[i / C16][(i % C16) * 8] = swv[k];
    }
    __syncthreads();
  }
  // ---- candidate masses: 8 fines of each chosen page, then the pending fines
  for (int base = wave * kRefreshRowsPerWave; base < E; base += NW * kRefreshRowsPerWave) {
    const int count = min(kRefreshRowsPerWave, E - base);
    const bf16_t* prow[kRefreshRowsPerWave];
    const bf16_t* srow[kRefreshRowsPerWave];
#pragma unroll
    for (int r = 0; r < kRefreshRowsPerWave; ++r) {
      const int j = base + min(r, count - 1);
      prow[r] = sm.pw[j < group * coarse ? sm.chosen[j / group] : K];
      srow[r] = sm.sw[j];
    }
    const float mass = staged_masses<D, kRefreshRowsPerWave>(sm.h, prow, srow, count, lane);
    if (lane < count) sm.keys[base + lane] = score_key(mass, base + lane);
  }
  __syncthreads();
  select_top_n<NT>(sm.keys, E, selected, sm.top);
  if (!write_out) return;
  int32_t* sel_out = p.sel + (size_t)bh * p.sel_cap;
  for (int m = tid; m < selected; m += NT) {
    const int j = key_index(sm.top[m]);
    sel_out[m] = j < group * coarse ? sm.chosen[j / group] * group + j % group
                                    : K * group + (j - group * coarse);
  }
  for (int i = tid; i < coarse; i += NT)
    p.chosen[(size_t)bh * p.chosen_cap + i] = sm.chosen[i];
  if (bh == 0 && tid == 0) p.header[1] = selected;
}

template <int D>
__global__ __launch_bounds__(kRefreshThreads) void route_refresh_kernel(RouteParams p) {
  __shared__ RefreshSmem<D> sm;
  if (gate_closed(p.gate)) return;   // uniform: every thread reads one header word
  refresh_select<D, kRefreshThreads>(p, blockIdx.x, sm, true);
}

// Route refresh and fold in one launch: the fold's CHUNKS workgroups of a
// (batch, head) each compute the head's selection (refresh_select on 16
// waves; the same arithmetic gives every workgroup the same route, and
// chunk 0 stores it), then fold their ROWS rows of G^T over the selected
// fines with fold_kernel's arithmetic and order: in slot order m, w_m[d] =
// pw[page(m)][d] * sw[m][d] (from the rows the selection staged in LDS,
// kRefreshFoldStage slots at a time), G^T[e][d] += w_m[d] * C^T_m[e][d] as
// one fp32 FMA, g[d] += w_m[d]. Thread (row, column pair) loads 4 bytes of
// each selected C^T row, so a wave reads one 256-byte row per slot. One
// launch instead of two removes a launch gap and the fold's wait for the
// route kernel's last workgroup.
constexpr int kRefreshFoldStage = 36;

template <int D>
__global__ __launch_bounds__(kRefreshThreads) void refresh_fold_kernel(RouteParams p,
                                                                        FoldParams f) {
  constexpr int NT = kRefreshThreads;
  constexpr int CP = D / 2, ROWS = NT / CP, CHUNKS = D / ROWS, U = kRefreshFoldStage;
  constexpr int group = 8;
  __shared__ RefreshSmem<D> sm;
  __shared__ float wts[U][D];
  __shared__ int slot_id[U];
  if (gate_closed(p.gate)) return;   // uniform: every thread reads one header word
  int bh, e_chunk;
  xcd_unit(blockIdx.x, p.B * p.H, CHUNKS, bh, e_chunk);
  refresh_select<D, NT>(p, bh, sm, e_chunk == 0);
  const int tid = threadIdx.x, cp = tid % CP, r = tid / CP;
  const int e = e_chunk * ROWS + r;
  const int K = p.completed, coarse = p.coarse, M = p.selected;
  const bf16_t* bank = f.bank + (size_t)bh * f.fine_cap * D * D;
  float acc0 = 0.0f, acc1 = 0.0f, den0 = 0.0f, den1 = 0.0f;
  for (int s0 = 0; s0 < M; s0 += U) {
    const int staged = min(U, M - s0);
    __syncthreads();                  // the previous stage is consumed (or the selection done)
    if (tid < staged) {
      const int j = key_index(sm.top[s0 + tid]);
      slot_id[tid] = j < group * coarse ? sm.chosen[j / group] * group + j % group
                                        : K * group + (j - group * coarse);
    }
    __syncthreads();
    // The stage's C^T loads first, then its weights (slot u's page row and
    // candidate row, both staged) while the loads are in flight.
    uint32_t cv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int m = min(u, staged - 1);
      cv[u] = *(const uint32_t*)(bank + ((size_t)slot_id[m] * D + e) * D + cp * 2);
    }
    for (int i = tid; i < staged * D; i += NT) {
      const int u = i / D, d = i % D;
      const int j = key_index(sm.top[s0 + u]);
      const int prow = j < group * coarse ? sm.chosen[j / group] : K;
      wts[u][d] = bf2f(sm.pw[prow][d]) * bf2f(sm.sw[j][d]);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u < staged) {
        const float2 w = *(const float2*)&wts[u][cp * 2];
        acc0 = fmaf(w.x, __uint_as_float(cv[u] << 16), acc0);
        acc1 = fmaf(w.y, __uint_as_float(cv[u] & 0xFFFF0000u), acc1);
        den0 += w.x;
        den1 += w.y;
      }
    }
  }
  *(float2*)(f.fold_g + ((size_t)bh * D + e) * D + cp * 2) = make_float2(acc0, acc1);
  if (e == 0) *(float2*)(f.fold_den + (size_t)bh * D + cp * 2) = make_float2(den0, den1);
}

// ---------------------------------------------------------------------------
// Routes of many queries at once: the per-query routes of the full-sequence
// read (route_interval = 1 in _read_training_group, tao_stream.py:596-665,
// with candidate_scores, routing_scores.py:7-47) and the turn routes of a
// prefill. The same candidates, masses, reduction order and stable top-k as
// route_kernel.
//
// What bounds them is VALU: every (query, row, channel) takes a product, its
// bf16 rounding and an fp32 add in the fold order. So a lane owns a query and
// keeps the rounded h * pw of one page in registers for the page's eight
// fines, and a row's weights are the same for the whole wave: they come
// through scalar loads and are widened on the scalar unit, which leaves 3.5
// vector instructions per channel (a lane per (query, row) pair with both
// rows in LDS needed about 9, and a wave per query 10 and a cross-lane fold
// per row). Masses of every visible fine are formed, also those of pages a
// query did not choose: the lanes of a wave choose different pages.
// A workgroup's waves share the fines evenly (with whole pages dealt to them, a
// short sequence's one page was a chain of up to eight fines in one wave), and
// a tile that reads every visible fine forms no mass.
// Measured (T16384 H7 D128): 404 us with a wave per query, 83 us now;
// (T16384 H32 D64): 403 us with a lane per (query, row) pair, 180 us now;
// (T2105 H7 D64): 11.3 us so, 3.7 now; (T3300 H1 D64): 10.8 so, 11.3 now.
// D = 128 is held to the 168 registers of three waves a SIMD: with 169, two a
// SIMD, T16384 H7 takes 101 us.
constexpr int kQThreads = 256;
constexpr int kQWaves = kQThreads / 64;

// Orders one wave's LDS accesses across its lanes (arrays private to a wave).
TAO_DEV void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

TAO_DEV void unpack8(const uint4& u, float out[8]) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    out[2 * i] = __uint_as_float(w[i] << 16);
    out[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
  }
}

// Wave-uniform read-only rows: the constant address space makes the loads
// scalar.
typedef const __attribute__((address_space(4))) uint32_t* const_words;
TAO_DEV const_words uniform_row(const bf16_t* p) { return (const_words)(uint64_t)p; }
TAO_DEV float word_bf(uint32_t w, int k) {
  return __uint_as_float(k ? (w & 0xFFFF0000u) : (w << 16));
}

// Sum over D channels in the fold order, the channels' values made as the
// tree reaches them: T(e, n) = T(e, 2n) + T(e + n, 2n), and pair(e) =
// y_e + y_(e + D/2) is a leaf.
template <int D, int E, int N, class Pair>
TAO_DEV float fold_tree(const Pair& pair) {
  if constexpr (N == D / 2) {
    return pair(E);
  } else {
    const float lo = fold_tree<D, E, 2 * N>(pair);
    const float hi = fold_tree<D, E + N, 2 * N>(pair);
    // Subtrees of 16 channels in turn: together they would not fit the registers.
    if constexpr (N == D / 16) __builtin_amdgcn_sched_barrier(0);
    return lo + hi;
  }
}

// 16-bit order key of a mass, never 0 (0 marks a fine that is no candidate).
TAO_DEV uint16_t mass_key(float mass) {
  bf16_t bits = f2bf(mass);
  if (bits == 0x8000) bits = 0;                      // -0 ties with +0, as in torch's sort
  const uint32_t key = bf16_order_key(bits);
  return (uint16_t)(key ? key : 1u);
}

// Keys of the fines [first, last) and of the pages that begin among them, one
// query per lane.
template <int D>
TAO_DEV void lane_masses(const bf16_t* hrow, int first, int last, bool write, bool pages, int K,
                         const bf16_t* pw, const SwRows& sw, uint16_t* pkey, uint16_t* fkey) {
  constexpr int G = 8, HALF = D / 2;
  for (int f = first; f < last;) {
    const int p = f / G, end = min(last, G * p + G);
    const const_words pwr = uniform_row(pw + (size_t)p * D);
    float x[D];
#pragma unroll
    for (int c = 0; c < HALF; c += 8) {
      float lo[8], hi[8];
      unpack8(*(const uint4*)(hrow + c), lo);
      unpack8(*(const uint4*)(hrow + HALF + c), hi);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t u = pack_bf16x2(lo[k] * word_bf(pwr[(c + k) / 2], k & 1),
                                       hi[k] * word_bf(pwr[(HALF + c + k) / 2], k & 1));
        x[c + k] = word_bf(u, 0);
        x[HALF + c + k] = word_bf(u, 1);
      }
    }
    if (pages && p < K && f == G * p) {
      const float m = fold_tree<D, 0, 1>([&](int e) __attribute__((always_inline)) {
        return x[e] + x[e + HALF];
      });
      if (write) pkey[p] = mass_key(rbf(m));
    }
    const_words s = uniform_row(sw.row(f, D));       // a page's rows are consecutive
    for (; f < end; ++f, s += D / 2) {
      const float m = fold_tree<D, 0, 1>([&](int e) __attribute__((always_inline)) {
        const uint32_t u = pack_bf16x2(x[e] * word_bf(s[e / 2], e & 1),
                                       x[e + HALF] * word_bf(s[(e + HALF) / 2], e & 1));
        return word_bf(u, 0) + word_bf(u, 1);
      });
      if (write) fkey[f] = mass_key(rbf(m));
    }
  }
}

// N masses of one query and one page per lane, in the lane's own rows:
// r(fold(r(r(h * pw) * sw_i))), or with PAGE r(fold(r(h * pw))). h * pw is
// rounded once for the N fines. The fold as eight partial sums of the
// channels 8c + k: chunks c and c + 2, then c and c + 1, then k by halves.
template <int D, int N, bool PAGE>
TAO_DEV void item_masses(const bf16_t* hrow, const bf16_t* pwrow, const bf16_t* const (&sw)[N],
                         float (&mass)[N]) {
  // Step n takes the channel blocks e and e + D / 2 of chunk c (D = 128: of
  // e = 8 c, then of 8 c + 32); the next step's rows are in flight meanwhile.
  constexpr int STEPS = D / 16;
  uint4 pr[2][2], sr[2][N][2];
  auto first = [](int n) __attribute__((always_inline)) {
    const int c = D == 128 ? n / 2 : n;            // chunks 0, 2, 1, 3
    return 8 * ((c & 1) * 2 + (c >> 1)) + (D == 128 ? 32 * (n & 1) : 0);
  };
  auto fetch = [&](int n) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int e0 = first(n) + (D / 2) * b;
      pr[n & 1][b] = *(const uint4*)(pwrow + e0);
#pragma unroll
      for (int i = 0; i < N; ++i)
        if constexpr (!PAGE) sr[n & 1][i][b] = *(const uint4*)(sw[i] + e0);
    }
  };
  float a[N][8], s[N][8], u[N][8];
  fetch(0);
#pragma unroll
  for (int n = 0; n < STEPS; ++n) {
    if (n + 1 < STEPS) fetch(n + 1);
    __builtin_amdgcn_sched_barrier(0);
    float t[N][8];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float hv[8], pv[8];
      unpack8(*(const uint4*)(hrow + first(n) + (D / 2) * b), hv);
      unpack8(pr[n & 1][b], pv);
      uint32_t x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        x[k] = pack_bf16x2(hv[2 * k] * pv[2 * k], hv[2 * k + 1] * pv[2 * k + 1]);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        float sv[8];
        if constexpr (!PAGE) unpack8(sr[n & 1][i][b], sv);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          float y = word_bf(x[k / 2], k & 1);
          if constexpr (!PAGE) y *= sv[k];
          if (b == 0) {
            t[i][k] = y;
          } else if constexpr (PAGE) {
            t[i][k] += y;
          } else {
            const uint32_t r = pack_bf16x2(t[i][k], y);
            t[i][k] = word_bf(r, 0) + word_bf(r, 1);
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        // Pinned: the compiler sinks the sums below every load otherwise.
        asm volatile("" : "+v"(t[i][k]));
        if (D == 128 && (n & 1) == 0) { u[i][k] = t[i][k]; continue; }
        const float v = D == 128 ? u[i][k] + t[i][k] : t[i][k];
        const int step = D == 128 ? n / 2 : n;
        if (step == 0) a[i][k] = v;
        if (step == 1) a[i][k] += v;
        if (step == 2) s[i][k] = v;
        if (step == 3) a[i][k] += s[i][k] + v;
      }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
    mass[i] = rbf(((a[i][0] + a[i][4]) + (a[i][2] + a[i][6])) +
                  ((a[i][1] + a[i][5]) + (a[i][3] + a[i][7])));
}

// h = r(softmax_D(raw_q)) of n <= 4 queries by one wave, as query_weights:
// sixteen lanes a query, lane i of them holding the channels i + 16 k, so the
// fold's first levels are in the lane and the last four are row rotations.
// row(q): raw_q row; dst(q): the row to store (bf16).
template <int CTRL>
TAO_DEV float row_ror(float v) { return dpp_partner<0x120 + CTRL>(v); }

template <int D, class Row, class Dst>
TAO_DEV void query_rows(int n, int lane, const Row& row, const Dst& dst) {
  constexpr int PER = D / 16;
  const int q = lane >> 4, i = lane & 15;
  const bf16_t* r = row(min(q, n - 1));
  float x[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) x[k] = bf2f(r[i + 16 * k]);
  float mx = x[0];
#pragma unroll
  for (int k = 1; k < PER; ++k) mx = fmaxf(mx, x[k]);
  mx = fmaxf(mx, row_ror<8>(mx));
  mx = fmaxf(mx, row_ror<4>(mx));
  mx = fmaxf(mx, row_ror<2>(mx));
  mx = fmaxf(mx, row_ror<1>(mx));
  float s[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) s[k] = x[k] = exp_cr(x[k] - mx);
#pragma unroll
  for (int w = PER / 2; w >= 1; w >>= 1)
#pragma unroll
    for (int k = 0; k < w; ++k) s[k] += s[k + w];
  float t = s[0];
  t += row_ror<8>(t);
  t += row_ror<4>(t);
  t += row_ror<2>(t);
  t += row_ror<1>(t);
  // x / t rounded to bf16: the product with the reciprocal is within 2 ulps
  // of the quotient, which alone decides near a bf16 rounding boundary.
  const float inv = 1.0f / t;
  bool near = false;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    s[k] = x[k] * inv;
    near |= near_bf16_midpoint(s[k], 4);
  }
  if (near) {
#pragma unroll
    for (int k = 0; k < PER; ++k) s[k] = x[k] / t;
  }
  if (q < n) {
    bf16_t* d = dst(q);
#pragma unroll
    for (int k = 0; k < PER; ++k) d[i + 16 * k] = f2bf(s[k]);
  }
}

TAO_DEV int quad_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);
  return v;
}
TAO_DEV uint32_t quad_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
}

// A quad's share of the keys: up to N in registers, or in LDS (N = 0).
template <int N>
struct QuadKeys {
  uint32_t k[N];
  TAO_DEV QuadKeys(const uint16_t* keys, int lo, int hi) {
#pragma unroll
    for (int i = 0; i < N; ++i) k[i] = lo + i < hi ? keys[lo + i] : 0u;
  }
  template <class F> TAO_DEV void each(const F& f) const {
#pragma unroll
    for (int i = 0; i < N; ++i) f(k[i], i);
  }
};
template <>
struct QuadKeys<0> {
  const uint16_t* p; int n;
  TAO_DEV QuadKeys(const uint16_t* keys, int lo, int hi) : p(keys + lo), n(hi - lo) {}
  template <class F> TAO_DEV void each(const F& f) const {
    for (int i = 0; i < n; ++i) f((uint32_t)p[i], i);
  }
};

template <int N, class Emit>
TAO_DEV void quad_select_n(const uint16_t* keys, int n, int m, int lane, const Emit& emit) {
  const int len = (n + 3) >> 2;
  const int lo = min(n, (lane & 3) * len), hi = min(n, lo + len);
  const QuadKeys<N> own(keys, lo, hi);
  // The bits that the largest and the smallest candidate share are the
  // threshold's too.
  uint32_t top = 0, low = 0;                    // low: largest of 0xFFFF - key
  own.each([&](uint32_t k, int) __attribute__((always_inline)) {
    top = max(top, k);
    low = max(low, k ? 0xFFFFu - k : 0u);
  });
  top = quad_max(top);
  low = 0xFFFFu - quad_max(low);
  const uint32_t differ = top ^ low;
  int bit = differ ? 31 - __clz((int)differ) : -1;
  uint32_t t = bit < 0 ? top : top & ~((2u << bit) - 1u);
  for (; bit >= 0; --bit) {
    const uint32_t c = t | (1u << bit);
    int count = 0;
    own.each([&](uint32_t k, int) __attribute__((always_inline)) { count += k >= c; });
    if (quad_sum(count) >= m) t = c;
  }
  int above = 0, ties = 0;
  own.each([&](uint32_t k, int) __attribute__((always_inline)) {
    above += k > t;
    ties += k == t;
  });
  int left = m - quad_sum(above);
  for (int i = 0; i < 3; ++i) {
    const int other = __shfl(ties, (lane & ~3) + i, 64);
    if (i < (lane & 3)) left -= other;
  }
  own.each([&](uint32_t k, int i) __attribute__((always_inline)) {
    if (k > t || (k == t && k && left-- > 0)) emit(lo + i);
  });
}

// The top m of keys[0, n) by (key descending, index ascending), 1 <= m <= the
// number of non-zero keys (the candidates): four lanes (a quad, sub = lane &
// 3) share the query and own a quarter of the indices each. The m-th largest
// key comes bit by bit from counts; ties at it are taken in index order.
// emit(index) runs in the owning lane, indices ascending over the quad.
template <class Emit>
TAO_DEV void quad_select(const uint16_t* keys, int n, int m, int lane, const Emit& emit) {
  if (n <= 32)
    quad_select_n<8>(keys, n, m, lane, emit);
  else if (n <= 64)
    quad_select_n<16>(keys, n, m, lane, emit);
  else
    quad_select_n<0>(keys, n, m, lane, emit);
}

// Opens the pages a query reads (open: one bit a page, zeroed) and clears the
// keys of the other pages' fines; four lanes a query.
TAO_DEV void quad_open_pages(const uint16_t* pkey, uint16_t* fkey, uint32_t* open, int K,
                             int coarse, int lane) {
  if (coarse < K) {
    if (coarse > 0)
      quad_select(pkey, K, coarse, lane,
                  [&](int pg) __attribute__((always_inline)) { atomicOr(&open[pg >> 5], 1u << (pg & 31)); });
    wave_sync();
    for (int f = lane & 3; f < 8 * K; f += 4)
      if (!(open[f >> 8] >> ((f >> 3) & 31) & 1u)) fkey[f] = 0;
  } else {
    for (int pg = lane & 3; pg < K; pg += 4) atomicOr(&open[pg >> 5], 1u << (pg & 31));
  }
  wave_sync();
}

// Per-query routes: a workgroup takes the queries of slots / 32 consecutive
// read tiles of one (batch, head). Selections are bitmasks over fine ids (the
// read needs the set, not the order).
template <int D, int W>
__global__ __launch_bounds__(64 * W, D == 128 ? 3 : 4) void route_queries_kernel(QueryRouteParams p,
                                                                  RouteLds lds) {
  extern __shared__ __align__(16) unsigned char route_smem[];
  constexpr int G = 8, PAD = D + 8;                // coarse_group (checked at launch)
  bf16_t* const hs = (bf16_t*)route_smem;
  uint16_t* const fkeys = (uint16_t*)(hs + lds.slots * PAD);
  uint16_t* const pkeys = fkeys + lds.slots * lds.fkeys;
  const int BH = p.B * p.H;
  const int bh = blockIdx.x % BH;
  const int b = bh / p.H, h = bh % p.H;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Tiles in reverse order: the latest tiles score the most keys.
  const int per = lds.slots / 32;
  const int t0 = ((int)gridDim.x / BH - 1 - (int)blockIdx.x / BH) * per;
  const int64_t* desc = p.tiles + 8 * (size_t)t0;
  const int tiles = min(per, p.n_tiles - t0);
  for (int a = 0; a < tiles;) {
    const int64_t* d0 = desc + 8 * a;
    int z = a + 1;                                 // tiles [a, z) share their route's shape
    while (z < tiles && desc[8 * z + 2] == d0[2] && desc[8 * z + 3] == d0[3] &&
           desc[8 * z + 4] == d0[4] && desc[8 * z + 6] == d0[6])
      ++z;
    if (!d0[6]) {                                  // no history: workgroup-uniform
      a = z;
      continue;
    }
    const int coarse = (int)d0[2], M = (int)d0[3], erel = (int)d0[4];
    const int epoch = p.first_epoch + erel, K = epoch / G;
    const int words = (epoch + 31) >> 5;
    const bf16_t* pw = p.pw_pool + ((size_t)erel * BH + bh) * p.pool_pcap * D;
    const SwRows sw{p.sw + (size_t)bh * p.fine_cap * D,
                    p.psw_pool + ((size_t)erel * BH + bh) * 8 * D, K * G};
    if (M == epoch) {          // every visible fine: no mass decides (up to six fines)
      for (int tl = a; tl < z; ++tl) {
        const int first = (int)desc[8 * tl], nq = (int)desc[8 * tl + 1];
        for (int i = threadIdx.x; i < nq * words; i += 64 * W) {
          const int q = i / words, left = epoch - 32 * (i - q * words);
          p.qsel[((size_t)(b * p.T + first + q) * p.H + h) * p.qsel_words + (i - q * words)] =
              left >= 32 ? ~0u : (1u << left) - 1u;
        }
      }
      a = z;
      continue;
    }
    // ---- h of each query
    for (int tl = a; tl < z; ++tl) {
      const int first = (int)desc[8 * tl], nq = (int)desc[8 * tl + 1];
      for (int q0 = 4 * w; q0 < nq; q0 += 4 * W)
        query_rows<D>(
            min(4, nq - q0), lane,
            [&](int i) __attribute__((always_inline)) {
              return p.rq + b * p.rq_sb + (int64_t)(first + q0 + i) * p.rq_st + h * p.rq_sh;
            },
            [&](int i) __attribute__((always_inline)) { return hs + (32 * tl + q0 + i) * PAD; });
    }
    __syncthreads();
    // ---- masses: lane = query slot (slots of no query compute and drop)
    {
      const int slot = lane & (lds.slots - 1);
      const bool write = lane >= 32 * a && lane < 32 * z;
      lane_masses<D>(hs + slot * PAD, w * epoch / W, (w + 1) * epoch / W, write, coarse < K, K,
                     pw, sw, pkeys + slot * lds.pkeys, fkeys + slot * lds.fkeys);
    }
    __syncthreads();
    // ---- selection: four lanes a query; open pages and bitmasks where h was
    uint32_t* const bits = (uint32_t*)hs;                    // [slot][words]
    uint32_t* const opens = bits + lds.slots * words;        // [slot][4]
    for (int i = threadIdx.x; i < lds.slots * (words + 4); i += 64 * W) bits[i] = 0u;
    __syncthreads();
    const int slot = 16 * w + (lane >> 2), tl = slot >> 5;
    if (tl >= a && tl < z && (slot & 31) < (int)desc[8 * tl + 1]) {
      uint16_t* fkey = fkeys + slot * lds.fkeys;
      quad_open_pages(pkeys + slot * lds.pkeys, fkey, opens + 4 * slot, K, coarse, lane);
      quad_select(fkey, epoch, M, lane, [&](int id) __attribute__((always_inline)) {
        atomicOr(&bits[slot * words + (id >> 5)], 1u << (id & 31));
      });
    }
    __syncthreads();
    for (int i = threadIdx.x + 32 * a * words; i < 32 * z * words; i += 64 * W) {
      const int s = i / words, wd = i - s * words;
      const int64_t* d = desc + 8 * (s >> 5);
      if ((s & 31) < (int)d[1])
        p.qsel[((size_t)(b * p.T + (int)d[0] + (s & 31)) * p.H + h) * p.qsel_words + wd] = bits[i];
    }
    __syncthreads();                               // h rows and keys are reused
    a = z;
  }
}

// Turn routes of a prefill (route_kernel's turn mode): one workgroup per
// (seal epoch, batch, head), sixteen of the epoch's turns at a time. A period
// of 24 tokens gives an epoch at most 11, too few for a lane per query: the
// lanes take (turn, page) items for the page masses, then (turn, chosen page,
// pair of its fines) items, so only candidates are scored and no lane waits
// for a turn that is not there. Outputs as route_kernel: ids in score order
// into the turn's sel_pool slot; the publishing turn also writes the state's
// route, chosen pages and route size. Measured at a 16K prompt (H32 D128):
// 87 us with a lane per (turn, row) pair in groups of sixteen turns over two
// or three epochs, 57 us now; one 16K call at 128K (rows beyond that form's
// LDS, a workgroup per turn): 350 -> 150 us.
TAO_DEV uint32_t score_key32(float score_bf, int index) {
  bf16_t bits = f2bf(score_bf);
  if (bits == 0x8000) bits = 0;                      // -0 ties with +0, as in torch's sort
  return (bf16_order_key(bits) << 16) | (uint32_t)(0xFFFF - index);
}

template <int D>
__global__ __launch_bounds__(kQThreads, 2) void route_turns_kernel(RouteParams p, int cap) {
  extern __shared__ __align__(16) unsigned char route_smem[];
  constexpr int G = 8, PAD = D + 8;
  bf16_t* const hs = (bf16_t*)route_smem;                      // [slot][PAD]
  uint32_t* const keys = (uint32_t*)(hs + kTurnSlots * PAD);   // [slot][cap]
  uint8_t* const chosen = (uint8_t*)(keys + kTurnSlots * cap); // [slot][cap]
  __shared__ uint32_t opens[kTurnSlots][kTurnMaxEpoch / 8 / 32];
  const int BH = p.B * p.H;
  const int bh = blockIdx.x % BH;
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Epochs in reverse order: the latest turns score the most rows.
  const int erel = p.n_epochs - 1 - (int)blockIdx.x / BH;
  // First turn of the epoch (turns ascend by epoch), 64 ways at a time: the
  // groups of `step` turns whose last turn is below the epoch are skipped.
  int s0 = 0, span = p.n_turns;
  while (span > 0) {
    const int step = (span + 63) / 64;
    const int at = s0 + min((lane + 1) * step, span) - 1;
    const int below = __popcll(__ballot(p.turns[8 * (size_t)at + 1] < erel));
    const int skip = min(below * step, span);
    s0 += skip;
    span = min(step, span - skip);
    if (step == 1) break;
  }
  s0 = __builtin_amdgcn_readfirstlane(s0);
  while (s0 < p.n_turns && p.turns[8 * (size_t)s0 + 1] == erel) {
    const int64_t* d0 = p.turns + 8 * (size_t)s0;
    const int64_t* dl = d0 + 8 * min(lane, min(kTurnSlots, p.n_turns - s0) - 1);
    const uint64_t same = __ballot(lane < min(kTurnSlots, p.n_turns - s0) && dl[1] == erel &&
                                   dl[4] == d0[4]);
    const int nq = __ffsll((unsigned long long)~same) - 1;
    const int K = (int)d0[2], pending = (int)d0[3], coarse = (int)d0[4];
    const int E = G * coarse + pending;
    const bf16_t* pw = p.pw_pool + ((size_t)erel * BH + bh) * p.pool_pcap * D;
    const SwRows sw{p.sw + (size_t)bh * p.fine_cap * D,
                    p.psw_pool + ((size_t)erel * BH + bh) * 8 * D, K * G};
    for (int i = tid; i < kTurnSlots * (kTurnMaxEpoch / 256); i += kQThreads) (&opens[0][0])[i] = 0u;
    for (int q0 = 4 * w; q0 < nq; q0 += 4 * kQWaves)
      query_rows<D>(
          min(4, nq - q0), lane,
          [&](int i) __attribute__((always_inline)) {
            return p.rq + b * p.rq_sb + d0[8 * (q0 + i)] * p.rq_st + h * p.rq_sh;
          },
          [&](int i) __attribute__((always_inline)) { return hs + (q0 + i) * PAD; });
    __syncthreads();
    // ---- coarse pages: stable top-`coarse` by page mass, listed ascending
    if (coarse < K) {
      for (int i = tid; i < nq * K; i += kQThreads) {
        const int pg = i / nq, q = i - pg * nq;
        const bf16_t* const none[1] = {nullptr};
        float m[1];
        item_masses<D, 1, true>(hs + q * PAD, pw + (size_t)pg * D, none, m);
        keys[q * cap + pg] = score_key32(m[0], pg);
      }
      __syncthreads();
      for (int i = tid; i < nq * K; i += kQThreads) {
        const int pg = i / nq, q = i - pg * nq;
        const uint32_t* row = keys + q * cap;
        const uint32_t mine = row[pg];
        int rank = 0;
        for (int j = 0; j < K; ++j) rank += row[j] > mine;
        if (rank < coarse) atomicOr(&opens[q][pg >> 5], 1u << (pg & 31));
      }
      __syncthreads();
      for (int i = tid; i < nq * K; i += kQThreads) {
        const int pg = i / nq, q = i - pg * nq;
        const uint32_t word = opens[q][pg >> 5], bit = 1u << (pg & 31);
        if (!(word & bit)) continue;
        int pos = __popc(word & (bit - 1));
        for (int j = 0; j < (pg >> 5); ++j) pos += __popc(opens[q][j]);
        chosen[q * cap + pos] = (uint8_t)pg;
      }
    } else {
      for (int i = tid; i < nq * K; i += kQThreads) {
        const int pg = i / nq, q = i - pg * nq;
        chosen[q * cap + pg] = (uint8_t)pg;
      }
    }
    __syncthreads();
    // ---- candidate masses: 8 fines of each chosen page, then the pending
    // fines, two a lane (candidates 2 i and 2 i + 1 share their page)
    auto cand = [&](int q, int j) __attribute__((always_inline)) {
      return j < G * coarse ? chosen[q * cap + j / G] * G + j % G : K * G + (j - G * coarse);
    };
    const int pairs = (E + 1) / 2;
    for (int i = tid; i < nq * pairs; i += kQThreads) {
      const int j = 2 * (i / nq), q = i - (j / 2) * nq;
      const int id = cand(q, j);
      const bf16_t* const rows[2] = {sw.row(id, D), sw.row(min(id + 1, K * G + pending - 1), D)};
      float m[2];
      item_masses<D, 2, false>(hs + q * PAD, pw + (size_t)(id / G) * D, rows, m);
      keys[q * cap + j] = score_key32(m[0], j);
      if (j + 1 < E) keys[q * cap + j + 1] = score_key32(m[1], j + 1);
    }
    __syncthreads();
    // ---- stable top-M in score order
    for (int i = tid; i < nq * E; i += kQThreads) {
      const int j = i / nq, q = i - j * nq;
      const int64_t* d = d0 + 8 * q;
      const uint32_t* row = keys + q * cap;
      const uint32_t mine = row[j];
      int rank = 0;
      for (int l = 0; l < E; ++l) rank += row[l] > mine;
      if (rank < (int)d[5]) {
        const int id = cand(q, j);
        p.sel_pool[((size_t)d[6] * BH + bh) * p.sel_cap + rank] = id;
        if (d[7]) p.sel[(size_t)bh * p.sel_cap + rank] = id;
      }
    }
    for (int q = 0; q < nq; ++q) {
      if (!d0[8 * q + 7]) continue;                // workgroup-uniform
      for (int i = tid; i < coarse; i += kQThreads)
        p.chosen[(size_t)bh * p.chosen_cap + i] = chosen[q * cap + i];
      if (bh == 0 && tid == 0) p.header[1] = (int)d0[8 * q + 5];
    }
    __syncthreads();                               // h rows, keys and lists are reused
    s0 += nq;
  }
}

}  // namespace

hipError_t launch_route_queries(const QueryRouteParams& p, int head_dim, hipStream_t s) {
  if (p.n_tiles <= 0) return hipSuccess;
  if (p.qsel_words < 1 || p.group != 8 || p.max_epoch < 1 || p.max_epoch > kQueryRouteMaxEpoch)
    return hipErrorInvalidValue;
  if (head_dim != 64 && head_dim != 128) return hipErrorInvalidValue;
  // Two read tiles a workgroup fill a wave's lanes (T16384 H16 D64: 95 us, 154
  // with one). One where the chip would not be full of them, up to four
  // workgroups a CU (D = 128: three): half of a wave's lanes idle, but so would
  // CUs (T3300 H7 D64: 14.5 us with two, 11.7 with one; T9008 H7: 24 with two,
  // 32 with one). And one where the keys of two do not fit the LDS (from 1,015
  // fines at D = 128).
  const int64_t singles = (int64_t)p.n_tiles * p.B * p.H;
  RouteLds lds = route_lds(64, p.max_epoch);
  if (singles <= (head_dim == 64 ? 1024 : 768) || lds.bytes(head_dim) > kLdsBytes)
    lds = route_lds(32, p.max_epoch);
  const size_t bytes = lds.bytes(head_dim);
  const int per = lds.slots / 32;
  const dim3 grid((unsigned)((p.n_tiles + per - 1) / per * p.B * p.H));
  // Eight waves where few workgroups route many fines: a wave's share of the
  // fines is then a serial chain (T9008 H2 D64: 20.5 us with four, 17.5 with
  // eight; T5000 H2: 12.4 with four, 13.0 with eight).
  const bool wide = per == 1 && p.max_epoch >= 32 && singles <= (head_dim == 64 ? 576 : 384);
  const auto kernel = head_dim == 128
                          ? (wide ? route_queries_kernel<128, 8> : route_queries_kernel<128, 4>)
                          : (wide ? route_queries_kernel<64, 8> : route_queries_kernel<64, 4>);
  if (bytes > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, grid, dim3(wide ? 512 : 256), bytes, s, p, lds);
  return hipGetLastError();
}

hipError_t launch_route(const RouteParams& p, int head_dim, hipStream_t s) {
  if (p.completed > kMaxSort || p.group * p.coarse + p.pending > kMaxSort)
    return hipErrorInvalidValue;
  if (p.turns && p.gate.header) return hipErrorInvalidValue;   // gates serve single turns
  // Turn mode: a workgroup per epoch when the turns ascend by epoch and the
  // keys of sixteen turns fit the LDS (those of a route of up to 512 fines, all
  // that a state keeps, do: at most 1,031 candidates); a workgroup per turn
  // otherwise.
  if (p.turns && p.n_turns > 0 && p.n_epochs > 0 && p.group == 8 &&
      (head_dim == 64 || head_dim == 128) &&
      turn_route_fits(head_dim, p.max_epoch, p.max_keys)) {
    const int cap = turn_route_cap(p.max_keys);
    const size_t bytes = turn_route_bytes(head_dim, cap);
    const dim3 tgrid((unsigned)(p.B * p.H * p.n_epochs));
    const auto kernel = head_dim == 128 ? route_turns_kernel<128> : route_turns_kernel<64>;
    if (bytes > 60 * 1024) {
      const hipError_t e = hipFuncSetAttribute(
          (const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
      if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kernel, tgrid, dim3(kQThreads), bytes, s, p, cap);
    return hipGetLastError();
  }
  // Single turn (a stream's refresh): the LDS-staged kernel when its rows fit.
  const int pages = p.completed + (p.pending > 0 ? 1 : 0);
  if (!p.turns && pages <= kRefreshPages && p.group * p.coarse + p.pending <= kRefreshRows &&
      p.group == 8) {
    const dim3 rgrid((unsigned)(p.B * p.H));
    if (head_dim == 128)
      hipLaunchKernelGGL(route_refresh_kernel<128>, rgrid, dim3(kRefreshThreads), 0, s, p);
    else if (head_dim == 64)
      hipLaunchKernelGGL(route_refresh_kernel<64>, rgrid, dim3(kRefreshThreads), 0, s, p);
    else
      return hipErrorInvalidValue;
    return hipGetLastError();
  }
  const dim3 grid((unsigned)(p.B * p.H * (p.turns ? p.n_turns : 1)));
  if (head_dim == 128)
    hipLaunchKernelGGL(route_kernel<128>, grid, dim3(kRouteThreads), 0, s, p);
  else if (head_dim == 64)
    hipLaunchKernelGGL(route_kernel<64>, grid, dim3(kRouteThreads), 0, s, p);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// The refresh and its fold in one launch when the route fits the staged
// refresh (single turn, group 8, rows within kRefreshPages / kRefreshRows);
// returns hipErrorNotSupported otherwise (the caller launches the two).
hipError_t launch_refresh_fold(const RouteParams& p, const FoldParams& f, int head_dim,
                               hipStream_t s) {
  const int pages = p.completed + (p.pending > 0 ? 1 : 0);
  if (p.turns || pages > kRefreshPages || p.group * p.coarse + p.pending > kRefreshRows ||
      p.group != 8 || f.group != 8 || p.selected != f.M || p.selected <= 0)
    return hipErrorNotSupported;
  if (head_dim == 128) {
    constexpr int CHUNKS = 128 / (kRefreshThreads / 64);
    hipLaunchKernelGGL(refresh_fold_kernel<128>, dim3((unsigned)(p.B * p.H * CHUNKS)),
                       dim3(kRefreshThreads), 0, s, p, f);
  } else if (head_dim == 64) {
    constexpr int CHUNKS = 64 / (kRefreshThreads / 32);
    hipLaunchKernelGGL(refresh_fold_kernel<64>, dim3((unsigned)(p.B * p.H * CHUNKS)),
                       dim3(kRefreshThreads), 0, s, p, f);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace tao
