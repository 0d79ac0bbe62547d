// fp32 full-sequence read: tao_attention on fp32 operands.
//
// Reference: tao_attention (operator.py:40-54) = read_training
// (tao_stream.py:668-757, route_interval=1) followed by _fuse_training
// (operator.py:21-38), with the softmax fine writer of _seal_training_all
// (tao_stream.py:80-123), the page metadata of _training_metadata /
// _tile_metadata (:530-593), the local tiles of _local_training_corrected_4k
// (:760-787) and the per-query route and read of _read_training_group
// (:596-665).
//
// fp32 semantics. The reference's torch operations follow the operand dtype;
// its Triton kernels hard-cast their products to bf16 (routing_scores.py:28,
// selected_read.py:31, 48), which has no fp32 meaning. Here every rounding
// point of the bf16 contract rounds to fp32 instead, so:
//  * everything that decides a route is bit-reproducible: exp and log are
//    fp64 evaluations rounded once to fp32; sums over channels, pages and
//    slots use the butterfly order (pad to a power of two, add the upper half
//    onto the lower); the writer's token sums run four sequential 64-token
//    quarters added pairwise; every product and sum is one IEEE fp32
//    operation (no contraction in this file);
//  * the local attention, the value matrices, the coarse read and the
//    selected read's numerator accumulate in fp32 in their own order, within
//    the 1e-4 tolerance of exact arithmetic.
// The contractions run on the fp32 matrix instructions (fp32 products and
// sums); everything else is VALU code.
#pragma clang fp contract(off)

#include "schedule.h"
#include "tao_common.h"
#include "tao_fusion.h"
#include "tao_launch.h"

namespace tao {
namespace {

constexpr int kFine = 256;          // fine_tokens
constexpr int kGroup = 8;           // coarse_group
constexpr int kKeep = 512;          // local_keep
constexpr int kRowsPerPage = 36;    // segment-weight rows of a page: prefixes n = 1..8
constexpr int kChunk = 16;          // queries per read block
constexpr float kLogTwoF32 = 0.693147180559945309f;   // fp32(log 2)

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// fp32 matrix instructions, accumulated in fp32. 32x32x2: lane l gives A row
// l % 32 and B column l % 32 of k = l / 32, accumulator i is row
// acc_row(i, l / 32) of column l % 32. 16x16x4: A row / B column l % 16 of
// k = l / 16, accumulator i is row 4 (l / 16) + i of column l % 16.
TAO_DEV f32x16 mfma32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
TAO_DEV f32x4 mfma16(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
TAO_DEV int acc_row(int i, int half) { return 8 * (i / 4) + 4 * half + i % 4; }

TAO_DEV float ld(const F32View& v, int b, int64_t t, int h, int d) {
  return v.p[b * v.sb + t * v.st + h * v.sh + d];
}
// Four channels; 16-byte loads where every row of the view allows them.
TAO_DEV f32x4 ld4(const float* p, bool vec) {
  if (vec) return *(const f32x4*)p;
  return (f32x4){p[0], p[1], p[2], p[3]};
}
bool rows_aligned(const F32View& v) {
  return ((uintptr_t)v.p & 15) == 0 && v.sb % 4 == 0 && v.st % 4 == 0 && v.sh % 4 == 0;
}

// Butterfly sum of the 64 lanes' values (fold halves: lane i adds lane
// i + half for half = 32 .. 1), broadcast to every lane.
TAO_DEV float wave_fold(float x) {
#pragma unroll
  for (int half = 32; half >= 1; half >>= 1) x = x + __shfl_down(x, half);
  return __shfl(x, 0);
}

TAO_DEV float wave_top(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
  return x;
}

// --------------------------------------------------------------- local tiles
// Query t of tile j attends causally to keys [max(0, 256 j - 512), t]
// (_local_training_corrected_4k and its ragged fallback); softmax scale
// 1/sqrt(D) as SDPA's default. A workgroup takes 32 queries and deals their
// 32-key blocks to eight waves, each with its own online softmax; the waves'
// partials are merged in wave order: M = max m_w, l = sum l_w e^(m_w - M),
// o = sum acc_w e^(m_w - M) / l. Scores are K Q^T on the fp32 matrix cores,
// so a lane holds sixteen keys of one query: its probabilities are the
// operand of V^T P^T as they stand, and only K passes through LDS. B1 T2048 H4
// D64 fills the chip with 256 workgroups, about 10 us of matrix time each:
// 124 us with a query per lane on the VALU and K, V through LDS; 29 us now,
// the writer's blocks included (50 us before in a launch of their own).
constexpr int kLocalWaves = 8;
constexpr int kLocalRows = 65;       // padded lanes of a merge row

template <int D>
struct F32LocalSmem {
  union {
    float k[kLocalWaves][32][D + 4];             // a wave's block, padded rows
    float red[kLocalWaves][16][kLocalRows];
  };
  float wm[kLocalWaves][32], wl[kLocalWaves][32];
  uint32_t bad;                                  // queries whose output holds a NaN
};

// Orders one wave's LDS accesses across its lanes (scratch private to a wave).
TAO_DEV void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Local attention of query t over its keys [k0, t], by one wave: lane = channel.
template <int D>
TAO_DEV void local_row(const F32Params& p, int k0, int t, int b, int h, int lane) {
  constexpr int R = D / 64;
  const float scale = 1.0f / sqrtf((float)D);
  float q[R], acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    q[r] = ld(p.q, b, t, h, lane + 64 * r);
    acc[r] = 0.0f;
  }
  float m = -__builtin_inff(), l = 0.0f;
  for (int key = k0; key <= t; ++key) {
    float dot = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) dot = fmaf(q[r], ld(p.k, b, key, h, lane + 64 * r), dot);
    const float s = wave_fold(dot) * scale;
    if (s == -__builtin_inff()) continue;        // weighs 0; the same in every lane
    const float mn = fmaxf(m, s), corr = expf(m - mn), wgt = expf(s - mn);
    l = l * corr + wgt;
#pragma unroll
    for (int r = 0; r < R; ++r)
      acc[r] = fmaf(wgt, ld(p.v, b, key, h, lane + 64 * r), acc[r] * corr);
    m = mn;
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    p.local[(((size_t)b * p.T + t) * p.H + h) * D + lane + 64 * r] = acc[r] / l;
}

template <int D>
TAO_DEV void local_tile(const F32Params& p, bool vec, int t0, int b, int h, F32LocalSmem<D>& sm) {
  constexpr int CT = D / 32;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int t = t0 + col;
  const int k0 = max(0, (t0 / kFine) * kFine - kKeep);
  auto& red = sm.red;
  auto& wm = sm.wm;
  auto& wl = sm.wl;
  const float scale = 1.0f / sqrtf((float)D);
  // Lane: channels half * D / 2 + i of its query (and of a block's key).
  const int c0 = half * (D / 2);
  f32x4 q[D / 8];
  const float* qp = p.q.p + b * p.q.sb + (int64_t)min(t, p.T - 1) * p.q.st + h * p.q.sh + c0;
#pragma unroll
  for (int i = 0; i < D / 8; ++i) q[i] = ld4(qp + 4 * i, vec);
  f32x16 acc[CT] = {};
  float m = -__builtin_inff(), l = 0.0f;
  if (threadIdx.x == 0) sm.bad = 0u;             // published by the merge's barriers
  // Keys past the sequence (the last block's) repeat its last row; the causal
  // mask drops them. K rows come whole (a row per 16 or 32 lanes) and turn to
  // a row per lane in LDS: read a row per lane from memory, every load touches
  // 64 cache lines, which the eight waves evict before their next piece.
  f32x4 k[D / 8];
  float v[CT][16];
  auto load = [&](int kb) __attribute__((always_inline)) {
    constexpr int ROWS = 256 / D;                // rows of one load
    const int row0 = lane / (D / 4), c = 4 * (lane % (D / 4));
    const float* kp = p.k.p + b * p.k.sb + h * p.k.sh + c;
#pragma unroll
    for (int i = 0; i < D / 8; ++i)
      k[i] = ld4(kp + (int64_t)min(kb + ROWS * i + row0, p.T - 1) * p.k.st, vec);
  };
  auto load_v = [&](int kb) __attribute__((always_inline)) {
    const float* vp = p.v.p + b * p.v.sb + h * p.v.sh + col;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float* row = vp + (int64_t)min(kb + acc_row(i, half), p.T - 1) * p.v.st;
#pragma unroll
      for (int c2 = 0; c2 < CT; ++c2) v[c2][i] = row[32 * c2];
    }
  };
  for (int kb = k0 + 32 * w; kb <= t0; kb += 32 * kLocalWaves) {
    load(kb);
    if (D == 64) load_v(kb);                     // D = 128: once K's registers are free
    wave_sync();                                 // the previous block's rows are read
    {
      constexpr int ROWS = 256 / D;
#pragma unroll
      for (int i = 0; i < D / 8; ++i)
        *(f32x4*)&sm.k[w][ROWS * i + lane / (D / 4)][4 * (lane % (D / 4))] = k[i];
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < D / 8; ++i) k[i] = *(const f32x4*)&sm.k[w][col][c0 + 4 * i];
    f32x16 s = {};
#pragma unroll
    for (int i = 0; i < D / 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) s = mfma32(k[i][j], q[i][j], s);
    if (D == 128) {
      __builtin_amdgcn_sched_barrier(0);
      load_v(kb);
    }
    float top = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = kb + acc_row(i, half) <= t ? s[i] * scale : -__builtin_inff();
      top = fmaxf(top, s[i]);
    }
    top = fmaxf(top, __shfl_xor(top, 32));
    const float mn = fmaxf(m, top);
    // No finite score yet (every visible one -inf): they weigh 0.
    const float at = mn > -__builtin_inff() ? mn : 0.0f;
    const float corr = expf(m - at);
    l *= corr;
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[c] *= corr;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = expf(s[i] - at);
      l += s[i];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[c] = mfma32(v[c][i], s[i], acc[c]);
    m = mn;
  }
  l += __shfl_xor(l, 32);
  // Merge the waves' partials (a wave without a block or a finite score has
  // m = -inf and weighs 0).
  if (half == 0) wm[w][col] = m;
  __syncthreads();                               // also: the K blocks are read
  float top = wm[0][col];
#pragma unroll
  for (int v = 1; v < kLocalWaves; ++v) top = fmaxf(top, wm[v][col]);
  const float f = m > -__builtin_inff() ? expf(m - top) : 0.0f;
  if (half == 0) wl[w][col] = l * f;
  // 32 channels a round; thread -> (channel, query), rows of 128 bytes.
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    if (c) __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) red[w][i][lane] = acc[c][i] * f;
    __syncthreads();
    for (int i = threadIdx.x; i < 32 * 32; i += 64 * kLocalWaves) {
      const int ch = i & 31, qi = i >> 5;
      if (t0 + qi >= p.T) continue;
      float sum = 0.0f, lsum = 0.0f;
#pragma unroll
      for (int v = 0; v < kLocalWaves; ++v) {
        sum += red[v][(ch >> 3) * 4 + (ch & 3)][qi + 32 * ((ch >> 2) & 1)];
        lsum += wl[v][qi];
      }
      const float o = sum / lsum;
      p.local[(((size_t)b * p.T + t0 + qi) * p.H + h) * D + 32 * c + ch] = o;
      if (o != o) atomicOr(&sm.bad, 1u << qi);
    }
  }
  __syncthreads();
  // The products give a key that a query does not see a weight of 0, and 0
  // times an infinite or NaN value is NaN. A NaN outlives every later sum, so
  // the queries that hold one are computed again over their own keys alone, a
  // wave each.
  for (uint32_t bad = sm.bad; bad; bad &= bad - 1) {
    const int qi = __builtin_ctz(bad);
    if (qi % kLocalWaves == w) local_row<D>(p, k0, t0 + qi, b, h, lane);
  }
}

// ------------------------------------------------------------------- writer
// 32 channels d of one visible block (fine f) of one head: per channel over
// its 256 tokens, top = max k, e = exp(k - top), Z = quarter sums, P = e / Z,
// z = top + log Z; then C[d][e] = sum_t P[t][d] v[t][e] on the fp32 matrix
// cores, the tokens dealt to the waves and their partials added in order.
// Bound by the fp64 exps and the latency of its phases: sixteen tokens a
// thread (50 us for the 20 blocks of B1 T2048 H4 D64 with a workgroup per
// block, sixty-four tokens a thread and the product on the VALU; 14 us now,
// alone).
struct F32WriterSmem {
  float prob[kFine][32];
  float red[16][32];
  float part_c[6][16][64];
};

template <int D>
TAO_DEV void writer_slice(const F32Params& p, int f, int c0, int b, int h, F32WriterSmem& sm) {
  constexpr int CT = D / 32, PARTS = 8 / CT, STEP = kFine / PARTS;
  const int tid = threadIdx.x, d = tid & 31, seg = tid >> 5;
  auto& prob = sm.prob;
  auto& red = sm.red;
  auto& part_c = sm.part_c;
  const int64_t base = (int64_t)f * kFine;
  const size_t bh = (size_t)b * p.H + h;
  float x[16];
  float top = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    x[i] = ld(p.rk, b, base + 16 * seg + i, h, c0 + d);
    top = fmaxf(top, x[i]);
  }
  red[seg][d] = top;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) top = fmaxf(top, red[i][d]);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    x[i] = exp_cr(x[i] - top);
    prob[16 * seg + i][d] = x[i];
  }
  __syncthreads();
  if (seg < 4) {                       // the quarter's tokens in order
    float acc = 0.0f;
#pragma unroll 16
    for (int i = 0; i < 64; ++i) acc = acc + prob[64 * seg + i][d];
    red[seg][d] = acc;
  }
  __syncthreads();
  const float total = (red[0][d] + red[1][d]) + (red[2][d] + red[3][d]);
#pragma unroll
  for (int i = 0; i < 16; ++i) prob[16 * seg + i][d] = x[i] / total;
  if (seg == 0) p.fine_z[(bh * p.S + f) * D + c0 + d] = top + log_cr(total);
  __syncthreads();
  const int lane = tid & 63, half = lane >> 5, col = lane & 31;
  const int ct = (tid >> 6) % CT, part = (tid >> 6) / CT;
  f32x16 acc = {};
  const float* vp = p.v.p + b * p.v.sb + h * p.v.sh + 32 * ct + col;
#pragma unroll 16
  for (int i = 0; i < STEP / 2; ++i) {
    const int tok = STEP * part + 2 * i + half;
    acc = mfma32(prob[tok][col], vp[(base + tok) * p.v.st], acc);
  }
  if (part)
#pragma unroll
    for (int i = 0; i < 16; ++i) part_c[(part - 1) * CT + ct][i][lane] = acc[i];
  __syncthreads();
  if (part) return;
  float* out = p.bank + ((bh * p.S + f) * D + c0) * D + 32 * ct + col;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float sum = acc[i];
#pragma unroll
    for (int v = 1; v < PARTS; ++v) sum += part_c[(v - 1) * CT + ct][i][lane];
    out[(size_t)acc_row(i, half) * D] = sum;
  }
}

// Both in one launch: they do not depend on each other, and the writer's few
// workgroups (dispatched first) run beside the local tiles. One workgroup a
// CU: two of them would share its matrix cores while other CUs are idle (46
// against 37 us at B1 T2048 H4 D64, measured before the tiles went out in
// descending order over all heads).
template <int D>
__global__ __launch_bounds__(64 * kLocalWaves, 2) void f32_front_kernel(
    F32Params p, bool vec, int writers) {
  __shared__ union {
    F32LocalSmem<D> local;
    F32WriterSmem writer;
  } sm;
  constexpr int SL = D / 32;
  const int BH = p.B * p.H;
  const int x = blockIdx.x / BH, bh = blockIdx.x % BH, b = bh / p.H, h = bh % p.H;
  if (x < writers)
    writer_slice<D>(p, x / SL, 32 * (x % SL), b, h, sm.writer);
  else   // the longest windows first
    local_tile<D>(p, vec, ((int)gridDim.x / BH - 1 - x) * 32, b, h, sm.local);
}

// -------------------------------------------------------------------- pages
// Prefix n of page pg (a workgroup each): pz[n - 1] = logsumexp of its first
// n fines (a completed page's summary is n = 8, a pending page's the prefix a
// tile sees), the segment weights exp(z - pz[n - 1]) of those n fines, and,
// with coarse values, the completed page's value matrix
// PC[d][e] = sum_s w_s[d] C_s[d][e] (tao_stream.py:486-499).
template <int D>
__global__ __launch_bounds__(256) void f32_pages_kernel(F32Params p) {
  const int pg = blockIdx.x / kGroup, n = 1 + blockIdx.x % kGroup;
  const int h = blockIdx.y, b = blockIdx.z;
  const size_t bh = (size_t)b * p.H + h;
  const int first = pg * kGroup;
  if (n > p.S - first) return;
  __shared__ float wfull[kGroup][D];
  const int d = threadIdx.x;
  if (d < D) {
    float z[kGroup], e[kGroup];
    float top = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < kGroup; ++i) {
      z[i] = i < n ? p.fine_z[(bh * p.S + first + i) * D + d] : -__builtin_inff();
      top = fmaxf(top, z[i]);
    }
    if (__builtin_isinf(top)) top = 0.0f;
#pragma unroll
    for (int i = 0; i < kGroup; ++i) e[i] = i < n ? exp_cr(z[i] - top) : 0.0f;
    int width = 1;
    while (width < n) width <<= 1;
    for (int half = width / 2; half >= 1; half >>= 1)
#pragma unroll
      for (int i = 0; i < kGroup / 2; ++i)
        if (i < half) e[i] = e[i] + e[i + half];
    const float v = log_cr(e[0]) + top;
    p.pz[((bh * p.P8 + pg) * kGroup + n - 1) * D + d] = v;
    float* sw = p.swt + ((bh * p.P8 + pg) * kRowsPerPage + n * (n - 1) / 2) * D + d;
#pragma unroll
    for (int j = 0; j < kGroup; ++j)
      if (j < n) {
        const float w = exp_cr(z[j] - v);
        sw[(size_t)j * D] = w;
        wfull[j][d] = w;
      }
  }
  if (!p.pc || n < kGroup) return;
  __syncthreads();
  const float* c = p.bank + (bh * p.S + first) * D * D;
  float* out = p.pc + (bh * p.Pc + pg) * D * D;
  for (int i = threadIdx.x; i < D * D; i += 256) {
    float acc = 0.0f;
#pragma unroll
    for (int s = 0; s < kGroup; ++s) acc = fmaf(wfull[s][i / D], c[(size_t)s * D * D + i], acc);
    out[i] = acc;
  }
}

// --------------------------------------------------------------------- read
// kChunk queries of one tile and head per workgroup of four waves. Tile
// prologue: the pages the tile sees (completed pages' summaries, the pending
// page's prefix summary), page weights softmax over them per channel and,
// with coarse values, the coarse weights softmax over the completed pages.
// Then h = softmax(raw_q); page masses of the (query, page) pairs and
// candidate masses of the (query, candidate) pairs, a lane each with the
// channel sum in registers; ranks by counting; and the reads on the fp32
// matrix cores: per fine that any of the queries selected, the rows
// ch = (h pw) sw of the queries that did (0 for the others) against its
// matrix, a wave per 16 columns. B1 T2048 H4 D64: 57 us with a wave per query
// (a cross-lane fold per mass, the read on the VALU), 22 us now.
constexpr int kMaxPages = 64;
constexpr int kMaxCand = 256;
constexpr int kReadThreads = 256;

// LDS of a read workgroup in floats; pages and cand: the call's largest.
struct F32ReadLds {
  int pages, cand;
  __host__ __device__ size_t floats(int D) const {
    return (size_t)2 * pages * D + 3 * kChunk * (D + 4) +
           (size_t)kChunk * cand * 3 + kChunk;
  }
};

// Monotone key of a mass: larger mass -> larger key, -0 as +0; a NaN has a
// place in the order too, so every rank is taken once.
TAO_DEV uint32_t f32_order_key(float x) {
  uint32_t u = __float_as_uint(x);
  if (u == 0x80000000u) u = 0u;
  return u & 0x80000000u ? ~u : u | 0x80000000u;
}

TAO_DEV int stable_rank(int idx, int n, const float* all) {
  const uint32_t mine = f32_order_key(all[idx]);
  int r = 0;
  for (int j = 0; j < n; ++j) {
    const uint32_t o = f32_order_key(all[j]);
    r += o > mine || (o == mine && j < idx);
  }
  return r;
}

// Fold of (h pw) [sw] over the D channels by one lane: eight partial sums of
// the channels 8 c + k (blocks e, e + 64 and e + 32, then the chunks c, c + 2
// and c, c + 1), then k by halves.
template <int D, bool SW>
TAO_DEV float lane_fold(const float* h, const float* pw, const float* sw) {
  auto block = [&](int e0, float (&y)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const f32x4 a = *(const f32x4*)(h + e0 + 4 * v), c = *(const f32x4*)(pw + e0 + 4 * v);
      f32x4 x;
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = a[k] * c[k];
      if constexpr (SW) {
        const f32x4 g = *(const f32x4*)(sw + e0 + 4 * v);
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = x[k] * g[k];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) y[4 * v + k] = x[k];
    }
  };
  float chunk[4][8];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float y[D / 32][8];
#pragma unroll
    for (int i = 0; i < D / 32; ++i) block(8 * c + 32 * i, y[i]);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if constexpr (D == 64)
        chunk[c][k] = y[0][k] + y[1][k];
      else
        chunk[c][k] = (y[0][k] + y[2][k]) + (y[1][k] + y[3][k]);
    }
  }
  float s[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) s[k] = (chunk[0][k] + chunk[2][k]) + (chunk[1][k] + chunk[3][k]);
  return ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
}

template <int D>
__global__ __launch_bounds__(kReadThreads) void f32_read_kernel(F32Params p, F32ReadLds lds) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int h = blockIdx.y, b = blockIdx.z;
  const int t0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * kChunk;
  const int nq = min(p.T - t0, kChunk);
  const int tile = t0 / kFine;
  const int visible = max(0, tile - kKeep / kFine);
  const size_t bh = (size_t)b * p.H + h;
  float* out = p.out + b * p.out_sb + (int64_t)t0 * p.out_st + h * p.out_sh;
  const float* local = p.local + ((size_t)b * p.T + t0) * p.H * D + (size_t)h * D;
  int32_t* sel_out = p.sel_out ? p.sel_out + (((size_t)b * p.T + t0) * p.H + h) * p.sel_cap : nullptr;
  if (!visible) {   // neither history branch present: the output is local
    for (int i = tid; i < nq * D; i += kReadThreads)
      out[(i / D) * p.out_st + i % D] = local[(size_t)(i / D) * p.H * D + i % D];
    if (sel_out)
      for (int i = tid; i < nq * p.sel_cap; i += kReadThreads)
        sel_out[(size_t)(i / p.sel_cap) * p.H * p.sel_cap + i % p.sel_cap] = -1;
    return;
  }
  const int completed = visible / kGroup, pending = visible % kGroup;
  const int P = completed + (pending > 0);
  int64_t coarse64 = 0, elig64 = 0, sel64 = 0;
  sched::routed_counts(p.cfg, completed, pending, &coarse64, &elig64, &sel64);
  const int coarse = (int)coarse64, M = (int)sel64, E = coarse * kGroup + pending;
  const bool coarse_on = p.coarse_values && tile * kFine >= kKeep + kGroup * kFine;

  extern __shared__ __align__(16) float read_smem[];
  constexpr int HP = D + 4;                            // padded h / ch row
  float* const pw = read_smem;                         // [page][D]
  float* const cw = pw + lds.pages * D;                // [page][D]
  float* const hs = cw + lds.pages * D;                // [query][HP]
  float* const ch = hs + kChunk * HP;                  // [2][query][HP]
  float* const mass = ch + 2 * kChunk * HP;            // [query][cand]
  float* const slots = mass + kChunk * lds.cand;       // [query][cand] masses by rank
  int16_t* const cand = (int16_t*)(slots + kChunk * lds.cand);   // [query][cand] fine ids
  int16_t* const sel = cand + kChunk * lds.cand;       // [query][cand] ids by rank
  float* const den = (float*)(sel + kChunk * lds.cand);          // [query]
  __shared__ uint32_t picked[kChunk][kMaxPages * kGroup / 32];   // bit per fine
  __shared__ uint32_t open[kChunk][kMaxPages / 32];
  __shared__ uint32_t bad;                             // queries whose numerator holds a NaN
  const int PC = lds.cand;

  for (int i = tid; i < kChunk * (kMaxPages * kGroup / 32); i += kReadThreads) (&picked[0][0])[i] = 0u;
  if (tid < kChunk * (kMaxPages / 32)) (&open[0][0])[tid] = 0u;
  if (tid == 0) bad = 0u;
  // Page z the tile sees, page weights and coarse weights: a thread per
  // channel for up to 8 pages (the fold over the next power of two), else
  // lanes = pages and the waves take the channels in turn.
  const float* pzt = p.pz + bh * p.P8 * kGroup * D;
  auto page_z = [&](int pg, int d) __attribute__((always_inline)) {
    return pzt[((size_t)pg * kGroup + (pg < completed ? kGroup : pending) - 1) * D + d];
  };
  if (P <= kGroup) {
    for (int i = tid; i < 2 * D; i += kReadThreads) {
      const int d = i % D, n = i < D ? P : completed;
      if (i >= D && !coarse_on) break;
      float e[kGroup];
      float top = -__builtin_inff();
#pragma unroll
      for (int g = 0; g < kGroup; ++g) {
        e[g] = g < n ? page_z(g, d) : -__builtin_inff();
        top = fmaxf(top, e[g]);
      }
      float s[kGroup];
#pragma unroll
      for (int g = 0; g < kGroup; ++g) s[g] = e[g] = g < n ? exp_cr(e[g] - top) : 0.0f;
#pragma unroll
      for (int half = kGroup / 2; half >= 1; half >>= 1)
#pragma unroll
        for (int g = 0; g < half; ++g) s[g] = s[g] + s[g + half];
      float* dst = (i < D ? pw : cw) + d;
#pragma unroll
      for (int g = 0; g < kGroup; ++g)
        if (g < n) dst[g * D] = e[g] / s[0];
    }
  } else {
    for (int d = w; d < D; d += kReadThreads / 64) {
      const float zp = lane < P ? page_z(lane, d) : -__builtin_inff();
      const float top = wave_top(zp);                  // all lanes take part
      const float e = lane < P ? exp_cr(zp - top) : 0.0f;
      const float total = wave_fold(e);
      if (lane < P) pw[lane * D + d] = e / total;
      if (coarse_on) {
        const float zc = lane < completed ? zp : -__builtin_inff();
        const float tc = wave_top(zc);
        const float ec = lane < completed ? exp_cr(zc - tc) : 0.0f;
        const float tot = wave_fold(ec);
        if (lane < completed) cw[lane * D + d] = ec / tot;
      }
    }
  }
  // h = softmax over channels of raw_q: sixteen lanes a query, lane i of
  // them the channels i + 16 k.
  {
    const int q = tid >> 4, i = tid & 15;
    float x[D / 16], s[D / 16];
#pragma unroll
    for (int k = 0; k < D / 16; ++k) x[k] = ld(p.rq, b, t0 + min(q, nq - 1), h, i + 16 * k);
    float top = x[0];
#pragma unroll
    for (int k = 1; k < D / 16; ++k) top = fmaxf(top, x[k]);
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
#pragma unroll
    for (int k = 0; k < D / 16; ++k) s[k] = x[k] = exp_cr(x[k] - top);
#pragma unroll
    for (int half = D / 32; half >= 1; half >>= 1)
#pragma unroll
      for (int k = 0; k < half; ++k) s[k] = s[k] + s[k + half];
    float total = s[0];
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) total = total + __shfl_xor(total, off);
#pragma unroll
    for (int k = 0; k < D / 16; ++k) hs[q * HP + i + 16 * k] = x[k] / total;
  }
  __syncthreads();

  const float* swt = p.swt + bh * p.P8 * kRowsPerPage * D;
  auto sw_row = [&](int id) __attribute__((always_inline)) {
    const int pg = id / kGroup, j = id % kGroup;
    const int n = pg < completed ? kGroup : pending;
    return swt + ((size_t)pg * kRowsPerPage + n * (n - 1) / 2 + j) * D;
  };
  // Chosen pages: stable top-`coarse` of the completed pages' masses.
  if (coarse < completed) {
    for (int i = tid; i < kChunk * completed; i += kReadThreads) {
      const int q = i % kChunk, pg = i / kChunk;
      mass[q * PC + pg] = lane_fold<D, false>(hs + q * HP, pw + pg * D, nullptr);
    }
    __syncthreads();
    for (int i = tid; i < kChunk * completed; i += kReadThreads) {
      const int q = i % kChunk, pg = i / kChunk;
      if (stable_rank(pg, completed, mass + q * PC) < coarse)
        atomicOr(&open[q][pg >> 5], 1u << (pg & 31));
    }
    __syncthreads();
  }
  for (int i = tid; i < kChunk * P; i += kReadThreads) {
    const int q = i % kChunk, pg = i / kChunk;
    int pos = pg;
    if (coarse < completed && pg < completed) {
      const uint32_t word = open[q][pg >> 5], bit = 1u << (pg & 31);
      if (!(word & bit)) continue;
      pos = __popc(word & (bit - 1)) + (pg >= 32 ? __popc(open[q][0]) : 0);
    } else if (pg == completed) {
      pos = coarse;
    }
    for (int s = 0; s < (pg < completed ? kGroup : pending); ++s)
      cand[q * PC + pos * kGroup + s] = (int16_t)(pg * kGroup + s);
  }
  __syncthreads();
  // Candidate masses sum_d (h pw[page]) sw[fine], then the stable top-M.
  for (int i = tid; i < kChunk * E; i += kReadThreads) {
    const int q = i % kChunk, c = i / kChunk, id = cand[q * PC + c];
    mass[q * PC + c] = lane_fold<D, true>(hs + q * HP, pw + (id / kGroup) * D, sw_row(id));
  }
  __syncthreads();
  for (int i = tid; i < kChunk * E; i += kReadThreads) {
    const int q = i % kChunk, c = i / kChunk, id = cand[q * PC + c];
    const int rank = stable_rank(c, E, mass + q * PC);
    if (rank >= M) continue;
    sel[q * PC + rank] = (int16_t)id;
    slots[q * PC + rank] = mass[q * PC + c];
    atomicOr(&picked[q][id >> 5], 1u << (id & 31));
  }
  __syncthreads();
  // den = butterfly over the slots of the selected masses (a wave per query).
  for (int q = w; q < nq; q += kReadThreads / 64) {
    int width = 1;
    while (width < M) width <<= 1;
    float v[kMaxCand / 64];
#pragma unroll
    for (int k = 0; k < kMaxCand / 64; ++k)
      v[k] = lane + 64 * k < M ? slots[q * PC + lane + 64 * k] : 0.0f;
    for (int half = width / 2; half >= 64; half >>= 1)
#pragma unroll
      for (int k = 0; k < kMaxCand / 128; ++k)
        if (k < half / 64) v[k] = v[k] + v[k + half / 64 < kMaxCand / 64 ? k + half / 64 : k];
    const float total = wave_fold(v[0]);
    if (lane == 0) den[q] = total;
    if (sel_out)
      for (int m = lane; m < p.sel_cap; m += 64)
        sel_out[(size_t)q * p.H * p.sel_cap + m] = m < M ? sel[q * PC + m] : -1;
  }

  // Reads: num = sum over fines of ch C, coarse = sum over pages of (h cw) PC.
  constexpr int TW = D / 64;                           // 16-column tiles a wave
  const int k4 = lane >> 4, col = lane & 15;
  f32x4 num[TW] = {}, co[TW] = {};
  int buf = 0;
  auto product = [&](const float* c, f32x4 (&acc)[TW]) __attribute__((always_inline)) {
    const float* row = ch + buf * kChunk * HP + col * HP + k4;
    const float* cp = c + (size_t)k4 * D + 16 * TW * w + col;
#pragma unroll 16
    for (int s = 0; s < D / 4; ++s)
#pragma unroll
      for (int j = 0; j < TW; ++j)
        acc[j] = mfma16(row[4 * s], cp[(size_t)4 * s * D + 16 * j], acc[j]);
  };
  // Two row buffers: a buffer is written again only after the barrier of the
  // other's product, which every wave reaches when it is done with this one.
  for (int id = 0; id < visible; ++id) {
    uint32_t any = 0;
#pragma unroll
    for (int q = 0; q < kChunk; ++q) any |= picked[q][id >> 5];
    if (!(any >> (id & 31) & 1u)) continue;            // workgroup-uniform
    const float* sw = sw_row(id);
    const float* pg = pw + (id / kGroup) * D;
    float* dst = ch + buf * kChunk * HP;
    for (int i = tid; i < kChunk * D; i += kReadThreads) {
      const int q = i / D, d = i % D;
      const bool on = picked[q][id >> 5] >> (id & 31) & 1u;
      dst[q * HP + d] = on ? (hs[q * HP + d] * pg[d]) * sw[d] : 0.0f;
    }
    __syncthreads();
    product(p.bank + (bh * p.S + id) * D * D, num);
    buf ^= 1;
  }
  if (coarse_on) {
    for (int pg = 0; pg < completed; ++pg) {
      float* dst = ch + buf * kChunk * HP;
      for (int i = tid; i < kChunk * D; i += kReadThreads) {
        const int q = i / D, d = i % D;
        dst[q * HP + d] = hs[q * HP + d] * cw[pg * D + d];
      }
      __syncthreads();
      product(p.pc + (bh * p.Pc + pg) * D * D, co);
      buf ^= 1;
    }
  }
  // A query that did not select a fine of the union has rows of 0 against its
  // matrix, and 0 times an infinite or NaN entry is NaN. A NaN outlives the
  // sums, so a query that holds one sums its own fines again.
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < TW; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (num[j][r] != num[j][r]) mine |= 1u << (4 * k4 + r);
  if (mine) atomicOr(&bad, mine);
  __syncthreads();                                     // den, bad
  for (uint32_t left = bad; left; left &= left - 1) {
    const int q = __builtin_ctz(left);
    float sum[TW] = {};
    for (int m = 0; q < nq && m < M; ++m) {
      const int id = sel[q * PC + m];
      const float* sw = sw_row(id);
      const float* pg = pw + (id / kGroup) * D;
      const float* c = p.bank + (bh * p.S + id) * D * D + 16 * TW * w + col;
      for (int d = k4; d < D; d += 4) {
        const float x = (hs[q * HP + d] * pg[d]) * sw[d];
#pragma unroll
        for (int j = 0; j < TW; ++j) sum[j] = fmaf(x, c[(size_t)d * D + 16 * j], sum[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < TW; ++j) {
      sum[j] += __shfl_xor(sum[j], 16);
      sum[j] += __shfl_xor(sum[j], 32);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * k4 + r == q) num[j][r] = sum[j];
    }
  }

  // _fuse_training at fp32 (operator.py:21-38); both history branches
  // present only with coarse values past first_coarse.
  const float bias = coarse_on ? kLogTwoF32 : 0.0f;
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    const int d = 16 * (TW * w + j) + col;
    float a[3], fb[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      a[i] = load_param(p.fa, p.f_dtype, h * p.fa_s[0] + d * p.fa_s[1] + i * p.fa_s[2]);
      fb[i] = load_param(p.fb, p.f_dtype, h * p.fb_s[0] + d * p.fb_s[1] + i * p.fb_s[2]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int q = 4 * k4 + r;
      if (q >= nq) continue;
      const float x = ld(p.rq, b, t0 + q, h, d);
      const float loc = local[(size_t)q * p.H * D + d];
      float s[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) s[i] = (a[i] * x) + fb[i];
      s[0] = s[0] + bias;
      if (!coarse_on) s[1] = -__builtin_inff();
      const float top3 = fmaxf(s[0], fmaxf(s[1], s[2]));
      const float e0 = exp_cr(s[0] - top3);
      const float e1 = coarse_on ? exp_cr(s[1] - top3) : 0.0f;
      const float e2 = exp_cr(s[2] - top3);
      const float tot = (e0 + e2) + e1;   // butterfly order over [e0, e1, e2, 0]
      const float r0 = e0 / tot, r1 = e1 / tot, r2 = e2 / tot;
      const float lt = r0 * (2.0f * loc);
      const float ct = r1 * (p.gain * co[j][r]);
      const float ft = r2 * (p.gain * (num[j][r] / den[q]));
      out[q * p.out_st + d] = (lt + ct) + ft;
    }
  }
}

}  // namespace

size_t f32_workspace_floats(int B, int H, int D, int64_t T, int coarse_values) {
  const int64_t tiles = (T + kFine - 1) / kFine;
  const int64_t S = tiles > 3 ? tiles - 3 : 0;
  const int64_t P8 = (S + kGroup - 1) / kGroup;
  const int64_t Pc = coarse_values ? S / kGroup : 0;
  const int64_t bh = (int64_t)B * H;
  auto align = [](int64_t n) { return (n + 63) & ~(int64_t)63; };
  return (size_t)(align(bh * T * D) + align(bh * S * D) + align(bh * S * D * D) +
                  align(bh * P8 * kGroup * D) + align(bh * P8 * kRowsPerPage * D) +
                  align(bh * Pc * D * D));
}

int f32_layout(F32Params& p, float* ws, int64_t T, int coarse_values) {
  const int64_t tiles = (T + kFine - 1) / kFine;
  p.S = (int)(tiles > 3 ? tiles - 3 : 0);
  p.P8 = (p.S + kGroup - 1) / kGroup;
  p.Pc = coarse_values ? p.S / kGroup : 0;
  p.T = (int)T;
  p.coarse_values = coarse_values;
  const int64_t bh = (int64_t)p.B * p.H;
  const int D = p.D;
  auto align = [](int64_t n) { return (n + 63) & ~(int64_t)63; };
  float* cur = ws;
  p.local = cur; cur += align(bh * T * D);
  p.fine_z = cur; cur += align(bh * p.S * D);
  p.bank = cur; cur += align(bh * (int64_t)p.S * D * D);
  p.pz = cur; cur += align(bh * p.P8 * kGroup * D);
  p.swt = cur; cur += align(bh * p.P8 * kRowsPerPage * D);
  p.pc = coarse_values && p.Pc ? cur : nullptr;
  return 0;
}

int f32_limits(const tao_stream_cfg& cfg, int64_t T, int64_t* pages, int64_t* cand) {
  const int64_t tiles = (T + kFine - 1) / kFine;
  const int64_t vmax = tiles > 3 ? tiles - 3 : 0;
  int64_t coarse = 0, elig = 0, sel = 0;
  if (vmax) sched::routed_counts(cfg, vmax / kGroup, vmax % kGroup, &coarse, &elig, &sel);
  *pages = vmax / kGroup + (vmax % kGroup > 0);
  *cand = coarse * kGroup + kGroup - 1;
  return *pages <= kMaxPages && *cand <= kMaxCand && sel <= kMaxCand;
}

namespace {

template <int D>
hipError_t launch_d(const F32Params& p, hipStream_t s, bool own_local) {
  auto grid = [&](int64_t x) { return dim3((unsigned)x, (unsigned)p.H, (unsigned)p.B); };
  const int64_t writers = (int64_t)p.S * (D / 32), tiles = own_local ? (p.T + 31) / 32 : 0;
  if (writers + tiles)
    hipLaunchKernelGGL(f32_front_kernel<D>, dim3((unsigned)((writers + tiles) * p.B * p.H)),
                       dim3(64 * kLocalWaves), 0, s, p, rows_aligned(p.q) && rows_aligned(p.k),
                       (int)writers);
  if (p.S) hipLaunchKernelGGL(f32_pages_kernel<D>, grid((int64_t)p.P8 * kGroup), dim3(256), 0, s, p);
  int64_t pages = 0, cand = 0;
  f32_limits(p.cfg, p.T, &pages, &cand);
  // Rows of an odd number of 4-byte words: a column of them spreads over the
  // banks.
  const F32ReadLds lds{(int)(pages ? pages : 1), (int)(cand < pages ? pages : cand) | 1};
  const size_t bytes = lds.floats(D) * sizeof(float);
  if (bytes > 60 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)f32_read_kernel<D>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(f32_read_kernel<D>, grid((p.T + kChunk - 1) / kChunk), dim3(kReadThreads),
                     bytes, s, p, lds);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_full_f32(const F32Params& p, hipStream_t s, bool own_local) {
  if (p.D == 64) return launch_d<64>(p, s, own_local);
  if (p.D == 128) return launch_d<128>(p, s, own_local);
  return hipErrorInvalidValue;
}

}  // namespace tao

namespace {

int f32_fail(int code, const char* msg) {
  tao::set_error(msg);
  return code;
}

tao::F32View f32_view(const void* p, const int64_t* s) {
  tao::F32View v;
  v.p = (const float*)p;
  v.sb = s[0];
  v.st = s[1];
  v.sh = s[2];
  return v;
}

}  // namespace

extern "C" {

size_t tao_full_sequence_f32_workspace_bytes(int32_t batch, int32_t heads, int32_t head_dim,
                                             int64_t tokens, int32_t coarse_values) {
  if (batch <= 0 || heads <= 0 || tokens < 0 || (head_dim != 64 && head_dim != 128)) return 0;
  return tao::f32_workspace_floats(batch, heads, head_dim, tokens, coarse_values ? 1 : 0) *
         sizeof(float);
}

}  // extern "C"

namespace {

// tao_full_sequence_f32 and tao_full_sequence_f32_local: local null computes
// the local attention, else the read takes it from `local`.
int full_f32(const tao_stream_cfg* cfg, const tao_tokens* tok, const tao_fusion* fu,
             int32_t batch, int32_t heads, int32_t head_dim, int32_t coarse_values,
             const void* local, void* out, const int64_t* out_s, int32_t* sel_out,
             int32_t sel_cap, void* workspace, size_t workspace_bytes, void* stream) {
  if (!cfg || !tok || !fu || !out || !out_s || !workspace)
    return f32_fail(TAO_E_ARGUMENT, "null fp32 full-sequence argument");
  if (!tok->q || !tok->k || !tok->v || !tok->raw_q || !tok->raw_k)
    return f32_fail(TAO_E_ARGUMENT, "null token operand");
  if (!fu->fusion_a || !fu->fusion_b ||
      (fu->dtype != TAO_BF16 && fu->dtype != TAO_FP32 && fu->dtype != TAO_FP16))
    return f32_fail(TAO_E_ARGUMENT, "invalid fusion parameters");
  if (cfg->fine_tokens != 256 || cfg->local_keep != 512 || cfg->coarse_group != 8)
    return f32_fail(TAO_E_ARGUMENT, "the fp32 read implements fine_tokens=256, local_keep=512, "
                                    "coarse_group=8");
  if (head_dim != 64 && head_dim != 128)
    return f32_fail(TAO_E_SHAPE, "head_dim must be 64 or 128");
  if (batch <= 0 || heads <= 0 || tok->tokens < 0)
    return f32_fail(TAO_E_SHAPE, "batch, heads and tokens must be positive");
  const int64_t T = tok->tokens;
  if (T == 0) return TAO_OK;
  if (T > (int64_t)1 << 30) return f32_fail(TAO_E_SHAPE, "sequence too long");
  int64_t pages = 0, cand = 0;
  if (!tao::f32_limits(*cfg, T, &pages, &cand))
    return f32_fail(TAO_E_CAPACITY, "the fp32 read holds at most 64 pages and 256 route "
                                    "candidates per query (sequence too long)");
  const size_t need = tao::f32_workspace_floats(batch, heads, head_dim, T, coarse_values ? 1 : 0) *
                      sizeof(float);
  if (sel_out && sel_cap <= 0) return f32_fail(TAO_E_ARGUMENT, "sel_out needs sel_cap > 0");
  if (workspace_bytes < need)
    return f32_fail(TAO_E_WORKSPACE, "workspace smaller than "
                                     "tao_full_sequence_f32_workspace_bytes()");
  tao::F32Params p{};
  p.q = f32_view(tok->q, tok->q_s);
  p.k = f32_view(tok->k, tok->k_s);
  p.v = f32_view(tok->v, tok->v_s);
  p.rq = f32_view(tok->raw_q, tok->rq_s);
  p.rk = f32_view(tok->raw_k, tok->rk_s);
  p.fa = fu->fusion_a;
  p.fb = fu->fusion_b;
  p.f_dtype = fu->dtype;
  for (int i = 0; i < 3; ++i) { p.fa_s[i] = fu->a_s[i]; p.fb_s[i] = fu->b_s[i]; }
  p.gain = fu->gain;
  p.out = (float*)out;
  p.out_sb = out_s[0];
  p.out_st = out_s[1];
  p.out_sh = out_s[2];
  p.sel_out = sel_out;
  p.sel_cap = sel_out ? sel_cap : 0;
  p.cfg = *cfg;
  p.B = batch;
  p.H = heads;
  p.D = head_dim;
  tao::f32_layout(p, (float*)workspace, T, coarse_values ? 1 : 0);
  if (local) p.local = const_cast<float*>((const float*)local);   // read only
  const hipError_t e = tao::launch_full_f32(p, (hipStream_t)stream, local == nullptr);
  if (e != hipSuccess) return f32_fail((int)e, hipGetErrorString(e));
  return TAO_OK;
}

}  // namespace

extern "C" {

int tao_full_sequence_f32(const tao_stream_cfg* cfg, const tao_tokens* tok, const tao_fusion* fu,
                          int32_t batch, int32_t heads, int32_t head_dim, int32_t coarse_values,
                          void* out, const int64_t* out_s, int32_t* sel_out, int32_t sel_cap,
                          void* workspace, size_t workspace_bytes, void* stream) {
  return full_f32(cfg, tok, fu, batch, heads, head_dim, coarse_values, nullptr, out, out_s,
                  sel_out, sel_cap, workspace, workspace_bytes, stream);
}

int tao_full_sequence_f32_local(const tao_stream_cfg* cfg, const tao_tokens* tok,
                                const tao_fusion* fu, int32_t batch, int32_t heads,
                                int32_t head_dim, int32_t coarse_values, const void* local,
                                void* out, const int64_t* out_s, int32_t* sel_out,
                                int32_t sel_cap, void* workspace, size_t workspace_bytes,
                                void* stream) {
  if (!local) return f32_fail(TAO_E_ARGUMENT, "null local attention output");
  return full_f32(cfg, tok, fu, batch, heads, head_dim, coarse_values, local, out, out_s,
                  sel_out, sel_cap, workspace, workspace_bytes, stream);
}

}  // extern "C"
