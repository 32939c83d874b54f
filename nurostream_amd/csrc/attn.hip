// The step either side of the MoE FFN in a GPT-OSS decode token (gfx950):
// YaRN rotary embedding + KV-cache append, and sink attention with the
// alternating sliding window, for one query token.
//
// Semantics follow the reference's model/gpt_oss.py: yarn_tables (42-58),
// the attention block (101-114) and sink_attention (73-85); compute in fp32
// like its torch path. The position of the token is read from device memory
// (`pos`), so a captured graph of a whole decode token can be replayed token
// after token; nsx_pos_advance moves it on inside the graph.
//
// KV cache layout: K and V each [n_kv][ctx_max][head_dim] fp32.
// Attention is split over the keys (one workgroup per kv head and split, each
// handling the kv head's n_rep query heads), and a combine kernel merges the
// splits together with the sink; a layer whose keys always fit one workgroup
// (a 128-key sliding window) finishes in the split kernel.
// Both grids are sized for ctx_max, so their shape does not depend on the
// position; each workgroup takes its share of the keys up to it.
#include "nsx_common.h"

#include <algorithm>
#include <type_traits>
#include <math.h>

namespace {

constexpr int ATTN_D = 64;        // head_dim (GPT-OSS)
constexpr int ATTN_TILE = 16;     // keys per wave and matrix-core step
constexpr int ATTN_NW = 4;        // waves of a split's workgroup
constexpr int ATTN_FINAL_NW = 8;  // waves of the only workgroup of a kv head: a tile each at 128 keys
constexpr int ATTN_FINAL_KEYS = 128;  // up to this many keys one workgroup per kv head does everything
constexpr int ATTN_MAX_REP = 16;  // query heads per kv head (columns of the matrix-core step)
// Splits of a kv head's keys: enough workgroups for two on each of the 256 CUs, at most what the combine
// kernel's lanes hold, and none shorter than a tile per wave.
constexpr int ATTN_MAX_SPLIT = 128;
constexpr int ATTN_GRID = 512;
// A running maximum's start. Finite, not -infinity: keys that all score -infinity (overflowed scores) then get weight
// e^-infinity = 0 beside it, where the difference of two infinities would make the head NaN.
constexpr float ATTN_LOWEST = -3.4028235e38f;

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Rotary of element d of a 64-element head row at position p: x = the
// element, partner = element d ^ 32 (both with bias), rotate_half pairing
// (gpt_oss.py:42-58, ops.py:95-104). Explicit fmaf so that every kernel that
// applies it rounds the same way.
__device__ __forceinline__ float rope_elem(float x, float partner, int d, int p, const float* __restrict__ inv_freq,
                                           float amp) {
  const float ang = (float)p * inv_freq[d & (ATTN_D / 2 - 1)];  // fp32, as positions.float() * inv
  float s, c;
  sincosf(ang, &s, &c);
  c *= amp;
  s *= amp;
  const float ps = partner * s;
  return d < ATTN_D / 2 ? fmaf(x, c, -ps) : fmaf(x, c, ps);
}

// The same for the pair (element d < 32, element d + 32): one sine and cosine serve both.
__device__ __forceinline__ void rope_pair(float& x0, float& x1, int p, float inv_freq, float amp) {
  const float ang = (float)p * inv_freq;
  float s, c;
  sincosf(ang, &s, &c);
  c *= amp;
  s *= amp;
  const float y0 = fmaf(x0, c, -(x1 * s));
  x1 = fmaf(x1, c, x0 * s);
  x0 = y0;
}

// One wave per row of the q | k | v block: bias, then rotary for q and k
// rows; k and v rows go into the cache at the token's position.
__global__ __launch_bounds__(64) void rope_kv_append_kernel(
    float* __restrict__ qkv, const float* __restrict__ bq, const float* __restrict__ bk,
    const float* __restrict__ bv, int n_head, int n_kv, const float* __restrict__ inv_freq, float amp,
    const int32_t* __restrict__ pos_ptr, float* __restrict__ k_cache, float* __restrict__ v_cache,
    int64_t ctx_max) {
  const int r = blockIdx.x, lane = threadIdx.x;
  const int p = *pos_ptr;
  if (p < 0 || p >= ctx_max) return;  // the host keeps p < ctx_max; never write outside the cache
  float x = qkv[(int64_t)r * ATTN_D + lane];
  if (r < n_head) {
    if (bq) x += bq[(int64_t)r * ATTN_D + lane];
  } else if (r < n_head + n_kv) {
    if (bk) x += bk[(int64_t)(r - n_head) * ATTN_D + lane];
  } else {
    if (bv) x += bv[(int64_t)(r - n_head - n_kv) * ATTN_D + lane];
    const int g = r - n_head - n_kv;
    v_cache[((int64_t)g * ctx_max + p) * ATTN_D + lane] = x;
    return;
  }
  const float y = rope_elem(x, __shfl_xor(x, ATTN_D / 2, 64), lane, p, inv_freq, amp);
  if (r < n_head) {
    qkv[(int64_t)r * ATTN_D + lane] = y;
  } else {
    const int g = r - n_head;
    k_cache[((int64_t)g * ctx_max + p) * ATTN_D + lane] = y;
  }
}

__device__ __forceinline__ void attn_span(int p, int window, int& lo, int& total) {
  lo = window > 0 ? max(0, p + 1 - window) : 0;
  total = p + 1 - lo;
}

// Keys per split: the token's keys in equal parts, whole tiles for each of the workgroup's waves.
__device__ __forceinline__ int attn_per(int total, int nsplit, int nw) {
  const int step = ATTN_TILE * nw;
  return ((total + nsplit - 1) / nsplit + step - 1) / step * step;
}

// Workgroup (kv head g, split c): the attention of the kv head's n_rep query
// heads over the split's keys. The token's keys are cut into gridDim.y splits
// of equal length (a multiple of one ATTN_TILE per wave), so the number of
// partials to merge does not grow with the history; splits past the current
// length return at once.
//
// Wave w takes key tiles w, w + NW, ... of the split and multiplies them by
// all query heads at once with v_mfma_f32_16x16x4_f32 (exact fp32 products
// and sums), so every key and value row is loaded once, by one wave:
//   scores: A = the tile's 16 keys x 4 dimensions, B = 4 dimensions x 16
//     query heads. Lane l holds key l % 16 and, of every 16 dimensions, the
//     four from 4 (l / 16): a 16-byte load serves four instructions. D: lane l
//     holds query head l % 16 and keys 4 (l / 16) .. + 3.
//   values: the D layout of the scores is the B layout of the next product (4
//     keys x 16 heads) when instruction r takes keys r, 4 + r, 8 + r, 12 + r;
//     A = 16 dimensions x those keys, lane l key 4 (l / 16) + r, dimensions
//     4 (l % 16) .. + 3, one per instruction: coalesced 16-byte loads. D of
//     instruction dt: lane l holds head l % 16, dimensions 16 (l / 16) + 4 i + dt.
// A running softmax per head in registers (maximum over the four lane groups
// by two shuffles), the next tile's rows in flight during a tile's products.
// The waves are merged in wave order through LDS.
//
// Bound: the cache rows (67 MB for 8 kv heads x 16384 keys: 10 us at the card's read rate); the
// products take 1024 cycles of a SIMD's matrix core per tile, about a third of that. Measured at 64 / 8
// heads, 16384 keys: 17.2 us (3.9 TB/s) against 33 for a kernel whose four waves each loaded every key row
// and multiplied on the VALU; 128 keys in one workgroup 6.9 us against 12.7. A second tile in flight per
// wave: 20.5 against 19.1 us for the call, so one.
//
// part: for query head h and split c the values acc[ATTN_D] at (h * nsplit +
// c) * ATTN_D, and behind all of those (m, l) at (h * nsplit + c) * 2.
// FINAL (one split covers every position: a sliding window or a cache of at
// most ATTN_FINAL_KEYS keys): the workgroup also merges the sink and writes out[h].
// ROPE: q is the token's raw q | k | v block; each workgroup adds the bias
// and applies the rotary to its query heads itself. The workgroup whose split
// holds the token's position does the same for the token's k row, adds v's
// bias and appends both to the cache; its own products take the two rows from
// LDS (no other workgroup reads them), so no separate rotary + append launch is needed.
struct RopeArgs {
  const float *bq, *bk, *bv, *inv_freq;
  float amp;
};

// rows of one key tile in a wave's registers
struct AttnTile {
  v4f k[ATTN_D / 16], v[4];
};

__device__ __forceinline__ void attn_lds_barrier() {  // LDS writes visible; the tile loads stay in flight
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <bool FINAL, bool ROPE, int NW>
__global__ __launch_bounds__(64 * NW) void attn_split_kernel(
    const float* __restrict__ q, float* __restrict__ k_cache, float* __restrict__ v_cache,
    const int32_t* __restrict__ pos_ptr, int64_t ctx_max, int window, float scale, int n_rep, int n_head, int nsplit,
    float* __restrict__ part, const float* __restrict__ sinks, float* __restrict__ out, RopeArgs ra) {
  constexpr int NT = 64 * NW, HALF = ATTN_D / 2;
  constexpr int PAIRS = (ATTN_MAX_REP * HALF + NT - 1) / NT;  // (d, d + 32) pairs of the query heads per thread
  __shared__ __align__(16) float qs[ATTN_MAX_REP][ATTN_D + 4];
  __shared__ __align__(16) float own[2][ATTN_D];  // the token's k and v rows
  __shared__ float sm[NW][ATTN_MAX_REP], sl[NW][ATTN_MAX_REP];
  __shared__ __align__(16) float sacc[NW][ATTN_MAX_REP][ATTN_D];
  const int g = blockIdx.x, c = blockIdx.y, t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, i16 = lane & 15, kq = lane >> 4;
  // loads that do not depend on the position go out first
  float x0[PAIRS], x1[PAIRS], fr[PAIRS], b0[PAIRS] = {}, b1[PAIRS] = {};
#pragma unroll
  for (int u = 0; u < PAIRS; ++u) {
    const int i = min(t + u * NT, n_rep * HALF - 1);
    const int64_t at = ((int64_t)g * n_rep + i / HALF) * ATTN_D + i % HALF;
    x0[u] = q[at];
    x1[u] = q[at + HALF];
    if constexpr (ROPE) {
      fr[u] = ra.inv_freq[i % HALF];
      if (ra.bq) {
        b0[u] = ra.bq[at];
        b1[u] = ra.bq[at + HALF];
      }
    }
  }
  float n0 = 0.f, n1 = 0.f, nf = 0.f;  // threads 0..31: the token's k pair; 64..127: its v element
  if constexpr (ROPE) {
    static_assert(NT >= 128, "the token's own rows take two waves");
    if (t < HALF) {
      const float* kr = q + ((int64_t)n_head + g) * ATTN_D;
      n0 = kr[t];
      n1 = kr[t + HALF];
      nf = ra.inv_freq[t];
      if (ra.bk) {
        n0 += ra.bk[(int64_t)g * ATTN_D + t];
        n1 += ra.bk[(int64_t)g * ATTN_D + t + HALF];
      }
    } else if (t >= 64 && t < 128) {
      n0 = q[((int64_t)n_head + n_head / n_rep + g) * ATTN_D + t - 64];  // v rows follow the n_kv k rows
      if (ra.bv) n0 += ra.bv[(int64_t)g * ATTN_D + t - 64];
    }
  }
  const int p = *pos_ptr;
  if (p < 0 || p >= ctx_max) return;
  int lo, total;
  attn_span(p, window, lo, total);
  const int per = attn_per(total, FINAL ? 1 : nsplit, NW);
  const int k0 = c * per;
  if (k0 >= total) return;  // past the current length
  const int nk = min(per, total - k0), ntile = (nk + ATTN_TILE - 1) / ATTN_TILE;
  const int rel = k0 + nk == total ? nk - 1 : -1;  // ROPE: the token's own key in this split
  const float* kb = k_cache + ((int64_t)g * ctx_max + lo + k0) * ATTN_D + 4 * kq;
  const float* vb = v_cache + ((int64_t)g * ctx_max + lo + k0) * ATTN_D + 4 * i16;
  // a tile's rows; rows past the split's keys are clamped to its last key and get weight 0
  auto load = [&](int tile, AttnTile& T) {
    const int r0 = tile * ATTN_TILE;
    const float* kr = kb + (int64_t)min(r0 + i16, nk - 1) * ATTN_D;
#pragma unroll
    for (int j = 0; j < ATTN_D / 16; ++j) T.k[j] = *(const v4f*)(kr + 16 * j);
#pragma unroll
    for (int r = 0; r < 4; ++r) T.v[r] = *(const v4f*)(vb + (int64_t)min(r0 + 4 * kq + r, nk - 1) * ATTN_D);
  };
  AttnTile T[2];
  load(min(wave, ntile - 1), T[0]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < PAIRS; ++u) {
    const int i = t + u * NT;
    if (i >= n_rep * HALF) break;
    float y0 = x0[u], y1 = x1[u];
    if constexpr (ROPE) {
      if (ra.bq) {
        y0 += b0[u];
        y1 += b1[u];
      }
      rope_pair(y0, y1, p, fr[u], ra.amp);
    }
    qs[i / HALF][i % HALF] = y0;
    qs[i / HALF][i % HALF + HALF] = y1;
  }
  if constexpr (ROPE) {
    if (rel >= 0) {
      const int64_t at = ((int64_t)g * ctx_max + p) * ATTN_D;
      if (t < HALF) {
        rope_pair(n0, n1, p, nf, ra.amp);
        own[0][t] = n0;
        own[0][t + HALF] = n1;
        k_cache[at + t] = n0;
        k_cache[at + t + HALF] = n1;
      } else if (t >= 64 && t < 128) {
        own[1][t - 64] = n0;
        v_cache[at + t - 64] = n0;
      }
    }
  }
  attn_lds_barrier();
  v4f qr[ATTN_D / 16];  // query head i16 (heads past n_rep repeat the last and are not stored)
#pragma unroll
  for (int j = 0; j < ATTN_D / 16; ++j) qr[j] = *(const v4f*)&qs[min(i16, n_rep - 1)][16 * j + 4 * kq];
  float m = ATTN_LOWEST, l = 0.f;
  v4f acc[4] = {};
  auto step = [&](int tile, AttnTile& cur) {
    const int r0 = tile * ATTN_TILE;
    if constexpr (ROPE) {
      if (rel >= r0 && rel < r0 + ATTN_TILE) {  // the token's own rows, which this launch appends
        if (r0 + i16 == rel) {
#pragma unroll
          for (int j = 0; j < ATTN_D / 16; ++j) cur.k[j] = *(const v4f*)&own[0][16 * j + 4 * kq];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (min(r0 + 4 * kq + r, nk - 1) == rel) cur.v[r] = *(const v4f*)&own[1][4 * i16];
      }
    }
    v4f s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < ATTN_D / 16; ++j) {
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.k[j][e], qr[j][e], s, 0, 0, 0);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = r0 + 4 * kq + r < nk ? s[r] * scale : -INFINITY;
      mx = fmaxf(mx, s[r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    const float mn = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)));
    const float corr = expf(m - mn);  // (first tile: of nothing)
    m = mn;
    float ls = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = r0 + 4 * kq + r < nk ? expf(s[r] - mn) : 0.f;
      ls += s[r];
    }
    l = fmaf(l, corr, ls);  // this lane group's keys; the groups are added at the end
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) acc[dt] *= corr;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.v[r][dt], s[r], acc[dt], 0, 0, 0);
    }
  };
  for (int tile = wave; tile < ntile; tile += 2 * NW) {
    if (tile + NW < ntile) load(tile + NW, T[1]);
    __builtin_amdgcn_sched_barrier(0);
    step(tile, T[0]);
    if (tile + NW >= ntile) break;
    if (tile + 2 * NW < ntile) load(tile + 2 * NW, T[0]);
    __builtin_amdgcn_sched_barrier(0);
    step(tile + NW, T[1]);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (i16 < n_rep) {
    if (kq == 0) {
      sm[wave][i16] = m;
      sl[wave][i16] = l;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *(v4f*)&sacc[wave][i16][16 * kq + 4 * i] = v4f{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
  }
  attn_lds_barrier();
  for (int i = t; i < n_rep * ATTN_D; i += NT) {
    const int h = i / ATTN_D, d = i % ATTN_D, hq = g * n_rep + h;
    const float sink = FINAL && sinks ? sinks[hq] : -INFINITY;
    float M = sink;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, sm[w][h]);
    float Z = FINAL && sinks ? expf(sink - M) : 0.f, a = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {  // (a wave without a tile has weight 0)
      const float e = expf(sm[w][h] - M);
      Z = fmaf(e, sl[w][h], Z);
      a = fmaf(e, sacc[w][h][d], a);
    }
    if constexpr (FINAL) {
      out[(int64_t)hq * ATTN_D + d] = a / Z;
    } else {
      part[((int64_t)hq * nsplit + c) * ATTN_D + d] = a;
      if (d == 0) {
        float* ml = part + (int64_t)n_head * nsplit * ATTN_D + ((int64_t)hq * nsplit + c) * 2;
        ml[0] = M;
        ml[1] = Z;
      }
    }
  }
}

// One workgroup per query head: merge the live splits with the sink (softmax
// over [scores, sink], the sink column dropped). Every wave forms all the
// splits' weights (lane = split), then wave w sums the values of splits w,
// w + 4, ... (lane = dimension) with all its loads in flight, and the four
// sums meet in LDS: one round trip for (m, l), one for the values. Bound by
// those two and the launch; at 128 chunks in one serial loop the first version
// took 64 us, this one 4.0.
__global__ __launch_bounds__(256) void attn_combine_kernel(
    const float* __restrict__ part, const float* __restrict__ sinks, const int32_t* __restrict__ pos_ptr,
    int64_t ctx_max, int window, int n_head, int nsplit, int nw, float* __restrict__ out) {
  constexpr int LPS = ATTN_MAX_SPLIT / 64;  // splits per lane
  __shared__ float ws[ATTN_MAX_SPLIT];
  __shared__ float red[4][ATTN_D];
  const int h = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float* ml = part + ((int64_t)n_head * ATTN_D + 2 * h) * nsplit;  // (m, l) pairs; the workspace is 4-byte aligned
  const float sink = sinks ? sinks[h] : -INFINITY;
  const int p = *pos_ptr;
  if (p < 0 || p >= ctx_max) return;
  int lo, total;
  attn_span(p, window, lo, total);
  const int per = attn_per(total, nsplit, nw), nc = (total + per - 1) / per;  // 1 <= nc <= nsplit
  float2 v[LPS];
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const float* p2 = ml + 2 * min(lane + 64 * i, nc - 1);
    v[i] = float2{p2[0], p2[1]};
  }
  float M = sink;
#pragma unroll
  for (int i = 0; i < LPS; ++i) M = fmaxf(M, v[i].x);
  M = wave_max(M);
  float z = 0.f;
#pragma unroll
  for (int i = 0; i < LPS; ++i) {
    const float e = lane + 64 * i < nc ? expf(v[i].x - M) : 0.f;
    if (wave == 0) ws[lane + 64 * i] = e;
    z = lane + 64 * i < nc ? fmaf(e, v[i].y, z) : z;
  }
  const float Z = wave_sum(z) + (sinks ? expf(sink - M) : 0.f);
  __syncthreads();
  const float* pv = part + (int64_t)h * nsplit * ATTN_D + lane;
  float a = 0.f;
  for (int c0 = wave; c0 < nc; c0 += 4 * 16) {
    float x[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) x[u] = pv[(int64_t)min(c0 + 4 * u, nc - 1) * ATTN_D];
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (c0 + 4 * u < nc) a = fmaf(ws[c0 + 4 * u], x[u], a);
  }
  red[wave][lane] = a;
  __syncthreads();
  if (wave == 0) out[(int64_t)h * ATTN_D + lane] = ((red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane])) / Z;
}

__global__ void pos_advance_kernel(int32_t* pos, int32_t n) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *pos += n;
}

}  // namespace

static inline hipStream_t S(void* s) { return (hipStream_t)s; }

extern "C" int nsx_rope_kv_append(float* qkv, const float* q_bias, const float* k_bias, const float* v_bias,
                                  int n_head, int n_kv, int head_dim, const float* inv_freq, float amplitude,
                                  const int32_t* pos, float* k_cache, float* v_cache, int64_t ctx_max,
                                  void* stream) {
  NSX_REQUIRE(head_dim == ATTN_D, NSX_ENOTIMPL, "head_dim %d (the kernels are written for 64)", head_dim);
  NSX_REQUIRE(n_head > 0 && n_kv > 0 && n_head % n_kv == 0 && n_head / n_kv <= ATTN_MAX_REP, NSX_EINVAL,
              "n_head=%d, n_kv=%d: n_head must be a multiple of n_kv, at most %d per kv head", n_head, n_kv,
              ATTN_MAX_REP);
  NSX_REQUIRE(ctx_max > 0 && ctx_max < (1ll << 31), NSX_EINVAL, "ctx_max=%lld", (long long)ctx_max);
  NSX_REQUIRE(qkv && inv_freq && pos && k_cache && v_cache, NSX_EINVAL, "null buffer");
  hipLaunchKernelGGL(rope_kv_append_kernel, dim3(n_head + 2 * n_kv), dim3(64), 0, S(stream), qkv, q_bias, k_bias,
                     v_bias, n_head, n_kv, inv_freq, amplitude, pos, k_cache, v_cache, ctx_max);
  NSX_LAUNCHED();
  return NSX_OK;
}

// Splits per kv head for a cache of ctx_max rows (window bounds the keys when positive).
static int attn_splits(int n_kv, int64_t ctx_max, int window) {
  const int64_t keys = window > 0 ? std::min<int64_t>(ctx_max, window) : ctx_max;
  const int64_t fill = std::min<int64_t>(ATTN_MAX_SPLIT, nsx_cdiv(ATTN_GRID, n_kv));
  return (int)std::min<int64_t>(nsx_cdiv(keys, ATTN_TILE * ATTN_NW), fill);
}

extern "C" int64_t nsx_attn_workspace_bytes(int n_head, int head_dim, int64_t ctx_max) {
  if (head_dim != ATTN_D || n_head <= 0 || ctx_max <= 0) return -1;
  return (int64_t)n_head * attn_splits(1, ctx_max, 0) * (ATTN_D + 2) * (int64_t)sizeof(float);
}

// Checks shared by both attention entry points, then the split launch (and
// the combine unless one workgroup per kv head covers every position).
static int attn_launch(const float* q, float* k_cache, float* v_cache, const float* sinks, int n_head, int n_kv,
                       int head_dim, const int32_t* pos, int64_t ctx_max, int window, float scale,
                       void* workspace, float* out, bool rope, const RopeArgs& ra, hipStream_t st) {
  NSX_REQUIRE(head_dim == ATTN_D, NSX_ENOTIMPL, "head_dim %d (the kernels are written for 64)", head_dim);
  NSX_REQUIRE(n_head > 0 && n_kv > 0 && n_head % n_kv == 0 && n_head / n_kv <= ATTN_MAX_REP, NSX_EINVAL,
              "n_head=%d, n_kv=%d: n_head must be a multiple of n_kv, at most %d per kv head", n_head, n_kv,
              ATTN_MAX_REP);
  NSX_REQUIRE(ctx_max > 0 && ctx_max < (1ll << 31) && window >= 0, NSX_EINVAL, "ctx_max=%lld window=%d",
              (long long)ctx_max, window);
  NSX_REQUIRE(q && k_cache && v_cache && pos && workspace && out, NSX_EINVAL, "null buffer");
  NSX_REQUIRE(((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) % 16 == 0, NSX_EINVAL,
              "q, the caches and out must be 16-byte aligned");
  const int n_rep = n_head / n_kv, nsplit = attn_splits(n_kv, ctx_max, window);
  // a sliding window bounds the keys; up to ATTN_FINAL_KEYS of them one workgroup and no combine launch
  const bool final_ = std::min<int64_t>(ctx_max, window > 0 ? window : ctx_max) <= ATTN_FINAL_KEYS;
  auto split = [&](auto final_tag, auto rope_tag) {
    constexpr bool F = decltype(final_tag)::value;
    constexpr int NW = F ? ATTN_FINAL_NW : ATTN_NW;
    hipLaunchKernelGGL((attn_split_kernel<F, decltype(rope_tag)::value, NW>), dim3(n_kv, F ? 1 : nsplit),
                       dim3(64 * NW), 0, st, q, k_cache, v_cache, pos, ctx_max, window, scale, n_rep, n_head, nsplit,
                       (float*)workspace, sinks, out, ra);
  };
  auto by_rope = [&](auto final_tag) {
    if (rope) split(final_tag, std::true_type{});
    else split(final_tag, std::false_type{});
  };
  if (final_) {
    by_rope(std::true_type{});
    NSX_LAUNCHED();
    return NSX_OK;
  }
  by_rope(std::false_type{});
  NSX_LAUNCHED();
  hipLaunchKernelGGL(attn_combine_kernel, dim3(n_head), dim3(256), 0, st, (const float*)workspace, sinks, pos,
                     ctx_max, window, n_head, nsplit, ATTN_NW, out);
  NSX_LAUNCHED();
  return NSX_OK;
}

extern "C" int nsx_attn_decode(const float* q, const float* k_cache, const float* v_cache, const float* sinks,
                               int n_head, int n_kv, int head_dim, const int32_t* pos, int64_t ctx_max,
                               int window, float scale, void* workspace, float* out, void* stream) {
  // the caches are only read on this path
  return attn_launch(q, const_cast<float*>(k_cache), const_cast<float*>(v_cache), sinks, n_head, n_kv, head_dim,
                     pos, ctx_max, window, scale, workspace, out, false, RopeArgs{}, S(stream));
}

extern "C" int nsx_attn_decode_qkv(const float* qkv, const float* q_bias, const float* k_bias, const float* v_bias,
                                   const float* inv_freq, float amplitude, const float* sinks, int n_head, int n_kv,
                                   int head_dim, const int32_t* pos, float* k_cache, float* v_cache,
                                   int64_t ctx_max, int window, float scale, void* workspace, float* out,
                                   void* stream) {
  NSX_REQUIRE(inv_freq, NSX_EINVAL, "null inv_freq");
  return attn_launch(qkv, k_cache, v_cache, sinks, n_head, n_kv, head_dim, pos, ctx_max, window, scale, workspace,
                     out, true, RopeArgs{q_bias, k_bias, v_bias, inv_freq, amplitude}, S(stream));
}

extern "C" int nsx_pos_advance(int32_t* pos, int32_t n, void* stream) {
  NSX_REQUIRE(pos, NSX_EINVAL, "null position");
  hipLaunchKernelGGL(pos_advance_kernel, dim3(1), dim3(64), 0, S(stream), pos, n);
  NSX_LAUNCHED();
  return NSX_OK;
}
