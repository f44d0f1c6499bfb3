// The exact path: RoPE, the K/V write and decode attention over fp32 caches,
// each bit for bit with the reference's CPU forward (run.cpp:506-526 and
// 597-641), as the reference's GPTOSS_EXACT engine build runs them
// (getp-csrc/engine/gpu_engine.hpp:478-488: rope_exact, kv_write_kernel,
// attention_exact of getp-csrc/kernels/misc.hpp:55-85 and attention.hpp:18-83).
//
// Bits, not speed, set the design: every sum the CPU takes in order is taken
// in the same order here (a score's 64 products in fp64, the softmax sum over
// the positions and the sink in fp64, each output dim's weighted values with
// FMA in time order), with the CPU's rounding of every step (products rounded
// to fp32 before the fp64 add, fp32 <-> fp64 conversions where the CPU has
// them, glibc's expf). What runs in parallel is what the CPU computes
// independently: the positions' scores, their exponentials and quotients,
// the 64 output dims, the query heads.
//
// Attention: one workgroup per (sequence, kv head, chunk of hc query heads),
// `parts` waves per head. Bound by latency: chains whose order is the CPU's (a
// score's 64 fp64 adds, a head's n adds of the softmax sum, a dim's n FMAs), so
// each phase runs as many chains side by side as it has and keeps loads out of
// them:
//   scores   a wave takes 64 positions, a lane walks one position's K row, 16
//            dims fetched ahead, with up to eight heads' chains at once on it;
//   softmax  max, exponentials and quotients over the waves of a head; the
//            sum in order by one wave per head, its values made fp64 64 at a time;
//   output   a wave per head, lane = output dim, V rows through a 4-stage LDS
//            ring that the other waves fill.
// The scores stay in LDS, hc rows of n + 1 floats (hc is chosen on the host so
// they fit). Before, K and V went through one LDS tile for one wave per head,
// and the sum's values were fetched one by one: 32 sequences of 128 .. 2048
// tokens, 64 / 8 heads, 294 us, now 90 - 95 (the longest sequence's scores 35, sum 17,
// output 35). Short contexts keep that one-tile form: a kernel of its own where
// the host bound is short, a branch where only a row's own context is.
#include <algorithm>

#include "exact_math.hpp"
#include "gkv_device.hpp"
#include "lds_dma.hpp"

namespace gkv {

constexpr int kExactTile = 64;
constexpr int kExactRow = kHeadDim + 1; // LDS row of a staged position (short contexts), in floats
constexpr int kExactMaxWaves = 16;
// Contexts of up to this many positions take the one-tile form: there a row per
// lane, read by every head's waves, costs more than the chains it saves (32
// sequences on a 128-slot ring: 15.9 us against 19.7; 200 positions level; 600
// positions, 4 sequences: 68.7 us against 35.4).
constexpr int kExactShort = 192;
// Where one workgroup per CU does not hold the call (kExactTwo workgroups, 256
// CUs) and two fit a CU's LDS, the long form runs with 64 registers and a smaller
// V ring, two workgroups of 16 waves to a CU, or (past kExactFour) up to four of
// 8: their chains overlap each other's. 8 heads a workgroup, us, one-tile form / one
// to a CU / so: 512 workgroups of 1 .. 40 positions under a bound of 1024 12.5 / 24.3 / 12.0,
// of 1 .. 1000 161 / 88.8 / 94.5 (384), 1024 of 1 .. 500 under 1500 161 / 128 / 105, 4096 of
// 1 .. 40 under 1024 57 / 167 / 57, of 1 .. 500 under 1500 565 / 452 / 333.
// The one-tile form, of which a CU holds four (8 heads), stays ahead further up
// while that leaves it fewer rounds: to 256 positions with 257 .. 512 workgroups of
// five or more heads (384 of 1 .. 224 34.6 against 37.3, 512 of 200 each 40 - 42 against 38),
// to 300 with 513 .. 1024 of 5 to 8 (1024 of 200 each 58.5 against 69.5, 768 of 1 .. 300
// 58.1 against 69.7, 1024 of 300 level).
constexpr int kExactShortTwo = 256, kExactShortFour = 300;
constexpr int64_t kExactTwo = 256, kExactMany = 2 * 256, kExactFour = 4 * 256;

// Four floats at any float's alignment (the fp32 caches' rows).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct ExactAttnArgs {
  const float *q;
  int64_t q_stride;
  const float *kc, *vc;
  int slots, n_kv_heads, G, hc, n_chunks, window;
  int parts;                // waves per head
  int att_row;              // floats per score row (a multiple of 4)
  int v_early;              // the V ring has LDS of its own
  int v_rows;               // V rows per stage of the output's ring (16 per loading wave at most)
  int one_tile_n;           // rows of at most this many positions take the one-tile form
  const float *sinks;
  int pos;                  // every row's position (positions == nullptr)
  const int32_t *positions; // device [B], or nullptr
  int n_cap;                // positions attended at most (sizes the score rows)
  float *out;
  int64_t out_stride;
  uint32_t *dev_err;
};

// Scores of this lane's position (its K row at kr) for heads h0 .. h0 + NH - 1
// of the chunk: (float)((sum_i (double)(q_i * k_i)) / sqrt(64)), products rounded
// to fp32, the sum in order (the division by 8 is exact as a product). The
// heads' chains run side by side over the row (kWhole: fetched at once, else 16 dims
// ahead).
// Heads past the last one repeat it (the same value to the same place).
template <int NH, bool kWhole>
__device__ __forceinline__ void exact_scores(const float *kr, const float *qs, int h0, int hc,
                                             int j, int n, float *att, int att_row) {
  double s[NH];
  const float *q0[NH];
#pragma unroll
  for (int hh = 0; hh < NH; hh++) {
    s[hh] = 0.0;
    q0[hh] = qs + min(h0 + hh, hc - 1) * kHeadDim;
  }
  if constexpr (kWhole) { // the whole row at once: one round trip
    f32x4 k[16];
#pragma unroll
    for (int i = 0; i < 16; i++)
      k[i] = *(const f32x4u *)(kr + 4 * i);
#pragma unroll
    for (int i = 0; i < 16; i++)
#pragma unroll
      for (int hh = 0; hh < NH; hh++) {
        const f32x4 q = *(const f32x4 *)&q0[hh][4 * i];
#pragma unroll
        for (int e = 0; e < 4; e++)
          s[hh] = __dadd_rn(s[hh], (double)__fmul_rn(q[e], k[i][e]));
      }
  } else {
    f32x4 cur[4], nxt[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
      cur[i] = *(const f32x4u *)(kr + 4 * i);
#pragma unroll 1
    for (int d = 0; d < kHeadDim; d += 16) {
      const int dn = min(d + 16, kHeadDim - 16); // (the last round re-reads its own)
#pragma unroll
      for (int i = 0; i < 4; i++)
        nxt[i] = *(const f32x4u *)(kr + dn + 4 * i);
#pragma unroll
      for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int hh = 0; hh < NH; hh++) {
          const f32x4 q = *(const f32x4 *)&q0[hh][d + 4 * i];
#pragma unroll
          for (int e = 0; e < 4; e++)
            s[hh] = __dadd_rn(s[hh], (double)__fmul_rn(q[e], cur[i][e]));
        }
        __builtin_amdgcn_sched_barrier(0); // (no registers to fetch every query at once)
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
        cur[i] = nxt[i];
    }
  }
  if (j < n) {
#pragma unroll
    for (int hh = 0; hh < NH; hh++)
      att[min(h0 + hh, hc - 1) * att_row + j] = (float)__dmul_rn(s[hh], 0.125);
  }
}

// The one-tile form: a wave per head (waves past the hc heads only load; kAll:
// there are none), K and V through one LDS tile of 64 positions (65-float rows so
// that lane t reading row t meets no bank conflict).
template <bool kAll>
__device__ __forceinline__ void exact_one_tile(const ExactAttnArgs &a, float *lds, double *s_sum,
                                               int b, int g, int hq0, int t0, int n) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool head = kAll || wave < a.hc;
  const int hw = kAll ? wave : min(wave, a.hc - 1), h = hq0 + hw;
  const int kv_dim = a.n_kv_heads * kHeadDim;
  float *kt = lds;                                   // [64][65]
  float *qs = kt + kExactTile * kExactRow;           // [hc][64]
  float *att = qs + a.hc * kHeadDim + hw * (n + 1); // this head's scores
  const int ring = a.window; // a window layer's cache is a ring of window slots
  const float *kbase = a.kc + (int64_t)b * a.slots * kv_dim + (int64_t)g * kHeadDim;
  const float *vbase = a.vc + (int64_t)b * a.slots * kv_dim + (int64_t)g * kHeadDim;
  if (head)
    qs[hw * kHeadDim + lane] = a.q[(int64_t)b * a.q_stride + (int64_t)h * kHeadDim + lane];

  // scores: (float)((sum_i (double)(q_i * k_i)) / 8), products rounded to fp32
  const double scale = (double)__fsqrt_rn((float)kHeadDim);
  for (int tile = 0; tile < n; tile += kExactTile) {
    __syncthreads();
    for (int idx = threadIdx.x; idx < kExactTile * kHeadDim; idx += blockDim.x) {
      const int r = idx >> 6, c = idx & 63, j = tile + r;
      if (j < n) {
        const int t = t0 + j;
        const int slot = ring > 0 ? t % ring : t;
        kt[r * kExactRow + c] = kbase[(int64_t)slot * kv_dim + c];
      }
    }
    __syncthreads();
    const int j = tile + lane;
    if (head && j < n) {
      double s = 0.0;
      for (int i = 0; i < kHeadDim; i++)
        s = __dadd_rn(s, (double)__fmul_rn(qs[hw * kHeadDim + i], kt[lane * kExactRow + i]));
      att[j] = (float)__ddiv_rn(s, scale);
    }
  }
  if (head && lane == 0)
    att[n] = a.sinks[h];
  __syncthreads();

  // softmax over att[0..n] (run.cpp:335-353): the max (exact in any order),
  // expf((float)((double)x - max)), the fp64 sum in index order, the quotients
  if (head) {
    float m = -INFINITY;
    for (int j = lane; j <= n; j += 64)
      m = fmaxf(m, att[j]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
      m = fmaxf(m, __shfl_xor(m, off));
    const double md = (double)m;
    for (int j = lane; j <= n; j += 64)
      att[j] = expf_cpu_exact((float)__dsub_rn((double)att[j], md));
  }
  __syncthreads();
  if (head && lane == 0) {
    double s = 0.0;
#pragma unroll 8
    for (int j = 0; j <= n; j++)
      s = __dadd_rn(s, (double)att[j]);
    s_sum[hw] = s;
  }
  __syncthreads();
  if (head) {
    const double sum = s_sum[hw];
    for (int j = lane; j <= n; j += 64)
      att[j] = (float)__ddiv_rn((double)att[j], sum);
  }
  __syncthreads();

  // out[d] = fma(w_t, v_t[d], out[d]) over t in order; the V rows go through
  // the K tile's LDS, 64 positions at a time, read once for the hc heads
  float acc = 0.0f;
  for (int tile = 0; tile < n; tile += kExactTile) {
    __syncthreads();
    for (int idx = threadIdx.x; idx < kExactTile * kHeadDim; idx += blockDim.x) {
      const int r = idx >> 6, c = idx & 63, j = tile + r;
      if (j < n) {
        const int t = t0 + j;
        const int slot = ring > 0 ? t % ring : t;
        kt[r * kExactRow + c] = vbase[(int64_t)slot * kv_dim + c];
      }
    }
    __syncthreads();
    if (head) {
      const int m_t = min(kExactTile, n - tile);
      for (int r = 0; r < m_t; r++)
        acc = __fmaf_rn(att[tile + r], kt[r * kExactRow + lane], acc);
    }
  }
  if (head)
    a.out[(int64_t)b * a.out_stride + (int64_t)h * kHeadDim + lane] = acc;
}

// A workgroup's row: positions t0 .. t0 + n - 1, or false after zeros and the
// length flag for a position the cache cannot hold (full layer: p >= slots) or
// beyond the host bound (uniform per workgroup).
__device__ __forceinline__ bool exact_row(const ExactAttnArgs &a, int b, int hq0, int &t0, int &n) {
  const int p = a.positions ? a.positions[b] : a.pos;
  t0 = a.window > 0 ? max(0, p - a.window + 1) : 0;
  n = p - t0 + 1;
  if (p >= 0 && n <= a.n_cap && (a.window > 0 || p < a.slots))
    return true;
  for (int i = threadIdx.x; i < a.hc * kHeadDim; i += blockDim.x)
    a.out[(int64_t)b * a.out_stride + (int64_t)hq0 * kHeadDim + i] = 0.0f;
  if (threadIdx.x == 0 && a.dev_err)
    atomicOr(a.dev_err, GKV_DEVERR_LENGTH);
  return false;
}

__global__ __launch_bounds__(64 * kExactMaxWaves) void attention_exact_short_kernel(ExactAttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ double s_sum[kExactMaxWaves];
  const int b = blockIdx.x, g = blockIdx.y / a.n_chunks;
  const int hq0 = g * a.G + (blockIdx.y % a.n_chunks) * a.hc; // the chunk's first query head
  int t0, n;
  if (exact_row(a, b, hq0, t0, n))
    exact_one_tile<true>(a, lds, s_sum, b, g, hq0, t0, n);
}

// kLite: 64 registers, so that the waves of two workgroups of 16 or four of 8 fit a
// CU (the rule is in the host code).
template <bool kLite>
__global__ __launch_bounds__(64 * kExactMaxWaves)
__attribute__((amdgpu_waves_per_eu(kLite ? 8 : 4)))
void attention_exact_kernel(ExactAttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ double s_sum[kExactMaxWaves];
  __shared__ float s_max[kExactMaxWaves];
  const int b = blockIdx.x;
  const int g = blockIdx.y / a.n_chunks;
  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n_waves = blockDim.x >> 6; // hc * parts
  const int hc = a.hc;
  const int hq0 = g * a.G + (blockIdx.y % a.n_chunks) * hc; // the chunk's first query head
  const int kv_dim = a.n_kv_heads * kHeadDim;
  float *qs = lds;                  // [hc][64]
  float *att = qs + hc * kHeadDim;  // [hc][att_row]
  double *s_dbl = (double *)(att + hc * a.att_row); // [hc][2][64], then the V ring

  int t0, n;
  if (!exact_row(a, b, hq0, t0, n))
    return;
  if (n <= a.one_tile_n) { // (the host bound may be far above a row's own context)
    exact_one_tile<false>(a, lds, s_sum, b, g, hq0, t0, n);
    return;
  }
  // a window layer's cache is a ring of window slots (n <= ring: position j of
  // the n attended wraps at most once)
  const int ring = a.window, s0 = ring > 0 ? t0 % ring : 0;
  auto slot_of = [&](int j) { return ring > 0 && s0 + j >= ring ? s0 + j - ring : s0 + j; };
  const float *kbase = a.kc + (int64_t)b * a.slots * kv_dim + (int64_t)g * kHeadDim;
  const float *vbase = a.vc + (int64_t)b * a.slots * kv_dim + (int64_t)g * kHeadDim;
  // V ring of the output phase (its comment is there); where the LDS holds it
  // beside the sums' fp64 values, its first stages are fetched from the start.
  float *ring_v = (float *)(s_dbl + (a.v_early ? 128 * hc : 0));
  const int R = a.v_rows;
  const bool split = n_waves > hc;
  const int n_load = split ? n_waves - hc : n_waves, me = split ? wave - hc : wave;
  const int per = (R + n_load - 1) / n_load;
  auto issue = [&](int c) {
    if (me < 0)
      return;
    int r = min(me, R - 1);
    for (int i = 0; i < per; i++) {
      dma4(vbase + (int64_t)slot_of(min(c * R + r, n - 1)) * kv_dim + lane,
           ring_v + ((c & 3) * R + r) * kHeadDim);
      r = min(r + n_load, R - 1);
    }
  };
  if (a.v_early)
    for (int c = 0; c < 3; c++)
      issue(c);
  for (int i = threadIdx.x; i < hc * kHeadDim; i += blockDim.x)
    qs[i] = a.q[(int64_t)b * a.q_stride + (int64_t)hq0 * kHeadDim + i];
  if ((int)threadIdx.x < hc)
    att[threadIdx.x * a.att_row + n] = a.sinks[hq0 + threadIdx.x];
  __syncthreads();

  // Items of one 64-position tile and up to 8 heads, fewer heads where there
  // would be fewer items than waves (a window, a short context).
  const int tiles = (n + kExactTile - 1) / kExactTile;
  int hg = kLite ? 4 : 8;
  while (hg > 1 && tiles * ((hc + hg - 1) / hg) < n_waves)
    hg >>= 1;
  const int n_hg = (hc + hg - 1) / hg;
  for (int it = wave; it < tiles * n_hg; it += n_waves) {
    const int tile = it / n_hg, h = (it - tile * n_hg) * hg;
    const int j = tile * kExactTile + lane;
    const float *kr = kbase + (int64_t)slot_of(min(j, n - 1)) * kv_dim;
    const int nh = min(hg, hc - h);
    if (!kLite && nh > 4)
      exact_scores<8, false>(kr, qs, h, hc, j, n, att, a.att_row);
    else if (nh > 2)
      exact_scores<4, false>(kr, qs, h, hc, j, n, att, a.att_row);
    else if (nh == 2)
      exact_scores<2, !kLite>(kr, qs, h, hc, j, n, att, a.att_row);
    else
      exact_scores<1, !kLite>(kr, qs, h, hc, j, n, att, a.att_row);
  }
  __syncthreads();

  // softmax over att[0..n] (run.cpp:335-353): the max (exact in any order),
  // expf((float)((double)x - max)), the fp64 sum in index order, the quotients
  const int hl = wave % hc, part = wave / hc; // this wave's head and share
  float *row = att + hl * a.att_row;
  float m = -INFINITY;
  for (int j = part * 64 + lane; j <= n; j += 64 * a.parts)
    m = fmaxf(m, row[j]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    m = fmaxf(m, __shfl_xor(m, off));
  if (lane == 0)
    s_max[wave] = m;
  __syncthreads();
  for (int i = 0; i < a.parts; i++)
    m = fmaxf(m, s_max[hl + i * hc]);
  const double md = (double)m;
  for (int j = part * 64 + lane; j <= n; j += 64 * a.parts)
    row[j] = expf_cpu_exact((float)__dsub_rn((double)row[j], md));
  __syncthreads();
  if (part == 0) {
    // 64 values at a time become fp64 side by side and come back two per LDS
    // read, every lane adding them in order: the chain is the additions alone.
    // (Values past the sink are +0, which changes no sum of non-negatives.)
    double *sd = s_dbl + hl * 128;
    auto stage = [&](int c) {
      const int j = 64 * c + lane;
      sd[64 * (c & 1) + lane] = j <= n ? (double)row[j] : 0.0;
    };
    double s = 0.0;
    stage(0);
    for (int c = 0; 64 * c <= n; c++) {
      stage(c + 1);
      typedef double f64x2 __attribute__((ext_vector_type(2)));
      const f64x2 *x = (const f64x2 *)(sd + 64 * (c & 1));
      for (int k = 0; k < 32 && 64 * c + 2 * k <= n; k += 8) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const f64x2 v = x[k + i];
          s = __dadd_rn(s, v[0]);
          s = __dadd_rn(s, v[1]);
        }
      }
    }
    if (lane == 0)
      s_sum[hl] = s;
  }
  __syncthreads();
  // The quotients x / sum in fp64: with the correctly rounded reciprocal y, q =
  // x y and one correction q + y (x - q sum), the remainder exact by FMA, is
  // the correctly rounded quotient (Markstein, 1990). x in [0, 1] and sum in [1,
  // n + 1]: nothing over- or underflows; a NaN stays one.
  const double sum = s_sum[hl], y = __ddiv_rn(1.0, sum);
  for (int j = part * 64 + lane; j <= n; j += 64 * a.parts) {
    const double x = (double)row[j], q = __dmul_rn(x, y);
    row[j] = (float)__fma_rn(__fma_rn(-q, sum, x), y, q);
  }
  __syncthreads();

  // out[d] = fma(w_t, v_t[d], out[d]) over t in order: wave h < hc takes head h,
  // lane = output dim. The other waves (all, if there are no others) bring V
  // rows into a ring of 4 stages of R rows, row i of
  // a stage by loader i % n_load; rows past the last position re-read it, and
  // loaders short of a row repeat their stage's last, so every loader issues
  // `per` loads a stage and the wait for all but the two younger stages' (or
  // fewer) is enough.
  if (!a.v_early)
    for (int c = 0; c < 3; c++)
      issue(c);
  const float *w = att + min(wave, hc - 1) * a.att_row;
  float acc = 0.0f;
  for (int c = 0; c * R < n; c++) {
    if (per >= 16)
      wait_vmcnt<32>();
    else if (per >= 8)
      wait_vmcnt<16>();
    else if (per >= 4)
      wait_vmcnt<8>();
    else if (per >= 2)
      wait_vmcnt<4>();
    else
      wait_vmcnt<2>();
    lds_barrier(); // stage c is whole; every wave is done with stage c - 1
    issue(c + 3);
    if (wave >= hc)
      continue;
    const float *v = ring_v + (c & 3) * R * kHeadDim + lane;
    const int m_t = min(R, n - c * R);
    int r = 0;
    for (; r + 16 <= m_t; r += 16) {
#pragma unroll
      for (int e = 0; e < 16; e += 4) {
        const f32x4 x = *(const f32x4 *)&w[c * R + r + e];
#pragma unroll
        for (int i = 0; i < 4; i++)
          acc = __fmaf_rn(x[i], v[(r + e + i) * kHeadDim], acc);
      }
    }
    if (r + 8 <= m_t) {
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const f32x4 x = *(const f32x4 *)&w[c * R + r + e];
#pragma unroll
        for (int i = 0; i < 4; i++)
          acc = __fmaf_rn(x[i], v[(r + e + i) * kHeadDim], acc);
      }
      r += 8;
    }
    for (; r < m_t; r++)
      acc = __fmaf_rn(w[c * R + r], v[r * kHeadDim], acc);
  }
  wait_vmcnt<0>(); // no load may still write into LDS when the workgroup ends
  if (wave < hc)
    a.out[(int64_t)b * a.out_stride + (int64_t)(hq0 + wave) * kHeadDim + lane] = acc;
}

// run.cpp's apply_rotary_emb on heads 0..n_heads-1 of each row, in place.
__global__ __launch_bounds__(256) void rope_exact_kernel(float *qkv, int64_t row_stride,
                                                         const float *cos_tab,
                                                         const float *sin_tab,
                                                         const int32_t *positions, int n_heads) {
  const int b = blockIdx.x;
  constexpr int half = kHeadDim / 2;
  const int64_t p = positions ? positions[b] : 0;
  const float *cv = cos_tab + p * half, *sv = sin_tab + p * half;
  float *row = qkv + (int64_t)b * row_stride;
  for (int idx = threadIdx.x; idx < n_heads * half; idx += blockDim.x) {
    const int hh = idx / half, i = idx % half;
    float *x = row + hh * kHeadDim;
    const float x1 = x[i], x2 = x[half + i];
    x[i] = rope_first(x1, x2, cv[i], sv[i]);
    x[half + i] = rope_second(x1, x2, cv[i], sv[i]);
  }
}

// Each row's K and V (kv_dim floats each) into the fp32 caches at its slot.
__global__ __launch_bounds__(256) void kv_write_exact_kernel(
    const float *qkv, int64_t row_stride, int k_off, int v_off, float *kc, float *vc, int slots,
    int kv_dim, int slot, const int32_t *positions, int window, uint32_t *dev_err) {
  const int b = blockIdx.x;
  int s = slot;
  if (positions) {
    const int p = positions[b];
    s = p < 0 ? -1 : window > 0 ? p % window : p;
  }
  if (s < 0 || s >= slots) {
    if (threadIdx.x == 0 && dev_err)
      atomicOr(dev_err, GKV_DEVERR_LENGTH);
    return;
  }
  const float *row = qkv + (int64_t)b * row_stride;
  const int64_t dst = ((int64_t)b * slots + s) * kv_dim;
  for (int i = threadIdx.x; i < kv_dim; i += blockDim.x) {
    kc[dst + i] = row[k_off + i];
    vc[dst + i] = row[v_off + i];
  }
}

// LDS a workgroup may take (queried once per device).
static size_t lds_limit() {
  static thread_local int dev = -1;
  static thread_local size_t lim = 0;
  int d = 0;
  if (hipGetDevice(&d) != hipSuccess)
    return 64 * 1024;
  if (d != dev) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, d) != hipSuccess ||
        v <= 0)
      v = 64 * 1024;
    dev = d;
    lim = (size_t)v;
  }
  return lim;
}

} // namespace gkv

using namespace gkv;

extern "C" int gkv_rope_exact(void *stream, int32_t B, float *qkv, int64_t row_stride,
                              const float *cos_tab, const float *sin_tab,
                              const int32_t *positions, int32_t n_heads) {
  if (B < 0 || !qkv || !cos_tab || !sin_tab || n_heads <= 0 ||
      row_stride < (int64_t)n_heads * kHeadDim)
    return GKV_ERR_ARG;
  if (B == 0)
    return GKV_OK;
  hipLaunchKernelGGL(rope_exact_kernel, dim3(B), dim3(256), 0, (hipStream_t)stream, qkv,
                     row_stride, cos_tab, sin_tab, positions, (int)n_heads);
  return launch_status("rope_exact_kernel");
}

extern "C" int gkv_kv_write_exact(void *stream, int32_t B, const float *qkv, int64_t row_stride,
                                  int32_t k_off, int32_t v_off, float *kc, float *vc,
                                  int32_t slots, int32_t kv_dim, int32_t slot,
                                  const int32_t *positions, int32_t window, uint32_t *dev_err) {
  if (B < 0 || !qkv || !kc || !vc || slots <= 0 || kv_dim <= 0 || k_off < 0 || v_off < 0 ||
      (int64_t)k_off + kv_dim > row_stride || (int64_t)v_off + kv_dim > row_stride ||
      window < 0 || (window > 0 && slots < window) ||
      (!positions && (slot < 0 || slot >= slots)))
    return GKV_ERR_ARG;
  if (B == 0)
    return GKV_OK;
  hipLaunchKernelGGL(kv_write_exact_kernel, dim3(B), dim3(256), 0, (hipStream_t)stream, qkv,
                     row_stride, (int)k_off, (int)v_off, kc, vc, (int)slots, (int)kv_dim,
                     (int)slot, positions, (int)window, dev_err);
  return launch_status("kv_write_exact_kernel");
}

extern "C" int gkv_attention_exact(void *stream, int32_t B, int32_t n_q_heads,
                                   int32_t n_kv_heads, const float *q, int64_t q_stride,
                                   const float *kc, const float *vc, int32_t slots,
                                   const float *sinks, int32_t pos, const int32_t *positions,
                                   int32_t max_pos, int32_t window, float *out,
                                   int64_t out_stride, uint32_t *dev_err) {
  if (B < 0 || !q || !kc || !vc || !sinks || !out || n_kv_heads <= 0 || n_q_heads <= 0 ||
      n_q_heads % n_kv_heads || slots <= 0 || window < 0 || (window > 0 && slots < window) ||
      q_stride < (int64_t)n_q_heads * kHeadDim || out_stride < (int64_t)n_q_heads * kHeadDim)
    return GKV_ERR_ARG;
  const int G = n_q_heads / n_kv_heads;
  if (G > 16)
    return GKV_ERR_UNSUPPORTED;
  const int p_bound = positions ? max_pos : pos;
  if (p_bound < 0 || (!positions && window == 0 && pos >= slots))
    return GKV_ERR_ARG;
  if (B == 0)
    return GKV_OK;
  // positions attended at most, then the most query heads per workgroup whose
  // score rows fit the LDS (kFixed: the part of it that stays free of them, the
  // limit on the positions of one head)
  const int n_cap = window > 0 ? std::min(p_bound + 1, (int)window) : p_bound + 1;
  constexpr size_t kFixed = (size_t)kExactTile * (kHeadDim + 1) * sizeof(float) + 256;
  const size_t lim = lds_limit();
  int hc = 0;
  for (int c = G; c >= 1; c--) {
    if (G % c)
      continue;
    const size_t need = kFixed + (size_t)c * (kHeadDim + n_cap + 1) * sizeof(float);
    if (need <= lim) {
      hc = c;
      break;
    }
  }
  if (hc == 0)
    return GKV_ERR_CAPACITY;
  ExactAttnArgs a{};
  a.q = q;
  a.q_stride = q_stride;
  a.kc = kc;
  a.vc = vc;
  a.slots = slots;
  a.n_kv_heads = n_kv_heads;
  a.G = G;
  a.hc = hc;
  a.n_chunks = G / hc;
  a.window = window;
  a.sinks = sinks;
  a.pos = pos;
  a.positions = positions;
  a.n_cap = n_cap;
  a.out = out;
  a.out_stride = out_stride;
  a.dev_err = dev_err;
  size_t lds;
  int threads;
  void (*fn)(ExactAttnArgs);
  const int64_t wgs = (int64_t)B * n_kv_heads * a.n_chunks;
  int short_cap = kExactShort;
  if (wgs > kExactTwo && wgs <= kExactMany && hc >= 5)
    short_cap = kExactShortTwo;
  else if (wgs > kExactMany && wgs <= kExactFour && hc >= 5 && hc <= 8)
    short_cap = kExactShortFour;
  if (n_cap <= short_cap) {
    lds = kFixed - 256 + (size_t)hc * (kHeadDim + n_cap + 1) * sizeof(float);
    threads = 64 * hc;
    fn = attention_exact_short_kernel;
  } else {
    a.att_row = (n_cap + 1 + 3) / 4 * 4;
    const int tiles = (n_cap + kExactTile - 1) / kExactTile;
    const size_t rows_bytes = (size_t)hc * (kHeadDim + a.att_row) * sizeof(float);
    const size_t dbl_bytes = (size_t)hc * 128 * sizeof(double);
    auto ring_bytes = [](int rows) { return (size_t)4 * rows * kHeadDim * sizeof(float); };
    // The V ring's smallest form (16 rows a stage, in the place of the sums' fp64
    // values) is what kFixed always holds.
    const size_t least = rows_bytes + std::max(ring_bytes(16), dbl_bytes);
    const bool lite = wgs > kExactTwo && 2 * (least + 256) <= lim;
    // waves: a whole number per head, at most one per head and 64-position tile
    const int most = lite && wgs > kExactFour && hc <= kExactMaxWaves / 2 ? kExactMaxWaves / 2
                                                                          : kExactMaxWaves;
    a.parts = std::max(1, std::min(most / hc, tiles));
    const int waves = hc * a.parts, n_load = waves > hc ? waves - hc : waves;
    // The ring's stages: as many rows (at most 16 loads a loading wave) as leave room
    // for the workgroups a CU is to hold (256: the static arrays)
    const size_t hold = !lite ? 1 : most == kExactMaxWaves ? 2 : std::min<size_t>(4, lim / (least + 256));
    const size_t room = lim / hold - 256 - rows_bytes;
    a.v_rows = 64;
    while (a.v_rows > 16 && (a.v_rows > 16 * n_load || std::max(ring_bytes(a.v_rows), dbl_bytes) > room))
      a.v_rows -= 8;
    a.v_early = ring_bytes(a.v_rows) + dbl_bytes <= room;
    lds = rows_bytes + (a.v_early ? ring_bytes(a.v_rows) + dbl_bytes
                                  : std::max(ring_bytes(a.v_rows), dbl_bytes));
    const int one_tile_floats = (int)(lds / sizeof(float)) - kExactTile * kExactRow - hc * kHeadDim;
    a.one_tile_n = std::min(kExactShort, one_tile_floats / hc - 1);
    threads = 64 * waves;
    fn = lite ? attention_exact_kernel<true> : attention_exact_kernel<false>;
  }
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)lds) != hipSuccess)
    return hip_status(hipGetLastError(), "attention_exact_kernel (LDS size)");
  hipLaunchKernelGGL(fn, dim3(B, n_kv_heads * a.n_chunks), dim3(threads), lds,
                     (hipStream_t)stream, a);
  return launch_status("attention_exact_kernel");
}
