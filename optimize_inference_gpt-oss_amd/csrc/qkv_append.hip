// QKV projection with the KV append in its epilogue.
//
// Replaces the pair gemm_bf16 (getp-csrc/kernels/fast_gemm.hpp:888-899) +
// rope_kv_bf16 (fast_misc.hpp:112-127) of layer_attention
// (getp-csrc/engine/gpu_engine.hpp:493-496): qkv = x . W^T + bias, with x
// bf16 [M][K] and W bf16 [N][K] row-major, fp32 accumulation, the bias added
// to the finished sum, as gemm_bf16 computes it; then the K part rotated and
// the K and V parts rounded into the paged cache exactly as gkv_kv_append
// stores them (same rotation, rounding and placement code), without the fp32
// K/V rows going through memory. The fp32 qkv rows (Q, K, V unrotated, what
// gemm_bf16 writes) are stored too when asked: the attention reads Q from
// them.
//
// Work: one workgroup per output tile (shapes and the rule that picks one:
// qkv_shape below), the K dimension in stages of one or more 64-wide pieces,
// fed by direct-to-LDS loads (16-byte slots XOR-swizzled per row, as in the
// prefill kernel). A wave owns some row tiles of 16 and one head of the tile
// (and, where the rows are few, every kWK-th 32-wide K slice):
// v_mfma_f32_16x16x32_bf16 with W as the first operand, so a lane holds 4
// consecutive dims of one row (16-byte stores of the fp32 rows), d and d + 32
// alike -- both halves of a RoPE pair. The operands of a slice are read from
// LDS into registers among the matrix ops of the slice before, and one
// barrier per stage both publishes the next stage and frees this one.
// What bounds it: with many rows the matrix cores (9507 rows: 249 us = 1126
// TFLOP/s, 243 - 256 by GPU, of which 200 in the K loop, the fp32 rows' 195 MB most of the rest;
// 128 x 128 tiles without the operand buffering, the workgroups of an XCD
// spread over all row blocks: 372 in turn with it), at 512 rows the operands' way
// into LDS (640 tiles bring 471 MB; under that load an operand takes 1.2 us from
// its load's issue) and the third tile on half the CUs, with few rows the chain of
// K steps.
//
// Placement of each row (its sequence, position, slot and block) is loaded by
// the first waves in three dependent hops of direct-to-LDS loads spread over the
// stages (the largest tile: the first loads), so its round trips overlap them instead of
// adding to it.
#include "gkv_device.hpp"
#include "kv_append.hpp"
#include "lds_dma.hpp"

#include <algorithm>
#include <type_traits>

namespace gkv {

struct QkvArgs {
  const uint16_t *x; // bf16 [M][x_stride]
  int64_t x_stride;
  const uint16_t *w; // bf16 [N][K]
  const float *bias; // [N] or nullptr
  float *out;        // fp32 [M][out_stride] or nullptr
  int64_t out_stride;
  int M, N, K, m_blocks, n_blocks;
  AppendArgs ap; // placement, tables and cache of the append (qkv/q_out/packs unused)
};

// Four floats at any float's alignment: this entry point asks none of the
// output rows, the bias and the angle tables.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kQkvBK = 64; // K per pipeline stage: 128 bytes of a row, 8 slots of 16 bytes

// The 16-byte slot of stage row r that holds K piece s (8 values): 8 rows see
// every slot, so the 16 lanes reading one piece of 16 rows hit distinct banks.
__device__ __forceinline__ int qkv_slot(int r, int s) { return s ^ (r & 7); }

// Row placement in the paged cache: the rows' sequence, position, slot and
// block, one row per lane of the first waves (row 64 * wave + lane of the
// tile), as three dependent hops of direct-to-LDS loads issued among the main
// loop's (a register load would be left in flight across code the compiler
// schedules freely).
template <int kGM>
struct QkvPlace {
  static constexpr int kRows = (kGM + 63) / 64 * 64; // 64 per placing wave
  int *s_seq, *s_rpos, *s_len, *s_id; // kRows ints each, 16-byte aligned
  int *s_pos, *s_off;                 // the results: position, slot in the block (-1: not stored)
  int64_t *s_base;                    // and the block's first element
  int m0, wave;
  bool place, need_len;

  // The row of this lane within the tile, formed afresh at each use (kept, it
  // and what is derived from it would hold registers through the main loop).
  __device__ __forceinline__ int tile_row() const {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  }
  __device__ __forceinline__ int row(int M) const { return min(m0 + tile_row(), M - 1); }
  __device__ __forceinline__ int row_seq_of(const AppendArgs &ap, int M) const {
    return ap.row_seq ? s_seq[tile_row()] : row(M);
  }
  __device__ __forceinline__ void hop1(const AppendArgs &ap, int M) {
    if (!place)
      return;
    if (ap.row_seq)
      dma4(ap.row_seq + row(M), s_seq + 64 * wave);
    if (ap.row_pos)
      dma4(ap.row_pos + row(M), s_rpos + 64 * wave);
  }
  __device__ __forceinline__ void hop2(const AppendArgs &ap, int M) { // hop 1 has landed
    if (!place || !need_len)
      return;
    dma4(ap.seq_lens + row_seq_of(ap, M), s_len + 64 * wave);
  }
  __device__ __forceinline__ void hop3(const AppendArgs &ap, int M) { // hop 2 has landed
    if (!place)
      return;
    const int r = tile_row();
    const int seq = row_seq_of(ap, M);
    const int len = need_len ? s_len[r] : 0;
    const int pos = ap.row_pos ? s_rpos[r] : len - 1;
    const int slot = ap.ring > 0 ? pos % ap.ring : pos;
    bool store = r < kGM && m0 + r < M && pos >= 0;
    if (store && ap.ring > 0 && ap.seq_lens && pos + ap.ring < len)
      store = false; // a later row of this call takes the ring slot
    const int blk = slot / kBlockTokens;
    if (store && blk >= ap.table_stride) {
      if (ap.dev_err)
        atomicOr(ap.dev_err, GKV_DEVERR_LENGTH);
      store = false;
    }
    s_pos[r] = max(pos, 0);
    s_off[r] = store ? slot % kBlockTokens : -1;
    // rows that are not stored load entry 0 (any valid address)
    dma4(ap.table + (store ? (int64_t)seq * ap.table_stride + blk : 0), s_id + 64 * wave);
  }
  __device__ __forceinline__ void finish(const AppendArgs &ap) { // every load has landed
    if (!place)
      return;
    const int r = tile_row(), id = s_id[r];
    s_base[r] = (int64_t)id * ap.n_kv_heads * (kBlockTokens * kHeadDim);
    if (s_off[r] >= 0 && (id < 0 || id >= ap.num_blocks)) {
      if (ap.dev_err)
        atomicOr(ap.dev_err, GKV_DEVERR_BLOCK_ID);
      s_off[r] = -1;
    }
  }
};

// Staged V rows: row r of a wave (its 64 values of one head) in LDS as bf16, or
// as codes of one byte. The 16-byte slots of a bf16 row (8 slots) and the
// 8-byte ones of a row of codes are XOR-swizzled by the row, so that the 16
// lanes writing one piece of 16 rows spread over the banks.
__device__ __forceinline__ int v_stage_bf16(int r, int d) { // element offset
  return r * 64 + 8 * ((d >> 3) ^ (r & 7)) + (d & 7);
}
__device__ __forceinline__ int v_stage_code(int r, int d) { // byte offset
  return r * 64 + 8 * ((d >> 3) ^ (r & 7)) + (d & 7);
}

// One row tile of 16 rows x one head from its finished sums: lane (kg, n)
// holds row m (lr within the workgroup's tile), dims 16 j + 4 kg + r in
// acc[j][r], both halves (d, d + 32) of its RoPE pairs. Adds the bias, stores
// the fp32 row; a K head goes into the cache exactly as gkv_kv_append rounds
// and places it, a V head's cache values into vst (the wave's staged rows, row
// vr) for qkv_store_values.
template <int kGM>
__device__ __forceinline__ void qkv_store_row(const QkvArgs &a, const QkvPlace<kGM> &pl,
                                              f32x4 (&acc)[4], const f32x4 (&bias)[4], int hd,
                                              int lr, int kg, char *vst, int vr) {
  constexpr int D = kHeadDim, HALF = kHeadDim / 2;
  const AppendArgs &ap = a.ap;
  const int m = pl.m0 + lr, c0 = D * hd + 4 * kg;
#pragma unroll
  for (int j = 0; j < 4; j++)
    acc[j] += bias[j];
  if (a.out && m < a.M) {
    float *o = a.out + (int64_t)m * a.out_stride + c0;
#pragma unroll
    for (int j = 0; j < 4; j++)
      *(f32x4u *)(o + 16 * j) = acc[j];
  }
  if (!ap.kc || hd < ap.n_q_heads)
    return;
  const bool is_k = hd < ap.n_q_heads + ap.n_kv_heads;
  const int g = is_k ? hd - ap.n_q_heads : hd - ap.n_q_heads - ap.n_kv_heads;
  const int off = pl.s_off[lr];
  const int64_t base = pl.s_base[lr] + (int64_t)g * (kBlockTokens * D);
  const bool st_ok = off >= 0; // (rows past the last have none)
  f32x4 y[4];
  if (is_k) {
    const int pos = pl.s_pos[lr];
#pragma unroll
    for (int j = 0; j < 2; j++) { // dims 16 j + 4 kg .. +3 and those + 32
      const f32x4 c = *(const f32x4u *)(ap.cos_tab + (int64_t)pos * HALF + 16 * j + 4 * kg);
      const f32x4 s = *(const f32x4u *)(ap.sin_tab + (int64_t)pos * HALF + 16 * j + 4 * kg);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        y[j][r] = rope_first(acc[j][r], acc[j + 2][r], c[r], s[r]);
        y[j + 2][r] = rope_second(acc[j][r], acc[j + 2][r], c[r], s[r]);
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++)
      y[j] = acc[j];
  }
  const bool quant = ap.kv_fp8 || (ap.v_int8 && !is_k);
  uint32_t code[4]; // of dims 16 j + 4 kg .. +3
  if (quant) {
    float amax = 0.0f; // of the head's 64 dims: 16 in this lane, 4 lanes
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        amax = fmaxf(amax, fabsf(y[j][r]));
    amax = fmaxf(amax, __shfl_xor(amax, 16));
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    if (ap.kv_fp8) {
      // e4m3: one scale per token and head (K's, then V's)
      const float inv = amax > 0.0f ? 448.0f / amax : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; j++)
        code[j] = fp8x4(y[j][0], y[j][1], y[j][2], y[j][3], inv);
      if (st_ok && kg == 0)
        ap.vs[base / 32 + (is_k ? 0 : kBlockTokens) + off] = amax / 448.0f;
    } else {
      // the reference's rule, getp-csrc/kernels/fast_misc.hpp:74-84
      const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        code[j] = 0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float cq = fminf(fmaxf(rintf(y[j][r] * inv), -127.0f), 127.0f);
          code[j] |= (uint32_t)(uint8_t)(int8_t)cq << (8 * r);
        }
      }
      if (st_ok && kg == 0)
        ap.vs[base / D + off] = amax / 127.0f;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int d = 16 * j + 4 * kg;
    const u32x2 w{f32x2_to_bf16_rne(y[j][0], y[j][1]), f32x2_to_bf16_rne(y[j][2], y[j][3])};
    if (!is_k && quant)
      *(uint32_t *)(vst + v_stage_code(vr, d)) = code[j];
    else if (!is_k)
      *(u32x2 *)(vst + 2 * v_stage_bf16(vr, d)) = w;
    else if (st_ok && quant)
      *(uint32_t *)((uint8_t *)ap.kc + base + k_fp8_offset(off, d)) = code[j];
    else if (st_ok)
      *(u32x2 *)(ap.kc + base + k_offset(off, d)) = w;
  }
}

// The staged V rows of one head (rows lr0 .. lr0 + n_rows - 1 of the tile, at
// most 64, staged as rows 0 ..) into the cache, by one wave. Four rows holding
// slots 4m .. 4m+3 of one block (consecutive tokens of a prompt) go together
// as 16-byte pieces (bf16: dims d and d + 16 of the 4 tokens; codes: dims d,
// d + 16, d + 32, d + 48); a row alone goes as one store of its 64 dims, whose
// lanes then meet in few cache lines. (Stored straight from the matrix layout,
// 16 rows x 4 dims an instruction, the V heads' workgroups took 7.5 us longer
// than the others at 512 decode rows.)
template <int kGM>
__device__ __forceinline__ void qkv_store_values(const AppendArgs &ap, const QkvPlace<kGM> &pl,
                                                 const char *vst, int lr0, int n_rows, int g,
                                                 int lane) {
  const bool code = ap.v_int8 || ap.kv_fp8;
  const int64_t hb = (int64_t)g * (kBlockTokens * kHeadDim);
  const int off = lane < n_rows ? pl.s_off[lr0 + lane] : -1;
  bool lead = lane + 3 < n_rows && off >= 0 && (off & 3) == 0;
#pragma unroll
  for (int k = 1; k < 4; k++) {
    const int r = min(lane + k, n_rows - 1) + lr0;
    lead = lead && pl.s_off[r] == off + k && pl.s_base[r] == pl.s_base[lr0 + lane];
  }
  uint64_t quads = __ballot(lead);
  uint64_t alone = __ballot(off >= 0) & ~(quads | quads << 1 | quads << 2 | quads << 3);
  const int per = code ? 16 : 32; // lanes per quad
  while (quads) {
    int r0 = -1; // this lane's quad
    for (int k = 0; k < 64 / per && quads; k++) {
      const int r = __builtin_ctzll(quads);
      quads &= quads - 1;
      r0 = lane / per == k ? r : r0;
    }
    if (r0 < 0)
      continue;
    const int t0 = pl.s_off[lr0 + r0];
    const int64_t base = pl.s_base[lr0 + r0] + hb;
    if (code) {
      const int d = lane & 15;
      uint32_t w[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        w[q] = 0;
#pragma unroll
        for (int k = 0; k < 4; k++)
          w[q] |= (uint32_t)(uint8_t)vst[v_stage_code(r0 + k, d + 16 * q)] << (8 * k);
      }
      *(u32x4 *)((uint8_t *)ap.vc + base + v_int8_offset(d, t0)) = u32x4{w[0], w[1], w[2], w[3]};
    } else {
      const int d = 32 * ((lane >> 4) & 1) + (lane & 15);
      uint16_t h[8];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        h[k] = ((const uint16_t *)vst)[v_stage_bf16(r0 + k, d)];
        h[4 + k] = ((const uint16_t *)vst)[v_stage_bf16(r0 + k, d + 16)];
      }
      *(u32x4 *)(ap.vc + base + v_offset(t0, d)) = pack8(h);
    }
  }
  while (alone) {
    const int r = __builtin_ctzll(alone);
    alone &= alone - 1;
    const int t = pl.s_off[lr0 + r];
    const int64_t base = pl.s_base[lr0 + r] + hb;
    if (code)
      ((uint8_t *)ap.vc)[base + v_int8_offset(lane, t)] = (uint8_t)vst[v_stage_code(r, lane)];
    else
      ap.vc[base + v_offset(t, lane)] = ((const uint16_t *)vst)[v_stage_bf16(r, lane)];
  }
}

// kGM x kGN output tile, kWM x (kGN / 64) x kWK waves, kSub 64-wide K pieces per
// stage: wave (wm, wn, wk) sums rows [wm] of head [wn] over the 32-wide slices
// wk, wk + kWK, .. of every stage; with kWK > 1 the sums of a tile meet in LDS
// after the loop.
template <int kGM, int kGN, int kWM, int kWK, int kSub, int kGStages, bool kWide = false>
__global__ __launch_bounds__(64 * kWM * (kGN / 64) * kWK) void qkv_append_kernel(QkvArgs a) {
  constexpr int kWN = kGN / 64, kNW = kWM * kWN * kWK;
  constexpr int kRT = kGM / 16 / kWM;            // 16-row tiles per wave
  constexpr int kSl = 2 * kSub / kWK;            // slices per wave and stage
  constexpr int kXC = kGM / 8, kWC = kGN / 8;    // 1 KB direct-to-LDS loads per 64 of K: x, W
  constexpr int kUnits = kSub * (kXC + kWC);
  constexpr int kGPer = (kUnits + kNW - 1) / kNW; // per wave and stage
  static_assert(kRT >= 1 && kGM % (16 * kWM) == 0 && (2 * kSub) % kWK == 0 &&
                    kNW >= QkvPlace<kGM>::kRows / 64,
                "launch shape");
  static_assert((kWK - 1) * kGM * kGN * 4 <= kGStages * kSub * (kGM + kGN) * kQkvBK * 2 &&
                    kGM * kGN * 2 * (kWK > 1 ? 2 : 1) <= kGStages * kSub * (kGM + kGN) * kQkvBK * 2,
                "the slices' sums and the staged V rows fit the stages");
  using Place = QkvPlace<kGM>;
  constexpr int kSubElems = (kGM + kGN) * kQkvBK, kStageElems = kSub * kSubElems;
  __shared__ __attribute__((aligned(16))) uint16_t stage[kGStages * kStageElems];
  __shared__ __attribute__((aligned(16))) int s_place[6 * Place::kRows];
  __shared__ int64_t s_base[Place::kRows];

  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int n = lane & 15, kg = lane >> 4;
  int mb, nb;
  {
    // workgroup id -> tile: the ids of one XCD (id % 8) take consecutive tiles,
    // in groups of 8 row blocks x all column blocks, rows fastest, so that the
    // tiles an XCD holds at once share their rows and columns in its L2. The
    // columns go round the XCDs (column c of an XCD's n / 8 is block 8 c + its
    // index), from the last one down: the K and V heads, whose epilogue is
    // longer, are spread over all XCDs and start first.
    const int x = blockIdx.x % 8, q = gridDim.x / 8, rem = gridDim.x % 8;
    const int t = x * q + min(x, rem) + blockIdx.x / 8;
    const int width = 8 * a.n_blocks, grp = t / width, in = t - grp * width;
    const int gm = min(a.m_blocks - 8 * grp, 8);
    mb = 8 * grp + in % gm;
    nb = in / gm;
    if (a.n_blocks % 8 == 0) {
      const int per = a.n_blocks / 8;
      nb = nb % per * 8 + nb / per;
    }
    nb = a.n_blocks - 1 - nb;
  }
  const int m0 = mb * kGM, n0 = nb * kGN;
  const int n64 = a.K / kQkvBK, nk = (n64 + kSub - 1) / kSub;
  const AppendArgs &ap = a.ap;

  // This wave's loads of a stage: load u = wave + kNW i of its kUnits 1 KB
  // loads, in each 64-wide K piece those of x (8 rows of 128 bytes each), then
  // those of W; a wave past the last load repeats it (the same bytes to the
  // same place), so every wave issues kGPer loads and the waits are exact.
  // A lane's offset from the tile's first row is 32 bits (kWide: 64).
  using Off = std::conditional_t<kWide, uint64_t, uint32_t>;
  const char *xb = (const char *)(a.x + (int64_t)m0 * a.x_stride);
  const char *wb = (const char *)(a.w + (int64_t)n0 * a.K);
  // the wave's loads split evenly between x and W: which is which is known when
  // compiling; and each of W's covers a head's 64 rows (N is whole heads), so
  // that one offset serves them all
  constexpr bool kEven = kSub == 1 && kXC % kNW == 0 && kWC % kNW == 0;
  constexpr bool kOneW = kEven && kNW == 8 && !kWide;
  constexpr int kOffs = kOneW ? kXC / kNW + 1 : kGPer;
  Off off[kOffs];
#pragma unroll
  for (int i = 0; i < kOffs; i++) {
    const int c = min(wave + kNW * i, kUnits - 1) % (kXC + kWC);
    const int r8 = lane >> 3, s = lane & 7;
    if (c < kXC) {
      const int r = 8 * c + r8;
      off[i] = (Off)((int64_t)min(r, a.M - 1 - m0) * a.x_stride + 8 * qkv_slot(r, s)) * 2;
    } else {
      const int r = 8 * (c - kXC) + r8;
      off[i] = (Off)((int64_t)min(r, a.N - 1 - n0) * a.K + 8 * qkv_slot(r, s)) * 2;
    }
  }
  // load i of chunk kc into stage st; K pieces past the last re-read the last one
  const uint32_t stage_lds = lds_addr(stage);
  auto dma = [&](int kc, int st, int i) {
    const int u = kEven ? wave + kNW * i : min(wave + kNW * i, kUnits - 1);
    const int sub = kEven ? 0 : u / (kXC + kWC);
    const bool is_x = kEven ? i < kXC / kNW : u % (kXC + kWC) < kXC;
    const int64_t kb = (int64_t)min(kc * kSub + sub, n64 - 1) * (kQkvBK * 2);
    const char *base = (is_x ? xb : wb) + kb;
    const uint32_t dst = stage_lds + 2 * (st * kStageElems + u * 512);
    if constexpr (kWide)
      dma16(base + off[i], &stage[st * kStageElems + u * 512]);
    else if (kOneW && !is_x) // 64 columns on, or the last 64
      dma16_at<kEven>(base + (int64_t)min(64 * (i - kXC / kNW), (a.N - 64 - n0)) * a.K * 2,
               off[kXC / kNW], dst);
    else
      dma16_at<kEven>(base, off[i], dst); // (kEven: no part of the base is the wave's)
  };
  auto dma_chunk = [&](int kc, int st) {
#pragma unroll
    for (int i = 0; i < kGPer; i++)
      dma(kc, st, i);
  };

  Place pl;
  pl.s_seq = s_place;
  pl.s_rpos = s_place + Place::kRows;
  pl.s_len = s_place + 2 * Place::kRows;
  pl.s_id = s_place + 3 * Place::kRows;
  pl.s_pos = s_place + 4 * Place::kRows;
  pl.s_off = s_place + 5 * Place::kRows;
  pl.s_base = s_base;
  pl.m0 = m0;
  pl.wave = wave;
  pl.place = wave < Place::kRows / 64 && ap.kc != nullptr;
  pl.need_len = ap.seq_lens && (!ap.row_pos || ap.ring > 0);

  const int wm = wave % kWM, wn = (wave / kWM) % kWN, wk = wave / (kWM * kWN);
  f32x4 acc[kRT][4];
#pragma unroll
  for (int i = 0; i < kRT; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
      acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // operands of one slice, double-buffered: operand q of slice sl of stage st
  // (W's four, then the row tiles' of x)
  bf16x8 xo[2][kRT], wo[2][4];
  auto read = [&](int st, int sl, int q, bf16x8 (&xr)[kRT], bf16x8 (&wr)[4]) {
    const int k32 = wk + kWK * sl; // slice of the stage
    const uint16_t *xs = &stage[st * kStageElems + (k32 >> 1) * kSubElems];
    const uint16_t *ws = xs + kGM * kQkvBK;
    const int s = 4 * (k32 & 1) + kg;
    if (q < 4) {
      const int r = 64 * wn + 16 * q + n;
      wr[q] = *(const bf16x8 *)&ws[r * kQkvBK + 8 * qkv_slot(r, s)];
    } else {
      const int r = 16 * (kRT * wm + q - 4) + n;
      xr[q - 4] = *(const bf16x8 *)&xs[r * kQkvBK + 8 * qkv_slot(r, s)];
    }
  };
  pl.hop1(ap, a.M);
  // The placement's later hops: with 8 row tiles a wave has no registers for
  // them in the main loop, so hop 1 is waited for behind chunk 0's loads, and
  // hop 2 goes out before chunk 1 and lands with chunk 0.
  constexpr bool kEarly = kRT >= 8;
  if constexpr (kEarly) {
    dma_chunk(0, 0);
    wait_vmcnt<kGPer>();
    pl.hop2(ap, a.M);
  }
#pragma unroll
  for (int p = kEarly ? 1 : 0; p < kGStages; p++)
    dma_chunk(p, p);
  wait_vmcnt<(kGStages - 1) * kGPer>();
  lds_barrier();
  if constexpr (kEarly)
    pl.hop3(ap, a.M);
  else
    pl.hop2(ap, a.M); // hop 1 was issued before chunk 0
#pragma unroll
  for (int q = 0; q < 4 + kRT; q++)
    read(0, 0, q, xo[0], wo[0]);
  int st = 0; // stage of chunk kc
  // One chunk, its first slice's operands in buffer b0. Before its last slice's
  // matrix ops, chunk kc + 1 has landed, every wave has read the whole of chunk
  // kc (its reads were waited for before the barrier) and chunk kc + kGStages
  // goes into its stage. The reads of the next slice and those loads are laid
  // between the row tiles' matrix ops, in this order (the scheduling barriers:
  // the compiler else moves the reads down to their use and the loads in front
  // of the matrix ops, and both are waited for).
  auto chunk = [&](int kc, auto b0c) {
    constexpr int b0 = decltype(b0c)::value;
    const int nst = st == kGStages - 1 ? 0 : st + 1;
#pragma unroll
    for (int sl = 0; sl < kSl; sl++) {
      const int cur = (b0 + sl) & 1, nxt = cur ^ 1;
      const bool last = sl == kSl - 1;
      if (last) {
        wait_vmcnt<(kGStages - 2) * kGPer>();
        lds_barrier();
        if (!kEarly && kc == kGStages)
          pl.hop3(ap, a.M); // hop 2 was issued before chunk kGStages's loads
      }
      // a K piece past the last adds nothing
      const bool real = kSub == 1 || kc * kSub + ((wk + kWK * sl) >> 1) < n64;
#pragma unroll
      for (int i = 0; i < kRT; i++) {
#pragma unroll
        for (int q = i * (4 + kRT) / kRT; q < (i + 1) * (4 + kRT) / kRT; q++)
          read(last ? nst : st, last ? 0 : sl + 1, q, xo[nxt], wo[nxt]);
        __builtin_amdgcn_sched_barrier(0);
        if (real) {
#pragma unroll
          for (int j = 0; j < 4; j++)
            acc[i][j] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(wo[cur][j], xo[cur][i], acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (last) {
#pragma unroll
          for (int d = i * kGPer / kRT; d < (i + 1) * kGPer / kRT; d++)
            dma(kc + kGStages, st, d);
        }
      }
    }
    st = nst;
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  for (int kc = 0; kc < nk; kc += 2 - (kSl + 1) % 2) {
    chunk(kc, I0{});
    if constexpr (kSl % 2 == 1) {
      if (kc + 1 < nk)
        chunk(kc + 1, I1{});
    }
  }
  wait_vmcnt<0>(); // every load landed, none still writes LDS
  if (!kEarly && nk <= kGStages) { // a short K left hop 3 for here
    pl.hop3(ap, a.M);
    wait_vmcnt<0>();
  }
  pl.finish(ap);
  __syncthreads();
  // (the lane's indices formed afresh: kept, they would hold registers through
  // the main loop)
  const int elane = pl.tile_row() & 63, en = elane & 15, ekg = elane >> 4;
  if constexpr (kWK > 1) { // the stages are free: the other slices' sums, in wave order
    f32x4 *red = (f32x4 *)stage + elane;
    constexpr int kTile = kRT * 4 * 64;
    if (wk > 0) {
#pragma unroll
      for (int i = 0; i < kRT; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          red[(wave - kWM * kWN) * kTile + (4 * i + j) * 64] = acc[i][j];
    }
    __syncthreads();
    if (wk > 0)
      return;
#pragma unroll
    for (int k = 1; k < kWK; k++)
#pragma unroll
      for (int i = 0; i < kRT; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          acc[i][j] += red[(wave + (k - 1) * kWM * kWN) * kTile + (4 * i + j) * 64];
  }

  const int hd = (n0 >> 6) + wn;
  if (64 * hd >= a.N)
    return;
  f32x4 bias[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    bias[j] = a.bias ? (f32x4) * (const f32x4u *)(a.bias + 64 * hd + 16 * j + 4 * kg)
                     : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // the wave's staged V rows: its own part of the stages (with kWK > 1 the
  // part its second slice sums came in)
  constexpr int kStBytes = kRT * 16 * 128;
  char *vst = (char *)stage + (wm + kWM * wn) * (kWK > 1 ? 2 : 1) * kStBytes;
#pragma unroll
  for (int i = 0; i < kRT; i++)
    qkv_store_row<kGM>(a, pl, acc[i], bias, hd, 16 * (kRT * wm + i) + en, ekg, vst, 16 * i + en);
  const int gv = hd - ap.n_q_heads - ap.n_kv_heads;
  if (ap.kc && gv >= 0) {
    const int row_bytes = ap.v_int8 || ap.kv_fp8 ? 64 : 128;
    for (int r = 0; r < 16 * kRT; r += 64)
      qkv_store_values<kGM>(ap, pl, vst + r * row_bytes, 16 * kRT * wm + r,
                            min(16 * kRT - r, 64), gv, elane);
  }
}

// ---- launch shapes ----------------------------------------------------------------

struct QkvShape {
  int bm, bn, threads;
  void (*fn)(QkvArgs);
};

template <int kGM, int kGN, int kWM, int kWK, int kSub, int kGStages, bool kWide = false>
static QkvShape shape_of() {
  return QkvShape{kGM, kGN, 64 * kWM * (kGN / 64) * kWK,
                  qkv_append_kernel<kGM, kGN, kWM, kWK, kSub, kGStages, kWide>};
}

// The launch shape for M rows and N columns. Times below: N = 5120, K = 2880,
// the append included, one MI355X.
static QkvShape qkv_shape(int M, int N, int64_t x_stride, int K) {
  auto blocks = [](int64_t n, int b) { return (n + b - 1) / b; };
  auto tiles = [&](int bm, int bn) { return blocks(M, bm) * blocks(N, bn); };
  // offsets within a tile beyond 32 bits (a row stride of millions of values)
  const int64_t x_span = (int64_t)std::min(M, 256) * x_stride * 2;
  const int64_t w_span = (int64_t)std::min(N, 256) * K * 2;
  if (x_span > UINT32_MAX || w_span > UINT32_MAX)
    return shape_of<64, 64, 4, 1, 1, 3, true>();
  // Few rows: a pass is the chain of its K steps, so each step is wide and its
  // 32-wide slices are dealt to the waves (16-row tiles, 256-wide steps: 12
  // steps instead of 45; 24 rows 11.8 us, 32-row tiles 12.3, 64-row ones with
  // 64-wide steps 16.8). 32-row tiles while every CU gets at most one (64 rows
  // 12.9 us, 64-row tiles 17.3) or two (128 rows 16.9 against 18.0).
  if (M <= 32)
    return shape_of<16, 64, 1, 8, 4, 3>();
  if (tiles(32, 64) <= 256)
    return shape_of<32, 64, 2, 4, 2, 4>();
  if (tiles(32, 64) <= 512)
    return shape_of<32, 64, 2, 2, 1, 4>();
  // 64 x 64 tiles up to two per CU, and where a third one goes to a good part of
  // the CUs (512 rows, 640 tiles: 29.9 us, 128 x 64 ones 30.7); with a third on
  // few CUs only 128 x 64 ones are ahead (416 rows, 560 tiles: 30.1 against 29.3; N
  // = 2560, 800 rows, 520 tiles: 30.9 against 28.1), and they are beyond 640 tiles
  // (540 rows, 720 tiles: 34.8 against 29.1), up to two of them per CU (640 rows
  // 32.1 us against 41.2).
  const int64_t t64 = tiles(64, 64);
  if (t64 <= 512 || (t64 > 576 && t64 <= 640))
    return shape_of<64, 64, 4, 1, 1, 3>();
  if (tiles(128, 64) <= 512)
    return shape_of<128, 64, 4, 2, 1, 3>();
  // 128 x 128 tiles while the GPU holds them at two per CU, then 256 x 256 ones
  // (one per CU, rounds of 256, 67 - 78 us each): N = 2560, 3072 rows 48 us against 69,
  // 3328 rows 79.6 against 69, 6400 rows 108 against 82. A second or third round of
  // the large tiles pays from some 1420 and 2130 small ones on: N = 2560, 8192
  // rows (1280) 124.6 against 133.8, 8960 rows (1400) 136.5 against 139.6, 9216 rows
  // (1440) 146.1 against 140.9; N = 5120, 4352 rows (1360) 129.9 against 140, 4864 rows
  // (1520) 160 against 141, 6656 rows (2080) level, 7424 rows (2320) 217 against 209.
  const int64_t t128 = tiles(128, 128), rounds = blocks(tiles(256, 256), 256);
  if (t128 <= (rounds > 1 ? rounds * 710 : 512))
    return shape_of<128, 128, 4, 1, 1, 2>();
  return shape_of<256, 256, 2, 1, 1, 2>();
}

} // namespace gkv

extern "C" int gkv_qkv_append(void *stream, int32_t n_rows, const void *x, int64_t x_stride,
                              int32_t hidden, const void *w_qkv, const float *b_qkv,
                              int32_t n_q_heads, const float *cos_tab, const float *sin_tab,
                              const int32_t *row_pos, const int32_t *row_seq,
                              const int32_t *seq_lens, gkv_cache_view cache, float *qkv_out,
                              int64_t out_stride, uint32_t *dev_err) {
  using namespace gkv;
  if (n_rows < 0 || !x || !w_qkv || n_q_heads <= 0 || cache.n_kv_heads <= 0 || hidden <= 0 ||
      cache.ring < 0)
    return GKV_ERR_ARG;
  if (n_q_heads % cache.n_kv_heads != 0)
    return GKV_ERR_ARG;
  const int64_t n_cols = (int64_t)(n_q_heads + 2 * cache.n_kv_heads) * kHeadDim;
  if (n_cols >= INT32_MAX || x_stride < hidden || (qkv_out && out_stride < n_cols))
    return GKV_ERR_ARG;
  if (hidden % kQkvBK != 0)
    return GKV_ERR_UNSUPPORTED;
  // 16-byte direct-to-LDS loads of x and W rows
  if (x_stride % 8 != 0 || ((uintptr_t)x | (uintptr_t)w_qkv) % 16 != 0)
    return GKV_ERR_ARG;
  const bool to_cache = cache.k != nullptr || cache.v != nullptr;
  if (!to_cache && !qkv_out)
    return GKV_ERR_ARG; // nothing to write
  if (to_cache && (!cache.k || !cache.v || !cache.block_table || cache.table_stride <= 0 ||
                   cache.num_blocks <= 0 || !cos_tab || !sin_tab))
    return GKV_ERR_ARG;
  if (to_cache && !row_pos && !seq_lens)
    return GKV_ERR_ARG; // no way to find the rows' positions
  if (to_cache && cache.ring > 0 && !seq_lens)
    return GKV_ERR_ARG; // rows W positions apart share a ring slot: the lengths pick the kept one
  if (cache.ring % kBlockTokens != 0)
    return GKV_ERR_UNSUPPORTED;
  if (cache.v_format != GKV_V_BF16 && cache.v_format != GKV_V_INT8 &&
      cache.v_format != GKV_KV_FP8)
    return GKV_ERR_ARG;
  if (to_cache && cache.v_format != GKV_V_BF16 && !cache.v_scale)
    return GKV_ERR_ARG;
  if (n_rows == 0)
    return GKV_OK;
  QkvArgs a;
  a.x = (const uint16_t *)x;
  a.x_stride = x_stride;
  a.w = (const uint16_t *)w_qkv;
  a.bias = b_qkv;
  a.out = qkv_out;
  a.out_stride = out_stride;
  a.M = n_rows;
  a.N = (int)n_cols;
  a.K = hidden;
  const QkvShape sh = qkv_shape(n_rows, (int)n_cols, x_stride, hidden);
  a.m_blocks = (n_rows + sh.bm - 1) / sh.bm;
  a.n_blocks = (int)((n_cols + sh.bn - 1) / sh.bn);
  const int64_t grid = (int64_t)a.m_blocks * a.n_blocks;
  if (grid >= INT32_MAX)
    return GKV_ERR_ARG;
  AppendArgs &ap = a.ap;
  ap.qkv = nullptr;
  ap.row_stride = 0;
  ap.n_q_heads = n_q_heads;
  ap.n_kv_heads = cache.n_kv_heads;
  ap.cos_tab = cos_tab;
  ap.sin_tab = sin_tab;
  ap.row_pos = row_pos;
  ap.row_seq = row_seq;
  ap.seq_lens = seq_lens;
  ap.kc = to_cache ? (uint16_t *)cache.k : nullptr;
  ap.vc = to_cache ? (uint16_t *)cache.v : nullptr;
  ap.table = cache.block_table;
  ap.table_stride = cache.table_stride;
  ap.num_blocks = cache.num_blocks;
  ap.ring = cache.ring;
  ap.q_out = nullptr;
  ap.q_out_stride = 0;
  ap.k_pack = nullptr;
  ap.v_pack = nullptr;
  ap.dev_err = dev_err;
  ap.v_int8 = cache.v_format == GKV_V_INT8;
  ap.kv_fp8 = cache.v_format == GKV_KV_FP8;
  ap.vs = (float *)cache.v_scale;
  hipLaunchKernelGGL(sh.fn, dim3((unsigned)grid), dim3(sh.threads), 0, (hipStream_t)stream, a);
  return launch_status(__func__);
}
