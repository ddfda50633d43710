// sk_attn.hip - decode attention side of the Qwen3 decode step on gfx950:
//   * per-head RMSNorm + rotary embedding + KV-cache write of the QKV
//     projection (engine/kernels/rope.py:94-188), and
//   * split-K grouped-query flash-decoding over the KV cache with a
//     device-side sequence length (engine/kernels/attention.py:23-202).
// Both are memory-bound: the first touches (HQ + 2*HKV) * D values per row,
// the second streams K and V of every valid position once per KV head.
#include "starter_amd.h"

#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include <math.h>
#include <string.h>

#include "sk_stream.hpp"

namespace sk {

constexpr int HEAD_D = 128;   // head width of Qwen3 (the only one compiled)

// ---------------------------------------------------------------------------
// q/k RMSNorm + RoPE + cache write (rope.py:94-188 cast placement):
//   n = bf16(x * rsqrt(mean(x^2) + eps)); y = bf16(w * n)
//   o1 = bf16(bf16(y1 * cos1) + bf16(-y2 * sin1)); o2 = bf16(bf16(y2 * cos2) + bf16(y1 * sin2))
// with (y1, y2) = (y[i], y[i + D/2]).  One wave per head: lane i holds the
// rotation pair (i, i + 64), so the rotation needs no lane exchange.  Workgroup
// (row, head group): 4 waves, heads 4*hg .. 4*hg+3 of projection row (b, t);
// heads < HQ are query heads (to q_out), then HKV key heads (normalised and
// rotated into k_cache at slot pos[b] + t, their value heads copied raw to
// v_cache).  The rotary angle is that of position pos[b] + t (a chain), or of
// pos[b] + depth[t] when depth is given (draft-tree rows, whose siblings share
// one absolute position: rope.py:94-122).  A row whose rotary position is
// outside the table, or a key/value row whose slot is outside [0, cap), is
// skipped.
// ---------------------------------------------------------------------------
struct RopeArgs {
  const uint16_t* qkv;
  int64_t ld_qkv;
  const uint16_t* qw;
  const uint16_t* kw;
  const uint16_t* cos;
  const uint16_t* sin;
  int rope_rows;
  const int32_t* pos;
  const int32_t* depth;   // [T] rotary position offsets, or nullptr (chain: t)
  uint16_t* q_out;
  uint16_t* k_cache;
  uint16_t* v_cache;
  int T, HQ, HKV, cap;
  float eps;
};

// One wave, one head row src[0..127]: lane i returns the normalised and
// rotated pair (o1, o2) = output dims (i, i + 64).  Shared by the standalone
// kernel and the attention prologue, so both produce the same bits.
__device__ __forceinline__ void rope_head(const uint16_t* src, const uint16_t* w, const uint16_t* cs,
                                          const uint16_t* sn, float eps, int lane, uint16_t& o1, uint16_t& o2) {
  const float x1 = bf2f(src[lane]), x2 = bf2f(src[lane + 64]);
  const float ss = wave_sum(x1 * x1 + x2 * x2);
  const float r = 1.0f / sqrtf(ss / (float)HEAD_D + eps);
  const float y1 = round_bf(bf2f(w[lane]) * round_bf(x1 * r));
  const float y2 = round_bf(bf2f(w[lane + 64]) * round_bf(x2 * r));
  const float c1 = bf2f(cs[lane]), c2 = bf2f(cs[lane + 64]);
  const float s1 = bf2f(sn[lane]), s2 = bf2f(sn[lane + 64]);
  o1 = f2bf(round_bf(y1 * c1) + round_bf(-y2 * s1));
  o2 = f2bf(round_bf(y2 * c2) + round_bf(y1 * s2));
}

__global__ void __launch_bounds__(256) qk_norm_rope_kernel(RopeArgs a) {
  const int row = blockIdx.x;                       // (b, t)
  const int head = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (head >= a.HQ + a.HKV) return;                 // wave-uniform
  const int b = row / a.T, t = row - (row / a.T) * a.T;
  const int p0 = a.pos[b];
  const int slot = p0 + t;
  const int angle = a.depth ? p0 + a.depth[t] : slot;
  if (angle < 0 || angle >= a.rope_rows) return;
  const bool is_q = head < a.HQ;
  if (!is_q && (slot < 0 || slot >= a.cap)) return;
  const uint16_t* src = a.qkv + (int64_t)row * a.ld_qkv + (int64_t)head * HEAD_D;
  uint16_t o1, o2;
  rope_head(src, is_q ? a.qw : a.kw, a.cos + (int64_t)angle * HEAD_D, a.sin + (int64_t)angle * HEAD_D, a.eps, lane,
            o1, o2);
  if (is_q) {
    uint16_t* dst = a.q_out + ((int64_t)(b * a.HQ + head) * a.T + t) * HEAD_D;
    dst[lane] = o1;
    dst[lane + 64] = o2;
  } else {
    const int kh = head - a.HQ;
    const int64_t cslot = ((int64_t)(b * a.HKV + kh) * a.cap + slot) * HEAD_D;
    a.k_cache[cslot + lane] = o1;
    a.k_cache[cslot + lane + 64] = o2;
    const uint16_t* vsrc = a.qkv + (int64_t)row * a.ld_qkv + (int64_t)(a.HQ + a.HKV + kh) * HEAD_D;
    a.v_cache[cslot + lane] = vsrc[lane];
    a.v_cache[cslot + lane + 64] = vsrc[lane + 64];
  }
}

// The same over 16-byte aligned rows, for prefill and verify row counts: 16
// lanes per head, lane j (< 8) holding dims 8j .. 8j+7 and lane j + 8 dims
// 64 + 8j .. +7, so every access is 16 bytes per lane and a rotation pair
// sits in lanes j and j ^ 8 of one 16-lane row (a DPP row rotation by 8).  The
// sum of squares is added in rope_head's order (a leaf per pair, a tree over
// 16 leaves, then the four 16-leaf sums in order; squares of bf16 are exact),
// so both kernels give the same bits.  A workgroup takes 16 heads of one row,
// value heads (copied) after the key heads.  Bound by memory: 16 x 1024 rows
// of 32 + 2 x 8 heads (402 MB) 90-96 us, where one element per lane took
// 177-182 us.
__device__ __forceinline__ u32x4 row_swap8(u32x4 v) {
  u32x4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r[q] = (uint32_t)__builtin_amdgcn_mov_dpp((int)v[q], 0x128, 0xF, 0xF, false);
  return r;
}
__device__ __forceinline__ float row_lane(float v, int sel) {   // lane 2 * sel of the 16-lane row
  const int i = __float_as_int(v);
  switch (sel) {
    case 0: return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x150, 0xF, 0xF, false));
    case 1: return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x152, 0xF, 0xF, false));
    case 2: return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x154, 0xF, 0xF, false));
    default: return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x156, 0xF, 0xF, false));
  }
}
__device__ __forceinline__ float bf_at(const u32x4& v, int e) {
  return bf2f((e & 1) ? v[e >> 1] >> 16 : v[e >> 1] & 0xFFFFu);
}

__global__ void __launch_bounds__(256) qk_norm_rope_vec_kernel(RopeArgs a) {
  const int row = blockIdx.x;                       // (b, t)
  const int head = blockIdx.y * 16 + (threadIdx.x >> 4);
  const int j = threadIdx.x & 15;                   // lane of the head: dims 8j .. 8j + 7
  if (head >= a.HQ + 2 * a.HKV) return;             // uniform over the head's 16 lanes
  const int b = row / a.T, t = row - (row / a.T) * a.T;
  const int p0 = a.pos[b];
  const int slot = p0 + t;
  const int angle = a.depth ? p0 + a.depth[t] : slot;
  if (angle < 0 || angle >= a.rope_rows) return;
  const bool is_q = head < a.HQ, is_v = head >= a.HQ + a.HKV;
  if (!is_q && (slot < 0 || slot >= a.cap)) return;
  const u32x4 x = ld16_stream(a.qkv + (int64_t)row * a.ld_qkv + (int64_t)head * HEAD_D + 8 * j);
  if (is_v) {
    const int kh = head - a.HQ - a.HKV;
    *reinterpret_cast<u32x4*>(a.v_cache + ((int64_t)(b * a.HKV + kh) * a.cap + slot) * HEAD_D + 8 * j) = x;
    return;
  }
  const u32x4 w = ld16((is_q ? a.qw : a.kw) + 8 * j);
  const u32x4 c = ld16(a.cos + (int64_t)angle * HEAD_D + 8 * j);
  const u32x4 s = ld16(a.sin + (int64_t)angle * HEAD_D + 8 * j);
  const u32x4 xo = row_swap8(x);
  float leaf[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float p = bf_at(x, e), q = bf_at(xo, e);
    leaf[e] = p * p + q * q;
  }
  const float h = ((leaf[0] + leaf[1]) + (leaf[2] + leaf[3])) + ((leaf[4] + leaf[5]) + (leaf[6] + leaf[7]));
  const float r = dpp_add(h, 0);                    // the 16-leaf sum, with the neighbour's eight
  const float ss = ((row_lane(r, 0) + row_lane(r, 1)) + row_lane(r, 2)) + row_lane(r, 3);
  const float rstd = 1.0f / sqrtf(ss / (float)HEAD_D + a.eps);
  u32x4 y;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    y[q] = (uint32_t)f2bf(bf_at(w, 2 * q) * round_bf(bf_at(x, 2 * q) * rstd)) |
           ((uint32_t)f2bf(bf_at(w, 2 * q + 1) * round_bf(bf_at(x, 2 * q + 1) * rstd)) << 16);
  const u32x4 yo = row_swap8(y);
  const bool lo = j < 8;
  u32x4 o;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint16_t v[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float mine = bf_at(y, 2 * q + e), other = bf_at(yo, 2 * q + e), sn = bf_at(s, 2 * q + e);
      v[e] = f2bf(round_bf(mine * bf_at(c, 2 * q + e)) + round_bf((lo ? -other : other) * sn));
    }
    o[q] = (uint32_t)v[0] | ((uint32_t)v[1] << 16);
  }
  if (is_q) {
    *reinterpret_cast<u32x4*>(a.q_out + ((int64_t)(b * a.HQ + head) * a.T + t) * HEAD_D + 8 * j) = o;
  } else {
    const int kh = head - a.HQ;
    *reinterpret_cast<u32x4*>(a.k_cache + ((int64_t)(b * a.HKV + kh) * a.cap + slot) * HEAD_D + 8 * j) = o;
  }
}

// ---------------------------------------------------------------------------
// Split-K GQA flash-decoding (attention.py:23-149 numerics: scores and
// softmax statistics in fp32, probabilities rounded to bf16 before the PV
// product, fp32 accumulation, one normalisation at the end).
//
// Workgroup (kv head, key range of a sequence, row block): ATTN_WAVES waves
// stream the range's keys, clipped to the row's valid length pos[b] + t + 1, 16
// keys per wave and block.  The scores of the KV head's query rows (QR = G*R of
// them, the columns of a 16-wide MFMA) come from v_mfma_f32_16x16x32_bf16 with
// the key rows as the A operand; each lane runs the online softmax of its own
// score column (4 keys of one row per block, the row max shared by the row's
// 4 lanes through permlane row swaps), and P.V runs on
// v_mfma_f32_16x16x16_bf16 with the probabilities as they sit in the score
// layout.  The waves' (m, l, acc) are merged in LDS in wave order.
// With several ranges, the partial (m, l, acc) goes to the workspace and the
// last workgroup of the (sequence, kv head) to arrive merges the ranges in
// order (no second kernel).
// ---------------------------------------------------------------------------
struct AttnArgs {
  const uint16_t* q;        // [B, HQ, R, D]
  const uint16_t* k;        // [B, HKV, cap, D]
  const uint16_t* v;
  const int32_t* pos;       // [B]: position of query row 0
  const int64_t* tree;      // [R] ancestor bit masks, or nullptr for the chain (causal) mask
  uint16_t* out;            // [B, R, HQ, D]
  float* part_o;            // [B*HKV, S, NRB, QR, D]
  float* part_ml;           // [B*HKV, S, NRB, QR, 2]
  unsigned* tickets;        // [B*HKV, NRB]
  int B, HQ, HKV, R, G, cap, S, NRB;
  int cover;                // keys the plan covers (the splits of the planned length)
  float scale;
  // ROPE instances: q rows and the new K/V rows come from the projection
  // buffer (rows (b, t)) through the per-head norm + rotary step.
  const uint16_t* qkv;
  int64_t ld_qkv;
  const uint16_t* qw;
  const uint16_t* kw;
  const uint16_t* cos;
  const uint16_t* sin;
  uint16_t* k_out;          // writable views of k / v
  uint16_t* v_out;
  int rope_rows;
  float eps;
  const int32_t* depth;     // ROPE with TREE: [R] rotary offsets (row t rotates by pos + depth[t])
  int rb_xcd;               // row blocks of one (b, kv head, split) launched 8 apart (one XCD)
};


// Reductions over lanes l, l^16, l^32, l^48 (the four 16-lane rows), by
// row swaps: every lane ends with the same value.
__device__ __forceinline__ float rows4_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows4_sum(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// VEC floats per lane, device-coherent (sc1), at byte off of descriptor r.
template <int VEC>
__device__ __forceinline__ void store_agent_vec(__amdgpu_buffer_rsrc_t r, int off, const float* v) {
  if constexpr (VEC == 4) {
    __builtin_amdgcn_raw_buffer_store_b128(
        u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])}, r, off, 0, 16);
  } else if constexpr (VEC == 2) {
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(v[0]), __float_as_uint(v[1])}, r, off, 0, 16);
  } else {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[0]), r, off, 0, 16);
  }
}
template <int VEC>
__device__ __forceinline__ void load_agent_vec(__amdgpu_buffer_rsrc_t r, int off, float* v) {
  if constexpr (VEC == 4) {
    const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(x[e]);
  } else if constexpr (VEC == 2) {
    const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 16);
    v[0] = __uint_as_float(x[0]);
    v[1] = __uint_as_float(x[1]);
  } else {
    v[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 16));
  }
}

// Key ranges.  The host knows only the planned length, so the S ranges of a
// sequence are cut here, from its own length, in grains of KEY_GRAIN keys:
// ranges of the planned length left most workgroups of a shorter sequence
// without keys (one sequence, 2000 of 4096 planned keys: half of them, 14.2 us
// against 9.9; 4 of 4000 of 8192: 19.8 against 14.4).  A sequence of at most
// WHOLE_GRAINS keeps one range: another block of 16 keys per wave costs less
// than 1 us, publishing and merging ranges about 1.5 (one query row, 300 keys:
// 7.3 us in one range, 8.1 in three; 16 sequences of 300: 9.4 and 10.4; past it,
// one of 500 keys 9.8 in one range, 8.7 in four; 16 of up to 500 10.6 and 10.3).
constexpr int KEY_GRAIN = 64, WHOLE_GRAINS = 6;
struct KeyRange {
  int pos, len;        // the sequence's position and keys
  int count, grains;   // its ranges, grains per range (the last may be shorter)
};
__device__ __forceinline__ KeyRange key_range(const AttnArgs& a, int b) {
  KeyRange k;
  k.pos = a.pos[b];
  k.len = max(min(min(k.pos + a.R, a.cap), a.cover), 0);
  const int total = max((k.len + KEY_GRAIN - 1) / KEY_GRAIN, 1);
  k.grains = total <= WHOLE_GRAINS ? total : max((total + a.S - 1) / a.S, 2);
  k.count = (total + k.grains - 1) / k.grains;
  return k;
}

// A wave's LDS slot: one block of 16 keys (K rows, then V rows); after the
// keys the space holds the waves' partial accumulators.
constexpr int KV_SLOT = 2 * 16 * 2 * HEAD_D;
constexpr int ACC_LD = HEAD_D + 8;   // (the lanes of one f32x4 store hold 16 different rows, and 128-float rows
                                     // put all of them on the same banks)
constexpr int attn_lds(int QR, int waves) {
  const int ring = waves * KV_SLOT, acc = waves * QR * ACC_LD * 4;
  return ring > acc ? ring : acc;
}

template <int QR, int ATTN_WAVES, bool TREE, bool ROPE = false>
__global__ void __launch_bounds__(64 * ATTN_WAVES, 4) decode_attn_kernel(AttnArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char dyn[];
  __shared__ float s_m[ATTN_WAVES][QR], s_l[ATTN_WAVES][QR];
  float* const s_acc = reinterpret_cast<float*>(dyn);   // [wave][row][ACC_LD]
  __shared__ int s_last;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int dg = lane & 15, kr = lane >> 4;
  // Workgroup (key range, sequence, KV head, row block): query rows rbk*QR ..
  // +QR-1 of the KV head's G*R rows (row = t*G + g).  The range is the slowest
  // index: ranges that a short sequence does not need leave every XCD alike.
  // With rb_xcd, launch position 8i + x runs row block i mod NRB of the (range,
  // sequence, KV head) unit 8(i / NRB) + x: workgroups are dealt to the 8 XCDs
  // round-robin, so the row blocks of one unit run side by side on one XCD and
  // the later ones read the keys from its L2.
  int unit, rbk;
  if (a.rb_xcd) {
    const int i = blockIdx.x >> 3, x = blockIdx.x & 7;
    unit = 8 * (i / a.NRB) + x;
    rbk = i % a.NRB;
  } else {
    unit = blockIdx.x / a.NRB;
    rbk = blockIdx.x - unit * a.NRB;
  }
  const int sb = unit / a.HKV, kh = unit - sb * a.HKV;
  const int split = sb / a.B, b = sb - split * a.B, bk = b * a.HKV + kh;
  const KeyRange rng = key_range(a, b);
  if (split >= rng.count) return;   // uniform: nothing left for this workgroup
  const int rows = a.G * a.R;
  const int pos = rng.pos;
  const int start = split * rng.grains * KEY_GRAIN;
  const int range_end = start + rng.grains * KEY_GRAIN;
  const bool last_range = split == rng.count - 1;
  // keys this workgroup may touch: below the longest row's length, the cache
  // and the planned length
  const int end = min(range_end, rng.len);

  // Wave w processes the 16-key blocks start + 16 (w + ATTN_WAVES i).  A
  // block's K and V rows (4 KB each) are loaded straight into the wave's own
  // LDS slot, four whole 256-byte rows per load, and read back in the layouts
  // of the two products.  Each half of the slot is loaded again as soon as its
  // fragments are in registers, so four to eight loads of a wave are always in
  // flight, and nothing is staged in registers: 119 of them at most, two
  // workgroups per CU (blocks staged in registers took 180 and one: 64
  // sequences of up to 200 keys 14.4 us, now 11.5; 5 x 8 tree rows of up to 1000
  // 16.4 us, now 13.1).  A second slot per wave is slower (16 sequences of up
  // to 500 keys 10.6 -> 10.9 us, 64 of up to 200 12.0 -> 15.6): it takes the CU's
  // second workgroup, and more requests in flight per wave bring nothing.  Long
  // contexts are bound by memory (2 x 32000 keys 44.7 us, 5.9 TB/s), short ones
  // by the chain of round trips position, projection row, keys, merge.
  //  * Scores: S^T[key][row] = K[16 keys, 128] . Q^T by four MFMAs with K as
  //    the A operand (lane l: key l%16, dims 32s + 8*(l/16)).  Chunk c (16
  //    bytes) of key r lies at position c ^ r of its row, so the 16 keys of a
  //    fragment read fall on 16 bank groups.  Lane l then holds keys
  //    4*(l/16) + i (i < 4) of query row l%16.
  //  * P.V: lane l reads dims 8*(l%16) .. +7 of keys 4*(l/16) + j, the keys of
  //    its scores.
  const uint32_t slot_off =
      (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)dyn) + wave * KV_SLOT;
  const char* const slot = dyn + wave * KV_SLOT;
  const int64_t kv_row0 = (int64_t)bk * a.cap;
  const int wk0 = start + 16 * wave;
  const int nblk = wk0 < end ? (end - 1 - wk0) / (16 * ATTN_WAVES) + 1 : 0;   // blocks of this wave (uniform)
  const int kx16 = 16 * (dg ^ kr);   // chunk dg ^ r of row r = kr + 4 j lies at kx16 ^ 64 j
  // Keys past `end` in the wave's last block load its last valid row again and
  // are masked.  K and V rows are read once per launch: non-temporal.
  auto issue = [&](int i, auto what) {
    constexpr bool V = decltype(what)::value;
    const int n0 = wk0 + 16 * ATTN_WAVES * i;
    const int lim = end - 1 - n0;   // >= 0
    const i32x4 rows16 = buf_of((V ? a.v : a.k) + (kv_row0 + n0) * HEAD_D, 16 * 2 * HEAD_D);
    int kr256 = 2 * HEAD_D * kr;   // (the offsets are formed again for each block: eight of them kept would spill)
    asm volatile("" : "+v"(kr256));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      load_lds16<true>(slot_off + (V ? 4096 : 0) + 1024 * j,
                       min(kr256 | (1024 * j), lim * (2 * HEAD_D)) | (V ? 16 * dg : kx16 ^ (64 * j)), rows16, 0);
  };
  const std::false_type keys{};
  const std::true_type values{};
  const int r16 = lane & 15;
  const int my_gr = rbk * QR + r16;
  const bool my_real = r16 < QR && my_gr < rows;
  const int my_t = my_gr / a.G;
  // (requested before any key, so that nothing waits for it behind those)
  long long my_tree = 0ll;
  if constexpr (TREE) my_tree = my_real ? (long long)a.tree[min(my_t, a.R - 1)] : 0ll;
  // The first block's keys are on their way while the query rows are formed,
  // unless it holds rows that this launch writes (the caches below pos are not
  // written).  Not its values: loads return in order, so everything the query
  // rows need would wait behind them too (with the values: 16 sequences of 300
  // keys, one row, 9.2 us, without 9.0; 64 of up to 200 12.0 and 11.5; 32 x 4
  // tree rows of up to 500 15.6 and 15.2; 5 x 8 of up to 1000 13.5 and 13.1).
  const bool early = nblk > 0 && wk0 + 16 <= min(end, pos);   // (uniform)
  if (early) issue(0, keys);
  // (ancestor masks wait in LDS for the few masked blocks; every wave stores the
  // same values and reads them back itself, in order)
  __shared__ long long s_tree[TREE ? QR : 1];
  auto issue_rest = [&]() {
    if (TREE && r16 < QR) s_tree[r16] = my_tree;
    if (nblk > 0) {
      if (!early) issue(0, keys);
      issue(0, values);
    }
  };

  // Query rows r = t*G + g (head kh*G + g, query row t) as the B operand of
  // v_mfma_f32_16x16x32_bf16: lane l supplies row l%16, dims 32s + 8*(l/16)
  // for K step s (rows >= QR are zero columns).
  bf16x8 qb[HEAD_D / 32];
  if constexpr (ROPE) {
    // Query rows through the norm + rotary step (one wave per row), into LDS.
    // Row t rotates by position pos + t (chain) or pos + depth[t] (draft
    // tree); a row whose rotary position is outside the table stays zero.
    __shared__ __attribute__((aligned(16))) uint16_t s_q[QR][HEAD_D];
    const int T = a.R;
    auto rot_of = [&](int t) { return TREE ? pos + a.depth[t] : pos + t; };
    for (int r = wave; r < QR; r += ATTN_WAVES) {   // wave-uniform
      const int gr = rbk * QR + r;
      const int t = gr / a.G, g = gr - (gr / a.G) * a.G;
      const int rot = gr < rows ? rot_of(t) : -1;
      uint16_t o1 = 0, o2 = 0;
      if (rot >= 0 && rot < a.rope_rows)
        rope_head(a.qkv + (int64_t)(b * T + t) * a.ld_qkv + (int64_t)(kh * a.G + g) * HEAD_D, a.qw,
                  a.cos + (int64_t)rot * HEAD_D, a.sin + (int64_t)rot * HEAD_D, a.eps, lane, o1, o2);
      s_q[r][lane] = o1;
      s_q[r][lane + 64] = o2;
    }
    // The new K/V rows of this (b, kv head) are written by every workgroup
    // whose key range holds their slot (the last range also takes slots past
    // the planned length), before any of its K/V loads: the stores are
    // complete (vmcnt 0) before the barrier.  Only those workgroups read
    // these slots, and each reads them after its own stores; several row
    // blocks write the same values, so a read never sees an older row.
    // Row t goes to wave (QR + t) mod ATTN_WAVES, so with fewer query rows
    // than waves the K/V rows run beside the query rows, not after them.
    constexpr int KV_WAVE0 = QR % ATTN_WAVES;
    for (int t = (wave - KV_WAVE0 + ATTN_WAVES) % ATTN_WAVES; t < T; t += ATTN_WAVES) {   // wave-uniform
      const int slot = pos + t, rot = rot_of(t);
      const bool mine = slot >= start && (slot < range_end || last_range);
      if (mine && slot < a.cap && rot >= 0 && rot < a.rope_rows) {
        const uint16_t* row = a.qkv + (int64_t)(b * T + t) * a.ld_qkv;
        uint16_t o1, o2;
        rope_head(row + (int64_t)(a.HQ + kh) * HEAD_D, a.kw, a.cos + (int64_t)rot * HEAD_D,
                  a.sin + (int64_t)rot * HEAD_D, a.eps, lane, o1, o2);
        const int64_t cs = ((int64_t)bk * a.cap + slot) * HEAD_D;
        a.k_out[cs + lane] = o1;
        a.k_out[cs + lane + 64] = o2;
        const uint16_t* vsrc = row + (int64_t)(a.HQ + a.HKV + kh) * HEAD_D;
        a.v_out[cs + lane] = vsrc[lane];
        a.v_out[cs + lane + 64] = vsrc[lane + 64];
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    issue_rest();
    const bool real = r16 < QR;
#pragma unroll
    for (int st = 0; st < HEAD_D / 32; ++st) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(&s_q[min(r16, QR - 1)][32 * st + 8 * kr]);
      qb[st] = __builtin_bit_cast(bf16x8, real ? v : u32x4{0u, 0u, 0u, 0u});
    }
  } else {
    const int gr = rbk * QR + r16;
    const int t = gr / a.G, g = gr - (gr / a.G) * a.G;
    const bool real = r16 < QR && gr < rows;
    const uint16_t* qp =
        a.q + ((int64_t)(b * a.HQ + kh * a.G + min(g, a.G - 1)) * a.R + min(t, a.R - 1)) * HEAD_D + 8 * kr;
#pragma unroll
    for (int st = 0; st < HEAD_D / 32; ++st) {
      const u32x4 v = ld16(qp + 32 * st);
      qb[st] = __builtin_bit_cast(bf16x8, real ? v : u32x4{0u, 0u, 0u, 0u});
    }
    issue_rest();
  }
  // Lane l owns query row l%16 (its MFMA column) and, in each 16-key block,
  // keys 4*(l/16) .. +3 of that row; the 4 lanes of a row share its running
  // max and keep partial sums.  acc[c][k] = O[row l%16][dim 8*(4*(l/16)+k) + c].
  // Visibility of key n to the row: keys before pos always; key pos + j
  // (j < R) iff j <= t (chain) or bit j of tree[t] is set (draft tree).
  const int row_lim = my_real ? pos + my_t : -1;   // last visible key of the row (chain)

  float m = -INFINITY, l = 0.f;
  f32x4 acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};

  // MASKED: the block may hold keys a row must not see; blocks wholly below
  // min(end, pos) need no masks (every real row sees every key below pos, and
  // padding rows are never written out).
  float p[4];
  auto softmax = [&](int n0, const f32x4& sacc, auto masked) {
    constexpr bool MASKED = decltype(masked)::value;
    const int key0 = n0 + 4 * kr;   // keys key0 .. key0+3 of this lane's row
    float sc[4];
    float mx = m;
    long long row_tree = 0ll;
    if constexpr (MASKED && TREE) row_tree = s_tree[min(r16, QR - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float dot = sacc[j] * a.scale;
      if constexpr (MASKED) {
        const int key = key0 + j;
        bool vis;
        if constexpr (TREE) {
          const int rel = key - pos;
          vis = row_lim >= 0 && (rel < 0 || (rel < a.R && ((row_tree >> rel) & 1ll)));
        } else {
          vis = key <= row_lim;
        }
        sc[j] = (key < end && vis) ? dot : -INFINITY;
      } else {
        sc[j] = dot;
      }
      mx = fmaxf(mx, sc[j]);
    }
    mx = rows4_max(mx);
    const float msafe = mx == -INFINITY ? 0.f : mx;
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = __expf(sc[j] - msafe);
    // Rescale only when some row's max moved (alpha == 1 elsewhere, so the
    // skipped multiplications are exact).
    if (__builtin_amdgcn_ballot_w64(mx != m)) {   // wave-uniform
      const float alpha = __expf(m - msafe);
      l *= alpha;
#pragma unroll
      for (int c = 0; c < 8; ++c) acc[c] *= alpha;
    }
    l += (p[0] + p[1]) + (p[2] + p[3]);
    m = mx;
  };
  const int unmasked_end = min(end, pos);   // keys below it need no masks
  for (int i = 0; i < nblk; ++i) {
    const bool more = i + 1 < nblk;
    const int n0 = wk0 + 16 * ATTN_WAVES * i;
    wait_loads<4>();   // the keys; the values may be in flight
    bf16x8 kf[HEAD_D / 32];
#pragma unroll
    for (int st = 0; st < HEAD_D / 32; ++st)
      kf[st] = *reinterpret_cast<const bf16x8*>(slot + 2 * HEAD_D * r16 + 16 * ((4 * st + kr) ^ r16));
    wait_lds();
    if (more) issue(i + 1, keys);   // (the keys' half of the slot is in registers)
    f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < HEAD_D / 32; ++st)
      sacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[st], qb[st], sacc, 0, 0, 0);
    if (n0 + 16 <= unmasked_end) softmax(n0, sacc, std::false_type{});   // (uniform)
    else softmax(n0, sacc, std::true_type{});
    if (more) wait_loads<4>();   // the values
    else wait_loads<0>();
    u32x4 vv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) vv[j] = *reinterpret_cast<const u32x4*>(slot + 4096 + 2 * HEAD_D * (4 * kr + j) + 16 * dg);
    wait_lds();
    if (more) issue(i + 1, values);
    // P.V on MFMA: O^T[dims][rows] += V^T[dims][16 keys] . P^T[16 keys][rows].
    // B = the probabilities as they sit (lane l: row l%16, keys 4*(l/16)+j),
    // rounded to bf16 (RNE) as the reference's tl.dot does; A for dim offset
    // c = V[keys 4*(l/16)+j][8*(l%16) + c], key pairs packed by v_perm.
    const bf16x2 p01 = {(__bf16)p[0], (__bf16)p[1]}, p23 = {(__bf16)p[2], (__bf16)p[3]};
    const s16x4 pb = __builtin_bit_cast(s16x4, u32x2{__builtin_bit_cast(uint32_t, p01), __builtin_bit_cast(uint32_t, p23)});
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t sel = h ? 0x07060302u : 0x05040100u;
        const u32x2 vt = {__builtin_amdgcn_perm(vv[1][c4], vv[0][c4], sel), __builtin_amdgcn_perm(vv[3][c4], vv[2][c4], sel)};
        acc[2 * c4 + h] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, vt), pb, acc[2 * c4 + h], 0, 0, 0);
      }
  }
  __syncthreads();   // the slots give way to the partial accumulators

  // Per wave: the row sums of the 4 lanes of each row, then the waves'
  // results merge in LDS in wave order.
  const float lw = rows4_sum(l);
  if (r16 < QR) {
    if (kr == 0) {
      s_m[wave][r16] = m;
      s_l[wave][r16] = lw;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float* dst = s_acc + (wave * QR + r16) * ACC_LD + 8 * (4 * kr + k);
      *reinterpret_cast<f32x4*>(dst) = f32x4{acc[0][k], acc[1][k], acc[2][k], acc[3][k]};
      *reinterpret_cast<f32x4*>(dst + 4) = f32x4{acc[4][k], acc[5][k], acc[6][k], acc[7][k]};
    }
  }
  __syncthreads();
  // Per row: the merged max, each wave's weight and the merged sum (waves in
  // order); then every output of the real rows combines the waves' partial
  // accumulators with those weights.
  __shared__ float s_w[ATTN_WAVES][QR], s_rowM[QR], s_rowL[QR];
  if (threadIdx.x < QR) {
    const int r = threadIdx.x;
    float M = -INFINITY;
#pragma unroll
    for (int wv = 0; wv < ATTN_WAVES; ++wv) M = fmaxf(M, s_m[wv][r]);
    float L = 0.f;
#pragma unroll
    for (int wv = 0; wv < ATTN_WAVES; ++wv) {
      const float w = s_m[wv][r] == -INFINITY ? 0.f : __expf(s_m[wv][r] - M);
      s_w[wv][r] = w;
      L += w * s_l[wv][r];
    }
    s_rowM[r] = M;
    s_rowL[r] = L;
  }
  __syncthreads();
  const bool single = rng.count == 1;
  const int nreal = min(QR, rows - rbk * QR);   // rows of this block that exist
  // Every thread takes VEC neighbouring outputs of the QR x HEAD_D.
  constexpr int VEC = QR * HEAD_D / (64 * ATTN_WAVES);
  static_assert(VEC * 64 * ATTN_WAVES == QR * HEAD_D && (VEC == 1 || VEC == 2 || VEC == 4), "outputs of a thread");
  const int r = threadIdx.x * VEC / HEAD_D, d = threadIdx.x * VEC % HEAD_D;
  auto store_out = [&](const float* O, float L) {
    const int gr = rbk * QR + r;
    const int t = gr / a.G, g = gr - (gr / a.G) * a.G;
    uint16_t* const o = a.out + ((int64_t)(b * a.R + t) * a.HQ + kh * a.G + g) * HEAD_D + d;
    uint16_t y[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) y[e] = f2bf(L > 0.f ? O[e] / L : 0.f);
    if (VEC > 1 && (reinterpret_cast<uintptr_t>(a.out) & (2 * VEC - 1)) == 0) {   // (uniform)
      uint32_t w[VEC > 1 ? VEC / 2 : 1];
#pragma unroll
      for (int e = 0; e < VEC / 2; ++e) w[e] = (uint32_t)y[2 * e] | ((uint32_t)y[2 * e + 1] << 16);
      __builtin_memcpy(__builtin_assume_aligned(o, 2 * VEC), w, 2 * VEC);
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[e] = y[e];
    }
  };
  const int64_t part0 = ((int64_t)bk * a.S * a.NRB + rbk) * QR;   // partial row of (range 0, row 0)
  const int64_t stride = (int64_t)a.NRB * QR;                     // partial rows per range
  const auto part_rows = [&](int64_t pr, int n) {                 // n partial rows from pr
    return __builtin_amdgcn_make_buffer_rsrc(a.part_o + pr * HEAD_D, 0, n * HEAD_D * 4, 0x00020000);
  };
  {
    float O[VEC] = {};
#pragma unroll
    for (int wv = 0; wv < ATTN_WAVES; ++wv) {
      float v[VEC];
      __builtin_memcpy(v, __builtin_assume_aligned(&s_acc[(wv * QR + r) * ACC_LD + d], 4 * VEC), 4 * VEC);
#pragma unroll
      for (int e = 0; e < VEC; ++e) O[e] += s_w[wv][r] * v[e];
    }
    if (single) {
      if (r < nreal) store_out(O, s_rowL[r]);
      return;
    }
    if (r < nreal) {
      const int64_t pr = part0 + split * stride;
      store_agent_vec<VEC>(part_rows(pr, QR), 4 * VEC * threadIdx.x, O);
      if (d == 0) {
        store_agent(&a.part_ml[2 * (pr + r)], s_rowM[r]);
        store_agent(&a.part_ml[2 * (pr + r) + 1], s_rowL[r]);
      }
    }
  }

  // Last workgroup of this (sequence, KV head, row block) merges the ranges.
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) s_last = take_ticket(&a.tickets[bk * a.NRB + rbk], (unsigned)rng.count) ? 1 : 0;
  __syncthreads();
  if (!s_last || r >= nreal) return;
  // A thread folds its outputs of the ranges in order, a batch at a time with
  // all its loads issued before any arithmetic: the merge is a chain of memory
  // round trips, one per batch (one row, 32 ranges: two trips instead of the 16
  // of a pass over the maxima and batches of four).
  float M = -INFINITY, L = 0.f, O[VEC] = {};
  const auto fold = [&](int s0, auto batch) {
    constexpr int MB = decltype(batch)::value;
    const int n = min(rng.count - s0, MB);
    const auto src = part_rows(part0 + s0 * stride, (int)((n - 1) * stride) + QR);
    float ms[MB], ls[MB], os[MB][VEC];
#pragma unroll
    for (int k = 0; k < MB; ++k) {
      const int s = min(k, n - 1);   // (past the end: the last again, not added)
      const int64_t pr = part0 + (s0 + s) * stride + r;
      ms[k] = load_agent(&a.part_ml[2 * pr]);
      ls[k] = load_agent(&a.part_ml[2 * pr + 1]);
      load_agent_vec<VEC>(src, (int)(s * stride) * (HEAD_D * 4) + 4 * VEC * (int)threadIdx.x, os[k]);
    }
    float Mb = M;
#pragma unroll
    for (int k = 0; k < MB; ++k) Mb = fmaxf(Mb, ms[k]);
    if (Mb == -INFINITY) return;   // no visible key so far
    const float keep = __expf(M - Mb);   // 0 before the first visible key
    L *= keep;
#pragma unroll
    for (int e = 0; e < VEC; ++e) O[e] *= keep;
    M = Mb;
#pragma unroll
    for (int k = 0; k < MB; ++k) {
      if (k < n) {
        const float w = __expf(ms[k] - M);
        L += w * ls[k];
#pragma unroll
        for (int e = 0; e < VEC; ++e) O[e] += w * os[k][e];
      }
    }
  };
  int s0 = 0;
  for (; rng.count - s0 > 8; s0 += 16) fold(s0, std::integral_constant<int, 16>{});
  if (s0 < rng.count) fold(s0, std::integral_constant<int, 8>{});
  store_out(O, L);
}

}  // namespace sk

namespace {

constexpr int kAttnMaxRows = 64;   // (HQ/HKV) * R

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
int cdiv(int a, int b) { return (a + b - 1) / b; }
size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// Waves per workgroup, 16 keys each per block.
constexpr int kAttnWaves = 8;

struct AttnPlan {
  int QR = 0, NRB = 0, S = 0, split_len = 0;
  size_t tickets = 0, part_o = 0, part_ml = 0, need = 0;
};

// S: the most key ranges of a (sequence, KV head) pair (the kernel cuts them
// from each sequence's length: key_range), no more than the planned length has
// workgroup blocks (16 keys per wave).  split_len: the planned length over S,
// in whole blocks; S of them are the keys the plan covers.
int attn_plan(int B, int HQ, int HKV, int D, int R, int cap, int max_len, int nsplit, AttnPlan* p) {
  if (B < 1 || HKV < 1 || HQ < HKV || HQ % HKV != 0 || R < 1 || cap < 1 || D != sk::HEAD_D) return SK_ERR_SHAPE;
  const int G = HQ / HKV;
  const int rows = G * R;
  if (rows > kAttnMaxRows) return SK_ERR_SHAPE;
  // Query rows per workgroup: up to 16, the columns of the MFMA tiles (the
  // per-lane state does not grow with them); more rows take several row
  // blocks, each streaming the keys once more.  The smaller instances have
  // less prologue and epilogue work (one row, 300 keys: 7.3 us with 4 rows, 7.5
  // with 8; 16 sequences of up to 1088 keys, R = 2: 18.0 with 8, 18.1 with 16).
  p->QR = rows <= 4 ? 4 : rows <= 8 ? 8 : 16;
  p->NRB = cdiv(rows, p->QR);
  const int work = max_len > 0 && max_len < cap ? max_len : cap;
  const int block = 16 * kAttnWaves;   // keys per workgroup block
  const int blocks = cdiv(work, block);
  int S = nsplit;
  if (S <= 0) {
    // One query row: about one workgroup per CU (256; 16 x 2000 keys in one
    // range 28.7 us, in two 25.1, in three 26.1, in four 24.7).  Verify rows
    // (R > 1): half of that (16 x 8 rows of up to 1000 keys in one range 18.9
    // us, in two 22.3; 16 x 2 rows 17.9 and 17.2).
    const long pairs = (long)B * HKV, groups = pairs * p->NRB;
    const long target = R == 1 ? 256 : 128;
    S = (int)((target + pairs - 1) / pairs);
    // Between one workgroup per CU and two, some CUs hold two and the rest wait
    // for them; then only as many ranges as fit the CUs once.  3 x 16000 keys
    // 45.0 us in 11 ranges (264 workgroups), 35.3 in 10 (240); 12 x 4000 42.4
    // in 3 (288), 34.2 in 2 (192); 6 x 8 tree rows of up to 4000 35.3 in 3 (two
    // row blocks each, 288), 29.3 in 2 (192).
    if (groups * S > 256 && groups * S < 512) S = (int)(256 / groups);
    if (S > 32) S = 32;
  }
  if (S > blocks) S = blocks;
  if (S < 1) S = 1;
  p->split_len = cdiv(blocks, S) * block;
  p->S = cdiv(work, p->split_len);
  if (p->S == 1) {
    p->need = 0;
    return SK_OK;
  }
  const size_t pairs = (size_t)B * HKV * p->NRB;
  p->tickets = align256(pairs * sizeof(unsigned));
  p->part_o = pairs * p->S * p->QR * sk::HEAD_D * sizeof(float);
  p->part_ml = pairs * p->S * p->QR * 2 * sizeof(float);
  p->need = p->tickets + align256(p->part_o) + p->part_ml;
  return SK_OK;
}

int attn_launch_status() { return hipGetLastError() == hipSuccess ? SK_OK : SK_ERR_LAUNCH; }

int attn_device_ok() {
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return SK_ERR_DEVICE;
  return strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? SK_OK : SK_ERR_DEVICE;
}

}  // namespace

extern "C" {

int sk_qk_norm_rope_cache_bf16(const sk_bf16* qkv, int64_t ld_qkv, const sk_bf16* q_norm_w, const sk_bf16* k_norm_w,
                               const sk_bf16* cos, const sk_bf16* sin, int rope_rows, const int32_t* pos,
                               const int32_t* depth, sk_bf16* q_out, sk_bf16* k_cache, sk_bf16* v_cache, int B, int T,
                               int HQ, int HKV, int D, int cap, float eps, hipStream_t stream) {
  if (B < 0 || T < 0 || HQ < 1 || HKV < 1 || cap < 1 || rope_rows < 1 || D != sk::HEAD_D) return SK_ERR_SHAPE;
  if (ld_qkv < (int64_t)(HQ + 2 * HKV) * D) return SK_ERR_SHAPE;
  if ((long)B * T > 0x7FFFFFFFL) return SK_ERR_SHAPE;
  if (B == 0 || T == 0) return SK_OK;
  if (!qkv || !q_norm_w || !k_norm_w || !cos || !sin || !pos || !q_out || !k_cache || !v_cache) return SK_ERR_NULL;
  int st = attn_device_ok();
  if (st) return st;
  sk::RopeArgs a;
  a.qkv = qkv;
  a.ld_qkv = ld_qkv;
  a.qw = q_norm_w;
  a.kw = k_norm_w;
  a.cos = cos;
  a.sin = sin;
  a.rope_rows = rope_rows;
  a.pos = pos;
  a.depth = depth;
  a.q_out = q_out;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.T = T;
  a.HQ = HQ;
  a.HKV = HKV;
  a.cap = cap;
  a.eps = eps;
  // 16-byte accesses from about a thousand heads on: with fewer, one lane's
  // chain of eight elements costs more than the loads it saves (32 + 2 x 8 heads,
  // us, one element per lane against eight: 8 rows 2.54, 2.63; 24 2.64, 2.68; 32
  // 2.77, 2.72; 128 3.75, 3.39).  Both give the same bits.
  const bool many = (int64_t)B * T * (HQ + 2 * HKV) >= 1024;
  if (many && aligned16(qkv) && (ld_qkv & 7) == 0 && aligned16(q_norm_w) && aligned16(k_norm_w) && aligned16(cos) &&
      aligned16(sin) && aligned16(q_out) && aligned16(k_cache) && aligned16(v_cache)) {
    sk::qk_norm_rope_vec_kernel<<<dim3((unsigned)(B * T), (unsigned)cdiv(HQ + 2 * HKV, 16)), dim3(256), 0, stream>>>(a);
    return attn_launch_status();
  }
  const unsigned groups = (unsigned)cdiv(HQ + HKV, 4);
  sk::qk_norm_rope_kernel<<<dim3((unsigned)(B * T), groups), dim3(256), 0, stream>>>(a);
  return attn_launch_status();
}

size_t sk_decode_attention_workspace_bytes(int B, int HQ, int HKV, int D, int R, int cap, int max_len, int nsplit) {
  AttnPlan p;
  if (attn_plan(B, HQ, HKV, D, R, cap, max_len, nsplit, &p)) return 0;
  return p.need;
}

}  // extern "C"

namespace {

template <int QR, bool TREE, bool ROPE>
int attn_launch(const sk::AttnArgs& a, unsigned grid, hipStream_t stream) {
  constexpr int lds = sk::attn_lds(QR, kAttnWaves);
  const auto fn = &sk::decode_attn_kernel<QR, kAttnWaves, TREE, ROPE>;
  // (once per device: the runtime call is host time of every eager call)
  static std::atomic<unsigned long long> allowed{0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return SK_ERR_DEVICE;
  const unsigned long long bit = dev >= 0 && dev < 64 ? 1ull << dev : 0ull;
  if (!(allowed.load(std::memory_order_acquire) & bit)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds) !=
        hipSuccess)
      return SK_ERR_LAUNCH;
    allowed.fetch_or(bit, std::memory_order_release);
  }
  fn<<<dim3(grid), dim3(64 * kAttnWaves), lds, stream>>>(a);
  return attn_launch_status();
}

// Fills the plan-dependent fields of a and launches the instance for
// (QR, tree, rope).
int attn_run(const AttnPlan& p, sk::AttnArgs& a, int B, int HQ, int HKV, int R, int cap, float scale, void* ws,
             bool rope, hipStream_t stream) {
  if (p.need > 0) {
    char* w = static_cast<char*>(ws);
    a.tickets = reinterpret_cast<unsigned*>(w);
    a.part_o = reinterpret_cast<float*>(w + p.tickets);
    a.part_ml = reinterpret_cast<float*>(w + p.tickets + align256(p.part_o));
  }
  a.HQ = HQ;
  a.HKV = HKV;
  a.R = R;
  a.G = HQ / HKV;
  a.cap = cap;
  a.B = B;
  a.S = p.S;
  a.cover = (int)std::min<int64_t>((int64_t)p.S * p.split_len, cap);
  a.NRB = p.NRB;
  a.rb_xcd = p.NRB > 1 && (B * HKV * p.S) % 8 == 0;
  a.scale = scale;
  const unsigned grid = (unsigned)(B * HKV * p.NRB * p.S);
  const auto launch = [&](auto tree_c, auto rope_c) {
    constexpr bool TREE = decltype(tree_c)::value, ROPE = decltype(rope_c)::value;
    if (p.QR == 4) return attn_launch<4, TREE, ROPE>(a, grid, stream);
    if (p.QR == 8) return attn_launch<8, TREE, ROPE>(a, grid, stream);
    return attn_launch<16, TREE, ROPE>(a, grid, stream);
  };
  const std::true_type yes{};
  const std::false_type no{};
  if (rope) return a.tree ? launch(yes, yes) : launch(no, yes);
  return a.tree ? launch(yes, no) : launch(no, no);
}

bool overlaps(const void* a, size_t na, const void* b, size_t nb) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return x < y + nb && y < x + na;
}

// The fused rotary step + attention of both entry points: tree and depth
// (the draft-tree masks and rotary offsets, both [R]) or both nullptr (chain).
int rope_attention(const sk_bf16* qkv, int64_t ld_qkv, const sk_bf16* q_norm_w, const sk_bf16* k_norm_w,
                   const sk_bf16* cos, const sk_bf16* sin, int rope_rows, float eps, sk_bf16* k_cache,
                   sk_bf16* v_cache, const int32_t* pos, const int64_t* tree, const int32_t* depth, sk_bf16* out,
                   int B, int HQ, int HKV, int D, int R, int cap, int max_len, float scale, int nsplit, void* ws,
                   size_t ws_bytes, hipStream_t stream) {
  if (B < 0) return SK_ERR_SHAPE;
  if (B == 0) return SK_OK;
  AttnPlan p;
  int st = attn_plan(B, HQ, HKV, D, R, cap, max_len, nsplit, &p);
  if (st) return st;
  if (rope_rows < 1 || ld_qkv < (int64_t)(HQ + 2 * HKV) * D || (long)B * R > 0x7FFFFFFFL) return SK_ERR_SHAPE;
  if (!qkv || !q_norm_w || !k_norm_w || !cos || !sin || !k_cache || !v_cache || !pos || !out) return SK_ERR_NULL;
  if (!aligned16(k_cache) || !aligned16(v_cache)) return SK_ERR_ALIGN;
  if (p.need > 0 && (!ws || ws_bytes < p.need)) return SK_ERR_WORKSPACE;
  // The output is written while the projection rows and the caches are read.
  const size_t out_bytes = (size_t)B * R * HQ * D * 2, cache_bytes = (size_t)B * HKV * cap * D * 2;
  const size_t qkv_bytes = ((size_t)(B * R - 1) * ld_qkv + (size_t)(HQ + 2 * HKV) * D) * 2;
  if (overlaps(out, out_bytes, qkv, qkv_bytes) || overlaps(out, out_bytes, k_cache, cache_bytes) ||
      overlaps(out, out_bytes, v_cache, cache_bytes) || overlaps(k_cache, cache_bytes, v_cache, cache_bytes) ||
      overlaps(k_cache, cache_bytes, qkv, qkv_bytes) || overlaps(v_cache, cache_bytes, qkv, qkv_bytes))
    return SK_ERR_ALIAS;
  st = attn_device_ok();
  if (st) return st;
  sk::AttnArgs a;
  memset(&a, 0, sizeof(a));
  a.k = k_cache;
  a.v = v_cache;
  a.pos = pos;
  a.out = out;
  a.qkv = qkv;
  a.ld_qkv = ld_qkv;
  a.qw = q_norm_w;
  a.kw = k_norm_w;
  a.cos = cos;
  a.sin = sin;
  a.k_out = k_cache;
  a.v_out = v_cache;
  a.rope_rows = rope_rows;
  a.eps = eps;
  a.tree = tree;
  a.depth = depth;
  return attn_run(p, a, B, HQ, HKV, R, cap, scale, ws, true, stream);
}


}  // namespace

extern "C" {

int sk_decode_attention_bf16(const sk_bf16* q, const sk_bf16* k_cache, const sk_bf16* v_cache, const int32_t* pos,
                             const int64_t* tree, sk_bf16* out, int B, int HQ, int HKV, int D, int R, int cap,
                             int max_len, float scale, int nsplit, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (B < 0) return SK_ERR_SHAPE;
  if (B == 0) return SK_OK;
  AttnPlan p;
  int st = attn_plan(B, HQ, HKV, D, R, cap, max_len, nsplit, &p);
  if (st) return st;
  if (!q || !k_cache || !v_cache || !pos || !out) return SK_ERR_NULL;
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache)) return SK_ERR_ALIGN;
  if (p.need > 0 && (!ws || ws_bytes < p.need)) return SK_ERR_WORKSPACE;
  st = attn_device_ok();
  if (st) return st;
  sk::AttnArgs a;
  memset(&a, 0, sizeof(a));
  a.q = q;
  a.k = k_cache;
  a.v = v_cache;
  a.pos = pos;
  a.tree = tree;
  a.out = out;
  return attn_run(p, a, B, HQ, HKV, R, cap, scale, ws, false, stream);
}

int sk_decode_attention_rope_bf16(const sk_bf16* qkv, int64_t ld_qkv, const sk_bf16* q_norm_w,
                                  const sk_bf16* k_norm_w, const sk_bf16* cos, const sk_bf16* sin, int rope_rows,
                                  float eps, sk_bf16* k_cache, sk_bf16* v_cache, const int32_t* pos, sk_bf16* out,
                                  int B, int HQ, int HKV, int D, int R, int cap, int max_len, float scale,
                                  int nsplit, void* ws, size_t ws_bytes, hipStream_t stream) {
  return rope_attention(qkv, ld_qkv, q_norm_w, k_norm_w, cos, sin, rope_rows, eps, k_cache, v_cache, pos, nullptr,
                        nullptr, out, B, HQ, HKV, D, R, cap, max_len, scale, nsplit, ws, ws_bytes, stream);
}

int sk_decode_attention_rope_tree_bf16(const sk_bf16* qkv, int64_t ld_qkv, const sk_bf16* q_norm_w,
                                       const sk_bf16* k_norm_w, const sk_bf16* cos, const sk_bf16* sin,
                                       int rope_rows, float eps, sk_bf16* k_cache, sk_bf16* v_cache,
                                       const int32_t* pos, const int64_t* tree, const int32_t* depth, sk_bf16* out,
                                       int B, int HQ, int HKV, int D, int R, int cap, int max_len, float scale,
                                       int nsplit, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (B > 0 && (!tree || !depth)) return SK_ERR_NULL;
  return rope_attention(qkv, ld_qkv, q_norm_w, k_norm_w, cos, sin, rope_rows, eps, k_cache, v_cache, pos, tree,
                        depth, out, B, HQ, HKV, D, R, cap, max_len, scale, nsplit, ws, ws_bytes, stream);
}

}  // extern "C"
