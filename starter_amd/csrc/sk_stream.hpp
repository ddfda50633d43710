// sk_stream.hpp - the stream path: weight rows and activation rows go from
// memory straight into LDS (buffer_load_dwordx4 ... lds), without passing
// through registers, and are read back as MFMA fragments.
//
// One workgroup computes one tile of weight rows against up to 128 activation
// rows over one K slice.  Its W = KG x MG waves form KG K groups (group kg
// takes the units kg, kg + KG, ... of the slice, a unit being UC columns) of
// MG waves, each owning MT 16-row activation tiles and all NT 16-row slabs of
// weight rows.  Every K group has an LDS ring of D units.  While a wave
// multiplies unit i out of registers, unit i + 1 is read from LDS into the
// other fragment registers and unit i + D is requested into the slot that
// unit i left, one load between every few MFMAs (issued together, the loads
// of a unit held the MFMAs behind the address unit: gate_up at 128 rows 32.2
// against 26.5 us).  With MG = 1 a ring belongs to one wave and the loop has
// no barrier at all; with MG > 1 the waves of the workgroup meet once a unit.
//
// What bounds it.  A direct load needs no register and no LDS store
// instruction, so the bytes in flight per CU are bounded by LDS (up to
// 150 KB) and the wave's time is left to MFMAs.  Each load instruction
// covers RPI = 1024 / (2 UC) rows with 128 (UC = 64) or 256 (UC = 128)
// contiguous bytes each, in lane order, so the address unit sees whole
// cache lines; the order a fragment read needs comes from the LDS side: the
// 16-byte chunk c of row r lies at chunk position c ^ sw(r) of its row, so
// the 16 rows of one fragment read fall on 16 different bank groups.
// Loads in fragment order (16 rows x 64 B) measured 1.5-2x slower, loads of
// 64 B per row (UC = 32) 1.6x.  Splitting K over the waves (KG) instead of
// sharing every unit reads each staged byte once; past 64 rows the
// activation rows would not fit KG rings, so MG waves share one.
//
// Rows past the tile, past N or past M are outside their slab's buffer
// descriptor: the hardware returns without touching memory and what the slot
// then holds only reaches outputs that are never written.
//
// Epilogue: the K groups' fp32 tiles meet in LDS as [group][row][column]
// planes, are summed in group order, and every thread finishes four
// consecutive columns of a row, so outputs and split-K partials are written
// in 8- and 16-byte pieces (2-byte stores from the accumulator layout cost
// ~5 us at 128 rows).  Split K (S > 1): the workgroup's tile of partials goes
// to its own contiguous block of the workspace, the last workgroup of a tile
// sums the S blocks in split order.
#pragma once

#include "sk_kernels.hpp"

namespace sk {

typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kStreamLds = 160 * 1024;

// LDS bytes of one ring slot, units in flight per K group, and the workgroup's
// dynamic LDS (ring or epilogue planes, whichever is larger, and the flag).
constexpr int stream_slot(int MG, int MT, int NT, int UC) { return (MG * MT + NT) * 16 * 2 * UC; }
constexpr int stream_planes(int KG, int MG, int MT, int NT) { return KG * 16 * MG * MT * (16 * NT + 4) * 4; }
constexpr int stream_depth(int KG, int MG, int MT, int NT, int UC) {
  const int d = (kStreamLds - 64) / (KG * stream_slot(MG, MT, NT, UC));
  return d > 4 ? 4 : d;
}
constexpr int stream_lds(int KG, int MG, int MT, int NT, int UC) {
  const int ring = KG * stream_depth(KG, MG, MT, NT, UC) * stream_slot(MG, MT, NT, UC);
  const int planes = stream_planes(KG, MG, MT, NT);
  return (ring > planes ? ring : planes) + 64;
}
constexpr bool stream_fits(int KG, int MG, int MT, int NT, int UC) {
  return stream_depth(KG, MG, MT, NT, UC) >= 2 && stream_lds(KG, MG, MT, NT, UC) <= kStreamLds;
}
// Rows one load instruction covers, and the tile row at which the up half of
// a gate/up tile starts (its loads must not mix the two matrices).
constexpr int stream_rpi(int UC) { return 512 / UC; }
constexpr int stream_half(int tr, int UC) { return (tr + stream_rpi(UC) - 1) / stream_rpi(UC) * stream_rpi(UC); }
// Floats per row of a tile's block of split-K partials.
constexpr int stream_part_pitch(int tr) { return (tr + 3) / 4 * 4; }

// Buffer descriptor of `bytes` readable bytes from p (uniform).
__device__ __forceinline__ i32x4 buf_of(const void* p, int bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xFFFF);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000;
  return r;
}

// 16 bytes per lane from descriptor r at byte voff + soff into LDS at lds_off
// + 16 * lane.  No vector register is written, so the compiler need not track
// it; the caller waits on vmcnt.  m0 is overwritten and cannot be declared: it
// is a reserved register, which the compiler warns about in a clobber list and
// does not preserve.  It never allocates m0 either, so this is safe as long as a
// kernel has no instruction of the compiler's own that reads it (indexed
// register access, messages, LDS-direct builtins); tests/test_build_tiers.py
// checks the assembly.
template <bool STREAM>
__device__ __forceinline__ void load_lds16(uint32_t lds_off, int voff, i32x4 r, int soff) {
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 ::"s"(lds_off), "v"(voff), "s"(r), "s"(soff) : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"s"(lds_off), "v"(voff), "s"(r), "s"(soff) : "memory");
}

template <int N0>
__device__ __forceinline__ void wait_loads() {
  constexpr int N = N0 > 63 ? 63 : N0;   // the counter's width; fewer outstanding is only stricter
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// 16-byte device-coherent (sc1) accesses of the split-K partials.
__device__ __forceinline__ void store_agent16(__amdgpu_buffer_rsrc_t r, int off, f32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 16);
}
__device__ __forceinline__ f32x4 load_agent16(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16));
}

template <int KG, int MG, int MT, int NT, int UC, int EPI>
__device__ __forceinline__ void stream_body(const Args& p) {
  constexpr bool GATEUP = EpiTraits<EPI>::gateup;
  constexpr int BASE = EpiTraits<EPI>::base;
  constexpr bool RESID = EpiTraits<EPI>::resid;
  static_assert(BASE == EPI_STORE || BASE == EPI_SWIGLU || BASE == EPI_PART, "epilogues of the stream path");
  static_assert(!EpiTraits<EPI>::norm && !EpiTraits<EPI>::pre, "the activations are taken as they are");
  static_assert(UC == 64 || UC == 128, "whole cache lines per row and load");
  static_assert(stream_fits(KG, MG, MT, NT, UC), "ring and planes fit the LDS");
  constexpr int W = KG * MG;               // waves
  constexpr int MTT = MG * MT;             // activation tiles
  constexpr int D = stream_depth(KG, MG, MT, NT, UC);
  constexpr int KS = UC / 32;              // MFMA K steps per unit
  constexpr int RPI = stream_rpi(UC);      // rows per load instruction
  constexpr int LPR = 64 / RPI;            // lanes (16-byte chunks) per row
  constexpr int NB = 16 / RPI;             // loads per 16-row slab
  constexpr int SLOT = stream_slot(MG, MT, NT, UC);
  constexpr int WLD = (NT * NB + MG - 1) / MG;   // weight loads per wave and unit (the last may repeat one)
  constexpr int ALD = MT * NB;                   // activation loads per wave and unit: its own rows
  constexpr int NI = WLD + ALD;

  extern __shared__ __attribute__((aligned(1024))) float lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / MG, mg = wave % MG;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int M = p.M, N = p.N, TR = p.tr, S = p.S;
  const int slice = blockIdx.x % (unsigned)S;
  const int rb = blockIdx.x / (unsigned)S;
  const int units = p.K / UC;              // the host guarantees K % UC == 0
  const int s_lo = slice * p.slice_units;
  const int s_hi = min(s_lo + p.slice_units, units);
  const int nu = s_hi - s_lo;
  // units of this K group; waves that meet at barriers all run as many
  const int nit = MG == 1 ? (nu > kg ? (nu - 1 - kg) / KG + 1 : 0) : (nu + KG - 1) / KG;

  char* const ring = reinterpret_cast<char*>(lds) + kg * (D * SLOT);
  const uint32_t ring_off =
      (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)reinterpret_cast<char*>(lds)) +
      kg * (D * SLOT);

  // Lane l of a load covers chunk (l % LPR) ^ sw(row) of row l / LPR; sw
  // spreads the 16 rows of a slab over the 16 bank groups of a fragment read.
  auto sw = [](int r) { return UC == 64 ? (r & 15) >> 1 : (r & 15); };
  const int lrow = lane / LPR;
  const int n0 = rb * TR;                        // first output column of the tile
  const int cols = min(TR, N - n0);              // output columns that exist
  const int HU = GATEUP ? stream_half(TR, UC) : 0;   // tile row of the first up row
  // Byte offsets of this wave's loads from the operand's descriptor base (the
  // tile's first row, activation row 0); kNoRow lies past every descriptor.
  // The host guarantees that rows * stride fits.
  constexpr int kNoRow = 0x7FFF0000;
  int woff[WLD], wslot[WLD], aoff[ALD];
  bool wup[WLD];
#pragma unroll
  for (int j = 0; j < WLD; ++j) {
    const int blk = min(j * MG + mg, NT * NB - 1);
    const int t = RPI * blk + lrow;              // tile row of this lane
    wup[j] = GATEUP && RPI * blk >= HU;          // uniform: HU is a multiple of RPI
    const int r = wup[j] ? t - HU : t;
    woff[j] = r < cols ? r * (int)p.ldw * 2 + 16 * ((lane % LPR) ^ sw(t)) : kNoRow;
    wslot[j] = blk * 1024;
  }
#pragma unroll
  for (int j = 0; j < ALD; ++j) {
    const int m = 16 * MT * mg + RPI * j + lrow;
    aoff[j] = m < M ? m * (int)p.lda * 2 + 16 * ((lane % LPR) ^ sw(m)) : kNoRow;
  }
  const int wbytes = ((cols - 1) * (int)p.ldw + p.K) * 2;
  const i32x4 buf_w0 = buf_of(p.W0 + (int64_t)n0 * p.ldw, wbytes);
  const i32x4 buf_w1 = GATEUP ? buf_of(p.W1 + (int64_t)n0 * p.ldw, wbytes) : buf_w0;
  const i32x4 buf_a = buf_of(p.A, ((M - 1) * (int)p.lda + p.K) * 2);
  // Load j of the unit at byte column so, into the slot at LDS offset base.
  auto load1 = [&](int j, int so, uint32_t base) {
    if (j < WLD)
      load_lds16<true>(base + wslot[j], woff[j], wup[j] ? buf_w1 : buf_w0, so);
    else
      load_lds16<false>(base + (NT * NB + mg * ALD + j - WLD) * 1024, aoff[j - WLD], buf_a, so);
  };
  auto unit_of = [&](int i) { return s_lo + kg + KG * i; };   // the group's i-th unit
  // Fragments of K step u: chunk g4 + 4u of row r16 of every slab.
  int foff[KS];
#pragma unroll
  for (int u = 0; u < KS; ++u)
    foff[u] = (r16 / RPI) * 1024 + 16 * ((r16 % RPI) * LPR + ((g4 + 4 * u) ^ sw(r16)));

  f32x4 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Frags {
    bf16x8 w[KS][NT], a[KS][MT];
  };
  auto read = [&](int slot, Frags& f) {
    const char* const b = ring + slot * SLOT;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) f.w[u][nt] = *reinterpret_cast<const bf16x8*>(b + nt * NB * 1024 + foff[u]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        f.a[u][mt] = *reinterpret_cast<const bf16x8*>(b + (NT + mg * MT + mt) * NB * 1024 + foff[u]);
    }
  };
  // One unit's MFMAs, with the loads of unit i + D spread between them (FILL).
  constexpr int TOT = KS * MT * NT;
  auto multiply = [&](const Frags& f, auto fill, int so, uint32_t base) {
#pragma unroll
    for (int k = 0; k < TOT; ++k) {
      const int u = k / (MT * NT), mt = (k / NT) % MT, nt = k % NT;
      if constexpr (decltype(fill)::value) {
#pragma unroll
        for (int j = 0; j < NI; ++j)
          if (j * TOT / NI == k) {
            __builtin_amdgcn_sched_barrier(0);
            load1(j, so, base);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
      acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[u][nt], f.a[u][mt], acc[nt][mt], 0, 0, 0);
    }
  };
  auto meet = [&]() {
    if constexpr (MG > 1) {
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
  };
  // Unit i's fragments are in cur, its slot (sc) is free once every wave of
  // the group has them; unit i + 1 is in slot sn.  Loads were issued in unit
  // order, NI per unit, so at most (D - 2) * NI may be outstanding when unit
  // i + 1 must have landed (units i + 2 .. i + D - 1 follow it).
  auto step = [&](int i, const Frags& cur, Frags& next, int sc, int sn) {
    if (i + 1 < nit) {
      if (min(i + D - 1, nit - 1) - (i + 1) >= D - 2) wait_loads<(D - 2) * NI>();
      else wait_loads<0>();
      wait_lds();   // the reads of unit i's slot have returned
      meet();
      read(sn, next);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i + D < nit)
      multiply(cur, std::true_type{}, 2 * UC * unit_of(i + D), ring_off + sc * SLOT);
    else if (MG == 1 || unit_of(i) < s_hi)   // (a group's last unit may lie past the slice)
      multiply(cur, std::false_type{}, 0, 0u);
    __builtin_amdgcn_sched_barrier(0);
  };
  if (nit > 0) {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < nit) {
#pragma unroll
        for (int j = 0; j < NI; ++j) load1(j, 2 * UC * unit_of(d), ring_off + d * SLOT);
      }
    if (nit >= D) wait_loads<(D - 1) * NI>();
    else wait_loads<0>();
    meet();
    Frags f0, f1;
    read(0, f0);
    int sc = 0, sn = 1, i = 0;
    auto advance = [&]() {
      sc = sn;
      sn = sn + 1 == D ? 0 : sn + 1;
    };
    for (; i + 1 < nit; i += 2) {
      step(i, f0, f1, sc, sn);
      advance();
      step(i + 1, f1, f0, sc, sn);
      advance();
    }
    if (i < nit) step(i, f0, f1, sc, sn);
  }

  // The K groups' tiles to LDS planes [group][row][column] (rows padded by
  // four floats: the 16 rows of one store on different bank groups).
  constexpr int PITCH = 16 * NT + 4;
  float* const planes = lds;
  wait_loads<0>();
  __syncthreads();
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      *reinterpret_cast<f32x4*>(planes + (kg * 16 * MTT + 16 * (mg * MT + mt) + r16) * PITCH + 16 * nt + 4 * g4) =
          acc[nt][mt];
  __syncthreads();
  // Four columns c .. c+3 of row m, summed over the K groups in order.
  auto sum4 = [&](int m, int c) {
    f32x4 s = *reinterpret_cast<const f32x4*>(planes + m * PITCH + c);
#pragma unroll
    for (int k = 1; k < KG; ++k) s += *reinterpret_cast<const f32x4*>(planes + (k * 16 * MTT + m) * PITCH + c);
    return s;
  };
  // Finish columns n0 + c .. + 3 of row m: bf16 store, or the residual
  // hand-off (the tile's columns are whole 16-column groups then, and a
  // group's four threads are the four lanes of a quad).
  auto finish4 = [&](int m, int c, const uint16_t (&y)[4]) {
    if constexpr (RESID) {
      const bool ok = c < cols;   // N is a multiple of 4
      const int64_t at = (int64_t)m * p.ldr + n0 + c;
      float sq = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool oke = ok && c + e < cols;
        const float xo = oke ? round_bf(bf2f(p.R[at + e]) + bf2f(y[e])) : 0.f;
        if (oke) p.RO[at + e] = f2bf(xo);
        sq += xo * xo;
      }
      sq += __shfl_xor(sq, 1);
      sq += __shfl_xor(sq, 2);
      if ((c & 15) == 0 && ok) p.SQ[(int64_t)m * p.sq_ld + ((n0 + c) >> 4)] = sq;
    } else {
      uint16_t* const d = p.C + (int64_t)m * p.ldc + n0 + c;
      if (c + 4 <= cols && (reinterpret_cast<uintptr_t>(d) & 7) == 0) {
        *reinterpret_cast<u32x2*>(d) =
            u32x2{(uint32_t)y[0] | ((uint32_t)y[1] << 16), (uint32_t)y[2] | ((uint32_t)y[3] << 16)};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < cols) d[e] = y[e];
      }
    }
  };
  const int PP = stream_part_pitch(TR), Q = PP / 4;   // four-column pieces per row
  if constexpr (BASE != EPI_PART) {
    for (int idx = tid; idx < M * Q; idx += 64 * W) {
      const int m = idx / Q, c = 4 * (idx - m * Q);
      const f32x4 s = sum4(m, c);
      uint16_t y[4];
      if constexpr (GATEUP) {
        const f32x4 u = sum4(m, HU + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = swiglu_bf(s[e], u[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = f2bf(s[e]);
      }
      finish4(m, c, y);
    }
  } else {
    // Partials [tile][split][row][PP]; see splitk_fixup for the ordering rule
    // (device-coherent stores complete before the ticket is taken).
    const int64_t tile_floats = (int64_t)M * PP;
    float* const mine = p.part + ((int64_t)rb * S + slice) * tile_floats;
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(mine, 0, (int)(tile_floats * 4), 0x00020000);
    for (int idx = tid; idx < M * Q; idx += 64 * W) store_agent16(rs, 16 * idx, sum4(idx / Q, 4 * (idx % Q)));
    __builtin_amdgcn_s_waitcnt(0);
    int* const flag = reinterpret_cast<int*>(reinterpret_cast<char*>(lds) + stream_lds(KG, MG, MT, NT, UC) - 64);
    __syncthreads();
    if (tid == 0) *flag = take_ticket(&p.tickets[rb], (unsigned)S) ? 1 : 0;
    __syncthreads();
    if (!*flag) return;
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(p.part + (int64_t)rb * S * tile_floats, 0,
                                                      (int)(S * tile_floats * 4), 0x00020000);
    for (int idx = tid; idx < M * Q; idx += 64 * W) {
      const int m = idx / Q, c = 4 * (idx - m * Q);
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
      for (int k0 = 0; k0 < S; k0 += kFixupBatch) {
        f32x4 v[kFixupBatch];
#pragma unroll
        for (int k = 0; k < kFixupBatch; ++k)   // (past S: the last split again, not added)
          v[k] = load_agent16(ra, (int)(min(k0 + k, S - 1) * tile_floats * 4) + 16 * idx);
#pragma unroll
        for (int k = 0; k < kFixupBatch; ++k)
          if (k0 + k < S) s = k0 + k == 0 ? v[k] : s + v[k];
      }
      uint16_t y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = f2bf(s[e]);
      finish4(m, c, y);
    }
  }
}

// ---------------------------------------------------------------------------
// Persistent tiles: many more weight rows than one tile per CU holds (a
// vocabulary head).  One workgroup of eight waves per CU walks a contiguous
// range of the 16-row slabs in tiles of kTilesRows rows; the ring runs on across
// the tiles, so the next tile's first units are in flight while a tile is
// finished.  The waves are four row groups of MT activation tiles by two
// column groups of NT slabs, and share every unit of 64 columns.
//
// What bounds it.  Each tile reads the activation rows again (from L2), so the
// bytes through a CU per weight row fall with the tile's height: 160 rows is
// the most that leaves a ring four units deep beside 128 activation rows
// (36 KB a unit).  The slabs are dealt out evenly (they differ by one between
// workgroups) and start on 16 columns, so a row's four lanes store whole
// 32-byte pieces straight from the accumulators.
// Measured over 151936 x 2560 weights (two-operand wide path before): logits
// at 128 rows 203 -> 177 us, 96 rows 176 -> 169, 64 rows 157 -> 152, 40 rows
// 142 -> 137; fused argmax 128 rows 191 -> 151 (5.2 TB/s of weights), 96 rows
// 159 -> 145, 64 rows 145 -> 131.  The logits' 39 MB of stores cost the
// difference of the two.
// ---------------------------------------------------------------------------
constexpr int kTilesMG = 4, kTilesNG = 2, kTilesNT = 5, kTilesUC = 64;
constexpr int kTilesRows = 16 * kTilesNG * kTilesNT;
constexpr int tiles_slot(int MT) { return (kTilesMG * MT * 16 + kTilesRows) * 2 * kTilesUC; }
constexpr int tiles_lds(int MT) { return 4 * tiles_slot(MT); }

template <int MT, int EPI>
__device__ __forceinline__ void stream_tiles_body(const Args& p) {
  constexpr int BASE = EpiTraits<EPI>::base;
  static_assert(BASE == EPI_STORE || BASE == EPI_ARGMAX, "epilogues of the persistent tiles");
  static_assert(!EpiTraits<EPI>::norm && !EpiTraits<EPI>::pre && !EpiTraits<EPI>::resid, "plain operands");
  constexpr int MG = kTilesMG, NT = kTilesNT, UC = kTilesUC, W = kTilesMG * kTilesNG, D = 4;
  constexpr int KS = UC / 32;
  constexpr int WB = kTilesRows / 8, AB = MG * MT * 2;   // loads (8 rows each) of a unit's weights and activations
  constexpr int NI = (WB + AB + W - 1) / W;              // loads per wave and unit (the last may repeat one)
  constexpr int SLOT = tiles_slot(MT);
  static_assert(SLOT == (WB + AB) * 1024 && tiles_lds(MT) <= kStreamLds - 2048, "ring and argmax bests fit the LDS");

  extern __shared__ __attribute__((aligned(1024))) float lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mg = wave % MG, ng = wave / MG;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int M = p.M, N = p.N;
  const int units = p.K / UC;   // the host guarantees K % UC == 0
  // this workgroup's slabs [lo, hi) and tiles (the host launches no more
  // workgroups than slabs)
  const int slabs = (N + 15) >> 4, wg = blockIdx.x, nwg = gridDim.x;
  const int each = slabs / nwg, extra = slabs - each * nwg;
  const int lo = wg * each + min(wg, extra), hi = lo + each + (wg < extra ? 1 : 0);
  const int n_hi = min(16 * hi, N);
  const int ntiles = (hi - lo + kTilesRows / 16 - 1) / (kTilesRows / 16);
  const int total = ntiles * units;

  unsigned long long* const lds_best =
      reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(lds) + tiles_lds(MT));
  if constexpr (BASE == EPI_ARGMAX)
    for (int i = tid; i < M; i += 64 * W) lds_best[i] = 0ull;   // ordered by the first unit's barrier

  const char* const ring = reinterpret_cast<const char*>(lds);
  const uint32_t ring_off =
      (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)reinterpret_cast<char*>(lds));

  // Load q of a unit covers rows 8q .. 8q + 7 of the slot: the tile's weight
  // rows, then the activation rows; wave w issues loads w, w + W, ...  Rows
  // past a tile's last lie past the descriptor (row strides are at least K),
  // as does the offset that rows past M get.
  auto sw = [](int r) { return (r & 15) >> 1; };
  int off[NI], slot_at[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int q = min(j * W + wave, WB + AB - 1);
    const bool weight = q < WB;
    const int r = 8 * (weight ? q : q - WB) + (lane >> 3);
    const int at = 16 * ((lane & 7) ^ sw(r));
    off[j] = weight ? r * (int)p.ldw * 2 + at : r < M ? r * (int)p.lda * 2 + at : 0x7FFF0000;
    slot_at[j] = q * 1024;
  }
  const i32x4 buf_a = buf_of(p.A, ((M - 1) * (int)p.lda + p.K) * 2);
  i32x4 buf_w;
  auto weights_of = [&](int t) {
    const int n0 = 16 * lo + kTilesRows * t;
    const int cols = min(kTilesRows, n_hi - n0);
    buf_w = buf_of(p.W0 + (int64_t)n0 * p.ldw, ((cols - 1) * (int)p.ldw + p.K) * 2);
  };
  auto load1 = [&](int j, int so, uint32_t base) {
    if (j * W + W <= WB || (j * W < WB && j * W + wave < WB))   // (uniform)
      load_lds16<true>(base + slot_at[j], off[j], buf_w, so);
    else
      load_lds16<false>(base + slot_at[j], off[j], buf_a, so);
  };
  int foff[KS];   // chunk g4 + 4u of row r16 of every slab
#pragma unroll
  for (int u = 0; u < KS; ++u) foff[u] = (r16 >> 3) * 1024 + 16 * ((r16 & 7) * 8 + ((g4 + 4 * u) ^ sw(r16)));

  f32x4 acc[NT][MT];
  auto zero_acc = [&]() {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  zero_acc();
  struct Frags {
    bf16x8 w[KS][NT], a[KS][MT];
  };
  auto read = [&](int slot, Frags& f) {
    const char* const b = ring + slot * SLOT;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        f.w[u][nt] = *reinterpret_cast<const bf16x8*>(b + (ng * NT + nt) * 2048 + foff[u]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        f.a[u][mt] = *reinterpret_cast<const bf16x8*>(b + WB * 1024 + (mg * MT + mt) * 2048 + foff[u]);
    }
  };
  constexpr int TOT = KS * MT * NT;
  auto multiply = [&](const Frags& f, auto fill, int so, uint32_t base) {
#pragma unroll
    for (int k = 0; k < TOT; ++k) {
      const int u = k / (MT * NT), mt = (k / NT) % MT, nt = k % NT;
      if constexpr (decltype(fill)::value) {
#pragma unroll
        for (int j = 0; j < NI; ++j)
          if (j * TOT / NI == k) {
            __builtin_amdgcn_sched_barrier(0);
            load1(j, so, base);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
      acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[u][nt], f.a[u][mt], acc[nt][mt], 0, 0, 0);
    }
  };
  // Lane l holds columns 4 * (l / 16) .. + 3 of each slab for row l % 16.
  // (Counting a tile's stores in the waits of the next units instead of
  // draining them changed nothing.)
  const bool vec = ((p.ldc & 3) == 0) && (reinterpret_cast<uintptr_t>(p.C) & 7) == 0;
  auto finish = [&](int t) {
    const int n0 = 16 * lo + kTilesRows * t + 16 * NT * ng + 4 * g4;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = 16 * (mg * MT + mt) + r16;
      if constexpr (BASE == EPI_ARGMAX) {
        uint32_t bo = 0u;
        int bn = 0;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int n = n0 + 16 * nt + e;
            const uint32_t o = argmax_ord(f2bf(acc[nt][mt][e]));
            if (n < n_hi && o > bo) {   // increasing columns: ties keep the lowest
              bo = o;
              bn = n;
            }
          }
        unsigned long long key = bo ? argmax_pack(bo, bn) : 0ull;
#pragma unroll
        for (int x = 16; x <= 32; x <<= 1) {
          const unsigned long long o = ((unsigned long long)(uint32_t)__shfl_xor((int)(key >> 32), x) << 32) |
                                       (uint32_t)__shfl_xor((int)(key & 0xFFFFFFFFu), x);
          key = o > key ? o : key;
        }
        if (g4 == 0 && m < M && key) atomicMax(&lds_best[m], key);
      } else if (m < M) {
        uint16_t* const row = p.C + (int64_t)m * p.ldc;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int n = n0 + 16 * nt;
          uint16_t y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = f2bf(acc[nt][mt][e]);
          if (vec && n + 4 <= n_hi) {
            *reinterpret_cast<u32x2*>(row + n) =
                u32x2{(uint32_t)y[0] | ((uint32_t)y[1] << 16), (uint32_t)y[2] | ((uint32_t)y[3] << 16)};
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < n_hi) row[n + e] = y[e];
          }
        }
      }
    }
  };
  // The loads run D units ahead: unit lu of tile lt is the next to request, the
  // ln-th of the tile.  Where the row stride is a multiple of 4 KB, every row of
  // a unit lies on the same one of an XCD's 16 L2 channels (256 bytes each), and
  // workgroups in step would load one channel at a time: each then starts its
  // tiles at a unit of its own (65536 x 2048, 64 rows: logits 64.8 -> 51.5 us,
  // argmax 63.4 -> 51.2; 100352 x 4096, 128 rows: 342 -> 310; 40960 x 8192: 245 ->
  // 208.  Other strides gain nothing: 151936 x 2560 177 either way).
  const int first =
      (p.ldw & 2047) == 0 ? (int)((unsigned)(wg >> 3) * (unsigned)units / (unsigned)((nwg + 7) >> 3)) : 0;
  int lt = 0, lu = first, ln = 0;
  auto advance_loads = [&]() {
    if (++lu == units) lu = 0;
    if (++ln == units) {
      ln = 0;
      if (++lt < ntiles) weights_of(lt);
    }
  };
  int ct = 0, cu = 0;   // the unit being multiplied
  // As in stream_body: unit i's fragments are in cur, its slot (sc) is free
  // past the barrier; unit i + 1 is in slot sn once every wave's loads of it
  // have landed.  (The stores of a finished tile count as outstanding too:
  // they only make the wait stricter.)
  auto step = [&](int i, const Frags& cur, Frags& next, int sc, int sn) {
    if (i + 1 < total) {
      if (i + D <= total) wait_loads<(D - 2) * NI>();
      else wait_loads<0>();
      wait_lds();
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      read(sn, next);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (i + D < total) {
      multiply(cur, std::true_type{}, 2 * UC * lu, ring_off + sc * SLOT);
      advance_loads();
    } else {
      multiply(cur, std::false_type{}, 0, 0u);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (++cu == units) {
      finish(ct);
      __builtin_amdgcn_sched_barrier(0);
      zero_acc();
      cu = 0;
      ++ct;
    }
  };
  weights_of(0);
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < total) {
#pragma unroll
      for (int j = 0; j < NI; ++j) load1(j, 2 * UC * lu, ring_off + d * SLOT);
      advance_loads();
    }
  if (total >= D) wait_loads<(D - 1) * NI>();
  else wait_loads<0>();
  wait_lds();   // (the argmax bests)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f0, f1;
  read(0, f0);
  int i = 0, sc = 0;
  for (; i + 1 < total; i += 2) {
    step(i, f0, f1, sc, (sc + 1) & (D - 1));
    step(i + 1, f1, f0, (sc + 1) & (D - 1), (sc + 2) & (D - 1));
    sc = (sc + 2) & (D - 1);
  }
  if (i < total) step(i, f0, f1, sc, (sc + 1) & (D - 1));

  if constexpr (BASE == EPI_ARGMAX) {
    __syncthreads();
    argmax_fixup(p, lds_best, reinterpret_cast<int*>(lds_best + M));
  }
}

}  // namespace sk
