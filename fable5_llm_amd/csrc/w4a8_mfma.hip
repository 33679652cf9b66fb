// Batched W4A8 (several tokens): int8 MFMA on gfx950 with the per-group
// scale applied after accumulation.  Per token the result is bit-identical
// to ref/w4a8_ref.py:254-289 matvec_y32: every group sum is exact in int32
// (|16 * sum w*x| <= 2^21) and the scale products are summed in int64.
//
// v_mfma_i32_16x16x64_i8: A = 16 tokens x 64 k, B = 64 k x 16 weight rows,
// D = 16 x 16 int32.  Lane l feeds token / row (l % 16) and k-quarter l / 16
// of A and B alike, so A and B share one lane->k mapping and the dot product
// does not depend on the order in which the hardware walks k.  D element
// (4 * (l / 16) + r, l % 16) lands in lane l, register r: a lane holds four
// tokens of ONE weight row, so a group's scale is one value per lane, read
// from that row's own bytes of the scale block.  It enters through
// v_mad_i64_i32, which runs at the rate of a double-precision FMA (measured:
// 2.4 against 2.2 ns per instruction and SIMD) and needs no conversion.
//
// Four wavefronts per workgroup, two workgroups per CU (or one of eight
// wavefronts).  What bounds it is the
// weight stream, and next to it the activations: 16 tokens of a group are
// 2 KiB for every KiB of weights they meet.  Loaded straight into the MFMA's
// layout they touch 16 cache lines per 16 lanes, and the address unit takes
// one line a cycle; so they are copied into LDS in whole lines (8 tokens x 128
// bytes a copy), with the 16-byte pieces of token t stored at piece ^ (t % 8),
// which keeps the LDS reads free of bank conflicts.  Two ways to split a
// unit (up to TM tiles per wavefront, all of K) over the wavefronts:
//
//  * shared (KS = 1): every wavefront takes its own TM tiles and all of K, and
//    all four or eight share one copy of the activations (one workgroup
//    barrier per four groups).  Nothing is reduced; best where tiles are plenty.
//  * split (KS = 4): the wavefronts take the same tile and every fourth quad
//    of groups, each with its own copies (no barrier), and meet in an LDS
//    table at the end of the unit.
//
// A workgroup runs its units one after another; the weight ring (4 groups per
// wavefront) and the copies run on across them, so the stream does not drain
// between tiles or matrices.  No wait depends on another workgroup.
//
// Measured in a graph of launches, us each, weights cold in all of them, with
// one workgroup per CU, loader wavefronts and 8 slots -> now:
//   12288 + 12288 rows, K 4096:  B = 8: 18.9 -> 12.9, B = 64: 100 -> 19.4
//   4096 rows, K 12288:          B = 8: 12.9 -> 9.4, B = 64: 52.5 -> 18.5
//   60,000 rows, K 4096:         B = 8: 32.7 -> 25.4, B = 32: 51.4 -> 27.6, B = 64: 240 -> 35.8
//   a pass of 96 FFN matrices:   B = 8: 525 -> 400, B = 32: 695 -> 450, B = 64: 4052 -> 539
//   ... three passes' plans in turn:    538 -> 415,         708 -> 498,         4052 -> 568
// Repeated, a pass finds part of its y32 (117 MB at B = 32) still in the
// last-level cache; in turn, it does not.  Likewise three sets of 12288 +
// 12288 rows in turn (156 MB) partly stay there: B = 8 11.9.  The pass's
// weights alone take 360 us at the read ceiling.
#include <algorithm>

#include "w4a8_device.h"

namespace w4a8 {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kMBufDword3 = 0x00020000;    // raw buffer, 32-bit data format
constexpr int kMAuxNt = 2;                 // buffer-load cache policy: non-temporal
constexpr int kMPast = 0x40000000;         // a buffer offset past every range
constexpr int kLdsBytes = 160 * 1024;
constexpr int kMWaves = 4;
constexpr int kMWide = 8;                  // wavefronts of a wide shared workgroup

// A unit: up to TM * TS consecutive row tiles of one matrix, over all of K.
struct MmUnit {
  const uint8_t *W;     // first tile
  const int8_t *x8;     // [B][K]
  int32_t *y32;         // [B][nrows]
  int32_t tile_bytes, ntiles;   // tiles from W on
  int32_t nrows, row0;  // row0: the first tile's first row
  int32_t NG, K, sh;
  int32_t pad[3];
};
static_assert(sizeof(MmUnit) == 64, "one scalar load of 16 words");

struct MmJob {
  MmUnit u;             // the job's first unit
  int32_t unit0;        // its number
  int32_t pad[3];
};

struct MmParams {
  MmJob job[kMmJobs];   // the jobs, when they travel in the parameters ...
  const MmUnit *tab;    // ... or a device table of the units (a matmul plan)
  int32_t njobs, units;
  int32_t B;
  int32_t *err;
};

__device__ __forceinline__ int cvt_lo16(uint32_t w) {
  // offset-form low nibbles u = w + 8 -> bytes 16*w (exact int8)
  return (int)(((w << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
}
__device__ __forceinline__ int cvt_hi16(uint32_t w) {
  return (int)(w & 0xF0F0F0F0u);   // two's-complement high nibbles -> 16*w
}

typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t mm_rsrc(const void *p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, bytes, kMBufDword3);
}

// A group's activations, both 16-byte halves of a lane's 32 k for every tile
// of 16 tokens (2 KiB apart).  In assembly, with the wait in the same block:
// the compiler would make an LDS read wait for the newest LDS copy in flight.
template <int CT>
__device__ __forceinline__ void mm_read(v4i (&x)[CT][2], uint32_t o0, uint32_t o1) {
  if constexpr (CT == 1) {
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]) : "v"(o0), "v"(o1) : "memory");
  } else if constexpr (CT == 2) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\t"
                 "ds_read_b128 %2, %4 offset:2048\n\tds_read_b128 %3, %5 offset:2048\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1])
                 : "v"(o0), "v"(o1) : "memory");
  } else if constexpr (CT == 3) {
    asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\t"
                 "ds_read_b128 %2, %6 offset:2048\n\tds_read_b128 %3, %7 offset:2048\n\t"
                 "ds_read_b128 %4, %6 offset:4096\n\tds_read_b128 %5, %7 offset:4096\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]),
                   "=&v"(x[2][0]), "=&v"(x[2][1])
                 : "v"(o0), "v"(o1) : "memory");
  } else {
    asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\t"
                 "ds_read_b128 %2, %8 offset:2048\n\tds_read_b128 %3, %9 offset:2048\n\t"
                 "ds_read_b128 %4, %8 offset:4096\n\tds_read_b128 %5, %9 offset:4096\n\t"
                 "ds_read_b128 %6, %8 offset:6144\n\tds_read_b128 %7, %9 offset:6144\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]),
                   "=&v"(x[2][0]), "=&v"(x[2][1]), "=&v"(x[3][0]), "=&v"(x[3][1])
                 : "v"(o0), "v"(o1) : "memory");
  }
}

__device__ __forceinline__ int32_t mm_opaque(int32_t v) {
  asm("" : "+v"(v));
  return v;
}
__device__ __forceinline__ void mm_lds_add(int64_t *p, int64_t v) {
  asm volatile("ds_add_u64 %0, %1" :: "v"(lds_off(p)), "v"(v) : "memory");
}
// the entry's value, the entry cleared
__device__ __forceinline__ int64_t mm_lds_take(int64_t *p) {
  int64_t v;
  asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)\n\tds_write_b64 %1, %2"
               : "=&v"(v) : "v"(lds_off(p)), "v"((int64_t)0) : "memory");
  return v;
}

// s_waitcnt vmcnt(N) alone (gfx9 encoding: vmcnt in bits 3:0 and 15:14)
template <int N>
__device__ __forceinline__ void mm_wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

struct MmSrc {
  const uint8_t *w;
  const int8_t *x;
  int32_t tile_bytes, ntiles, K, NG;
};
// tile j's buffer: its range ends with the tile's data, and is empty (loads
// return zeros without a memory access) where there is no such tile
__device__ __forceinline__ __amdgpu_buffer_rsrc_t mm_tile_rsrc(const MmSrc &S, int j) {
  return mm_rsrc(S.w + (int64_t)j * S.tile_bytes, j < S.ntiles ? S.tile_bytes : 0);
}

// A wavefront's step (the groups of one copy) and its LDS buffers: 4 groups
// and two buffers where a buffer stays within 8 KiB per wavefront (32 KiB
// shared), else one group and four buffers -- a step's copies are then
// issued three groups ahead (17..32 tokens, 4096 rows, K 12288: 14.9 us with
// two buffers, 13.8 with four).
constexpr int mm_q(int CT, int KS) { return KS == 1 || CT == 1 ? 4 : 1; }
constexpr int mm_nbuf(int CT, int KS) { return KS == 1 || CT == 1 ? 2 : 4; }
constexpr int mm_octets(int CT, bool half8) { return half8 ? 1 : 2 * CT; }   // of tokens
constexpr size_t mm_x_bytes(int CT, int KS, bool half8) {
  return (size_t)KS * mm_nbuf(CT, KS) * mm_q(CT, KS) * mm_octets(CT, half8) * 1024;
}

// half8: at most 8 tokens (one octet is copied, and read by both halves of
// the MFMA's 16 rows)
template <int NW, int TM, int CT, int KS, bool half8, bool plan>
__global__ __launch_bounds__(64 * NW, 2) void matmul_kernel(MmParams P) {
  extern __shared__ __align__(1024) uint8_t smem[];
  constexpr int TS = NW / KS;
  constexpr int Q = mm_q(CT, KS), NBUF = mm_nbuf(CT, KS);
  constexpr int NO = mm_octets(CT, half8);
  constexpr int kGrp = NO * 1024;                   // LDS bytes of a group's activations
  constexpr int kBuf = Q * kGrp;                    // ... of a step
  constexpr int ND = TS == 1 ? Q * NO : Q * NO / NW;   // copies per wavefront and step
  constexpr int D = 4;                           // groups in flight
  constexpr int kTurn = KS * D;                     // groups of a turn of the ring, all slices
  constexpr int kXBytes = (int)mm_x_bytes(CT, KS, half8);
  // the scales' 256 bytes of a block are read twice, half a block apart: kept
  // in the cache, except beyond 48 tokens, where the activations need it more
  // (96 FFN matrices: B = 32 493 us non-temporal, 477 not; B = 64 586 and 598)
  constexpr int kMAuxM = CT == 4 ? kMAuxNt : 0;
  constexpr int NR = TM * CT * 4 * 64;              // a wavefront's sums
  static_assert(KS == 1 || KS == NW, "the copies are shared by all wavefronts or by none");
  static_assert(ND * 1024 * (TS == 1 ? 1 : NW) == kBuf, "whole copies per wavefront");
  static_assert(NBUF - 1 <= D / Q || NBUF == 2, "a step's copies reach one turn ahead at most");
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ks = TS == 1 ? wave : 0, ts = TS == 1 ? 0 : wave;
  const int B = P.B, G = gridDim.x, r = blockIdx.x;
  typedef const __attribute__((address_space(4))) MmUnit CUnit;

  // unit number i of this workgroup (an empty one past its last)
  auto unit_at = [&](int i) {
    const int64_t pos = (int64_t)i * G + r;
    MmUnit U{};
    if constexpr (plan) {
      if (pos < P.units) U = *(const MmUnit *)((CUnit *)P.tab + pos);
    } else if (pos < P.units) {
      const int u = (int)pos;
      int jb = 0;
#pragma unroll
      for (int k = 1; k < kMmJobs; ++k) jb += (k < P.njobs && u >= P.job[k].unit0) ? 1 : 0;
      jb = __builtin_amdgcn_readfirstlane(jb);
      U = P.job[jb].u;
      const int t = (u - P.job[jb].unit0) * (TM * TS);
      U.W += (int64_t)t * U.tile_bytes;
      U.ntiles -= t;
      U.row0 = t * kTileRows;
    }
    return U;
  };
  // where a turn's loads come from
  auto src_of = [&](const MmUnit &U) {
    return MmSrc{U.W + (int64_t)(ts * TM) * U.tile_bytes, U.x8, U.tile_bytes, U.ntiles - ts * TM,
                 U.K, U.NG};
  };

  // a step's copies: 8 tokens of one group at a time (1 KiB): lane l brings
  // piece (l % 8) ^ (token % 8) of token l / 8
  const int dtok = lane >> 3, dpiece = (lane & 7) ^ (dtok & 7);
  uint8_t *const xmine = smem + (TS == 1 ? wave * (NBUF * kBuf) : 0);
  // the copies of a step whose first group (over all slices) is gs
  auto copy_x = [&](const MmSrc &S, int gs, int buf) {
    const __amdgpu_buffer_rsrc_t rx = mm_rsrc(S.x, B * S.K);
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const int n = TS == 1 ? d : wave * ND + d;    // (group, token octet)
      const int g = n / NO, o = n % NO;
      const int gg = gs + ks * D + g;
      const int off = (8 * o + dtok) * S.K + gg * kGroup + 16 * dpiece;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rx, (lds_void_t *)(xmine + buf * kBuf + n * 1024), 16, gg < S.NG ? off : kMPast, 0, 0, 0);
    }
  };
  const int wlane = kScaleChunk + (c * 4 + q) * 16, slane = c * 16;
  u4 w[TM][D];
  // the turn's scales and the next turn's, a lane's four groups in one load
  // (a load per group and tile, 2 bytes a lane: B = 8 432 us, 423 so)
  u2 m[TM], mn[TM];
  auto load_w = [&](const MmSrc &S, int g, const int slot) {
    const int off = (g >> 3) * kBlockBytes + (g & 7) * kGroupChunk + wlane;
#pragma unroll
    for (int j = 0; j < TM; ++j)
      w[j][slot] = __builtin_amdgcn_raw_buffer_load_b128(mm_tile_rsrc(S, j), off, 0, kMAuxNt);
  };
  auto load_m = [&](const MmSrc &S, int g) {
    const int off = (g >> 3) * kBlockBytes + (g & 7) * 2 + slane;   // g: a multiple of 4
#pragma unroll
    for (int j = 0; j < TM; ++j)
      mn[j] = __builtin_amdgcn_raw_buffer_load_b64(mm_tile_rsrc(S, j), off, 0, kMAuxM);
  };

  int64_t p[TM][CT][4];
#pragma unroll
  for (int j = 0; j < TM; ++j)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int e = 0; e < 4; ++e) p[j][ct][e] = 0;

  MmUnit U = unit_at(0), V = unit_at(1);
  MmSrc S = src_of(U);
  int64_t *const red = (int64_t *)(smem + kXBytes);   // KS > 1: two tables of NR sums
  if constexpr (KS > 1) {
    for (int i = tid; i < 2 * NR; i += NW * 64) red[i] = 0;
    wait_lds();
    __builtin_amdgcn_s_barrier();
  }
  load_m(S, ks * D);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < NBUF - 1; ++s) copy_x(S, s / (D / Q) * kTurn + s % (D / Q) * Q, s);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < D; ++i) {
    load_w(S, ks * D + i, i);
  }
  // the first step's activations: everything issued after them may be in flight
  mm_wait_vm<(NBUF - 2) * ND + TM * D>();
  if constexpr (TS > 1) __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);

  const int crow = half8 ? c & 7 : c;
  const uint32_t xbase = lds_off(xmine) + crow * 128;
  const uint32_t x0 = xbase + (((2 * q) ^ (c & 7)) * 16), x1 = xbase + (((2 * q + 1) ^ (c & 7)) * 16);
  int buf = 0;    // the step's buffer
  int tb = 0;     // KS > 1: the unit's table
  bool ovf = false;
  for (int i_unit = 0; U.ntiles > 0; ++i_unit) {
    for (int g0 = 0; g0 < U.NG; g0 += kTurn) {
      const bool last = g0 + kTurn >= U.NG;
      const MmSrc T = last ? src_of(V) : S;      // the next turn's loads
      const int gt = last ? 0 : g0 + kTurn;
#pragma unroll
      for (int j = 0; j < TM; ++j) m[j] = mn[j];
      load_m(T, gt + ks * D);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < D; ++i) {
        if (i % Q == 0) {
          // a step begins (its activations have landed): refill the buffer
          // that the step before it has left
          const int ahead = i / Q + NBUF - 1;
          const int nb = buf + NBUF - 1 >= NBUF ? buf - 1 : buf + NBUF - 1;
          if (ahead < D / Q) copy_x(S, g0 + ahead * Q, nb);
          else copy_x(T, gt + (ahead - D / Q) * Q, nb);
          __builtin_amdgcn_sched_barrier(0);
        }
        v4i x[CT][2];
        const uint32_t xo = buf * kBuf + (i % Q) * kGrp;
        mm_read<CT>(x, x0 + xo, x1 + xo);
        __builtin_amdgcn_sched_barrier(0);
        v4i acc[TM][CT];
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          const u4 wp = w[j][i];
          const v4i a0 = {cvt_lo16(wp.x), cvt_hi16(wp.x), cvt_lo16(wp.y), cvt_hi16(wp.y)};
          const v4i a1 = {cvt_lo16(wp.z), cvt_hi16(wp.z), cvt_lo16(wp.w), cvt_hi16(wp.w)};
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
            acc[j][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[ct][0], a0, v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
            acc[j][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[ct][1], a1, acc[j][ct], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_w(T, gt + ks * D + i, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          // opaque, so that the compiler forms 32 x 32 + 64 signed multiply-adds
          const int32_t mv = mm_opaque((int32_t)(i & 1 ? m[j][i / 2] >> 16 : m[j][i / 2] & 0xFFFFu));
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              p[j][ct][e] += (int64_t)mv * (int64_t)acc[j][ct][e];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (i % Q == Q - 1) {
          // the next step's activations: issued NBUF - 1 steps ago
          mm_wait_vm<(NBUF - 2) * (ND + TM * Q) + TM * Q>();
          if constexpr (TS > 1) __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
          buf = buf + 1 == NBUF ? 0 : buf + 1;
        }
      }
      S = T;
    }
    // the unit's sums: rounded, checked and stored
    const int sh = U.sh, nrows = U.nrows;
    const int64_t half = sh > 0 ? (int64_t)1 << (sh - 1) : 0;
    int32_t *const y32 = U.y32;
    auto put = [&](int64_t t, int row, int tok) {
      const int64_t v = t >> 4;   // t is 16 * the row's sum exactly
      const int64_t a = ((v < 0 ? -v : v) + half) >> sh;
      const int64_t y = v < 0 ? -a : a;
      if (row < nrows && tok < B) {
        ovf = ovf || y > 2147483647LL || y < -2147483647LL;
        y32[(int64_t)tok * nrows + row] = (int32_t)y;
      }
    };
    if constexpr (KS == 1) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < TM; ++j) {
            put(p[j][ct][e], U.row0 + (ts * TM + j) * kTileRows + c, 16 * ct + 4 * q + e);
            p[j][ct][e] = 0;
          }
    } else {
      // the slices meet in one of two LDS tables (alternating by unit, so
      // that one barrier per unit keeps its readers and the next unit's
      // adders apart); each wavefront stores, and clears, its share
      int64_t *const tab = red + tb * NR;
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            mm_lds_add(tab + ((j * CT + ct) * 4 + e) * 64 + lane, p[j][ct][e]);
            p[j][ct][e] = 0;
          }
      wait_lds();
      __builtin_amdgcn_s_barrier();
      static_assert(NR % (NW * 64) == 0, "");
#pragma unroll
      for (int k = 0; k < NR / (NW * 64); ++k) {
        const int n = k * NW + wave;            // (j, ct, e)
        int64_t *const s = tab + n * 64 + lane;
        const int64_t t = mm_lds_take(s);
        const int j = n / (CT * 4), ct = n / 4 % CT, e = n % 4;
        put(t, U.row0 + j * kTileRows + c, 16 * ct + 4 * q + e);
      }
      tb ^= 1;
    }
    U = V;
    V = unit_at(i_unit + 2);
  }
  // copies issued past the last unit (empty ranges) have landed before the
  // LDS is given back
  mm_wait_vm<0>();
  if (ovf) atomicOr(P.err, 1);
}

// How a launch runs for B tokens on ncu CUs.
struct MmShape {
  int CT, TM, KS, NW, units, wgs;
};

// `tiles` row tiles of `groups` groups in all, the longest of NG, which make
// `quads` units of four tiles and `wide` units of sixteen.
static MmShape mm_shape(int64_t tiles, int64_t groups, int64_t quads, int64_t wide, int NG,
                        int32_t B, int ncu) {
  MmShape s{};
  s.CT = (B + 15) / 16;
  // Shared where its units (4 tiles a workgroup) still fill the CUs (K 4096,
  // B = 8: 768 tiles, 3 per CU, 9.8 us shared, 9.3 split; 832 9.8 and 10.0;
  // 512 9.2 and 7.1).  Beyond 32 tokens the shared copies are worth more (K
  // 4096, B = 48: 384 tiles 12.7 and 13.3, 512 12.8 and 14.0), and up to K =
  // 2048 the split leaves wavefronts without groups (B = 24: 640 tiles, K 1024
  // 6.2 and 7.7, K 2048 7.9 and 8.2; 384 tiles, K 1024 5.7 and 6.5, but K 2048,
  // B = 8 6.0 and 5.1).  Tiles of 48 groups and more (K = 6144): few tokens
  // stay split for longer, their copies being small beside the weights (K
  // 12288: 768 tiles, B = 8 24.5 and 18.7, B = 16 24.8 and 23.5; 960 tiles, B
  // = 8 23.8 and 23.3, B = 16 23.9 and 29.0), 17 to 32 go shared once the
  // split's two workgroups per CU are full (K 12288, B = 24: 640 tiles 25.6
  // and 26.8, 512 23.5 and 20.5).
  int64_t need = B > 32 || NG <= 16 ? ncu * 3 / 2 : ncu * 3;
  if (groups >= 48 * tiles) {
    if (B <= 8) need = ncu * 4;
    else if (B <= 16) need = ncu * 3 + 1;
    else if (B <= 32) need = ncu * 2 + 1;
  }
  s.KS = tiles >= need ? 1 : kMWaves;
  s.TM = 1;
  s.NW = kMWaves;
  // Beyond one unit of four tiles per CU eight wavefronts share the copies,
  // one tile each, which keeps a workgroup on every CU busy where four
  // would leave most CUs with one (1280 tiles, K 4096, B = 8 / 64: 12.4 / 19.0
  // on eight, 12.6 / 21.5 on four, K 12288, B = 64 45.2 and 53.8; up to one
  // per CU four are better: 1024 tiles, K 4096 12.0 / 18.0 and 10.7 / 15.8, K
  // 12288, B = 8 28.7 and 23.7).
  if (s.KS == 1 && tiles >= ncu * 4 && quads > ncu) {
    s.NW = kMWide;
    // Beyond 8 tiles per CU two tiles a wavefront share its reads of the
    // activations (K 4096: 2049 tiles, B = 8 / 64 16.8 / 28.2 with two on four
    // wavefronts, 18.9 / 31.4 with one on eight; 1800 tiles, B = 64 22.6 and
    // 20.8), on eight wavefronts (3750 tiles: B = 64 36.7 on four, 33.5; 96
    // FFN matrices: B = 32 470 and 453, B = 64 586 and 536), except up to 8
    // tokens (24.2 and 24.6) and where more than a tenth of the places for
    // tiles stays empty in the rounds (4800 tiles, B = 32 36.7 and 41.2; 10560
    // tiles of a plan of K 2048 and 6016, B = 24 51.4 and 55.6; but 2300 to
    // 3000 tiles, and 10560 of K 4096, run 5 to 9 % faster on eight).
    if (tiles > (int64_t)ncu * kMWide) {
      s.TM = 2;
      const int64_t places = (wide + ncu - 1) / ncu * ncu * (2 * kMWide);
      if (B <= 8 || tiles * 10 < places * 9) s.NW = kMWaves;
    }
  }
  return s;
}
static int mm_tiles_per_unit(const MmShape &s) { return s.TM * (s.NW / s.KS); }

// Workgroups: all units at once up to two workgroups per CU.  Eight
// wavefronts are one workgroup per CU, and so is a long pass of up to 32
// tokens: fewer streams read faster (96 FFN matrices, B = 8: 401 us against
// 410; beyond 32 tokens the second workgroup's overlap is worth more).
static int mm_wgs(int units, int NW, int32_t B, int ncu) {
  const int most = NW > kMWaves || (units >= 8 * ncu && B <= 32) ? ncu : 2 * ncu;
  return units < most ? units : most;
}

static int mm_ncu() {
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess)
    (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  return ncu;
}

static MmShape mm_setup(const MmJobSpec *jobs, int n, int32_t B, MmJob *out) {
  int64_t tiles = 0, groups = 0, quads = 0, wide = 0;
  int NG = 0;
  for (int j = 0; j < n; ++j) {
    const int64_t t = (jobs[j].nrows + kTileRows - 1) / kTileRows;
    tiles += t;
    groups += t * jobs[j].L.NG;
    quads += (t + kMWaves - 1) / kMWaves;
    wide += (t + 2 * kMWide - 1) / (2 * kMWide);
    NG = jobs[j].L.NG > NG ? jobs[j].L.NG : NG;
  }
  const int ncu = mm_ncu();
  MmShape s = mm_shape(tiles, groups, quads, wide, NG, B, ncu);
  const int per = mm_tiles_per_unit(s);
  int unit = 0;
  for (int j = 0; j < n; ++j) {
    MmJob &J = out[j];
    const MmJobSpec &q = jobs[j];
    J = MmJob{};
    J.u.W = q.w;
    J.u.x8 = q.x8;
    J.u.y32 = q.y32;
    J.u.tile_bytes = (int32_t)q.L.tile_bytes;
    J.u.nrows = q.nrows;
    J.u.ntiles = (q.nrows + kTileRows - 1) / kTileRows;
    J.u.NG = q.L.NG;
    J.u.sh = q.sh;
    J.u.K = q.L.K;
    J.unit0 = unit;
    unit += (J.u.ntiles + per - 1) / per;
  }
  s.units = unit;
  s.wgs = mm_wgs(unit, s.NW, B, ncu);
  return s;
}

template <int NW, int TM, int CT, int KS, bool half8, bool plan>
static hipError_t mm_launch1(const MmParams &P, int wgs, hipStream_t s) {
  auto *const k = &matmul_kernel<NW, TM, CT, KS, half8, plan>;
  // dynamic LDS beyond the default limit: allowed once per process
  static const hipError_t attr = hipFuncSetAttribute(
      (const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
  if (attr != hipSuccess) return attr;
  constexpr size_t lds = mm_x_bytes(CT, KS, half8) +
                         (KS > 1 ? (size_t)2 * TM * CT * 4 * 64 * sizeof(int64_t) : 0);
  static_assert(lds <= kLdsBytes, "LDS of one workgroup");
  hipLaunchKernelGGL(k, dim3(wgs), dim3(64 * NW), lds, s, P);
  return hipGetLastError();
}

template <int CT, bool plan>
static hipError_t mm_launch2(const MmParams &P, const MmShape &c, hipStream_t s) {
  if constexpr (CT == 1) {
    // the split's private copies are halved for up to 8 tokens
    if (c.KS > 1 && P.B <= 8) return mm_launch1<kMWaves, 1, CT, kMWaves, true, plan>(P, c.wgs, s);
  }
  if (c.KS > 1) return mm_launch1<kMWaves, 1, CT, kMWaves, false, plan>(P, c.wgs, s);
  if (c.NW > kMWaves)
    return c.TM == 1 ? mm_launch1<kMWide, 1, CT, 1, false, plan>(P, c.wgs, s)
                     : mm_launch1<kMWide, 2, CT, 1, false, plan>(P, c.wgs, s);
  return c.TM == 1 ? mm_launch1<kMWaves, 1, CT, 1, false, plan>(P, c.wgs, s)
                   : mm_launch1<kMWaves, 2, CT, 1, false, plan>(P, c.wgs, s);
}

template <bool plan>
static hipError_t mm_launch(const MmParams &P, const MmShape &c, hipStream_t s) {
  switch (c.CT) {
    case 1: return mm_launch2<1, plan>(P, c, s);
    case 2: return mm_launch2<2, plan>(P, c, s);
    case 3: return mm_launch2<3, plan>(P, c, s);
    case 4: return mm_launch2<4, plan>(P, c, s);
    default: return hipErrorInvalidValue;   // 1..64 tokens
  }
}

}  // namespace

hipError_t matmul_plan_prepare(const MmJobSpec *jobs, int n, int32_t B,
                               std::vector<uint8_t> &table, MmPlanCfg *cfg) {
  if (n < 1 || n > kMmPlanJobs || B < 1 || B > 64 || !cfg) return hipErrorInvalidValue;
  std::vector<MmJob> J(n);
  const MmShape s = mm_setup(jobs, n, B, J.data());
  const int per = mm_tiles_per_unit(s);
  // The units one after another, those of the longest matrices first:
  // workgroup r takes units r, r + wgs, ..., so the shares differ by less
  // than one unit of each K.
  std::vector<int> order(n);
  for (int j = 0; j < n; ++j) order[j] = j;
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int b) { return J[a].u.NG > J[b].u.NG; });
  table.resize((size_t)s.units * sizeof(MmUnit));
  MmUnit *out = (MmUnit *)table.data();
  for (int j : order)
    for (int t = 0; t < J[j].u.ntiles; t += per) {
      MmUnit &u = *out++;
      u = J[j].u;
      u.W += (int64_t)t * u.tile_bytes;
      u.ntiles -= t;
      u.row0 = t * kTileRows;
    }
  *cfg = MmPlanCfg{B, s.CT, s.TM, s.KS, s.NW, s.units, s.wgs};
  return hipSuccess;
}

hipError_t launch_matmul_plan(const void *d_table, const MmPlanCfg &cfg, int32_t *err,
                              hipStream_t s) {
  if (!d_table) return hipErrorInvalidValue;
  MmParams P{};
  P.units = cfg.units;
  P.B = cfg.B;
  P.err = err;
  P.tab = (const MmUnit *)d_table;
  return mm_launch<true>(P, MmShape{cfg.CT, cfg.TM, cfg.KS, cfg.NW, cfg.units, cfg.wgs}, s);
}

hipError_t launch_matmul_multi(const MmJobSpec *jobs, int n, int32_t B, int32_t *err,
                               hipStream_t s) {
  if (n < 1 || n > kMmJobs || B < 1 || B > 64) return hipErrorInvalidValue;
  MmParams P{};
  const MmShape c = mm_setup(jobs, n, B, P.job);
  P.njobs = n;
  P.units = c.units;
  P.B = B;
  P.err = err;
  return mm_launch<false>(P, c, s);
}

hipError_t launch_matmul(const uint8_t *w, int32_t nrows, const Layout &L, int32_t sh,
                         const int8_t *x8, int32_t B, int32_t *y32, int32_t *err,
                         hipStream_t s) {
  const MmJobSpec j{w, nrows, L, sh, x8, y32};
  return launch_matmul_multi(&j, 1, B, err, s);
}

}  // namespace w4a8
