// HIP kernels of the W4A8 matvec engine for gfx950 (MI355X).
//
// The integer law is the reference's: ref/w4a8_ref.py:254-289 (matvec_y32),
// ref/fixedpoint.py:24-75 (DYNQ8, rsqrt), ref/layer_fixed.py:1242-1278
// (RMSNorm), seq_model.py:1027-1050 + seq_movers.sv:759-836 (MOVY),
// gen_layer_script.py:1397-1433 (ALU ops, AMAX32).  Every product and sum is
// an exact integer, so any summation order gives bit-identical results.
#include <hip/hip_ext.h>

#include "w4a8_device.h"

namespace w4a8 {

// ---------------------------------------------------------------------------
// prologue: produce x8 (and e_x) in LDS.  Every workgroup computes the same
// values (DYNQ8 is one exponent over the whole vector and cannot be chunked,
// SEQ_ISA.md:560-569), so no grid-wide synchronisation is needed.  NT
// threads take pieces of 8 elements: thread t holds elements
// [c*NT*8 + 8t, +8) of piece c, so the 4 threads of a DPP quad hold 32
// consecutive elements -- one (group, k-quarter) of the weight layout.
//
// It stands between a launch's start and its first dot product, one chain of
// load, reductions and arithmetic on a few wavefronts, so its length is its
// instruction count and its LDS round trips.  One kernel instance per
// prologue kind, no branch per element: 16-bit steps run two elements an
// instruction (v_pk_*_i16), wide products are 32 x 32 + 64 multiply-adds on
// magnitudes, and a reduction is one LDS round trip (GroupRed).  From the
// first workgroup's start to the first dot product, K = 4096: DYNQ8 3.3 ->
// 2.4 us, RMSNorm 5.6 -> 3.9 us; with the way tiles meet (below) a layer's FFN
// block 25.4 -> 23.2 us, the chained step in graph mode 1.404 -> 1.291 ms.
// ---------------------------------------------------------------------------
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ s16x2 as_s16x2(int v) { return __builtin_bit_cast(s16x2, v); }
__device__ __forceinline__ int piece_word(const int4 &p, int i) {
  return i == 0 ? p.x : (i == 1 ? p.y : (i == 2 ? p.z : p.w));
}
__device__ __forceinline__ int pack16(int lo, int hi) {
  return (int)__builtin_amdgcn_perm((uint32_t)hi, (uint32_t)lo, 0x05040100u);
}

// clip16 of a magnitude with its sign
__device__ __forceinline__ int32_t clip16_mag(uint32_t q, bool neg) {
  const int32_t m = (int32_t)min(q, 32767u + (neg ? 1u : 0u));
  return neg ? -m : m;
}

// ALU EMUL32 at p0 = 12 (gen_layer_script.py:1414-1418):
// clip16(rshift_round(a * b, 12)), b int16
__device__ __forceinline__ int32_t emul12(int32_t a, int32_t b) {
  static_assert(kEmulP0 == 12, "");
  const uint32_t ma = a < 0 ? 0u - (uint32_t)a : (uint32_t)a, mb = (uint32_t)abs(b);
  const uint64_t v = (uint64_t)ma * mb + 2048u;     // |a * b| <= 2^46
  const uint32_t q = (uint32_t)(v >> 32) ? 0xFFFFFFFFu : (uint32_t)v;
  return clip16_mag(q >> 12, (a ^ b) < 0);
}

// 1/sqrt(v * 2^-P) ~= r * 2^(e-30), v >= 1: fixedpoint.py:56-75.  Every value
// of its int64 steps fits 32 bits (m < 2^32, r and r^2 >> 30 at most 2^30,
// m r^2 near 2^30), so each step is one 32 x 32 -> 64 product.
template <typename T>
__device__ __forceinline__ void rsqrt32(uint64_t v, int P, const T *lut, uint32_t *r_out,
                                        int *e_out) {
  int s = 32 - __clzll((long long)v);
  if ((s - P) & 1) s += 1;
  const uint32_t m = (uint32_t)(s >= 0 ? (v >> s) : (v << (-s)));
  const uint32_t idx = m < 0x80000000u ? (m >> 22) & 0xFFu : 256u | ((m >> 23) & 0xFFu);
  uint32_t r = (uint32_t)lut[idx] << 15;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const uint32_t r2 = (uint32_t)(((uint64_t)r * r) >> 30);
    const uint32_t mr2 = (uint32_t)(((uint64_t)m * r2) >> 30);
    r = (uint32_t)(((uint64_t)r * (0xC0000000u - mr2)) >> 31);
  }
  *r_out = r;
  *e_out = -((s - P + 30) / 2);
}

template <int PRO, int NT>
struct ProRegs {
  static constexpr int kPer = PRO == PRO_X8 ? 16 : 8;            // elements of a piece
  static constexpr int kK = PRO == PRO_RMSNORM_DYNQ8 ? 8192 : kKMax;
  static constexpr int kPc = (kK + NT * kPer - 1) / (NT * kPer);
  int4 pc[kPc];   // int16 x (PRO_X8: 16 int8 per piece), zeros past K
  int4 wv[PRO == PRO_RMSNORM_DYNQ8 ? kPc : 1];   // int16 RMSNorm weights
};

// the loads of x (and of the norm weights): issued before any weight load
template <int PRO, int NT>
__device__ __forceinline__ void pro_load(const GemvParams &P, ProRegs<PRO, NT> &X, int tid) {
  typedef ProRegs<PRO, NT> R;
  const int K = P.K;
  const int4 z = make_int4(0, 0, 0, 0);
#pragma unroll
  for (int c = 0; c < R::kPc; ++c) {
    const int i = (c * NT + tid) * R::kPer;
    X.pc[c] = z;
    if constexpr (PRO == PRO_RMSNORM_DYNQ8) X.wv[c] = z;
    if (i < K) {
      if constexpr (PRO == PRO_X8) X.pc[c] = *(const int4 *)((const int8_t *)P.x + i);
      else X.pc[c] = *(const int4 *)((const int16_t *)P.x + i);
      if constexpr (PRO == PRO_RMSNORM_DYNQ8) X.wv[c] = *(const int4 *)(P.norm_w + i);
    }
  }
  if constexpr (PRO == PRO_EMUL_DYNQ8) {
    int4 a[R::kPc][2];
#pragma unroll
    for (int c = 0; c < R::kPc; ++c) {
      const int i = (c * NT + tid) * 8;
      a[c][0] = a[c][1] = z;
      if (i < K) {
        a[c][0] = *(const int4 *)(P.x2 + i);
        a[c][1] = *(const int4 *)(P.x2 + i + 4);
      }
    }
#pragma unroll
    for (int c = 0; c < R::kPc; ++c)
      if (c * NT * 8 < K) {
        const int av[8] = {a[c][0].x, a[c][0].y, a[c][0].z, a[c][0].w,
                           a[c][1].x, a[c][1].y, a[c][1].z, a[c][1].w};
        int o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const s16x2 g = as_s16x2(piece_word(X.pc[c], i));
          o[i] = pack16(emul12(av[2 * i], g.x), emul12(av[2 * i + 1], g.y));
        }
        X.pc[c] = make_int4(o[0], o[1], o[2], o[3]);
      }
  }
}

// The prologue's reductions over its wavefronts when the whole workgroup
// runs it (sm: 2 * NW int64 of LDS).
template <int NW>
struct WgRed {
  int64_t *sm;
  __device__ uint64_t sum(uint64_t v, int wave, int lane) {
    if (lane == 0) sm[wave] = (int64_t)v;
    __syncthreads();
    uint64_t t = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) t += (uint64_t)sm[w];
    return t;
  }
  __device__ int32_t max(int32_t v, int wave, int lane) {
    if (lane == 0) sm[NW + wave] = v;
    __syncthreads();
    int32_t t = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) t = ::max(t, (int32_t)sm[NW + w]);
    return t;
  }
  __device__ void done(int, int) { __syncthreads(); }
};

// ... and when 8 wavefronts of a larger workgroup run it: no workgroup
// barrier, since the others may be stalled behind their weight loads.  Each
// wavefront posts its value with a valid bit, and polls the eight words until
// all have it: one LDS round trip for value and flag, the eight lanes of a
// half row holding the eight values.
struct ProWords {
  uint64_t sum[8];    // zero at the launch's start; bit 63: valid
  uint32_t max[8];    // bit 31: valid
  int32_t ready[8];   // the wavefront's share of x8 is stored
};
__device__ __forceinline__ uint64_t lds_read_u64(const uint64_t *p) {
  uint64_t v;
  asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(lds_off(p)) : "memory");
  return v;
}
__device__ __forceinline__ void lds_post_u64(uint64_t *p, uint64_t v) {
  asm volatile("ds_write_b64 %0, %1" :: "v"(lds_off(p)), "v"(v) : "memory");
}
__device__ __forceinline__ void lds_post_i32(int32_t *p, int32_t v) {
  asm volatile("ds_write_b32 %0, %1" :: "v"(lds_off(p)), "v"(v) : "memory");
}
struct GroupRed {
  ProWords *w;
  bool ok;    // false once a poll gave up
  __device__ uint64_t sum(uint64_t v, int wave, int lane) {
    if (lane == 0) lds_post_u64(&w->sum[wave], v | (1ull << 63));
    uint64_t t = 0;
    bool got = false;
    for (uint32_t n = 0; n < kLdsSpin && !got; ++n) {
      t = lds_read_u64(&w->sum[lane & 7]);
      got = __all((int64_t)t < 0);
    }
    ok = ok && got;
    t &= ~(1ull << 63);
    t += dpp_u64<0xB1, 0xF>(t);    // pairs, quads, half rows
    t += dpp_u64<0x4E, 0xF>(t);
    t += dpp_u64<0x141, 0xF>(t);
    return t;
  }
  __device__ int32_t all_max(int lane) {
    int32_t t = 0;
    bool got = false;
    for (uint32_t n = 0; n < kLdsSpin && !got; ++n) {
      t = lds_read_i32((const int32_t *)&w->max[lane & 7]);
      got = __all(t < 0);
    }
    ok = ok && got;
    t &= 0x7FFFFFFF;
    t = ::max(t, W4A8_DPP(t, 0, 0xB1, 0xF));
    t = ::max(t, W4A8_DPP(t, 0, 0x4E, 0xF));
    return ::max(t, W4A8_DPP(t, 0, 0x141, 0xF));
  }
  __device__ int32_t max(int32_t v, int wave, int lane) {
    if (lane == 0) lds_post_i32((int32_t *)&w->max[wave], v | (int32_t)0x80000000);
    return all_max(lane);
  }
  // every wavefront's share of x8 is stored (a wavefront's LDS instructions
  // execute in order); backoff: 64 cycles between polls
  template <bool backoff = false>
  __device__ void wait_ready(int lane) {
    bool got = false;
    for (uint32_t n = 0; n < kLdsSpin && !got; ++n) {
      got = __all(lds_read_i32(&w->ready[lane & 7]) != 0);
      if (backoff && !got) __builtin_amdgcn_s_sleep(1);
    }
    ok = ok && got;
  }
  __device__ void done(int wave, int lane) {
    if (lane == 0) lds_post_i32(&w->ready[wave], 1);
    wait_ready(lane);
  }
};

// A workgroup barrier that waits for LDS alone: __syncthreads may also wait
// for the weight loads in flight.
__device__ __forceinline__ void meet() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// fixedpoint.py:24-33: the least e with rshift_round(max, e) <= 127 is
// bitlen(max) - 7, or one more when rounding carries past 127
__device__ __forceinline__ int dynq8_exponent(int32_t mx) {
  int e = mx > 127 ? 25 - __clz(mx) : 0;
  if (e > 0 && ((mx + (1 << (e - 1))) >> e) > 127) ++e;
  return e;
}

// Leaves x8 in xs[0, K) and the offset corrections -8 * (sum of the x8 met by
// the offset-form low nibbles of each (group, k-quarter)) in xlo; returns e_x.
template <int PRO, int NT, typename TabT, typename Red>
__device__ __forceinline__ int pro_compute(const GemvParams &P, ProRegs<PRO, NT> &X, int8_t *xs,
                                           int32_t *xlo, const TabT *rsqrt_lut, int tid,
                                           Red &red) {
  typedef ProRegs<PRO, NT> R;
  const int K = P.K;
  const int lane = tid & 63, wave = tid >> 6;
  const bool writer = blockIdx.x == 0;
  if constexpr (PRO == PRO_X8) {
#pragma unroll
    for (int c = 0; c < R::kPc; ++c) {
      const int i = (c * NT + tid) * 16;
      // the two threads of a pair hold one (group, k-quarter)
      int s = __builtin_amdgcn_sdot4(X.pc[c].x, 0x01010101, 0, false);
      s = __builtin_amdgcn_sdot4(X.pc[c].z, 0x01010101, s, false);
      s += W4A8_DPP(s, 0, 0xB1, 0xF);
      if (i < K) {
        *(int4 *)(xs + i) = X.pc[c];
        if ((tid & 1) == 0) xlo[i / 32] = -8 * s;
        if (writer && P.x8_out) *(int4 *)(P.x8_out + i) = X.pc[c];
      }
    }
    if (writer && P.e_x_out && tid == 0) *P.e_x_out = P.e_x_given;
    red.done(wave, lane);
    return P.e_x_given;
  }
  if constexpr (PRO == PRO_RMSNORM_DYNQ8) {
    // layer_fixed.py:1262-1278 in sign-magnitude form: rshift_round rounds
    // the magnitude, so |x * r| and |y * sc| carry the rounding and the
    // sign is restored afterwards
    uint64_t ss = 0;
#pragma unroll
    for (int c = 0; c < R::kPc; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const s16x2 v = as_s16x2(piece_word(X.pc[c], i));
        ss += (uint32_t)__builtin_amdgcn_sdot2(v, v, 0, false);   // at most 2^31
      }
    ss = red.sum(wave_sum_u64(ss), wave, lane);
    if (ss == 0) ss = 1;
    uint32_t r;
    int e;
    rsqrt32(ss, 2 * P.in_f + (31 - __clz(K)), rsqrt_lut, &r, &e);
    // r < 2^31 (a Q30 reciprocal square root) and |x| <= 2^15; for in_f in
    // 0..40 (checked on the host) a left shift is at most 17, so the shifted
    // |x| * r stays below 2^63
    const int s1 = 30 - e;
    const int32_t one = P.one_plus ? (1 << 14) : 0;
    const int rs = s1 < 0 ? 0 : (s1 > 63 ? 63 : s1), ls = s1 < 0 ? -s1 : 0;
    const uint64_t half1 = rs > 0 ? ((uint64_t)1 << (rs - 1)) : 0;
    auto norm = [&](int32_t xv, int32_t wv, bool left) {
      const int32_t sc = wv + one;
      const uint64_t mag = (uint64_t)(uint32_t)abs(xv) * (uint64_t)r + half1;
      const uint64_t ym = left ? mag << ls : mag >> rs;
      // y is clipped to [-2^32, 2^32 - 1]; a magnitude of 2^32 or more
      // saturates the int16 result for any nonzero scale exactly as
      // 2^32 - 1 does, so the product is formed in 32 x 32 bits
      const uint32_t y = (uint32_t)(ym >> 32) ? 0xFFFFFFFFu : (uint32_t)ym;
      const uint64_t qv = (uint64_t)y * (uint64_t)(uint32_t)abs(sc) + 8192u;
      // qv >> 14, saturated: above 2^32 it is past the clip
      const uint32_t q = (uint32_t)(qv >> 32) ? 0xFFFFFFFFu : (uint32_t)qv;
      return clip16_mag(q >> 14, (xv ^ sc) < 0);
    };
    auto pieces = [&](bool left) {
#pragma unroll
      for (int c = 0; c < R::kPc; ++c)
        if (c * NT * 8 < K) {
          int o[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const s16x2 v = as_s16x2(piece_word(X.pc[c], i)), w = as_s16x2(piece_word(X.wv[c], i));
            o[i] = pack16(norm(v.x, w.x, left), norm(v.y, w.y, left));
          }
          X.pc[c] = make_int4(o[0], o[1], o[2], o[3]);
          const int base = (c * NT + tid) * 8;
          if (writer && P.xn_out && base < K) *(int4 *)(P.xn_out + base) = X.pc[c];
        }
    };
    if (s1 >= 0) pieces(false);
    else pieces(true);
  }
  s16x2 hi = {0, 0}, lo = {0, 0};
#pragma unroll
  for (int c = 0; c < R::kPc; ++c)
    if (c * NT * 8 < K)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const s16x2 v = as_s16x2(piece_word(X.pc[c], i));
        hi = __builtin_elementwise_max(hi, v);
        lo = __builtin_elementwise_min(lo, v);
      }
  int32_t mx = max(max((int)hi.x, (int)hi.y), -min((int)lo.x, (int)lo.y));
  const int e = dynq8_exponent(red.max(wave_max_i32(mx), wave, lane));
  // magnitudes in 16 bits: |x| <= 2^15, plus half (at most 2^8)
  const unsigned short half = (unsigned short)((1 << e) >> 1), sh = (unsigned short)e;
  const u16x2 halves = {half, half}, shifts = {sh, sh}, most = {127, 127};
#pragma unroll
  for (int c = 0; c < R::kPc; ++c)
    if (c * NT * 8 < K) {
      const int base = (c * NT + tid) * 8;
      uint32_t q[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const s16x2 v = as_s16x2(piece_word(X.pc[c], i)), sg = v >> 15;
        u16x2 m = __builtin_bit_cast(u16x2, (v ^ sg) - sg);
        m = __builtin_elementwise_min((m + halves) >> shifts, most);
        q[i] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(s16x2, m) ^ sg) - sg);
      }
      const uint32_t lo8 = __builtin_amdgcn_perm(q[1], q[0], 0x06040200u);
      const uint32_t hi8 = __builtin_amdgcn_perm(q[3], q[2], 0x06040200u);
      int t4 = __builtin_amdgcn_sdot4((int)lo8, 0x01010101, 0, false);
      t4 += __builtin_amdgcn_update_dpp(0, t4, 0xB1, 0xF, 0xF, false);
      t4 += __builtin_amdgcn_update_dpp(0, t4, 0x4E, 0xF, 0xF, false);
      if (base < K) {
        *(uint2 *)(xs + base) = make_uint2(lo8, hi8);
        if ((tid & 3) == 0) xlo[base / 32] = -8 * t4;
        if (writer && P.x8_out) *(uint2 *)(P.x8_out + base) = make_uint2(lo8, hi8);
      }
    }
  if (writer && P.e_x_out && tid == 0) *P.e_x_out = e;
  red.done(wave, lane);
  return e;
}

// ---------------------------------------------------------------------------
// the GEMV: one 768-thread workgroup per CU, 3 teams of 4 wavefronts that
// share one prologue.  Team v of workgroup r takes tiles r + G*(v + 3i);
// its wavefronts split a tile's scale blocks, each keeping its next two
// blocks in flight.  Where no workgroup has a second tile and a tile has more
// than 4 blocks (a 4096 x 12288 down projection on 256 CUs), the 12
// wavefronts are one team.  A tile's sums meet in an LDS slot; the wavefront
// that adds last finishes the tile, so no team waits for another.
// ---------------------------------------------------------------------------
__device__ __forceinline__ const uint8_t *block_addr(const GemvParams &P, int tg, int b) {
  const int j = job_of(P, tg);
  return P.job[j].w + (int64_t)(tg - P.job[j].tile0) * P.tile_bytes +
         (int64_t)b * kBlockBytes;
}

// This wavefront's blocks over the kernel: for its team's tiles it = 0, 1,
// ... (tile tg0 + VS * it < total_tiles), blocks b = wt, wt + W, ... < nblk --
// nbw blocks per tile, the same for every tile.
struct Item {
  int k;    // position in the sequence
  int it;   // tile iteration
  int j;    // b = wt + W * j
};
__device__ __forceinline__ void item_next(Item &c, int nbw) {
  ++c.k;
  if (++c.j == nbw) {
    c.j = 0;
    ++c.it;
  }
}

// Put a block in flight: always exactly 1 + kGroupsPerBlock loads, so the
// compiler's count of outstanding loads is the same on every path.  The loads are
// buffer loads whose range ends with the block's data: past the end of the
// sequence (range 0), and for the missing groups of a short block, they are
// out of range, return zero and make no memory access.
constexpr int kBufDword3 = 0x00020000;   // raw buffer, 32-bit data format (gfx9)

// The buffer resource of block b of global tile tg (an empty range when not
// real: its loads return zero without a memory access).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t block_rsrc(const GemvParams &P, int tg, int b,
                                                            bool real) {
  const uint8_t *bb = real ? block_addr(P, tg, b) : (const uint8_t *)P.tables;
  const int len = real ? kScaleChunk + groups_in(P.NG, b) * kGroupChunk : 0;
  return __builtin_amdgcn_make_buffer_rsrc((void *)bb, (short)0, len, kBufDword3);
}
__device__ __forceinline__ void issue_rsrc(BlockRegs &R, __amdgpu_buffer_rsrc_t rs, int lane) {
  const u32x4_t sc = __builtin_amdgcn_raw_buffer_load_b128(rs, (lane >> 2) * 16, 0, kAuxNt);
  R.sc = make_uint4(sc.x, sc.y, sc.z, sc.w);
#pragma unroll
  for (int i = 0; i < kGroupsPerBlock; ++i) {
    const u32x4_t w = __builtin_amdgcn_raw_buffer_load_b128(
        rs, kScaleChunk + i * kGroupChunk + lane * 16, 0, kAuxNt);
    R.w[i] = make_uint4(w.x, w.y, w.z, w.w);
  }
}
__device__ __forceinline__ void issue_block(BlockRegs &R, const GemvParams &P, int tg, int b,
                                            bool real, int lane) {
  issue_rsrc(R, block_rsrc(P, tg, b, real), lane);
}

// v is computed at this point
__device__ __forceinline__ void computed(__amdgpu_buffer_rsrc_t rs) {
  asm volatile("" ::"s"(rs));
}
// a copy of v that the compiler knows nothing about
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

constexpr int kGT = 768;
constexpr int kGWaves = kGT / 64;
constexpr int kGTeams = kGWaves / 4;
constexpr int kPW0 = 4;                // teams 1 and 2 (wavefronts 4..11) run the prologue
constexpr int kPT = kGT - 64 * kPW0;   // 512 threads

// The LDS slots in which a team's tiles meet, where it has no more than two
// (a longer stream goes in step, below): tile iteration `it` in slot it, used
// once, so nothing is cleared for reuse or waited for.  Zeroed before the
// workgroup meets, so their number is on the launch's path (eight a team:
// 4096 x 4096 5.26 us in a graph of launches, two: 5.10).
constexpr int kSlots = 2;
struct TileSlot {
  uint64_t sum[kTileRows];   // 16 * p of each row
  int32_t cnt;               // wavefronts that have added
  int32_t pad;
};
__device__ __forceinline__ void lds_add_u64(uint64_t *p, uint64_t v) {
  asm volatile("ds_add_u64 %0, %1" :: "v"(lds_off(p)), "v"(v) : "memory");
}
__device__ __forceinline__ int32_t lds_add_rtn(int32_t *p, int32_t v) {
  int32_t old;
  asm volatile("ds_add_rtn_u32 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)"
               : "=v"(old) : "v"(lds_off(p)), "v"(v) : "memory");
  return old;
}

// 16 * p reduced over the 4 k-quarter lanes
__device__ __forceinline__ int64_t quarter_sum(int64_t p) {
  p = (int64_t)((uint64_t)p + dpp_u64<0xB1, 0xF>((uint64_t)p));
  return (int64_t)((uint64_t)p + dpp_u64<0x4E, 0xF>((uint64_t)p));
}

// Add this wavefront's share of a tile (quarter_sum) to the tile's slot; true
// in the wavefront that adds last of nw, which gets lane l < 16's row sum in
// tot.  (A wavefront's LDS instructions execute in order, so the count
// follows the sums.)
__device__ __forceinline__ bool tile_add(TileSlot &S, int nw, int64_t p, int lane, int64_t &tot) {
  if ((lane & 3) == 0) lds_add_u64(&S.sum[lane >> 2], (uint64_t)p);
  int32_t old = 0;
  if (lane == 0) old = lds_add_rtn(&S.cnt, 1);
  if (__builtin_amdgcn_readfirstlane(old) != nw - 1) return false;
  if (lane < kTileRows) tot = (int64_t)lds_read_u64(&S.sum[lane]);
  return true;
}

// round, check and write the 16 rows of tile t (lane l: row 16 t + l)
__device__ __forceinline__ void tile_finish(const GemvJob &J, int t, int64_t tot, int lane,
                                            int e_x, const uint16_t *sig, int32_t *err,
                                            uint64_t &best) {
  const int row = t * kTileRows + lane;
  if (lane < kTileRows && row < J.nrows) {
    const int64_t y = rshr64(tot >> 4, J.sh);   // tot is 16 * p exactly
    if (y > 2147483647LL || y < -2147483647LL) atomicOr(err, 1);
    const int shift = J.p0 - e_x;
    switch (J.epi) {
      case EPI_Y32:
        ((int32_t *)J.out)[row] = (int32_t)y;
        break;
      case EPI_MOVY_I16:
        ((int16_t *)J.out)[row] = (int16_t)clamp64(movy_shift(y, shift), -32768, 32767);
        break;
      case EPI_MOVY_I16_ADD: {
        const int64_t v = clamp64(movy_shift(y, shift), -32768, 32767);
        if (J.out) ((int16_t *)J.out)[row] = (int16_t)v;
        J.res_out[row] = (int16_t)clamp64(v + J.res[row], -32768, 32767);
        break;
      }
      case EPI_MOVY_P32:
        ((int32_t *)J.out)[row] =
            (int32_t)clamp64(movy_shift(y, shift), -2147483648LL, 2147483647LL);
        break;
      case EPI_SILU32:
        ((int16_t *)J.out)[row] = (int16_t)silu32(y, shift, sig);
        break;
      case EPI_SHIFT_I64:
        ((int64_t *)J.out)[row] = movy_shift(y, shift);
        break;
      default: {   // EPI_ARGMAX: raw y32 (shift 0), seq_format.py:2225-2226
        const uint64_t k = argmax_key((int32_t)y, (uint32_t)row);
        best = k > best ? k : best;
      }
    }
  }
}

template <int PRO>
__global__ __launch_bounds__(kGT) void gemv_kernel(GemvParams P) {
  __shared__ __align__(16) int8_t xs[kKMax];
  __shared__ int32_t xlo[kKMax / 32];
  __shared__ TileSlot slots[kGTeams][kSlots];
  __shared__ int64_t red[2][kGTeams][4][kTileRows];   // lockstep
  __shared__ uint64_t keys[kGWaves];
  __shared__ uint16_t tab_rsqrt[PRO == PRO_RMSNORM_DYNQ8 ? 512 : 1], tab_sig[264];
  __shared__ ProWords words;

  const int tid = threadIdx.x, lane = tid & 63;
  // wave index as a scalar so the block loops below branch on SGPRs
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NG = P.NG, nblk = P.nblk, T = P.total_tiles;
  const int G = gridDim.x, r = blockIdx.x;
  // one team of 12: 4096 x 12288 8.4 -> 6.4 us from the first workgroup's start
  // to the last's end (a tile's 24 blocks on 12 wavefronts, two each, instead
  // of six in turn on four)
  const bool wide = T <= G && nblk > 4;
  const int W = wide ? kGWaves : 4;                 // wavefronts of a team
  const int team = wide ? 0 : wave >> 2, wt = wide ? wave : wave & 3;
  const int VS = wide ? G : G * kGTeams;
  const int nw = min(W, nblk);                      // ... that have blocks of a tile
  if (tid < (int)(sizeof(words) / 4)) ((int32_t *)&words)[tid] = 0;
  for (int i = tid; i < (int)(sizeof(slots) / 4); i += kGT) ((int32_t *)slots)[i] = 0;
  // A long stream (the LM head) keeps its wavefronts in step, one barrier per
  // tile iteration: the GPU then sweeps one window of memory, where drifting
  // wavefronts read at 0.92 of that (248,320 x 4096: 81.3 us in step, 89 us
  // without).  Short launches (up to two tiles per team) run without: no team
  // waits for another's first blocks (chained step in graph mode 1.33 ms in
  // step from the second tile on, 1.29 ms without).
  const bool lockstep = T > kSlots * VS;
  if (lockstep)
    for (int i = tid; i < (int)(sizeof(red) / 4); i += kGT) ((int32_t *)red)[i] = 0;

  // A CU's first weight blocks take microseconds to drain at its share of
  // HBM bandwidth, and a wavefront cannot issue past a load the memory
  // pipeline has no room for.  So teams 1 and 2 issue the activation and
  // table loads, the workgroup meets once (nothing is waited for), and only
  // then do wavefronts 0-3 put their first blocks in flight, behind the
  // activations.  Wavefronts 4-11 issue theirs after the prologue: issued
  // before its arithmetic, they stall it for as long as the memory pipeline is
  // full (chained step in graph mode 1.44 -> 1.61 ms).
  // Two register sets per wavefront, A and B, hold its next two blocks.
  const int tg0 = r + G * team;
  const int nbw = wt >= nblk ? 0 : wide ? (nblk - wt + kGWaves - 1) / kGWaves : (nblk - wt + 3) / 4;
  const int nitems = tg0 < T ? ((T - 1 - tg0) / VS + 1) * nbw : 0;
  Item ca{0, 0, 0}, cb = ca;
  if (nbw > 0) item_next(cb, nbw);
  Item cn = cb;
  if (nbw > 0) item_next(cn, nbw);
  BlockRegs A, B;
  const int pt = tid - kPW0 * 64;   // thread index within the prologue group
  GroupRed grp{&words, true};
  int e_x;
  if (wave < kPW0) {
    // the blocks' addresses first (the kernel arguments they need come in by
    // scalar loads, a round trip or two at a launch's start), so that the
    // loads go out as soon as the workgroup has met: C0 as one launch per
    // matrix 5.49 -> 5.38 us
    const __amdgpu_buffer_rsrc_t rsA = block_rsrc(P, tg0, wt, nitems > 0);
    const __amdgpu_buffer_rsrc_t rsB =
        block_rsrc(P, tg0 + VS * cb.it, wt + W * cb.j, cb.k < nitems);
    computed(rsA);
    computed(rsB);
    meet();
    issue_rsrc(A, rsA, lane);
    issue_rsrc(B, rsB, lane);
    grp.wait_ready<true>(lane);
    e_x = PRO == PRO_X8 ? P.e_x_given : dynq8_exponent(grp.all_max(lane));
    e_x = __builtin_amdgcn_readfirstlane(e_x);
  } else {
    static_assert(kPT >= 512 && kPT >= 257, "one table entry per thread");
    ProRegs<PRO, kPT> X;
    pro_load<PRO, kPT>(P, X, pt);
    int trs = 0;
    if constexpr (PRO == PRO_RMSNORM_DYNQ8) trs = P.tables[kRsqrtOff + pt];
    const int tsg = P.tables[kSigmoidOff + (pt < 257 ? pt : 0)];
    meet();
    if constexpr (PRO == PRO_RMSNORM_DYNQ8) tab_rsqrt[pt] = (uint16_t)trs;
    if (pt < 257) tab_sig[pt] = (uint16_t)tsg;
    e_x = pro_compute<PRO, kPT>(P, X, xs, xlo, tab_rsqrt, pt, grp);
    e_x = __builtin_amdgcn_readfirstlane(e_x);
    if (nitems > 0) {
      issue_block(A, P, tg0, wt, true, lane);
      issue_block(B, P, tg0 + VS * cb.it, wt + W * cb.j, cb.k < nitems, lane);
    }
  }

  // the first tile's job, its fields read before anything waits for them
  int jcur = job_of(P, tg0 < T ? tg0 : 0);
  GemvJob J = P.job[jcur];
  const uint16_t *sig = tab_sig;
  uint64_t best = 0;   // argmax key (0 == none)
  int64_t p = 0;
  auto finish = [&](int tg, int64_t tot, int lane) {
    const int j = job_of(P, tg);
    if (j != jcur) {
      jcur = j;
      J = P.job[j];
    }
    tile_finish(J, tg - J.tile0, tot, lane, e_x, sig, P.err, best);
  };
  // In step, a team's wavefronts finish its tiles in turn, those without
  // blocks of a tile (K <= 3072) too.  Left to the wavefronts that have
  // blocks, the epilogues are all one wavefront's where a tile is one block
  // (K <= 1024): 248,320 x 1024 with argmax 53.5 us, 43.9 in turn; 64,000 x
  // 640 with MOVY int16 15.4 and 13.1; nothing changes from K = 4096 on.
  int fin = 0;   // tile iterations finished
  auto finish_in_step = [&](int tg, int lane) {
    const int par = fin & 1;
    const bool mine = wt == (fin & 3);
    meet();
    ++fin;
    if (mine && tg < T)
      finish(tg, red[par][team][0][lane & 15] + red[par][team][1][lane & 15] +
                     red[par][team][2][lane & 15] + red[par][team][3][lane & 15], lane);
  };
  // consume the block in R (item c), add to its tile after the wavefront's
  // last block of it, and refill R with the item two ahead
  auto step = [&](BlockRegs &R, Item &c) {
    // lane-derived offsets are recomputed from an opaque copy of the thread
    // index, so the compiler does not keep them all live across the loop
    const int tid_s = opaque(tid);
    const int lane = tid_s & 63, q = lane & 3;
    const int b = wt + W * c.j;
    const int tg = tg0 + VS * c.it, it = c.it;
    const bool last = c.j == nbw - 1;
    p = dot_block(R, groups_in(NG, b), b * kGroupsPerBlock, q, xs, xlo, p);
    if (last) {
      p = quarter_sum(p);
      if (lockstep) {
        if ((lane & 3) == 0) red[it & 1][team][wt][lane >> 2] = p;
        finish_in_step(tg, lane);
      } else {
        int64_t tot = 0;
        if (tile_add(slots[team][it], nw, p, lane, tot)) finish(tg, tot, lane);
      }
      p = 0;
    }
    c = cn;
    item_next(cn, nbw);
    issue_block(R, P, tg0 + VS * c.it, wt + W * c.j, c.k < nitems, lane);
  };
  for (int k = 0; k < nitems; k += 2) {
    step(A, ca);
    if (k + 1 >= nitems) break;
    step(B, cb);
  }
  // tile iterations this wavefront has no block of (team 0 has the most tiles)
  if (lockstep)
    for (const int iters = (T - r + VS - 1) / VS; fin < iters;)
      finish_in_step(tg0 + VS * fin, lane);
  if (!grp.ok && lane == 0) atomicOr(P.err, 4);
  if (P.partials) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const uint64_t other = __shfl_xor(best, o);
      best = other > best ? other : best;
    }
    if (lane == 0) keys[wave] = best;
    __syncthreads();
    if (tid == 0) {
      uint64_t k = keys[0];
      for (int w = 1; w < kGWaves; ++w) k = keys[w] > k ? keys[w] : k;
      P.partials[r] = k;
    }
  }
}

__global__ __launch_bounds__(kWG) void argmax_final_kernel(
    const uint64_t *partials, int n, int32_t *result) {
  __shared__ uint64_t keys[kWaves];
  uint64_t best = 0;
  for (int i = threadIdx.x; i < n; i += kWG) best = partials[i] > best ? partials[i] : best;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t other = __shfl_xor(best, o);
    best = other > best ? other : best;
  }
  if ((threadIdx.x & 63) == 0) keys[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kWaves; ++w) best = keys[w] > best ? keys[w] : best;
    best = keys[0] > best ? keys[0] : best;
    result[0] = (int32_t)(0xFFFFFFFFu - (uint32_t)(best & 0xFFFFFFFFu));
    result[1] = (int32_t)((uint32_t)(best >> 32) ^ 0x80000000u);
  }
}

// prologue only: DYNQ8 / RMSNorm(+DYNQ8) of one vector, one workgroup
template <int PRO>
__global__ __launch_bounds__(kWG) void vec_prologue_kernel(GemvParams P) {
  __shared__ __align__(16) int8_t xs[kKMax];
  __shared__ int32_t xlo[kKMax / 32];
  __shared__ int64_t sm[2 * kWaves];
  ProRegs<PRO, kWG> X;
  pro_load<PRO, kWG>(P, X, threadIdx.x);
  WgRed<kWaves> red{sm};
  pro_compute<PRO, kWG>(P, X, xs, xlo, P.tables + kRsqrtOff, threadIdx.x, red);
}

// ---------------------------------------------------------------------------
// repack: row image (w4a8_ref.py:349-370) <-> tile layout
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t to_tile_word(uint32_t in) {
  // nibble t of `in` is w[k0+t] (two's complement)
  uint32_t out = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t lo = ((in >> (4 * i)) & 15u) ^ 8u;
    const uint32_t hi = (in >> (4 * (4 + i))) & 15u;
    out |= (lo | (hi << 4)) << (8 * i);
  }
  return out;
}
__device__ __forceinline__ uint32_t from_tile_word(uint32_t out) {
  uint32_t in = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t byte = (out >> (8 * i)) & 0xFFu;
    in |= ((byte & 15u) ^ 8u) << (4 * i);
    in |= (byte >> 4) << (4 * (4 + i));
  }
  return in;
}

__device__ __forceinline__ uint8_t *group_piece(uint8_t *base, const Layout &L,
                                                int64_t r, int g) {
  const int64_t t = r / kTileRows;
  const int rr = (int)(r % kTileRows);
  return base + t * L.tile_bytes + (int64_t)(g / kGroupsPerBlock) * kBlockBytes +
         kScaleChunk + (g % kGroupsPerBlock) * kGroupChunk + rr * 64;
}
__device__ __forceinline__ uint8_t *scale_piece(uint8_t *base, const Layout &L,
                                                int64_t r, int b) {
  const int64_t t = r / kTileRows;
  const int rr = (int)(r % kTileRows);
  return base + t * L.tile_bytes + (int64_t)b * kBlockBytes + rr * 16;
}

__global__ void repack_groups_kernel(const uint8_t *img, int64_t nrows, Layout L,
                                     int64_t stride, uint8_t *dst) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= nrows * L.NG) return;
  const int64_t r = gid / L.NG;
  const int g = (int)(gid % L.NG);
  const uint4 *src = (const uint4 *)(img + r * stride + 64 * g);
  uint4 *d = (uint4 *)group_piece(dst, L, r, g);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint4 v = src[q];
    d[q] = make_uint4(to_tile_word(v.x), to_tile_word(v.y), to_tile_word(v.z),
                      to_tile_word(v.w));
  }
}

__global__ void repack_scales_kernel(const uint8_t *img, int64_t nrows, Layout L,
                                     int64_t stride, uint8_t *dst) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= nrows * L.nblk) return;
  const int64_t r = gid / L.nblk;
  const int b = (int)(gid % L.nblk);
  const uint8_t *s = img + r * stride + L.K / 2;
  uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int g = b * kGroupsPerBlock + j;
    if (g < L.NG) {
      const uint32_t m = (uint32_t)s[2 * g] | ((uint32_t)s[2 * g + 1] << 8);
      w[j >> 1] |= m << (16 * (j & 1));
    }
  }
  *(uint4 *)scale_piece(dst, L, r, b) = make_uint4(w[0], w[1], w[2], w[3]);
}

__global__ void unpack_groups_kernel(const uint8_t *src, int64_t nrows, Layout L,
                                     int64_t stride, uint8_t *img) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= nrows * L.NG) return;
  const int64_t r = gid / L.NG;
  const int g = (int)(gid % L.NG);
  const uint4 *s = (const uint4 *)group_piece(const_cast<uint8_t *>(src), L, r, g);
  uint4 *d = (uint4 *)(img + r * stride + 64 * g);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint4 v = s[q];
    d[q] = make_uint4(from_tile_word(v.x), from_tile_word(v.y),
                      from_tile_word(v.z), from_tile_word(v.w));
  }
}

__global__ void unpack_scales_kernel(const uint8_t *src, int64_t nrows, Layout L,
                                     int64_t stride, uint8_t *img) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= nrows * L.nblk) return;
  const int64_t r = gid / L.nblk;
  const int b = (int)(gid % L.nblk);
  const uint4 v = *(const uint4 *)scale_piece(const_cast<uint8_t *>(src), L, r, b);
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint8_t *s = img + r * stride + L.K / 2;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int g = b * kGroupsPerBlock + j;
    if (g < L.NG) {
      const uint32_t m = (w[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
      s[2 * g] = (uint8_t)(m & 0xFF);
      s[2 * g + 1] = (uint8_t)(m >> 8);
    }
  }
}

// ---------------------------------------------------------------------------
// elementwise law ops
// ---------------------------------------------------------------------------
__global__ void fill_i32_kernel(int32_t *p, int32_t v, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// One workgroup: the copies are a few KB to 150 KB, and a single group can
// tell when all of it has been written.  Bound by the link's round trip.
__global__ __launch_bounds__(1024) void host_copy_kernel(HostCopy c) {
  const uint4 *src = (const uint4 *)c.src;
  uint4 *dst = (uint4 *)c.dst;
  const int n16 = c.n / 16;
  for (int i = threadIdx.x; i < n16; i += 1024) dst[i] = src[i];
  if (!c.flag) return;
  if (threadIdx.x == 0) *c.err_out = *c.err;
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(c.flag, c.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void rshift_round_kernel(const int64_t *v, int64_t n, int s, int64_t *out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = rshr64(v[i], s);
}

__global__ void movy_kernel(const int32_t *y, int64_t n, int shift, int mode, void *out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t v = movy_shift(y[i], shift);
    if (mode == 1) ((int16_t *)out)[i] = (int16_t)clamp64(v, -32768, 32767);
    else ((int32_t *)out)[i] = (int32_t)clamp64(v, -2147483648LL, 2147483647LL);
  }
}

__global__ void alu_kernel(int op, const int32_t *y, const int16_t *b, int64_t n,
                           int p0, const int32_t *tables, void *out) {
  const int32_t *sig = tables + kSigmoidOff;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t v = y[i];
    switch (op) {
      case 1:   // SHIFT32
        ((int16_t *)out)[i] = (int16_t)clamp64(movy_shift(v, p0), -32768, 32767);
        break;
      case 6:   // SILU32
        ((int16_t *)out)[i] = (int16_t)silu32(v, p0, sig);
        break;
      case 8:   // EMUL32: clip16(rshift_round(y * b, p0))
        ((int16_t *)out)[i] = (int16_t)clamp64(movy_shift(v * (int64_t)b[i], p0),
                                               -32768, 32767);
        break;
      default:  // 9 SHIFT32W
        ((int32_t *)out)[i] = (int32_t)clamp64(movy_shift(v, p0),
                                               -2147483648LL, 2147483647LL);
    }
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int blocks_for(int64_t n, int threads, int cap) {
  int64_t b = (n + threads - 1) / threads;
  if (b < 1) b = 1;
  return (int)(b > cap ? cap : b);
}

// The HBM read ceiling: every 16-byte piece of buf read once with
// non-temporal loads (the weight stream's access), XOR-folded so that no
// load can be dropped, one word per workgroup into sink.  Grid-stride, each
// thread keeping 8 loads in flight.
__global__ __launch_bounds__(256) void read_kernel(const uint4 *__restrict__ buf, int64_t n16,
                                                   uint32_t *__restrict__ sink) {
  const int64_t stride = (int64_t)gridDim.x * 256 * 8;
  uint32_t acc = 0;
  for (int64_t base = (int64_t)blockIdx.x * 256 * 8 + threadIdx.x; base < n16; base += stride) {
    uint4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t i = base + (int64_t)k * 256;
      v[k] = i < n16 ? ldg16_nt((const uint8_t *)(buf + i)) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) acc ^= v[k].x ^ v[k].y ^ v[k].z ^ v[k].w;
  }
  __shared__ uint32_t red[256];
  red[threadIdx.x] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t a = 0;
    for (int i = 0; i < 256; ++i) a ^= red[i];
    sink[blockIdx.x] = a;
  }
}

hipError_t launch_read(const void *buf, int64_t nbytes, uint32_t *sink, int grid,
                       hipStream_t s, hipEvent_t start, hipEvent_t stop) {
  hipExtLaunchKernelGGL(read_kernel, dim3(grid), dim3(256), 0, s, start, stop, 0,
                        (const uint4 *)buf, nbytes / 16, sink);
  return hipGetLastError();
}

hipError_t launch_fill_i32(int32_t *p, int32_t v, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(fill_i32_kernel, dim3(blocks_for(n, 256, 4096)), dim3(256),
                     0, s, p, v, n);
  return hipGetLastError();
}

hipError_t launch_host_copy(const HostCopy &c, hipStream_t s) {
  hipLaunchKernelGGL(host_copy_kernel, dim3(1), dim3(1024), 0, s, c);
  return hipGetLastError();
}

hipError_t launch_repack(const uint8_t *img, int64_t nrows, const Layout &L,
                         int64_t stride, uint8_t *dst, hipStream_t s) {
  const int64_t ntiles = (nrows + kTileRows - 1) / kTileRows;
  hipError_t e = hipMemsetAsync(dst, 0, (size_t)(ntiles * L.tile_bytes), s);
  if (e != hipSuccess) return e;
  const int64_t ng = nrows * L.NG, nb = nrows * L.nblk;
  hipLaunchKernelGGL(repack_groups_kernel, dim3((unsigned)((ng + 255) / 256)),
                     dim3(256), 0, s, img, nrows, L, stride, dst);
  hipLaunchKernelGGL(repack_scales_kernel, dim3((unsigned)((nb + 255) / 256)),
                     dim3(256), 0, s, img, nrows, L, stride, dst);
  return hipGetLastError();
}

hipError_t launch_unpack(const uint8_t *src, int64_t nrows, const Layout &L,
                         int64_t stride, uint8_t *img, hipStream_t s) {
  hipError_t e = hipMemsetAsync(img, 0, (size_t)(nrows * stride), s);
  if (e != hipSuccess) return e;
  const int64_t ng = nrows * L.NG, nb = nrows * L.nblk;
  hipLaunchKernelGGL(unpack_groups_kernel, dim3((unsigned)((ng + 255) / 256)),
                     dim3(256), 0, s, src, nrows, L, stride, img);
  hipLaunchKernelGGL(unpack_scales_kernel, dim3((unsigned)((nb + 255) / 256)),
                     dim3(256), 0, s, src, nrows, L, stride, img);
  return hipGetLastError();
}

hipError_t launch_gemv_timed(const GemvParams &p, int grid, hipStream_t s,
                             hipEvent_t start, hipEvent_t stop) {
  const dim3 g(grid), b(kGT);
  switch (p.pro) {
    case PRO_X8:
      hipExtLaunchKernelGGL(gemv_kernel<PRO_X8>, g, b, 0, s, start, stop, 0, p);
      break;
    case PRO_DYNQ8:
      hipExtLaunchKernelGGL(gemv_kernel<PRO_DYNQ8>, g, b, 0, s, start, stop, 0, p);
      break;
    case PRO_RMSNORM_DYNQ8:
      hipExtLaunchKernelGGL(gemv_kernel<PRO_RMSNORM_DYNQ8>, g, b, 0, s, start, stop, 0, p);
      break;
    case PRO_EMUL_DYNQ8:
      hipExtLaunchKernelGGL(gemv_kernel<PRO_EMUL_DYNQ8>, g, b, 0, s, start, stop, 0, p);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gemv(const GemvParams &p, int grid, hipStream_t s) {
  switch (p.pro) {
    case PRO_X8:
      hipLaunchKernelGGL(gemv_kernel<PRO_X8>, dim3(grid), dim3(kGT), 0, s, p);
      break;
    case PRO_DYNQ8:
      hipLaunchKernelGGL(gemv_kernel<PRO_DYNQ8>, dim3(grid), dim3(kGT), 0, s, p);
      break;
    case PRO_RMSNORM_DYNQ8:
      hipLaunchKernelGGL(gemv_kernel<PRO_RMSNORM_DYNQ8>, dim3(grid), dim3(kGT), 0, s, p);
      break;
    case PRO_EMUL_DYNQ8:
      hipLaunchKernelGGL(gemv_kernel<PRO_EMUL_DYNQ8>, dim3(grid), dim3(kGT), 0, s, p);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_argmax_final(const uint64_t *partials, int n, int32_t *result,
                               hipStream_t s) {
  if (!partials || !result || n < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(argmax_final_kernel, dim3(1), dim3(kWG), 0, s, partials, n,
                     result);
  return hipGetLastError();
}

hipError_t launch_vec_prologue(const GemvParams &p, hipStream_t s) {
  if (p.pro == PRO_RMSNORM_DYNQ8)
    hipLaunchKernelGGL(vec_prologue_kernel<PRO_RMSNORM_DYNQ8>, dim3(1), dim3(kWG), 0, s, p);
  else
    hipLaunchKernelGGL(vec_prologue_kernel<PRO_DYNQ8>, dim3(1), dim3(kWG), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_rshift_round(const int64_t *v, int64_t n, int sft, int64_t *out,
                               hipStream_t s) {
  hipLaunchKernelGGL(rshift_round_kernel, dim3(blocks_for(n, 256, 4096)), dim3(256),
                     0, s, v, n, sft, out);
  return hipGetLastError();
}

hipError_t launch_movy(const int32_t *y, int64_t n, int shift, int mode, void *out,
                       hipStream_t s) {
  hipLaunchKernelGGL(movy_kernel, dim3(blocks_for(n, 256, 4096)), dim3(256), 0, s,
                     y, n, shift, mode, out);
  return hipGetLastError();
}

// MOVX (seq_model.py:929-952): the int8 values held in int16 scratch words
// src[0, n) into the engine's x window, the ragged tail of the last 4-byte
// word zeroed (SEQ_ISA B6); a value outside int8 sets bit 4 of err.
__global__ void movx_kernel(const int16_t *src, int64_t n, int64_t nb, int8_t *dst,
                            int32_t *err) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nb;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int16_t v = i < n ? src[i] : 0;
    if (v < -128 || v > 127) atomicOr(err, 16);
    dst[i] = (int8_t)v;
  }
}

hipError_t launch_movx(const int16_t *src, int64_t n, int8_t *dst, int32_t *err,
                       hipStream_t s) {
  const int64_t nb = (n + 3) & ~(int64_t)3;
  hipLaunchKernelGGL(movx_kernel, dim3(blocks_for(nb, 256, 4096)), dim3(256), 0, s, src, n,
                     nb, dst, err);
  return hipGetLastError();
}

hipError_t launch_alu(int op, const int32_t *y, const int16_t *b, int64_t n, int p0,
                      const int32_t *tables, void *out, hipStream_t s) {
  hipLaunchKernelGGL(alu_kernel, dim3(blocks_for(n, 256, 4096)), dim3(256), 0, s,
                     op, y, b, n, p0, tables, out);
  return hipGetLastError();
}

int gemv_max_blocks_per_cu() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, gemv_kernel<PRO_DYNQ8>, kGT, 0) !=
          hipSuccess || n < 1)
    n = 1;
  return n;
}

}  // namespace w4a8
