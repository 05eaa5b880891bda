// Batched quantised matmul on CDNA4 MFMA (gfx950): out[b, i] = W[i, :] . x[b, :]
// for B tokens, m rows of GGUF block-quantised weights and f32 activations.
//
// Replaces the prefill projections of vantablack's CPU prefill,
// matmulBatched (src/runtime/prefill.zig:325-378, called at :170-226):
// every weight row dequantised as dequantToF32 does
// (src/runtime/forward.zig:654-730) and dotted with each token in f32.
//
// Precision.  Each token's activations are scaled by a power of two 2^e that
// puts the token's largest |x| in [2^14, 2^15), then cut into two f16 pieces
// rounded to nearest (pre-pass vtb_xsplit): h1 = f16(x 2^e),
// h2 = f16(x 2^e - h1).  h1 + h2 holds x 2^e to 22 significant bits (to an
// absolute 2^-25 where the remainder falls below f16's normal range, i.e.
// 2^-40 of the token's largest |x|).  Weights enter as exact integers in f16,
// so products are exact and v_mfma_f32_32x32x16_f16 sums them in f32; the
// token's 2^-e comes back out exactly in the epilogue.  (Three truncated bf16
// pieces would be exact, at 3/2 the MFMA work and operand traffic: measured
// 4-16% slower over the Llama-3-8B shapes.)
//
// What the MFMAs sum, and what the VALU then does per output:
//   Q4_K, Q5_K  the integers sc * q (at most 63 * 31 = 1953, exact in f16) over
//               a whole 256-column block, T = sum sc q x, and beside them
//               T2 = sum mn * (sum of x over the sub-block), one MFMA per tile
//               (the sub-block sums, scaled by 2^-5, as two f16 pieces in the
//               two K halves).  acc += d T - 32 dmin T2: two FMAs per output
//               and 256 columns.
//   Q6_K        sc * (q - 32), up to 2^12 in magnitude, as an f16 (rounded to
//               11 bits) and the remainder, -1, 0 or 1, which only needs h1:
//               three MFMAs per step, one FMA (by d) per 256 columns.
//   Q8_0        q over a 32-column block, one FMA (by d) per 32 columns.
// Scaling sub-blocks on the VALU instead, two FMAs per output and 32 columns,
// made as many VALU cycles as MFMA cycles and held the kernel at 290-325
// TFLOP/s (4096-14336 rows, 2048-8192 tokens).
//
// Tiling.  A workgroup computes 32 TT tokens x 256 rows; its four waves own 64
// rows each (2 row tiles x TT token tiles of 32x32, D = x . W^T: lane column =
// one weight row, so a lane needs one scale per row tile).  Each weight is
// then unpacked by one wave of the workgroup only, straight into the MFMA's
// B layout: lane (row, half) unpacks the 16 + 16 columns of its half of every
// 64-column chunk, and no weight crosses lanes or LDS.  Activations go
// through LDS, shared by the four waves: the pre-pass stores them in fragment
// order, so a chunk is a linear copy of 8 KB per token tile and a fragment read
// is 64 lanes x 16 contiguous bytes.  The next chunk's activations and quants
// are loaded into registers (about 230 of the 256 that two waves per SIMD
// leave) while a chunk is computed; one barrier per chunk, which waits for LDS
// only.  (Weights as a queue of LDS DMA in each lane's own order, with the
// waits counted by hand, measured the same for Q4_K and slower for Q8_0.)
// Workgroup ids are remapped so that each XCD works through 8 x 8 squares of
// (token block, row block): what the workgroups of an XCD read at one time
// is shared eightfold in its L2.
//
// Few tokens or rows leave CUs idle, so the K range is split over `n_split`
// workgroups (whole 256-column blocks each); their f32 partials are added in
// split order by vtb_qgemm_reduce.
//
// Measured (before: 128 x 128 tiles, weights unpacked into LDS, sub-blocks
// scaled on the VALU; us per call with its pre-pass): Q4_K 14336 x 4096, 2048
// tokens 794 -> 506 (475 TFLOP/s of the reference's flops, 0.98 PFLOP/s of
// MFMA work, where a plain f16 matrix product of the library runs at
// 1.1-1.2); Q5_K 797 -> 537, Q8_0 736 -> 585, Q6_K 903 -> 720; 4096 x 4096 with 33
// tokens, Q8_0: 122 -> 21.  With the unpacking, the flush into acc or the
// staging of x taken out (timing only) Q4_K takes 471, 465 and 456 us against
// 501: no one part bounds it.
#include "common.h"

namespace vtb {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ inline float wave_max(float v) {
  v = fmaxf(v, dpp<DPP_XOR1>(v));
  v = fmaxf(v, dpp<DPP_XOR2>(v));
  v = fmaxf(v, dpp<DPP_HALF_MIRROR>(v));
  v = fmaxf(v, dpp<DPP_MIRROR>(v));
  v = xor_max<16>(v);
  return xor_max<32>(v);
}

// Activation fragments: [token tile of 32][64-column chunk][piece 2][i 4]
// [lane 64][8 halves].  Lane (t, h) of step i holds token t's columns
// 32 (i / 2) + 16 h + 8 (i % 2) + {0, 2, 1, 3, 4, 6, 5, 7} of the chunk: the
// columns whose weights the lanes of half h unpack for that step, in the
// order a masked dword yields its bytes.
constexpr int kQgChunkBytes = 8192;  // of one token tile, both pieces

// NT tokens per workgroup of 256 threads: each token's largest |x| fixes its
// power of two, then a thread splits one token's groups of 8 columns.  NT = 8
// writes whole 128-byte lines; NT = 1 spreads few tokens over more CUs.
template <int NT>
__device__ __forceinline__ void xsplit_body(const XSplitArgs& a) {
  __shared__ float s_max[4][NT];
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t0 = (int)blockIdx.x * NT;
  constexpr int TPW = NT >= 4 ? NT / 4 : 1;  // tokens per wave in the max pass
  constexpr int WPT = NT >= 4 ? 1 : 4;       // waves per token
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int tl = NT >= 4 ? wave * TPW + j : 0;
    float mx = 0.0f;
    if (t0 + tl < a.B) {
      const float* row = a.x + (size_t)(t0 + tl) * a.k;
#pragma unroll 4
      for (int c = 4 * (NT >= 4 ? lane : tid); c < a.k; c += 256 * WPT) {
        const float4 v = *reinterpret_cast<const float4*>(row + c);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
      }
    }
    mx = wave_max(mx);
    if (lane == 0) s_max[NT >= 4 ? 0 : wave][tl] = mx;
  }
  __syncthreads();
  const int tl = tid % NT, t = t0 + tl;
  float mx = s_max[0][tl];
  if constexpr (NT < 4) mx = fmaxf(fmaxf(mx, s_max[1][tl]), fmaxf(s_max[2][tl], s_max[3][tl]));
  // 2^e with mx 2^e in [2^14, 2^15); e clamped so that 2^e and 2^-e stay
  // normal f32 (a row that small is then scaled less, not wrongly).
  int e = mx > 0.0f ? 14 - ilogbf(mx) : 0;
  e = e > 100 ? 100 : (e < -100 ? -100 : e);
  const float scale = ldexpf(1.0f, e);
  if (tid < NT) a.inv_scale[t] = ldexpf(1.0f, -e);
  const bool live = t < a.B;
  const float* row = a.x + (size_t)t * a.k;
  const int n64 = (a.k + 63) >> 6, n256 = (a.k + 255) >> 8;
  uint8_t* dst = reinterpret_cast<uint8_t*>(a.planes) + (size_t)(t >> 5) * n64 * kQgChunkBytes + 16 * (t & 31);
  uint16_t* sdst = a.sums + (size_t)(t >> 5) * n256 * 512 + 8 * (t & 31);
  // Groups of 8 columns, padded to whole 256-column blocks so that every lane
  // runs the same trips (the sums below are taken across lanes).
  for (int g = tid / NT; g < 32 * n256; g += 256 / NT) {
    const int c = 8 * g;
    float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (live && c < a.k) {
      const float4 q0 = *reinterpret_cast<const float4*>(row + c), q1 = *reinterpret_cast<const float4*>(row + c + 4);
      v[0] = q0.x, v[1] = q0.z, v[2] = q0.y, v[3] = q0.w;
      v[4] = q1.x, v[5] = q1.z, v[6] = q1.y, v[7] = q1.w;
    }
    uint32_t w1[4], w2[4];
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float xs = v[j] * scale;  // exact (power of two)
      sum += xs;
      const _Float16 h1 = (_Float16)xs;                 // round to nearest even
      const _Float16 h2 = (_Float16)(xs - (float)h1);  // the difference is exact in f32
      const uint32_t b1 = __builtin_bit_cast(uint16_t, h1), b2 = __builtin_bit_cast(uint16_t, h2);
      if (j & 1) {
        w1[j >> 1] |= b1 << 16;
        w2[j >> 1] |= b2 << 16;
      } else {
        w1[j >> 1] = b1;
        w2[j >> 1] = b2;
      }
    }
    const int q = g & 7;  // 8-column group of the chunk
    if ((g >> 3) < n64) {
      uint8_t* d = dst + (size_t)(g >> 3) * kQgChunkBytes + 1024 * (2 * (q >> 2) + (q & 1)) + 512 * ((q >> 1) & 1);
      *reinterpret_cast<uint4*>(d) = make_uint4(w1[0], w1[1], w1[2], w1[3]);
      *reinterpret_cast<uint4*>(d + 4096) = make_uint4(w2[0], w2[1], w2[2], w2[3]);
    }
    // Sums of 32 columns (4 groups, NT lanes apart), scaled by 2^-5 into f16's
    // range, as two pieces: half 0's and half 1's K rows of the min MFMA.
    float s32 = sum;
    if constexpr (NT == 8) {
      s32 = xor_sum<16>(xor_sum<8>(s32));
    } else {
      s32 += dpp<DPP_XOR1>(s32);
      s32 += dpp<DPP_XOR2>(s32);
    }
    if ((g & 3) == 0) {
      s32 *= 0.03125f;
      const _Float16 h1 = (_Float16)s32, h2 = (_Float16)(s32 - (float)h1);
      uint16_t* d = sdst + (size_t)(g >> 5) * 512 + ((g >> 2) & 7);
      d[0] = __builtin_bit_cast(uint16_t, h1);
      d[256] = __builtin_bit_cast(uint16_t, h2);
    }
  }
}

__device__ inline uint32_t qperm(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }
__device__ inline float qh_lo(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(v & 0xffffu)); }
__device__ inline float qh_hi(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16)); }
__device__ inline f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ inline uint32_t as_u(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ inline f16x2 splat_h2(float v) { return f16x2{(_Float16)v, (_Float16)v}; }
__device__ inline f16x2 pk_fma(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ inline f16x8 frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_bit_cast(f16x8, u32x4{a, b, c, d});
}
// Lanes 32..63 of x and lanes 0..31 of y change places (v_permlane32_swap; the
// s_nop as in xchg32).  Every lane of the wave must be active.
__device__ inline void swap32(uint32_t& x, uint32_t& y) {
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "+v"(y));
}
// Bytes (0, 2) and (1, 3) of u over 0x64: the f16 pairs 1024 + byte.
constexpr uint32_t kK64 = 0x64646464u;
__device__ inline uint32_t pair02(uint32_t u) { return qperm(kK64, u, 0x04020400u); }
__device__ inline uint32_t pair13(uint32_t u) { return qperm(kK64, u, 0x04030401u); }

// Four dwords / one dword of a raw buffer (zeros past its end).
__device__ inline u32x4 load4(__amdgpu_buffer_rsrc_t r, int voff, int soff = 0) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ inline uint32_t load1(__amdgpu_buffer_rsrc_t r, int voff, int soff = 0) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}
// This wave's LDS operations are done, and every wave of the workgroup says
// the same.  Not __syncthreads: loads of the next chunks stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

enum { QG8_0 = 0, QG4_K = 1, QG5_K = 2, QG6_K = 3 };
constexpr int kQgRows = 256;  // rows per workgroup, 64 per wave

// Per format: what a lane loads of one row, and how it turns that into B
// fragments.
//   WU    chunks per load of quants (Next: as loaded; Raw: ready to unpack)
// Fields of Q8_0 and Q6_K are 2-byte aligned: they are read as the aligned
// dwords that cover them (16 + 4 bytes) and realigned by v_perm.
template <int KIND> struct Qf;

// The eight 6-bit scales and mins of a block as bytes (simd.zig:211-219).
__device__ inline void k45_scales(const uint32_t (&h)[4], uint32_t (&sc)[2], uint32_t (&mn)[2]) {
  sc[0] = h[1] & 0x3F3F3F3Fu;
  mn[0] = h[2] & 0x3F3F3F3Fu;
  sc[1] = (h[3] & 0x0F0F0F0Fu) | ((h[1] >> 2) & 0x30303030u);
  mn[1] = ((h[3] >> 4) & 0x0F0F0F0Fu) | ((h[2] >> 2) & 0x30303030u);
}

// simd.zig:192-243 (Q4_K), 275-317 (Q5_K).  Chunk j of a block holds
// sub-blocks 2j (low nibbles of qs[32 j + l]) and 2j + 1 (high nibbles); lane
// half h unpacks l = 16 h + [0, 16).  Q5_K adds bit 2j (2j + 1) of qh[l].
template <bool FIVE> struct QfK45 {
  static constexpr int BE = 256, BB = FIVE ? 176 : 144, WU = 1;
  struct NextHead {
    u32x4 h, qh;
  };
  struct Head {
    uint32_t h[4], qh[FIVE ? 4 : 1];
    uint32_t sc[2], mn[2];
  };
  struct Next {
    u32x4 q;
  };
  struct Raw {
    uint32_t q[4];
  };
  __device__ static void load_head(__amdgpu_buffer_rsrc_t r, int off, int half, NextHead& n) {
    n.h = load4(r, off);
    if constexpr (FIVE) n.qh = load4(r, off + 16 + 16 * half);
  }
  __device__ static void load_raw(__amdgpu_buffer_rsrc_t r, int off, int j, int half, Next& n) {
    n.q = load4(r, off + (FIVE ? 48 : 16) + 32 * j + 16 * half);
  }
  __device__ static void head(const NextHead& n, int, Head& hd) {
    hd.h[0] = n.h.x, hd.h[1] = n.h.y, hd.h[2] = n.h.z, hd.h[3] = n.h.w;
    if constexpr (FIVE) hd.qh[0] = n.qh.x, hd.qh[1] = n.qh.y, hd.qh[2] = n.qh.z, hd.qh[3] = n.qh.w;
    k45_scales(hd.h, hd.sc, hd.mn);
  }
  __device__ static void raw(const Next& n, const Head&, int, Raw& raw) {
    raw.q[0] = n.q.x, raw.q[1] = n.q.y, raw.q[2] = n.q.z, raw.q[3] = n.q.w;
  }
  // The scale operands of sub-block 2j + hi: sc, and -(bias + centre) sc.
  struct Sc {
    f16x2 a, b;
  };
  __device__ static Sc scales(const Head& hd, int j, int hi) {
    const int s = 2 * j + hi;
    const uint32_t sel = 0x04000400u + 0x00010001u * (s & 3);
    Sc o;
    o.a = as_h2(qperm(kK64, hd.sc[s >> 2], sel)) - splat_h2(1024.0f);
    o.b = o.a * splat_h2(FIVE ? -144.0f : -72.0f);  // 9 sc 2^3 or 2^4: exact
    return o;
  }
  // sc (q - centre).  A quant in the top mantissa bits of an f16 whose ulp
  // there is 1 is bias + q: Q4_K bits 4..7 under 0x5400 (64 + q), Q5_K bits
  // 3..7 under 0x5800 (128 + q).
  __device__ static f16x8 unpack(const Raw& raw, const Head& hd, const Sc& sc, int j, int i, uint32_t m, uint32_t bias) {
    const int hi = i >> 1;
    uint32_t p[4];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const uint32_t v = raw.q[2 * (i & 1) + d];
      if constexpr (FIVE) {
        const int s = 2 * j + hi;
        const uint32_t u = ((hi ? v >> 1 : v << 3) & 0x78787878u) |
                           ((hd.qh[2 * (i & 1) + d] << (7 - s)) & 0x80808080u);
        p[2 * d] = qperm(0x58585858u, u, 0x04020400u);
        p[2 * d + 1] = qperm(0x58585858u, u, 0x04030401u);
      } else {
        p[2 * d] = ((hi ? v : v << 4) & m) | bias;
        p[2 * d + 1] = ((hi ? v >> 8 : v >> 4) & m) | bias;
      }
    }
    return frag(as_u(pk_fma(as_h2(p[0]), sc.a, sc.b)), as_u(pk_fma(as_h2(p[1]), sc.a, sc.b)),
                as_u(pk_fma(as_h2(p[2]), sc.a, sc.b)), as_u(pk_fma(as_h2(p[3]), sc.a, sc.b)));
  }
  static constexpr float CENTRE = FIVE ? 16.0f : 8.0f;
  // Eight bytes (the block's scales or mins) as a fragment, both K halves alike.
  __device__ static f16x8 bytes8(const uint32_t (&b)[2]) {
    uint32_t p[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t u = qperm(kK64, b[d >> 1], (d & 1) ? 0x04030402u : 0x04010400u);
      p[d] = as_u(as_h2(u) - splat_h2(1024.0f));
    }
    return frag(p[0], p[1], p[2], p[3]);
  }
};
template <> struct Qf<QG4_K> : QfK45<false> {};
template <> struct Qf<QG5_K> : QfK45<true> {};

// simd.zig:349-404.  Chunk j = 2 hb + jj of a block holds quadrants 2 jj and
// 2 jj + 1 of half hb: quadrant qd's weight l is nibble qd / 2 of
// ql[64 hb + 32 (qd % 2) + l] | bits 2qd..2qd+1 of qh[32 hb + l] << 4, minus 32,
// scaled by d * sc[8 hb + l / 16 + 2 qd].  A lane loads the three 16-byte
// fields of a half at once.
template <> struct Qf<QG6_K> {
  static constexpr int BE = 256, BB = 210, WU = 2;
  struct NextHead {
    u32x4 sc;
    uint32_t d;
  };
  struct Head {
    uint32_t sc[4];    // bytes + 128
    uint32_t d;        // f16 bits
    uint32_t realign;  // v_perm selector of this block
  };
  struct Next {
    u32x4 q[3];
    uint32_t t[3];
  };
  struct Raw {
    uint32_t ql[2][4], qh[4];
  };
  __device__ static void load_head(__amdgpu_buffer_rsrc_t r, int off, int, NextHead& n) {
    n.sc = load4(r, (off & ~3) + 192);
    n.d = load1(r, (off & ~3) + 208);
  }
  __device__ static void load_raw(__amdgpu_buffer_rsrc_t r, int off, int j, int half, Next& n) {
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      const int o = (off & ~3) + (f < 2 ? 64 * (j >> 1) + 32 * f : 128 + 32 * (j >> 1)) + 16 * half;
      n.q[f] = load4(r, o);
      n.t[f] = load1(r, o + 16);
    }
  }
  __device__ static void head(const NextHead& n, int off, Head& hd) {
    const bool sh = (off & 2) != 0;
    const uint32_t w[5] = {n.sc.x, n.sc.y, n.sc.z, n.sc.w, n.d};
    hd.realign = sh ? 0x05040302u : 0x03020100u;
#pragma unroll
    for (int i = 0; i < 4; ++i) hd.sc[i] = qperm(w[i + 1], w[i], hd.realign) ^ 0x80808080u;
    hd.d = n.d >> (sh ? 16 : 0);
  }
  __device__ static void raw(const Next& n, const Head& hd, int, Raw& raw) {
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      const uint32_t w[5] = {n.q[f].x, n.q[f].y, n.q[f].z, n.q[f].w, n.t[f]};
#pragma unroll
      for (int i = 0; i < 4; ++i) (f < 2 ? raw.ql[f & 1][i] : raw.qh[i]) = qperm(w[i + 1], w[i], hd.realign);
    }
  }
  // sc of the lane's 16-column group: byte 2 (qd % 2) + half of its dword.
  __device__ static f16x2 scales(const Head& hd, int j, int hi, int half) {
    const int qd = 2 * (j & 1) + hi;
    const uint32_t sel = 0x04000400u + 0x00010001u * (uint32_t)(2 * (qd & 1) + half);
    return as_h2(qperm(kK64, hd.sc[2 * (j >> 1) + (qd >> 1)], sel)) - splat_h2(1152.0f);
  }
  __device__ static void unpack(const Raw& raw, f16x2 sc, int j, int i, f16x8& hi_o, f16x8& lo_o) {
    const int w = i >> 1, qd = 2 * (j & 1) + w;
    uint32_t a[4], b[4];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const int n = 2 * (i & 1) + d;
      const uint32_t u = ((raw.ql[w][n] >> (4 * (qd >> 1))) & 0x0F0F0F0Fu) |
                         (((raw.qh[n] >> (2 * qd)) & 0x03030303u) << 4);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const f16x2 q = as_h2(s ? pair13(u) : pair02(u)) - splat_h2(1056.0f);
        const f16x2 p = q * sc;  // rounded to 11 bits
        a[2 * d + s] = as_u(p);
        b[2 * d + s] = as_u(pk_fma(q, sc, -p));  // -1, 0 or 1
      }
    }
    hi_o = frag(a[0], a[1], a[2], a[3]);
    lo_o = frag(b[0], b[1], b[2], b[3]);
  }
};

// simd.zig:145-157.  A chunk is two 34-byte blocks.  Lane half h loads block h
// whole (nine aligned dwords) and the halves then swap: half h unpacks
// qs[16 h, 16 h + 16) of each.
template <> struct Qf<QG8_0> {
  static constexpr int BE = 32, BB = 8 * 34, WU = 1;  // BB: 256 columns, as for the others
  struct NextHead {};
  struct Head {};
  struct Next {
    u32x4 q[2];
    uint32_t t;
  };
  struct Raw {
    uint32_t q[2][4];  // bytes + 128
    uint32_t d[2];     // f16 bits
  };
  __device__ static void load_head(__amdgpu_buffer_rsrc_t, int, int, NextHead&) {}
  __device__ static void head(const NextHead&, int, Head&) {}
  __device__ static void load_raw(__amdgpu_buffer_rsrc_t r, int off, int j, int half, Next& n) {
    const int o = (off + (2 * j + half) * 34) & ~3;
    n.q[0] = load4(r, o);
    n.q[1] = load4(r, o + 16);
    n.t = load1(r, o + 32);
  }
  // off: the lane's block.
  __device__ static void raw(const Next& n, const Head&, int off, Raw& raw) {
    const uint32_t w[9] = {n.q[0].x, n.q[0].y, n.q[0].z, n.q[0].w, n.q[1].x, n.q[1].y, n.q[1].z, n.q[1].w, n.t};
    const bool sh = (off & 2) != 0;
    // qs starts 2 bytes into w[0], or with w[1]
    const uint32_t sel = sh ? 0x07060504u : 0x05040302u;
    uint32_t d0 = sh ? w[0] >> 16 : w[0], d1 = d0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t lo = qperm(w[i + 1], w[i], sel) ^ 0x80808080u, hi = qperm(w[i + 5], w[i + 4], sel) ^ 0x80808080u;
      // lo: block h's first half in lanes of half h; hi: its second half
      swap32(lo, hi);
      raw.q[0][i] = lo;
      raw.q[1][i] = hi;
    }
    swap32(d0, d1);
    raw.d[0] = d0 & 0xffffu;
    raw.d[1] = d1 & 0xffffu;
  }
  __device__ static f16x8 unpack(const Raw& raw, int i) {
    uint32_t p[4];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const uint32_t u = raw.q[i >> 1][2 * (i & 1) + d];
      p[2 * d] = as_u(as_h2(pair02(u)) - splat_h2(1152.0f));
      p[2 * d + 1] = as_u(as_h2(pair13(u)) - splat_h2(1152.0f));
    }
    return frag(p[0], p[1], p[2], p[3]);
  }
};

__device__ inline f32x16 mfma(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ inline f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.0f;
  return z;
}

template <int KIND, int TT>
__device__ __forceinline__ void qgemm_body(const QGemmArgs& a) {
  using F = Qf<KIND>;
  constexpr bool K45 = KIND == QG4_K || KIND == QG5_K;
  constexpr int XB = TT * kQgChunkBytes;  // one activation slot
  constexpr int NX = 2 * TT;              // its 16-byte pieces per thread
  __shared__ __attribute__((aligned(16))) uint8_t s_x[2][XB];

  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fl = lane & 31, half = lane >> 5;

  // Workgroup -> (split, row block, token block): each XCD (consecutive ids go
  // to different XCDs) takes a contiguous range of the list, in which 8 row
  // blocks advance over the token blocks together.
  const int total = a.n_rb * a.n_tb * a.n_split;
  const int per = total >> 3;
  int wi = (int)blockIdx.x;
  if (wi < 8 * per) wi = (wi & 7) * per + (wi >> 3);
  const int split = wi / (a.n_rb * a.n_tb);
  wi -= split * a.n_rb * a.n_tb;
  const int rg = wi / (8 * a.n_tb);
  wi -= rg * 8 * a.n_tb;
  const int gw = a.n_rb - 8 * rg < 8 ? a.n_rb - 8 * rg : 8;
  const int tb = wi / gw, rb = 8 * rg + wi % gw;
  const int tok0 = 32 * TT * tb, row0 = kQgRows * rb + 64 * wave;

  // This split's chunks [c_lo, c_hi).
  const int n64 = (a.k + 63) >> 6, n256 = (a.k + 255) >> 8;
  const int b_lo = split * a.split_blocks;
  const int b_hi = b_lo + a.split_blocks < n256 ? b_lo + a.split_blocks : n256;
  const int c_lo = 4 * b_lo, c_hi = 4 * b_hi < n64 ? 4 * b_hi : n64;

  const auto wr = buffer_rsrc(a.w, a.w_bytes);
  const size_t tile_bytes = (size_t)n64 * kQgChunkBytes;
  const auto xr = buffer_rsrc(reinterpret_cast<const uint8_t*>(a.planes) + (size_t)(tok0 >> 5) * tile_bytes,
                              (unsigned)(TT * tile_bytes));
  const auto sr = buffer_rsrc(a.sums + (size_t)(tok0 >> 5) * n256 * 512, (unsigned)(TT * n256 * 1024));
  // Rows past m read zeros from the end of the range.
  int ro[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) ro[rt] = row0 + 32 * rt + fl < a.m ? (row0 + 32 * rt + fl) * a.row_bytes : (int)a.w_bytes;

  // The next chunk's activations, the next quants and block header.  Chunks
  // past the range load its last one again, unused.
  u32x4 xn[NX];
  auto load_x = [&](int c) __attribute__((always_inline)) {
    const int cc = c < c_hi ? c : c_hi - 1;
#pragma unroll
    for (int n = 0; n < NX; ++n)
      xn[n] = load4(xr, 16 * tid, (int)((n >> 1) * tile_bytes) + cc * kQgChunkBytes + 4096 * (n & 1));
  };
  auto store_x = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NX; ++n) *reinterpret_cast<u32x4*>(&s_x[0][0] + slot * XB + 4096 * n + 16 * tid) = xn[n];
  };
  typename F::Next wn[2];
  auto load_w = [&](int c) __attribute__((always_inline)) {
    const int cc = c < c_hi ? c : c_hi - 1;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) F::load_raw(wr, ro[rt] + (cc >> 2) * F::BB, cc & 3, half, wn[rt]);
  };
  typename F::NextHead hn[2];
  auto load_head = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) F::load_head(wr, ro[rt] + (blk < b_hi ? blk : b_hi - 1) * F::BB, half, hn[rt]);
  };

  f32x16 acc[TT][2];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) acc[tt][rt] = zero16();

  auto xfrag = [&](int slot, int tt, int p, int i) __attribute__((always_inline)) {
    return *reinterpret_cast<const f16x8*>(&s_x[0][0] + slot * XB + 8192 * tt + 4096 * p + 1024 * i + 16 * lane);
  };

  // Q4_K's mask and bias, one in an SGPR and one in a VGPR and out of the
  // compiler's sight: as literals they make two instructions of every and-or
  // (14336 x 4096, 2048 tokens: 514 us, 506 so).
  uint32_t k_mask = 0x00F000F0u, k_bias = 0x54005400u;
  asm("" : "+s"(k_mask));
  asm("" : "+v"(k_bias));

  load_x(c_lo);
  load_head(b_lo);
  load_w(c_lo);
  store_x(0);
  lds_barrier();
  for (int blk = b_lo; blk < b_hi; ++blk) {
    typename F::Head hd[2];
    typename F::Raw raw[2];
    f32x16 T[TT][2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 4 * blk + j;
      if (KIND == QG8_0 && c >= c_hi) break;  // k ends inside a block of 256
      const int xs = j & 1;  // a block starts with an even chunk
      load_x(c + 1);
      if (j == 0) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) F::head(hn[rt], ro[rt] + blk * F::BB, hd[rt]);
        load_head(blk + 1);
      }
      if (j % F::WU == 0) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
          F::raw(wn[rt], hd[rt], ro[rt] + blk * F::BB + (KIND == QG8_0 ? (2 * j + half) * 34 : 0), raw[rt]);
        if constexpr (F::WU == 1) load_w(c + 1);
      }
      if constexpr (F::WU == 2)
        if (j % 2 == 1) load_w(c + 1);  // (a step earlier it spills)
      __builtin_amdgcn_sched_barrier(0);  // (the scheduler would sink the loads to their use)
      if constexpr (KIND == QG8_0) {
        // T per block of 32 columns; one token tile's FMAs run beside the next
        // one's MFMAs
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          f16x8 w[2][2];
          float d[2];
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) {
            // k may end in half a chunk: what follows it has no columns
            d[rt] = b == 0 || 64 * c + 32 < a.k ? qh_lo(raw[rt].d[b]) : 0.0f;
#pragma unroll
            for (int i = 0; i < 2; ++i) w[rt][i] = F::unpack(raw[rt], 2 * b + i);
          }
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) {
            f32x16 U[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
              for (int p = 0; p < 2; ++p) {
                const f16x8 x = xfrag(xs, tt, p, 2 * b + i);
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) U[rt] = mfma(x, w[rt][i], i == 0 && p == 0 ? zero16() : U[rt]);
              }
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
              for (int e = 0; e < 16; ++e) acc[tt][rt][e] = fmaf(d[rt], U[rt][e], acc[tt][rt][e]);
          }
        }
      } else {
      // T starts anew with each block of 256 columns (K45) or 128 (Q6_K).
      constexpr int kTSteps = K45 ? 4 : 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f16x8 w[2], wl[2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          if constexpr (KIND == QG6_K)
            F::unpack(raw[rt], F::scales(hd[rt], j, i >> 1, half), j, i, w[rt], wl[rt]);
          else
            w[rt] = F::unpack(raw[rt], hd[rt], F::scales(hd[rt], j, i >> 1), j, i, k_mask, k_bias);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) {
            const f16x8 x = xfrag(xs, tt, p, i);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
              T[tt][rt] = mfma(x, w[rt], i == 0 && j % kTSteps == 0 && p == 0 ? zero16() : T[tt][rt]);
              if constexpr (!K45)
                if (p == 0) T[tt][rt] = mfma(x, wl[rt], T[tt][rt]);
            }
          }
      }
      if (j % kTSteps == kTSteps - 1) {
        __builtin_amdgcn_sched_barrier(0);  // (keeps the Q4_K and Q5_K bodies out of scratch)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          if constexpr (K45) {
            // acc += d T + 32 centre d sum(sc S) - 32 dmin sum(mn S), S the
            // sub-block sums of x 2^-5
            const float d = qh_lo(hd[rt].h[0]), dc = 32.0f * F::CENTRE * d, dm = -32.0f * qh_hi(hd[rt].h[0]);
            const f16x8 sc = F::bytes8(hd[rt].sc), mn = F::bytes8(hd[rt].mn);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
              const f16x8 sx = __builtin_bit_cast(f16x8, load4(sr, 16 * lane, (tt * n256 + blk) * 1024));
              const f32x16 C1 = mfma(sx, sc, zero16()), C2 = mfma(sx, mn, zero16());
#pragma unroll
              for (int e = 0; e < 16; ++e)
                acc[tt][rt][e] = fmaf(d, T[tt][rt][e], fmaf(dc, C1[e], fmaf(dm, C2[e], acc[tt][rt][e])));
            }
          } else {
            const float d = qh_lo(hd[rt].d);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
              for (int e = 0; e < 16; ++e) acc[tt][rt][e] = fmaf(d, T[tt][rt][e], acc[tt][rt][e]);
          }
        }
      }
      }
      store_x(xs ^ 1);
      lds_barrier();
    }
  }

  // out[token][row], or this workgroup's partial [token][256 rows]: lanes
  // 0..31 of one register hold 32 consecutive rows of one token.
  const bool whole = a.n_split == 1;
  float* out = whole ? a.out + (size_t)tok0 * a.m + row0
                     : a.part + ((size_t)(split * a.n_tb + tb) * a.n_rb + rb) * (32 * TT * kQgRows) + 64 * wave;
  const size_t ld = whole ? (size_t)a.m : (size_t)kQgRows;
  // (every load is back and every product formed before the first store, also
  // where the compiler would sink them into the store's branch: the wait for
  // a load would there wait for the stores before it)
  float inv[TT][16];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(a.inv_scale + tok0 + 32 * tt + 8 * q + 4 * half);
      inv[tt][4 * q] = v.x, inv[tt][4 * q + 1] = v.y, inv[tt][4 * q + 2] = v.z, inv[tt][4 * q + 3] = v.w;
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float v = acc[tt][rt][e] * inv[tt][e];
        asm volatile("" : "+v"(v));
        acc[tt][rt][e] = v;
      }
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int row = 32 * rt + fl;
    if (row0 + row < a.m) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int tok = 32 * tt + 8 * (e >> 2) + 4 * half + (e & 3);
          if (tok0 + tok < a.B) out[(size_t)tok * ld + row] = acc[tt][rt][e];
        }
    }
  }
}

}  // namespace vtb

extern "C" __global__ __launch_bounds__(256) void vtb_xsplit(vtb::XSplitArgs a) { vtb::xsplit_body<8>(a); }
extern "C" __global__ __launch_bounds__(256) void vtb_xsplit_1(vtb::XSplitArgs a) { vtb::xsplit_body<1>(a); }

// out = the n_split partials of each output, added in split order.  One wave
// per token and row block, four rows per lane; a tile's rows past m were not
// written: they are read with the others and not stored.
extern "C" __global__ __launch_bounds__(256) void vtb_qgemm_reduce(vtb::QReduceArgs a) {
  const int lane = (int)threadIdx.x & 63, tok = 4 * (int)blockIdx.y + ((int)threadIdx.x >> 6), rb = (int)blockIdx.x;
  const int row = vtb::kQgRows * rb + 4 * lane;
  if (tok >= a.B || row >= a.m) return;
  const int tb = tok / a.tile_tokens;
  const size_t tile = (size_t)a.tile_tokens * vtb::kQgRows;
  const float* p = a.part + ((size_t)tb * a.n_rb + rb) * tile + (size_t)(tok - tb * a.tile_tokens) * vtb::kQgRows + 4 * lane;
  float* o = a.out + (size_t)tok * a.m + row;
  const size_t step = (size_t)a.n_tb * a.n_rb * tile;
  // Eight partials in flight; past the last one it is read again and not added.
  // (One after the other, and the last rows of m % 4 on their own, 4096 x 4096
  // with 33 tokens took 1.6 us more per call, 374 x 9216 with 40 12.)
  float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int s0 = 0; s0 < a.n_split; s0 += 8) {
    float4 u[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      u[i] = *reinterpret_cast<const float4*>(p + (size_t)(s0 + i < a.n_split ? s0 + i : a.n_split - 1) * step);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s0 + i < a.n_split) v = make_float4(v.x + u[i].x, v.y + u[i].y, v.z + u[i].z, v.w + u[i].w);
  }
  const float r[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (row + e < a.m) o[e] = r[e];
}

// Two workgroups per CU (at most 256 registers per lane).
#define VTB_QGEMM(NAME, KIND)                                                                       \
  extern "C" __global__ __launch_bounds__(256, 2) void vtb_qgemm_##NAME##_t64(vtb::QGemmArgs a) { \
    vtb::qgemm_body<vtb::KIND, 2>(a);                                                              \
  }                                                                                                \
  extern "C" __global__ __launch_bounds__(256, 2) void vtb_qgemm_##NAME##_t32(vtb::QGemmArgs a) { \
    vtb::qgemm_body<vtb::KIND, 1>(a);                                                              \
  }
VTB_QGEMM(q8_0, QG8_0)
VTB_QGEMM(q4_k, QG4_K)
VTB_QGEMM(q5_k, QG5_K)
VTB_QGEMM(q6_k, QG6_K)
