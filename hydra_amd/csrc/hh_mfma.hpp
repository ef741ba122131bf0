// hh_mfma.hpp — device code shared by the expert products' translation units (hh_gemm.hip and
// hh_gemm_block.hip, hh_prefill.hip): weight formats, the canonical arithmetic of one chunk, epilogue values, and the
// task order and direct-to-LDS loads of the prefill kernels.
#pragma once
#include "hh_common.hpp"

#include <type_traits>

namespace hh {

enum { PH_UP = 0, PH_DOWN = 1 };

__device__ __forceinline__ f32x4 mfma(const bf16x8 &a, const bf16x8 &b, const f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Two unsigned integers < 256 → packed bf16 pair (exact: 8 significant bits).
__device__ __forceinline__ uint32_t u8pair_to_bf16x2(uint32_t lo, uint32_t hi) {
  const uint32_t a = __float_as_uint((float)lo), b = __float_as_uint((float)hi);
  return __builtin_amdgcn_perm(b, a, 0x07060302u);   // the upper halves
}

// 8 8-bit MLX values of two words → bf16 integers.
__device__ __forceinline__ bf16x8 mlx8_to_bf16(uint32_t w0, uint32_t w1) {
  u32x4 r = {u8pair_to_bf16x2(w0 & 0xFF, (w0 >> 8) & 0xFF),
             u8pair_to_bf16x2((w0 >> 16) & 0xFF, w0 >> 24),
             u8pair_to_bf16x2(w1 & 0xFF, (w1 >> 8) & 0xFF),
             u8pair_to_bf16x2((w1 >> 16) & 0xFF, w1 >> 24)};
  return as_bf16x8(r);
}

template <int FMT> struct Fmt;

// ---- MXFP4 blocks without their scales (decode kernels stage a tile's scales in LDS): 128-column
// chunks, one 16-byte block per lane
constexpr int Q_MXFP4_W = 4;
// Rows are read through a buffer resource over the whole weight matrix of the expert: the lane's
// row offset is computed once and a chunk's offset (64 bytes per chunk) goes into the
// instruction's immediate field, so a stream of chunks costs no address registers. Chunks are
// not clamped: a lane past K reads the next row (its weights are zeroed by lane_valid) and reads
// past the matrix return zeros. Streams of this format walk K with stride 1.
template <> struct Fmt<Q_MXFP4_W> {
  static constexpr int CHUNK = 128, NB = 4;
  struct A { u32x4 w; };
  struct Row {
    __amdgpu_buffer_rsrc_t rs;
    int voff;   // row · K/2 + 16·(lane group): the lane's block of chunk 0
  };
  __device__ static Row row(const uint8_t *matrix, uint64_t bytes, int r, int K) {
    Row rw;
    rw.rs = __builtin_amdgcn_make_buffer_rsrc((void *)matrix, (short)0, (int)bytes, 0x00020000);
    rw.voff = r * (K / 2) + 16 * ((threadIdx.x & 63) >> 4);
    return rw;
  }
  __device__ static void load(A &a, const Row &rw, int c, int, int) {
    a.w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw.rs, rw.voff + 64 * c, 0, 0));
  }
  __device__ static bool lane_valid(int c, int g, int K) { return 128 * c + 32 * g < K; }
};

// ---- BF16: 128-column chunks; step v (32 columns) of a chunk holds, in lane (g, l16), row l16's
// columns 128c + 32v + 8g .. +7: a lane's four 16-byte pieces lie 64 bytes apart, so a load of
// one step reads 64 contiguous bytes of each of 16 rows. K is a multiple of 64: a step lies wholly
// inside or wholly past K, and steps past K are skipped (uniformly) by every kernel.
template <> struct Fmt<Q_BF16> {
  static constexpr int CHUNK = 128, NB = 4, VS = 32;   // VS: B columns between steps
  struct A { u32x4 w[4]; };
  struct Row { const uint8_t *w; };
  __device__ static Row row(const uint8_t *base, int r, int K) { return {base + (size_t)r * K * 2}; }
  __device__ static void load(A &a, const Row &rw, int c, int g, int K) {
#pragma unroll
    for (int s = 0; s < 4; ++s) a.w[s] = *(const u32x4 *)(rw.w + 2 * min(128 * c + 32 * s + 8 * g, K - 8));
  }
  __device__ static int bcol(int c, int g, int) { return 128 * c + 8 * g; }
  __device__ static bool step_ok(int c, int v, int K) { return 128 * c + 32 * v < K; }
};

// ---- MLX affine: 64-column chunks (one group) ------------------------------------------------
// The lane's stage also carries its row's group scale and bias (bf16 pair); the D rows' values
// are fetched from the lanes of those rows by shuffle (affine_sb).
template <int BITS> struct FmtMLX {
  static constexpr int CHUNK = 64, NB = 2, VS = 8;
  struct A { uint32_t w[BITS / 2]; uint32_t sb; };  // 4-bit: 2 words (16 values); 8-bit: 4 words
  struct Row { const uint8_t *w; const uint16_t *sc, *bi; };
  __device__ static Row row(const uint8_t *words, const uint8_t *scales, const uint8_t *biases,
                            int r, int K) {
    return {words + (size_t)r * (K * BITS / 8), (const uint16_t *)scales + (size_t)r * (K / 64),
            (const uint16_t *)biases + (size_t)r * (K / 64)};
  }
  __device__ static void load(A &a, const Row &rw, int c, int g, int K) {
    const uint8_t *p = rw.w + (64 * c + 16 * g) * BITS / 8;
    if constexpr (BITS == 4) {
      u32x2 v = *(const u32x2 *)p;
      a.w[0] = v[0]; a.w[1] = v[1];
    } else {
      u32x4 v = *(const u32x4 *)p;
      a.w[0] = v[0]; a.w[1] = v[1]; a.w[2] = v[2]; a.w[3] = v[3];
    }
    a.sb = (uint32_t)rw.sc[c] | ((uint32_t)rw.bi[c] << 16);
  }
  // The codes only (the group's scale and bias come from elsewhere: MlxSb).
  __device__ static void load_w(A &a, const Row &rw, int c, int g, int K) {
    const uint8_t *p = rw.w + (64 * c + 16 * g) * BITS / 8;
    if constexpr (BITS == 4) {
      u32x2 v = *(const u32x2 *)p;
      a.w[0] = v[0]; a.w[1] = v[1];
    } else {
      u32x4 v = *(const u32x4 *)p;
      a.w[0] = v[0]; a.w[1] = v[1]; a.w[2] = v[2]; a.w[3] = v[3];
    }
    a.sb = 0u;
  }
  __device__ static int bcol(int c, int g, int) { return 64 * c + 16 * g; }
};
template <> struct Fmt<Q_MLX4> : FmtMLX<4> {};
template <> struct Fmt<Q_MLX8> : FmtMLX<8> {};

template <int FMT> constexpr bool is_mlx() { return FMT == Q_MLX4 || FMT == Q_MLX8; }

// ---- shared pieces of the canonical arithmetic -------------------------------------------------

// One 16-row A tile of a wave: the lane's weight row.
template <int FMT> struct ATile {
  typename Fmt<FMT>::Row row;
};

// One 16-row A tile: output rows r0 .. r0+15 (lane l16 takes r0 + l16); PH_UP picks the gate
// (is_up false) or the up matrix.
template <int PH, int FMT>
__device__ __forceinline__ ATile<FMT> tile_of(const uint8_t *blob, const ExpertGroup &grp, int r0, bool is_up,
                                              int K, int l16) {
  ATile<FMT> t;
  const int orow = r0 + l16;
  const int I = grp.inter;
  if constexpr (FMT == Q_MXFP4_W) {
    // GPT-OSS gate_up rows interleave gate and up (ReferenceLayer.swift:11). The matrix extends to the next
    // sub-tensor of the blob (its scales).
    if (PH == PH_UP) t.row = Fmt<FMT>::row(blob + grp.off[0], grp.off[1] - grp.off[0], 2 * orow + (is_up ? 1 : 0), K);
    else t.row = Fmt<FMT>::row(blob + grp.off[3], grp.down_bytes ? grp.down_bytes : grp.off[4] - grp.off[3], orow, K);
  } else if constexpr (FMT == Q_BF16) {
    // Gemma gate_up: gate = rows 0..I-1, up = rows I..2I-1 (Gemma4Weights.swift:107-112).
    if (PH == PH_UP) t.row = Fmt<FMT>::row(blob + grp.off[0], orow + (is_up ? I : 0), K);
    else t.row = Fmt<FMT>::row(blob + grp.off[1], orow, K);
  } else {
    const int mat = (PH == PH_UP) ? (is_up ? 1 : 0) : 2;
    t.row = Fmt<FMT>::row(blob + grp.off[3 * mat], blob + grp.off[3 * mat + 1], blob + grp.off[3 * mat + 2],
                          orow, K);
  }
  return t;
}

// The MFMA sequence of chunk c for NM A tiles × NT token tiles. `bv(st, hh, v)` returns the
// lane's 8 B values of token tile st, term hh (x | h_hi, h_lo), step v, at columns
// Fmt::bcol(c, g, K) + 8v.
// MLX: `sbf(m)`, when given, returns the (scale | bias << 16) words of D rows 4g .. 4g+3 of tile m
// for this chunk; otherwise they come from the A operands' rows by shuffles.
template <int FMT, int NM, int NT, int NH, class BV, class SBF = std::nullptr_t>
__device__ __forceinline__ void chunk_mfma(f32x4 (&acc)[NM][NT], const typename Fmt<FMT>::A (&w)[NM],
                                           const ATile<FMT> (&at)[NM], BV bv, int c, int g, int K,
                                           SBF sbf = nullptr) {
  using F = Fmt<FMT>;
  if constexpr (FMT == Q_BF16) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (!F::step_ok(c, v, K)) break;
      u32x4 b[NT][NH];
#pragma unroll
      for (int st = 0; st < NT; ++st)
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) b[st][hh] = bv(st, hh, v);
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int st = 0; st < NT; ++st)
#pragma unroll
          for (int hh = 0; hh < NH; ++hh) acc[m][st] = mfma(as_bf16x8(w[m].w[v]), as_bf16x8(b[st][hh]), acc[m][st]);
    }
  } else {
    // MLX affine, one 64-column group: P = Σ q·x on the bf16 MFMA (steps v = 0, 1: word v of the
    // lane's codes), G = Σ x on the MFMA with an all-ones A operand (every row of its D holds the
    // column sums, so each lane gets its column's), then acc += s·P + b·G per D row
    // (gemma.metal:234-236's factorisation). 4-bit codes enter the MFMA as bf16 (128 + q), two
    // per instruction pair: ((w >> 4k) & 0x000F000F) | 0x43004300 holds codes k and k+4, so the
    // B values are paired the same way (x_k, x_{k+4}) and the 128·G term goes into the bias:
    // acc += s·P' + (b − 128·s)·G.
    u32x4 b[NT][NH][2];
#pragma unroll
    for (int st = 0; st < NT; ++st)
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const u32x4 raw = bv(st, hh, v);
          if constexpr (FMT == Q_MLX4) {
            // (x0,x1)(x2,x3)(x4,x5)(x6,x7) → (x0,x4)(x1,x5)(x2,x6)(x3,x7)
            b[st][hh][v] = u32x4{__builtin_amdgcn_perm(raw[2], raw[0], 0x05040100u),
                                 __builtin_amdgcn_perm(raw[2], raw[0], 0x07060302u),
                                 __builtin_amdgcn_perm(raw[3], raw[1], 0x05040100u),
                                 __builtin_amdgcn_perm(raw[3], raw[1], 0x07060302u)};
          } else {
            b[st][hh][v] = raw;
          }
        }
    f32x4 P[NM][NT], G[NT];
#pragma unroll
    for (int st = 0; st < NT; ++st) {
      G[st] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < NM; ++m) P[m][st] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};   // bf16 1.0
#pragma unroll
    for (int v = 0; v < 2; ++v) {
#pragma unroll
      for (int st = 0; st < NT; ++st)
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) G[st] = mfma(as_bf16x8(ones), as_bf16x8(b[st][hh][v]), G[st]);
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        bf16x8 av;
        if constexpr (FMT == Q_MLX4) {
          const uint32_t wv = w[m].w[v];
          u32x4 r;
#pragma unroll
          for (int k = 0; k < 4; ++k) r[k] = ((wv >> (4 * k)) & 0x000F000Fu) | 0x43004300u;
          av = as_bf16x8(r);
        } else {
          av = mlx8_to_bf16(w[m].w[2 * v], w[m].w[2 * v + 1]);
        }
#pragma unroll
        for (int st = 0; st < NT; ++st)
#pragma unroll
          for (int hh = 0; hh < NH; ++hh) P[m][st] = mfma(av, as_bf16x8(b[st][hh][v]), P[m][st]);
      }
    }
    // D row 4g + ii is the A row of lane 4g + ii: its scale and bias by shuffle (all four
    // shuffles issued before the first is used).
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      uint32_t sbs[4];
      if constexpr (std::is_same_v<SBF, std::nullptr_t>) {
        const int sbl = (int)w[m].sb;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) sbs[ii] = (uint32_t)__shfl(sbl, 4 * g + ii);
      } else {
        const u32x4 v = sbf(m);
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) sbs[ii] = v[ii];
      }
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const uint32_t sbv = sbs[ii];
        const float sc = bf16_bits_to_f32(sbv & 0xFFFF);
        const float bi0 = bf16_bits_to_f32(sbv >> 16);
        const float bi = FMT == Q_MLX4 ? __builtin_fmaf(-128.f, sc, bi0) : bi0;
#pragma unroll
        for (int st = 0; st < NT; ++st) {
          acc[m][st][ii] = __builtin_fmaf(sc, P[m][st][ii], acc[m][st][ii]);
          acc[m][st][ii] = __builtin_fmaf(bi, G[st][ii], acc[m][st][ii]);
        }
      }
    }
  }
}

// acc = p0 + p1 per element (the two chains of the canonical arithmetic).
__device__ __forceinline__ f32x4 sum_chains(const f32x4 &p0, const f32x4 &p1) {
  f32x4 r;
#pragma unroll
  for (int ii = 0; ii < 4; ++ii) r[ii] = p0[ii] + p1[ii];
  return r;
}

// Gated activations of 4 intermediates (BF16 and MLX layers, which have no expert bias).
__device__ __forceinline__ f32x4 up_values(const GemmArgs &a, const f32x4 &gate, const f32x4 &up) {
  float gv[4], uv[4], yv[4];
#pragma unroll
  for (int ii = 0; ii < 4; ++ii) {
    gv[ii] = gate[ii] + 0.f;
    uv[ii] = up[ii] + 0.f;
  }
  activate_n<4>(a.act, gv, uv, yv, a.alpha, a.limit);
  return f32x4{yv[0], yv[1], yv[2], yv[3]};
}

// The same with the GPT-OSS bias of the 4 intermediates, already loaded: 16 bytes from the bias
// row at element 2·i0, (gate, up) bf16 pairs in order.
__device__ __forceinline__ f32x4 up_values_mx(const GemmArgs &a, const u32x4 &bias, const f32x4 &gate,
                                              const f32x4 &up) {
  float gv[4], uv[4], yv[4];
#pragma unroll
  for (int ii = 0; ii < 4; ++ii) {
    gv[ii] = gate[ii] + bf16_bits_to_f32(bias[ii] & 0xFFFFu);
    uv[ii] = up[ii] + bf16_bits_to_f32(bias[ii] >> 16);
  }
  activate_n<4>(a.act, gv, uv, yv, a.alpha, a.limit);
  return f32x4{yv[0], yv[1], yv[2], yv[3]};
}

// Gate-up epilogue of 4 intermediates i0..i0+3 of slot `slot` (BF16 and MLX layers): activation, bf16 hi/lo.
__device__ __forceinline__ void up_epilogue(const GemmArgs &a, int i0, int slot, const f32x4 &gate, const f32x4 &up) {
  const f32x4 yv = up_values(a, gate, up);
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int ii = 0; ii < 4; ++ii) {
    const float y = yv[ii];
    hi[ii] = f32_to_bf16_bits(y);
    lo[ii] = f32_to_bf16_bits(y - bf16_bits_to_f32(hi[ii]));
  }
  const size_t o = (size_t)slot * a.ldh + i0;
  *(u32x2 *)(a.h_hi + o) = u32x2{hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
  *(u32x2 *)(a.h_lo + o) = u32x2{lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
}

// ---- MXFP4 on the scaled MFMA -------------------------------------------------------------------
typedef int v8i __attribute__((ext_vector_type(8)));

// D += A·B, v_mfma_scale_f32_16x16x128_f8f6f4 with A = 16 rows × 128 K of fp4 e2m1 and B =
// 128 K × 16 columns of fp8 e4m3. A lane (g, l16): row l16, the 32 values of K block g (low nibble
// first: exactly one MXFP4 block as stored) and that block's e8m0 scale. B lane (g, l16): column
// l16, K 16g..16g+15 in bytes 0-15 and K 64+16g..64+16g+15 in bytes 16-31, and the e8m0 scale of
// K block g. D as the 16x16 bf16 MFMA.
__device__ __forceinline__ f32x4 smfma(const u32x4 &a, const u32x4 &blo, const u32x4 &bhi, uint32_t sa,
                                       uint32_t sb, const f32x4 &c) {
  const v8i av = {(int)a[0], (int)a[1], (int)a[2], (int)a[3], 0, 0, 0, 0};
  const v8i bv = {(int)blo[0], (int)blo[1], (int)blo[2], (int)blo[3],
                  (int)bhi[0], (int)bhi[1], (int)bhi[2], (int)bhi[3]};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 4, 0, 0, (int)sa, 0, (int)sb);
}

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// Tasks of a prefill launch: task τ, on XCD τ mod 8 (workgroups go to the XCDs in turn), is a row tile
// and a work item, or nothing past the row tiles or the items. The 8 XCDs form P row-tile parts ×
// 8/P work-item parts: XCD x takes row tiles of part x mod P and work items of part x / P, work item
// by work item (each item's row tiles consecutively). An expert's slice of weight rows stays in
// the XCD's L2 across the expert's consecutive items, and an item's operand rows are fetched by
// the P XCDs of its item part.
struct PrefillTasks {
  int RT, nwork, P, rtp, nq, lim;
  __device__ __forceinline__ PrefillTasks(int RT_, int nwork_, int P_)
      : RT(RT_), nwork(nwork_), P(P_), rtp((RT_ + P_ - 1) / P_), nq((nwork_ + 8 / P_ - 1) / (8 / P_)), lim(8 * rtp * nq) {}
  __device__ __forceinline__ bool tile(int tau, int &rt, int &wi) const {
    if (tau >= lim) return false;
    const int x = tau & 7, j = tau >> 3, q = j / rtp;
    rt = (x & (P - 1)) * rtp + (j - q * rtp);
    wi = (x / P) * nq + q;
    return rt < RT && wi < nwork;
  }
};

// Where an MXFP4 prefill wave finds its row scales in LDS. A row's three stages of scales come as the 16
// bytes from the dword that holds block sc0 of the row, moved back where they would pass the
// matrix's last byte: mx_scale_src is their offset in the matrix (rows of nsb blocks),
// mx_scale_back how far they were moved. Only a wave that holds the matrix's last rows has any that
// were (mx_last_rows, rw its first row): a wave wholly past them loads the last row's bytes, uses none,
// and must not form a distance from rows that do not exist.
__host__ __device__ constexpr bool mx_last_rows(int rw, int out_dim) { return rw < out_dim && rw + 64 >= out_dim; }
__host__ __device__ constexpr int mx_scale_src(int row, int out_dim, int nsb, int sc0) {
  const int at = (row * nsb + sc0) & ~3, end = out_dim * nsb - 16;
  return at < end ? at : end;
}
__host__ __device__ constexpr int mx_scale_back(int row, int out_dim, int nsb, int sc0) {
  const int past = ((row * nsb + sc0) & ~3) - (out_dim * nsb - 16);
  return past > 0 ? past : 0;
}

// At most N of the wave's loads outstanding.
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

}  // namespace hh
