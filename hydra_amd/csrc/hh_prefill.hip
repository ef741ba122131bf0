// hh_prefill.hip — expert products grouped by expert, on gfx950 MFMA: batches above 16 tokens, and of 5 to 16
// tokens on BF16 and MLX layers large enough for it (hh_api.hip:mid_batch). One four-wave workgroup per task (a row tile × a work item), two workgroups per compute unit.
#include "hh_mfma.hpp"

#include <algorithm>
#include <mutex>

namespace hh {

constexpr int kRowParts = 2;   // row-tile parts of the XCDs (PrefillTasks)

// 16 bytes per lane from global memory straight into LDS: base (uniform) + off (per lane) to LDS
// byte `l` + 16·lane. Written in assembly so that the compiler does not order the wave's own LDS
// reads after its loads in flight (it would wait for all of them); the kernels wait with wait_vm.
// The instruction has no register result; its LDS address goes through m0.
__device__ __forceinline__ void dma16(const void *base, uint32_t off, uint32_t l) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(l), "v"(off), "s"(base)
               : "memory", "m0");
}
__device__ __forceinline__ void dma16(const void *p, uint32_t l) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(l), "v"(p) : "memory", "m0");
}
// 4 (2) bytes per lane to LDS byte `l` + 4·lane.
__device__ __forceinline__ void dma4(const void *p, uint32_t l) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(l), "v"(p) : "memory", "m0");
}
__device__ __forceinline__ void dma2(const void *p, uint32_t l) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, off" ::"s"(l), "v"(p) : "memory", "m0");
}
// Barrier after the wave's own LDS reads have returned: the next stage may overwrite what they read.
__device__ __forceinline__ void step_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ uint32_t lds_addr(const uint8_t *l) { return (uint32_t)(uintptr_t)(lds_ptr_t)(void *)l; }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// One task per workgroup; two four-wave workgroups (BF16 160-token items: one of eight waves) per
// compute unit, so that one's loads, barriers and epilogue pass under the other's MFMAs. Every wave
// both loads and multiplies: a stage of K columns of the row tile's weights and of the item's
// token rows goes straight to an S-deep LDS ring, S − 1 stages ahead. Before (one persistent
// workgroup per compute unit, four loader waves and four MFMA waves) each SIMD had a single MFMA
// wave, which sat through its own LDS reads and barrier at every stage (with no global traffic at
// all the BF16 T = 2048 gate-up still took 350 of its 415 us).
// Weight loads take whole 128-byte (4-bit MLX: 64-byte) pieces of a row with consecutive lanes: 50 B/clk
// per compute unit from L2, against 15.5 for the MFMA lane order (16 rows × 64 bytes, consecutive
// lanes on different rows), which the L1 serves a row at a time when the row stride is a multiple
// of 128 bytes. The XOR of the 16-byte segments by the row keeps the MFMA lanes' LDS reads at full rate for BF16
// and 8-bit MLX (no conflict cycles counted; a fifth of MXFP4's and 4-bit MLX's LDS cycles are conflicts).
// The output tiles' arithmetic is the canonical one (chunk_mfma, prefill equals decode bit for bit).
//
// XCD order (PrefillTasks): two row-tile parts × four item parts, so an item's token rows reach two
// XCDs' L2: BF16 T = 2048 gate-up 430 us with four parts, 349 with two, 359 with one.

// ---- BF16 -----------------------------------------------------------------------------------------
// NT token tiles × NM weight tiles of 16 per wave; WT token groups of four waves; SV MFMA steps of
// 32 columns per stage.
// Tiles, timed on the 128-expert layer (H 2816, I 704; gate-up / down us at T tokens):
//   T = 2048 (128 tokens an expert): 64-token items of 128 intermediates 300 / 222, 128-token items
//     285 / 217, 160-token items 278 / 194 (an expert's weights are in 2.5, 1.5, 1.0 items; at 160 the
//     counters show 1.18 / 1.11 times the bytes needed);
//     with 32-column stages (64-byte pieces) 349 for the 64-token gate-up;
//   T = 700 (44 an expert): 160-token 206 / 144, 32-token 243 / 141;
//   T = 400 (25 an expert): 160-token 195 / 133, 32-token 196 / 112, hence the line at 40;
//   T = 100 (6 an expert; the weights' 1.03 GB stream at 5.8 TB/s): 32-token gate-up of 64
//     intermediates 179, of 128 201.
// The previous kernels: 415 / 284 at T = 2048, 302 / 177 at 700, 189 / 105 at 100.
template <int PH, int NT_, int RT_, int SV_, int WT_> struct Bf {
  static constexpr int NT = NT_, NH = PH == PH_UP ? 1 : 2, SV = SV_, WT = WT_;
  static constexpr int RT = RT_, NM = (PH == PH_UP ? 2 : 1) * RT;   // gate-up: RT gate and RT up tiles
  static constexpr int NW = 4 * WT;                          // waves
  static constexpr int ROWS = 64 * RT;                       // output rows per workgroup
  static constexpr int TB = 1024 * SV;                       // bytes of a 16-row tile
  static constexpr int A_INS = 4 * NM * SV, B_INS = NH * NT * WT * SV;   // 1 KiB loads per stage
  static constexpr int APW = A_INS / NW, BPW = (B_INS + NW - 1) / NW;
  static constexpr int L = APW + BPW;
  static constexpr int OFF_B = A_INS * 1024;
  static constexpr int STAGE = OFF_B + B_INS * 1024;
  static constexpr int S_FIT = (80 * WT * 1024) / STAGE, S = S_FIT > 4 ? 4 : S_FIT;
  static constexpr int LDS = S * STAGE;
  static_assert(S >= 2, "ring depth");
};

template <int PH, int NT_, int RT_, int SV_, int WT_>
__global__ __launch_bounds__(256 * WT_) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_bf16(GemmArgs a) {
  using C = Bf<PH, NT_, RT_, SV_, WT_>;
  constexpr int NM = C::NM, NT = C::NT, NH = C::NH, RT = C::RT, S = C::S, L = C::L, SV = C::SV, WT = C::WT, TB = C::TB;
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63, g = lane >> 4, l16 = lane & 15;
  const int wave = uniform(threadIdx.x >> 6), wr = wave & 3, wt = wave >> 2;
  const int H = a.hidden, E = a.experts;
  const int nwork = *a.n_work;
  int rt, wi;
  if (!PrefillTasks(a.row_tiles, nwork, kRowParts).tile(a.first_task + (int)blockIdx.x, rt, wi)) return;
  const int4 it = a.work[wi];
  const int e = uniform(it.x), pos = uniform(it.y), cnt = uniform(it.z);
  const ExpertGroup &grp = a.grp[e == E ? 1 : 0];
  const uint8_t *blob = grp.blobs + (e == E ? 0 : (size_t)e * grp.stride);
  const int I = grp.inter;
  const int K = PH == PH_UP ? H : I, out_dim = PH == PH_UP ? I : H;
  const int n = K / (32 * SV);   // stages
  if (rt * C::ROWS >= out_dim) return;
  const int rb = rt * C::ROWS + wr * 16 * RT, tb = wt * 16 * NT;
  const bool active = rb < out_dim && tb < cnt;

  constexpr int RPI = 16 / SV, SEGS = 4 * SV;   // rows per load, 16-byte segments per row
  const size_t rowb = (size_t)K * 2;
  const int lr = lane / SEGS;   // row of the load
  auto swz = [](int r) { return SV == 1 ? (r >> 1) & 3 : r & 7; };
  const int seg = (lane % SEGS) ^ swz(lr);
  const uint32_t aoff = (uint32_t)(lr * rowb + 16 * seg);
  const uint8_t *abase[C::APW];
#pragma unroll
  for (int i = 0; i < C::APW; ++i) {
    const int j = wave * C::APW + i;   // load j of the stage: tile j / SV, rows RPI·(j % SV) ..
    const int tl = j / SV, w = tl / NM, m = tl % NM;
    const int r0 = min(rt * C::ROWS + w * 16 * RT + 16 * (m % RT), out_dim - 16) + (PH == PH_UP && m >= RT ? I : 0);
    abase[i] = blob + grp.off[PH == PH_UP ? 0 : 1] + (r0 + RPI * (j % SV)) * rowb;
  }
  const uint8_t *bsrc[C::BPW];
  uint32_t bdst[C::BPW];
#pragma unroll
  for (int i = 0; i < C::BPW; ++i) {
    const int j = (wave * C::BPW + i) % C::B_INS, hh = j / (NT * WT * SV), tl = j % (NT * WT * SV);
    const int sl = a.order[pos + min(RPI * tl + lr, cnt - 1)];
    const uint16_t *row = PH == PH_UP ? a.x + (size_t)(sl / a.slots) * H : (hh ? a.h_lo : a.h_hi) + (size_t)sl * a.ldh;
    bsrc[i] = (const uint8_t *)row + 16 * seg;
    bdst[i] = lds_addr(lds) + C::OFF_B + 1024 * j;
  }
  int es[NT];
#pragma unroll
  for (int st = 0; st < NT; ++st) es[st] = a.order[pos + min(tb + 16 * st + l16, cnt - 1)];

  const uint32_t adst = lds_addr(lds) + wave * C::APW * 1024;
  int q = 0, qs = 0;   // stages issued, the ring slot of the next
  auto issue = [&]() {
    const uint32_t so = (uint32_t)(qs * C::STAGE);
#pragma unroll
    for (int i = 0; i < C::APW; ++i) dma16(abase[i] + 64 * SV * q, aoff, adst + so + 1024 * i);
#pragma unroll
    for (int i = 0; i < C::BPW; ++i) dma16(bsrc[i] + 64 * SV * q, bdst[i] + so);
    ++q;
    qs = qs == S - 1 ? 0 : qs + 1;
  };
  for (int u = 0; u < S - 1 && q < n; ++u) issue();

  f32x4 acc[2][NM][NT];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int st = 0; st < NT; ++st) acc[p][m][st] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int roff = l16 * 64 * SV + 16 * (g ^ swz(l16));   // step v: ^ 64·v
  int s = 0, ss = 0;   // stage computed, its ring slot
  auto step = [&](f32x4 (&ac)[NM][NT]) {
    // Stage s has landed once at most the later issued stages' loads are outstanding.
    const int later = q - 1 - s;
    if (later >= S - 2) wait_vm<(S - 2) * L>();
    else if (S > 3 && later == 1) wait_vm<L>();
    else wait_vm<0>();
    step_barrier();
    if (q < n) issue();
    const uint8_t *stg = lds + ss * C::STAGE;
    if (active) {
#pragma unroll
      for (int v = 0; v < SV; ++v) {
        const int ro = roff ^ (64 * v);
        u32x4 w[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) w[m] = *(const u32x4 *)(stg + (wr * NM + m) * TB + ro);
#pragma unroll
        for (int st = 0; st < NT; ++st) {
          if (st > 0 && tb + 16 * st >= cnt) break;   // token tiles wholly past the item
#pragma unroll
          for (int hh = 0; hh < NH; ++hh) {
            const u32x4 b = *(const u32x4 *)(stg + C::OFF_B + (hh * NT * WT + wt * NT + st) * TB + ro);
#pragma unroll
            for (int m = 0; m < NM; ++m) ac[m][st] = mfma(as_bf16x8(w[m]), as_bf16x8(b), ac[m][st]);
          }
        }
      }
    }
    ++s;
    ss = ss == S - 1 ? 0 : ss + 1;
  };
  // Chunks of 128 columns: the even ones into chain 0, the odd ones into chain 1.
  constexpr int SPC = 4 / SV;
  for (int c0 = 0; c0 < n; c0 += 2 * SPC) {
    const int n0 = min(n, c0 + SPC), n1 = min(n, c0 + 2 * SPC);
#pragma unroll 1
    while (s < n0) step(acc[0]);
#pragma unroll 1
    while (s < n1) step(acc[1]);
  }
  if (!active) return;
#pragma unroll
  for (int st = 0; st < NT; ++st) {
    if (tb + 16 * st + l16 >= cnt) continue;
    const float ew = PH == PH_DOWN ? a.slot_w[es[st]] : 0.f;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int r0 = rb + 16 * r;
      if (r0 >= out_dim) continue;
      if constexpr (PH == PH_UP) {
        up_epilogue(a, r0 + 4 * g, es[st], sum_chains(acc[0][r][st], acc[1][r][st]),
                    sum_chains(acc[0][RT + r][st], acc[1][RT + r][st]));
      } else {
        const f32x4 v = sum_chains(acc[0][r][st], acc[1][r][st]);
        f32x4 o;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) o[ii] = ew * (v[ii] + 0.f);   // down_value's arithmetic
        *(f32x4 *)(a.slot_out + (size_t)es[st] * H + r0 + 4 * g) = o;
      }
    }
  }
}

// ---- MLX affine -----------------------------------------------------------------------------------
// A stage is two 64-column groups. Bound by VALU work where experts have many tokens: per group and wave, 14
// operations to expand a 16-row tile's 4-bit codes (24 for 8-bit), and eight per tile and token tile
// to scale the group's partial sums; the MFMAs take a third of that. Two things keep the rest small:
// the group scales become fp32 once per row (one row per lane, through LDS) instead of in every
// lane of the 16 that share a D row (48 operations per group, T = 1024 gate-up 151 -> 135 us), and the
// lane's LDS offsets are formed once. 256-expert layer (H 2048, I 512), gate-up / down us:
//   4-bit T = 1024 135 / 112 (before: 227 / 160), T = 333 110 / 67 (158 / 104), T = 60 85 / 53 (125 / 85);
//   8-bit T = 333 137 / 79 (170 / 99), T = 1024 176 / 126 (237 / 154).
// RT: 4-bit gate-up tiles of 128 intermediates 135, of 64 157 (an operand pair is expanded for half
// the rows); 4-bit down tiles of 192 rows 112, of 256 115 (spills), of 128 120; 8-bit down tiles of 128
// rows 79 at T = 333, of 64 115; wider 8-bit tiles leave one stage in LDS.
template <int PH, int BITS, int RT_, int NT_> struct Ml {
  static constexpr int NT = NT_, NH = PH == PH_UP ? 1 : 2;
  static constexpr int RT = RT_, NM = (PH == PH_UP ? 2 : 1) * RT;
  static constexpr int ROWS = 64 * RT;
  static constexpr int AK = BITS / 4;                        // KiB of a 16-row tile per stage
  static constexpr int APW = NM * AK, BPW = NH * NT;         // 1 KiB loads per wave per stage
  static constexpr int L = APW + BPW + 2;
  static constexpr int OFF_B = 4 * APW * 1024;
  static constexpr int OFF_SB = OFF_B + 4 * BPW * 1024;      // per wave: scale words, bias words of 64 rows
  static constexpr int STAGE = OFF_SB + 4 * 512;
  static constexpr int S_FIT = (76 * 1024) / STAGE, S = S_FIT > 4 ? 4 : S_FIT;
  static constexpr int OFF_F = S * STAGE;                    // per wave: [group][scale, bias][64 rows] fp32
  static constexpr int LDS = OFF_F + 4 * 1024;
  static_assert(S >= 2 && NM <= 4, "ring depth");
};

template <int PH, int BITS, int RT_, int NT_>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_mlx(GemmArgs a) {
  using C = Ml<PH, BITS, RT_, NT_>;
  constexpr int NM = C::NM, NT = C::NT, NH = C::NH, RT = C::RT, S = C::S, L = C::L, AK = C::AK;
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63, g = lane >> 4, l16 = lane & 15;
  const int wave = uniform(threadIdx.x >> 6);
  const int H = a.hidden, E = a.experts;
  const int nwork = *a.n_work;
  int rt, wi;
  if (!PrefillTasks(a.row_tiles, nwork, kRowParts).tile(a.first_task + (int)blockIdx.x, rt, wi)) return;
  const int4 it = a.work[wi];
  const int e = uniform(it.x), pos = uniform(it.y), cnt = uniform(it.z);
  const ExpertGroup &grp = a.grp[e == E ? 1 : 0];
  const uint8_t *blob = grp.blobs + (e == E ? 0 : (size_t)e * grp.stride);
  const int I = grp.inter;
  const int K = PH == PH_UP ? H : I, out_dim = PH == PH_UP ? I : H;
  const int ng = K / 64, n = (ng + 1) / 2;   // groups; stages of two
  if (rt * C::ROWS >= out_dim) return;
  const int rb = rt * C::ROWS + wave * 16 * RT;
  const bool active = rb < out_dim;

  constexpr int SEGS = 4 * AK, RPI = 16 / AK;   // 16-byte segments per weight row, rows per load
  const int rowb = K * BITS / 8;
  auto aswz = [](int r) { return AK == 1 ? (r >> 1) & 3 : r & 7; };
  const int lr = lane / SEGS, seg = (lane % SEGS) ^ aswz(lr);
  // The last stage of an odd group count has one group: lanes past it repeat that group's bytes.
  const uint32_t aoff = (uint32_t)(lr * rowb + 16 * seg);
  const uint32_t aoff_t = (ng & 1) ? (uint32_t)(lr * rowb + 16 * (seg & (SEGS / 2 - 1))) : aoff;
  const uint8_t *abase[C::APW];
#pragma unroll
  for (int i = 0; i < C::APW; ++i) {
    const int m = i / AK, mat = PH == PH_UP ? (m >= RT ? 1 : 0) : 2;
    const int r0 = min(rb + 16 * (m % RT), out_dim - 16);
    abase[i] = blob + grp.off[3 * mat] + (size_t)(r0 + RPI * (i % AK)) * rowb;
  }
  // Lane 16m + r: the two groups' scales (biases) of row r of tile m, one dword.
  const uint8_t *ssrc, *zsrc;
  {
    const int m = min(lane >> 4, NM - 1), mat = PH == PH_UP ? (m >= RT ? 1 : 0) : 2;
    const size_t r = min(rb + 16 * (m % RT), out_dim - 16) + l16;
    ssrc = blob + grp.off[3 * mat + 1] + r * ng * 2;
    zsrc = blob + grp.off[3 * mat + 2] + r * ng * 2;
  }
  // Operand load j of the stage: 4 token rows of 256 bytes.
  const uint8_t *bsrc[C::BPW];
  uint32_t bdst[C::BPW];
  int btail[C::BPW];
#pragma unroll
  for (int i = 0; i < C::BPW; ++i) {
    const int j = wave * C::BPW + i, hh = j / (4 * NT), tl = j % (4 * NT);
    const int tn = 4 * tl + (lane >> 4), sl = a.order[pos + min(tn, cnt - 1)];
    const uint16_t *row = PH == PH_UP ? a.x + (size_t)(sl / a.slots) * H : (hh ? a.h_lo : a.h_hi) + (size_t)sl * a.ldh;
    const int sg = l16 ^ (tn & 15);
    bsrc[i] = (const uint8_t *)row + 16 * sg;
    btail[i] = (ng & 1) && sg >= 8 ? 128 : 0;
    bdst[i] = lds_addr(lds) + C::OFF_B + 1024 * j;
  }
  int es[NT];
#pragma unroll
  for (int st = 0; st < NT; ++st) es[st] = a.order[pos + min(16 * st + l16, cnt - 1)];

  const uint32_t adst = lds_addr(lds) + wave * C::APW * 1024;
  const uint32_t sdst = lds_addr(lds) + C::OFF_SB + wave * 512;
  int q = 0, qs = 0;
  auto issue = [&]() {
    const uint32_t so = (uint32_t)(qs * C::STAGE);
    const bool tail = q == n - 1;
    const uint32_t ao = tail ? aoff_t : aoff;
#pragma unroll
    for (int i = 0; i < C::APW; ++i) dma16(abase[i] + 64 * AK * q, ao, adst + so + 1024 * i);
#pragma unroll
    for (int i = 0; i < C::BPW; ++i) dma16(bsrc[i] + (256 * q - (tail ? btail[i] : 0)), bdst[i] + so);
    // A dword holds groups 2q and 2q + 1; the last stage of an odd count reads its group alone.
    if (tail && (ng & 1)) {
      dma2(ssrc + 4 * q, sdst + so);
      dma2(zsrc + 4 * q, sdst + so + 256);
    } else {
      dma4(ssrc + 4 * q, sdst + so);
      dma4(zsrc + 4 * q, sdst + so + 256);
    }
    ++q;
    qs = qs == S - 1 ? 0 : qs + 1;
  };
  for (int u = 0; u < S - 1 && q < n; ++u) issue();

  f32x4 acc[2][NM][NT];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int st = 0; st < NT; ++st) acc[p][m][st] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The lane's offsets in a stage: its codes (group 1: ^ 32 · AK), its operand segments (group, step: ^ 128, ^ 16).
  const uint32_t alo = wave * NM * AK * 1024 + 64 * AK * l16 +
                       (BITS == 4 ? 16 * ((g >> 1) ^ aswz(l16)) + 8 * (g & 1) : 16 * (g ^ aswz(l16)));
  const uint32_t blo = C::OFF_B + 256 * l16 + 16 * ((2 * g) ^ l16);
  float *fsb = (float *)(lds + C::OFF_F) + 256 * wave + lane;
  const float *fsr = (const float *)(lds + C::OFF_F) + 256 * wave + 4 * g;
  int ss = 0;
#pragma unroll 1
  for (int s = 0; s < n; ++s) {
    const int later = q - 1 - s;
    if (later >= S - 2) wait_vm<(S - 2) * L>();
    else if (S > 3 && later == 1) wait_vm<L>();
    else wait_vm<0>();
    step_barrier();
    if (q < n) issue();
    const uint8_t *stg = lds + ss * C::STAGE;
    ss = ss == S - 1 ? 0 : ss + 1;
    if (!active) continue;
    {
      // The wave's 64 rows, one per lane: scale and bias of both groups as fp32 (the 4-bit bias
      // less 128 scales), written for the D rows' reads below. Every lane would otherwise convert
      // the values of its four D rows of each tile.
      const uint32_t sw = *(const uint32_t *)(stg + C::OFF_SB + wave * 512 + 4 * lane);
      const uint32_t zw = *(const uint32_t *)(stg + C::OFF_SB + wave * 512 + 256 + 4 * lane);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const float sc = __uint_as_float(p ? sw & 0xFFFF0000u : sw << 16);
        const float z = __uint_as_float(p ? zw & 0xFFFF0000u : zw << 16);
        fsb[128 * p] = sc;
        fsb[128 * p + 64] = BITS == 4 ? __builtin_fmaf(-128.f, sc, z) : z;
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if (2 * s + p >= ng) break;   // an odd group count's last stage has one
      // Codes of group 2s + p as bf16 (chunk_mfma's forms); its scales and biases of D rows 4g .. 4g + 3.
      u32x4 av[NM][2];
      f32x4 sc[NM], bi[NM];
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const uint8_t *tile = stg + m * AK * 1024;
        if constexpr (BITS == 4) {
          const u32x2 c = *(const u32x2 *)(tile + (alo ^ (32 * p)));
#pragma unroll
          for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int k = 0; k < 4; ++k) av[m][v][k] = ((c[v] >> (4 * k)) & 0x000F000Fu) | 0x43004300u;
        } else {
          const u32x4 c = *(const u32x4 *)(tile + (alo ^ (64 * p)));
#pragma unroll
          for (int v = 0; v < 2; ++v) av[m][v] = __builtin_bit_cast(u32x4, mlx8_to_bf16(c[2 * v], c[2 * v + 1]));
        }
        sc[m] = *(const f32x4 *)(fsr + 128 * p + 16 * m);
        bi[m] = *(const f32x4 *)(fsr + 128 * p + 64 + 16 * m);
      }
      const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};   // bf16 1.0
#pragma unroll
      for (int st = 0; st < NT; ++st) {
        if (st > 0 && 16 * st >= cnt) break;   // token tiles wholly past the item
        u32x4 b[NH][2];
#pragma unroll
        for (int hh = 0; hh < NH; ++hh)
#pragma unroll
          for (int v = 0; v < 2; ++v) {
            const u32x4 r = *(const u32x4 *)(stg + (hh * NT + st) * 4096 + (blo ^ (128 * p + 16 * v)));
            if constexpr (BITS == 4) {
              // (x0,x1)(x2,x3)(x4,x5)(x6,x7) → (x0,x4)(x1,x5)(x2,x6)(x3,x7), the codes' pairing
              b[hh][v] = u32x4{__builtin_amdgcn_perm(r[2], r[0], 0x05040100u), __builtin_amdgcn_perm(r[2], r[0], 0x07060302u),
                               __builtin_amdgcn_perm(r[3], r[1], 0x05040100u), __builtin_amdgcn_perm(r[3], r[1], 0x07060302u)};
            } else {
              b[hh][v] = r;
            }
          }
        f32x4 G = {0.f, 0.f, 0.f, 0.f}, P[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) P[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
          for (int hh = 0; hh < NH; ++hh) {
            G = mfma(as_bf16x8(ones), as_bf16x8(b[hh][v]), G);
#pragma unroll
            for (int m = 0; m < NM; ++m) P[m] = mfma(as_bf16x8(av[m][v]), as_bf16x8(b[hh][v]), P[m]);
          }
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) {
            acc[p][m][st][ii] = __builtin_fmaf(sc[m][ii], P[m][ii], acc[p][m][st][ii]);
            acc[p][m][st][ii] = __builtin_fmaf(bi[m][ii], G[ii], acc[p][m][st][ii]);
          }
      }
    }
  }
  if (!active) return;
#pragma unroll
  for (int st = 0; st < NT; ++st) {
    if (16 * st + l16 >= cnt) continue;
    const float ew = PH == PH_DOWN ? a.slot_w[es[st]] : 0.f;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int r0 = rb + 16 * r;
      if (r0 >= out_dim) continue;
      if constexpr (PH == PH_UP) {
        up_epilogue(a, r0 + 4 * g, es[st], sum_chains(acc[0][r][st], acc[1][r][st]),
                    sum_chains(acc[0][RT + r][st], acc[1][RT + r][st]));
      } else {
        const f32x4 v = sum_chains(acc[0][r][st], acc[1][r][st]);
        f32x4 o;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) o[ii] = ew * (v[ii] + 0.f);   // down_value's arithmetic
        *(f32x4 *)(a.slot_out + (size_t)es[st] * H + r0 + 4 * g) = o;
      }
    }
  }
}

// ---- MXFP4 ----------------------------------------------------------------------------------------
// A stage is 128 columns: 16-row weight tiles of 64 bytes a row (one MFMA's K), the token rows' fp8
// terms, and, every third stage, the scales of three stages. A wave owns 64 weight rows (32
// intermediates of gate-up, gate and up rows interleaved) and all the item's tokens.
// What bounds it: the weight rows' arrival. Without weight traffic the T = 2048 gate-up takes 305 of its
// 411 us (and 224 without its MFMAs, 360 without its epilogue; the MFMA pipes are busy a third of the time, and 2.1 times the
// bytes needed are fetched, 1.4 at T = 512), so three things keep more of them in flight or make them cheaper, on the 128-expert layer (H = I = 2880, Zipf load; gate-up / down us):
//   - scales 16 bytes a row every three stages instead of 4 every stage (a row's scales lie 90
//     bytes from the next row's, so every lane of such a load takes a cache line of its own): T = 2048
//     447 / 312 -> 413 / 283, T = 512 212 / 135 -> 193 / 124;
//   - a stage's weight tiles are private to a wave, which reloads their slot as soon as they are in
//     its registers: two stages in flight from two slots, T = 512 193 / 124 -> 183 / 116;
//   - two workgroups per compute unit: eight waves sharing a 64- or 128-token operand tile 514-540 at T = 2048.
// Before (persistent kernels with loader waves): T = 2048 483 / 368, T = 512 222 / 148, and 102 / 55 at
// T = 45 of the 32-expert layer, now 405 / 279, 183 / 116 and 92 / 49.
// Gate-up items hold 64 tokens where experts average 16 or more (T = 2048 405, with 32 tokens 480;
// T = 512 183 against 199), 16 where few experts have few tokens each (three gate-up workgroups per
// compute unit: 92 -> 78 at T = 45; the down product's three terms leave room for two), down items otherwise 32
// (a 64-token stage leaves one slot).
template <int PH, int NT_> struct Mx {
  static constexpr int NT = NT_, NTERM = PH == PH_UP ? NTX : NTH;
  static constexpr int NJ = 4;                               // 16-row tiles per wave, their 1 KiB loads per stage
  static constexpr int ROWS = 256, TOK = 16 * NT;            // weight rows, tokens of a work item
  static constexpr int B_INS = NTERM * TOK / 8, BPW = (B_INS + 3) / 4;   // 1 KiB operand loads per stage
  static constexpr int BR = NTERM * TOK, BSL = (BR + 63) / 64;           // operand rows; loads of their scales
  static constexpr int OFF_B = 16 * 1024;
  static constexpr int STAGE = OFF_B + B_INS * 1024;
  // Scales of three stages: 16 bytes of each weight row, then of each operand row; two such sets.
  static constexpr int OFF_Q = 2 * STAGE, QB = 4096, QUAD = QB + BSL * 1024;
  static constexpr int LDS = OFF_Q + 2 * QUAD;
  static constexpr int WGS = LDS <= 160 * 1024 / 3 ? 3 : 2;   // workgroups per compute unit
  static_assert(BSL <= 4 && LDS <= 80 * 1024, "two workgroups per compute unit");
};
static_assert(Mx<PH_UP, 1>::WGS == 3 && Mx<PH_DOWN, 1>::WGS == 2, "16-token items: 50 KB, and 54 KB with three terms");

template <int PH, int NT_>
__global__ __launch_bounds__(256, (Mx<PH, NT_>::WGS)) void prefill_mx(GemmArgs a) {
  using C = Mx<PH, NT_>;
  constexpr int NT = C::NT, NTERM = C::NTERM, NJ = C::NJ, TOK = C::TOK;
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63, g = lane >> 4, l16 = lane & 15;
  const int wave = uniform(threadIdx.x >> 6);
  const int H = a.hidden;
  const int nwork = *a.n_work;
  int rt, wi;
  if (!PrefillTasks(a.row_tiles, nwork, kRowParts).tile(a.first_task + (int)blockIdx.x, rt, wi)) return;
  const int4 it = a.work[wi];
  const int e = uniform(it.x), pos = uniform(it.y), cnt = uniform(it.z);
  const ExpertGroup &grp = a.grp[e == a.experts ? 1 : 0];
  const uint8_t *blob = grp.blobs + (e == a.experts ? 0 : (size_t)e * grp.stride);
  const int I = grp.inter;
  const int K = PH == PH_UP ? H : I, out_dim = PH == PH_UP ? 2 * I : H;
  const int nsb = K / 32, n = (K + 127) / 128;   // blocks of a row; stages
  const int ld = PH == PH_UP ? a.xld : a.hld;
  const uint8_t *qbase = PH == PH_UP ? a.xq : a.hq, *sbase = PH == PH_UP ? a.xs : a.hs;
  if (rt * C::ROWS >= out_dim) return;
  const int rw = rt * C::ROWS + 64 * wave;   // the wave's first row
  const bool active = rw < out_dim;
  const bool part = (K & 127) != 0;   // the last stage holds 64 columns
  const bool last_rows = mx_last_rows(rw, out_dim);   // holds the rows within 16 bytes of the scales' end

  const int rowb = K / 2;
  const int lr = lane >> 2, seg = (lane & 3) ^ ((lr >> 1) & 3);
  const uint32_t aoff = (uint32_t)(lr * rowb + 16 * seg);
  const uint32_t aoff_t = part ? (uint32_t)(lr * rowb + 16 * (seg & 1)) : aoff;   // lanes past K repeat the half before it
  const uint8_t *abase[NJ];
#pragma unroll
  for (int i = 0; i < NJ; ++i) {
    const int r0 = min(rw + 16 * i, out_dim - 16);
    abase[i] = blob + grp.off[PH == PH_UP ? 0 : 3] + (size_t)r0 * rowb;
  }
  // Block scales of row rw + lane: 16 bytes from the dword that holds a stage's
  // first, which covers three stages; moved back where they would pass the matrix's last byte.
  const uint8_t *sbase_w = blob + grp.off[PH == PH_UP ? 1 : 4];
  const int srow = min(rw + lane, out_dim - 1);
  const int ntok = (cnt + 15) & ~15;   // operand rows past the last used token tile are not loaded
  const uint8_t *bsrc[C::BPW];
  bool bon[C::BPW];
#pragma unroll
  for (int i = 0; i < C::BPW; ++i) {
    const int j = (wave * C::BPW + i) % C::B_INS, r = 8 * j + (lane >> 3), t = r / TOK, tn = r % TOK;
    bon[i] = (8 * j) % TOK < ntok;
    const int sl = a.order[pos + min(tn, cnt - 1)];
    bsrc[i] = qbase + ((size_t)(PH == PH_UP ? sl / a.slots : sl) * NTERM + t) * ld + 16 * ((lane & 7) ^ (tn & 7));
  }
  const uint8_t *bssrc;
  {
    const int d = min(min(wave, C::BSL - 1) * 64 + lane, C::BR - 1), t = d / TOK, tn = d % TOK;
    const int sl = a.order[pos + min(tn, cnt - 1)];
    bssrc = sbase + ((size_t)(PH == PH_UP ? sl / a.slots : sl) * NTERM + t) * (ld / 32);
  }
  int es[NT];
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) es[tt] = a.order[pos + min(16 * tt + l16, cnt - 1)];

  const uint32_t l0 = lds_addr(lds);
  int q = 0, qs = 0, q3 = 0, qset = 0;   // stages issued, its ring slot, stage mod 3, scale set
  auto issue = [&]() {
    const uint32_t st = l0 + (uint32_t)(qs * C::STAGE);
    if (q3 == 0) {
      const uint32_t qd = l0 + C::OFF_Q + qset * C::QUAD;
      dma16(sbase_w + mx_scale_src(srow, out_dim, nsb, 4 * q), qd + 1024 * wave);
      if (wave < C::BSL) dma16(bssrc + 4 * q, qd + C::QB + 1024 * wave);
      qset ^= 1;
    }
    q3 = q3 == 2 ? 0 : q3 + 1;
#pragma unroll
    for (int i = 0; i < C::BPW; ++i)
      if (bon[i]) dma16(bsrc[i] + 128 * q, st + C::OFF_B + 1024 * ((wave * C::BPW + i) % C::B_INS));
    ++q;
    qs ^= 1;
  };
  // Weight tiles of stage s (the wave's own: only it reads them) into slot s & 1.
  auto issue_a = [&](int s) {
    const uint32_t ao = part && s == n - 1 ? aoff_t : aoff;
#pragma unroll
    for (int i = 0; i < NJ; ++i) dma16(abase[i] + 64 * s, ao, l0 + (s & 1) * C::STAGE + 1024 * (wave * NJ + i));
  };
  issue_a(0);
  issue();
  if (n > 1) issue_a(1);

  f32x4 acc[NJ][NT];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) acc[j][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int aro = 4096 * wave + 64 * l16 + 16 * (g ^ ((l16 >> 1) & 3));
  const int bro = C::OFF_B + 128 * l16 + 16 * (g ^ (l16 & 7));   // the high half: ^ 64
  const int sro = C::OFF_Q + 16 * (64 * wave + l16) + g + (((rw + l16) * nsb) & 3), bso = C::OFF_Q + C::QB + 16 * l16 + g;
  int ss = 0, s3 = 0, sset = 0;
#pragma unroll 1
  for (int s = 0; s < n; ++s) {
    // Stage s has landed; the weight tiles of stage s + 1, issued after it, may be in flight.
    if (s + 1 < n) wait_vm<NJ>();
    else wait_vm<0>();
    step_barrier();
    if (q < n) issue();
    const uint8_t *stg = lds + ss * C::STAGE;
    ss ^= 1;
    const uint8_t *qd = lds + sset * C::QUAD + 4 * s3;   // this stage's scales in its set
    const int sc0 = 4 * (s - s3);
    s3 = s3 == 2 ? 0 : s3 + 1;
    if (s3 == 0) sset ^= 1;
    u32x4 w[NJ];
    uint32_t sa[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      w[j] = *(const u32x4 *)(stg + aro + 1024 * j);
      int back = 0;   // how far the row's 16 bytes were moved back
      if (last_rows) back = mx_scale_back(rw + 16 * j + l16, out_dim, nsb, sc0);
      sa[j] = qd[sro + 256 * j + back];
    }
    // The wave's weight tiles are in registers: their slot takes the stage after the next, two
    // steps ahead of its use.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (s + 2 < n) issue_a(s + 2);
    if (!active) continue;
    const bool tail = part && s == n - 1;
    // Lanes past K take zero weights and operand terms with scales 2^0 (whatever bytes they read).
    const bool ok = !tail || g < 2;
    if (tail) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if (!ok) w[j] = u32x4{0u, 0u, 0u, 0u};
        if (!ok) sa[j] = 127u;
      }
    }
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
      if (tt > 0 && 16 * tt >= cnt) break;   // token tiles wholly past the item
#pragma unroll
      for (int t = 0; t < NTERM; ++t) {
        const u32x4 blo = *(const u32x4 *)(stg + bro + 128 * (TOK * t + 16 * tt));
        u32x4 bhi = *(const u32x4 *)(stg + (bro ^ 64) + 128 * (TOK * t + 16 * tt));
        uint32_t bs = qd[bso + 16 * (TOK * t + 16 * tt)];
        if (tail) {
          bhi = u32x4{0u, 0u, 0u, 0u};
          if (!ok) bs = 127u;
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[j][tt] = smfma(w[j], blo, bhi, sa[j], bs, acc[j][tt]);
      }
    }
  }
  if (!active) return;
  float bias[NJ][4];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) bias[j][ii] = 0.f;
  if (a.expert_bias) {
    const uint16_t *bp = (const uint16_t *)(blob + grp.off[PH == PH_UP ? 2 : 5]) + rw + 4 * g;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const u32x2 bw = *(const u32x2 *)(bp + 16 * j);
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) bias[j][ii] = bf16_bits_to_f32((bw[ii >> 1] >> (16 * (ii & 1))) & 0xFFFFu);
    }
  }
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    if (16 * tt >= cnt) break;
    const bool in = 16 * tt + l16 < cnt;
    if constexpr (PH == PH_UP) {
      float v[8], gv[8], uv[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 d = acc[j][tt];
        gv[2 * j] = d[0] + bias[j][0];
        uv[2 * j] = d[1] + bias[j][1];
        gv[2 * j + 1] = d[2] + bias[j][2];
        uv[2 * j + 1] = d[3] + bias[j][3];
      }
      activate_n<8>(a.act, gv, uv, v, a.alpha, a.limit);
      uint32_t hq[NTH][2], sbq[NTH], he[NTH][2];
      quant_block<NTH>(v, hq, sbq);
      // Each lane's 8 contiguous bytes of every term (one store each).
#pragma unroll
      for (int t = 0; t < NTH; ++t) transpose_pieces(hq[t][0], hq[t][1], g, he[t][0], he[t][1]);
      if (in) {
        const int i0 = rw / 2;
#pragma unroll
        for (int t = 0; t < NTH; ++t) {
          *(u32x2 *)(a.hq + ((size_t)es[tt] * NTH + t) * a.hld + i0 + 8 * g) = u32x2{he[t][0], he[t][1]};
          if (g == 0) a.hs[((size_t)es[tt] * NTH + t) * (a.hld / 32) + i0 / 32] = (uint8_t)sbq[t];
        }
      }
    } else if (in) {
      const float ew = a.slot_w[es[tt]];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        f32x4 o;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) o[ii] = ew * (acc[j][tt][ii] + bias[j][ii]);   // down_value's arithmetic
        *(f32x4 *)(a.slot_out + (size_t)es[tt] * H + rw + 16 * j + 4 * g) = o;
      }
    }
  }
}

// One workgroup per task; launches of at most 2^22 workgroups (a launch's threads are counted in 32
// bits), each told its first task.
template <class C> static hipError_t launch_tasks(void (*kernel)(GemmArgs), int threads, int rows, GemmArgs a, int max_work,
                                                  hipStream_t s, Timing tm, std::once_flag &once) {
  std::call_once(once, [&] {
    (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    (void)hipGetLastError();
  });
  a.row_tiles = (rows + C::ROWS - 1) / C::ROWS;
  constexpr int P = kRowParts;
  const int64_t tasks = 8ll * ((a.row_tiles + P - 1) / P) * ((max_work + 8 / P - 1) / (8 / P));
  constexpr int64_t most = 1ll << 22;
  for (int64_t t0 = 0; t0 < tasks; t0 += most) {
    a.first_task = (int32_t)t0;
    hipExtLaunchKernelGGL(kernel, dim3((unsigned)std::min(most, tasks - t0)), dim3(threads), C::LDS, s,
                          t0 == 0 ? tm.start : nullptr, t0 + most >= tasks ? tm.stop : nullptr, 0, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
// Tasks of a launch at most, with `rows` output rows each.
static int64_t tasks(int max_work, int out, int rows) { return (int64_t)max_work * ((out + rows - 1) / rows); }
template <int PH> static int out_rows(const GemmArgs &a) {
  return PH == PH_UP ? std::max(a.grp[0].inter, a.grp[1].inter) : a.hidden;
}
template <int PH, int NT, int RT, int SV, int WT> static hipError_t launch_bf16(const GemmArgs &a, int max_work, hipStream_t s, Timing tm) {
  static std::once_flag once;
  return launch_tasks<Bf<PH, NT, RT, SV, WT>>(prefill_bf16<PH, NT, RT, SV, WT>, 256 * WT, out_rows<PH>(a), a, max_work, s, tm, once);
}
template <int PH, int BITS, int RT, int NT> static hipError_t launch_mlx(const GemmArgs &a, int max_work, hipStream_t s, Timing tm) {
  static std::once_flag once;
  return launch_tasks<Ml<PH, BITS, RT, NT>>(prefill_mlx<PH, BITS, RT, NT>, 256, out_rows<PH>(a), a, max_work, s, tm, once);
}
template <int PH, int NT> static hipError_t launch_mx(const GemmArgs &a, int max_work, hipStream_t s, Timing tm) {
  static std::once_flag once;
  return launch_tasks<Mx<PH, NT>>(prefill_mx<PH, NT>, 256, (PH == PH_UP ? 2 : 1) * out_rows<PH>(a), a, max_work, s, tm, once);
}

// The tile of each call (`max_work`: its work items at most). BF16 work items hold 160 tokens (nt 10: experts averaging 40 tokens or
// more) or 32, MXFP4 items 16 (nt 1), 32, or 64 for the gate-up
// (nt 4), MLX items 32.
hipError_t launch_gemm(int phase, int quant, int nt, const GemmArgs &a, int max_work, hipStream_t s, Timing tm) {
  const bool up = phase == PH_UP;
  if (quant == Q_MLX4) {
    // Tiles of 64 rows where even they do not fill the two workgroups a compute unit holds (tasks counted at the
    // wide tiles, of twice and three times the rows). Gate-up, us, wide / 64 (tasks): 1 expert of H 2880, I 512 T = 100
    // 40 / 28 (20), 16 experts of H 2048, I 768 (K 4) T = 100 29 / 21 (174), 256 experts of H 2048, I 512 (K 8)
    // T = 8 26 / 24 (268), T = 12 36 / 37 (400). Down: 4 experts of H 2048, I 1536 (K 2) T = 100 24 / 17 (121), T = 300
    // 24 / 32 (253). Down tiles of 128 rows where those of 192 would be a tenth padding, with up to two tasks a
    // compute unit: 512 x 2880 T = 2000 55 / 48 (189), 1024 x 1024 T = 2000 33 / 30 (378), T = 8000 77 / 82 (1500).
    if (up) return tasks(max_work, a.grp[0].inter, 128) <= 300 ? launch_mlx<PH_UP, 4, 1, 2>(a, max_work, s, tm) : launch_mlx<PH_UP, 4, 2, 2>(a, max_work, s, tm);
    const int64_t wide = tasks(max_work, a.hidden, 192);
    if (wide <= 130) return launch_mlx<PH_DOWN, 4, 1, 2>(a, max_work, s, tm);
    const int pad128 = (a.hidden + 127) / 128 * 128, pad192 = (a.hidden + 191) / 192 * 192;
    if (wide <= 512 && 10 * pad192 > 11 * pad128) return launch_mlx<PH_DOWN, 4, 2, 2>(a, max_work, s, tm);
    return launch_mlx<PH_DOWN, 4, 3, 2>(a, max_work, s, tm);
  }
  if (quant == Q_MLX8) {
    // The same for 8-bit down tiles: 4 experts of H 2048, I 1536 (K 2) T = 40 the layer 60 / 55 (tasks of 128 rows: 112),
    // 1 expert of H 2880, I 512 T = 300 61 / 65 (253).
    if (up) return launch_mlx<PH_UP, 8, 1, 2>(a, max_work, s, tm);
    return tasks(max_work, a.hidden, 128) <= 200 ? launch_mlx<PH_DOWN, 8, 1, 2>(a, max_work, s, tm) : launch_mlx<PH_DOWN, 8, 2, 2>(a, max_work, s, tm);
  }
  if (quant == Q_MXFP4) {
    if (nt == 1) return up ? launch_mx<PH_UP, 1>(a, max_work, s, tm) : launch_mx<PH_DOWN, 1>(a, max_work, s, tm);
    if (up) return nt == 4 ? launch_mx<PH_UP, 4>(a, max_work, s, tm) : launch_mx<PH_UP, 2>(a, max_work, s, tm);
    return launch_mx<PH_DOWN, 2>(a, max_work, s, tm);
  }
  if (nt == 10) return up ? launch_bf16<PH_UP, 5, 2, 2, 2>(a, max_work, s, tm) : launch_bf16<PH_DOWN, 5, 4, 2, 2>(a, max_work, s, tm);
  return up ? launch_bf16<PH_UP, 2, 1, 2, 1>(a, max_work, s, tm) : launch_bf16<PH_DOWN, 2, 2, 2, 1>(a, max_work, s, tm);
}

}  // namespace hh
