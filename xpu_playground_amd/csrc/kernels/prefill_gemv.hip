// Batched canonical GEMV of the prompt on the FP32 MFMA (prompt chunks past a
// few tokens; pf_gemv in qwen3_ops.hip for the rest).
//
// Out[t][row] for rows of W (M x K, K = 512 NC, M % 16 == 0) and token rows
// In[t] (T x K), bit for bit the decode GEMV's: element k of a dot product
// belongs to canonical lane l = (k / 8) % 64, slot k % 8, chunk k / 512; each
// (lane, slot) chain runs over its chunks by FMA from +0, the slots fold as a
// balanced tree, then the lanes l ^ 32, 16, 8, 4, 2, 1.
// v_mfma_f32_16x16x1_4b (K = 1) is one IEEE FMA per element of four
// independent 16 x 16 tiles, so one instruction advances one slot's chain of
// four canonical lanes (its four blocks) for 16 tokens x 16 rows, and a fold
// is a plain v_add_f32 of two accumulator registers: no lane exchange and no
// per-(row, token) unpacking, which were half of pf_gemv's instructions.
//
// A block owns 16 output rows (EPI 2: 16 gate and 16 up rows) and walks the
// token tiles of its group with the weight fragments held in registers.
// Its wavefronts split the canonical lanes: wavefront q of four takes lanes
// 16 i + 4 q + b for blocks b = 0..3 and steps i = 0, 2, 1, 3 (64 contiguous
// bytes per row and load), so the l ^ 32 and l ^ 16 folds stay in its
// registers; with eight wavefronts each half takes i = 0, 2 or i = 1, 3. The
// l ^ 16 (eight wavefronts), 8 and 4 folds cross wavefronts through LDS, the
// l ^ 2 and 1 folds are the four blocks. Tokens are the first MFMA operand,
// so a lane's result is one row of W and a wavefront's stores are 32
// contiguous bytes per token.
//
// Bound: FP32 MFMA and VALU issue together. The K = 1 MFMA runs 32 FMAs per
// clock and SIMD, the VALU about as many, and the two do not overlap
// (measured: 32 clocks per MFMA plus 2.25 per v_add with two wavefronts), so
// K FMAs and 511 adds per output take 46 TMAC/s at K = 1024 and 60 at K =
// 3072; measured at 2048 tokens 38 and 42, against 20-23 for pf_gemv. Each
// pair of slots unpacks all its operands, then issues its MFMAs back to back,
// then folds: alternating one MFMA with its two unpacks cost 6%.
// At 128 tokens (us, 0.6B rows): QKV 29.0 -> 20.3, o_proj 16.9 -> 13.7,
// [gate; up] 47.5 -> 33.8, down 25.3 -> 19.3. That rate allows 12, 5, 18 and 7
// there: a block's few token tiles do not cover its first weight loads.
#include "qwen3_core.hpp"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// EPI 0: Out = bf16(y); 1: Out = bf16(Out + bf16(y)); 2: W is [gate; up], 2 M
// rows, Out[t][i] = bf16(bf16(silu(bf16(g))) * bf16(u)). HOLD: the weight
// fragments stay in registers over the block's token tiles; otherwise they
// are read again for each tile. Grid 8 ceil(M / 16 / 8) groups: token tile
// group g of `groups` takes tiles [n g / groups, n (g + 1) / groups).
template <int NC, int EPI, bool HOLD, int WAVES>
XPU_DEVICE void pf_rows(const uint16_t *__restrict__ W, const uint16_t *__restrict__ In, uint16_t *Out, uint32_t M,
                        uint32_t T, uint32_t groups) {
  constexpr uint32_t K = 512u * NC;
  constexpr int RT = EPI == 2 ? 2 : 1;  // gate rows and up rows
  __shared__ float xch[2 * 4 * RT * 16 * 64];
  constexpr int S = 16 / WAVES;  // lane groups per wavefront
  const uint32_t lane = xpu::lane_id(), wv_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wave = wv_id & 3u, half = WAVES == 8 ? wv_id >> 2 : 0u;
  const uint32_t ntt = (T + 15u) / 16u, nrt = M / 16u;
  // XCD x (workgroup b runs on XCD b % 8) takes row tiles x, x + 8, ...
  const uint32_t idx = blockIdx.x >> 3;
  const uint32_t rt_i = (idx / groups) * 8u + (blockIdx.x & 7u), grp = idx % groups;
  if (rt_i >= nrt) return;
  const uint32_t tt_beg = ntt * grp / groups, tt_end = ntt * (grp + 1u) / groups;
  if (tt_beg >= tt_end) return;
  const uint32_t o0 = rt_i * 16u;
  const uint32_t j = lane & 15u, b = lane >> 4;
  const uint32_t lcol = (16u * half + 4u * wave + b) * 8u;
  const uint16_t *wp[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) wp[r] = W + static_cast<uint64_t>((r ? M : 0u) + o0 + j) * K + lcol;
  auto xrow = [&](uint32_t tt) { return In + static_cast<uint64_t>(min(16u * tt + j, T - 1u)) * K + lcol; };
  constexpr int order[4] = {0, 2, 1, 3};  // canonical lanes l and l ^ 32, then l ^ 16
  u32x4 wv[HOLD ? S : 1][RT][NC], xv[2][NC];
  auto load_w = [&](int at, int i) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c) wv[at][r][c] = *reinterpret_cast<const u32x4 *>(wp[r] + c * 512 + i * 128);
  };
  auto load_x = [&](int at, const uint16_t *xp, int i) {
#pragma unroll
    for (int c = 0; c < NC; ++c) xv[at][c] = *reinterpret_cast<const u32x4 *>(xp + c * 512 + i * 128);
  };
  auto word = [](const u32x4 &v, int e) { return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; };
  auto elem = [&](const u32x4 &v, int e) {
    return e & 1 ? xpu::hi16<xpu::kBf16>(word(v, e >> 1)) : xpu::lo16<xpu::kBf16>(word(v, e >> 1));
  };
  const uint16_t *xp = xrow(tt_beg);
  // the first step's operands first: its products start while the rest of
  // the weights are still on their way
  if constexpr (HOLD) load_w(0, order[0]);
  load_x(0, xp, order[0]);
  if constexpr (HOLD) {
#pragma unroll
    for (int s = 1; s < S; ++s) load_w(s, order[s]);
  }
  for (uint32_t tt = tt_beg; tt < tt_end; ++tt) {
    const uint16_t *xnext = xrow(min(tt + 1u, tt_end - 1u));
    f32x16 part[RT];
    if constexpr (!HOLD) {
#pragma unroll
      for (int r = 0; r < RT; ++r) asm volatile("" : "+v"(wp[r]));  // the loads stay in the loop
    } else {
#pragma unroll
      for (int q = 0; q < S * RT * NC; ++q)
        asm volatile("" : "+v"(wv[q / (RT * NC)][q / NC % RT][q % NC]));  // unpacked where they are used
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      load_x((s + 1) & 1, s < S - 1 ? xp : xnext, order[(s + 1) % S]);
      if constexpr (!HOLD) load_w(0, order[s]);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const auto &w = wv[HOLD ? s : 0][r];
        f32x16 lvl[2], f;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          // two slots' chains, then the balanced tree over the slots
          float xf[2][NC], wf[2][NC];
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              xf[h][c] = elem(xv[s & 1][c], e + h);
              wf[h][c] = elem(w[c], e + h);
            }
          __builtin_amdgcn_sched_barrier(0);
          f32x16 f0 = {}, f1 = {};
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            f0 = __builtin_amdgcn_mfma_f32_16x16x1f32(xf[0][c], wf[0][c], f0, 0, 0, 0);
            f1 = __builtin_amdgcn_mfma_f32_16x16x1f32(xf[1][c], wf[1][c], f1, 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          f = f0 + f1;
          if (e & 2) {
            f = lvl[0] + f;
            if (e & 4) f = lvl[1] + f;
            else lvl[1] = f;
          } else {
            lvl[0] = f;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (s == 0 || s == 2) {
          part[r] = f;
        } else {
          part[r] = part[r] + f;
          if (s == 1 && r == 0) __syncthreads();  // the previous tile's reads are done
#pragma unroll
          for (int g = 0; g < 16; ++g) xch[((((WAVES == 8 ? half : s >> 1)) * 4 + wave) * RT + r) * 1024 + g * 64 + lane] = part[r][g];
        }
      }
    }
    xp = xnext;
    // lanes l ^ 8 and l ^ 4 across the wavefronts, through LDS
    __syncthreads();
    if (WAVES == 8 && half) continue;
    float y[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      float v[4];
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        float u[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t at = (q * RT + r) * 1024 + (4 * bb + wave) * 64 + lane;
          u[q] = xch[at] + xch[4 * RT * 1024 + at];
        }
        v[bb] = (u[0] + u[2]) + (u[1] + u[3]);
      }
      y[r] = (v[0] + v[2]) + (v[1] + v[3]);
    }
    const uint32_t tok = 16u * tt + 4u * b + wave;
    if (tok < T) {
      uint16_t *out = Out + static_cast<uint64_t>(tok) * M + o0 + j;
      if constexpr (EPI == 0) {
        *out = static_cast<uint16_t>(xpu::f32_to_bf16(y[0]));
      } else if constexpr (EPI == 1) {
        *out = static_cast<uint16_t>(xpu::f32_to_bf16(xpu::bf16_to_f32(*out) + xpu::round_bf16(y[0])));
      } else {
        *out = static_cast<uint16_t>(silu_mul_code(xpu::round_bf16(y[0]), xpu::round_bf16(y[1])));
      }
    }
  }
}

}  // namespace

// xpu_q3_pf_rows_e<EPI>_c<NC>_w<WAVES>, OCC wavefronts per SIMD: without
// spills, four wavefronts per block where eight cost registers or idle
// blocks, eight where K = 1024 leaves room for two such blocks per compute
// unit (128 tokens x 4096 rows: 19.9 -> 18.0 us) or K = 4096 needs the
// weight fragments spread over more wavefronts. K = 4096: checkpoints with
// hidden or query width 4096 and an intermediate size of 512 {2, 4, 6, 8} (the
// 8B shape's 12288 has no down_proj kernel, so its default prompt is stepwise)
#define XPU_Q3_PF_ROWS(EPI, NC, HOLD, WAVES, OCC)                                                                   \
  extern "C" __global__ __launch_bounds__(64 * WAVES, OCC) void xpu_q3_pf_rows_e##EPI##_c##NC##_w##WAVES(           \
      const uint16_t *__restrict__ W, const uint16_t *__restrict__ In, uint16_t *Out, uint32_t M, uint32_t T,       \
      uint32_t groups) {                                                                                            \
    pf_rows<NC, EPI, HOLD, WAVES>(W, In, Out, M, T, groups);                                                        \
  }
XPU_Q3_PF_ROWS(0, 2, true, 8, 4)
XPU_Q3_PF_ROWS(0, 4, true, 4, 2)
XPU_Q3_PF_ROWS(0, 8, true, 8, 2)
XPU_Q3_PF_ROWS(1, 2, true, 8, 4)
XPU_Q3_PF_ROWS(1, 4, true, 4, 2)
XPU_Q3_PF_ROWS(1, 6, true, 4, 2)
XPU_Q3_PF_ROWS(1, 8, true, 8, 2)
XPU_Q3_PF_ROWS(2, 2, true, 4, 2)
XPU_Q3_PF_ROWS(2, 4, true, 8, 2)
XPU_Q3_PF_ROWS(2, 8, false, 8, 2)
