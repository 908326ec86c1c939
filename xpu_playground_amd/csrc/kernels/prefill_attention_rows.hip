// Causal attention of a prompt chunk on the FP32 MFMA, bit for bit the decode
// attention (attention_head in qwen3_core.hpp, qwen3/kernels.hpp:157-192), for
// contexts of one softmax chunk (up to kAttnChunk positions) and chunks that
// start at a multiple of 16 (p0 % 16 == 0, the caller's check: a tile of 16
// queries has to be one group of 16 positions, for the residue classes, the
// diagonal and the last V stage).
//
// One block per (16 queries, head); its eight wavefronts share the LDS rows
// of scores. v_mfma_f32_16x16x1_4b (K = 1) is one IEEE FMA per element of
// four independent 16 x 16 tiles, so it runs the decode attention's FMA
// chains as they are:
// - scores: a score's slot e sums q[8 c + e] k[8 c + e] over chunks c; one
//   instruction advances slot e of 64 keys x 16 queries (blocks = four groups
//   of 16 keys), the slots fold by register adds;
// - softmax: canonical lane L of a row is lane L, holding positions 512 c +
//   8 L + e, as in attention_tail;
// - P.V: residue class t mod 16 = 4 h + k is accumulator h, block k, so each
//   16 positions are four instructions for 16 queries x 16 dims, and a
//   wavefront owns 16 dims for all positions.
// Masked probabilities are exact zeros, which leave a chain as it is (a chain
// starts at +0 and only a non-finite V could change that; see the P.V loop).
//
// Bound: FP32 MFMA issue (2 x 2 n instructions of 32 clocks per 16 queries and
// head over four SIMDs), then LDS latency in P.V: with one stage of V loads
// in flight a 64-position step took 2600 clocks, with four 1640. One block
// per compute unit (accumulators of 128 registers), so a chunk needs at
// least 256 of them. Chunks of 256 queries of a 1531-id prompt, 16 heads: 187
// us per layer with one block per token, 32 us here.
#include "qwen3_core.hpp"

namespace xpu {

constexpr uint32_t kRowsWaves = 8, kRowsKeys = 64, kRowsStage = 64;  // keys per score tile, V rows staged at once
// LDS: 16 rows of score / probability codes (a pitch of 32 bytes mod 128
// spreads the 16 rows over the banks), then the block's Q rows, whose space
// the wavefronts' V stages (64 rows x 16 dims each) take over
constexpr uint32_t kRowsQPitch = kHeadDim * 2 + 16;
XPU_DEVICE constexpr uint32_t rows_pitch(uint32_t n) { return (n + 63u) / 64u * 128u + 32u; }

typedef float f32x16r __attribute__((ext_vector_type(16)));

XPU_DEVICE float code_at(const u32x4 &v, int e) {
  const uint32_t w = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
  return e & 1 ? hi16<kBf16>(w) : lo16<kBf16>(w);
}

}  // namespace xpu

extern "C" __global__ __launch_bounds__(512, 2) void xpu_q3_pf_attention_rows(
    const uint16_t *__restrict__ Q, const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache,
    uint16_t *__restrict__ A, uint32_t p0, uint32_t T, uint32_t heads, uint32_t kv_heads, uint32_t max_seq,
    float scale) {
  using namespace xpu;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  extern __shared__ __align__(128) uint8_t rows_lds[];
  __shared__ float red[kRowsWaves][16];
  const uint32_t lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t j = lane & 15u, b = lane >> 4;
  // the longest contexts first; a kv head's blocks on one XCD for 8 kv heads
  const uint32_t ntiles = (T + 15u) / 16u, group = heads / kv_heads;
  const uint32_t kv = blockIdx.x % kv_heads, head = kv * group + blockIdx.x / kv_heads % group;
  const uint32_t qt = ntiles - 1u - blockIdx.x / heads;
  const uint32_t first = p0 + qt * 16u;          // position of the tile's first query
  const uint32_t last = p0 + min(qt * 16u + 15u, T - 1u);  // position of its last
  const uint32_t n = last + 1u;
  const uint32_t pitch = rows_pitch(p0 + T);
  uint8_t *const srow = rows_lds;
  uint8_t *const tail = rows_lds + 16u * pitch;  // Q rows, then V stages
  const uint64_t head_base = static_cast<uint64_t>(kv) * max_seq * kHeadDim;
  const uint16_t *const kc = kcache + head_base, *const vc = vcache + head_base;
  const uint64_t chunk = static_cast<uint64_t>(max_seq) * 8u;

  // ---- scores: tiles of 64 keys, lane (j, b) <-> key 16 b + j of a tile.
  // Slot e's chain of every (key, query) of the tile is one accumulator of
  // 4 blocks (16 keys each) x 16 queries; register 4 bb + r of lane l holds
  // key 16 bb + 4 (l / 16) + r of query l % 16.
  float vmax = -__builtin_inff();
  const uint32_t ktiles = (n + kRowsKeys - 1u) / kRowsKeys;
  {
    u32x4 kf[16];
    auto load_k = [&](uint32_t kt, int c) {
      const uint64_t t = min(kt * kRowsKeys + lane, n - 1u);
      kf[c] = *reinterpret_cast<const u32x4 *>(kc + c * chunk + t * 8u);
    };
    if (wave < ktiles)
#pragma unroll
      for (int c = 0; c < 16; ++c) load_k(wave, c);
    // Q rows to LDS (rows past the last query repeat it)
    if (threadIdx.x < 256) {
      const uint32_t r = threadIdx.x >> 4, c = threadIdx.x & 15u;
      const uint64_t t = min(qt * 16u + r, T - 1u);
      *reinterpret_cast<u32x4 *>(tail + r * kRowsQPitch + c * 16u) =
          *reinterpret_cast<const u32x4 *>(Q + (t * heads + head) * kHeadDim + c * 8u);
    }
    __syncthreads();
    for (uint32_t kt = wave; kt < ktiles; kt += kRowsWaves) {
      const uint32_t nt = min(kt + kRowsWaves, ktiles - 1u);  // (the last one reads its own tile again)
      f32x16r acc[8];
      auto q_read = [&](int c) { return *reinterpret_cast<const u32x4 *>(tail + j * kRowsQPitch + c * 16u); };
      u32x4 qnext = q_read(0);
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const u32x4 qf = qnext;
        if (c < 15) qnext = q_read(c + 1);
        float kx[8], qx[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          kx[e] = code_at(kf[c], e);
          qx[e] = code_at(qf, e);
        }
        load_k(nt, c);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (c == 0) acc[e] = f32x16r{};
          acc[e] = __builtin_amdgcn_mfma_f32_16x16x1f32(kx[e], qx[e], acc[e], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      const f32x16r s = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
      const uint32_t limit = first + j;  // keys 0 .. limit of this lane's query
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        const uint32_t t = kt * kRowsKeys + 16u * bb + 4u * b;
        uint32_t code[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          code[r] = f32_to_bf16(round_bf16(s[4 * bb + r]) * scale);
          if (t + r <= limit) vmax = fmaxf(vmax, bf16_to_f32(code[r]));
        }
        *reinterpret_cast<u32x2 *>(srow + j * pitch + t * 2u) = u32x2{code[0] | (code[1] << 16), code[2] | (code[3] << 16)};
      }
    }
  }
  // the maximum of query j over the block's lanes (j, *) and wavefronts
  vmax = fmaxf(vmax, xor16_f(vmax));
  vmax = fmaxf(vmax, xor32_f(vmax));
  if (b == 0) red[wave][j] = vmax;
  __syncthreads();

  // V rows t0 .. t0 + 63 of the wavefront's 16 dims (rows past the last query
  // repeat it); the first stages arrive during the softmax
  constexpr int kAhead = 4;
  u32x4 vring[kAhead][2];
  const uint16_t *const vsrc = vc + (2u * wave + (lane >> 5)) * chunk;
  auto load_v = [&](int at, uint32_t t0) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      vring[at][i] = *reinterpret_cast<const u32x4 *>(
          vsrc + static_cast<uint64_t>(min(t0 + 32u * i + (lane & 31u), n - 1u)) * 8u);
  };
  auto store_v = [&](const u32x4 (&v)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<u32x4 *>(tail + wave * kRowsStage * 32u + (32u * i + (lane & 31u)) * 32u + (lane >> 5) * 16u) = v[i];
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) load_v(i, i * kRowsStage);

  // ---- softmax of two queries per wavefront: canonical lane L = lane holds
  // positions 512 c + 8 L + e of its row. The probabilities go back over the
  // scores, each 16 of them in the order the P.V operand reads: position
  // 4 h + k of the 16 at place 4 k + h.
  {
    constexpr int kChunks = kAttnChunk / 512;
    float ex[2][kChunks][8], mx[2], inv[2];
    uint32_t len[2];  // (rows past the last query are not stored)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t row = wave + i * kRowsWaves;
      len[i] = min(first + row, last) + 1u;
      mx[i] = red[0][row];
#pragma unroll
      for (uint32_t w = 1; w < kRowsWaves; ++w) mx[i] = fmaxf(mx[i], red[w][row]);
    }
    float acc[2][8] = {};
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      if (c * 512u >= n) break;  // uniform
      const uint32_t t = c * 512u + lane * 8u;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint8_t *const p = srow + (wave + i * kRowsWaves) * pitch;
        const u32x4 v = t < n ? *reinterpret_cast<const u32x4 *>(p + t * 2u) : u32x4{0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          ex[i][c][e] = t + e < len[i] ? canonical_exp_nonpos(code_at(v, e) - mx[i]) : 0.0f;
          acc[i][e] = acc[i][e] + ex[i][c][e];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) inv[i] = 1.0f / (0.0f + wave_butterfly(fold8(acc[i])));
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      if (c * 512u >= n) break;  // uniform
      const uint32_t t = c * 512u + lane * 8u;
      if (t >= (n + 15u) / 16u * 16u) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        uint8_t *const g = srow + (wave + i * kRowsWaves) * pitch + (t & ~15u) * 2u + (lane & 1u) * 4u;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          *reinterpret_cast<uint32_t *>(g + k * 8u) =
              f32_to_bf16(ex[i][c][k] * inv[i]) | (f32_to_bf16(ex[i][c][k + 4] * inv[i]) << 16);
      }
    }
  }
  __syncthreads();

  // ---- P.V: wavefront w owns dims 16 w .. 16 w + 15 (cache chunks 2 w and
  // 2 w + 1); accumulator h, block k is residue class 4 h + k of t mod 16
  f32x16r pv[4] = {};
  {
    uint8_t *const stage = tail + wave * kRowsStage * 32u;
    const uint32_t stage_at = lds_addr(stage);
    // P.V of the 16 positions from t, staged at row m of the stage
    auto p_read = [&](uint32_t t) { return *reinterpret_cast<const u32x2 *>(srow + j * pitch + t * 2u + b * 8u); };
    auto v_read = [&](uint32_t m) {
      const uint32_t at = stage_at + (m + 4u * (j >> 2) + b) * 32u + (j & 3u) * 8u;
      return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(at)));
    };
    auto products = [&](const u32x2 &pc, const u32x2 &vv) {
      const float pf[4] = {lo16<kBf16>(pc.x), hi16<kBf16>(pc.x), lo16<kBf16>(pc.y), hi16<kBf16>(pc.y)};
      const float vf[4] = {lo16<kBf16>(vv.x), hi16<kBf16>(vv.x), lo16<kBf16>(vv.y), hi16<kBf16>(vv.y)};
#pragma unroll
      for (int h = 0; h < 4; ++h) pv[h] = __builtin_amdgcn_mfma_f32_16x16x1f32(pf[h], vf[h], pv[h], 0, 0, 0);
    };
    // positions before the tile's own 16, 64 at a time, with the loads of
    // kAhead stages in flight
    uint32_t t0 = 0;
    auto whole = [&](int at) {
      store_v(vring[at]);
      load_v(at, t0 + kAhead * kRowsStage);
      __builtin_amdgcn_wave_barrier();
      u32x2 pc[4], vv[4];
#pragma unroll
      for (uint32_t m = 0; m < 4; ++m) {
        pc[m] = p_read(t0 + 16u * m);
        vv[m] = v_read(16u * m);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) products(pc[m], vv[m]);
      __builtin_amdgcn_wave_barrier();
      t0 += kRowsStage;
    };
    for (; t0 + kAhead * kRowsStage <= first;)
#pragma unroll
      for (int at = 0; at < kAhead; ++at) whole(at);
    int left = 0;
#pragma unroll
    for (int at = 0; at + 1 < kAhead; ++at)
      if (t0 + kRowsStage <= first) {  // uniform
        whole(at);
        left = at + 1;
      }
    // the rest, with the tile's own positions last, zeros past the last
    // query. An infinity or NaN among their V rows must not meet the zero
    // probability of an earlier query: then those 16 go one query and
    // position at a time.
    u32x4 rest[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      rest[i] = left == 0 ? vring[0][i] : left == 1 ? vring[1][i] : left == 2 ? vring[2][i] : vring[3][i];
      if (t0 + 32u * i + (lane & 31u) >= n) rest[i] = u32x4{0, 0, 0, 0};
    }
    store_v(rest);
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int w = 0; w < 4; ++w)
        odd = odd || (t0 + 32u * i + (lane & 31u) >= first &&
                      ((rest[i][w] & 0x7f80u) == 0x7f80u || (rest[i][w] & 0x7f800000u) == 0x7f800000u));
    const bool one_by_one = __builtin_amdgcn_ballot_w64(odd) != 0;
    __builtin_amdgcn_wave_barrier();
    for (uint32_t m = 0; t0 + m < n; m += 16u) {
      if (t0 + m < first || !one_by_one) {
        products(p_read(t0 + m), v_read(m));
        continue;
      }
#pragma unroll
      for (uint32_t h = 0; h < 4; ++h)
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          const float x = bf16_to_f32(*reinterpret_cast<const uint16_t *>(stage + (m + 4u * h + k) * 32u + j * 2u));
#pragma unroll
          for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t q = 4u * b + r;
            const uint8_t *const at = srow + q * pitch + (t0 + m + 4u * k + h) * 2u;
            const float f = __builtin_fmaf(bf16_to_f32(*reinterpret_cast<const uint16_t *>(at)), x, pv[h][4 * k + r]);
            pv[h][4 * k + r] = 4u * h + k <= q ? f : pv[h][4 * k + r];
          }
        }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float s[4];
#pragma unroll
    for (int h = 0; h < 4; ++h)
      s[h] = ((0.0f + pv[h][r]) + (0.0f + pv[h][4 + r])) + ((0.0f + pv[h][8 + r]) + (0.0f + pv[h][12 + r]));
    const uint32_t q = qt * 16u + 4u * b + r;
    if (q < T)
      A[(static_cast<uint64_t>(q) * heads + head) * kHeadDim + wave * 16u + j] =
          static_cast<uint16_t>(f32_to_bf16((s[0] + s[1]) + (s[2] + s[3])));
  }
}
