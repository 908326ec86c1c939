// GEMM entry points: xpu_gemm (kernel launch) and the run_gemm command-line
// program (reference gemm.cpp and the GEMM mode of level_zero/peak_l0.cpp:895-949).
#include "../../include/xpu_kernels.h"
#include "host_common.hpp"
#include "runtime_internal.hpp"

#include <algorithm>
#include <cstdlib>
#include <iomanip>
#include <iostream>
#include <type_traits>

using xpu::set_error;

namespace {

uint64_t round_up8(uint64_t v) { return (v + 7) & ~uint64_t{7}; }

// Block tiles of the MFMA kernels (kernels/gemm.hip), largest first. Rates
// are FLOP per compute unit relative to the large tile, measured with one
// block per busy compute unit: a 224 x 256 block runs at 0.89-0.97 (median
// 0.93 over six shapes; its four wavefronts each read all 224 A rows, and
// its B rows cost as much as in the 256 x 256 block); a 128 x 256 block at
// 0.85; a 128 x 128 block alone at 0.59, and two of them sharing a unit (its
// LDS holds two) at 0.82 together.
struct GemmTile {
  const char *tag;  // kernel name part: xpu_gemm_<type><tag>[_odd]_dma[u][_edge]
  uint32_t rows, cols;
  uint32_t per_cu;   // blocks one compute unit holds at once
  double solo_rate;  // one block on a unit
  double pair_rate;  // two blocks on a unit, together (per_cu == 2)
  bool odd_forms;    // has _odd kernels (an odd count, 3 or more, of 64-deep K-slices)
  bool nt_forms;     // has [n][k] (_nt) kernels for the prompt projections
};
constexpr GemmTile kTiles[] = {{"", 256, 256, 1, 1.0, 0.0, true, true},
                               {"_m224", 224, 256, 1, 0.93, 0.0, true, false},
                               {"_m128", 128, 256, 1, 0.85, 0.0, false, true},
                               {"_t128", 128, 128, 2, 0.59, 0.82, false, true}};

// The tile with the least estimated time. The blocks spread evenly over the
// compute units, so the busiest unit gets w = ceil(tiles / CUs) of them and
// runs them in pairs where it holds two. The larger tile wins ties. The
// reference takes its small tile when M or N is below 2560 (gemm.cpp:145);
// here the 256 x 256 tile stays where it gives each compute unit one block
// (4096^3), 224 x 256 takes outputs where it still does and cuts each unit's
// work by 1/8 (3000 x 4097: 238 blocks instead of 204), and outputs that
// leave most compute units idle take a smaller one.
// (32-bit divisions: the plan is host time of every call)
uint32_t ceil_div(uint32_t a, uint32_t b) { return a ? (a - 1) / b + 1 : 0; }

uint64_t ceil_div(uint64_t a, uint32_t b) {
  return a >> 32 ? (a + b - 1) / b : ceil_div(static_cast<uint32_t>(a), b);
}

uint64_t tile_count(uint32_t M, uint32_t N, uint32_t rows, uint32_t cols) {
  return static_cast<uint64_t>(ceil_div(M, rows)) * ceil_div(N, cols);
}

double tile_cost(const GemmTile &t, uint32_t compute_units, uint32_t M, uint32_t n_cols) {
  const uint64_t w = ceil_div(tile_count(M, n_cols, t.rows, t.cols), std::max(1u, compute_units));
  const double area = static_cast<double>(t.rows) * t.cols;
  return t.per_cu == 2 ? static_cast<double>(w / 2) * 2.0 * area / t.pair_rate +
                             static_cast<double>(w % 2) * area / t.solo_rate
                       : static_cast<double>(w) * area / t.solo_rate;
}

const GemmTile &choose_tile(uint32_t compute_units, uint32_t M, uint32_t n_cols, bool nt = false) {
  const GemmTile *best = &kTiles[0];
  double best_cost = 0;
  for (const GemmTile &t : kTiles) {
    if (nt && !t.nt_forms) continue;
    const double cost = tile_cost(t, compute_units, M, n_cols);
    if (&t == &kTiles[0] || cost < best_cost) {
      best = &t;
      best_cost = cost;
    }
  }
  return *best;
}

// The most ranges xpu_gemm cuts K into (1: whole K): where 128 x 128 tiles
// leave at least half the compute units idle, about CUs / tiles ranges of a
// multiple of 2 slices, for K of 24 slices or more or partials of at most
// 4 MiB (1024^3, 16 slices and 16 MB of partials, is slower split at any
// tile: 12.8 us against 6.7).
uint32_t max_splits(uint32_t compute_units, const GemmTile &tile, uint32_t M, uint32_t N, uint32_t K) {
  const uint64_t tiles = tile_count(M, N, 128, 128);
  const uint32_t slices = (K + 63) / 64;
  if (tile.rows != 128 || tile.cols != 128 || tiles * 2 > compute_units || slices < 8) return 1;
  const uint32_t want = ceil_div(compute_units, static_cast<uint32_t>(tiles));
  const uint32_t spl = (ceil_div(slices, want) + 1) / 2 * 2, splits = ceil_div(slices, spl);
  const uint64_t bytes = static_cast<uint64_t>(splits) * M * ((N + 3) / 4 * 4) * 4;
  return splits >= 2 && (slices >= 24 || bytes <= (4ull << 20)) ? splits : 1;
}

// The small tiles (kernels/gemm.hip): stages
// (slices per group) and us per 64-deep slice with w blocks on the busiest
// unit, w * pair_us for w >= 2.
struct SmallTile {
  const char *tag;
  uint32_t rows, cols, stages;
  double solo_us, pair_us;
};
constexpr SmallTile kSmallTiles[] = {{"_m32", 32, 128, 4, 0.26, 0.27}, {"_m64", 64, 128, 3, 0.33, 0.36}};

struct SmallPlan {
  const SmallTile *tile = nullptr;  // null: the tile of choose_tile, whole K
  uint64_t tiles = 0;
  uint32_t splits = 1, slices = 0;  // K ranges, and slices per range
};

// A small tile, with K whole or in up to `limit` ranges, where its estimated
// time is below the chosen tile's: us per slice (a group of slices past K
// costs as much) over the busiest unit's blocks, plus for a split the second
// launch (2 us), each range's load in the reduction (0.12 us) and the
// partials' round trip (0.55 us per MB). Fitted to 19 swept shapes, bf16 and
// back to back: it takes the measured fastest plan or one within 8% of it.
// Against 128 x 128 tiles, K split as max_splits says: 24 x 4096 x 4096 (8
// ranges of 32 x 128) 12.0 -> 9.1 us, 64 x 1024 x 4096 13.1 -> 8.1, 512^3
// (whole K) 8.9 -> 4.3, 1024^3 9.5 -> 6.7, 300 x 3000 x 3000 20.5 -> 17.3,
// 1500 x 1000 x 600 (64 x 128) 7.7 -> 6.6; 2048 x 2048 x 512 stays (8.0
// against 9.0).
SmallPlan choose_small(uint32_t compute_units, const GemmTile &tile, uint32_t M, uint32_t N, uint32_t K,
                       uint32_t limit) {
  SmallPlan plan;
  if (tile.rows > 128) return plan;
  const uint32_t slices = (K + 63) / 64, cus = std::max(1u, compute_units);
  // 0.375 us is a slice's share of 128 x 128 outputs at the large tile's rate
  double best = tile_cost(tile, cus, M, N) / (128 * 128) * 0.375 * slices;
  const double mb = static_cast<double>(M) * ((N + 3) / 4 * 4) * 4e-6;
  auto consider = [&](auto index) {
    constexpr const SmallTile &t = kSmallTiles[index];  // (its divisors are constants)
    const uint64_t tiles = tile_count(M, N, t.rows, t.cols);
    // as many ranges as fill the units, then fewer, halving
    for (uint32_t want = limit == 1 || tiles >= cus ? 1u : std::min(limit, cus / static_cast<uint32_t>(tiles));;
         want /= 2) {
      const uint32_t per = ceil_div(want == 1 ? slices : ceil_div(slices, want), t.stages) * t.stages;
      const uint32_t splits = want == 1 ? 1 : ceil_div(slices, per);
      const uint64_t w = tiles * splits <= cus ? 1 : ceil_div(tiles * splits, cus);
      const double us = per * (w == 1 ? t.solo_us : static_cast<double>(w) * t.pair_us) +
                        (splits >= 2 ? 2.0 + splits * (0.12 + 0.55 * mb) : 0.0);
      if (us < best) {
        best = us;
        plan = {&t, tiles, splits, per};
      }
      if (want <= 1) break;
    }
  };
  consider(std::integral_constant<size_t, 0>{});
  consider(std::integral_constant<size_t, 1>{});
  return plan;
}

}  // namespace

namespace xpu {

int gemm_run(xpu_runtime *rt, int dtype, const void *A, const void *B, void *C, uint32_t M, uint32_t N, uint32_t K,
             void *fixed_workspace, uint64_t fixed_capacity) {
  if (!rt || !A || !B || !C) return set_error(XPU_ERR_INVALID, "xpu_gemm: null argument");
  if (dtype != XPU_DTYPE_BF16 && dtype != XPU_DTYPE_FP16)
    return set_error(XPU_ERR_INVALID, "xpu_gemm: dtype must be bf16 (0) or fp16 (1)");
  if (M == 0 || N == 0 || K == 0) return set_error(XPU_ERR_INVALID, "xpu_gemm: M, N, K must be positive");
  // 32-bit buffer offsets: 256 rows of A and 64 rows of B per K-slice
  const uint64_t kp = round_up8(K), np = round_up8(N);
  if (kp * 256 * 2 >= (1ull << 31) || np * 64 * 2 >= (1ull << 31))
    return set_error(XPU_ERR_INVALID, "xpu_gemm: K must be below 4M and N below 16M");
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C)) % 2)
    return set_error(XPU_ERR_INVALID, "xpu_gemm: A, B and C must be 2-byte aligned (16-bit elements)");
  // A and B are read in place at any K, N and alignment: the kernels stage
  // unaligned rows by LDS-DMA and handle the K and N edges themselves
  // (kernels/gemm.hip); nothing is copied or padded
  const void *a_use = A, *b_use = B;
  const uint32_t k_run = K, n_run = N;
  const bool c16 = reinterpret_cast<uintptr_t>(C) % 16 == 0 && N % 8 == 0;
  const GemmTile &tile = choose_tile(rt->compute_units, M, n_run);
  // K % 8 != 0 or N odd: the _edge form cuts the chunk that straddles
  // column K and restores the elements the range check cuts at the
  // operands' ends (kernels/gemm.hip)
  const bool edge = K % 8 != 0 || N % 2 != 0;
  const char *dt = dtype ? "fp16" : "bf16";
  // Where K may be split, the FP32 partials [split][M][pitch] go into the
  // workspace (the runtime's, or the caller's fixed array) and one reduction
  // in split order rounds to the output type. Within the GEMM's tolerance,
  // not bit-equal to one chain (the FP32 sum is re-associated at the range
  // boundaries). The fixed array's limit is stated on max_splits' partials,
  // which no plan exceeds, so that the accepted shapes do not depend on the
  // tile a plan takes.
  const uint32_t pitch = (N + 3) / 4 * 4;
  const uint64_t split_bytes = static_cast<uint64_t>(M) * pitch * 4;
  const uint32_t limit = max_splits(rt->compute_units, tile, M, N, K);
  if (fixed_workspace && limit >= 2 && limit * split_bytes > fixed_capacity)
    return set_error(XPU_ERR_INVALID, "xpu_gemm_noalloc: K may be split in up to " + std::to_string(limit) +
                                          " ranges at this shape, whose partials would need " +
                                          std::to_string(limit * split_bytes) + " bytes, above the " +
                                          std::to_string(fixed_capacity) + "-byte scratch array");
  if (const SmallPlan plan = choose_small(rt->compute_units, tile, M, N, K, limit); plan.tile) {
    const std::string stem = std::string("xpu_gemm_") + dt + plan.tile->tag;
    const bool part = plan.splits >= 2;
    const std::string name = stem + (part ? "_part_dma" : c16 ? "_dma" : "_dmau") + (edge ? "_edge" : "");
    const xpu::KernelInfo *k = rt->find_exact(name);
    const xpu::KernelInfo *kr = part ? rt->find_exact("xpu_gemm_splitk_reduce_any") : nullptr;
    if (!k || (part && !kr)) return set_error(XPU_ERR_NOT_FOUND, "kernel is absent from module: " + name);
    void *out = C;
    uint32_t kb = K, ld_out = N, n_out = N;
    int rc = XPU_OK;
    if (part) {
      out = fixed_workspace;
      if (!out && (rc = rt->scratch(plan.splits * split_bytes, &out))) return rc;
      kb = plan.slices;
      ld_out = pitch;
    }
    const xpu_kernel_arg args[] = {{8, &a_use}, {8, &b_use}, {8, &out},    {4, &M},    {4, &n_run},
                                   {4, &k_run}, {4, &kb},    {4, &ld_out}, {4, &n_out}};
    if ((rc = rt->launch(*k, static_cast<uint32_t>(plan.tiles * plan.splits), 1, 256, 0, args, 9)) || !part) return rc;
    const uint64_t threads = static_cast<uint64_t>(M) * (pitch / 4);
    const uint32_t grid = static_cast<uint32_t>(std::min<uint64_t>((threads + 255) / 256, rt->compute_units * 8ull));
    uint32_t ldc = N, ns = plan.splits, d = static_cast<uint32_t>(dtype);
    const xpu_kernel_arg rargs[] = {{8, &out}, {8, &C}, {4, &M}, {4, &n_run}, {4, &ld_out}, {4, &ldc}, {4, &ns}, {4, &d}};
    return rt->launch(*kr, grid, 1, 256, 0, rargs, 8);
  }
  // the 256 x 256 and 224 x 256 kernels come in a form for an odd number (3
  // or more) of 64-deep K-slices, which skips the slice of zeros that closes
  // the last pair and the last slice's k-steps past K
  const uint32_t slices = (k_run + 63) / 64;
  const bool odd = tile.odd_forms && slices % 2 == 1 && slices >= 3;
  const std::string name = std::string("xpu_gemm_") + dt + tile.tag + (odd ? "_odd" : "") +
                           (c16 ? "_dma" : "_dmau") + (edge ? "_edge" : "");
  const xpu::KernelInfo *k = rt->find_exact(name);
  if (!k) return set_error(XPU_ERR_NOT_FOUND, "kernel is absent from module: " + name);
  const uint64_t tiles = ((static_cast<uint64_t>(M) + tile.rows - 1) / tile.rows) *
                         ((static_cast<uint64_t>(n_run) + tile.cols - 1) / tile.cols);
  if (tiles > 0x7fffffffu) return set_error(XPU_ERR_INVALID, "xpu_gemm: too many tiles");
  const uint32_t kb = K, ldc = N, n_out = N;
  const xpu_kernel_arg args[] = {{8, &a_use}, {8, &b_use}, {8, &C},   {4, &M},     {4, &n_run},
                                 {4, &k_run}, {4, &kb},    {4, &ldc}, {4, &n_out}};
  return rt->launch(*k, static_cast<uint32_t>(tiles), 1, 256, 0, args, 9);
}

}  // namespace xpu

// For the tests of the dispatch: the tile, the number of K ranges and the slices
// per range (all of K if 1) that xpu_gemm takes on a GPU with that many compute
// units, and the largest number of ranges. Not part of the C ABI.
extern "C" void xpu_internal_gemm_plan(uint32_t compute_units, uint32_t M, uint32_t N, uint32_t K, uint32_t *rows,
                                       uint32_t *cols, uint32_t *splits, uint32_t *slices, uint32_t *limit) {
  const GemmTile &tile = choose_tile(compute_units, M, N);
  *limit = max_splits(compute_units, tile, M, N, K);
  const SmallPlan plan = choose_small(compute_units, tile, M, N, K, *limit);
  *rows = plan.tile ? plan.tile->rows : tile.rows;
  *cols = plan.tile ? plan.tile->cols : tile.cols;
  *splits = plan.splits;
  *slices = plan.splits >= 2 ? plan.slices : (K + 63) / 64;
}

namespace xpu {

// C[M x N] = A[M x K] W^T for W given [N][K] (bf16, K and N multiples of 8,
// every pointer 16-byte aligned, row strides K, K and N), the projections of
// the batched prompt (qwen3_engine.cpp); residual: C = bf16(C + bf16(A W^T)).
// The block tile and the odd-slice form are chosen as for xpu_gemm.
uint64_t gemm_nt_workspace_bound(const xpu_runtime *rt) {
  // split K only with tiles <= CUs / 2, and splits <= ceil(CUs / tiles):
  // splits x tiles <= CUs + tiles <= 1.5 CUs tiles of 128 x 64 FP32
  return (static_cast<uint64_t>(rt->compute_units) * 3 / 2 + 1) * 128 * 64 * 4;
}

int gemm_nt(xpu_runtime *rt, const void *A, const void *W, void *C, uint32_t M, uint32_t N, uint32_t K,
            bool residual, const void *norm_w, void *Xn, float eps, bool *normed) {
  if (normed) *normed = false;
  if (!rt || !A || !W || !C) return set_error(XPU_ERR_INVALID, "gemm_nt: null argument");
  if (M == 0 || N == 0 || K == 0 || K % 8 || N % 8 || (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W) |
                                                       reinterpret_cast<uintptr_t>(C)) % 16)
    return set_error(XPU_ERR_INVALID, "gemm_nt: needs positive M, N, K with K, N multiples of 8 and 16-byte aligned "
                                      "operands");
  if (static_cast<uint64_t>(K) * 256 * 2 >= (1ull << 31) || static_cast<uint64_t>(N) >= (1u << 24))
    return set_error(XPU_ERR_INVALID, "gemm_nt: K must be below 4M and N below 16M");
  const GemmTile &tile = choose_tile(rt->compute_units, M, N, true);
  const uint32_t slices = (K + 63) / 64;
  const bool odd = tile.tag[0] == '\0' && slices % 2 == 1 && slices >= 3;
  auto count = [&](uint32_t rows, uint32_t cols) {
    return ((static_cast<uint64_t>(M) + rows - 1) / rows) * ((static_cast<uint64_t>(N) + cols - 1) / cols);
  };
  uint64_t tiles = count(tile.rows, tile.cols);
  std::string tag = tile.tag;
  // 128 x 64 tiles where even 128 x 128 ones leave compute units idle
  if (tag == "_t128" && tiles < rt->compute_units) {
    tag = "_n64";
    tiles = count(128, 64);
  }
  // Split K where even 128 x 64 tiles leave half the compute units idle (a
  // short prompt's projections): splits of a multiple of 4 slices (the
  // kernel's stage group) so that tiles x splits about fills the CUs; FP32
  // partials in the workspace, then one reduction (split order) that
  // rounds and applies the residual.
  if (tag == "_n64" && tiles * 2 <= rt->compute_units) {
    const uint32_t want = static_cast<uint32_t>((rt->compute_units + tiles - 1) / tiles);
    const uint32_t spl = ((slices + want - 1) / want + 3) / 4 * 4, splits = (slices + spl - 1) / spl;
    if (splits >= 2) {
      const xpu::KernelInfo *kp = rt->find_exact("xpu_gemm_bf16_n64_nt_part_dma");
      const xpu::KernelInfo *kr = rt->find_exact("xpu_gemm_splitk_reduce");
      if (!kp || !kr) return set_error(XPU_ERR_NOT_FOUND, "kernel is absent from module: split-K GEMM");
      void *part = nullptr;
      int rc = rt->scratch(static_cast<uint64_t>(splits) * M * N * 4, &part);
      if (rc) return rc;
      uint32_t kb = spl, ldc = N, n_out = N, res = residual ? 1u : 0u, nsplit = splits;
      const xpu_kernel_arg pargs[] = {{8, &A}, {8, &W},  {8, &part}, {4, &M},    {4, &N},
                                      {4, &K}, {4, &kb}, {4, &ldc},  {4, &n_out}};
      if ((rc = rt->launch(*kp, static_cast<uint32_t>(tiles * splits), 1, 256, 0, pargs, 9))) return rc;
      const xpu::KernelInfo *kn = rt->find_exact("xpu_gemm_splitk_reduce_norm");
      if (norm_w && Xn && normed && kn && (N == 512 || N == 1024)) {
        const xpu_kernel_arg nargs[] = {{8, &part}, {8, &C},      {4, &M},  {4, &N},  {4, &nsplit},
                                        {4, &res},  {8, &norm_w}, {8, &Xn}, {4, &eps}};
        if ((rc = rt->launch(*kn, (M + 3) / 4, 1, 256, 0, nargs, 9))) return rc;
        *normed = true;
        return XPU_OK;
      }
      const uint64_t threads = static_cast<uint64_t>(M) * N / 8;
      const uint32_t grid = static_cast<uint32_t>(std::min<uint64_t>((threads + 255) / 256, rt->compute_units * 8ull));
      const xpu_kernel_arg rargs[] = {{8, &part}, {8, &C}, {4, &M}, {4, &N}, {4, &nsplit}, {4, &res}};
      return rt->launch(*kr, grid, 1, 256, 0, rargs, 6);
    }
  }
  const std::string name = "xpu_gemm_bf16" + tag + (odd ? "_odd" : "") + "_nt" + (residual ? "_res" : "") + "_dma";
  const xpu::KernelInfo *k = rt->find_exact(name);
  if (!k) return set_error(XPU_ERR_NOT_FOUND, "kernel is absent from module: " + name);
  uint32_t kb = K, ldc = N, n_out = N;
  const xpu_kernel_arg args[] = {{8, &A}, {8, &W},  {8, &C},   {4, &M},    {4, &N},
                                 {4, &K}, {4, &kb}, {4, &ldc}, {4, &n_out}};
  return rt->launch(*k, static_cast<uint32_t>(tiles), 1, 256, 0, args, 9);
}

}  // namespace xpu

extern "C" int xpu_gemm(xpu_runtime *rt, int dtype, const void *A, const void *B, void *C,
                        uint32_t M, uint32_t N, uint32_t K) {
  return xpu::gemm_run(rt, dtype, A, B, C, M, N, K, nullptr, 0);
}

extern "C" int xpu_gemm_tile(const xpu_runtime *rt, uint32_t M, uint32_t N, uint32_t *rows, uint32_t *cols) {
  if (!rt || !rows || !cols) return set_error(XPU_ERR_INVALID, "xpu_gemm_tile: null argument");
  if (M == 0 || N == 0) return set_error(XPU_ERR_INVALID, "xpu_gemm_tile: M and N must be positive");
  const GemmTile &t = choose_tile(rt->compute_units, M, static_cast<uint32_t>(round_up8(N)));
  *rows = t.rows;
  *cols = t.cols;
  return XPU_OK;
}

namespace {

struct GemmOptions {
  uint32_t m = 4096, n = 4096, k = 4096;  // gemm.cpp:19
  unsigned iterations = 20, warmups = 5;  // gemm.cpp:20
  int dtype = XPU_DTYPE_BF16;
  // gemm.cpp:81-85: the reference's only input is A = 0.5, B = 0.25 with the
  // known answer 0.125 * K (:109-117), so it is the default here too;
  // --init uniform selects the seeded U[-1,1] data of the benchmark
  // configurations (checked against an FP64 host product)
  bool constant_init = true;
  uint64_t seed = 1;
  uint32_t check_rows = 64;
};

[[noreturn]] void gemm_usage(const char *program, int status) {
  std::ostream &out = status ? std::cerr : std::cout;
  out << "Usage: " << program << " [--size N | --m M --n N --k K] [--type bf16|fp16]\n"
      << "       [--iterations N] [--warmups N] [--init constant|uniform] [--seed N]\n"
      << "       [--check-rows N]\n";
  std::exit(status);
}

// gemm.cpp:40-59
GemmOptions parse_gemm(int argc, char **argv) {
  GemmOptions o;
  for (int i = 1; i < argc; ++i) {
    const std::string_view arg(argv[i]);
    if (arg == "-h" || arg == "--help") gemm_usage(argv[0], 0);
    if (++i == argc) throw std::invalid_argument(std::string(arg) + " requires a value");
    const std::string_view value(argv[i]);
    if (arg == "--size") o.m = o.n = o.k = xpu::parse_positive<uint32_t>(value, arg);
    else if (arg == "--m") o.m = xpu::parse_positive<uint32_t>(value, arg);
    else if (arg == "--n") o.n = xpu::parse_positive<uint32_t>(value, arg);
    else if (arg == "--k") o.k = xpu::parse_positive<uint32_t>(value, arg);
    else if (arg == "--iterations") o.iterations = xpu::parse_positive<unsigned>(value, arg);
    else if (arg == "--warmups") o.warmups = xpu::parse_positive<unsigned>(value, arg);
    else if (arg == "--type" && value == "fp16") o.dtype = XPU_DTYPE_FP16;
    else if (arg == "--type" && value == "bf16") o.dtype = XPU_DTYPE_BF16;
    else if (arg == "--type") throw std::invalid_argument("--type must be bf16 or fp16");
    else if (arg == "--init" && value == "uniform") o.constant_init = false;
    else if (arg == "--init" && value == "constant") o.constant_init = true;
    else if (arg == "--init") throw std::invalid_argument("--init must be uniform or constant");
    else if (arg == "--seed") o.seed = xpu::parse_unsigned<uint64_t>(value, arg);
    else if (arg == "--check-rows") o.check_rows = xpu::parse_unsigned<uint32_t>(value, arg);
    else throw std::invalid_argument("unknown option: " + std::string(arg));
  }
  return o;
}

void check(int rc) {
  if (rc) throw std::runtime_error(xpu_last_error());
}

struct RuntimeGuard {
  xpu_runtime *rt = nullptr;
  ~RuntimeGuard() { xpu_rt_destroy(rt); }
};

}  // namespace

extern "C" int run_gemm(int argc, char **argv) {
  try {
    const GemmOptions o = parse_gemm(argc, argv);
    RuntimeGuard guard;
    check(xpu_rt_create(nullptr, -1, &guard.rt));
    xpu_runtime *rt = guard.rt;
    std::cout << "Device: " << rt->name << " (" << rt->arch << ", " << rt->compute_units << " CUs)\n";
    const uint64_t as = static_cast<uint64_t>(o.m) * o.k, bs = static_cast<uint64_t>(o.k) * o.n,
                   cs = static_cast<uint64_t>(o.m) * o.n;
    check(xpu_rt_require_device_and_memory(rt, (as + bs + cs) * 2));
    void *a = nullptr, *b = nullptr, *c = nullptr;
    check(xpu_rt_alloc(rt, as * 2, 256, &a));
    check(xpu_rt_alloc(rt, bs * 2, 256, &b));
    check(xpu_rt_alloc(rt, cs * 2, 256, &c));
    if (o.constant_init) {
      // gemm.cpp:81-85: A = 0.5, B = 0.25 (no padding needed here)
      const uint16_t ha = xpu::encode16(0.5f, o.dtype), hb = xpu::encode16(0.25f, o.dtype);
      std::vector<uint16_t> fill(std::max(as, bs));
      std::fill(fill.begin(), fill.begin() + as, ha);
      check(xpu_rt_copy_to_device(rt, a, fill.data(), as * 2));
      std::fill(fill.begin(), fill.begin() + bs, hb);
      check(xpu_rt_copy_to_device(rt, b, fill.data(), bs * 2));
    } else {
      check(xpu_fill_uniform(rt, o.dtype, a, as, o.seed));
      check(xpu_fill_uniform(rt, o.dtype, b, bs, o.seed + 1));
    }
    check(xpu_rt_memset(rt, c, 0, cs * 2));
    for (unsigned i = 0; i < o.warmups; ++i) check(xpu_gemm(rt, o.dtype, a, b, c, o.m, o.n, o.k));
    check(xpu_rt_synchronize(rt));
    void *start = nullptr, *stop = nullptr;
    check(xpu_rt_event_create(rt, &start));
    check(xpu_rt_event_create(rt, &stop));
    // gemm.cpp:102-108: one timed launch per iteration, 2*M*N*K FLOP
    const double flops = 2.0 * o.m * o.n * o.k;
    std::vector<double> rates, times;
    for (unsigned i = 0; i < o.iterations; ++i) {
      check(xpu_rt_event_record(rt, start));
      check(xpu_gemm(rt, o.dtype, a, b, c, o.m, o.n, o.k));
      check(xpu_rt_event_record(rt, stop));
      float ms = 0;
      check(xpu_rt_event_elapsed_ms(start, stop, &ms));
      times.push_back(ms * 1e-3);
      rates.push_back(flops / (ms * 1e-3) / 1e12);
    }
    xpu_rt_event_destroy(start);
    xpu_rt_event_destroy(stop);

    // Verification: constant init checks 0.125 * K (gemm.cpp:109-117); the
    // uniform init checks the first rows against an FP64 host product,
    // rounded to the output type, within 2 output ulps + gamma_K sum|a b|.
    double err2 = 0, ref2 = 0, max_ulps = 0;
    const uint32_t rows = std::min(o.m, o.check_rows);
    if (rows) {
      std::vector<uint16_t> hc(static_cast<size_t>(rows) * o.n), ha(static_cast<size_t>(rows) * o.k),
          hb(bs);
      check(xpu_rt_copy_from_device(rt, hc.data(), c, hc.size() * 2));
      if (o.constant_init) {
        const float expected = o.k * 0.125f, tolerance = std::max(0.5f, expected * 0.01f);
        for (uint16_t v : hc)
          if (std::fabs(xpu::decode16(v, o.dtype) - expected) > tolerance)  // gemm.cpp:111-117
            throw std::runtime_error("GEMM verification failed: expected " + std::to_string(expected) + ", got " +
                                     std::to_string(xpu::decode16(v, o.dtype)));
      } else {
        check(xpu_rt_copy_from_device(rt, ha.data(), a, ha.size() * 2));
        check(xpu_rt_copy_from_device(rt, hb.data(), b, hb.size() * 2));
        std::vector<double> bd(bs);
        for (uint64_t i = 0; i < bs; ++i) bd[i] = xpu::decode16(hb[i], o.dtype);
        const double gamma = o.k * 0x1p-24 / (1 - o.k * 0x1p-24);
        std::vector<double> acc(o.n), absacc(o.n);
        for (uint32_t r = 0; r < rows; ++r) {
          std::fill(acc.begin(), acc.end(), 0.0);
          std::fill(absacc.begin(), absacc.end(), 0.0);
          for (uint32_t kk = 0; kk < o.k; ++kk) {
            const double av = xpu::decode16(ha[static_cast<size_t>(r) * o.k + kk], o.dtype);
            const double *brow = bd.data() + static_cast<size_t>(kk) * o.n;
            for (uint32_t j = 0; j < o.n; ++j) {
              acc[j] += av * brow[j];
              absacc[j] += std::fabs(av * brow[j]);
            }
          }
          for (uint32_t j = 0; j < o.n; ++j) {
            const double ref = xpu::decode16(xpu::encode16(static_cast<float>(acc[j]), o.dtype), o.dtype);
            const double got = xpu::decode16(hc[static_cast<size_t>(r) * o.n + j], o.dtype);
            const double ulp = o.dtype ? xpu::fp16_ulp(ref) : xpu::bf16_ulp(ref);
            err2 += (got - ref) * (got - ref);
            ref2 += ref * ref;
            max_ulps = std::max(max_ulps, std::fabs(got - ref) / ulp);
            if (std::fabs(got - ref) > 2 * ulp + gamma * absacc[j])
              throw std::runtime_error("GEMM verification failed: C[" + std::to_string(r) + "][" + std::to_string(j) +
                                       "] expected " + std::to_string(ref) + ", got " + std::to_string(got));
          }
        }
        if ((ref2 > 0 ? std::sqrt(err2 / ref2) : std::sqrt(err2)) > 1e-3)
          throw std::runtime_error("GEMM verification failed: relative L2 error above 1e-3");
      }
    }
    std::cout << "Type: " << (o.dtype ? "FP16" : "BF16") << ", shape: " << o.m << 'x' << o.n << 'x' << o.k
              << '\n';
    if (o.constant_init)
      std::cout << "Input: constant A = 0.5, B = 0.25 (gemm.cpp:81-85), expected 0.125 * K = "
                << std::defaultfloat << o.k * 0.125 << '\n';
    else
      std::cout << "Input: uniform [-1,1), seed " << o.seed << '\n';
    std::cout << std::fixed << std::setprecision(2) << "Median: " << xpu::median_of(rates)
              << " TFLOP/s\nBest:   " << xpu::max_of(rates) << " TFLOP/s\n"
              << "MFMA roofline: " << (xpu::median_of(rates) / 2500.0 * 100.0)
              << "% of 2500 TFLOP/s dense (median " << xpu::median_of(times) * 1e6 << " us)\n";
    if (rows && !o.constant_init)
      std::cout << std::scientific << std::setprecision(3) << "Accuracy: rel-L2 "
                << (ref2 > 0 ? std::sqrt(err2 / ref2) : std::sqrt(err2)) << ", max " << std::fixed
                << std::setprecision(2) << max_ulps << " ulp over " << rows << " rows\n";
    std::cout << "Verification: PASS\n";
    return 0;
  } catch (const std::exception &error) {
    std::cerr << "Error: " << error.what() << '\n';
    return 1;
  }
}
