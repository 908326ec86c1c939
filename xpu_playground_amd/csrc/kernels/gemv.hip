// GEMV entry kernels: y[M] = A[M x K] . x[K], bf16 or fp16 storage, FP32
// accumulation (reference: gemv_kernel.hpp:21-63, entries
// level_zero/gem_spv_entry.cpp:11-27 with argument order (A, x, y, m, k)).
//
// Launch: 256 threads (4 wavefronts, fixed at compile time); dynamic LDS = round_up(K, 512) * 2
// bytes for the staged vector; the grid walks tiles of 4*R rows with a
// grid-stride loop so each block stages the vector once. Any M, K >= 1 and
// any leading dimension lda >= K are accepted; the _vec, _vecg and _ends
// variants need A, x 16-byte aligned and K, lda multiples of 8 (the host
// checks), the _any variants load 16 bytes at any element. The _vecg variants
// read the vector from global memory when it does not fit in LDS.
#include "gemv_core.hpp"

namespace xpu {

// XG: read the vector from global memory (cached loads) instead of LDS, for
// vectors longer than the LDS holds; needs the _vec alignment conditions.
template <int DT, int R, int U, bool VEC, bool XG, bool EARLY, bool CACHED>
XPU_DEVICE void gemv_entry(const uint16_t *__restrict__ A, const uint16_t *__restrict__ x,
                           uint16_t *__restrict__ y, uint32_t M, uint32_t K, uint64_t lda) {
  extern __shared__ __align__(16) uint16_t lds_x[];
  const uint16_t *xs = x;
  constexpr uint32_t kBlock = 256;  // launched with 256 threads (gemv_api.cpp)
  const uint32_t wave = threadIdx.x >> 6;
  const uint32_t rows_per_block = (kBlock >> 6) * R;
  if constexpr (!XG) {
    const uint32_t kpad = (K + 511u) & ~511u;
    stage_vector<VEC, kBlock>(lds_x, x, K, kpad);
    __syncthreads();
    xs = lds_x;
  }
  for (uint32_t base = blockIdx.x * rows_per_block; base < M; base += gridDim.x * rows_per_block) {
    const uint32_t row0 = base + wave * R;
    if (row0 >= M) continue;
    float out[R];
    gemv_rows<DT, R, U, VEC, EARLY, CACHED>(A, lda, K, M, xs, row0, out);
    const uint32_t lane = lane_id();
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (lane == static_cast<uint32_t>(r) && row0 + r < M)
        y[row0 + r] = static_cast<uint16_t>(encode<DT>(out[r]));
  }
}

}  // namespace xpu

#define XPU_GEMV_VARIANT(NAME, DT, R, U, VEC, XG, EARLY, CACHED)                           \
  extern "C" __global__ __launch_bounds__(256) void NAME(                                  \
      const uint16_t *__restrict__ A, const uint16_t *__restrict__ x,                      \
      uint16_t *__restrict__ y, uint32_t M, uint32_t K, uint64_t lda) {                    \
    XPU_STAMP(xpu::kStampGemv);                                                            \
    xpu::gemv_entry<DT, R, U, VEC, XG, EARLY, CACHED>(A, x, y, M, K, lda);                 \
  }
#define XPU_GEMV_TYPES(FORM, R, U, VEC, XG, EARLY)                                  \
  XPU_GEMV_VARIANT(xpu_gemv_bf16_##FORM, xpu::kBf16, R, U, VEC, XG, EARLY, false)   \
  XPU_GEMV_VARIANT(xpu_gemv_fp16_##FORM, xpu::kFp16, R, U, VEC, XG, EARLY, false)

// name: xpu_gemv_<type>_r<R>u<U>_<vec|ends|any|vecg>; R rows per wavefront, U
// 512-column chunks per pipelined load batch. The two-chunk forms _ends and
// _any load the row's end (the chunk that crosses K, the full chunk left over)
// ahead of the batches. Not where it costs: rows of 4096 columns or more that
// are whole batches take _vec (65536 x 4096 76.2 us, 78.0 with _ends; x 8192
// 151.5 and 155.8), and so do long rows (16384^2 fp16 5%) and the decode
// kernels, whose usual widths have no such end and whose wavefronts per SIMD
// its registers would reduce (135 instead of 123; no difference in time was
// measured at hidden 5120, 322 us a token for two layers either way). The bf16
// _ends loads each row's first batch cached: from the Infinity Cache that is 2%
// faster (16384 x 2048 12.0 us against 12.2 with streaming loads), from memory
// 2% faster past 256 MB (151936 x 2560 114 against 117) and up to 11% slower
// below 2048 columns (151936 x 1024 53.5 against 47.8); fp16 streams it.
XPU_GEMV_TYPES(r1u4_vec, 1, 4, true, false, false)
XPU_GEMV_TYPES(r1u4_any, 1, 4, false, false, false)
XPU_GEMV_TYPES(r2u2_vec, 2, 2, true, false, false)
XPU_GEMV_VARIANT(xpu_gemv_bf16_r2u2_ends, xpu::kBf16, 2, 2, true, false, true, true)
XPU_GEMV_VARIANT(xpu_gemv_fp16_r2u2_ends, xpu::kFp16, 2, 2, true, false, true, false)
XPU_GEMV_TYPES(r2u2_any, 2, 2, false, false, true)
XPU_GEMV_TYPES(r1u8_vecg, 1, 8, true, true, false)
