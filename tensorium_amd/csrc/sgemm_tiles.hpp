// SGEMM arguments and the epilogue of the bf16-part tiles (sgemm.hip,
// sgemm_ragged.hip).
#pragma once
#include "common.hpp"
#include "split_loop.hpp"

namespace tnh {

struct SgemmArgs {
  const float* A;
  const float* B;
  float* C;
  int64_t M, N, K, lda, ldb, ldc;
  int64_t strideA, strideB, strideC;
  int64_t aBytes, bBytes;  // extent of one batch item of A / B
  int64_t cBytes;          // extent of one batch item of C
  float alpha, beta;
  int tilesM, tilesN;
  // splits > 1 (one batch item): workgroup (tile, split) sums kChunk of K and
  // stores it raw in part [splits][M][N], which sgemm_reduce adds up
  int splits;
  int64_t kChunk;
  float* part;
};

// The K range of this workgroup's split (blockIdx.z).
__device__ inline void sgemm_range(const SgemmArgs& a, int64_t& kBegin, int64_t& kEnd) {
  kBegin = blockIdx.z * a.kChunk;
  kEnd = min(a.K, kBegin + a.kChunk);
}

template <class Cfg>
__device__ inline void sgemm_store(const SgemmArgs& a, int64_t bz, int64_t m0, int64_t n0,
                                   const f32x16 (&acc)[Cfg::FM][Cfg::FN]) {
  // C = alpha*acc (+ beta*C): lane columns n, wave-uniform row offsets in the
  // scalar operand, out-of-range elements at kOOB (dropped); every C load is
  // issued before the first store.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  const int64_t m0w = m0 + wm * Cfg::WTM, n0w = n0 + wn * Cfg::WTN;
  const int h = lane >> 5;
  const int rowBase = static_cast<int>(m0w) + 4 * h;
  const bool allRows = m0w + Cfg::FM * 32 <= a.M;
  const uint32_t ldc4 = static_cast<uint32_t>(a.ldc) * 4u;
  const __amdgpu_buffer_rsrc_t cR = make_rsrc(a.C + bz * a.strideC, a.cBytes);
  uint32_t vo[Cfg::FN];
#pragma unroll
  for (int j = 0; j < Cfg::FN; ++j) {
    const int64_t n = n0w + j * 32 + (lane & 31);
    vo[j] = sel_off(n < a.N, static_cast<uint32_t>(rowBase) * ldc4 + static_cast<uint32_t>(n) * 4u);
  }
  auto rowOk = [&](int i, int r) { return allRows || rowBase + i * 32 + 8 * (r >> 2) + (r & 3) < a.M; };
  auto off = [&](int i, int j, int r) { return rowOk(i, r) ? vo[j] : kOOB; };
  // the row of a scalar offset: none past the last (kOOB)
  const int lastRow = __builtin_amdgcn_readfirstlane(max(static_cast<int>(a.M - 1 - m0w), 0));
  auto rowOff = [&](int i, int r) { return static_cast<uint32_t>(min(i * 32 + 8 * (r >> 2) + (r & 3), lastRow)); };
  const float alpha = a.alpha, beta = a.beta;
  if (a.splits > 1) {
    const __amdgpu_buffer_rsrc_t pR = make_rsrc(a.part + blockIdx.z * a.M * a.N, a.M * a.N * 4);
    const uint32_t n4 = static_cast<uint32_t>(a.N) * 4u;
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j) {
        const int64_t n = n0w + j * 32 + (lane & 31);
        const uint32_t pv =
            sel_off(n < a.N, static_cast<uint32_t>(rowBase) * n4 + static_cast<uint32_t>(n) * 4u);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          conv::buf_st1s(pR, acc[i][j][r], rowOk(i, r) ? pv : kOOB, rowOff(i, r) * n4);
      }
    return;
  }
  if (beta != 0.f) {
    float cv[Cfg::FM][Cfg::FN][16];
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) cv[i][j][r] = buf_ld1s(cR, off(i, j, r), rowOff(i, r) * ldc4);
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          conv::buf_st1s(cR, alpha * acc[i][j][r] + beta * cv[i][j][r], off(i, j, r), rowOff(i, r) * ldc4);
  } else {
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) conv::buf_st1s(cR, alpha * acc[i][j][r], off(i, j, r), rowOff(i, r) * ldc4);
  }
}

// Tile shapes of the tiles for any operands: the index into kRaggedCfgs.
struct RaggedInfo {
  int rows, cols, perCU;
};
constexpr int kNumRagged = 3;
constexpr RaggedInfo kRaggedCfgs[kNumRagged] = {{128, 128, 1}, {64, 128, 2}, {64, 64, 3}};

// Any sizes, leading dimensions and alignment; C (and part) within 2 GiB.
int launch_sgemm_ragged(int i, SgemmArgs a, int64_t batch, bool ta, bool tb, hipStream_t s);

}  // namespace tnh
