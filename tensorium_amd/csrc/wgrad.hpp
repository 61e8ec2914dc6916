// The weight-gradient product's arguments and its launch (wgrad.hip).
#pragma once
#include "common.hpp"

namespace tnh {

struct WgradArgs {
  const float* A;
  const float* B;
  float* C;
  float* part;
  int64_t M, N, L, lda, ldb, ldc, strideA, strideB, batch;
  int64_t aBytes, bBytes, kChunk;
  float alpha, beta;
  int tilesM, tilesN, splits;
  int rawPieces;  // store every split's raw sums in part, no reduction (also one split)
};

// weight gradients of fewer elements sum their pieces a wave per element
constexpr int64_t kWaveReduceBelow = 8192;

// A convolution's input as the column operand: [C][H][W] images, kernel, stride, padding, dilation.
struct ColGeom {
  int64_t xBatchStride, xBytes;
  int C, H, W, OW, L, kh, kw, sY, sX, pH, pW, dY, dX;
};

// C = beta*C + alpha * sum_b A_b * B_b^T over batch images of L pixels, any
// L: A_b = A + b*strideA ([M][L], rows lda apart), B_b the rows of B + b*strideB
// ([N][L], rows ldb apart), or with geom the im2col of the image there.  The
// split partials go to the stream's workspace (whole K without one): with
// a->splits > 1 they are in a->part and left to be summed into C.  With
// a->rawPieces they go to the caller's a->part, one split's too; without it
// nothing runs and a->splits says how many there are.
int wgrad_any(Context* cx, WgradArgs* a, const ColGeom* geom);

}  // namespace tnh
