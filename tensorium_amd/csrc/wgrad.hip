// Weight gradients over any geometry: dW = beta*dW + alpha * sum over images
// and output pixels of delta[f] * column[n], the column matrix gathered from
// the input.  It replaces im2col and a product per image (two launches an
// image: 64 -> 128 channels, 3x3, 56x56, batch 32 took 835 us).
//
// The reduction axis is the output pixels of all images in quads of four of
// one output row; a row of OW pixels has ceil(OW / 4) quads, the elements past
// its end are zeros in both operands.  A panel of the split loop is eight
// quads, wherever they lie, so no size is special; a quad's image, row and
// place in it are found per panel (two divisions by a float reciprocal,
// corrected to the exact quotient).
#include <algorithm>

#include "gemm_core.hpp"
#include "split_loop.hpp"
#include "wgrad.hpp"

namespace tnh {
namespace {

struct QuadAxis {
  int quads;          // of all images
  int OW, OH, perRow; // pixels of a row, rows of an image, quads of a row
  float invRow, invImage;  // 1 / perRow, 1 / OH
  int exact;          // too many rows for the reciprocals: integer division
};

struct Quad {
  int b, oy, x;  // image, output row, first pixel in it
  bool in;
};

// n / d for 0 <= n: the float quotient is within one of it while it is below 2^22
__device__ inline int quotient(int n, int d, float inv, bool exact) {
  if (exact) return n / d;
  int q = static_cast<int>(static_cast<float>(n) * inv);
  const int r = n - q * d;
  q += r >= d ? 1 : 0;
  q -= r < 0 ? 1 : 0;
  return q;
}

__device__ inline Quad quad_at(const QuadAxis& x, int q) {
  Quad r;
  r.in = q < x.quads;
  const int row = quotient(q, x.perRow, x.invRow, x.exact != 0);
  r.x = 4 * (q - row * x.perRow);
  r.b = quotient(row, x.OH, x.invImage, x.exact != 0);
  r.oy = row - r.b * x.OH;
  return r;
}

// Thread t holds quad t % 8 of rows t / 8 + v * ROWSTEP of a panel.
template <int ROWS, int NT, template <int, int> class Panel>
struct QuadRows {
  static constexpr int BK = 32, ROWSTEP = NT / 8, QUADS = ROWS / ROWSTEP;
  using L = Panel<ROWS, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(ROWS % ROWSTEP == 0 && ROWSTEP % 16 == 0, "QuadRows split");
  __amdgpu_buffer_rsrc_t rsrc;
  QuadAxis ax;
  int kq, ldsOff;
  f32x4 reg[QUADS];
  __device__ inline void init_quads(const float* p, int64_t bytes, const QuadAxis& axis, int tid) {
    rsrc = make_rsrc(p, bytes);
    ax = axis;
    kq = tid % 8;
    ldsOff = L::chunk(tid / 8, kq);
  }
  __device__ inline f32x4 quad(int u) const { return reg[u]; }
  __device__ inline int off(int u) const { return ldsOff + u * ROWSTEP * L::STRIDE; }
  __device__ inline void store(lds_t* stage) const { conv::store_quads(*this, stage); }
};

// Rows of pixels in memory, `ld` floats apart, an image every `stride`; four
// floats a load at any address (ragged_loaders.hpp).  With WHOLE (OW % 4 == 0)
// no quad crosses a row's end; else what it holds past it is cleared.
template <int ROWS, int NT, bool WHOLE, template <int, int> class Panel>
struct PixelRows : QuadRows<ROWS, NT, Panel> {
  using Base = QuadRows<ROWS, NT, Panel>;
  uint32_t rowOff[Base::QUADS];
  uint32_t stride4;
  int left;  // elements of this thread's quad before the row's end
  __device__ inline void init(const float* p, int64_t bytes, int64_t ld, int64_t stride, int64_t rows, int64_t r0,
                              const QuadAxis& axis, int tid) {
    Base::init_quads(p, bytes, axis, tid);
    stride4 = static_cast<uint32_t>(stride) * 4u;
#pragma unroll
    for (int v = 0; v < Base::QUADS; ++v) {
      const int64_t r = r0 + tid / 8 + v * Base::ROWSTEP;
      rowOff[v] = r < rows ? static_cast<uint32_t>(r * ld * 4) : kOOB;
    }
  }
  __device__ inline void load(int64_t k0) {
    const Quad q = quad_at(Base::ax, static_cast<int>(k0 >> 2) + Base::kq);
    const uint32_t o = static_cast<uint32_t>(q.b) * stride4 + static_cast<uint32_t>(q.oy * Base::ax.OW + q.x) * 4u;
#pragma unroll
    for (int v = 0; v < Base::QUADS; ++v) {
      const bool ok = q.in && rowOff[v] != kOOB;
      Base::reg[v] = buf_ld4s(Base::rsrc, sel_off(ok, rowOff[v] + o), 0);
    }
    left = Base::ax.OW - q.x;
  }
  // hides QuadRows::quad, so store() below calls this one
  __device__ inline f32x4 quad(int u) const {
    f32x4 v = Base::reg[u];
    if constexpr (!WHOLE) v = f32x4{v[0], left > 1 ? v[1] : 0.f, left > 2 ? v[2] : 0.f, left > 3 ? v[3] : 0.f};
    return v;
  }
  __device__ inline void store(lds_t* stage) const { conv::store_quads(*this, stage); }
};

// The im2col rows n = (c*kh + ky)*kw + kx of the input.
template <int ROWS, int NT, template <int, int> class Panel>
struct ColRows : QuadRows<ROWS, NT, Panel> {
  using Base = QuadRows<ROWS, NT, Panel>;
  int ry[Base::QUADS], rx[Base::QUADS];  // ky*dY - pH, kx*dX - pW
  uint32_t rowOff[Base::QUADS];          // the channel's plane in bytes
  uint32_t stride4;
  int H, W, sY, sX;
  __device__ inline void init(const float* p, const ColGeom& g, int64_t rows, int64_t r0, const QuadAxis& axis,
                              int tid) {
    Base::init_quads(p, g.xBytes, axis, tid);
    stride4 = static_cast<uint32_t>(g.xBatchStride) * 4u;
    H = g.H, W = g.W, sY = g.sY, sX = g.sX;
#pragma unroll
    for (int v = 0; v < Base::QUADS; ++v) {
      const int64_t r = r0 + tid / 8 + v * Base::ROWSTEP;
      const int n = static_cast<int>(r < rows ? r : 0), taps = g.kh * g.kw;
      const int c = n / taps, t = n - c * taps, ky = t / g.kw, kx = t - ky * g.kw;
      ry[v] = r < rows ? ky * g.dY - g.pH : -(1 << 30);  // no row of the image
      rx[v] = kx * g.dX - g.pW;
      rowOff[v] = static_cast<uint32_t>(c) * static_cast<uint32_t>(g.H * g.W) * 4u;
    }
  }
  __device__ inline void load(int64_t k0) {
    const Quad q = quad_at(Base::ax, static_cast<int>(k0 >> 2) + Base::kq);
    const int iy0 = q.oy * sY, ix0 = q.x * sX, left = q.in ? Base::ax.OW - q.x : 0;
    const uint32_t image = static_cast<uint32_t>(q.b) * stride4;
#pragma unroll
    for (int v = 0; v < Base::QUADS; ++v) {
      const int iy = iy0 + ry[v], ix = ix0 + rx[v];
      const bool row = static_cast<unsigned>(iy) < static_cast<unsigned>(H);
      const uint32_t o = image + rowOff[v] + static_cast<uint32_t>(iy * W + ix) * 4u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = row && e < left && static_cast<unsigned>(ix + e * sX) < static_cast<unsigned>(W);
        Base::reg[v][e] = buf_ld1s(Base::rsrc, sel_off(ok, o + static_cast<uint32_t>(e * sX) * 4u), 0);
      }
    }
  }
};

// The column operand, as bf16 parts and in fp32: gathered (COL) or in memory.
template <class Cfg, bool COL, bool VEC, template <int, int> class P>
struct ColOp {
  using type = PixelRows<Cfg::BN, Cfg::NT, VEC, P>;
};
template <class Cfg, bool VEC, template <int, int> class P>
struct ColOp<Cfg, true, VEC, P> {
  using type = ColRows<Cfg::BN, Cfg::NT, P>;
};

template <class Cfg, bool COL, bool VEC>
__global__ __launch_bounds__(Cfg::NT, Cfg::OCC) void wgrad_split_kernel(WgradArgs a, ColGeom g, QuadAxis ax) {
  using AL = PixelRows<Cfg::BM, Cfg::NT, VEC, conv::SplitPanel>;
  using AF = PixelRows<Cfg::BM, Cfg::NT, VEC, conv::SwzPanel>;
  using BL = typename ColOp<Cfg, COL, VEC, conv::SplitPanel>::type;
  using BF = typename ColOp<Cfg, COL, VEC, conv::SwzPanel>::type;
  using Loop = conv::SplitLoop<Cfg, AL, BL>;
  __shared__ __attribute__((aligned(16))) float smem[Loop::LDS_FLOATS];
  __shared__ int odd;
  lds_t* lds = (lds_t*)smem;
  int tm, tn;
  tile_coords(blockIdx.x, a.tilesM, a.tilesN, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * Cfg::BM, n0 = static_cast<int64_t>(tn) * Cfg::BN;
  auto init = [&](auto& al, auto& bl) {
    al.init(a.A, a.aBytes, a.lda, a.strideA, a.M, m0, ax, threadIdx.x);
    if constexpr (COL)
      bl.init(a.B, g, a.N, n0, ax, threadIdx.x);
    else
      bl.init(a.B, a.bBytes, a.ldb, a.strideB, a.N, n0, ax, threadIdx.x);
  };
  const int64_t panels = (ax.quads + 7) / 8;
  const int64_t p0 = blockIdx.y * a.kChunk / 32, np = min(panels - p0, a.kChunk / 32);
  AL al;
  BL bl;
  init(al, bl);
  f32x16 acc[Cfg::FM][Cfg::FN];
  Loop::exec(al, bl, p0 * 32, np, lds, &odd, acc);
  if (!Loop::finite(acc, &odd)) {
    AF af;
    BF bf;
    init(af, bf);
    conv::PlainLoop<Cfg, AF, BF>::exec(af, bf, p0 * 32, np, lds, acc);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t mw = m0 + wave / Cfg::WN * Cfg::WTM + 4 * (lane >> 5);
  const int64_t nw = n0 + wave % Cfg::WN * Cfg::WTN + (lane & 31);
  const bool raw = a.splits > 1 || a.rawPieces;
  float* out = raw ? a.part + static_cast<int64_t>(blockIdx.y) * a.M * a.N : a.C;
  const int64_t ld = raw ? a.N : a.ldc;
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j) {
      const int64_t n = nw + j * 32;
      if (n >= a.N) continue;
      auto at = [&](int r) { return mw + i * 32 + 8 * (r >> 2) + (r & 3); };
      float old[16];  // read together: a read after a store would wait for it
      if (!raw && a.beta != 0.f)
#pragma unroll
        for (int r = 0; r < 16; ++r) old[r] = at(r) < a.M ? out[at(r) * ld + n] : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (at(r) >= a.M) continue;
        float v = acc[i][j][r];
        if (!raw) {
          v = a.alpha * v;
          if (a.beta != 0.f) v = v + a.beta * old[r];
        }
        out[at(r) * ld + n] = v;
      }
    }
}

using W128 = conv::LeanCfg<128, 128, 32, 2, 4, 2>;
using W64x128 = conv::LeanCfg<64, 128, 32, 2, 2, 2>;
using W128x64 = conv::LeanCfg<128, 64, 32, 2, 2, 2>;
using W64 = conv::LeanCfg<64, 64, 32, 2, 2, 3>;

// What a tile costs a panel, in us: with one workgroup on its CU and, for each
// of several, where the CU is busy.
struct TileCost {
  int rows, cols;
  float alone, busy;
};
constexpr TileCost kTiles[] = {
    {128, 128, 1.55f, 1.55f}, {64, 128, 1.5f, 1.05f}, {128, 64, 1.3f, 1.05f}, {64, 64, 0.9f, 0.6f}};

struct Plan {
  int tile, splits;
  int64_t chunk;  // panels per split
};

// The tile and the split of the reduction axis, chosen together: a 128x128
// tile reads the fewest bytes per product, but a short axis then leaves most
// CUs without work, and each split costs its M*N floats written and read.
// Every tile is tried whole and with the splits that give one, two and three
// workgroups a CU, at least two panels each, and the least estimate taken.  The
// constants are fitted to 1300 timings of 39 products (M 17 to 1024, N 27 to
// 4608, 7 to 10816 panels), which they give within 10% in the mean; the choice
// is within 5% of the best of each in the mean, 17% at most.  Layers of
// 3 -> 32, 32 -> 64 and 64 -> 128 channels on 32x32, 16x16 and 8x8 pixels (us;
// first the widest tile that fits with at least eight panels a split, then
// this rule): batch 8 15.0, 19.7, 20.0 and 10.1, 10.5, 9.8; batch 32 16.0,
// 21.6, 21.1 and 13.5, 15.8, 14.5; batch 128 22.4, 33.7, 26.4 and 22.3, 29.1,
// 24.9.
Plan plan(int64_t M, int64_t N, int64_t panels, int64_t cus) {
  Plan best{0, 1, panels};
  float least = 0.f;
  for (int t = 0; t < 4; ++t) {
    const TileCost& c = kTiles[t];
    const int64_t tiles = ((M + c.rows - 1) / c.rows) * ((N + c.cols - 1) / c.cols);
    for (int64_t n = 0; n <= 3; ++n) {
      int64_t splits = std::max<int64_t>(1, std::min<int64_t>({n * cus / tiles, panels / 2, 1024}));
      const int64_t chunk = (panels + splits - 1) / splits;
      splits = (panels + chunk - 1) / chunk;  // no empty split
      const int64_t perCU = (tiles * splits + cus - 1) / cus;
      float us = static_cast<float>(chunk) * std::max(c.alone, static_cast<float>(perCU) * c.busy);
      if (splits > 1)  // the reduction: a wave an element, or a thread
        us += 2.f + static_cast<float>(splits) *
                        (M * N < kWaveReduceBelow ? 0.006f : static_cast<float>(M * N) * 2.5e-6f);
      if ((t == 0 && n == 0) || us < least) least = us, best = {t, static_cast<int>(splits), chunk};
    }
  }
  return best;
}

template <class Cfg>
int run(Context* cx, WgradArgs* a, const ColGeom* geom, const QuadAxis& ax, const Plan& pl) {
  const int64_t tm = (a->M + Cfg::BM - 1) / Cfg::BM, tn = (a->N + Cfg::BN - 1) / Cfg::BN;
  if (tm * tn > INT32_MAX) return fail(TNH_ERR_UNSUPPORTED, "conv2d_wgrad: grid too large");
  a->tilesM = static_cast<int>(tm);
  a->tilesN = static_cast<int>(tn);
  const int64_t panels = (ax.quads + 7) / 8;
  a->kChunk = pl.chunk * 32;
  a->splits = pl.splits;
  if (a->rawPieces && !a->part) return TNH_OK;
  if (a->splits > 1 && !a->rawPieces) {
    a->part = static_cast<float*>(workspace(cx, static_cast<size_t>(a->splits) * a->M * a->N * 4));
    if (!a->part) a->splits = 1, a->kChunk = panels * 32;
  }
  const ColGeom g = geom ? *geom : ColGeom{};
  const dim3 grid(static_cast<unsigned>(tm * tn), static_cast<unsigned>(a->splits));
  const bool vec = ax.OW % 4 == 0;
  if (geom && vec)
    hipLaunchKernelGGL((wgrad_split_kernel<Cfg, true, true>), grid, dim3(Cfg::NT), 0, cx->stream, *a, g, ax);
  else if (geom)
    hipLaunchKernelGGL((wgrad_split_kernel<Cfg, true, false>), grid, dim3(Cfg::NT), 0, cx->stream, *a, g, ax);
  else if (vec)
    hipLaunchKernelGGL((wgrad_split_kernel<Cfg, false, true>), grid, dim3(Cfg::NT), 0, cx->stream, *a, g, ax);
  else
    hipLaunchKernelGGL((wgrad_split_kernel<Cfg, false, false>), grid, dim3(Cfg::NT), 0, cx->stream, *a, g, ax);
  return launch_status("wgrad_split_kernel");
}

}  // namespace

int wgrad_any(Context* cx, WgradArgs* a, const ColGeom* geom) {
  QuadAxis ax{};
  // rows in memory, and a 1x1 window over every pixel, have no row ends inside an image
  const bool plane = !geom || (geom->kh == 1 && geom->kw == 1 && geom->sY == 1 && geom->sX == 1 && geom->pH == 0 &&
                               geom->pW == 0);
  ax.OW = static_cast<int>(plane ? a->L : geom->OW);
  ax.OH = static_cast<int>(a->L / ax.OW);
  ax.perRow = (ax.OW + 3) / 4;
  const int64_t rows = a->batch * ax.OH;
  if (rows * ax.perRow >= (int64_t(1) << 31) - 64)
    return fail(TNH_ERR_UNSUPPORTED, "conv2d_wgrad: reduction axis too long");
  ax.quads = static_cast<int>(rows * ax.perRow);
  ax.invRow = 1.f / static_cast<float>(ax.perRow);
  ax.invImage = 1.f / static_cast<float>(ax.OH);
  ax.exact = rows >= (int64_t(1) << 22);
  if (plane && geom) {
    WgradArgs b = *a;
    b.B = a->B;
    b.bBytes = geom->xBytes;
    b.ldb = a->L;
    b.strideB = geom->xBatchStride;
    *a = b;
    geom = nullptr;
  }
  const int64_t panels = (ax.quads + 7) / 8;
  Plan pl = plan(a->M, a->N, panels, cx->cu_count);
  // the update pass takes few weights in one piece only
  if (a->rawPieces && a->M * a->N < kWaveReduceBelow && panels < 16) pl = {3, 1, panels};
  switch (pl.tile) {
    case 0: return run<W128>(cx, a, geom, ax, pl);
    case 1: return run<W64x128>(cx, a, geom, ax, pl);
    case 2: return run<W128x64>(cx, a, geom, ax, pl);
    default: return run<W64>(cx, a, geom, ax, pl);
  }
}

}  // namespace tnh
