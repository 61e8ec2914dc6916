// NCHW convolution of any kernel size, channel count and weight layout on the
// bf16-part tiles: rows are filters (the weights [F][K], any K), columns are
// output pixels gathered element by element.
//
// A thread owns one pixel column for the whole K loop and a wave 64 columns of
// one k-quad, so what k means (channel, window row and column) is the same for
// the wave: it is found in scalar registers, rides in the load's scalar
// offset, and a lane only adds the window's place and tests two bits of its
// masks of window rows and columns inside the image.  It replaces fp32 tiles
// whose threads divided twice per element: 5x5, 48 -> 100 channels, 57x75,
// batch 8 206 -> 120 us.
#include <algorithm>

#include "common.hpp"
#include "conv_gather.hpp"
#include "ragged_loaders.hpp"

namespace tnh {
namespace conv {
namespace {

// floor(2^32 / d) + 1: k / d is the high word of k * magic for k * d < 2^32 (0: d is 1)
struct GatherDiv {
  uint32_t inner, kw;  // inner: C (tap-major) or kh * kw
};

__device__ inline int div_by(int k, uint32_t magic) {
  return magic ? static_cast<int>(__umulhi(static_cast<uint32_t>(k), magic)) : k;
}

template <class Cfg, template <int, int> class Panel>
struct GatherCols {
  static constexpr int BK = 32, BN = Cfg::BN, NT = Cfg::NT;
  static constexpr int QSTEP = NT / BN, NQ = 8 / QSTEP;
  using L = Panel<BN, BK>;
  static constexpr int SIZE = L::SIZE, QUADS = NQ;
  static_assert(BN % 64 == 0 && NT % BN == 0 && 8 % QSTEP == 0, "GatherCols split");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t colOff;        // bytes to (image, iy0, ix0), modulo 2^32
  uint32_t yMask, xMask;  // window rows and columns inside the image
  GatherDiv div;
  int q0, K, kw, W, C, inner;
  bool tap;
  uint32_t HW4;
  int ldsOff[NQ];
  float reg[NQ][4];

  __device__ inline void init(const ConvGeom& g, const GatherDiv& d, int64_t n0, int tid) {
    rsrc = make_rsrc(g.x, g.xBytes);
    div = d;
    K = static_cast<int>(g.K);
    kw = g.kw;
    W = g.W;
    C = g.C;
    tap = g.tapW != 0;
    inner = tap ? g.C : g.kh * g.kw;
    HW4 = static_cast<uint32_t>(g.H) * static_cast<uint32_t>(g.W) * 4u;
    const int col = tid % BN;
    q0 = __builtin_amdgcn_readfirstlane(tid / BN);
    const int64_t n = n0 + col;
    const bool ok = n < g.N;
    const int64_t nn = ok ? n : 0;
    const int64_t b = nn / g.OHW;
    const int p = static_cast<int>(nn - b * g.OHW);
    const int oy = p / g.OW, ox = p - (p / g.OW) * g.OW;
    const int iy0 = oy * g.sY - g.pH, ix0 = ox * g.sX - g.pW;
    colOff = static_cast<uint32_t>((b * g.xBatchStride + static_cast<int64_t>(iy0) * g.W + ix0) * 4);
    // bits lo .. hi-1 of a mask
    auto bits = [](int lo, int hi) {
      lo = max(lo, 0);
      hi = min(hi, 32);
      return hi <= lo ? 0u : (hi - lo == 32 ? ~0u : ((1u << (hi - lo)) - 1u) << lo);
    };
    yMask = ok ? bits(-iy0, min(g.kh, g.H - iy0)) : 0u;
    xMask = bits(-ix0, min(g.kw, g.W - ix0));
#pragma unroll
    for (int j = 0; j < NQ; ++j) ldsOff[j] = L::chunk(col, q0 + j * QSTEP);
  }
  __device__ inline void load(int64_t k0) {
#pragma unroll
    for (int j = 0; j < NQ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = static_cast<int>(k0) + 4 * (q0 + j * QSTEP) + e;  // uniform
        const int hi = div_by(k, div.inner), lo = k - hi * inner;
        const int t = tap ? hi : lo, c = tap ? lo : hi;
        const int ky = div_by(t, div.kw), kx = t - ky * kw;
        const bool ok = k < K && (yMask & (1u << (ky & 31))) && (xMask & (1u << kx));
        reg[j][e] = buf_ld1s(rsrc, sel_off(ok, colOff + static_cast<uint32_t>(ky * W + kx) * 4u),
                             static_cast<uint32_t>(min(c, C - 1)) * HW4);  // c past K: kOOB
      }
  }
  __device__ inline f32x4 quad(int u) const { return f32x4{reg[u][0], reg[u][1], reg[u][2], reg[u][3]}; }
  __device__ inline int off(int u) const { return ldsOff[u]; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

// A 1x1 window over every pixel: the columns are the channels' own rows of
// pixels, in RowsTailMN's units, none of which may cross an image's end.
// Loaded element by element such a layer, which multiplies little, waited on
// its loads: 200 -> 300 channels, 26x26, batch 4 15.2 -> 10.6 us, 48 -> 100,
// 60x60, batch 8 12.1 -> 9.5 (the fp32 tiles before 12.8 and 14.7).
template <class Cfg, template <int, int> class Panel>
struct PixelCols : RowsTailMN<Cfg::BN, Cfg::NT, Panel> {
  __device__ inline void init(const ConvGeom& g, const GatherDiv&, int64_t n0, int tid) {
    this->init_rows(g.x, g.xBytes, g.OHW, tid, [&](int col) {
      const int64_t n = n0 + col;
      if (n >= g.N) return kOOB;
      const int64_t b = n / g.OHW;
      return static_cast<uint32_t>((b * g.xBatchStride + (n - b * g.OHW)) * 4);
    });
    this->klimit(g.K);
  }
};

// One tile, its columns loaded by BL (in fp32: BF).  A function that takes the
// arguments by reference: with the same code in the kernel, on its own copy of
// them, the compiler spilled (64x64 over rows of pixels 168 registers and 40
// bytes of scratch, here 124; 5x5, 48 -> 100, 57x75, batch 8 124.3 -> 120.3 us).
// The SGEMM tiles, written so, use 40 registers less too and are 3 to 5% slower.
template <class Cfg, class BL, class BF>
__device__ inline void gather_tile(const ConvArgs& a, const GatherDiv& d, int64_t m0, int64_t n0, lds_t* lds, int* odd) {
  f32x16 acc[Cfg::FM][Cfg::FN];
  using AL = RowsTailK<Cfg::BM, Cfg::NT, SplitPanel>;
  using AF = RowsTailK<Cfg::BM, Cfg::NT, SwzPanel>;
  using Loop = SplitLoop<Cfg, AL, BL>;
  static_assert(Loop::LDS_FLOATS == kSplitLds<Cfg>, "panels");
  auto init = [&](auto& al, auto& bl) {
    al.init(a.w, a.wBytes, a.g.K, a.F, m0, threadIdx.x);
    al.klimit(a.g.K);
    bl.init(a.g, d, n0, threadIdx.x);
  };
  const int64_t kBegin = blockIdx.y * a.kChunk, kEnd = min(a.g.K, kBegin + a.kChunk);
  const int64_t nk = (kEnd - kBegin + 31) / 32;
  AL al;
  BL bl;
  init(al, bl);
  Loop::exec(al, bl, kBegin, nk, lds, odd, acc);
  if (!Loop::finite(acc, odd)) {
    AF af;
    BF bf;
    init(af, bf);
    PlainLoop<Cfg, AF, BF>::exec(af, bf, kBegin, nk, lds, acc);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  conv_store_buf<Cfg::FM, Cfg::FN>(a, acc, m0 + wm * Cfg::WTM, n0 + wn * Cfg::WTN, lane);
}

// How a kernel loads its columns: single elements, rows of pixels (1x1 windows,
// images of whole units), or rows of pixels but single ones in the tiles that
// hold an image's end (123 -> 37 channels, 187x187, batch 21 185 -> 155 us; 90
// -> 142, 43x51, batch 23 38.3 -> 29.5).  The last needs more registers: not
// for images of a few tiles (100 -> 255, 13x13, batch 16 11.0 -> 11.7), nor
// where no unit crosses an image's end.
enum GatherLoads { kElements, kPixels, kPixelsOrEnds };

template <class Cfg, GatherLoads LOADS>
__global__ __launch_bounds__(Cfg::NT, Cfg::OCC) void conv_gather_kernel(ConvArgs a, GatherDiv d) {
  __shared__ __attribute__((aligned(16))) float smem[kSplitLds<Cfg>];
  __shared__ int odd;
  lds_t* lds = (lds_t*)smem;
  int tm, tn;
  tile_coords(blockIdx.x, a.tilesM, a.tilesN, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * Cfg::BM, n0 = static_cast<int64_t>(tn) * Cfg::BN;
  bool pixels = LOADS == kPixels;
  if constexpr (LOADS == kPixelsOrEnds) pixels = n0 / a.g.OHW == (min(n0 + Cfg::BN, a.g.N) - 1) / a.g.OHW;
  if constexpr (LOADS != kElements)
    if (pixels) gather_tile<Cfg, PixelCols<Cfg, SplitPanel>, PixelCols<Cfg, SwzPanel>>(a, d, m0, n0, lds, &odd);
  if constexpr (LOADS != kPixels)
    if (!pixels) gather_tile<Cfg, GatherCols<Cfg, SplitPanel>, GatherCols<Cfg, SwzPanel>>(a, d, m0, n0, lds, &odd);
}

using G64 = LeanCfg<64, 64, 32, 2, 2, 3>;
using G64x128 = LeanCfg<64, 128, 32, 2, 2, 2>;
using G128 = LeanCfg<128, 128, 32, 2, 4, 2>;
using G32x128 = LeanCfg<32, 128, 32, 1, 4, 2>;

uint32_t magic(int64_t d) { return d == 1 ? 0u : static_cast<uint32_t>((uint64_t(1) << 32) / d + 1); }

template <class Cfg>
int run(ConvArgs a, hipStream_t s) {
  const int64_t tm = (a.F + Cfg::BM - 1) / Cfg::BM, tn = (a.g.N + Cfg::BN - 1) / Cfg::BN;
  if (tm * tn > INT32_MAX) return fail(TNH_ERR_UNSUPPORTED, "conv2d: grid too large");
  a.tilesM = static_cast<int>(tm);
  a.tilesN = static_cast<int>(tn);
  const GatherDiv d{magic(a.g.tapW ? a.g.C : a.g.kh * a.g.kw), magic(a.g.kw)};
  const dim3 grid(static_cast<unsigned>(tm * tn), static_cast<unsigned>(a.splits));
  const ConvGeom& g = a.g;
  const bool planes = g.kh == 1 && g.kw == 1 && g.sY == 1 && g.sX == 1 && g.pH == 0 && g.pW == 0;
  if (planes && g.OHW % 4 == 0)
    hipLaunchKernelGGL((conv_gather_kernel<Cfg, kPixels>), grid, dim3(Cfg::NT), 0, s, a, d);
  else if (planes && g.OHW >= 8 * Cfg::BN)
    hipLaunchKernelGGL((conv_gather_kernel<Cfg, kPixelsOrEnds>), grid, dim3(Cfg::NT), 0, s, a, d);
  else
    hipLaunchKernelGGL((conv_gather_kernel<Cfg, kElements>), grid, dim3(Cfg::NT), 0, s, a, d);
  return launch_status("conv_gather_kernel");
}

}  // namespace

bool gather_takes(int64_t C, int64_t taps, int64_t K) {
  return (K + 64) * std::max(C, taps) < (int64_t(1) << 31);
}

int launch_gather(int i, ConvArgs a, hipStream_t s) {
  switch (i) {
    case 0: return run<G64>(a, s);
    case 1: return run<G64x128>(a, s);
    case 2: return run<G128>(a, s);
    default: return run<G32x128>(a, s);
  }
}

}  // namespace conv
}  // namespace tnh
