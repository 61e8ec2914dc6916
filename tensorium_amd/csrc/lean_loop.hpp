// Operand loaders of the lean tiles and of the wave-split tiles (conv_wsplit),
// their fp32 LDS panels and the fp32 fragments.  The lean tiles' loop is
// split_loop.hpp's, which takes the loaders with its own panels.
//   * Both operand panels are k-contiguous in LDS with their 16-byte chunks
//     XOR-swizzled: every LDS access is a conflict-free 16-byte
//     ds_read/ds_write_b128 and no padding is needed.  The B gather writes 4
//     consecutive k of one output column per store.
//   * Per-lane global offsets are fixed for the whole K loop; what varies
//     along K is wave-uniform and rides in the buffer instruction's scalar
//     offset.  The 3x3 padding test is a per-lane 9-bit tap mask computed
//     once, so a K panel costs a few vector ALU operations instead of two per
//     load.
//
// Requirements (checked by the host): K % BK == 0 (tap-major 3x3 with
// C % BK == 0, or 1x1 stride 1 with C % BK == 0), 16-byte weight rows, and
// output / residual / split-K partials within 2 GiB each (conv_store_buf).
#pragma once
#include "conv_args.hpp"

namespace tnh {
namespace conv {

template <int BM_, int BN_, int BK_, int WM_, int WN_, int OCC_>
struct LeanCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, OCC = OCC_;
  static constexpr int NT = WM * WN * 64;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int FM = WTM / 32, FN = WTN / 32;
  static constexpr int KCH = BK / 16;
  static_assert(FM >= 1 && FN >= 1 && WTM % 32 == 0 && WTN % 32 == 0, "tile");
  static_assert(BK == 32, "panel depth");
};

// k-contiguous panel [ROWS][BK] (floats) whose 16-byte chunks are
// XOR-swizzled: logical chunk q of row r sits at physical chunk q ^ swz(r).
// The LDS has 64 four-byte banks (256 bytes) and serves a 16-byte access 16
// lanes at a time, so 16 consecutive rows at one logical chunk must land in
// 16 different 16-byte bank groups.  A 32-float row is half a bank line: the
// row parity picks the half and swz(r) = (r / 2) % 8 spreads each half's 8
// rows over its 8 groups.  One row's chunks, and two consecutive rows' chunks,
// are always distinct groups too (the row-wise stores of the loaders).
template <int ROWS, int BK>
struct SwzPanel {
  static constexpr int SIZE = ROWS * BK;
  static constexpr int STRIDE = BK;  // floats per row
  static_assert(BK == 32, "panel depth");
  __device__ static inline int swz(int row) { return (row >> 1) & 7; }
  __device__ static inline int chunk(int row, int q) { return row * BK + 4 * (q ^ swz(row)); }
  // four consecutive k of a row to the place chunk() names
  __device__ static inline void put(lds_t* p, f32x4 v) { *reinterpret_cast<lds_f4*>(p) = v; }
};

// A loader holds QUADS k-quads of its panel: quad(u) goes to off(u).
template <class Loader>
__device__ inline void store_quads(const Loader& x, lds_t* stage) {
#pragma unroll
  for (int u = 0; u < Loader::QUADS; ++u) Loader::L::put(stage + x.off(u), x.quad(u));
}

// k-contiguous operand: row r of the panel is memory row r0 + r (row stride
// ld floats, rows >= `rows` read 0), 16-byte loads.  Thread t owns chunk
// t % (BK/4) of rows t / (BK/4) + v * ROWSTEP (ROWSTEP % 16 == 0, so every row
// of a thread has the same swizzle).  The conv weights [F][K] (ld = K), and
// the GEMM operands A (not transposed) and B (transposed).  KT: K is not a
// multiple of BK (set by klimit()); a chunk at k >= K reads 0 instead of the
// start of the next row.
template <int ROWS, int BK_, int NT_, bool KT = false, template <int, int> class Panel = SwzPanel>
struct LeanRowsK {
  static constexpr int BK = BK_, NT = NT_;
  static constexpr int QPR = BK / 4;
  static constexpr int ROWSTEP = NT / QPR;
  static constexpr int PER = ROWS / ROWSTEP;
  using L = Panel<ROWS, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(NT % QPR == 0 && ROWS % ROWSTEP == 0 && PER >= 1 && ROWSTEP % 16 == 0, "LeanRowsK split");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t voff[PER];
  int ldsOff;
  int kq4, kLim;  // KT: this thread's k offset in a panel, and K
  f32x4 reg[PER];

  __device__ inline void init(const float* p, int64_t bytes, int64_t ld, int64_t rows, int64_t r0, int tid) {
    rsrc = make_rsrc(p, bytes);
    const int row = tid / QPR, kq = tid % QPR;
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int64_t gr = r0 + row + v * ROWSTEP;
      voff[v] = sel_off(gr < rows, static_cast<uint32_t>((gr * ld + kq * 4) * 4));
    }
    ldsOff = L::chunk(row, kq);
    kq4 = 4 * kq;
    kLim = 0;
  }
  __device__ inline void klimit(int64_t K) { kLim = static_cast<int>(K); }
  __device__ inline void load(int64_t k0) {
    const uint32_t so = static_cast<uint32_t>(k0) * 4u;
    if constexpr (KT) {
      const bool in = static_cast<int>(k0) + kq4 < kLim;  // K % 4 == 0: a chunk is whole or past K
#pragma unroll
      for (int v = 0; v < PER; ++v) reg[v] = buf_ld4s(rsrc, sel_off(in, voff[v]), so);
    } else {
#pragma unroll
      for (int v = 0; v < PER; ++v) reg[v] = buf_ld4s(rsrc, voff[v], so);
    }
  }
  static constexpr int QUADS = PER;
  __device__ inline f32x4 quad(int u) const { return reg[u]; }
  __device__ inline int off(int u) const { return ldsOff + u * ROWSTEP * L::STRIDE; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

template <class Cfg>
using LeanA = LeanRowsK<Cfg::BM, Cfg::BK, Cfg::NT>;

// Row-contiguous operand: element (row r, k) at (r0 + r) + k * ld floats
// (rows >= `rows` read 0): the GEMM operands A (transposed) and B (not
// transposed) in fp32.  Thread t owns row t % ROWS and the k-quads t / ROWS +
// j * QSTEP, four loads ld floats apart each.
template <int ROWS, int BK_, int NT_>
struct LeanRowsMN {
  static constexpr int BK = BK_, NT = NT_;
  static constexpr int QSTEP = NT / ROWS, NQ = (BK / 4) / QSTEP;
  using L = SwzPanel<ROWS, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(NT % ROWS == 0 && (BK / 4) % QSTEP == 0 && NQ >= 1, "LeanRowsMN split");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t voff, ld4;
  int ldsOff[NQ];
  float reg[NQ][4];

  __device__ inline void init(const float* p, int64_t bytes, int64_t ld, int64_t rows, int64_t r0, int tid) {
    rsrc = make_rsrc(p, bytes);
    ld4 = static_cast<uint32_t>(ld) * 4u;
    const int row = tid % ROWS, q0 = tid / ROWS;
    const int64_t gr = r0 + row;
    voff = sel_off(gr < rows, static_cast<uint32_t>((gr + 4 * q0 * ld) * 4));
#pragma unroll
    for (int j = 0; j < NQ; ++j) ldsOff[j] = L::chunk(row, q0 + j * QSTEP);
  }
  __device__ inline void load(int64_t k0) {
#pragma unroll
    for (int j = 0; j < NQ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        reg[j][e] = buf_ld1s(rsrc, voff, static_cast<uint32_t>(static_cast<int>(k0) + 4 * j * QSTEP + e) * ld4);
  }
  static constexpr int QUADS = NQ;
  __device__ inline f32x4 quad(int u) const { return f32x4{reg[u][0], reg[u][1], reg[u][2], reg[u][3]}; }
  __device__ inline int off(int u) const { return ldsOff[u]; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

// Channels-last tap gather as the A operand (row r of the panel = output
// pixel m0 + r, k = tap*C + c with a panel inside one tap): a row's BK
// channels are contiguous, so each thread issues PER 16-byte loads per panel.
// Thread t owns chunk t % (BK/4) of rows t / (BK/4) + v * ROWSTEP.  A row's
// pixel offset at tap (0, 0) is fixed for the K loop (modulo 2^32: it may
// point before the image at the border); the uniform tap offset is added per
// panel, the channel offset rides in the scalar operand, and a per-row tap
// mask (computed once) sends taps in the padding to kOOB.
template <int ROWS, int BK_, int NT_, int KH, int KW, template <int, int> class Panel = SwzPanel>
struct NhwcTapRows {
  static constexpr int BK = BK_, NT = NT_;
  static constexpr int QPR = BK / 4;
  static constexpr int ROWSTEP = NT / QPR;
  static constexpr int PER = ROWS / ROWSTEP;
  using L = Panel<ROWS, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(NT % QPR == 0 && ROWS % ROWSTEP == 0 && PER >= 1 && ROWSTEP % 16 == 0 && KH * KW <= 32,
                "NhwcTapRows split");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t rowOff[PER];
  uint32_t tapMask[PER];
  uint32_t pix4, rowPix4;  // bytes per pixel step, per image row
  int C;
  int ldsOff;
  f32x4 reg[PER];

  __device__ inline void init(const ConvGeom& g, int xPix, int64_t m0, int tid) {
    rsrc = make_rsrc(g.x, g.xBytes);
    C = g.C;
    pix4 = static_cast<uint32_t>(xPix) * 4u;
    rowPix4 = static_cast<uint32_t>(g.W) * pix4;
    const int row = tid / QPR, kq = tid % QPR;
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int64_t n = m0 + row + v * ROWSTEP;
      const bool ok = n < g.N;
      const int64_t nn = ok ? n : 0;
      const int64_t b = nn / g.OHW;
      const int p = static_cast<int>(nn - b * g.OHW);
      const int oy = p / g.OW, ox = p - (p / g.OW) * g.OW;
      const int iy0 = oy * g.sY - g.pH, ix0 = ox * g.sX - g.pW;
      rowOff[v] = static_cast<uint32_t>(((b * g.H + iy0) * g.W + ix0) * xPix * 4 + kq * 16);
      uint32_t m = 0;
#pragma unroll
      for (int ky = 0; ky < KH; ++ky)
#pragma unroll
        for (int kx = 0; kx < KW; ++kx) {
          const bool in = static_cast<unsigned>(iy0 + ky) < static_cast<unsigned>(g.H) &&
                          static_cast<unsigned>(ix0 + kx) < static_cast<unsigned>(g.W);
          m |= (ok && in ? 1u : 0u) << (ky * KW + kx);
        }
      tapMask[v] = m;
    }
    ldsOff = L::chunk(row, kq);
  }
  __device__ inline void load(int64_t k0) {
    const int kk = static_cast<int>(k0);
    const int tap = kk / C;  // uniform
    const int c0 = kk - tap * C;
    const int ky = tap / KW, kx = tap - (tap / KW) * KW;
    const uint32_t tapOff = static_cast<uint32_t>(ky) * rowPix4 + static_cast<uint32_t>(kx) * pix4;
#pragma unroll
    for (int v = 0; v < PER; ++v)
      reg[v] = buf_ld4s(rsrc, sel_off((tapMask[v] >> tap) & 1u, rowOff[v] + tapOff), static_cast<uint32_t>(c0) * 4u);
  }
  static constexpr int QUADS = PER;
  __device__ inline f32x4 quad(int u) const { return reg[u]; }
  __device__ inline int off(int u) const { return ldsOff + u * ROWSTEP * L::STRIDE; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

// NhwcTapRows for 3x3 windows over any C % 4 == 0: a panel may span taps
// (C = 4, 8, 16: 32/C taps per panel; C = 48, 80, ...: a panel crosses one
// tap boundary) and the last panel may run past K = 9C (those chunks read
// 0).  A thread's chunk sits at k = k0 + 4*(t % (BK/4)): its tap and channel
// are found per panel (one approximate float division, corrected to the
// exact quotient); the rows' tap masks and pixel offsets are as in
// NhwcTapRows, the channel offset is per thread.
template <int ROWS, int BK_, int NT_, template <int, int> class Panel = SwzPanel>
struct NhwcTapRowsAny {
  static constexpr int BK = BK_, NT = NT_;
  static constexpr int QPR = BK / 4;
  static constexpr int ROWSTEP = NT / QPR;
  static constexpr int PER = ROWS / ROWSTEP;
  using L = Panel<ROWS, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(NT % QPR == 0 && ROWS % ROWSTEP == 0 && PER >= 1 && ROWSTEP % 16 == 0, "NhwcTapRowsAny split");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t rowOff[PER];  // byte offset of the row's pixel at tap (0, 0), channel 0, modulo 2^32
  uint32_t tapMask[PER];
  uint32_t pix4, rowPix4;
  int C, K, kq4;
  float invC;
  int ldsOff;
  f32x4 reg[PER];

  __device__ inline void init(const ConvGeom& g, int xPix, int64_t m0, int tid) {
    rsrc = make_rsrc(g.x, g.xBytes);
    C = g.C;
    K = 9 * g.C;
    invC = 1.f / static_cast<float>(g.C);
    pix4 = static_cast<uint32_t>(xPix) * 4u;
    rowPix4 = static_cast<uint32_t>(g.W) * pix4;
    const int row = tid / QPR, kq = tid % QPR;
    kq4 = 4 * kq;
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int64_t n = m0 + row + v * ROWSTEP;
      const bool ok = n < g.N;
      const int64_t nn = ok ? n : 0;
      const int64_t b = nn / g.OHW;
      const int p = static_cast<int>(nn - b * g.OHW);
      const int oy = p / g.OW, ox = p - (p / g.OW) * g.OW;
      const int iy0 = oy * g.sY - g.pH, ix0 = ox * g.sX - g.pW;
      rowOff[v] = static_cast<uint32_t>(((b * g.H + iy0) * g.W + ix0) * xPix * 4);
      uint32_t m = 0;
#pragma unroll
      for (int ky = 0; ky < 3; ++ky)
#pragma unroll
        for (int kx = 0; kx < 3; ++kx) {
          const bool in = static_cast<unsigned>(iy0 + ky) < static_cast<unsigned>(g.H) &&
                          static_cast<unsigned>(ix0 + kx) < static_cast<unsigned>(g.W);
          m |= (ok && in ? 1u : 0u) << (ky * 3 + kx);
        }
      tapMask[v] = m;
    }
    ldsOff = L::chunk(row, kq);
  }
  __device__ inline void load(int64_t k0) {
    const int k = static_cast<int>(k0) + kq4;
    // k / C: the float quotient is within one of the exact one for k < 2^22
    int tap = static_cast<int>(static_cast<float>(k) * invC);
    tap += (tap + 1) * C <= k ? 1 : 0;
    tap -= tap * C > k ? 1 : 0;
    const int c = k - tap * C;
    const bool kin = k < K;  // past K: tap >= 9, at most 9 + 31/4
    const int ky = tap / 3, kx = tap - (tap / 3) * 3;
    const uint32_t off = static_cast<uint32_t>(ky) * rowPix4 + static_cast<uint32_t>(kx) * pix4 +
                         static_cast<uint32_t>(c) * 4u;
#pragma unroll
    for (int v = 0; v < PER; ++v)
      reg[v] = buf_ld4s(rsrc, sel_off(kin && ((tapMask[v] >> tap) & 1u), rowOff[v] + off), 0u);
  }
  static constexpr int QUADS = PER;
  __device__ inline f32x4 quad(int u) const { return reg[u]; }
  __device__ inline int off(int u) const { return ldsOff + u * ROWSTEP * L::STRIDE; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

// Tap-major 3x3 gather (k = tap*C + c, a panel inside one tap): thread t
// owns output column t % BN and the k-quads t / BN + j * QSTEP; a quad is 4
// consecutive channels of one input pixel (4 loads HW floats apart), stored
// with one 16-byte LDS write.
template <class Cfg, int KH, int KW, template <int, int> class Panel = SwzPanel>
struct LeanTapB {
  static constexpr int BK = Cfg::BK, BN = Cfg::BN, NT = Cfg::NT;
  static constexpr int QSTEP = NT / BN, NQ = (BK / 4) / QSTEP;
  using L = Panel<BN, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(NT % BN == 0 && (BK / 4) % QSTEP == 0 && NQ >= 1 && KH * KW <= 32, "LeanTapB split");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t colOff;   // byte offset of (image, iy0, ix0, channel 4 * first quad), modulo 2^32
  uint32_t tapMask;  // bit ky*KW + kx: that tap reads inside the image
  uint32_t HW4;
  int C, W;
  int ldsOff[NQ];
  float reg[NQ][4];

  __device__ inline void init(const ConvGeom& g, int64_t n0, int tid) {
    rsrc = make_rsrc(g.x, g.xBytes);
    C = g.C;
    W = g.W;
    HW4 = static_cast<uint32_t>(g.H) * static_cast<uint32_t>(g.W) * 4u;
    const int col = tid % BN, q0 = tid / BN;
    const int64_t n = n0 + col;
    const bool colOk = n < g.N;
    const int64_t nn = colOk ? n : 0;
    const int64_t b = nn / g.OHW;
    const int p = static_cast<int>(nn - b * g.OHW);
    const int oy = p / g.OW, ox = p - (p / g.OW) * g.OW;
    const int iy0 = oy * g.sY - g.pH, ix0 = ox * g.sX - g.pW;
    colOff = static_cast<uint32_t>((b * g.xBatchStride + static_cast<int64_t>(iy0) * g.W + ix0) * 4) +
             static_cast<uint32_t>(4 * q0) * HW4;
    uint32_t m = 0;
#pragma unroll
    for (int ky = 0; ky < KH; ++ky)
#pragma unroll
      for (int kx = 0; kx < KW; ++kx) {
        const bool in = static_cast<unsigned>(iy0 + ky) < static_cast<unsigned>(g.H) &&
                        static_cast<unsigned>(ix0 + kx) < static_cast<unsigned>(g.W);
        m |= (colOk && in ? 1u : 0u) << (ky * KW + kx);
      }
    tapMask = m;
#pragma unroll
    for (int j = 0; j < NQ; ++j) ldsOff[j] = L::chunk(col, q0 + j * QSTEP);
  }
  __device__ inline void load(int64_t k0) {
    const int kk = static_cast<int>(k0);
    const int tap = kk / C;  // uniform
    const int c0 = kk - tap * C;
    const int ky = tap / KW, kx = tap - (tap / KW) * KW;
    const uint32_t vo = sel_off((tapMask >> tap) & 1u, colOff + static_cast<uint32_t>(ky * W + kx) * 4u);
#pragma unroll
    for (int j = 0; j < NQ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        reg[j][e] = buf_ld1s(rsrc, vo, static_cast<uint32_t>(c0 + 4 * j * QSTEP + e) * HW4);
  }
  static constexpr int QUADS = NQ;
  __device__ inline f32x4 quad(int u) const { return f32x4{reg[u][0], reg[u][1], reg[u][2], reg[u][3]}; }
  __device__ inline int off(int u) const { return ldsOff[u]; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

// 1x1 stride 1: B[k = c][n = b*HW + p] = x_b[c][p].  Scalar: as LeanTapB
// without the tap (4 loads HW apart per quad).  VEC (HW % 4 == 0, batch
// stride % 4 == 0, x aligned): thread t owns columns 4 * (t % (BN/4)) .. +3
// and k-quads t / (BN/4) + j * QSTEP; it loads a 4 (k) x 4 (column) block
// with four 16-byte loads and stores its transpose, one 16-byte LDS write
// per column.
template <class Cfg, bool VEC, template <int, int> class Panel = SwzPanel>
struct Lean1x1B {
  static constexpr int BK = Cfg::BK, BN = Cfg::BN, NT = Cfg::NT;
  static constexpr int CPT = VEC ? 4 : 1;
  static constexpr int TPR = BN / CPT;
  static constexpr int QSTEP = NT / TPR, NQ = (BK / 4) / QSTEP;
  using L = Panel<BN, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(NT % TPR == 0 && (BK / 4) % QSTEP == 0 && NQ >= 1, "Lean1x1B split");
  using Reg = typename std::conditional<VEC, f32x4, float>::type;
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t voff, HW4;
  int ldsOff[NQ][CPT];
  Reg reg[NQ][4];

  __device__ inline void init(const ConvGeom& g, int64_t n0, int tid) {
    rsrc = make_rsrc(g.x, g.xBytes);
    const int64_t HW = g.OHW;
    HW4 = static_cast<uint32_t>(HW) * 4u;
    const int col = (tid % TPR) * CPT, q0 = tid / TPR;
    const int64_t n = n0 + col;
    const bool colOk = n < g.N;
    const int64_t nn = colOk ? n : 0;
    const int64_t b = nn / HW;
    voff = sel_off(colOk, static_cast<uint32_t>((b * g.xBatchStride + (nn - b * HW) + 4 * q0 * HW) * 4));
#pragma unroll
    for (int j = 0; j < NQ; ++j)
#pragma unroll
      for (int c = 0; c < CPT; ++c) ldsOff[j][c] = L::chunk(col + c, q0 + j * QSTEP);
  }
  __device__ inline void load(int64_t k0) {
#pragma unroll
    for (int j = 0; j < NQ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t so = static_cast<uint32_t>(static_cast<int>(k0) + 4 * j * QSTEP + e) * HW4;
        if constexpr (VEC)
          reg[j][e] = buf_ld4s(rsrc, voff, so);
        else
          reg[j][e] = buf_ld1s(rsrc, voff, so);
      }
  }
  static constexpr int QUADS = NQ * CPT;
  __device__ inline f32x4 quad(int u) const {
    const int j = u / CPT, c = u % CPT;
    if constexpr (VEC)
      return f32x4{reg[j][0][c], reg[j][1][c], reg[j][2][c], reg[j][3][c]};
    else
      return f32x4{reg[j][0], reg[j][1], reg[j][2], reg[j][3]};
  }
  __device__ inline int off(int u) const { return ldsOff[u / CPT][u % CPT]; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

template <class Cfg, class AL, class BL>
struct LeanLoop {
  static constexpr int FM = Cfg::FM, FN = Cfg::FN, KCH = Cfg::KCH, BK = Cfg::BK;

  // Eight k per lane and 32x32 block as two 16-byte halves: step s uses
  // element s % 4 of half s / 4 (k = 16*chunk + 8*(lane/32) + s).
  struct Frag {
    f32x4 a[FM][2];
    f32x4 b[FN][2];
  };

  // Per-lane float offsets inside a 32-row block of either panel (blocks
  // start at multiples of 32 rows, so a row's swizzle is that of lane % 32):
  // lo[c][e] addresses half e of chunk c.
  struct Lanes {
    int lo[KCH][2];
    int aRow, bRow;  // first row of the wave's blocks, times BK
  };

  __device__ static inline void read(const lds_t* stage, int c, const Lanes& L, Frag& f) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e)
        f.a[i][e] = *reinterpret_cast<const lds_f4*>(stage + L.aRow + i * 32 * BK + L.lo[c][e]);
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e)
        f.b[j][e] = *reinterpret_cast<const lds_f4*>(stage + AL::SIZE + L.bRow + j * 32 * BK + L.lo[c][e]);
  }

  __device__ static inline void mma(const Frag& f, f32x16 (&acc)[FM][FN]) {
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[i][s >> 2][s & 3], f.b[j][s >> 2][s & 3], acc[i][j], 0,
                                                           0, 0);
  }

  __device__ static inline Lanes lanes() {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
    const int r = lane & 31, h = lane >> 5;
    Lanes L;
#pragma unroll
    for (int c = 0; c < KCH; ++c)
#pragma unroll
      for (int e = 0; e < 2; ++e) L.lo[c][e] = SwzPanel<32, BK>::chunk(r, 4 * c + 2 * h + e);
    L.aRow = wm * Cfg::WTM * BK;
    L.bRow = wn * Cfg::WTN * BK;
    return L;
  }

  __device__ static inline void zero(f32x16 (&acc)[FM][FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  }

  __device__ static inline void add(f32x16 (&acc)[FM][FN], const f32x16 (&g)[FM][FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = acc[i][j][e] + g[i][j][e];
  }
};

}  // namespace conv
}  // namespace tnh
