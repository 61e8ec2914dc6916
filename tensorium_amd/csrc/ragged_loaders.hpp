// Operand loaders for the sizes and strides that the vector loaders of
// lean_loop.hpp and split_loop.hpp do not take: any K (elements past it read
// 0), any leading dimension, any row count, any float's address.
//
// They load four floats at a time all the same: a buffer load of several
// dwords needs only the first one's alignment, and its range is checked dword
// by dword against voffset + soffset (seen on gfx950), so a quad that runs
// past the operand's last element reads zeros there and nothing beyond.
#pragma once
#include "split_loop.hpp"

namespace tnh {
namespace conv {

// k-contiguous rows in LeanRowsK's split of the panel.  A quad that crosses K
// holds the next row's first elements, which are cleared when it is used.
template <int ROWS, int NT_, template <int, int> class Panel>
struct RowsTailK {
  static constexpr int BK = 32, NT = NT_, ROWSTEP = NT / 8, QUADS = ROWS / ROWSTEP;
  using L = Panel<ROWS, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(ROWS % ROWSTEP == 0 && ROWSTEP % 16 == 0, "RowsTailK split");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t voff[QUADS];
  int ldsOff, kq4, K, left;  // left: elements of this thread's quad before K
  f32x4 reg[QUADS];

  __device__ inline void init(const float* p, int64_t bytes, int64_t ld, int64_t rows, int64_t r0, int tid) {
    rsrc = make_rsrc(p, bytes);
    kq4 = 4 * (tid % 8);
#pragma unroll
    for (int v = 0; v < QUADS; ++v) {
      const int64_t gr = r0 + tid / 8 + v * ROWSTEP;
      voff[v] = gr < rows ? static_cast<uint32_t>((gr * ld + kq4) * 4) : kOOB;
    }
    ldsOff = L::chunk(tid / 8, tid % 8);
    K = left = 0;
  }
  __device__ inline void klimit(int64_t k) { K = static_cast<int>(k); }
  __device__ inline void load(int64_t k0) {
    const uint32_t so = static_cast<uint32_t>(k0) * 4u;
    left = K - static_cast<int>(k0) - kq4;
#pragma unroll
    for (int v = 0; v < QUADS; ++v) reg[v] = buf_ld4s(rsrc, sel_off(left > 0, voff[v]), so);
  }
  __device__ inline f32x4 quad(int u) const {
    return f32x4{reg[u][0], left > 1 ? reg[u][1] : 0.f, left > 2 ? reg[u][2] : 0.f, left > 3 ? reg[u][3] : 0.f};
  }
  __device__ inline int off(int u) const { return ldsOff + u * ROWSTEP * L::STRIDE; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

// Row-contiguous operand in SplitRowsMN's units.  A unit that crosses the last
// row holds elements of the next k there, which reach only sums that are not
// stored.
template <int ROWS, int NT_, template <int, int> class Panel>
struct RowsTailMN {
  static constexpr int BK = 32, NT = NT_;
  static constexpr int CPT = ROWS * 2 >= NT ? 4 : (ROWS * 4 >= NT ? 2 : 1);
  static constexpr int UNITS = ROWS / CPT * 8, NQ = UNITS / NT;
  using L = Panel<ROWS, BK>;
  static constexpr int SIZE = L::SIZE;
  static_assert(UNITS % NT == 0 && NQ >= 1 && NT % 32 == 0, "RowsTailMN split");
  using Reg = float __attribute__((ext_vector_type(CPT)));
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t voff[NQ], ld4;
  int ldsOff[NQ][CPT], k4[NQ], K;
  Reg reg[NQ][4];

  // rowOff(row): as SplitRowsMN's
  template <class F>
  __device__ inline void init_rows(const float* p, int64_t bytes, int64_t ld, int tid, F&& rowOff) {
    rsrc = make_rsrc(p, bytes);
    ld4 = static_cast<uint32_t>(ld) * 4u;
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      const int u = tid + j * NT;
      const int row = CPT * ((u & 3) | (u >> 5 << 2)), kq = (u >> 2) & 7;
      const uint32_t o = rowOff(row);
      voff[j] = o != kOOB ? o + static_cast<uint32_t>(4 * kq) * ld4 : kOOB;  // wraps only past K
      k4[j] = 4 * kq;
#pragma unroll
      for (int c = 0; c < CPT; ++c) ldsOff[j][c] = L::chunk(row + c, kq);
    }
    K = 0;
  }
  __device__ inline void init(const float* p, int64_t bytes, int64_t ld, int64_t rows, int64_t r0, int tid) {
    init_rows(p, bytes, ld, tid,
              [&](int row) { return r0 + row < rows ? static_cast<uint32_t>((r0 + row) * 4) : kOOB; });
  }
  __device__ inline void klimit(int64_t k) { K = static_cast<int>(k); }
  __device__ inline void load(int64_t k0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t so = static_cast<uint32_t>(min(static_cast<int>(k0) + e, K - 1)) * ld4;  // kOOB
#pragma unroll
      for (int j = 0; j < NQ; ++j) {
        const uint32_t vo = sel_off(static_cast<int>(k0) + k4[j] + e < K, voff[j]);
        if constexpr (CPT == 4)
          reg[j][e] = buf_ld4s(rsrc, vo, so);
        else if constexpr (CPT == 2)
          reg[j][e] = __builtin_bit_cast(Reg, __builtin_amdgcn_raw_buffer_load_b64(rsrc, vo, so, 0));
        else
          reg[j][e] = buf_ld1s(rsrc, vo, so);
      }
    }
  }
  static constexpr int QUADS = NQ * CPT;
  __device__ inline f32x4 quad(int u) const {
    const int j = u / CPT, c = u % CPT;
    return f32x4{reg[j][0][c], reg[j][1][c], reg[j][2][c], reg[j][3][c]};
  }
  __device__ inline int off(int u) const { return ldsOff[u / CPT][u % CPT]; }
  __device__ inline void store(lds_t* stage) const { store_quads(*this, stage); }
};

}  // namespace conv
}  // namespace tnh
