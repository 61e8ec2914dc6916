// SGEMM over any sizes, leading dimensions and alignment on the bf16-part
// tiles, with split K; the lean tiles (sgemm.hip) take what is whole panels of
// aligned vectors.  They replace fp32 tiles that loaded one float at a time
// through two registers of prefetch and never split K: 255x1531x10817 NT
// 325 -> 58 us.
#include "ragged_loaders.hpp"
#include "sgemm_tiles.hpp"

namespace tnh {
namespace {

template <int ROWS, int NT, bool KC, template <int, int> class P>
struct Op {  // k contiguous
  using type = conv::RowsTailK<ROWS, NT, P>;
};
template <int ROWS, int NT, template <int, int> class P>
struct Op<ROWS, NT, false, P> {  // rows contiguous
  using type = conv::RowsTailMN<ROWS, NT, P>;
};

template <class Cfg, bool TA, bool TB>
__global__ __launch_bounds__(Cfg::NT, Cfg::OCC) void sgemm_ragged_kernel(SgemmArgs a) {
  using AL = typename Op<Cfg::BM, Cfg::NT, !TA, conv::SplitPanel>::type;
  using AF = typename Op<Cfg::BM, Cfg::NT, !TA, conv::SwzPanel>::type;
  using BL = typename Op<Cfg::BN, Cfg::NT, TB, conv::SplitPanel>::type;
  using BF = typename Op<Cfg::BN, Cfg::NT, TB, conv::SwzPanel>::type;
  using Loop = conv::SplitLoop<Cfg, AL, BL>;
  __shared__ __attribute__((aligned(16))) float smem[Loop::LDS_FLOATS];
  __shared__ int odd;
  lds_t* lds = (lds_t*)smem;
  const int64_t bz = blockIdx.y;
  int tm, tn;
  tile_coords(blockIdx.x, a.tilesM, a.tilesN, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * Cfg::BM, n0 = static_cast<int64_t>(tn) * Cfg::BN;
  auto init = [&](auto& al, auto& bl) {
    al.init(a.A + bz * a.strideA, a.aBytes, a.lda, a.M, m0, threadIdx.x);
    al.klimit(a.K);
    bl.init(a.B + bz * a.strideB, a.bBytes, a.ldb, a.N, n0, threadIdx.x);
    bl.klimit(a.K);
  };
  int64_t kBegin, kEnd;
  sgemm_range(a, kBegin, kEnd);
  const int64_t nk = (kEnd - kBegin + 31) / 32;
  AL al;
  BL bl;
  init(al, bl);
  f32x16 acc[Cfg::FM][Cfg::FN];
  Loop::exec(al, bl, kBegin, nk, lds, &odd, acc);
  if (!Loop::finite(acc, &odd)) {
    AF af;
    BF bf;
    init(af, bf);
    conv::PlainLoop<Cfg, AF, BF>::exec(af, bf, kBegin, nk, lds, acc);
  }
  sgemm_store<Cfg>(a, bz, m0, n0, acc);
}

using R128 = conv::LeanCfg<128, 128, 32, 2, 4, 2>;
using R64x128 = conv::LeanCfg<64, 128, 32, 2, 2, 2>;
using R64 = conv::LeanCfg<64, 64, 32, 2, 2, 3>;

template <class Cfg>
int run(SgemmArgs a, int64_t batch, bool ta, bool tb, hipStream_t s) {
  const int64_t tm = (a.M + Cfg::BM - 1) / Cfg::BM, tn = (a.N + Cfg::BN - 1) / Cfg::BN;
  if (tm * tn > INT32_MAX || batch > 65535)
    return fail(TNH_ERR_UNSUPPORTED, "sgemm: grid too large (%lld tiles, batch %lld)", (long long)(tm * tn),
                (long long)batch);
  a.tilesM = static_cast<int>(tm);
  a.tilesN = static_cast<int>(tn);
  const dim3 grid(static_cast<unsigned>(tm * tn), static_cast<unsigned>(batch), static_cast<unsigned>(a.splits));
  if (!ta && !tb)
    hipLaunchKernelGGL((sgemm_ragged_kernel<Cfg, false, false>), grid, dim3(Cfg::NT), 0, s, a);
  else if (!ta)
    hipLaunchKernelGGL((sgemm_ragged_kernel<Cfg, false, true>), grid, dim3(Cfg::NT), 0, s, a);
  else if (!tb)
    hipLaunchKernelGGL((sgemm_ragged_kernel<Cfg, true, false>), grid, dim3(Cfg::NT), 0, s, a);
  else
    hipLaunchKernelGGL((sgemm_ragged_kernel<Cfg, true, true>), grid, dim3(Cfg::NT), 0, s, a);
  return launch_status("sgemm_ragged_kernel");
}

}  // namespace

int launch_sgemm_ragged(int i, SgemmArgs a, int64_t batch, bool ta, bool tb, hipStream_t s) {
  switch (i) {
    case 0: return run<R128>(a, batch, ta, tb, s);
    case 1: return run<R64x128>(a, batch, ta, tb, s);
    default: return run<R64>(a, batch, ta, tb, s);
  }
}

}  // namespace tnh
