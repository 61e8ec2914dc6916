"""SGEMM's K splits and its tiles for any operands (csrc/sgemm.hip,
csrc/sgemm_ragged.hip): pinned configurations, odd sizes, leading dimensions
and bases, against float64, element by element."""
import numpy as np
import pytest
import torch

from tensorium_amd import synth
from tensorium_amd.nnhip import SGEMM_SPLIT_UNIT

pytestmark = pytest.mark.gpu

LEAN, RAGGED = (2, 3, 4, 5), (10, 11, 12)
FORMS = [(0, 0), (0, 1), (1, 0), (1, 1)]


def gemm(hip, cfg, A, B, ta=0, tb=0, alpha=1.0, beta=0.0, C=None, pad=0, off=0):
    """alpha op(A) op(B) + beta C through leading dimensions `pad` past the
    rows, operands `off` floats into their buffers; what the pads hold (NaN
    beside the operands) must not be used or changed."""
    M, N = A.shape[0], B.shape[1]

    def put(x, fill):
        x = np.ascontiguousarray(x)
        buf = np.full(off + x.shape[0] * (x.shape[1] + pad), fill, np.float32)
        buf[off:].reshape(x.shape[0], -1)[:, :x.shape[1]] = x
        return torch.from_numpy(buf).cuda(), x.shape[1] + pad

    dA, lda = put(A.T if ta else A, np.nan)
    dB, ldb = put(B.T if tb else B, np.nan)
    dC, ldc = put(np.full((M, N), 9.0, np.float32) if C is None else C, 77.0)
    torch.cuda.synchronize()
    hip.setSgemmAutotune(True, cfg)
    try:
        hip.gemm(ta, tb, M, N, A.shape[1], alpha, dA, off, lda, dB, off, ldb, beta, dC, off, ldc)
    finally:
        hip.setSgemmAutotune(True, -1)
    hip.finish()
    got = dC.cpu().numpy()
    assert (got[:off] == 77).all()
    got = got[off:].reshape(M, -1)
    assert (got[:, N:] == 77).all()
    return got[:, :N]


def bound(A, B, splits=1):
    """24 bf16 instructions of a group of 64 k, the groups', the splits' and alpha's roundings."""
    K = A.shape[1]
    steps = min(24, 6 * -(-K // 16)) + -(-K // 64) + splits
    return (steps + 2) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))


@pytest.mark.parametrize("cfg", LEAN + RAGGED)
@pytest.mark.parametrize("splits", [2, 3, 7])
@pytest.mark.parametrize("ta,tb", FORMS)
def test_k_split(hip, cfg, splits, ta, tb):
    """Splits that K's panels do not divide into, the last one short, for the
    any-operand tiles with a last panel that is not whole; sizes below and past
    a tile."""
    lean = cfg in LEAN
    for M, N, K, pad, off in ([(132, 260, 352, 4, 4), (4, 8, 320, 0, 0)] if lean else
                              [(131, 259, 353, 3, 1), (5, 3, 321, 0, 0), (1, 70, 417, 1, 2)]):
        for alpha, beta in ((1.0, 0.0), (0.5, 1.0)):
            print(f"[case] sgemm split cfg {cfg} splits {splits} {M}x{N}x{K} ta {ta} tb {tb} beta {beta}", flush=True)
            A, B = synth.normal(300 + K, (M, K)), synth.normal(400 + K, (K, N))
            C = synth.normal(500, (M, N))
            got = gemm(hip, cfg + SGEMM_SPLIT_UNIT * splits, A, B, ta, tb, alpha, beta, C, pad, off)
            ref = alpha * (A.astype(np.float64) @ B.astype(np.float64)) + beta * C.astype(np.float64)
            assert np.all(np.abs(got - ref) <= alpha * bound(A, B, splits) + 2.0 ** -23 * np.abs(ref))


@pytest.mark.parametrize("cfg", (2, 5, 10, 12))
def test_more_splits_than_panels(hip, cfg):
    """K of three panels in 64 splits: one panel each."""
    print(f"[case] sgemm more splits than panels cfg {cfg}", flush=True)
    A, B = np.round(synth.normal(601, (40, 96), 2.0)), np.round(synth.normal(602, (96, 36), 2.0))
    assert np.array_equal(gemm(hip, cfg + SGEMM_SPLIT_UNIT * 64, A, B), A @ B)


def test_splits_that_are_refused(hip):
    A, B = np.ones((32, 64), np.float32), np.ones((64, 32), np.float32)
    for cfg in (0, 1, 6, 9):
        with pytest.raises(Exception, match="does not split"):
            gemm(hip, cfg + SGEMM_SPLIT_UNIT * 2, A, B)
    for bad in (13, 63, 64 + 13, 65 * 64):
        with pytest.raises(Exception, match="config"):
            hip.setSgemmAutotune(True, bad)


@pytest.mark.parametrize("cfg", RAGGED)
@pytest.mark.parametrize("ta,tb", FORMS)
@pytest.mark.parametrize("K", [1, 2, 5, 31, 33, 63, 67, 95, 129, 1153])
def test_any_operands_against_float64(hip, cfg, ta, tb, K):
    print(f"[case] ragged sgemm cfg {cfg} K {K} ta {ta} tb {tb}", flush=True)
    M, N = 135, 261
    A, B = synth.normal(700 + K, (M, K)), synth.uniform(800 + K, (K, N), 0.0, 1.0)
    A[7] *= 1e-12
    B[:, 5] *= 1e15
    got = gemm(hip, cfg, A, B, ta, tb, pad=5, off=3)
    assert np.all(np.abs(got - A.astype(np.float64) @ B.astype(np.float64)) <= bound(A, B))


@pytest.mark.parametrize("cfg", RAGGED)
@pytest.mark.parametrize("ta,tb", FORMS)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_any_operands_values_without_parts(hip, cfg, ta, tb, value):
    """One such value in A's last row and column, beside the padding; and in
    B's: the tile is computed again in fp32 through the same odd strides."""
    print(f"[case] ragged sgemm cfg {cfg} ta {ta} tb {tb} value {value}", flush=True)
    M, N, K = 131, 259, 67
    for where in ("A", "B"):
        A, B = synth.uniform(51, (M, K), -1, 1), synth.uniform(52, (K, N), 0.25, 0.75)
        B[K - 1, ::3] = 0.0  # inf * 0
        if where == "A":
            A[M - 1, K - 1] = value
        else:
            B[K - 1, N - 1] = value
        got = gemm(hip, cfg, A, B, ta, tb, pad=5, off=3)
        with np.errstate(all="ignore"):
            ref = A.astype(np.float64) @ B.astype(np.float64)
            limit = bound(A, B)
        plain = np.isfinite(ref)
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[~plain & ~np.isnan(ref)], ref[~plain & ~np.isnan(ref)])
        # the fp32 tile adds K products in one chain
        assert np.all(np.abs(got[plain] - ref[plain]) <= (limit * K)[plain])
