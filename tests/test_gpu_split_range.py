"""The bf16-part products (csrc/split_loop.hpp) over the whole range of floats,
on every kernel that forms them.  Each sum holds one product that is not zero,
so nothing else hides its error: the bound is six bf16 instructions and two
roundings, 2^-21 of the product, where a lost third part costs up to 2^-18 and
a lost second one 2^-9; or 2^-149, the smallest step of a float."""
import numpy as np
import pytest
import torch

from tensorium_amd import synth
from tensorium_amd.nnhip import WEIGHTS_REFERENCE, WEIGHTS_TAP_MAJOR, acLINEAR

pytestmark = pytest.mark.gpu

LEAN_SGEMM, RAGGED_SGEMM = (2, 3, 4, 5, 9), (10, 11, 12)
# exponents of the two operands: ordinary; parts under bf16's smallest step
# beside a large partner; subnormals; a partner past the lift; both at the
# range's ends; products at the smallest step
SCALES = [(0, 0), (-110, 90), (-116, 100), (-124, 101), (-126, 126), (-134, 126), (-140, 126), (-149, 120), (100, -126),
          (126, -140), (103, 0), (0, 104), (60, 60), (-75, -74), (-126, -10), (-100, -49)]


def values(seed, shape, e):
    """24-bit values of either sign times 2^e, as the nearest floats (e < -126: subnormals)."""
    v = synth.uniform(seed, shape, 1.0, 2.0).astype(np.float64) * np.where(synth.uniform(seed + 1, shape) < 0.5, -1, 1)
    return (v * 2.0 ** e).astype(np.float32)


def one_hot(seed, rows, K, e):
    """[rows][K] with one value a row, every k taken in turn."""
    a = np.zeros((rows, K), np.float32)
    a[np.arange(rows), (5 * np.arange(rows) + 3) % K] = values(seed, (rows,), e)
    return a


def check(got, a, b):
    """got [M][N] = a [M][K] times b [K][N], one product a sum."""
    ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.all(np.abs(got - ref) <= 8 * 2.0 ** -24 * np.abs(ref) + 2.0 ** -149)


def D(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("cfg", LEAN_SGEMM + RAGGED_SGEMM)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_sgemm(hip, cfg, ta, tb):
    lean = cfg in LEAN_SGEMM
    M, N, K = (132, 260, 96) if lean else (131, 259, 67)
    for e, f in SCALES:
        print(f"[case] sgemm range cfg {cfg} ta {ta} tb {tb} 2^{e} x 2^{f}", flush=True)
        A, B = one_hot(900, M, K, e), values(910, (K, N), f)
        dA, dB, dC = D(A.T if ta else A), D(B.T if tb else B), torch.zeros(M, N, device="cuda")
        torch.cuda.synchronize()
        hip.setSgemmAutotune(True, cfg)
        try:
            hip.gemm(ta, tb, M, N, K, 1.0, dA, 0, M if ta else K, dB, 0, K if tb else N, 0.0, dC, 0, N)
        finally:
            hip.setSgemmAutotune(True, -1)
        hip.finish()
        check(dC.cpu().numpy(), A, B)


@pytest.mark.parametrize("cfg", LEAN_SGEMM + RAGGED_SGEMM)
def test_one_tiny_value_among_ordinary_ones(hip, cfg):
    """One element of 2^-124 beside a row's 2^-40: with partners of 2^101 it decides its sums."""
    print(f"[case] sgemm one tiny value cfg {cfg}", flush=True)
    M, N, K = 132, 260, 96
    A, B = synth.uniform(920, (M, K), -1, 1) * np.float32(2.0 ** -40), synth.uniform(921, (K, N), -1, 1)
    A[:, 40] = 0
    A[77, 40], B[40] = np.float32(1.7 * 2.0 ** -124), values(922, (N,), 101)
    dA, dB, dC = D(A), D(B), torch.zeros(M, N, device="cuda")
    torch.cuda.synchronize()
    hip.setSgemmAutotune(True, cfg)
    try:
        hip.gemm(0, 0, M, N, K, 1.0, dA, 0, K, dB, 0, N, 0.0, dC, 0, N)
    finally:
        hip.setSgemmAutotune(True, -1)
    hip.finish()
    a, b = A.astype(np.float64), B.astype(np.float64)
    # 24 bf16 instructions of a group of 64 k, two groups, two roundings
    assert np.all(np.abs(dC.cpu().numpy() - a @ b) <= 28 * 2.0 ** -24 * (np.abs(a) @ np.abs(b)))


@pytest.mark.parametrize("cfg,nhwc", [(c, n) for n in (False, True) for c in [*range(11, 20), *range(27, 31)]
                                      if c < 27 or not n])
def test_conv_1x1(hip, cfg, nhwc):
    B, C, H, W, F = 2, 32, 9, 16, 72
    for e, f in SCALES:
        print(f"[case] conv range cfg {cfg} nhwc {nhwc} 2^{e} x 2^{f}", flush=True)
        w, x = one_hot(930, F, C, e), values(940, (C, B, H, W), f)
        dw, out = D(w), torch.zeros((B, H, W, F) if nhwc else (B, F, H, W), device="cuda")
        dx = D(x.transpose(1, 2, 3, 0) if nhwc else x.transpose(1, 0, 2, 3))
        torch.cuda.synchronize()
        hip.setConvAutotune(True, cfg)
        try:
            if nhwc:
                hip.conv2dForwardNHWC(B, C, H, W, F, 1, 1, 0, dx, 0, dw, None, acLINEAR, out, 0)
            else:
                hip.conv2dForward(B, C, H, W, F, 1, 1, 0, dx, 0, dw, None, acLINEAR, out, 0,
                                  weightLayout=WEIGHTS_TAP_MAJOR)
        finally:
            hip.setConvAutotune(True, -1)
        hip.finish()
        got = out.cpu().numpy()
        got = got.reshape(B * H * W, F).T if nhwc else got.transpose(1, 0, 2, 3).reshape(F, -1)
        check(got, w, x.reshape(C, -1))


@pytest.mark.parametrize("C", [12, 20])
def test_conv_channels_last_any_channels(hip, C):
    """The fixed tiles of channel counts that are no multiple of 32, 3x3: the middle tap's weights alone."""
    B, H, W, F = 2, 9, 16, 72
    for e, f in SCALES:
        print(f"[case] conv range any channels {C} 2^{e} x 2^{f}", flush=True)
        w1, x = one_hot(935, F, C, e), values(945, (B, H, W, C), f)
        w = np.zeros((F, 3, 3, C), np.float32)
        w[:, 1, 1] = w1
        out = torch.zeros((B, H, W, F), device="cuda")
        dx, dw = D(x), D(w)
        torch.cuda.synchronize()
        hip.conv2dForwardNHWC(B, C, H, W, F, 3, 1, 1, dx, 0, dw, None, acLINEAR, out, 0)
        hip.finish()
        check(out.cpu().numpy().reshape(-1, F).T, w1, x.reshape(-1, C).T)


@pytest.mark.parametrize("cfg", range(27, 31))
def test_conv_5x5(hip, cfg):
    """A window of which one weight a filter is not zero, over an image of one window."""
    C, k, F = 5, 5, 40
    for e, f in SCALES:
        print(f"[case] conv 5x5 range cfg {cfg} 2^{e} x 2^{f}", flush=True)
        w, x = one_hot(950, F, C * k * k, e), values(960, (C * k * k, 1), f)
        out, dw, dx = torch.zeros(F, 1, device="cuda"), D(w), D(x)
        torch.cuda.synchronize()
        hip.setConvAutotune(True, cfg)
        try:
            hip.conv2dForward(1, C, k, k, F, k, 1, 0, dx, 0, dw, None, acLINEAR, out, 0, weightLayout=WEIGHTS_REFERENCE)
        finally:
            hip.setConvAutotune(True, -1)
        hip.finish()
        check(out.cpu().numpy(), w, x)


@pytest.mark.parametrize("F,C,k,H,W", [(20, 5, 1, 7, 8), (70, 40, 3, 9, 5), (130, 40, 3, 8, 8), (40, 130, 1, 6, 7)])
def test_weight_gradient(hip, F, C, k, H, W):
    """One pixel's delta a filter: the gradients are single products (1x1 and the windows over it)."""
    L = H * W
    for e, f in SCALES:
        print(f"[case] wgrad range F {F} C {C} k {k} {H}x{W} 2^{e} x 2^{f}", flush=True)
        d, x = one_hot(970, F, L, e), values(980, (C, H, W), f)
        p = k // 2
        xp = np.pad(x, ((0, 0), (p, p), (p, p)))
        col = np.stack([xp[:, i:i + H, j:j + W] for i in range(k) for j in range(k)], 1).reshape(C * k * k, L)
        dW, dd, dx = torch.zeros(F, C * k * k, device="cuda"), D(d), D(x)
        torch.cuda.synchronize()
        hip.convWeightGradient(1, C, H, W, F, k, k, p, p, 1, 1, 1, 1, dx, C * L, dd, F * L, 1.0, 0.0, dW)
        hip.finish()
        check(dW.cpu().numpy(), d, col.T)
