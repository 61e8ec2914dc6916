"""Outputs and operands whose rows lie so far apart that 63 of them pass 2^31
bytes: a tile's rows past the last one write and read nothing.  Whole numbers,
every sum exact."""
import numpy as np
import pytest
import torch

from tensorium_amd.nnhip import CONV_SPLIT_UNIT, WEIGHTS_REFERENCE, WEIGHTS_TAP_MAJOR, acLINEAR

pytestmark = pytest.mark.gpu

SGEMM_CFGS = (-1, 2, 3, 4, 5, 9, 10, 11, 12)


def ints(shape, seed, lo=-4, hi=5):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(lo, hi, shape, generator=g, device="cuda").float()


@pytest.mark.parametrize("cfg", SGEMM_CFGS)
@pytest.mark.parametrize("M", [1, 3])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_sgemm_long_c_rows(hip, cfg, M, beta):
    N, K, ldc = 96, 32, 1 << 24  # row 32 of a tile is 2^31 bytes from row 0
    print(f"[case] sgemm long C rows cfg {cfg} M {M} beta {beta}", flush=True)
    A, B = ints((M, K), 1), ints((K, N), 2)
    C = torch.full(((M - 1) * ldc + N,), 7.0, device="cuda")
    torch.cuda.synchronize()
    hip.setSgemmAutotune(True, cfg)
    try:
        hip.gemm(0, 0, M, N, K, 1.0, A, 0, K, B, 0, N, beta, C, 0, ldc)
    finally:
        hip.setSgemmAutotune(True, -1)
    hip.finish()
    ref = A.cpu().numpy() @ B.cpu().numpy() + 7.0 * beta
    for m in range(M):
        assert np.array_equal(C[m * ldc:m * ldc + N].cpu().numpy(), ref[m])
    gaps = (C == 7.0).sum().item()
    assert gaps >= (M - 1) * (ldc - N)


@pytest.mark.parametrize("cfg", (-1, 10, 11, 12))
@pytest.mark.parametrize("log2ld", [28, 29])  # the third or second k is 2^31 bytes on
def test_sgemm_long_operand_rows(hip, cfg, log2ld):
    M, N, K, ld = 3, 5, 1, 1 << log2ld
    print(f"[case] sgemm long operand rows cfg {cfg} ld 2^{log2ld}", flush=True)
    A, B, C = ints((M,), 3, 1), ints((N,), 4, 1), torch.zeros(M, N, device="cuda")
    torch.cuda.synchronize()
    hip.setSgemmAutotune(True, cfg)
    try:
        hip.gemm(1, 0, M, N, K, 1.0, A, 0, ld, B, 0, ld, 0.0, C, 0, N)
    finally:
        hip.setSgemmAutotune(True, -1)
    hip.finish()
    assert np.array_equal(C.cpu().numpy(), np.outer(A.cpu().numpy(), B.cpu().numpy()))


@pytest.mark.parametrize("cfg", [27, 28, 29, 30, 28 + 2 * CONV_SPLIT_UNIT])
def test_gather_conv_large_image(hip, cfg):
    F, O, k = 3, 4096, 5  # 2^26 bytes a filter
    print(f"[case] gather conv {k}x{k} {O}x{O} cfg {cfg}", flush=True)
    x, w = ints((O + k - 1, O + k - 1), 5), ints((F, k, k), 6)
    out = torch.full((F, O, O), 77.0, device="cuda")
    torch.cuda.synchronize()
    hip.setConvAutotune(True, cfg)
    try:
        hip.conv2dForward(1, 1, O + k - 1, O + k - 1, F, k, 1, 0, x, 0, w, None, acLINEAR, out, 0,
                          weightLayout=WEIGHTS_REFERENCE)
    finally:
        hip.setConvAutotune(True, -1)
    hip.finish()
    for f in range(F):
        ref = torch.zeros(O, O, device="cuda")
        for i in range(k):
            for j in range(k):
                ref += w[f, i, j] * x[i:i + O, j:j + O]
        assert torch.equal(out[f], ref), f


@pytest.mark.parametrize("cfg", [11, 12, 13, 14, 15, 17, 18, 19])
def test_lean_conv_large_image(hip, cfg):
    C, F, H, W = 32, 3, 2932, 2936  # row 63 is 2^31 + 2^24 bytes from row 0
    print(f"[case] lean conv 1x1 {H}x{W} cfg {cfg}", flush=True)
    x, w = ints((C, H, W), 7), ints((F, C), 8)
    out = torch.full((F, H, W), 77.0, device="cuda")
    torch.cuda.synchronize()
    hip.setConvAutotune(True, cfg)
    try:
        hip.conv2dForward(1, C, H, W, F, 1, 1, 0, x, 0, w, None, acLINEAR, out, 0, weightLayout=WEIGHTS_TAP_MAJOR)
    finally:
        hip.setConvAutotune(True, -1)
    hip.finish()
    for f in range(F):
        ref = torch.zeros(H, W, device="cuda")
        for c in range(C):
            ref += w[f, c] * x[c]
        assert torch.equal(out[f], ref), f


@pytest.mark.parametrize("cfg", range(11, 20))
@pytest.mark.parametrize("res", [False, True])
def test_channels_last_long_pixels(hip, cfg, res):
    C, F, pix = 32, 8, 1 << 24  # one pixel, the next 2^26 bytes on
    print(f"[case] channels-last long pixels cfg {cfg} residual {res}", flush=True)
    x, w, r = ints((C,), 9), ints((F, C), 10), ints((F,), 11)
    out = torch.full((F,), 77.0, device="cuda")
    torch.cuda.synchronize()
    hip.setConvAutotune(True, cfg)
    try:
        hip.conv2dForwardNHWC(1, C, 1, 1, F, 1, 1, 0, x, 0, w, None, acLINEAR, out, 0, outPix=pix,
                              residual=r if res else None, resOffset=0, resPix=pix if res else None)
    finally:
        hip.setConvAutotune(True, -1)
    hip.finish()
    ref = w.cpu().numpy() @ x.cpu().numpy() + (r.cpu().numpy() if res else 0)
    assert np.array_equal(out.cpu().numpy(), ref)
