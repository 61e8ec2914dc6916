"""NCHW convolutions that no lean tile takes (csrc/conv_gather.hip): any
kernel size, channel count, weight layout and alignment, on integer data (every
partial sum is exact) against a float64 im2col product."""
import numpy as np
import pytest
import torch

from tensorium_amd import synth
from tensorium_amd.nnhip import CONV_SPLIT_UNIT, WEIGHTS_REFERENCE, WEIGHTS_TAP_MAJOR, acLEAKY

pytestmark = pytest.mark.gpu

GATHER = range(27, 31)
# (B, C, H, W, F, kh, kw, stride, padH, padW): K = 1; K % 4 = 1, 2, 3, 0; masks of 32 rows; windows wider than the
# image; filters and pixels around the tiles' edges
SHAPES = [
    (1, 1, 1, 1, 1, 1, 1, 1, 0, 0),
    (2, 5, 9, 7, 33, 5, 5, 1, 2, 2),
    (2, 3, 11, 11, 31, 7, 7, 2, 3, 3),
    (1, 31, 8, 9, 65, 1, 3, 1, 0, 1),
    (2, 13, 6, 10, 129, 1, 1, 2, 0, 0),
    (1, 2, 40, 5, 20, 32, 2, 1, 3, 0),
    (2, 2, 5, 40, 20, 2, 32, 3, 0, 5),
    (3, 48, 8, 17, 100, 3, 3, 1, 1, 1),
    (1, 70, 13, 13, 64, 3, 3, 1, 1, 1),
    (2, 3, 4, 4, 40, 5, 5, 1, 4, 4),
    # 1x1 over whole planes, pixels a multiple of 4: rows of pixels in units of 2 and 4
    (2, 13, 6, 10, 129, 1, 1, 1, 0, 0),
    (3, 70, 7, 8, 65, 1, 1, 1, 0, 0),
    (1, 33, 1, 4, 20, 1, 1, 1, 0, 0),
    (5, 1, 2, 2, 3, 1, 1, 1, 0, 0),
    # no multiple of 4: tiles with and without an image's end
    (3, 33, 13, 15, 40, 1, 1, 1, 0, 0),
    (2, 6, 1, 129, 33, 1, 1, 1, 0, 0),
    (2, 35, 23, 29, 130, 1, 1, 1, 0, 0),
    (3, 9, 37, 57, 40, 1, 1, 1, 0, 0),
]


def conv64(x, w, s, ph, pw):
    B, C, H, W = x.shape
    F, _, kh, kw = w.shape
    OH, OW = (H + 2 * ph - kh) // s + 1, (W + 2 * pw - kw) // s + 1
    xp = np.zeros((B, C, H + 2 * ph, W + 2 * pw))
    xp[:, :, ph:ph + H, pw:pw + W] = x
    out = np.zeros((B, F, OH, OW))
    for i in range(kh):
        for j in range(kw):
            win = xp[:, :, i:i + s * (OH - 1) + 1:s, j:j + s * (OW - 1) + 1:s]
            out += np.einsum("fc,bcyx->bfyx", w[:, :, i, j].astype(np.float64), win)
    return out


@pytest.mark.parametrize("cfg", list(GATHER) + [-1])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("layout", [WEIGHTS_REFERENCE, WEIGHTS_TAP_MAJOR])
def test_gather_integer(hip, cfg, shape, layout):
    B, C, H, W, F, kh, kw, s, ph, pw = shape
    print(f"[case] conv gather cfg {cfg} {shape} layout {layout}", flush=True)
    x, w = np.round(synth.normal(1200, (B, C, H, W), 2.0)), np.round(synth.normal(1201, (F, C, kh, kw), 1.5))
    bias = np.round(synth.normal(1202, (F,), 2.0))
    ref = conv64(x, w, s, ph, pw) + bias[:, None, None]
    ref = np.where(ref < 0, np.float32(0.1) * ref.astype(np.float32), ref).astype(np.float32)
    res = np.round(synth.normal(1203, ref.shape, 3.0))
    ref = ref + res
    n = ref[0].size
    wl = w if layout == WEIGHTS_REFERENCE else w.transpose(0, 2, 3, 1)
    # operands at odd offsets of their buffers: no 16-byte alignment anywhere; images apart
    dx = torch.zeros(3 + B * (C * H * W + 5), device="cuda")
    for b in range(B):
        dx[3 + b * (C * H * W + 5):][:C * H * W] = torch.from_numpy(x[b].ravel()).cuda()
    dw = torch.zeros(1 + w.size, device="cuda")
    dw[1:] = torch.from_numpy(np.ascontiguousarray(wl).ravel()).cuda()
    dr = torch.from_numpy(np.ascontiguousarray(res)).cuda()
    out = torch.full((2 + B * (n + 7),), 77.0, device="cuda")
    db = torch.from_numpy(bias).cuda()
    splits = [0] if cfg < 0 else [0, 2, 3]
    for sp in splits:
        out.fill_(77.0)
        torch.cuda.synchronize()
        hip.setConvAutotune(True, cfg + CONV_SPLIT_UNIT * sp if cfg >= 0 else -1)
        try:
            hip.conv2dForward(B, C, H, W, F, kh, s, ph, dx, 3, dw.data_ptr() + 4, db, acLEAKY, out, 2,
                              inBatchStride=C * H * W + 5, outBatchStride=n + 7, residual=dr, resBatchStride=n,
                              weightLayout=layout, kernelWidth=kw, padWidth=pw)
        finally:
            hip.setConvAutotune(True, -1)
        hip.finish()
        got = out.cpu().numpy()
        assert (got[:2] == 77).all()
        for b in range(B):
            at = 2 + b * (n + 7)
            assert np.array_equal(got[at:at + n], ref[b].ravel()), (b, sp)
            assert (got[at + n:at + n + 7] == 77).all()


@pytest.mark.parametrize("cfg", GATHER)
def test_gather_infinite_input_and_weight_rows(hip, cfg):
    """An infinite input value reaches only its windows; a filter of infinite
    weights only its own output, though the row before it ends (K % 4 = 3)
    inside the same four floats."""
    print(f"[case] conv gather infinite cfg {cfg}", flush=True)
    B, C, H, W, F, k = 1, 3, 9, 9, 6, 3
    x, w = np.round(synth.normal(1210, (B, C, H, W), 2.0)), np.ones((F, C, k, k), np.float32)
    x = np.abs(x) + 1
    x[0, 1, 4, 4] = np.inf
    w[3] = np.inf
    with np.errstate(invalid="ignore"):
        ref = conv64(x, w, 1, 0, 0)
    dx, dw = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    out = torch.zeros(1, F, 7, 7, device="cuda")
    torch.cuda.synchronize()
    hip.setConvAutotune(True, cfg)
    try:
        hip.conv2dForward(B, C, H, W, F, k, 1, 0, dx, 0, dw, None, 4, out, 0)
    finally:
        hip.setConvAutotune(True, -1)
    hip.finish()
    assert np.isinf(ref[0, 3]).all() and np.isfinite(ref[0, 2]).any()
    assert np.array_equal(out.cpu().numpy(), ref.astype(np.float32))


@pytest.mark.parametrize("cfg", GATHER)
@pytest.mark.parametrize("B,C,H,W,F,k,s,splits", [(1, 65, 15, 15, 35, 5, 1, 16), (2, 32, 13, 10, 32, 5, 2, 8),
                                                  (1, 7, 13, 13, 16, 7, 1, 4)])
def test_gather_splits_of_a_few_panels(hip, cfg, B, C, H, W, F, k, s, splits):
    """The K splits that small layers are timed with: two to four panels of 32 each, a remainder in the last."""
    print(f"[case] conv gather splits cfg {cfg} C {C} k {k} splits {splits}", flush=True)
    x, w = np.round(synth.normal(1220, (B, C, H, W), 2.0)), np.round(synth.normal(1221, (F, C, k, k), 1.5))
    ref = conv64(x, w, s, k // 2, k // 2).astype(np.float32)
    dx, dw, out = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), torch.zeros(ref.shape, device="cuda")
    torch.cuda.synchronize()
    hip.setConvAutotune(True, cfg + CONV_SPLIT_UNIT * splits)
    try:
        hip.conv2dForward(B, C, H, W, F, k, s, k // 2, dx, 0, dw, None, 4, out, 0)
    finally:
        hip.setConvAutotune(True, -1)
    hip.finish()
    assert np.array_equal(out.cpu().numpy(), ref)
