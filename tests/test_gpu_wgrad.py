"""Weight gradients over geometries no panel fits (csrc/wgrad.hip): rows of
any length, strides, dilations, tiles with remainders, against float64."""
import numpy as np
import pytest
import torch

from tensorium_amd import synth

pytestmark = pytest.mark.gpu


def im2col(x, kh, kw, ph, pw, sy, sx, dy, dx):
    B, C, H, W = x.shape
    OH, OW = (H + 2 * ph - dy * (kh - 1) - 1) // sy + 1, (W + 2 * pw - dx * (kw - 1) - 1) // sx + 1
    xp = np.zeros((B, C, H + 2 * ph, W + 2 * pw), x.dtype)
    xp[:, :, ph:ph + H, pw:pw + W] = x
    col = np.empty((B, C, kh, kw, OH, OW), x.dtype)
    for i in range(kh):
        for j in range(kw):
            col[:, :, i, j] = xp[:, :, i * dy:i * dy + sy * (OH - 1) + 1:sy, j * dx:j * dx + sx * (OW - 1) + 1:sx]
    return col.reshape(B, C * kh * kw, OH * OW), OH, OW


@pytest.mark.parametrize("B,C,H,W,F,kh,kw,ph,pw,sy,sx,dy,dx", [
    (1, 1, 1, 1, 1, 1, 1, 0, 0, 1, 1, 1, 1),          # one pixel
    (3, 2, 5, 1, 3, 3, 1, 1, 0, 1, 1, 1, 1),          # rows of one pixel
    (2, 3, 6, 2, 4, 3, 3, 1, 1, 1, 1, 1, 1),          # two
    (2, 5, 7, 3, 66, 3, 3, 1, 1, 1, 1, 1, 1),         # three; filters past a tile
    (5, 4, 13, 13, 20, 3, 3, 1, 1, 1, 1, 1, 1),       # 13 = 3 quads and one
    (2, 16, 9, 20, 130, 3, 3, 1, 1, 1, 1, 1, 1),      # whole quads, a remainder in both tile axes
    (2, 6, 17, 15, 9, 5, 3, 2, 0, 2, 3, 1, 2),        # strides, dilation, no padding across
    (4, 70, 11, 14, 65, 1, 1, 0, 0, 2, 2, 1, 1),      # 1x1 with a stride
    (3, 70, 11, 13, 65, 1, 1, 0, 0, 1, 1, 1, 1),      # 1x1 over planes of 143
    (32, 8, 30, 30, 16, 3, 3, 1, 1, 1, 1, 1, 1),      # many panels: several splits
])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_wgrad_any_geometry(hip, B, C, H, W, F, kh, kw, ph, pw, sy, sx, dy, dx, beta):
    print(f"[case] wgrad B{B} C{C} {H}x{W} F{F} k{kh}x{kw} s{sy},{sx} d{dy},{dx}", flush=True)
    geom = (kh, kw, ph, pw, sy, sx, dy, dx)
    for integers in (True, False):
        x = synth.normal(1100, (B, C, H, W), 2.0)
        x = np.round(x) if integers else x
        col, OH, OW = im2col(x, *geom)
        L, K = OH * OW, C * kh * kw
        delta = synth.normal(1101, (B, F, L), 2.0)
        delta = np.round(delta) if integers else delta
        dw0 = np.round(synth.normal(1102, (F, K), 3.0))
        dW, dx_, dd = (torch.from_numpy(a).cuda() for a in (dw0, x, delta))
        torch.cuda.synchronize()
        hip.convWeightGradient(B, C, H, W, F, *geom, dx_, C * H * W, dd, F * L, 1.0, beta, dW)
        hip.finish()
        got = dW.cpu().numpy()
        d, c = delta.astype(np.float64), col.astype(np.float64)
        ref = beta * dw0 + np.matmul(d, c.transpose(0, 2, 1)).sum(0)
        if integers:  # every partial sum is a whole number below 2^24
            assert np.array_equal(got, ref.astype(np.float32))
        else:  # 24 bf16 instructions and one sum per 64 pixels, the splits' sums, alpha and beta
            mag = np.matmul(np.abs(d), np.abs(c).transpose(0, 2, 1)).sum(0) + np.abs(dw0)
            assert np.all(np.abs(got - ref) <= (24 + B * L / 64 + 64) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("L", [1, 3, 30, 57 * 75])
def test_nt_batch_reduce_any_length(hip, L):
    print(f"[case] nt batch reduce L {L}", flush=True)
    B, F, K = 3, 70, 90
    a, b = np.round(synth.normal(1110, (B, F, L), 2.0)), np.round(synth.normal(1111, (B, K, L), 2.0))
    dC = torch.zeros(F, K, device="cuda")
    da, db = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    torch.cuda.synchronize()
    hip.gemmNTBatchReduce(F, K, L, 0.5, da, 0, L, F * L, db, 0, L, K * L, 0.0, dC, 0, K, B)
    hip.finish()
    ref = 0.5 * np.matmul(a.astype(np.float64), b.astype(np.float64).transpose(0, 2, 1)).sum(0)
    assert np.array_equal(dC.cpu().numpy(), ref.astype(np.float32))


def test_infinite_input_outside_the_rows(hip):
    """The padding of a row's last quad reads nothing: an infinite input value
    reaches only the gradients of the windows that hold it."""
    print("[case] wgrad infinite input", flush=True)
    B, C, H, W, F = 2, 2, 6, 6, 5
    x, delta = np.round(synth.normal(1120, (B, C, H, W), 2.0)), np.ones((B, F, 25), np.float32)
    x[0, 1, 2, 5] = np.inf  # the sixth column: one past the output row's end for kx = 0
    dW = torch.zeros(F, C * 4, device="cuda")
    dx, dd = torch.from_numpy(x).cuda(), torch.from_numpy(delta).cuda()
    torch.cuda.synchronize()
    hip.convWeightGradient(B, C, H, W, F, 2, 2, 0, 0, 1, 1, 1, 1, dx, C * H * W, dd, F * 25, 1.0, 0.0, dW)
    hip.finish()
    col, _, _ = im2col(x, 2, 2, 0, 0, 1, 1, 1, 1)
    ref = np.matmul(delta.astype(np.float64), col.astype(np.float64).transpose(0, 2, 1)).sum(0)
    assert np.isinf(ref).any() and np.isfinite(ref).any()
    assert np.array_equal(dW.cpu().numpy(), ref.astype(np.float32))


@pytest.mark.parametrize("B,C,H,F", [(8, 32, 16, 64), (8, 64, 8, 128), (32, 64, 8, 128), (128, 32, 16, 64), (128, 64, 8, 128)])
def test_short_axes_fill_the_gpu(hip, B, C, H, F):
    """A quarter of the workgroups that 64x64 tiles of two panels of 32 pixels
    would give, or one a CU: neither large tiles nor long splits leave the GPU
    idle."""
    print(f"[case] wgrad pieces B{B} C{C} {H}x{H} F{F}", flush=True)
    K, panels = C * 9, B * H * H // 32
    x, d = torch.zeros(B, C, H, H, device="cuda"), torch.zeros(B, F, H, H, device="cuda")
    n = hip.convWeightGradientPieces(B, C, H, H, F, 3, 3, 1, 1, 1, 1, 1, 1, x, C * H * H, d, F * H * H)
    tiles = -(-F // 64) * -(-K // 64)
    assert n * tiles >= min(tiles * panels // 8, 256)


def test_few_weights_on_a_short_axis_are_one_piece(hip):
    """Fewer than 8192 weights: one piece up to 15 panels of 32 pixels, refused above."""
    print("[case] wgrad pieces few weights", flush=True)
    C, H, F = 3, 8, 32
    for B in (1, 4, 7):
        x, d = torch.ones(B, C, H, H, device="cuda"), torch.ones(B, F, H, H, device="cuda")
        pieces = torch.zeros(F * C * 9, device="cuda")
        torch.cuda.synchronize()
        assert hip.convWeightGradientPieces(B, C, H, H, F, 3, 3, 1, 1, 1, 1, 1, 1, x, C * H * H, d, F * H * H, pieces,
                                            F * C * 9) == 1
        hip.finish()
        col, _, _ = im2col(np.ones((B, C, H, H), np.float32), 3, 3, 1, 1, 1, 1, 1, 1)
        assert np.array_equal(pieces.cpu().numpy().reshape(F, C * 9), np.tile(col.sum((0, 2)), (F, 1)))
    x, d = torch.ones(8, C, H, H, device="cuda"), torch.ones(8, F, H, H, device="cuda")
    with pytest.raises(Exception, match="sum their pieces a wave each"):
        hip.convWeightGradientPieces(8, C, H, H, F, 3, 3, 1, 1, 1, 1, 1, 1, x, C * H * H, d, F * H * H)
