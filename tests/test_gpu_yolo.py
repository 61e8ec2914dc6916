"""YOLOv3-416 end to end on the GPU against the CPU oracle: the three
pre-logistic head convolutions (darknet layers 81, 93, 105) within the
per-tensor 1e-5 bound, every intermediate convolution too, and the yolo
outputs.  Batch 2 checks that per-image results do not depend on the batch
(per-image route concat).  The benchmark configurations at their full sizes
(416 at batch 16, 608 at batch 32, channels-last, tuned for those shapes)
are tied to the oracle-checked batch-1 network image by image."""
import numpy as np
import pytest
import torch

from oracle import netref
from oracle import refcpu as R
from tensorium_amd import darknet, synth
from tensorium_amd.nnhip import DeviceArray, acLEAKY
from yolo_check import yolo_err

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module")
def yolo():
    net, layers = darknet.load_cfg("yolov3.cfg")
    return layers, darknet.synthetic_weights(layers)


def run_gpu(hip, layers, weights, x, fuse=True):
    n = darknet.Network(hip, layers, x.shape[0], weights, fuse=fuse)
    dx = DeviceArray.from_numpy(x)  # the library's own memory (any device buffer is taken)
    heads = n.forward(dx)
    hip.finish()
    return n, [h.numpy() for h in heads]


def test_yolov3_416_layerwise(hip, yolo):
    """Every conv layer of YOLOv3-416 fed the oracle's own input for that
    layer: per-layer output within the 1e-5 per-tensor bound."""
    layers, W = yolo
    print("[case] yolov3-416 batch 1 layer-wise vs oracle", flush=True)
    x = synth.uniform(7, (1, 3, 416, 416))
    ref = netref.forward(layers, W, x)
    n = darknet.Network(hip, layers, 1, W, fuse=False)
    worst = 0.0
    for L in layers:
        if L["type"] != "convolutional":
            continue
        i = L["index"]
        src = torch.from_numpy(ref[i - 1] if i > 0 else x).cuda()
        torch.cuda.synchronize()
        w, b, layout = n.w[i]
        C, h, ww = L["in"]
        out = torch.empty((1,) + L["out"], dtype=torch.float32, device="cuda")
        hip.conv2dForward(1, C, h, ww, L["filters"], L["size"], L["stride"], L["pad"], src, 0, w, b, L["act"], out,
                          0, weightLayout=layout)
        hip.finish()
        e = R.rel_err(out.cpu().numpy(), ref[i])
        worst = max(worst, e)
        assert e <= TOL, (i, e)
    print(f"worst per-layer conv error {worst:.3e}", flush=True)


def test_yolov3_416_batch1_heads(hip, yolo):
    """End to end: the three pre-logistic head convolutions (the parity
    checkpoint) within 1e-5 of the oracle; intermediate layers accumulate
    fp32 ordering differences over ~100 layers and are reported."""
    layers, W = yolo
    print("[case] yolov3-416 batch 1 end-to-end vs oracle", flush=True)
    x = synth.uniform(7, (1, 3, 416, 416))
    ref = netref.forward(layers, W, x)
    n, heads = run_gpu(hip, layers, W, x)
    errs = {}
    for L in layers:
        i = L["index"]
        if L["type"] == "convolutional" and i not in n.fused:
            errs[i] = R.rel_err(n.out[i].numpy(), ref[i])
    worst = max(errs, key=errs.get)
    print(f"worst intermediate conv error {errs[worst]:.3e} at layer {worst}", flush=True)
    for i in (81, 93, 105):
        print(f"head conv {i}: {errs[i]:.3e}", flush=True)
        assert errs[i] <= TOL, (i, errs[i])
    assert max(errs.values()) <= 5 * TOL
    for h, i in zip(heads, (82, 94, 106)):
        # The head convs reach |x| ~ 1e5 with random weights, so a 1e-6
        # relative difference moves logistic(x) near 0 by O(1): the parity
        # checkpoint is the pre-logistic conv above.  The yolo kernel itself
        # must be bit-exact on the GPU's own head-conv output.
        own = R.yolo_fwd(n.out[i - 1].numpy(), 3, 80, exact=True)
        assert np.array_equal(h, own)


def test_yolov3_fusion_is_exact(hip, yolo):
    """Shortcut fused into the conv epilogue == separate addvv, bit for bit,
    when both networks run the same tilings: with autotuning off the cost
    model picks each layer's tiling from its GEMM shape alone (the tuner
    times a convolution with and without a residual separately, so its
    choices, and the summation order, may differ between the two)."""
    layers, W = yolo
    print("[case] yolov3 fused vs unfused", flush=True)
    x = synth.uniform(8, (1, 3, 416, 416))
    hip.setConvAutotune(False, -1)
    try:
        _, a = run_gpu(hip, layers, W, x, fuse=True)
        _, b = run_gpu(hip, layers, W, x, fuse=False)
    finally:
        hip.setConvAutotune(True, -1)
    for u, v in zip(a, b):
        assert np.array_equal(u, v)


def test_yolov3_batch_independent(hip, yolo):
    layers, W = yolo
    print("[case] yolov3 batch 2 == two batch-1 runs", flush=True)
    x = synth.uniform(9, (2, 3, 416, 416))
    _, h2 = run_gpu(hip, layers, W, x)
    for b in range(2):
        _, h1 = run_gpu(hip, layers, W, x[b:b + 1].copy())
        for u, v in zip(h2, h1):
            assert R.rel_err(u[b:b + 1], v) <= TOL


def test_yolov3_graph_replay(hip, yolo):
    """The forward captured into a HIP graph and replayed several times, with
    eager work and synchronisations between replays: every replay equals the
    eager result bit for bit (same tuned kernels)."""
    layers, W = yolo
    print("[case] yolov3 HIP graph replay", flush=True)
    x = synth.uniform(10, (2, 3, 416, 416))
    n = darknet.Network(hip, layers, 2, W)
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    eager = [h.numpy() for h in n.forward(dx)]
    hip.finish()
    try:
        n.capture(dx)
        scratch = torch.zeros(n.out[0].shape, device="cuda")
        for rep in range(3):
            heads = n.replay()
            hip.finish()
            got = [h.numpy() for h in heads]
            for u, v in zip(got, eager):
                assert np.array_equal(u, v), rep
            # eager work between replays, on both streams
            hip.fill(scratch.numel(), scratch, 0, float(rep), 1)
            hip.finish()
            scratch.add_(1.0)
            torch.cuda.synchronize()
    finally:
        n.release_graph()
        hip.useTorchStream()


def test_yolov3_nhwc_heads(hip, yolo):
    """The channels-last network at batch 1 end to end (the benchmark's
    batch-1 configuration, tuned for its shapes: wave-split tiles on the
    small layers): the three pre-logistic head convolutions within 1e-5 of
    the oracle, every other unfused convolution within 5e-5, the yolo kernel
    bit-exact on the device's own head-conv output (written NCHW), and two
    graph replays equal to the eager forward bit for bit."""
    layers, W = yolo
    print("[case] yolov3-416 batch 1 channels-last end-to-end vs oracle", flush=True)
    x = synth.uniform(7, (1, 3, 416, 416))
    ref = netref.forward(layers, W, x)
    n = darknet.Network(hip, layers, 1, W, layout="nhwc")
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    heads = [h.numpy() for h in n.forward(dx)]
    hip.finish()
    errs = {}
    assert n.up_fused == {84, 96} and n.yolo_fused == {81, 93, 105}
    for L in layers:
        i = L["index"]
        if L["type"] == "convolutional" and i not in n.fused and i not in n.up_fused:
            errs[i] = R.rel_err(n.output(i), ref[i])
        if L["type"] == "upsample":  # written by the convolution before it
            errs[i] = R.rel_err(n.output(i), ref[i])
    worst = max(errs, key=errs.get)
    print(f"worst intermediate conv error {errs[worst]:.3e} at layer {worst}", flush=True)
    for i in (81, 93, 105):
        assert errs[i] <= TOL, (i, errs[i])
    assert max(errs.values()) <= 5 * TOL
    for h, i in zip(heads, (82, 94, 106)):
        own = R.yolo_fwd(n.output(i - 1), 3, 80, exact=True)
        assert np.array_equal(h, own)
    try:
        n.capture(dx)
        for rep in range(2):
            got = n.replay()
            hip.finish()
            for u, v in zip([g.numpy() for g in got], heads):
                assert np.array_equal(u, v), rep
            torch.cuda.synchronize()
    finally:
        n.release_graph()
        hip.useTorchStream()


@pytest.mark.parametrize("B", [1, 4])
def test_yolov3_nhwc_fusion_is_exact(hip, yolo, B):
    """Channels-last head fusions (the upsample written by the conv before
    it, the yolo head written by the head conv) against the network that
    launches them separately, bit for bit, when both run the same tilings
    (autotuning off: the cost model picks each tiling from the GEMM shape
    alone)."""
    layers, W = yolo
    print(f"[case] yolov3 batch {B} nhwc fused vs unfused", flush=True)
    x = synth.uniform(19, (B, 3, 416, 416))
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    hip.setConvAutotune(False, -1)
    try:
        a = darknet.Network(hip, layers, B, W, layout="nhwc")
        ha = [h.numpy() for h in a.forward(dx)]
        hip.finish()
        b = darknet.Network(hip, layers, B, W, layout="nhwc", fuse_heads=False)
        hb = [h.numpy() for h in b.forward(dx)]
        hip.finish()
    finally:
        hip.setConvAutotune(True, -1)
    assert a.up_fused and a.yolo_fused and not b.up_fused and not b.yolo_fused
    for u, v in zip(ha, hb):
        assert np.array_equal(u, v)
    for i in (85, 97, 81, 93, 105):
        assert np.array_equal(a.output(i), b.output(i)), i


@pytest.mark.parametrize("B", [1, 4])
def test_yolov3_nhwc_branches(hip, yolo, B):
    """The yolo head tails (layers 80-82 and 92-94) forked onto a second
    stream: the planner finds exactly those two tails, and the branched
    eager forward and two replays of its graph equal the single-stream
    forward bit for bit (the same tuned kernels run; only the stream and
    the split-K scratch differ)."""
    layers, W = yolo
    print(f"[case] yolov3-416 batch {B} nhwc head tails on a second stream", flush=True)
    x = synth.uniform(17, (B, 3, 416, 416))
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    n = darknet.Network(hip, layers, B, W, layout="nhwc")
    assert n.branches == {80: 82, 92: 94}
    single = [h.numpy() for h in n.forward(dx, branches=False)]
    hip.finish()
    got = [h.numpy() for h in n.forward(dx, branches=True)]
    hip.finish()
    for u, v in zip(got, single):
        assert np.array_equal(u, v)
    n.use_branches = True
    try:
        n.capture(dx)
        for rep in range(2):
            heads = n.replay()
            hip.finish()
            for u, v in zip([h.numpy() for h in heads], single):
                assert np.array_equal(u, v), rep
            torch.cuda.synchronize()
    finally:
        n.release_graph()
        hip.useTorchStream()


def test_yolov3_nhwc_matches_nchw_and_replays(hip, yolo):
    """Batch 2: the channels-last network's head convolutions equal the NCHW
    network's within the per-tensor bound, the route inputs written in place
    equal a concat, and graph replays of the channels-last forward equal its
    eager result bit for bit."""
    layers, W = yolo
    print("[case] yolov3 batch 2 nhwc vs nchw, graph replay", flush=True)
    x = synth.uniform(11, (2, 3, 416, 416))
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    a = darknet.Network(hip, layers, 2, W)
    a.forward(dx)
    hip.finish()
    b = darknet.Network(hip, layers, 2, W, layout="nhwc")
    eager = [h.numpy() for h in b.forward(dx)]
    hip.finish()
    for i in (81, 93, 105, 86, 98):  # head convs and the two multi-input routes
        assert R.rel_err(b.output(i), a.output(i)) <= 2 * TOL, i
    try:
        b.capture(dx)
        for rep in range(3):
            heads = b.replay()
            hip.finish()
            for u, v in zip([h.numpy() for h in heads], eager):
                assert np.array_equal(u, v), rep
            torch.cuda.synchronize()
    finally:
        b.release_graph()
        hip.useTorchStream()


def test_yolov3_416_b16_bench_config(hip, yolo):
    """The benchmark's own configuration: YOLOv3-416 at batch 16,
    channels-last, autotuned for batch-16 shapes (tail splits included).
    Images 0, 7 and 15 of the batch against the CPU oracle run on the same
    image and against the float64 evaluation of the network: the three
    pre-logistic head convolutions within 1e-5 of the oracle (the north
    star's bound) and of float64.  Two graph replays of the batch-16 forward
    equal its eager result bit for bit."""
    layers, W = yolo
    print("[case] yolov3-416 batch 16 nhwc (bench configuration) vs the oracle, graph replay", flush=True)
    x = synth.uniform(13, (16, 3, 416, 416))
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    big = darknet.Network(hip, layers, 16, W, layout="nhwc")
    eager = [h.numpy() for h in big.forward(dx)]
    hip.finish()
    heads16 = {i: big.output(i) for i in (81, 93, 105)}
    for img in (0, 7, 15):
        print(f"[case] oracle and float64 forwards of image {img}", flush=True)
        xi = np.ascontiguousarray(x[img:img + 1])
        ref = netref.forward(layers, W, xi)
        r64 = f64_heads(layers, W, xi)
        for i in (81, 93, 105):
            e = R.rel_err(heads16[i][img:img + 1], ref[i])
            e64 = R.rel_err(heads16[i][img:img + 1], r64[i])
            print(f"image {img} head conv {i}: vs oracle {e:.3e}, vs float64 {e64:.3e} "
                  f"(oracle vs float64 {R.rel_err(ref[i], r64[i]):.3e})", flush=True)
            assert e64 <= TOL, (img, i, e64)
            assert e <= TOL, (img, i, e)
        del ref
    try:
        big.capture(dx)
        for rep in range(2):
            heads = big.replay()
            hip.finish()
            for u, v in zip([h.numpy() for h in heads], eager):
                assert np.array_equal(u, v), rep
            torch.cuda.synchronize()
    finally:
        big.release_graph()
        hip.useTorchStream()


def f64_heads(layers, W, x, heads=(81, 93, 105)):
    """The network evaluated in float64 with torch on the CPU (conv2d,
    leaky 0.1, shortcut add, channel concat, nearest upsample): the head
    convolutions of an fp32 chain free of rounding, as a library-routine
    reference."""
    import torch.nn.functional as Fn

    outs, prev = [], torch.from_numpy(x).double()
    for L in layers:
        t = L["type"]
        if t == "convolutional":
            w, b = W[L["index"]]
            F, k, C = L["filters"], L["size"], L["in"][0]
            y = Fn.conv2d(prev, torch.from_numpy(w).double().reshape(F, C, k, k), torch.from_numpy(b).double(),
                          stride=L["stride"], padding=L["pad"])
            if L["act"] == acLEAKY:
                y = torch.where(y < 0, 0.1 * y, y)
        elif t == "shortcut":
            y = prev + outs[L["src"]]
        elif t == "route":
            y = torch.cat([outs[s_] for s_ in L["srcs"]], 1)
        elif t == "upsample":
            y = prev.repeat_interleave(L["stride"], 2).repeat_interleave(L["stride"], 3)
        else:
            y = prev
        outs.append(y)
        prev = y
    return {i: outs[i].numpy() for i in heads}


def test_yolov3_608_b32_bench_config(hip):
    """BASELINE config 5 at its size: YOLOv3-608 at batch 32, channels-last
    and autotuned for those shapes; images 0 and 31 against the CPU oracle
    run on the same image and against the float64 evaluation of the same
    network: the heads within 1e-5 of the oracle (the north star's bound)
    and of float64."""
    _, layers = darknet.load_cfg("yolov3.cfg", 608, 608)
    W = darknet.synthetic_weights(layers)
    print("[case] yolov3-608 batch 32 nhwc vs the oracle", flush=True)
    x = synth.uniform(17, (32, 3, 608, 608))
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    big = darknet.Network(hip, layers, 32, W, layout="nhwc")
    big.forward(dx)
    hip.finish()
    heads32 = {i: big.output(i) for i in (81, 93, 105)}
    del big
    for img in (0, 31):
        print(f"[case] oracle and float64 forwards of image {img} at 608", flush=True)
        xi = np.ascontiguousarray(x[img:img + 1])
        ref = netref.forward(layers, W, xi)
        r64 = f64_heads(layers, W, xi)
        for i in (81, 93, 105):
            e = R.rel_err(heads32[i][img:img + 1], ref[i])
            e64 = R.rel_err(heads32[i][img:img + 1], r64[i])
            o64 = R.rel_err(ref[i], r64[i])
            print(f"image {img} head conv {i}: vs oracle {e:.3e}, vs float64 {e64:.3e} "
                  f"(oracle vs float64 {o64:.3e})", flush=True)
            assert e64 <= TOL, (img, i, e64)
            assert e <= TOL, (img, i, e)
        del ref


@pytest.mark.parametrize("B", [2, 16])
def test_yolov3_reference_route_mode(hip, yolo, B):
    """The reference's whole-tensor route concat (nconcatlayer.pas:115 ->
    ntensors.pas:12045: every input's whole batched tensor copied back to
    back, which mixes images at batch > 1), NCHW network at batch 2 and 16,
    against the oracle run in the same mode on the whole batch: the three
    head convolutions within 1e-5, and at least one head differs from the
    per-image (darknet) concat by more than that bound."""
    layers, W = yolo
    print(f"[case] yolov3-416 batch {B} route_mode=reference vs the oracle", flush=True)
    x = synth.uniform(19 + B, (B, 3, 416, 416))
    dx = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    n = darknet.Network(hip, layers, B, W, route_mode="reference")
    n.forward(dx)
    hip.finish()
    got = {i: n.output(i) for i in (81, 93, 105)}
    del n
    ref = netref.forward(layers, W, x, route_mode="reference")
    for i in (81, 93, 105):
        e = R.rel_err(got[i], ref[i])
        print(f"batch {B} head conv {i}: {e:.3e}", flush=True)
        assert e <= TOL, (i, e)
    per_image = darknet.Network(hip, layers, B, W)
    per_image.forward(dx)
    hip.finish()
    assert max(R.rel_err(per_image.output(i), got[i]) for i in (93, 105)) > 10 * TOL


def test_nhwc_rejects_reference_route_mode(hip, yolo):
    layers, W = yolo
    with pytest.raises(NotImplementedError):
        darknet.Network(hip, layers, 2, W, layout="nhwc", route_mode="reference")


@pytest.mark.parametrize("layout", ["nchw", "nhwc"])
def test_yolov3_batch_in_passes(hip, layout):
    """A batch run as several passes over one-pass buffers (max_pass_batch=2:
    images 0-1, 2-3, then 4 alone) gives the heads of the single-pass network
    within the per-tensor bound, eagerly and in a graph replay; intermediate
    outputs are refused (only the last pass is held)."""
    print(f"[case] yolov3-128 batch 5 in passes of 2, {layout}", flush=True)
    _, layers = darknet.load_cfg("yolov3.cfg", 128, 128)
    W = darknet.synthetic_weights(layers)
    dx = torch.from_numpy(synth.uniform(11, (5, 3, 128, 128))).cuda()
    torch.cuda.synchronize()
    one = darknet.Network(hip, layers, 5, W, layout=layout)
    ref = [h.numpy() for h in one.forward(dx)]
    hip.finish()
    convs = [one.output(i) for i in (81, 93, 105)]
    net = darknet.Network(hip, layers, 5, W, layout=layout, max_pass_batch=2)
    assert (net.pass_batch, net.batch) == (2, 5)
    heads = net.forward(dx)
    hip.finish()
    for h, r, c in zip(heads, ref, convs):
        assert h.shape == r.shape
        assert yolo_err(h.numpy(), r, c, 3, 80, TOL) <= TOL
    heads = net.capture(dx)
    for _ in range(2):
        for h in heads:
            hip.fill(h.numel(), h, 0, 0.0, 1)
        hip.finish()
        net.replay()
        hip.finish()
        for h, r, c in zip(heads, ref, convs):
            assert yolo_err(h.numpy(), r, c, 3, 80, TOL) <= TOL
    net.release_graph()
    with pytest.raises(ValueError, match="passes"):
        net.output(3)


@pytest.mark.parametrize("layout", ["nchw", "nhwc"])
def test_yolov3_tiny_vs_oracle(hip, layout):
    """YOLOv3-tiny (maxpools, a stride-1 maxpool, a 16-channel convolution
    input, a route over a maxpool's input) end to end at batch 2 against the
    oracle run per image: the two pre-logistic head convolutions (15, 22)
    within the per-tensor bound, the yolo outputs within it too."""
    print(f"[case] yolov3-tiny-416 batch 2 {layout} vs oracle", flush=True)
    _, layers = darknet.load_cfg("yolov3-tiny.cfg")
    W = darknet.synthetic_weights(layers)
    x = synth.uniform(5, (2, 3, 416, 416))
    net = darknet.Network(hip, layers, 2, W, layout=layout)
    heads = net.forward(torch.from_numpy(x).cuda())
    hip.finish()
    for b in range(2):
        ref = netref.forward(layers, W, x[b:b + 1])
        for i in (15, 22):
            got = net.output(i)[b:b + 1]
            e = R.rel_err(got, ref[i])
            print(f"image {b} head conv {i}: {e:.3e}", flush=True)
            assert e <= TOL, (b, i, e)
        for h, i in zip(heads, (16, 23)):
            assert yolo_err(h[b:b + 1].numpy(), ref[i], ref[i - 1], 3, 80, TOL) <= TOL


@pytest.mark.parametrize("layout", ["nchw", "nhwc"])
def test_yolov3_tiny_scale_xy_vs_oracle(hip, layout):
    """YOLOv3-tiny with scale_x_y = 1.05 on both yolo layers (the value
    YOLOv4 cfgs use): the yolo outputs at batch 2 against the oracle run per
    image, within the per-tensor bound; the fused conv + yolo head path
    (channels-last) and the plain yolo kernel (NCHW) both take the step."""
    print(f"[case] yolov3-tiny-256 scale_x_y=1.05 batch 2 {layout} vs oracle", flush=True)
    import os
    with open(os.path.join(darknet.CFG_DIR, "yolov3-tiny.cfg")) as f:
        text = f.read().replace("[yolo]", "[yolo]\nscale_x_y=1.05")
    _, layers = darknet.parse_cfg(text, 256, 256)
    W = darknet.synthetic_weights(layers)
    x = synth.uniform(6, (2, 3, 256, 256))
    net = darknet.Network(hip, layers, 2, W, layout=layout)
    heads = net.forward(torch.from_numpy(x).cuda())
    hip.finish()
    for b in range(2):
        ref = netref.forward(layers, W, x[b:b + 1])
        for h, i in zip(heads, (16, 23)):
            e = yolo_err(h[b:b + 1].numpy(), ref[i], ref[i - 1], 3, 80, TOL, 1.05)
            print(f"image {b} yolo {i}: {e:.3e}", flush=True)
            assert e <= TOL, (b, i, e)


DEPTH_CFG = """[net]
width=64
height=64
channels=3

[convolutional]
batch_normalize=1
filters=32
size=3
stride=1
pad=1
activation=leaky

[maxpool]
maxpool_depth=1
out_channels=8

[convolutional]
filters=18
size=1
stride=1
pad=1
activation=linear

[yolo]
mask=0,1,2
anchors=10,13, 16,30, 33,23
classes=1
"""


def test_maxpool_depth_network_vs_oracle(hip):
    """A network with a maxpool_depth layer (32 channels -> 8 groups of 4):
    the NCHW network's yolo output against the oracle within the per-tensor
    bound, and the depth layer's output bit for bit; the channels-last planner
    refuses it."""
    print("[case] maxpool_depth network 64x64 batch 2", flush=True)
    _, layers = darknet.parse_cfg(DEPTH_CFG)
    assert layers[1]["out"] == (8, 64, 64)
    W = darknet.synthetic_weights(layers)
    x = synth.uniform(8, (2, 3, 64, 64))
    net = darknet.Network(hip, layers, 2, W, layout="nchw")
    heads = net.forward(torch.from_numpy(x).cuda())
    hip.finish()
    ref = netref.forward(layers, W, x)
    assert np.array_equal(net.output(1), R.maxpool_depth_fwd(net.output(0), 8)[0])
    assert yolo_err(heads[0].numpy(), ref[3], ref[2], 3, 1, TOL) <= TOL
    with pytest.raises(NotImplementedError, match="maxpool_depth"):
        darknet.Network(hip, layers, 2, W, layout="nhwc")
