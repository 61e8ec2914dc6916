"""The comparison of yolo outputs at the jumps of the reference's logistic (yolo_check.py)."""
import os

import numpy as np
import pytest
import yolo_check
from oracle import netref, refcpu as R
from tensorium_amd import darknet, synth

TOL = 1e-5
N, CLASSES = 3, 4


@pytest.mark.parametrize("k,jump", [(0, 8.62e-4), (1, 7.66e-4), (-1, 7.66e-4), (2, 5.52e-4)])
def test_logits_beside_a_jump(k, jump):
    conv = synth.normal(1, (2, N * (CLASSES + 5), 5, 6), 2.0)
    at = (1, CLASSES + 5 + 4, 2, 3)  # the second anchor's objectness
    x = np.float32(k * np.log(2))
    conv[at] = x - np.float32(1e-6)
    out = yolo_check.transform(conv, N, CLASSES)
    other = conv.copy()
    other[at] = x + np.float32(1e-6)
    got = yolo_check.transform(other, N, CLASSES)
    assert abs(np.abs(got - out).max() - jump) < 5e-6
    assert R.rel_err(got, out) > 5 * TOL  # what a plain comparison sees
    assert yolo_check.yolo_err(got, out, conv, N, CLASSES, TOL) <= TOL
    for wrong in ((1, CLASSES + 5 + 4, 2, 4), (0, 2, 1, 1), (1, 0, 0, 0)):  # elsewhere the same error is refused
        bad = got.copy()
        bad[wrong] += np.float32(jump)
        assert yolo_check.yolo_err(bad, out, conv, N, CLASSES, TOL) > TOL
    bad = got.copy()
    bad[at] += np.float32(jump)  # and another value at the jump
    assert yolo_check.yolo_err(bad, out, conv, N, CLASSES, TOL) > TOL


def test_yolov3_tiny_has_a_logit_beside_a_jump():
    """YOLOv3-tiny at 256x256 on the input of the scale_x_y parity test: a
    second-head logit of image 0 is 2e-6 from zero, under the rounding of the
    layers before it, so the output there is one of two values 1.65e-4 of the
    largest apart."""
    with open(os.path.join(darknet.CFG_DIR, "yolov3-tiny.cfg")) as f:
        text = f.read().replace("[yolo]", "[yolo]\nscale_x_y=1.05")
    _, layers = darknet.parse_cfg(text, 256, 256)
    W = darknet.synthetic_weights(layers)
    ref = netref.forward(layers, W, synth.uniform(6, (2, 3, 256, 256))[:1])
    conv, out = ref[22], ref[23]
    logits = conv.reshape(3, 85, -1).copy()
    logits[:, 2:4] = 1  # box sizes, which stay raw
    at = np.unravel_index(np.abs(logits).argmin(), logits.shape)
    assert 0 < logits[at] < 1e-5 * np.abs(conv).max()
    other = conv.copy()
    other.reshape(logits.shape)[at] *= -1
    got = yolo_check.transform(other, 3, 80, 1.05)
    assert 1.6e-4 < R.rel_err(got, out) < 1.8e-4
    assert yolo_check.yolo_err(got, out, conv, 3, 80, TOL, 1.05) <= TOL
