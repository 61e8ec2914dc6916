"""Comparison of yolo outputs across the jumps of the reference's logistic.

logistic_array (nactivation.pas:36-127) forms exp(-x) as 2^i p(f), t = -x log2(e)
= i + f, with a polynomial whose ends do not meet: p(0) = 1.00172, p(1)/2 =
0.99828.  Its output jumps wherever t passes a whole number, at x = 0 by 8.62e-4
and at x = k ln 2 by somewhat less.  A logit within rounding of such a point
falls on either side, whichever sums it came from, so there (and only there)
both sides are right."""
import numpy as np

from oracle import refcpu as R

LOG2E = 1.4426950408889634


def transform(conv, n, classes, scale_xy=1.0):
    """The oracle's yolo layer over a head convolution's output [B][n*(5+classes)][h][w]."""
    y = R.yolo_fwd(np.ascontiguousarray(conv, np.float32), n, classes, exact=True)
    s = np.float32(scale_xy)
    if s != 1:
        v = y.reshape(conv.shape[0], n, classes + 5, -1)
        v[:, :, :2] = (v[:, :, :2] * s).astype(np.float32) + np.float32(0.5) * (np.float32(1) - s)
    return y


def yolo_err(got, out, conv, n, classes, tol, scale_xy=1.0):
    """max |got - out| / max |out|, as the per-tensor bound has it, where out
    is the yolo output of the logits conv; at logits that a change within the
    bound (tol of the largest) takes over a jump, against the nearest of the
    outputs there."""
    d = np.float32(tol) * np.abs(conv).max()
    near = np.floor(-(conv - d).astype(np.float64) * LOG2E) != np.floor(-(conv + d).astype(np.float64) * LOG2E)
    got, out = np.asarray(got, np.float64), np.asarray(out, np.float64)
    diff = np.abs(got - out).reshape(conv.shape)
    if near.any():
        for shifted in (conv - d, conv + d):
            other = np.abs(got - transform(shifted, n, classes, scale_xy)).reshape(conv.shape)
            diff = np.where(near, np.minimum(diff, other), diff)
    return float(diff.max() / np.abs(out).max())
