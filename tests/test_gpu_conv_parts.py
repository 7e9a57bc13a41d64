"""Convolutions whose K is split: the last block to finish adds the parts four at a time and the rest one by
one, for part counts around multiples of four, ragged tiles and the K pieces of the last tiles; against float64
and, as the order of the sum is fixed, bit for bit on a second run."""
import numpy as np
import pytest

import oracle as O
from conftest import empty_dev, to_dev

pytestmark = pytest.mark.gpu

# few tiles and K = 9 Cin: up to one part per 128 taps, 16 at most
SHAPES = [(1, c, 7, 7, 64, 3, 1, 1) for c in (29, 43, 57, 72, 86, 100, 114, 128, 143, 230)] + [
    (1, 129, 9, 11, 70, 3, 1, 1),      # tiles ragged both ways
    (3, 46, 61, 53, 75, 5, 2, 2),
    (33, 64, 28, 28, 96, 3, 1, 1),     # whole tiles and K pieces of the last ones
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_parts(hip, shape):
    print(f"case {shape}", flush=True)
    N, Cin, H, W, Cout, k, stride, pad = shape
    x, w = O.randn((N, Cin, H, W), 21), O.randn((Cout, Cin, k, k), 22, 0.1)
    res_shape = (N, Cout, (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1)
    res, bias = O.randn(res_shape, 23), O.randn((Cout,), 24)
    one, zero = np.ones(Cout, np.float32), np.zeros(Cout, np.float32)
    d = lambda a: to_dev(hip, a)
    dx, dw = d(x), d(w)
    got = []
    for _ in range(2):
        dy = empty_dev(hip, res_shape)
        hip.HIPBackend.conv2dBiasBnAddAct(dx, dw, d(bias), d(one), d(zero), d(zero), d(one), 0.0, d(res), 0, dy, N, Cin, H,
                                          W, Cout, k, k, stride, pad)
        got.append(dy.numpy())
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    y, bound = O.conv_f64(x, w, bias, stride, pad)
    K = Cin * k * k
    # K products and sums (bias among them), the residual's addition
    assert np.all(np.abs(got[0] - (y + res)) <= 2.0 ** -24 * ((K + 3) * np.abs(bound) + np.abs(y) + np.abs(res)))
