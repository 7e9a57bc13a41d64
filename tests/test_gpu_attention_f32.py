"""fp32 attention: the fused kernel at the edges of its tiles (16 queries a wave, 64 a workgroup, 64 keys a
trip, head dimensions padded to 16), the sizes beside it that take the composed path, and scores that are
infinite or NaN, against float64.

Bound, per context element, in units of sum_j P_ij |V_jd| (u = 2^-24): the weight of a key carries its score's
error, at most (D + 3) u sum_d |scale q k| over scores of the two keys compared, plus 4 u of exp and its scale;
the sums over S keys of the numerator and of the weights add (S + 2) u each, the division 2 u.
"""
import numpy as np
import pytest

import oracle as O
from conftest import empty_dev, to_dev
from test_gpu_streams import streams  # noqa: F401  (fixture: caller-owned streams)

pytestmark = pytest.mark.gpu

# S: one key, around 16 and 64, several trips; D: each padded width, the largest, the composed path (10, 132)
SHAPES = [(2, s, 2, 64) for s in (1, 15, 16, 17, 63, 64, 65, 129, 300)] + \
         [(1, s, 3, d) for d in (4, 12, 16, 20, 32, 48, 80, 96, 100, 128, 10, 132) for s in (17, 70)] + \
         [(1, 384, 3, 64), (1, 449, 3, 64), (3, 500, 1, 64), (1, 512, 12, 64), (1, 700, 2, 32), (2, 577, 3, 80),
          (1, 1000, 12, 20), (2, 1030, 1, 64), (4, 520, 9, 128)]   # both sides of the line between the two paths


def _run(hip, qkv, B, S, H, D, scale, shift=0):
    """shift: floats by which input and output lie off the allocation's start."""
    dq = to_dev(hip, np.concatenate([np.zeros(shift, np.float32), qkv.reshape(-1)]))
    dout = empty_dev(hip, (B * S * H * D + shift,))
    hip.HIPBackend.attention(dq.ptr + 4 * shift, dout.ptr + 4 * shift, B, S, H, D, scale)
    return dout.numpy()[shift:].reshape(B * S, H * D)


def _tolerance(qkv, B, S, H, D, scale):
    q, k = (np.abs(qkv.reshape(B, S, 3, H, D)[:, :, i].astype(np.float64)) for i in (0, 1))
    worst = abs(scale) * np.einsum("bshd,bthd->bhst", q, k).max()
    return 2.0 ** -24 * (2 * (D + 3) * worst + 8 + 2 * (S + 2) + 2)


@pytest.mark.parametrize("B,S,H,D", SHAPES, ids=lambda v: str(v))
def test_edges(hip, B, S, H, D):
    print(f"case {B}x{S}x{H}x{D}", flush=True)
    qkv = O.randn((B * S, 3 * H * D), 31 * S + D, 1.0)
    scale = float(np.float32(D ** -0.5))
    got = _run(hip, qkv, B, S, H, D, scale, shift=S % 2)
    ref, bound = O.attention_f64(qkv, B, S, H, D, scale)
    assert O.normalized_error(got, ref, bound) <= _tolerance(qkv, B, S, H, D, scale)


def test_cold_capture(hip, streams):
    """Long, few heads take products with intermediates; a fresh stream that records a graph cannot allocate them
    and records the fused kernel, for the staging array as for the products' own workspace."""
    B, S, H, D = 1, 1024, 1, 64
    qkv = O.randn((B * S, 3 * H * D), 13, 1.0)
    scale = float(np.float32(D ** -0.5))
    ref, bound = O.attention_f64(qkv, B, S, H, D, scale)
    dq = to_dev(hip, qkv)
    s = streams.create()
    hip.set_stream(s)
    for warm in (None, (1, 1100, 1, 10)):   # nothing, or another call's staging array alone
        if warm:
            b, n, h, d = warm
            hip.HIPBackend.attention(to_dev(hip, np.zeros((b * n, 3 * h * d), np.float32)), empty_dev(hip, (b * n, h * d)), *warm, 1.0)
        dout = empty_dev(hip, (B * S, H * D))
        g = hip.Graph(lambda: hip.HIPBackend.attention(dq, dout, B, S, H, D, scale))
        try:
            for _ in range(2):
                g.launch()
                streams.sync(s)
                got = dout.numpy()
                assert O.normalized_error(got, ref, bound) <= _tolerance(qkv, B, S, H, D, scale)
        finally:
            g.destroy()


def test_negative_scale_and_large_scores(hip):
    """Maxima that grow over the trips (scores to several hundred) and a negative scale."""
    B, S, H, D = 1, 200, 2, 32
    qkv = O.randn((B * S, 3 * H * D), 7, 4.0)
    qkv *= np.linspace(0.1, 2.0, S, dtype=np.float32)[:, None]
    for scale in (0.5, -0.5):
        ref, bound = O.attention_f64(qkv, B, S, H, D, scale)
        got = _run(hip, qkv, B, S, H, D, scale)
        assert O.normalized_error(got, ref, bound) <= _tolerance(qkv, B, S, H, D, scale)


def test_values_near_the_largest(hip):
    """Weighted means of values near the largest float stay finite."""
    B, S, H, D = 1, 150, 1, 16
    qkv = O.randn((S, 3 * D), 9, 0.5)
    qkv[:, 2 * D:] = 3.0e38
    got = _run(hip, qkv, B, S, H, D, 0.25)
    assert np.all(np.abs(got / 3.0e38 - 1) <= 2.0 ** -24 * (2 * S + 8))


def test_non_finite(hip):
    """A key whose scores are -inf has weight 0, wherever it lies (whole leading trips of them); a row that has a
    +inf or NaN score, or only -inf, is NaN."""
    B, S, H, D = 1, 140, 1, 16
    qkv = O.randn((S, 3 * D), 11, 0.5)
    qkv[:, 0] = 1.0
    masked = qkv.copy()
    masked[:70, D] = -np.inf
    got = _run(hip, masked, B, S, H, D, 0.25)
    want = qkv.astype(np.float64)
    s = 0.25 * want[:, :D] @ want[70:, D:2 * D].T
    P = np.exp(s - s.max(1, keepdims=True))
    P /= P.sum(1, keepdims=True)
    bound = P @ np.abs(want[70:, 2 * D:])
    assert O.normalized_error(got, P @ want[70:, 2 * D:], bound) <= _tolerance(qkv, B, S, H, D, 0.25)
    for bad, rows in ((np.inf, slice(90, 91)), (np.nan, slice(3, 4)), (-np.inf, slice(0, S))):
        x = qkv.copy()
        x[rows, D] = bad
        assert np.all(np.isnan(_run(hip, x, B, S, H, D, 0.25)))
