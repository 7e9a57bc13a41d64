"""fp32 GEMM through bf16 pieces: every tile at its edges, and the values that the pieces carry with
difficulty (denormals) or not at all (infinities, NaN, huge values), against float64.

Bound: each output is a sum of K products; in any order, with every product and addition rounded to
fp32 and (6 of 9 piece products) at most 2^-24 of each product left out, it is within
(K + 2) 2^-24 sum |a b| of the exact sum, plus the smallest denormal for each of those roundings (tiles
recomputed on the fp32 MFMA round every addition to the denormal spacing).
"""
import numpy as np
import pytest

from conftest import empty_dev, to_dev

pytestmark = pytest.mark.gpu

# (M, N): 64x64 tiles, 128x128 tiles (one per CU / several), 256x256 tiles on a 256-CU device, each also ragged
TILES = [(64, 64), (65, 131), (2048, 2048), (1930, 2047), (2048, 4096), (2047, 3970), (4096, 4096), (4090, 3845)]
DEPTHS = [1, 15, 16, 17, 33, 64, 80, 81, 97, 112, 129]   # 1 .. 9 slices of 16, whole and partial


def _operands(M, N, K, seed):
    r = np.random.default_rng(seed)
    return r.standard_normal((M, K), dtype=np.float32), r.standard_normal((K, N), dtype=np.float32)


def _run(hip, layout, A, B):
    M, K = A.shape
    N = B.shape[1]
    dC = empty_dev(hip, (M, N))
    H = hip.HIPBackend
    if layout == "nn":
        H.matmul(to_dev(hip, A), to_dev(hip, B), dC, M, K, N)
    elif layout == "nt":
        H.matmulTransB(to_dev(hip, A), to_dev(hip, B.T), dC, M, K, N)
    elif layout == "tn":
        H.matmulTransA(to_dev(hip, A.T), to_dev(hip, B), dC, M, K, N)
    else:
        H.gemmStridedBatched(True, True, 1, M, N, K, to_dev(hip, A.T), M, 0, to_dev(hip, B.T), K, 0, dC, N, 0)
    return dC.numpy()


def _check(got, A, B, rows):
    a, b = A[rows].astype(np.float64), B.astype(np.float64)
    with np.errstate(all="ignore"):
        ref = a @ b
        mag = np.abs(a) @ np.abs(b)
    got = got[rows].astype(np.float64)
    fine = np.isfinite(ref) & (mag < 3.0e38)
    over = ~np.isfinite(ref)
    assert np.array_equal(np.isnan(got[over]), np.isnan(ref[over]))
    inf = over & np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf])
    bound = (A.shape[1] + 2) * (2.0 ** -24 * mag + 2.0 ** -149)
    assert np.all(np.abs(got[fine] - ref[fine]) <= bound[fine])
    return fine


def _rows(M):
    """All rows of a small product, else the edges of the tiles and some between."""
    if M <= 160:
        return np.arange(M)
    return np.unique(np.r_[0:3, 62:66, 126:130, 254:258, np.arange(300, M, 211), M - 70:M - 60, M - 3:M])


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N", TILES)
def test_tile_edges(hip, layout, M, N):
    for K in DEPTHS if M * N < 1 << 16 else DEPTHS[1::3]:
        print(f"case {layout} {M}x{N}x{K}", flush=True)
        A, B = _operands(M, N, K, M + N + K)
        assert _check(_run(hip, layout, A, B), A, B, _rows(M)).all()


# The plan's lines between the pieces and the fp32 MFMA on the 64x64 tile: few tiles (unsplit, split into short and
# long pieces), more tiles than CUs; row counts that are and are not multiples of four; the last slice of each length.
ROUTES = [(64, 60, k) for k in (1, 2, 3, 4, 5, 19, 31, 32, 33, 36, 511, 512, 530, 1000, 1023, 1024, 1030, 2047, 2048, 4100)] + \
         [(61, 131, k) for k in (1, 3, 18, 47, 512, 1023, 1025, 2050)] + [(9, 4096, k) for k in (2040, 4099)] + \
         [(1000, 2047, k) for k in (1, 30, 33, 191, 192, 193, 224, 288, 319, 320, 321, 322, 323, 338, 352)] + \
         [(1500, 1501, k) for k in (32, 33, 127, 128, 129)] + \
         [(100, 1000, k) for k in (1100, 1216, 1500, 2100)] + [(128, 4000, 2100), (333, 999, 321), (333, 999, 319)]


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N", sorted({r[:2] for r in ROUTES}))
def test_small_tile_routes(hip, layout, M, N):
    for K in [r[2] for r in ROUTES if r[:2] == (M, N)]:
        print(f"case {layout} {M}x{N}x{K}", flush=True)
        A, B = _operands(M, N, K, M + K)
        got = _run(hip, layout, A, B)
        assert _check(got, A, B, _rows(M)).all()
        if K == 1:   # one product: the nearest float, in any layout
            assert np.array_equal(got.view(np.uint32), (A * B).view(np.uint32))


@pytest.mark.parametrize("N", [260, 2048, 4096])
def test_one_term_sums(hip, N):
    """A diagonal matrix times another: each output is one product among zeros. Through the pieces it is off by at
    most the three piece products left out (2^-24 of it) and, as an MFMA's sum is one of the two floats beside the
    exact one, a unit in the last place and 2^-29 for the roundings of the smaller pieces."""
    r = np.random.default_rng(9)
    d, B = r.standard_normal(N).astype(np.float32), r.standard_normal((N, N), dtype=np.float32)
    exact = d.astype(np.float64)[:, None] * B
    got = _run(hip, "nn", np.diag(d), B)
    ulp = np.spacing(np.abs(exact).astype(np.float32)).astype(np.float64)
    assert np.all(np.abs(got - exact) <= (2.0 ** -24 + 2.0 ** -29) * np.abs(exact) + ulp)


@pytest.mark.parametrize("nz", [2, 7, 64])
@pytest.mark.parametrize("N", [2048, 4096])
def test_few_term_sums(hip, nz, N):
    """Rows with nz elements among zeros: each of the (at most nz) slices that hold them adds six piece products to
    the sums, each addition off by at most 2^-23 of sum |a b|, and leaves 2^-24 out."""
    r = np.random.default_rng(nz)
    A, B = np.zeros((N, N), np.float32), r.standard_normal((N, N), dtype=np.float32)
    for i in range(192):
        A[i, r.choice(N, nz, replace=False)] = r.standard_normal(nz)
    got = _run(hip, "nn", A, B)[:192].astype(np.float64)
    a = A[:192].astype(np.float64)
    assert np.all(np.abs(got - a @ B) <= (6 * nz * 2.0 ** -23 + 2.0 ** -24) * (np.abs(a) @ np.abs(B)))


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(70, 67, 40), (128, 256, 2048), (2048, 2048, 50), (2048, 4096, 50), (4096, 4096, 50)])
def test_special_values(hip, layout, M, N, K):
    """Infinities, NaN, huge values and denormals in single elements; 128x256x2048 splits K."""
    A, B = _operands(M, N, K, 7)
    A[3, 5], A[9, 0], A[M - 1, K - 1] = np.inf, np.nan, -np.inf
    A[12, :] = 0
    A[12, 7] = np.inf                       # inf * b, and 0 elsewhere
    A[20, 4], B[4, 11] = 3.3e38, 1e-30      # beyond the pieces' range, finite products
    A[21, 6] = -2.7e33                      # 2^111
    B[6, :] *= np.float32(1e-20)
    A[30, :] = np.float32(1e-42)            # denormal
    A[31, :] = np.float32(3e-39)
    A[32, :] *= np.float32(1e-36)
    B[:, 20] *= np.float32(1e-38)
    print(f"case {layout} {M}x{N}x{K}", flush=True)
    _check(_run(hip, layout, A, B), A, B, np.unique(np.r_[0:40, M - 2:M]))


@pytest.mark.parametrize("M,N", [(50, 45), (70, 67), (13, 131)])
@pytest.mark.parametrize("ta,tb", [(True, False), (False, False), (True, True)])
def test_row_padding_is_not_read(hip, ta, tb, M, N):
    """Rows of an operand stored K first are longer than the matrix: what lies behind them (NaN here) is read
    neither by whole slices nor by the last, partial one, so the sums are the same bits as with zeros there (a NaN
    in any lane's sums would send its block to the fp32 MFMA, which rounds differently)."""
    pad = 96
    for K in (7, 45, 128, 141):
        print(f"case {ta} {tb} {M}x{N}x{K}", flush=True)
        A, B = _operands(M, N, K, K)
        got = []
        for fill in (0.0, np.nan):
            a, b = (np.ascontiguousarray(x) for x in (A.T if ta else A, B.T if tb else B))
            lda, ldb = a.shape[1], b.shape[1]
            if ta:
                a, lda = np.c_[a, np.full((K, pad), fill, np.float32)], M + pad
            if not tb:
                b, ldb = np.c_[b, np.full((K, pad), fill, np.float32)], N + pad
            dC = empty_dev(hip, (M, N))
            hip.HIPBackend.gemmStridedBatched(ta, tb, 1, M, N, K, to_dev(hip, a), lda, 0, to_dev(hip, b), ldb, 0, dC, N, 0)
            got.append(dC.numpy())
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
        assert _check(got[0], A, B, np.arange(M)).all()


BF16_MAX = 2.0 ** 128 - 2.0 ** 120


# The scaled operand's first piece overflows from half a bf16 ulp above the largest bf16 on (2^-16 of it, about
# 2^112), a scaled sum at 2^128 (2^96 of the sum itself).
@pytest.mark.parametrize("big,other", [(2.0 ** 111, 1e-3), (BF16_MAX * 2.0 ** -16, 1e-3), (2.0 ** 112 - 2.0 ** 103, 1e-3),
                                       (2.0 ** 112, 1e-3), (3.4e38, 1e-3), (2.0 ** 94, 1.0), (2.0 ** 95, 1.0),
                                       (2.0 ** 96, 1.0), (2.0 ** 97, 1.0), (2.0 ** 120, 2.0 ** -25), (2.0 ** 60, 2.0 ** 40)])
@pytest.mark.parametrize("M,N,K", [(64, 64, 33), (130, 70, 600), (2048, 2048, 20), (4096, 4096, 20)])
def test_hand_over(hip, M, N, K, big, other):
    """One huge element alone in the whole product, below and above what the pieces carry: its row is as exact as
    any other, and so is the rest of its tile, which the fp32 MFMA computes again with it."""
    print(f"case {M}x{N}x{K} {big:.3g}", flush=True)
    A, B = _operands(M, N, K, 11)
    A[5, K - 2] = big
    B[K - 2, :] = (np.float32(other) * np.sign(B[K - 2, :])).astype(np.float32)
    assert _check(_run(hip, "nn", A, B), A, B, np.r_[0:9, 30:36, 62:64]).all()


@pytest.mark.parametrize("scale_a,scale_b", [(1e-42, 1e36), (1e-40, 1e-2), (1e-37, 1e-5), (1e32, 1e-32), (1e18, 1e19)])
def test_ranges(hip, scale_a, scale_b):
    """Whole operands of denormals, tiny and huge values (the last two near and past the pieces' range)."""
    A, B = _operands(130, 70, 45, 3)
    A, B = A * np.float32(scale_a), B * np.float32(scale_b)
    _check(_run(hip, "nn", A, B), A, B, np.arange(130))


def test_linear_backward_special_values(hip):
    """The fused backward's products and column sums with a huge and an infinite gradient element."""
    H = hip.HIPBackend
    nb, ni, no = 37, 70, 66
    r = np.random.default_rng(5)
    X, G, W = (r.standard_normal(s, dtype=np.float32) for s in ((nb, ni), (nb, no), (ni, no)))
    X[4, :] = 0
    G[4, 9], G[7, 20], G[8, 21] = 3e38, np.inf, 1e-42
    dW, db, dX = empty_dev(hip, (ni, no)), empty_dev(hip, (no,)), empty_dev(hip, (nb, ni))
    H.linearBackward(to_dev(hip, X), to_dev(hip, G), to_dev(hip, W), None, dW, db, dX, nb, ni, no)
    want = np.zeros(no, np.float32)
    for row in G:
        want = want + row
    assert np.array_equal(db.numpy(), want)
    _check(dW.numpy(), np.ascontiguousarray(X.T), G, np.arange(ni))
    keep = np.setdiff1d(np.arange(nb), [4])   # row 4 overflows
    _check(dX.numpy(), G, np.ascontiguousarray(W.T), keep)
