"""Finite inputs whose scores lie far below zero: one of the first key tiles, or all of them, more than 128 log2 units
down, so that 2^-maximum overflows.  Whichever wavefront meets such a tile first, forward and backward give
the oracle's numbers, in each form of the kernels.  On the CPU executor, and on the GPU."""
import numpy as np
import pytest

from oracle import oracle as O
from test_row_forms import TOL, force, where  # noqa: F401 (fixture)

TILE = {O.F32: 32, O.F16: 64, O.BF16: 64}  # keys per tile


def inputs(dtype, N, H, d, low):
    """Scores of the keys in tile `low` (None: of all keys) are below -128 log2 units, the others of order one.  The component
    that does it is a power of two in Q and in K: the kernels round c * Q and c * K to 16 bits, and so they round alike."""
    q, k, v, do = (O.round_to(O.fill_normal((1, N, H, d), 71, t), dtype) for t in (1, 2, 3, 7))
    q[..., 0] = 16.0
    k[..., 0] = 0.0
    k[:, slice(None) if low is None else slice(TILE[dtype] * low, TILE[dtype] * (low + 1)), :, 0] = -64.0 if d <= 64 else -128.0
    return q, k, v, do


def run(where, dtype, N, H, d, causal, q, k, v, do):
    (tq, pq), (tk, pk), (tv, pv), (tdo, pdo) = (where.put(x, dtype) for x in (q, k, v, do))
    outs = [where.out(q.shape, dtype) for _ in range(4)]
    n_ws = where.hip.flash_bwd_workspace_bytes(1, N, H)
    ws, pws = where.scratch(n_ws)
    scale, st = 1.0 / np.sqrt(d), (N * H * d, H * d, d)
    where.hip.flash_fwd_gqa(pq, pk, pv, outs[0][1], dtype, 1, N, H, H, d, st, st, scale, causal)
    where.hip.flash_bwd(pdo, pq, pk, pv, *(p for _, p in outs[1:]), dtype, 1, N, H, H, d, st, st, scale, causal, pws, n_ws)
    return [where.get(x, dtype) for x, _ in outs]


def check(got, q, k, v, do, dtype, N, H, d, causal):
    assert H == 1
    scale = 1.0 / np.sqrt(d)
    want = (O.attention(q, k, v, 1, N, H, d, scale, causal), *O.attention_backward(q, k, v, do, 1, N, H, d, scale, causal, H))
    # what dQ and dK are off by here, beside the ordinary tolerance: a component of size |K| or |Q| times the rounding of dS =
    # w (dP - delta) and, through the weights in delta = sum of w dP, of w (16 bits: 2^-9 of each; fp32: of scores near 200,
    # 2^-24 * 200 and a few of them)
    q2, k2, v2, do2 = (x[0, :, 0].astype(np.float64) for x in (q, k, v, do))
    s = q2 @ k2.T * scale
    if causal:
        s[np.triu_indices(N, 1)] = -np.inf
    w = np.exp(s - s.max(1, keepdims=True))
    w /= w.sum(1, keepdims=True)
    dp = do2 @ v2.T
    ds = np.abs(w * (dp - (w * dp).sum(1, keepdims=True))) + w * (w * np.abs(dp)).sum(1, keepdims=True)
    eps = 1e-4 if dtype == O.F32 else 2.0**-9
    more = (0.0, eps * scale * np.abs(k).max() * ds.sum(1).max(), eps * scale * np.abs(q).max() * ds.sum(0).max(), 0.0)
    for name, g, x, r in zip(("O", "dQ", "dK", "dV"), got, want, more):
        assert np.isfinite(g).all(), name
        bar = TOL[dtype] * max(1.0, np.abs(x).max()) + r
        assert np.abs(g - x).max() <= bar, (name, float(np.abs(g - x).max()), bar)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("low", [0, 1, 2, 3, None])
@pytest.mark.parametrize("rows", [32, 128])
def test_fp32(where, rows, low, causal):  # noqa: F811
    force(where, rows)
    N, H, d = 130, 1, 64
    x = inputs(O.F32, N, H, d, low)
    check(run(where, O.F32, N, H, d, causal, *x), *x, O.F32, N, H, d, causal)


@pytest.mark.parametrize("rows,N,d,causal", [(128, 130, 64, True), (128, 200, 128, False), (128, 130, 256, True),   # one walk
                                             (256, 260, 128, True), (256, 260, 64, False),                        # 256 rows
                                             (0, 577, 64, True), (0, 577, 128, False)])                           # two walks
@pytest.mark.parametrize("low", [0, 1, None])
@pytest.mark.parametrize("dtype", [O.BF16])
def test_16_bit(where, dtype, low, rows, N, d, causal):  # noqa: F811
    where.hip.set_tuning("flash_rows", rows)
    where.hip.set_tuning("flash_walks", 2 if rows == 0 else 1)
    H = 1
    x = inputs(dtype, N, H, d, low)
    check(run(where, dtype, N, H, d, causal, *x), *x, dtype, N, H, d, causal)


@pytest.mark.parametrize("dtype,rows,N,d,tile", [(O.F32, 32, 130, 64, 0), (O.F32, 32, 130, 64, 1), (O.F32, 32, 130, 128, 3), (O.F32, 128, 130, 64, 1),
                                                 (O.BF16, 0, 577, 64, 0), (O.BF16, 0, 577, 128, 1), (O.BF16, 128, 130, 64, 1)])
def test_a_tile_of_infinitely_low_scores(where, dtype, rows, N, d, tile):  # noqa: F811
    """Keys that an infinity in K takes out altogether: a tile of them, also as the first one a set of wavefronts meets."""
    where.hip.set_tuning("flash_rows", rows)
    where.hip.set_tuning("flash_walks", 2 if rows == 0 else 1)
    q, k, v, _ = inputs(dtype, N, 1, d, None)
    k[..., 0] = 0.0
    k[:, TILE[dtype] * tile:TILE[dtype] * (tile + 1), :, 0] = -np.inf
    (tq, pq), (tk, pk), (tv, pv), (o, po) = *(where.put(x, dtype) for x in (q, k, v)), where.out(q.shape, dtype)
    scale, st = 1.0 / np.sqrt(d), (N * d, d, d)
    where.hip.flash_fwd_gqa(pq, pk, pv, po, dtype, 1, N, 1, 1, d, st, st, scale, False)
    keep = np.r_[0:TILE[dtype] * tile, min(N, TILE[dtype] * (tile + 1)):N]
    s = q[0, :, 0].astype(np.float64) @ k[0, keep, 0].astype(np.float64).T * scale
    w = np.exp(s - s.max(1, keepdims=True))
    want = (w / w.sum(1, keepdims=True)) @ v[0, keep, 0].astype(np.float64)
    got = where.get(o, dtype)[0, :, 0]
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= TOL[dtype] * max(1.0, np.abs(want).max())
