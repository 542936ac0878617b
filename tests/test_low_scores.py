"""Finite inputs whose scores lie far below zero: one of the first key tiles, or all of them, more than 128 log2 units
down, so that 2^-maximum overflows.  Whichever wavefront meets such a tile first, forward and backward give
the oracle's numbers, in each form of the kernels.  On the CPU executor, and on the GPU."""
import numpy as np
import pytest

from oracle import oracle as O
from test_row_forms import TOL, force, where  # noqa: F401 (fixture)

TILE = {O.F32: 32, O.F16: 64, O.BF16: 64}  # keys per tile


def inputs(dtype, N, H, d, low):
    """Scores of the keys in tile `low` (None: of all keys) are -100 nats, the others of order one."""
    q, k, v, do = (O.round_to(O.fill_normal((1, N, H, d), 71, t), dtype) for t in (1, 2, 3, 7))
    q[..., 0] = 10.0
    k[..., 0] = 0.0
    k[:, slice(None) if low is None else slice(TILE[dtype] * low, TILE[dtype] * (low + 1)), :, 0] = -10.0 * np.sqrt(d)
    return q, O.round_to(k, dtype), v, do


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
    scale = 1.0 / np.sqrt(d)
    want = (O.attention(q, k, v, 1, N, H, d, scale, causal), *O.attention_backward(q, k, v, do, 1, N, H, d, scale, causal, H))
    # an error e in the weights is scale * |K| * e in dQ, scale * |Q| * e in dK
    reach = (1.0, scale * np.abs(k).max(), scale * np.abs(q).max(), 1.0)
    for name, g, w, r in zip(("O", "dQ", "dK", "dV"), got, want, reach):
        assert np.isfinite(g).all(), name
        bar = TOL[dtype] * max(1.0, np.abs(w).max(), r)
        assert np.abs(g - w).max() <= bar, (name, float(np.abs(g - w).max()), bar)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("low", [0, 1, 2, 3, None])
@pytest.mark.parametrize("rows", [32])
def test_fp32(where, rows, low, causal):  # noqa: F811
    force(where, rows)
    N, H, d = 130, 1, 64
    x = inputs(O.F32, N, H, d, low)
    check(run(where, O.F32, N, H, d, causal, *x), *x, O.F32, N, H, d, causal)
