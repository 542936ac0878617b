"""Dense masks made of blocks: the 16-bit forward walks only the 64 x 64 tiles that
hold a visible pair.  Masks whose first, last, odd or even tiles are empty for a query block, query blocks that see nothing,
one live row of 16 in a tile, more tiles than one 64-tile window, causal launches with paired query tiles.  On the CPU
executor, and on the GPU."""
import numpy as np
import pytest

from oracle import oracle as O
from simt import simt as S
from test_row_forms import Executor, Gpu


@pytest.fixture(params=["executor", pytest.param("gpu", marks=pytest.mark.gpu)])
def where(request):
    w = Gpu(request.getfixturevalue("gpu")) if request.param == "gpu" else Executor()
    before = w.hip.get_tuning("flash_pair_min_tiles")
    w.hip.set_tuning("flash_pair_min_tiles", 1)
    yield w
    w.hip.set_tuning("flash_pair_min_tiles", before)
    if request.param != "gpu":
        S.configure(False, 1)


def block_mask(B, N, share, seed):
    """Random live 64 x 64 tiles with a few single pairs in place of whole ones."""
    rng = np.random.default_rng(seed)
    t = (N + 63) // 64
    live = rng.random((B, t, t)) < share
    live[0, 0, :] = False            # a query block that sees nothing (its 128-row tile has another half)
    if t > 2:
        live[0, 2, :-1] = False      # only the last tile, which may be short
        live[0, 2, -1] = True
    mask = np.repeat(np.repeat(live, 64, 1), 64, 2)[:, :N, :N].astype(np.float32)
    mask *= rng.random(mask.shape) < 0.9
    mask[-1, N - 1, :] = 0.0
    mask[-1, N - 1, N // 2] = 1.0    # one pair in an otherwise empty row
    return np.ascontiguousarray(mask)


@pytest.mark.parametrize("dtype,B,N,H,H_kv,d,causal,share", [
    (O.F16, 2, 577, 2, 1, 64, False, 0.3), (O.BF16, 2, 577, 2, 1, 64, False, 0.3), (O.BF16, 2, 450, 1, 1, 128, True, 0.4),
    (O.F16, 1, 300, 2, 2, 96, False, 0.0), (O.F16, 1, 4100, 1, 1, 64, False, 0.01), (O.BF16, 1, 200, 1, 1, 256, False, 0.5)])
def test_tiles_without_a_visible_pair(where, dtype, B, N, H, H_kv, d, causal, share):
    if N > 4096 and isinstance(where, Executor):
        pytest.skip("more tiles than one window: minutes on the executor")
    mask = block_mask(B, N, share, N + d)
    q = O.round_to(O.fill_normal((B, N, H, d), 61, 1), dtype)
    k, v = (O.round_to(O.fill_normal((B, N, H_kv, d), 61, t), dtype) for t in (2, 3))
    (tq, pq), (tk, pk), (tv, pv) = (where.put(x, dtype) for x in (q, k, v))
    tm, pm = where.put(mask, O.F32)
    o, po = where.out(q.shape, dtype)
    rep = H // H_kv
    scale, st, kst = 1.0 / np.sqrt(d), (N * H * d, H * d, d), (N * H_kv * d, H_kv * d, d)
    where.hip.flash_fwd_gqa(pq, pk, pv, po, dtype, B, N, H, H_kv, d, st, kst, scale, causal, None, pm)
    want = O.attention(q, np.repeat(k, rep, axis=2), np.repeat(v, rep, axis=2), B, N, H, d, scale, causal, mask=mask)
    got = where.get(o, dtype)
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= 2e-2 * max(1.0, np.abs(want).max())
