"""Both forms of the kernels that exist in two: workgroups of 128 rows (32 per wavefront) and workgroups of 32 rows whose
wavefronts share the walk over the other side.  The launcher chooses by size; here each form is forced at the sizes where it
can go wrong: fewer tiles than wavefronts, a last tile of 1 to 31 rows, blocks at and beyond a 32- or 128-row boundary,
grouped heads, ragged batches with an empty sequence, head dimensions below the kernel's.  On the CPU executor, and on the GPU."""
import numpy as np
import pytest

from oracle import oracle as O
from simt import simt as S

TOL = {O.F32: 1e-4, O.F16: 2e-2, O.BF16: 2e-2}

DENSE = [(1, 1, 2, 2, 128, True), (2, 31, 2, 1, 64, False), (1, 33, 3, 3, 64, True), (1, 130, 2, 1, 128, True),
         (2, 129, 2, 2, 64, False), (1, 160, 4, 2, 96, False), (1, 290, 2, 1, 40, True)]
RAGGED = [((130, 0, 1, 33), 2, 1, 64, True), ((31, 160, 257), 2, 2, 128, False), ((97, 300, 16, 64), 4, 2, 80, True)]


class Executor:
    def __init__(self):
        S.load()
        S.configure(True, 3)
        self.hip = S.EmulatedHip()

    def put(self, x, dtype):
        x = S.guarded(S.to_storage(x, dtype))
        return x, S.ptr(x)

    def ints(self, x):
        x = S.guarded(np.asarray(x, np.int32))
        return x, S.ptr(x)

    def out(self, shape, dtype):
        x = S.guarded(S.empty_storage(shape, dtype))
        return x, S.ptr(x)

    def scratch(self, n):
        x = S.guarded(np.full(n // 4, np.nan, np.float32))
        return x, S.ptr(x)

    def get(self, x, dtype):
        return S.from_storage(x, dtype)


class Gpu:
    def __init__(self, hip):
        self.hip = hip

    def put(self, x, dtype):
        from gpu_util import to_dev
        t = to_dev(x, dtype)
        return t, t.data_ptr()

    def ints(self, x):
        from gpu_util import dev_i32
        t = dev_i32(x)
        return t, t.data_ptr()

    def out(self, shape, dtype):
        import torch
        from gpu_util import torch_dtype
        t = torch.full(shape, float("nan"), dtype=torch_dtype(dtype), device="cuda")
        return t, t.data_ptr()

    def scratch(self, n):
        import torch
        t = torch.full((n // 4,), float("nan"), dtype=torch.float32, device="cuda")
        return t, t.data_ptr()

    def get(self, x, dtype):
        import torch
        from gpu_util import to_host
        torch.cuda.synchronize()
        return to_host(x)


@pytest.fixture(params=["executor", pytest.param("gpu", marks=pytest.mark.gpu)])
def where(request):
    if request.param == "gpu":
        w = Gpu(request.getfixturevalue("gpu"))
    else:
        w = Executor()
    before = {n: w.hip.get_tuning(n) for n in ("flash_rows", "flash_walks", "bwd_split", "flash_pair_min_tiles")}
    yield w
    for n, v in before.items():
        w.hip.set_tuning(n, v)
    if request.param != "gpu":
        S.configure(False, 1)


def force(where, rows):
    where.hip.set_tuning("flash_rows", rows)
    where.hip.set_tuning("bwd_split", 3 if rows == 32 else 1)
    where.hip.set_tuning("flash_pair_min_tiles", 1)  # (128 rows: causal launches of two tiles and more take them in pairs)


def check(got, want, dtype):
    for name, g, w in zip(("O", "dQ", "dK", "dV"), got, want):
        assert np.isfinite(g).all(), name
        bar = TOL[dtype] * max(1.0, np.abs(w).max())
        assert np.abs(g - w).max() <= bar, (name, float(np.abs(g - w).max()), bar)


@pytest.mark.parametrize("rows", [32, 128])
@pytest.mark.parametrize("dtype", [O.F32])
@pytest.mark.parametrize("B,N,H,H_kv,d,causal", DENSE)
def test_dense(where, rows, dtype, B, N, H, H_kv, d, causal):
    force(where, rows)
    q, do = (O.round_to(O.fill_normal((B, N, H, d), 51, t), dtype) for t in (1, 7))
    k, v = (O.round_to(O.fill_normal((B, N, H_kv, d), 51, t), dtype) for t in (2, 3))
    (tq, pq), (tk, pk), (tv, pv), (tdo, pdo) = (where.put(x, dtype) for x in (q, k, v, do))
    (o, po), (gq, pgq) = where.out(q.shape, dtype), where.out(q.shape, dtype)
    (gk, pgk), (gv, pgv) = where.out(k.shape, dtype), where.out(k.shape, dtype)
    n_ws = where.hip.flash_bwd_workspace_bytes(B, N, H)
    ws, pws = where.scratch(n_ws)
    scale, st, kst = 1.0 / np.sqrt(d), (N * H * d, H * d, d), (N * H_kv * d, H_kv * d, d)
    where.hip.flash_fwd_gqa(pq, pk, pv, po, dtype, B, N, H, H_kv, d, st, kst, scale, causal)
    where.hip.flash_bwd(pdo, pq, pk, pv, pgq, pgk, pgv, dtype, B, N, H, H_kv, d, st, kst, scale, causal, pws, n_ws)
    rep = H // H_kv
    want = (O.attention(q, np.repeat(k, rep, axis=2), np.repeat(v, rep, axis=2), B, N, H, d, scale, causal),
            *O.attention_backward(q, k, v, do, B, N, H, d, scale, causal, H_kv))
    check([where.get(x, dtype) for x in (o, gq, gk, gv)], want, dtype)


@pytest.mark.parametrize("rows", [32, 128])
@pytest.mark.parametrize("dtype", [O.F32])
@pytest.mark.parametrize("lens,H,H_kv,d,causal", RAGGED)
def test_ragged(where, rows, dtype, lens, H, H_kv, d, causal):
    force(where, rows)
    ragged_forward_and_backward(where, dtype, lens, H, H_kv, d, causal)


def ragged_forward_and_backward(where, dtype, lens, H, H_kv, d, causal):
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, longest, n = int(cu[-1]), max(lens), len(lens)
    q, do = (O.round_to(O.fill_normal((T, H, d), 52, t), dtype) for t in (1, 7))
    k, v = (O.round_to(O.fill_normal((T, H_kv, d), 52, t), dtype) for t in (2, 3))
    (tq, pq), (tk, pk), (tv, pv), (tdo, pdo) = (where.put(x, dtype) for x in (q, k, v, do))
    (o, po), (gq, pgq) = where.out(q.shape, dtype), where.out(q.shape, dtype)
    (gk, pgk), (gv, pgv) = where.out(k.shape, dtype), where.out(k.shape, dtype)
    tcu, pcu = where.ints(cu)
    n_ws = where.hip.flash_bwd_workspace_bytes(n, longest, H)
    ws, pws = where.scratch(n_ws)
    scale = 1.0 / np.sqrt(d)
    where.hip.flash_fwd_varlen_gqa(pq, pk, pv, po, dtype, pcu, n, longest, H, H_kv, d, H * d, d, H_kv * d, d, scale, causal)
    where.hip.flash_bwd_varlen(pdo, pq, pk, pv, pgq, pgk, pgv, dtype, pcu, n, longest, H, H_kv, d, H * d, d, H_kv * d, d, scale,
                               causal, pws, n_ws)
    rep = H // H_kv
    want = [np.zeros_like(x) for x in (q, q, k, k)]
    for a, b in zip(cu, cu[1:]):
        if a == b:
            continue
        L = int(b - a)
        qs, ks, vs, ds = (x[None, a:b] for x in (q, k, v, do))
        parts = (O.attention(qs, np.repeat(ks, rep, axis=2), np.repeat(vs, rep, axis=2), 1, L, H, d, scale, causal),
                 *O.attention_backward(qs, ks, vs, ds, 1, L, H, d, scale, causal, H_kv))
        for w, x in zip(want, parts):
            w[a:b] = np.asarray(x).reshape(L, *w.shape[1:])
    check([where.get(x, dtype) for x in (o, gq, gk, gv)], want, dtype)


# The 16-bit backward of a ragged batch, tiles singly and in pairs: odd and even numbers of tiles, sequences of fewer than the
# longest one's, an empty one; head counts whose pairs are dealt to the XCDs whole, in 2 and in 8 slices.
@pytest.mark.parametrize("pair", [0, 1])
@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("lens,H,H_kv,d,causal", [((130, 0, 1, 33), 2, 1, 64, True), ((300, 129, 0, 257), 4, 4, 128, True),
                                                  ((31, 160), 8, 8, 96, True), ((200, 385), 3, 3, 64, False)])
def test_ragged_backward_16_bit(where, pair, dtype, lens, H, H_kv, d, causal):
    before = where.hip.get_tuning("bwd_pair")
    where.hip.set_tuning("bwd_pair", pair)
    try:
        ragged_forward_and_backward(where, dtype, lens, H, H_kv, d, causal)
    finally:
        where.hip.set_tuning("bwd_pair", before)


# The 16-bit forward whose workgroups walk the keys in two sets of wavefronts (by itself in launches of few tiles, more than 512
# keys; named here): odd and even numbers of key tiles, one tile, a last tile of one row, one that only the second set has, head
# dimensions below the kernel's.
WALKS = [(1, 50, 2, 1, 64, True), (2, 65, 1, 1, 128, False), (1, 129, 2, 2, 64, True), (1, 513, 2, 2, 64, True), (1, 577, 2, 1, 128, False), (2, 640, 2, 1, 96, True), (1, 769, 4, 2, 40, True), (1, 705, 1, 1, 128, True)]


@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("B,N,H,H_kv,d,causal", WALKS)
def test_two_walks_dense(where, dtype, B, N, H, H_kv, d, causal):
    q = O.round_to(O.fill_normal((B, N, H, d), 53, 1), dtype)
    k, v = (O.round_to(O.fill_normal((B, N, H_kv, d), 53, t), dtype) for t in (2, 3))
    k[:, 64:128] *= 3.0  # the second set's first tile holds the largest scores, and the sets' maxima differ
    (tq, pq), (tk, pk), (tv, pv) = (where.put(x, dtype) for x in (q, k, v))
    scale, st, kst = 1.0 / np.sqrt(d), (N * H * d, H * d, d), (N * H_kv * d, H_kv * d, d)
    n_st = where.hip.flash_row_stats_bytes(B, N, H)
    got, stats = [], []
    for walks in (2, 1):
        where.hip.set_tuning("flash_walks", walks)
        (o, po), (ws, pws) = where.out(q.shape, dtype), where.scratch(n_st)
        assert where.hip.flash_fwd_keep(pq, pk, pv, po, dtype, B, N, H, H_kv, d, st, kst, scale, causal, pws)
        got.append(where.get(o, dtype))
        stats.append((ws.cpu().numpy() if hasattr(ws, "cpu") else np.asarray(ws)).reshape(B * H, -1)[:, :N])
    rep = H // H_kv
    want = O.attention(q, np.repeat(k, rep, axis=2), np.repeat(v, rep, axis=2), B, N, H, d, scale, causal)
    check(got[:1], [want], dtype)
    check(got[1:], [want], dtype)
    if N > 512:
        assert not np.array_equal(got[0], got[1])  # two forms ran: their weights are rounded against different maxima
    # log2 of sums of up to N fp32 terms in two orders (N * 2^-24 / ln 2), and the reference maxima's own rounding (|m| < 64: 2^-18)
    assert np.abs(stats[0] - stats[1]).max() <= N * 2.0**-23 + 2.0**-16


@pytest.mark.parametrize("lens,H,H_kv,d,causal", [((513, 0, 1, 65), 2, 1, 64, True), ((64, 2, 128), 2, 2, 64, False), ((64, 600, 130), 2, 2, 128, False), ((300, 577, 16), 2, 1, 80, True)])
def test_two_walks_ragged(where, lens, H, H_kv, d, causal):
    dtype = O.BF16
    where.hip.set_tuning("flash_walks", 2)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, longest, n = int(cu[-1]), max(lens), len(lens)
    q = O.round_to(O.fill_normal((T, H, d), 54, 1), dtype)
    k, v = (O.round_to(O.fill_normal((T, H_kv, d), 54, t), dtype) for t in (2, 3))
    (tq, pq), (tk, pk), (tv, pv), (tcu, pcu), (o, po) = *(where.put(x, dtype) for x in (q, k, v)), where.ints(cu), where.out(q.shape, dtype)
    scale, rep = 1.0 / np.sqrt(d), H // H_kv
    where.hip.flash_fwd_varlen_gqa(pq, pk, pv, po, dtype, pcu, n, longest, H, H_kv, d, H * d, d, H_kv * d, d, scale, causal)
    want = np.zeros_like(q)
    for a, b in zip(cu, cu[1:]):
        if b > a:
            qs, ks, vs = (x[None, a:b] for x in (q, k, v))
            want[a:b] = np.asarray(O.attention(qs, np.repeat(ks, rep, axis=2), np.repeat(vs, rep, axis=2), 1, int(b - a), H, d, scale,
                                               causal)).reshape(b - a, H, d)
    check([where.get(o, dtype)], [want], dtype)
