"""fp32 tensors up to d = 128 are multiplied in three bf16 pieces on the matrix cores.  What can go wrong there: a piece left
out, and inputs that have no such pieces (infinities, magnitudes at the ends of the range), which are computed with the
fp32 instructions instead.  Both forms of the kernels (32 and 128 rows per workgroup), against 64-bit arithmetic."""
import numpy as np
import pytest

from oracle import oracle as O


class _Cpu:
    """The kernels on the CPU executor."""

    def __init__(self):
        from simt import simt as S
        S.load()
        S.configure(False, 1)
        self.S, self.hip = S, S.EmulatedHip()
        self.set_tuning = self.hip.set_tuning

    def forward(self, q, k, v, causal, scale):
        S = self.S
        B, N, H, d = q.shape
        H_kv = k.shape[2]
        dq, dk, dv, do = (S.guarded(np.ascontiguousarray(x)) for x in (q, k, v, np.zeros_like(q)))
        self.hip.flash_fwd_gqa(S.ptr(dq), S.ptr(dk), S.ptr(dv), S.ptr(do), O.F32, B, N, H, H_kv, d, (N * H * d, H * d, d),
                               (N * H_kv * d, H_kv * d, d), scale, causal, None, None)
        return np.array(do).reshape(q.shape).astype(np.float64)


class _Gpu:
    def __init__(self):
        import torch
        torch.cuda.init()
        from attention_amd import hip
        self.hip, self.set_tuning = hip, hip.set_tuning

    def forward(self, q, k, v, causal, scale):
        import torch
        B, N, H, d = q.shape
        H_kv = k.shape[2]
        dq, dk, dv = (torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (q, k, v))
        do = torch.zeros_like(dq)
        self.hip.flash_fwd_gqa(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), do.data_ptr(), O.F32, B, N, H, H_kv, d, (N * H * d, H * d, d),
                               (N * H_kv * d, H_kv * d, d), scale, causal, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return do.cpu().numpy().astype(np.float64)


@pytest.fixture(params=[_Cpu, pytest.param(_Gpu, marks=pytest.mark.gpu)], ids=["cpu", "gpu"])
def device(request):
    return request.param()


def exact(q, k, v, causal, scale):
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    N, group = q.shape[1], q.shape[2] // k.shape[2]
    out = np.empty_like(q)
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            s = q[b, :, h] @ k[b, :, h // group].T * scale
            if causal:
                s = np.where(np.tril(np.ones((N, N), bool)), s, -np.inf)
            p = np.exp(s - s.max(1, keepdims=True))
            out[b, :, h] = p @ v[b, :, h // group] / p.sum(1, keepdims=True)
    return out


def inputs(N, d, H_kv, seed):
    r = np.random.default_rng(seed)
    return tuple(r.standard_normal((1, N, h, d)).astype(np.float32) for h in (2, H_kv, H_kv))


@pytest.mark.parametrize("rows", [32, 128])
@pytest.mark.parametrize("N,d,H_kv,causal", [(33, 64, 2, False), (129, 64, 1, True), (95, 128, 2, True), (64, 128, 1, False), (40, 96, 2, False), (31, 100, 2, True)])
def test_all_pieces_count(device, rows, N, d, H_kv, causal):
    """A product of pieces that is left out would be an error of 2^-17 (a middle times a middle or a first times a last one) or more of
    single products: 3e-6 in the 2-norm of these sums, where fp32 rounding of inputs, weights and sums leaves 2e-7 (d = 64) to 4e-7."""
    q, k, v = inputs(N, d, H_kv, 5)
    device.set_tuning("flash_rows", rows)
    try:
        got = device.forward(q, k, v, causal, d ** -0.5)
    finally:
        device.set_tuning("flash_rows", 0)
    want = exact(q, k, v, causal, d ** -0.5)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 6e-7


@pytest.mark.parametrize("rows", [32, 128])
@pytest.mark.parametrize("d", [64, 128])
def test_values_without_pieces(device, rows, d):
    N = 70
    q, k, v = inputs(N, d, 2, 6)
    scale = d ** -0.5
    device.set_tuning("flash_rows", rows)
    try:
        # an infinite value: every query has an infinity in that column, nothing else changes
        v1 = v.copy()
        v1[0, 40, 1, 7] = np.inf
        got, want = device.forward(q, k, v1, False, scale), exact(q, k, v, False, scale)
        assert np.isposinf(got[0, :, 1, 7]).all()
        got[0, :, 1, 7] = want[0, :, 1, 7]
        assert np.abs(got - want).max() <= 1e-5
        # an infinite key element that every query meets with a factor of the other sign: weight 0
        k1 = k.copy()
        k1[0, 20, 0, 3] = -np.inf
        q1 = np.abs(q)
        keep = np.delete(np.arange(N), 20)
        got = device.forward(q1, k1, v, False, scale)
        s = q1[0, :, 0].astype(np.float64) @ k[0, keep, 0].T.astype(np.float64) * scale
        p = np.exp(s - s.max(1, keepdims=True))
        assert np.abs(got[0, :, 0] - p @ v[0, keep, 0] / p.sum(1, keepdims=True)).max() <= 1e-5
        # the lower end of the range: the last pieces of these are below the smallest normal number
        small = v * np.float32(1e-36)
        got, want = device.forward(q, k, small, False, scale) * 1e36, exact(q, k, small, False, scale) * 1e36
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 6e-7
    finally:
        device.set_tuning("flash_rows", 0)
