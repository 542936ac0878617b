"""The work that programs give this framework, as cases that can be timed: prefill, training steps (forward and backward)
and decode steps over a paged cache, each through the package's public entry points on torch tensors that live on the GPU.

A case is a dict of plain values; its "path" says which of four programs it belongs to:

  prefill   one dense forward: B sequences of N tokens, H query heads over H_kv, head dimension d, with or without a causal
            mask or a dense mask [B,N,N]
  serve     what a server does with a batch of new prompts of different lengths: one forward over the packed batch, then
            its K and V into the paged cache
  train     a forward that keeps its row statistics and the backward of the same tensors; with "lo" / "hi" a packed batch
            of sequences of different lengths
  decode    one step of generation for B sequences with a filled cache: the new token's K and V are appended, then its
            query attends to the whole context

Lengths and page orders follow from the case ("lens_seed"), the values in the tensors from the seed given to prepare().
"""
import math
import random

import torch

from attention_amd import hip

_CODE = {"fp32": hip.F32, "fp16": hip.F16, "bf16": hip.BF16}
_TYPE = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_PAGE = 16  # tokens per page of the cache


def listed():
    return [
        # one user at a chat prompt, generating: the smallest call there is, where latency is all that counts
        dict(name="decode_one", path="decode", dtype="bf16", B=1, H=32, H_kv=8, d=128, lo=777, hi=777, lens_seed=1),
        # a serving batch with grouped heads, contexts of a few thousand tokens
        dict(name="decode_grouped", path="decode", dtype="bf16", B=16, H=32, H_kv=8, d=128, lo=512, hi=4096, lens_seed=2),
        # a large serving batch, one cached head per query head: the repository's decode headline
        dict(name="decode_batch", path="decode", dtype="fp16", B=64, H=32, H_kv=32, d=128, lo=512, hi=4096, lens_seed=3),
        # a few long documents being continued
        dict(name="decode_long", path="decode", dtype="bf16", B=8, H=32, H_kv=32, d=128, lo=16384, hi=32768, lens_seed=4),
        # one prompt of ordinary, odd length with grouped heads: time to the first token
        dict(name="prefill_prompt", path="prefill", dtype="bf16", B=1, N=777, H=32, H_kv=8, d=128, causal=True, mask=False),
        # the repository's prefill headline
        dict(name="prefill_batch", path="prefill", dtype="bf16", B=4, N=4096, H=32, H_kv=32, d=128, causal=True, mask=False),
        # the small fp32 configuration of the C++ interface's own tests: default data type, no causal mask
        dict(name="prefill_fp32", path="prefill", dtype="fp32", B=2, N=512, H=8, H_kv=8, d=64, causal=False, mask=False),
        # an encoder over padded and packed documents: a dense mask, an odd length, a head dimension between the usual ones
        dict(name="prefill_masked", path="prefill", dtype="fp16", B=4, N=1001, H=16, H_kv=16, d=96, causal=False, mask=True),
        # a server's batch of new prompts of very different lengths, and their way into the cache
        dict(name="serve_ragged", path="serve", dtype="fp16", B=16, H=32, H_kv=32, d=64, lo=128, hi=8192, lens_seed=5),
        # a training step of a language model on long sequences
        dict(name="train_batch", path="train", dtype="bf16", B=4, N=4096, H=32, H_kv=32, d=128, causal=True),
        # fine-tuning on packed examples of different lengths, grouped heads
        dict(name="train_ragged", path="train", dtype="bf16", B=12, H=16, H_kv=4, d=64, lo=100, hi=2000, lens_seed=6, causal=True),
        # a small model trained in fp32, the interface's default data type
        dict(name="train_fp32", path="train", dtype="fp32", B=2, N=512, H=8, H_kv=8, d=64, causal=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng, most):
    """(H, H_kv): query heads and the heads of the cache they share."""
    group = rng.choice([1, 1, 2, 4, 4, 8, 16, 32])
    h = rng.choice([x for x in (4, 8, 12, 16, 24, 32, 40, 64) if x <= most and x % group == 0] or [group])
    return h, h // group


def _draw_once(rng):
    path = rng.choice(["prefill", "serve", "train", "decode", "decode"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp16", "fp32"])
    case = dict(path=path, dtype=dtype)
    if path == "decode":
        H, H_kv = _heads(rng, 64)
        lo = _log_int(rng, 16, 16384)
        case.update(B=_log_int(rng, 1, 128), H=H, H_kv=H_kv, d=rng.choice([64, 80, 96, 128, 128, 128, 256]), lo=lo,
                    hi=min(32768, lo * rng.choice([1, 2, 4, 8])), lens_seed=rng.randrange(1 << 20))
        return case
    if dtype == "fp32":  # small models and checks: what this type is used for
        H, H_kv = rng.choice([(4, 4), (8, 8), (12, 12), (8, 2), (16, 16)])
        d, most = rng.choice([32, 64, 64, 96, 128]), 2048
    else:
        H, H_kv = _heads(rng, 40)
        d, most = rng.choice([64, 64, 80, 96, 128, 128, 128, 256]), 16384
    case.update(H=H, H_kv=H_kv, d=d)
    if path == "serve" or (path == "train" and rng.random() < 0.35):
        lo = _log_int(rng, 16, most // 8)
        case.update(B=_log_int(rng, 2, 32), lo=lo, hi=min(most, lo * rng.choice([2, 4, 16])), lens_seed=rng.randrange(1 << 20))
    else:
        case.update(B=_log_int(rng, 1, 8), N=_log_int(rng, 64, most))
    if path != "serve":
        case.update(causal=rng.random() < 0.75)
    if path == "prefill":
        case.update(mask=case["N"] <= 4096 and rng.random() < 0.2)
    return case


def draw(rng):
    most = {}
    for c in listed():
        for k, v in work(c).items():
            most[k] = max(most.get(k, 0), v)
    while True:
        case = _draw_once(rng)
        w = work(case)
        rate = 16 if case["dtype"] == "fp32" else 1  # an fp32 product takes the matrix cores 16 times as long
        if w["bytes"] <= most["bytes"] and w["flops"] * rate <= most["flops"]:
            return case


def _lengths(case):
    rng = random.Random(case["lens_seed"])
    return [rng.randint(case["lo"], case["hi"]) for _ in range(case["B"])]


def _pages(lens, rng_seed):
    """A block table over shuffled pages: (rows of page ids, -1 behind a sequence's last page; pages in the pool)."""
    need = [-(-n // _PAGE) for n in lens]
    ids = list(range(sum(need) + 16))
    random.Random(rng_seed).shuffle(ids)
    table, at = [], 0
    for n in need:
        table.append(ids[at:at + n] + [-1] * (max(need) - n))
        at += n
    return table, len(ids)


def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    B, H, H_kv, d = case["B"], case["H"], case["H_kv"], case["d"]
    if case["path"] == "decode":
        lens = _lengths(case)
        # K and V of every cached token once, the new token's read and written, the query, the output, table and lengths
        n = 2 * sum(lens) * H_kv * d * size + 4 * B * H_kv * d * size + 2 * B * H * d * size
        return {"bytes": n + 4 * sum(-(-x // _PAGE) for x in lens) + 4 * B, "flops": 4 * H * d * sum(lens)}
    lens = _lengths(case) if "lo" in case else [case["N"]] * B
    tokens = sum(lens)
    causal = case.get("causal", True)
    pairs = sum(n * (n + 1) // 2 if causal else n * n for n in lens)
    forward = {"bytes": (2 * H + 2 * H_kv) * tokens * d * size, "flops": 4 * H * d * pairs}
    if case["path"] == "train":  # Q, K, V, dO in, O, dQ, dK, dV out; two products forward, five backward
        return {"bytes": (4 * H + 4 * H_kv) * tokens * d * size, "flops": forward["flops"] * 7 // 2}
    if case["path"] == "serve":  # and K and V written to the cache
        return {"bytes": forward["bytes"] + 2 * H_kv * tokens * d * size, "flops": forward["flops"]}
    return {"bytes": forward["bytes"] + (4 * B * case["N"] ** 2 if case["mask"] else 0), "flops": forward["flops"]}


# Against 64-bit arithmetic on the same inputs the listed cases are off by: fp32 8.7e-7 (2-norm) and 1.0e-5 (largest single
# value), fp16 forward 3.5e-4 and 6.7e-3, bf16 3.1e-3 and 0.13 (gradients; forward 2.5e-3 and 0.05: results and the weights
# of the second product are rounded to 16 bits, and late rows of a causal forward are small).  About four times that;
# fp16 gradients by the ratio of the two types' roundings.
def tolerance(case):
    return {"fp32": {"rel": 4e-6, "max": 6e-5}, "fp16": {"rel": 1.6e-3, "max": 6e-2}, "bf16": {"rel": 1.2e-2, "max": 0.4}}[case["dtype"]]


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind = _TYPE[case["dtype"]]
    B, H, H_kv, d = case["B"], case["H"], case["H_kv"], case["d"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(kind)

    def ints(values):
        return torch.tensor(values, dtype=torch.int32, device="cuda")

    s = dict(case, code=_CODE[case["dtype"]], scale=1.0 / math.sqrt(d))
    if case["path"] == "decode":
        lens = _lengths(case)
        table, n_pages = _pages(lens, case["lens_seed"])
        pool = (n_pages, _PAGE, H_kv, d)
        s.update(q=normal(B, H, d), k_new=normal(B, H_kv, d), v_new=normal(B, H_kv, d), k_pool=torch.empty(pool, dtype=kind, device="cuda"),
                 v_pool=torch.empty(pool, dtype=kind, device="cuda"))
        for name in ("k_pool", "v_pool"):  # page by page through a small fp32 buffer: the pools are the largest tensors here
            for part in s[name].split(4096):
                part.copy_(torch.randn(part.shape, generator=g, device="cuda", dtype=torch.float32))
        s.update(table=ints(table), lens=ints(lens), rows=ints(list(range(B))), at=ints([n - 1 for n in lens]), max_len=max(lens),
                 max_pages=len(table[0]))
        s["out"] = torch.empty_like(s["q"])
        s["ws_bytes"] = hip.paged_decode_workspace_bytes(B, H, d, s["max_len"], _PAGE)
        s["ws"] = torch.empty(max(s["ws_bytes"], 16), dtype=torch.uint8, device="cuda")
        return s
    ragged = "lo" in case
    lens = _lengths(case) if ragged else [case["N"]] * B
    lead = (sum(lens),) if ragged else (B, case["N"])
    s.update(q=normal(*lead, H, d), k=normal(*lead, H_kv, d), v=normal(*lead, H_kv, d), max_len=max(lens))
    s["out"] = torch.empty_like(s["q"])
    if ragged:
        at = [0]
        for n in lens:
            at.append(at[-1] + n)
        s.update(cu=ints(at), strides=(H * d, d), kv_strides=(H_kv * d, d))
    else:
        s.update(strides=(case["N"] * H * d, H * d, d), kv_strides=(case["N"] * H_kv * d, H_kv * d, d))
    if case["path"] == "serve":
        table, n_pages = _pages(lens, case["lens_seed"])
        s.update(table=ints(table), max_pages=len(table[0]), rows=ints(list(range(B))),
                 k_pool=torch.zeros((n_pages, _PAGE, H_kv, d), dtype=kind, device="cuda"),
                 v_pool=torch.zeros((n_pages, _PAGE, H_kv, d), dtype=kind, device="cuda"))
    if case["path"] == "train":
        s["d_out"] = normal(*lead, H, d)
        s.update(d_q=torch.empty_like(s["q"]), d_k=torch.empty_like(s["k"]), d_v=torch.empty_like(s["v"]))
        s["ws_bytes"] = hip.flash_bwd_workspace_bytes(B, s["max_len"], H)
        s["ws"] = torch.empty(s["ws_bytes"], dtype=torch.uint8, device="cuda")
        if not ragged:
            s["stats"] = torch.empty(hip.flash_row_stats_bytes(B, case["N"], H), dtype=torch.uint8, device="cuda")
    if case.get("mask"):
        # documents of about a third of the length side by side, padding behind the last, a few pairs dropped
        N = case["N"]
        doc = (torch.rand((B, N), generator=g, device="cuda") < 3.0 / N).cumsum(1)
        real = torch.arange(N, device="cuda") < torch.randint(N * 3 // 4, N + 1, (B, 1), generator=g, device="cuda")
        keep = (doc[:, :, None] == doc[:, None, :]) & real[:, None, :] & (torch.rand((B, N, N), generator=g, device="cuda") < 0.95)
        s["mask_values"] = keep.to(torch.float32)
    return s


def run(s):
    stream = torch.cuda.current_stream().cuda_stream
    code, B, H, H_kv, d, scale = s["code"], s["B"], s["H"], s["H_kv"], s["d"], s["scale"]
    q, out = s["q"].data_ptr(), s["out"].data_ptr()
    if s["path"] == "decode":
        kp, vp, table = s["k_pool"].data_ptr(), s["v_pool"].data_ptr(), s["table"].data_ptr()
        hip.kv_scatter(s["k_new"].data_ptr(), s["v_new"].data_ptr(), code, kp, vp, code, table, s["max_pages"], B, H_kv, d, _PAGE,
                       token_row=s["rows"].data_ptr(), token_pos=s["at"].data_ptr(), stream=stream)
        hip.paged_decode_gqa(q, out, code, kp, vp, code, table, s["lens"].data_ptr(), None, B, H, H_kv, d, _PAGE, s["max_pages"],
                             s["max_len"], scale, 0, s["ws"].data_ptr(), s["ws_bytes"], stream)
        return s["out"], s["k_pool"], s["v_pool"]
    k, v = s["k"].data_ptr(), s["v"].data_ptr()
    st, kst = s["strides"], s["kv_strides"]
    if s["path"] == "serve":
        hip.flash_fwd_varlen_gqa(q, k, v, out, code, s["cu"].data_ptr(), B, s["max_len"], H, H_kv, d, *st, *kst, scale, True, stream)
        hip.kv_scatter_batch(k, v, code, 0, H_kv * d, s["k_pool"].data_ptr(), s["v_pool"].data_ptr(), code, s["table"].data_ptr(),
                             s["max_pages"], s["rows"].data_ptr(), B, s["max_len"], H_kv, d, _PAGE, cu_seqlens=s["cu"].data_ptr(),
                             stream=stream)
        return s["out"], s["k_pool"], s["v_pool"]
    causal = s["causal"]
    if s["path"] == "prefill":
        mask = s["mask_values"].data_ptr() if s["mask"] else None
        hip.flash_fwd_gqa(q, k, v, out, code, B, s["N"], H, H_kv, d, st, kst, scale, causal, stream, mask)
        return s["out"]
    d_out, d_q, d_k, d_v, ws = (s[x].data_ptr() for x in ("d_out", "d_q", "d_k", "d_v", "ws"))
    if "cu" in s:
        cu = s["cu"].data_ptr()
        hip.flash_fwd_varlen_gqa(q, k, v, out, code, cu, B, s["max_len"], H, H_kv, d, *st, *kst, scale, causal, stream)
        hip.flash_bwd_varlen(d_out, q, k, v, d_q, d_k, d_v, code, cu, B, s["max_len"], H, H_kv, d, *st, *kst, scale, causal, ws,
                             s["ws_bytes"], stream)
    else:
        N, stats = s["N"], s["stats"].data_ptr()
        if hip.flash_fwd_keep(q, k, v, out, code, B, N, H, H_kv, d, st, kst, scale, causal, stats, stream):
            hip.flash_bwd_kept(d_out, q, k, v, out, stats, d_q, d_k, d_v, code, B, N, H, H_kv, d, st, kst, scale, causal, ws,
                               s["ws_bytes"], stream)
        else:
            hip.flash_bwd(d_out, q, k, v, d_q, d_k, d_v, code, B, N, H, H_kv, d, st, kst, scale, causal, ws, s["ws_bytes"], stream)
    return s["out"], s["d_q"], s["d_k"], s["d_v"]
