"""The workloads that this library's performance is followed on: what a program that trains or serves with its kernels
has them do, through the public entry points, from the calls that are over in a few launches to the ones that fill the
chip for a tenth of a millisecond.

``listed()`` names the fixed cases, ``draw(rng)`` gives further sizes of the same ranges, ``prepare`` makes the inputs on
the GPU, ``run`` is one pass, ``work`` the bytes and operations the pass cannot do without, ``tolerance`` how far two
correct implementations may be apart.
"""
from __future__ import annotations

import math

import torch

from __graft_entry__ import load_package

ct = load_package()
from cutile_jl_amd.examples import fmha, moe, softmax  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "e4m3": 1}


def listed():
    return [
        # The layernorm example's own largest size: forward and backward of one layer of a small model.  Four launches of a
        # few microseconds, so what counts is what a launch costs.
        dict(name="layernorm_1024", op="layernorm", M=1024, N=1024, groups=64),
        # The training step of the norm benchmark: 4096 rows of 4096, everything has to come from memory.
        dict(name="layernorm_4096", op="layernorm", M=4096, N=4096, groups=64),
        # Softmax over the logits of 1024 tokens and a vocabulary that is no multiple of anything.
        dict(name="softmax_vocabulary", op="softmax", M=1024, N=50257, dtype="bf16"),
        # The dense GEMM benchmark: f16 operands, fp32 result.
        dict(name="matmul_4096", op="matmul", M=4096, N=4096, K=4096, dtype="f16", out="f32"),
        # A product of ordinary, ragged size: none of the three extents fits a tile or a 16-byte vector.
        dict(name="matmul_ragged", op="matmul", M=2999, N=2100, K=3001, dtype="bf16", out="bf16"),
        # The batched GEMM benchmark in full fp32.
        dict(name="batchmatmul_f32", op="batchmatmul", batch=8, M=1024, N=2048, K=512, dtype="f32"),
        # Attention over a prompt, the attention benchmark: 16 heads of 64, causal.
        dict(name="attention_d64", op="attention", batch=8, heads=16, kv_heads=16, sq=1024, skv=1024, dim=64, causal=True, dtype="f16"),
        # Attention over a prompt as grouped-query models have it: heads of 128, four query heads to a key head, a prompt
        # length that is not a multiple of a tile.
        dict(name="attention_d128_grouped", op="attention", batch=2, heads=32, kv_heads=8, sq=2000, skv=2000, dim=128, causal=True, dtype="bf16"),
        # One new token per sequence against the cached keys of a serving batch.
        dict(name="attention_decode", op="attention", batch=16, heads=32, kv_heads=8, sq=1, skv=4000, dim=128, causal=True, dtype="bf16"),
        # The MoE benchmark: 256 tokens in flight, top-2 of 32 experts, every expert's weights are read.
        dict(name="moe_256", op="moe", tokens=256, hidden=1024, experts=32, inter=2048, topk=2, dtype="f16", weights="f16"),
        # The same layer with e4m3 weights and per-channel scales.
        dict(name="moe_256_e4m3", op="moe", tokens=256, hidden=1024, experts=32, inter=2048, topk=2, dtype="f16", weights="e4m3"),
        # The same layer over a prompt of 4096 tokens: the matrix cores count, not the weights.
        dict(name="moe_prefill", op="moe", tokens=4096, hidden=1024, experts=32, inter=2048, topk=2, dtype="f16", weights="f16"),
    ]


def _log(rng, lo, hi, step=1):
    """A size between lo and hi, uniform in its logarithm; one in three is left as it falls, the rest are multiples of step."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 1 / 3:
        return min(hi, n | 1)
    return min(hi, max(lo, n // step * step))


def draw(rng):
    op = rng.choice(["layernorm", "softmax", "matmul", "matmul", "batchmatmul", "prompt", "prompt", "decode", "moe", "moe"])
    if op == "layernorm":
        N = _log(rng, 256, 8192, 64)
        return dict(op=op, M=_log(rng, 256, min(8192, (1 << 24) // N)), N=N, groups=64)
    if op == "softmax":
        dtype = rng.choice(["f32", "f16", "bf16"])
        N = _log(rng, 512, 60000, 64)
        return dict(op=op, M=_log(rng, 64, min(8192, (1 << 26) // (N * BYTES[dtype] // 2))), N=N, dtype=dtype)
    if op == "matmul":
        dtype = rng.choice(["f16", "bf16"])
        return dict(op=op, M=_log(rng, 256, 4096, 64), N=_log(rng, 256, 4096, 64), K=_log(rng, 256, 4096, 64), dtype=dtype,
                    out=rng.choice([dtype, "f32"]))
    if op == "batchmatmul":
        return dict(op=op, batch=rng.randint(2, 12), M=_log(rng, 128, 1024, 64), N=_log(rng, 128, 2048, 64), K=_log(rng, 128, 512, 32), dtype="f32")
    if op == "prompt":
        dim, group = rng.choice([64, 128]), rng.choice([1, 4])
        kv_heads, S = rng.choice([4, 8]), _log(rng, 256, 4096, 64)
        per = 4 * kv_heads * group * S * S * dim
        batch = max(1, min(rng.randint(1, 8), int(9e10 // per)))
        return dict(op="attention", batch=batch, heads=kv_heads * group, kv_heads=kv_heads, sq=S, skv=S, dim=dim, causal=rng.random() < 0.75,
                    dtype=rng.choice(["f16", "bf16"]))
    if op == "decode":
        dim, group = rng.choice([64, 128]), rng.choice([1, 4, 8])
        kv_heads, S = rng.choice([4, 8, 16]), _log(rng, 512, 16384, 64)
        per = 4 * kv_heads * S * dim
        batch = max(1, min(rng.randint(1, 32), int(4e8 // per)))
        return dict(op="attention", batch=batch, heads=kv_heads * group, kv_heads=kv_heads, sq=1, skv=S, dim=dim, causal=True,
                    dtype=rng.choice(["f16", "bf16"]))
    topk = rng.choice([1, 2, 2, 4, 8])
    return dict(op="moe", tokens=_log(rng, 16, 8192 // topk, 16), hidden=rng.choice([512, 1024]), experts=rng.choice([8, 16, 32, 64]),
                inter=rng.choice([512, 1024, 1408, 2048]), topk=topk, dtype=rng.choice(["f16", "bf16"]), weights=rng.choice(["same", "same", "e4m3"]))


def _weights_type(c):
    return c["dtype"] if c["weights"] == "same" else c["weights"]


def prepare(case, seed):
    c = dict(case)
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, dtype=torch.float32, std=1.0, mean=0.0):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=g)

    def empty(*shape, dtype=torch.float32):
        return torch.empty(shape, dtype=dtype, device="cuda")

    op = c["op"]
    if op == "layernorm":
        M, N, G = c["M"], c["N"], c["groups"]
        return dict(c, X=normal(M, N), W=normal(N, std=0.1, mean=1.0), B=normal(N, std=0.1), DY=normal(M, N), Y=empty(M, N), DX=empty(M, N),
                    Mean=empty(M), Rstd=empty(M), partials=empty(2, G, N), dW=empty(N), dB=empty(N),
                    Locks=torch.zeros(G, dtype=torch.int64, device="cuda"))
    if op == "softmax":
        x = normal(c["M"], c["N"], dtype=DTYPES[c["dtype"]], std=2.0)
        return dict(c, x=x, y=torch.empty_like(x), tile=softmax.next_power_of_2(c["N"]))
    if op in ("matmul", "batchmatmul"):
        T = DTYPES[c["dtype"]]
        lead = (c["batch"],) if op == "batchmatmul" else ()
        # a Julia (M, K) array is a torch (K, M) tensor
        if op == "matmul":
            A, B = normal(c["K"], c["M"], dtype=T, std=0.125), normal(c["N"], c["K"], dtype=T, std=0.125)
        else:
            A, B = (empty(*lead, p, q, dtype=T).uniform_(-1, 1, generator=g) for p, q in ((c["K"], c["M"]), (c["N"], c["K"])))
        return dict(c, A=A, B=B, C=empty(*lead, c["N"], c["M"], dtype=DTYPES[c.get("out", c["dtype"])]))
    if op == "attention":
        T = DTYPES[c["dtype"]]
        kv = (c["batch"], c["kv_heads"], c["skv"], c["dim"])
        return dict(c, Q=normal(c["batch"], c["heads"], c["sq"], c["dim"], dtype=T), K=normal(*kv, dtype=T), V=normal(*kv, dtype=T))
    T, E, H, I, k = DTYPES[c["dtype"]], c["experts"], c["hidden"], c["inter"], c["topk"]
    logits = normal(c["tokens"], E)
    top = torch.topk(logits, k, dim=1)
    weights = dict(w1=normal(E, 2 * I, H, dtype=T, std=0.02), w2=normal(E, H, I, dtype=T, std=0.02), w1_scale=None, w2_scale=None)
    if _weights_type(c) == "e4m3":
        weights = vars(moe.quantize_weights(moe.namespace(w1=weights["w1"], w2=weights["w2"])))
    return dict(c, x=normal(c["tokens"], H, dtype=T), topk_ids=(top.indices + 1).t().contiguous(),
                topk_weights=torch.softmax(top.values, dim=1).to(T).t().contiguous(), **weights)


def run(state):
    s = state
    op = s["op"]
    if op == "layernorm":
        # forward, then the backward as the example runs it: zero-filled partial sums, dX with the partials, the final sums
        ct.layer_norm_fwd(s["X"], s["W"], s["B"], s["Y"], s["Mean"], s["Rstd"], 1e-5, 1024)
        s["partials"].zero_()
        dw, db = s["partials"]
        ct.layer_norm_bwd_dx_partial_dwdb(s["DX"], s["DY"], dw, db, s["X"], s["W"], s["Mean"], s["Rstd"], s["Locks"], s["groups"], 1024)
        ct.layer_norm_bwd_dwdb(dw, db, s["dW"], s["dB"], 32, 1024)
        return dict(y=s["Y"], mean=s["Mean"], rstd=s["Rstd"], dx=s["DX"], dw=s["dW"], db=s["dB"])
    if op == "softmax":
        ct.softmax_tma_kernel(s["y"], s["x"], s["tile"], num_programs=s["M"])
        return s["y"]
    if op == "matmul":
        ct.matmul_kernel(s["A"], s["B"], s["C"], 64, 64, 64)
        return s["C"]
    if op == "batchmatmul":
        ct.batch_matmul_kernel(s["A"], s["B"], s["C"], 64, 64, 64)
        return s["C"]
    if op == "attention":
        return fmha.cutile_fmha(s["Q"], s["K"], s["V"], input_pos=s["skv"] - s["sq"], query_group_size=s["heads"] // s["kv_heads"], causal=s["causal"])
    return moe.cutile_moe(s["x"], s["w1"], s["w2"], s["topk_weights"], s["topk_ids"], 128, 128, 64, w1_scale=s["w1_scale"], w2_scale=s["w2_scale"])


def work(case):
    c = case
    op = c["op"]
    if op == "layernorm":
        # forward: X in, Y out; backward: X and dY in, dX out; W twice, B, Mean, Rstd out and in; dW, dB out
        return dict(bytes=4 * (5 * c["M"] * c["N"] + 5 * c["N"] + 4 * c["M"]), flops=20 * c["M"] * c["N"])
    if op == "softmax":
        return dict(bytes=2 * c["M"] * c["N"] * BYTES[c["dtype"]], flops=4 * c["M"] * c["N"])
    if op in ("matmul", "batchmatmul"):
        n, M, N, K = c.get("batch", 1), c["M"], c["N"], c["K"]
        b = BYTES[c["dtype"]]
        return dict(bytes=n * (b * (M * K + K * N) + BYTES[c.get("out", c["dtype"])] * M * N), flops=2 * n * M * N * K)
    if op == "attention":
        sq, skv = c["sq"], c["skv"]
        pairs = sq * skv - sq * (sq - 1) // 2 if c["causal"] else sq * skv   # the queries are the last sq positions
        return dict(bytes=2 * c["batch"] * c["dim"] * 2 * (c["heads"] * sq + c["kv_heads"] * skv), flops=4 * c["batch"] * c["heads"] * c["dim"] * pairs)
    hit = c["experts"] * (1 - (1 - c["topk"] / c["experts"]) ** c["tokens"])      # experts that some token is sent to, on average
    matrices = hit * 3 * c["hidden"] * c["inter"] * BYTES[_weights_type(c)]
    if _weights_type(c) == "e4m3":
        matrices += hit * 4 * (2 * c["inter"] + c["hidden"])
    return dict(bytes=matrices + 2 * 2 * c["tokens"] * c["hidden"] + 10 * c["tokens"] * c["topk"],
                flops=6 * c["tokens"] * c["topk"] * c["hidden"] * c["inter"])


def tolerance(case):
    # Four times what the outputs of these cases and of two dozen drawn ones were seen to be off the same formulas in
    # float64 (f16 results of softmax and matmul: an eighth of the bf16 ones, by the three more bits of the type).
    op = case["op"]
    if op == "layernorm":
        return dict(rel=6e-7, max=2.5e-6)
    if op == "softmax":
        return dict(rel=dict(f32=4e-7, f16=9e-4, bf16=7e-3)[case["dtype"]], max=dict(f32=4e-6, f16=2e-3, bf16=1.6e-2)[case["dtype"]])
    if op == "matmul":
        return dict(rel=dict(f32=1.6e-6, f16=9e-4, bf16=7e-3)[case["out"]], max=dict(f32=1.5e-5, f16=2e-3, bf16=1.6e-2)[case["out"]])
    if op == "batchmatmul":
        return dict(rel=1.6e-6, max=1.5e-5)
    if op == "attention":
        return dict(rel=dict(f16=1.4e-3, bf16=1.2e-2)[case["dtype"]], max=dict(f16=4e-2, bf16=1.2e-1)[case["dtype"]])
    return dict(rel=dict(f16=2e-3, bf16=1.5e-2)[case["dtype"]], max=dict(f16=1e-2, bf16=7e-2)[case["dtype"]])
