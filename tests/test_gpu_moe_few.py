"""The grouped GEMM for few tokens per expert, whose waves split K (csrc/moe_few.hip): stand-in for the reference's
examples/moe.jl:45-105."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cutile_jl_amd.examples import moe
from test_gpu_moe import _every_path, _routed, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("make", [
    # replicas per expert on the edges of the 32-slot tiles, none, and a second tile; K of four stages, and part-filled last ones; N off the strips
    lambda: _routed([1, 31, 32, 33, 0, 7, 64, 16], hidden_size=256, intermediate_size=272),
    lambda: _routed([3, 0, 40, 20], topk=1, hidden_size=272, intermediate_size=400, T=torch.bfloat16),
    lambda: _routed([9, 11, 2, 10], topk=2, hidden_size=1008, intermediate_size=304, T=torch.bfloat16),
    lambda: _routed([70, 50, 33, 47], topk=2, hidden_size=512, intermediate_size=256),                        # more than 32 per expert
    lambda: moe.prepare(num_tokens=16, hidden_size=512, num_experts=8, intermediate_size=512, topk=8),
    lambda: moe.prepare(num_tokens=1, hidden_size=1024, num_experts=16, intermediate_size=1024, topk=2),
], ids=["edges", "small", "ragged", "two_tiles", "top8", "one_token"])
def test_few_tokens_per_expert(ct, orc, make, e4m3):
    """Every launch sequence gives the same bits, blocks of 32, 64 and 128 slots too; the float64 oracle on the (dequantised) weights."""
    d = make()
    J = orc.to_julia
    w1d, w2d, kw = J(d.w1), J(d.w2), {}
    if e4m3:
        q = moe.quantize_weights(d)
        d.w1, d.w2 = q.w1, q.w2
        kw = dict(w1_scale=q.w1_scale, w2_scale=q.w2_scale)
        w1d = orc.e4m3fn_decode(J(q.w1.view(torch.uint8))) * J(q.w1_scale)[None]
        w2d = orc.e4m3fn_decode(J(q.w2.view(torch.uint8))) * J(q.w2_scale)[None]
    outs = {}
    for tile_m in (128, 64, 32):
        for k, v in _every_path(d, tile_m, **kw).items():
            outs[k, tile_m] = v
    c = torch.full((d.num_tokens * d.topk, 2 * d.intermediate_size + 4), float("nan"), dtype=d.hidden_states.dtype, device="cuda")[:, :2 * d.intermediate_size]
    tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 32, d.num_experts)
    moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c, d.topk_weights, tok, exp, mul_routed_weight=True, num_token_replicas=d.topk,
                                tile_m=32, tile_n=128, tile_k=64, **({"b_scale": kw["w1_scale"]} if e4m3 else {}))
    assert ct.last_variant() == "fused_moe_few_t32_n64_k64_ksplit4" + ("_w8a16" if e4m3 else ""), ct.last_variant()
    assert not torch.isnan(c.float()).any()
    want = outs["separate", 128]
    for k, v in outs.items():
        assert torch.equal(v, want), k
    ref = orc.ref_moe(J(d.hidden_states), w1d, w2d, J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(want), ref, 5e-2 if d.hidden_states.dtype == torch.bfloat16 else 2e-2)


@pytest.mark.parametrize("K,N,routed,few", [
    (256, 20480, True, True), (256, 20544, True, False), (2048, 16320, True, True), (2048, 16384, True, False), (2064, 16384, True, True),
    (4096, 8128, True, True), (4096, 8192, True, False), (4096, 1024, True, True), (512, 8192, False, True), (4096, 7680, False, True), (4096, 8192, False, False),
])
def test_which_launches_of_e4m3_weights_the_rule_takes(ct, orc, K, N, routed, few):
    """Rows of 2 KB below 1024 workgroups, unless the other kernel has no 64-channel strips for their K; of 4 KB below 512; 1280 at most."""
    E, tokens = 4, 16
    rng = np.random.default_rng(K + N)
    tok, exp = orc.moe_align_tile_size(np.arange(tokens, dtype=np.int64)[:, None] % E + 1, 32, E)
    A = torch.from_numpy(rng.integers(-2, 3, (tokens, K)).astype(np.float16)).cuda()
    W = torch.randint(-1, 2, (E, N, K), dtype=torch.int8, generator=torch.Generator().manual_seed(K)).cuda().half()
    C = torch.empty(tokens, N, dtype=torch.float16, device="cuda")
    ct.fused_moe_kernel(A, W.to(torch.float8_e4m3fn), C, torch.ones(tokens, dtype=torch.float16, device="cuda"), torch.from_numpy(tok).cuda(),
                        torch.from_numpy(exp).cuda(), 1, routed, 32, 128, 64, b_scale=torch.ones(E, N, device="cuda"))
    assert ct.last_variant().startswith("fused_moe_few_") == few, ct.last_variant()
    # (integers below 2^11, so f16 holds them and fp32 sums are exact)
    assert torch.equal(C.float(), torch.stack([W[t % E].float() @ A[t].float() for t in range(tokens)]))


@pytest.mark.parametrize("tokens,E,K,N,off,routed,few", [
    (31, 1, 256, 256, 0, False, True), (16, 4, 256, 7680, 0, False, True), (16, 4, 256, 7744, 0, False, False),    # first projection: 480 workgroups
    (16, 4, 256, 8256, 0, True, True), (16, 4, 2048, 8192, 0, True, False), (16, 4, 2040, 8192, 0, True, True),    # second: rows of 4 KB from 512 on
    (16, 4, 2048, 8064, 0, True, True),
    (16, 4, 2048, 3008, 0, True, False), (16, 4, 2048, 3072, 0, True, True),                                        # and from 192 on
    (16, 4, 4096, 3072, 0, True, False), (16, 4, 4088, 3072, 0, True, True),                                        # of 8 KB never
    (16, 4, 256, 20480, 0, True, True), (16, 4, 256, 20544, 0, True, False),                                        # 1280 workgroups
    (128, 4, 2048, 3392, 0, False, True), (128, 4, 2048, 3456, 0, False, False),                                    # 32 per expert, rows of 4 KB: 320
    (128, 4, 512, 3712, 0, False, True), (128, 4, 512, 3776, 0, False, False), (128, 4, 512, 3776, 0, True, False),  # 32 per expert: 352 workgroups
    (16, 4, 248, 256, 0, False, False), (16, 4, 260, 256, 0, False, False), (16, 4, 256, 256, 4, False, False),    # K below 256, off the chunks; rows off 16 bytes
])
def test_which_launches_the_rule_takes(ct, orc, tokens, E, K, N, off, routed, few):
    """Both sides compute the same exact integers."""
    rng = np.random.default_rng(K + tokens + N)
    tok, exp = orc.moe_align_tile_size(np.arange(tokens, dtype=np.int64)[:, None] % E + 1, 32, E)
    A = torch.from_numpy(rng.integers(-2, 3, (tokens, K)).astype(np.float16)).cuda()
    W = torch.from_numpy(rng.integers(-1, 2, (E, N, K)).astype(np.float16))
    flat = torch.zeros(E * N * K + 16, dtype=torch.float16, device="cuda")
    B = flat[off:off + E * N * K].view(E, N, K)
    B.copy_(W)
    C = torch.empty(tokens, N, dtype=torch.float16, device="cuda")
    ct.fused_moe_kernel(A, B, C, torch.ones(tokens, dtype=torch.float16, device="cuda"), torch.from_numpy(tok).cuda(), torch.from_numpy(exp).cuda(),
                        1, routed, 32, 128, 64)
    assert ct.last_variant().startswith("fused_moe_few_") == few, ct.last_variant()
    ref = np.stack([W[t % E].float().numpy() @ A[t].float().cpu().numpy() for t in range(tokens)])
    assert np.array_equal(C.float().cpu().numpy(), ref)


def _exact(orc, tokens, topk, E, K, N, T, e4m3, seed=0):
    """Small integers, so every product below is exact: (A, B, b_scale, tok, exp, weights (tokens, topk), result before the weights)."""
    rng = np.random.default_rng(seed + K + N)
    A = rng.integers(-2, 3, (tokens, K)).astype(np.float32); W = rng.integers(-1, 2, (E, N, K)).astype(np.float32)
    ids = np.stack([rng.permutation(E)[:topk] + 1 for _ in range(tokens)]).astype(np.int64)
    tok, exp = orc.moe_align_tile_size(ids, 32, E)
    scale = 2.0 ** rng.integers(-1, 2, (E, N))
    ref = np.stack([W[e - 1] @ A[t] * (scale[e - 1] if e4m3 else 1) for t in range(tokens) for e in ids[t]])
    weights = (2.0 ** rng.integers(-1, 2, (tokens, topk))).astype(np.float32)
    cuda = lambda x, t: torch.from_numpy(np.ascontiguousarray(x)).to(t).cuda()
    return (cuda(A, T), cuda(W, torch.float8_e4m3fn if e4m3 else T), cuda(scale, torch.float32) if e4m3 else None, cuda(tok, torch.int32),
            cuda(exp, torch.int32), cuda(weights.T, T), weights, ref)


@pytest.mark.parametrize("T", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("N,pad,off", [(258, 0, 0), (257, 0, 0), (321, 7, 0), (256, 2, 0), (256, 4, 2), (260, 4, 4), (259, 5, 1), (63, 1, 3)])
def test_results_off_the_stores_of_four(ct, orc, N, pad, off, e4m3, T):
    """N, a leading dimension and a start of C that are no multiples of four: the stores go element by element, and nothing around them
    is touched."""
    A, B, scale, tok, exp, w2d, weights, ref = _exact(orc, 13, 2, 4, 272, N, T, e4m3)
    flat = torch.full((off + 26 * (N + pad) + 16,), 99.0, dtype=T, device="cuda")
    C = flat[off:off + 26 * (N + pad)].view(26, N + pad)[:, :N]
    for mul in (False, True):
        flat.fill_(99.0)
        ct.fused_moe_kernel(A, B, C, w2d, tok, exp, 2, mul, 32, 128, 64, b_scale=scale)
        assert ct.last_variant().startswith("fused_moe_few_t32"), ct.last_variant()
        want = ref * weights.reshape(-1, 1) if mul else ref
        # (integers up to 2^11 and a power of two are exact in f16; those beyond 2^8 in bf16 are rounded to nearest)
        assert torch.equal(C.cpu(), torch.from_numpy(want).to(T))
        assert flat.ne(99.0).sum().item() <= 26 * N and bool((flat[:off] == 99.0).all()) and bool((flat[off + 26 * (N + pad):] == 99.0).all())
        assert pad == 0 or bool((flat[off:off + 26 * (N + pad)].view(26, N + pad)[:, N:] == 99.0).all())


@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("half", [129, 130, 31, 128])
def test_silu_results_off_the_stores_of_four(ct, orc, half, e4m3):
    """The epilogue against the projection and silu_and_mul_kernel one after the other, bit for bit."""
    A, B, scale, tok, exp, w2d, weights, ref = _exact(orc, 13, 2, 4, 272, 2 * half, torch.float16, e4m3)
    A = A * 0.0625
    flat = torch.full((26 * (half + 1) + 8,), 99.0, dtype=torch.float16, device="cuda")
    C = flat[:26 * (half + 1)].view(26, half + 1)[:, :half]
    ct.fused_moe_silu_kernel(A, B, C, w2d, tok, exp, 2, False, 32, 128, 64, b_scale=scale)
    assert ct.last_variant().startswith("fused_moe_few_silu"), ct.last_variant()
    both = torch.empty(26, 2 * half, dtype=torch.float16, device="cuda"); want = torch.empty(26, half, dtype=torch.float16, device="cuda")
    ct.fused_moe_kernel(A, B, both, w2d, tok, exp, 2, False, 32, 128, 64, b_scale=scale)
    ct.silu_and_mul_kernel(both[:, :half], both[:, half:], want, 256)
    assert torch.equal(C, want) and bool((flat[:26 * (half + 1)].view(26, half + 1)[:, half:] == 99.0).all()) and bool((flat[26 * (half + 1):] == 99.0).all())


@pytest.mark.parametrize("form", ["plain", "silu", "accumulate"])
@pytest.mark.parametrize("bad", [0, 5, -3, 2**30])
def test_experts_out_of_range_and_slots_without_a_token(ct, orc, form, bad):
    """A block of an expert that does not exist writes nothing, neither does a slot whose token does not exist, and the routed weights may
    be a strided view."""
    N = 264
    A, B, _, tok, exp, w2d, weights, ref = _exact(orc, 13, 2, 4, 272, N, torch.float16, False)
    total, exp, tok = 26, exp.clone(), tok.clone()
    first = tok[:32].clone()
    exp[0] = bad                                                             # the first expert's tokens
    second = tok[32:64]; live = int((second <= total).sum())
    dropped = int(second[live - 1]); second[live - 1] = -7                     # and the last of the second's
    lost = sorted({int(t) - 1 for t in first if 1 <= int(t) <= total} | {dropped - 1})
    keep = [f for f in range(total) if f not in lost]
    wide = torch.full((3, 2 * 13 + 3), float("nan"), dtype=torch.float16, device="cuda")
    view = wide[:2, 1:27:2]; view.copy_(w2d)
    if form == "accumulate":
        # (one replica per column of A: the second projection's input)
        A2 = A.repeat_interleave(2, 0).contiguous()
        out = torch.zeros(13, N, dtype=torch.float16, device="cuda")
        ct.fused_moe_accumulate_kernel(A2, B, out, view, tok, exp, 32, 128, 64)
        want = ref * weights.reshape(-1, 1); want[lost] = 0
        assert ct.last_variant().startswith("fused_moe_few_acc"), ct.last_variant()
        assert torch.equal(out.cpu(), torch.from_numpy(want.reshape(13, 2, N).sum(1)).half())
        return
    n = N // 2 if form == "silu" else N
    C = torch.full((total, n), 99.0, dtype=torch.float16, device="cuda")
    launch = ct.fused_moe_silu_kernel if form == "silu" else ct.fused_moe_kernel
    launch(A * 0.0625 if form == "silu" else A, B, C, view, tok, exp, 2, form == "plain", 32, 128, 64)
    assert ct.last_variant().startswith("fused_moe_few_"), ct.last_variant()
    assert bool((C[lost] == 99.0).all()) and not bool((C[keep] == 99.0).all(1).any())
    if form == "plain":
        assert torch.equal(C[keep].cpu(), torch.from_numpy((ref * weights.reshape(-1, 1))[keep]).half())


@pytest.mark.parametrize("switch,value", [("MI_MOE_DENSE_J", "2"), ("MI_MOE_DENSE_J", "4"), ("MI_MOE_DENSE_WIDE", "0"), ("MI_MOE_DENSE_STREAM", "0"),
                                          ("MI_MOE_DENSE", "0"), ("MI_MOE_PREFILL", "0")])
def test_a_forced_kernel_is_forced(ct, orc, monkeypatch, switch, value):
    """The settings that force a kernel, or a shape of one, leave no launch to this one."""
    A, B, _, tok, exp, w2d, weights, ref = _exact(orc, 64, 2, 4, 512, 256, torch.float16, False)
    tok, exp = (x.cuda() for x in map(torch.from_numpy, orc.moe_align_tile_size(np.stack([[t % 4 + 1, (t + 1) % 4 + 1] for t in range(64)]).astype(np.int64), 128, 4)))
    C = torch.empty(128, 256, dtype=torch.float16, device="cuda")
    run = lambda: ct.fused_moe_kernel(A, B, C, w2d, tok, exp, 2, False, 128, 128, 64) or ct.last_variant()
    assert run().startswith("fused_moe_few_")
    want = C.clone()
    monkeypatch.setenv(switch, value)
    name = run()
    assert name.startswith("fused_moe_t64_" if switch == "MI_MOE_DENSE" else "fused_moe_dense_"), name
    assert torch.equal(C, want)
