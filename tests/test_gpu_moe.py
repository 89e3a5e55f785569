"""GPU parity tests for the MoE kernels through the C ABI.

Oracle: numpy restatement of ``ref_moe`` (examples/moe.jl:264-304) in float64, plus per-kernel
checks of the grouped GEMM, SiLU*mul and the top-k sum.  Shapes: the reference example's
``main()`` list (moe.jl:402-410), the measured top-2 configuration at reduced width, expert
counts that are not multiples of the tile (sentinel padding), and FP8-E4M3 weights.

Tolerance: |err| <= 2e-2 * (|ref| + max|ref|), and the reference's
``isapprox(rtol=1e-2, atol=1e-2)`` (moe.jl:370-374).  The f16 result is rounded to f16 three
times on the way (cache1, cache2, cache3) exactly as in the reference.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from cutile_jl_amd.examples import moe  # noqa: E402


def check(got, ref, tol=2e-2):
    got = np.asarray(got, dtype=np.float64)
    err = np.abs(got - ref)
    bound = tol * (np.abs(ref) + np.abs(ref).max())
    assert np.all(err <= bound), f"max err {err.max():.3e}, worst ratio {np.max(err / bound):.3f}"


class _dense_knob:
    """MI_MOE_DENSE=0 keeps every launch on the streaming kernels, =1 sends every launch the ring kernel can take to it
    (the library reads the variable at every call)."""
    def __init__(self, value):
        self.value = value

    def __enter__(self):
        import os
        self.old = os.environ.get("MI_MOE_DENSE")
        os.environ["MI_MOE_DENSE"] = self.value

    def __exit__(self, *exc):
        import os
        if self.old is None:
            os.environ.pop("MI_MOE_DENSE", None)
        else:
            os.environ["MI_MOE_DENSE"] = self.old


@pytest.mark.parametrize("tokens,hidden,experts,inter,topk,router", [
    (48, 512, 64, 1024, 8, "randperm"), (128, 512, 32, 1024, 4, "randperm"), (64, 1024, 64, 2048, 8, "randperm"),
    (256, 512, 32, 512, 2, "top2_logits"), (7, 256, 3, 128, 2, "randperm"), (300, 256, 2, 256, 2, "randperm"),
    (1, 128, 4, 64, 1, "randperm"), (96, 256, 256, 128, 8, "randperm"), (33, 128, 160, 64, 6, "randperm"),
])
def test_moe_end_to_end(orc, tokens, hidden, experts, inter, topk, router):
    d = moe.prepare(num_tokens=tokens, hidden_size=hidden, num_experts=experts, intermediate_size=inter, topk=topk,
                    router=router)
    r = moe.run(d)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(r.out), ref)
    assert orc.isapprox(J(r.out).astype(np.float64), ref, rtol=1e-2, atol=1e-2)


def test_moe_bf16(orc):
    d = moe.prepare(num_tokens=64, hidden_size=256, num_experts=8, intermediate_size=256, topk=2, T=torch.bfloat16)
    r = moe.run(d)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(r.out), ref, 5e-2)


def test_fused_moe_kernel_alone_with_sentinels(ct, orc):
    """One grouped GEMM against per-slot dot products; checks the replica -> token mapping
    (cld(token_id, replicas)), the routed-weight scaling, that sentinel slots write nothing
    and that untouched columns of C keep their contents."""
    rng = np.random.default_rng(0)
    K, N, E, tokens, topk, tile_m = 192, 160, 5, 9, 3, 16
    A = rng.standard_normal((K, tokens)).astype(np.float16)
    B = (rng.standard_normal((K, N, E)) * 0.1).astype(np.float16)
    ids = np.stack([rng.permutation(E)[:topk] + 1 for _ in range(tokens)]).astype(np.int64)
    w = rng.random((tokens, topk)).astype(np.float16)
    tok, exp = orc.moe_align_tile_size(ids, tile_m, E)
    total = tokens * topk
    dev = "cuda"
    C = torch.full((total + 2, N), 9.0, dtype=torch.float16, device=dev)  # two spare columns
    wflat = torch.from_numpy(w.reshape(-1)).to(dev)
    for mul in (False, True):
        C.fill_(9.0)
        ct.fused_moe_kernel(orc.from_julia(A).to(dev), orc.from_julia(B).to(dev), C[:total], wflat,
                            torch.from_numpy(tok).to(dev), torch.from_numpy(exp).to(dev), topk, mul, tile_m, 128, 64)
        got = orc.to_julia(C).astype(np.float64)
        flat_e = ids.reshape(-1)
        ref = np.zeros((N, total))
        for f in range(total):
            t = f // topk
            ref[:, f] = B[:, :, flat_e[f] - 1].astype(np.float64).T @ A[:, t].astype(np.float64)
            if mul:
                ref[:, f] *= float(w.reshape(-1)[f])
        check(got[:, :total], ref, 2e-2)
        assert np.all(got[:, total:] == 9.0)
    # The routed weights as the (num_tokens, topk) matrix itself, dense and as a strided view, instead of its
    # slot-fastest flattening (moe.jl:193): the kernel looks (token, slot) up, the result is the same bit for bit.
    flat_result = C.clone()
    w2d = torch.from_numpy(np.ascontiguousarray(w.T)).to(dev)                         # torch (topk, tokens)
    wide = torch.full((topk + 1, 2 * tokens + 3), float("nan"), dtype=torch.float16, device=dev)
    wide[:topk, 1:2 * tokens + 1:2] = w2d
    for wv in (w2d, wide[:topk, 1:2 * tokens + 1:2]):
        C.fill_(9.0)
        ct.fused_moe_kernel(orc.from_julia(A).to(dev), orc.from_julia(B).to(dev), C[:total], wv,
                            torch.from_numpy(tok).to(dev), torch.from_numpy(exp).to(dev), topk, True, tile_m, 128, 64)
        assert torch.equal(C, flat_result)
    with pytest.raises(ct.MiError):                                                  # a matrix of the wrong extent
        ct.fused_moe_kernel(orc.from_julia(A).to(dev), orc.from_julia(B).to(dev), C[:total], w2d[:, :tokens - 1],
                            torch.from_numpy(tok).to(dev), torch.from_numpy(exp).to(dev), topk, True, tile_m, 128, 64)


def test_silu_and_mul_and_topk_sum(ct, orc):
    rng = np.random.default_rng(1)
    inter, total = 300, 37
    AB = torch.from_numpy((rng.standard_normal((total, 2 * inter)) * 3).astype(np.float16)).cuda()
    C = torch.zeros((total, inter), dtype=torch.float16, device="cuda")
    moe.invoke_silu_and_mul_kernel(AB, C)
    a = orc.to_julia(AB[:, :inter]); b = orc.to_julia(AB[:, inter:])
    ref = orc.silu_and_mul(a, b)
    check(orc.to_julia(C), ref, 2e-3)
    x = torch.from_numpy(rng.standard_normal((19, 4, 130)).astype(np.float16)).cuda()  # Julia (130, 4, 19)
    out = torch.empty((19, 130), dtype=torch.float16, device="cuda")
    ct.moe_sum_topk(x, out)
    assert torch.equal(out, x.float().sum(dim=1).to(torch.float16))
    assert ct.last_variant() == "moe_sum_topk"
    # channel counts that are multiples of eight take 16-byte loads: the unrolled slot counts, a general one, bf16,
    # and a view whose token stride is padded
    for topk, H, T, dt in [(2, 1024, 256, torch.float16), (8, 136, 33, torch.float16), (3, 64, 5, torch.float16),
                           (4, 256, 70, torch.bfloat16), (1, 8, 1, torch.float16)]:
        x = torch.from_numpy(rng.standard_normal((T, topk + 1, H)).astype(np.float32)).to(dt).cuda()[:, :topk]
        out = torch.full((T, H + 8), 7.0, dtype=dt, device="cuda")
        ct.moe_sum_topk(x, out[:, :H])
        assert ct.last_variant() == "moe_sum_topk_vec8"
        ref = torch.zeros((T, H), dtype=torch.float32, device="cuda")
        for k in range(topk):
            ref += x[:, k].float()                                  # slots in ascending order, fp32
        assert torch.equal(out[:, :H], ref.to(dt)) and bool((out[:, H:] == 7.0).all())


def test_moe_fp8_weights(orc):
    """E4M3FN expert weights with per-(n, expert) fp32 scales: the oracle is ref_moe on the
    dequantised weights, so only accumulation order and the f16 cache roundings differ."""
    d = moe.prepare(num_tokens=96, hidden_size=512, num_experts=8, intermediate_size=512, topk=2,
                    router="top2_logits")
    J = orc.to_julia
    c1, s1 = orc.quantize_e4m3fn_per_channel(J(d.w1).astype(np.float32))
    c2, s2 = orc.quantize_e4m3fn_per_channel(J(d.w2).astype(np.float32))
    up = lambda c: orc.from_julia(c).cuda().view(torch.float8_e4m3fn)
    out = moe.cutile_moe(d.hidden_states, up(c1), up(c2), d.topk_weights, d.topk_ids, 128, 128, 64,
                         w1_scale=orc.from_julia(s1).cuda(), w2_scale=orc.from_julia(s2).cuda())
    w1d = orc.e4m3fn_decode(c1) * s1[None]; w2d = orc.e4m3fn_decode(c2) * s2[None]
    ref = orc.ref_moe(J(d.hidden_states), w1d, w2d, J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(out), ref)


@pytest.mark.parametrize("tokens,E,K,N,dtype,accumulate", [
    (100, 64, 512, 480, torch.float16, False),    # 7.5 strips of 64 channels, two K steps (the fewest)
    (64, 32, 768, 1024, torch.bfloat16, True),    # 512 strips in all and two replicas per expert: the smallest of the range
    (511, 32, 2048, 1024, torch.float16, True),   # almost 32 replicas per expert, most of them two tiles
    (65, 33, 512, 1022, torch.float16, False),    # a last strip of 62 channels
])
def test_e4m3_weights_in_strips_of_64_channels(ct, orc, tokens, E, K, N, dtype, accumulate):
    """One grouped GEMM against float64 dot products over the dequantised weights.  The products of f16 / bf16 and e4m3
    are exact in fp32, so a result is off by its sum's roundings (K * 2^-24 of the sum of magnitudes at most) and its
    own rounding to the storage type (2^-11 / 2^-8 of it, once per addend where replicas are added)."""
    g = torch.Generator(device="cuda").manual_seed(tokens)
    A = torch.randn(tokens, K, device="cuda", generator=g).to(dtype)
    W = torch.randn(E, N, K, device="cuda", generator=g).to(torch.float8_e4m3fn)
    scale = torch.rand(E, N, device="cuda", generator=g) * 0.1 + 0.05
    ids = torch.argsort(torch.rand(tokens, E, device="cuda", generator=g), dim=1)[:, :2].t().contiguous() + 1   # (2, tokens)
    w = torch.rand(2, tokens, device="cuda", generator=g).to(dtype)
    tok, exp = ct.moe_align_tile_size_device(ids, 128, E)
    ref, mag = [], []
    for k in range(2):
        r, m = torch.empty(tokens, N, dtype=torch.float64, device="cuda"), torch.empty(tokens, N, dtype=torch.float64, device="cuda")
        for t in range(tokens):
            x = A[t].double() * W[ids[k, t] - 1].double()
            f = scale[ids[k, t] - 1].double()
            r[t], m[t] = x.sum(dim=1) * f, x.abs().sum(dim=1) * f
        ref.append(r * w[k].double()[:, None])
        mag.append(m * w[k].double()[:, None])
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    if accumulate:
        # (replica r of token t belongs to column t: A's rows, one per token and slot)
        A2 = A.repeat_interleave(2, dim=0)
        out = torch.zeros(tokens, N, dtype=dtype, device="cuda")
        ct.fused_moe_accumulate_kernel(A2, W, out, w, tok, exp, 128, 128, 64, b_scale=scale)
        r, m = ref[0] + ref[1], mag[0] + mag[1]
        bound = (K + 2) * 2.0 ** -24 * m + 2 * eps * (ref[0].abs() + ref[1].abs()) + 2.0 ** -23
    else:
        out = torch.full((tokens * 2, N), float("nan"), dtype=dtype, device="cuda")
        ct.fused_moe_kernel(A, W, out, w, tok, exp, 2, True, 128, 128, 64, b_scale=scale)
        r, m = torch.stack(ref, dim=1).reshape(tokens * 2, N), torch.stack(mag, dim=1).reshape(tokens * 2, N)
        bound = (K + 2) * 2.0 ** -24 * m + 1.01 * eps * r.abs() + 2.0 ** -23
    assert ct.last_variant() == "fused_moe_t32_n64_k256_ksplit2_w8a16"
    err = (out.double() - r).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


def test_e4m3_weight_rows_off_16_bytes_take_strips_of_32_channels(ct):
    """The same weights in rows that are and are not 16-byte aligned (views of a wider buffer): two kernels, each off
    the exact sum by K * 2^-24 of the sum of magnitudes and by the result's rounding at most."""
    tokens, E, K, N = 64, 32, 512, 1024
    g = torch.Generator(device="cuda").manual_seed(3)
    A = torch.randn(tokens, K, device="cuda", generator=g).half()
    W = torch.randn(E, N, K + 8, device="cuda", generator=g).to(torch.float8_e4m3fn)[:, :, :K]
    scale = torch.rand(E, N, device="cuda", generator=g) * 0.1 + 0.05
    ids = torch.argsort(torch.rand(tokens, E, device="cuda", generator=g), dim=1)[:, :2].t().contiguous() + 1
    w = torch.rand(2, tokens, device="cuda", generator=g).half()
    tok, exp = ct.moe_align_tile_size_device(ids, 128, E)
    out, variant = [], []
    for weights in (W.contiguous(), W):
        out.append(torch.full((tokens * 2, N), float("nan"), dtype=torch.float16, device="cuda"))
        ct.fused_moe_kernel(A, weights, out[-1], w, tok, exp, 2, True, 128, 128, 64, b_scale=scale)
        variant.append(ct.last_variant())
    assert variant == ["fused_moe_t32_n64_k256_ksplit2_w8a16", "fused_moe_t32_n32_k256_ksplit4_w8a16"]
    f = (scale[ids.t().reshape(-1) - 1] * w.t().reshape(-1, 1)).double()      # (slot, channel)
    x = W.double()[ids.t().reshape(-1) - 1] * A.double().repeat_interleave(2, dim=0)[:, None]
    ref, mag = x.sum(dim=2) * f, x.abs().sum(dim=2) * f
    for o in out:
        assert bool(((o.double() - ref).abs() <= (K + 2) * 2.0 ** -24 * mag + 1.01 * 2.0 ** -11 * ref.abs() + 2.0 ** -23).all())


def test_fp8_dequant_covers_every_code(ct, orc):
    """Every finite E4M3FN code as a weight: K = 256 codes against a one-hot activation picks
    each dequantised value out exactly (checks subnormals, signs and the exponent rebias)."""
    codes = np.arange(256, dtype=np.uint8)
    codes[0x7F] = 0; codes[0xFF] = 0x80  # the two NaN codes never occur in weights
    K, N, E = 256, 32, 1
    Bq = np.repeat(codes[:, None, None], N, axis=1)           # (K, N, E)
    scale = np.linspace(0.5, 2.0, N, dtype=np.float32)[:, None]  # (N, E)
    A = np.eye(K, dtype=np.float16)                           # token t = one-hot at k = t
    ids = np.ones((K, 1), dtype=np.int64)
    tok, exp = orc.moe_align_tile_size(ids, 128, E)
    C = torch.zeros((K, N), dtype=torch.float16, device="cuda")
    ct.fused_moe_kernel(orc.from_julia(A).cuda(), orc.from_julia(Bq).cuda().view(torch.float8_e4m3fn), C,
                        torch.ones(K, dtype=torch.float16, device="cuda"), torch.from_numpy(tok).cuda(),
                        torch.from_numpy(exp).cuda(), 1, False, 128, 128, 64,
                        b_scale=orc.from_julia(scale).cuda())
    ref = (orc.e4m3fn_decode(codes)[None, :] * scale).astype(np.float16)  # (N, K)
    assert np.array_equal(orc.to_julia(C), ref)


def test_moe_full_size_top2(orc):
    """The measured configuration (256 tokens, hidden 1024, 32 experts, inter 2048, top-2)."""
    d = moe.prepare(benchmark=True, topk=2, router="top2_logits")
    r = moe.run(d)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float32)
    check(J(r.out), ref.astype(np.float64))


@pytest.mark.parametrize("num_tokens,topk,E,tile_m", [(256, 2, 32, 128), (48, 8, 64, 16), (7, 3, 5, 4), (1, 1, 1, 128),
                                                      (1000, 4, 9, 32), (130, 2, 1000, 8),
                                                      (512, 2, 32, 128), (512, 4, 7, 16), (513, 4, 7, 16), (2049, 1, 33, 64),
                                                      (4096, 2, 32, 128), (4100, 3, 11, 128),   # one and two batches of ids per wave
                                                      (16385, 2, 160, 64), (8193, 1, 1000, 8), (40000, 3, 3, 128),   # several workgroups:
                                                      (70000, 2, 1024, 16), (9000, 7, 64, 128)])                      # 33, 9, 64, 16 and 62 of them
def test_device_align_matches_host_routine(ct, orc, num_tokens, topk, E, tile_m):
    """The counting sort (one workgroup, or two launches of several from 8192 replicas on) gives the host routine's
    arrays (stable per-expert order, sentinel padding) in the leading part of its fixed-capacity outputs, and marks
    the rest unused."""
    rng = np.random.default_rng(num_tokens + topk)
    ids = rng.integers(1, E + 1, size=(topk, num_tokens), dtype=np.int64)   # torch layout of Julia (tokens, topk)
    ids_t = torch.from_numpy(ids)
    tok_h, exp_h = ct.moe_align_tile_size(ids_t, tile_m, E)
    tok_d, exp_d = ct.moe_align_tile_size_device(ids_t.cuda(), tile_m, E)
    nb = exp_h.numel()
    blocks, slots = ct.moe_align_capacity(num_tokens, topk, tile_m, E)
    assert tok_d.numel() == slots and exp_d.numel() == blocks and nb <= blocks
    assert torch.equal(exp_d[:nb].cpu(), exp_h) and torch.all(exp_d[nb:] == 0)
    assert torch.equal(tok_d[:nb * tile_m].cpu(), tok_h) and torch.all(tok_d[nb * tile_m:] == num_tokens * topk + 1)
    assert ct.last_variant() == ("moe_align_device_count_place" if num_tokens * topk >= 8192 else "moe_align_device_1wg")
    # oracle as a third opinion
    tok_o, exp_o = orc.moe_align_tile_size(ids.T, tile_m, E)
    assert np.array_equal(tok_h.numpy(), tok_o) and np.array_equal(exp_h.numpy(), exp_o)


def test_device_align_of_several_workgroups_in_a_row_and_under_capture(ct):
    """The two-launch sort keeps its counts in an array of the library: a smaller batch after a larger one, a batch
    with ids outside 1..E and one that clears an array on the way all match the host routine; a capturing stream is
    not given the array, sorts with one workgroup, and the replayed graph gives the same arrays."""
    rng = np.random.default_rng(5)
    E, tile_m = 48, 64
    for num_tokens, topk, bad in [(30000, 4, False), (5000, 2, False), (12000, 3, True), (9000, 1, False)]:
        ids = rng.integers(1, E + 1, size=(topk, num_tokens), dtype=np.int64)
        if bad:
            ids[rng.random(ids.shape) < 0.1] = 0
            ids[rng.random(ids.shape) < 0.05] = E + 7
        ids_t = torch.from_numpy(ids)
        valid = torch.from_numpy(((ids >= 1) & (ids <= E)).T.reshape(-1))   # replica order: slot fastest
        junk = torch.full((1024, 33), 3.0, dtype=torch.float16, device="cuda")
        tok_d, exp_d = ct.moe_align_tile_size_device(ids_t.cuda(), tile_m, E, clear=junk)
        multi = num_tokens * topk >= 8192
        assert ct.last_variant() == ("moe_align_device_count_place" if multi else "moe_align_device_1wg")
        assert not junk.any()
        if not bad:
            tok_h, exp_h = ct.moe_align_tile_size(ids_t, tile_m, E)
        else:   # the host routine takes valid ids only: sort the valid replicas, keep their original numbers
            flat = ids.T.reshape(-1)
            keep = np.nonzero(valid.numpy())[0]
            tok_s, exp_h = ct.moe_align_tile_size(torch.from_numpy(flat[keep].reshape(1, -1).copy()), tile_m, E)
            sentinel = tok_s == keep.size + 1
            tok_h = torch.from_numpy(keep.astype(np.int32) + 1)[(tok_s.long() - 1).clamp(max=keep.size - 1)]
            tok_h[sentinel] = num_tokens * topk + 1
        nb = exp_h.numel()
        assert torch.equal(exp_d[:nb].cpu(), exp_h) and torch.all(exp_d[nb:] == 0)
        assert torch.equal(tok_d[:nb * tile_m].cpu(), tok_h) and torch.all(tok_d[nb * tile_m:] == num_tokens * topk + 1)
    # the last batch again, captured
    ids_d = ids_t.cuda()
    tok_g, exp_g = torch.empty_like(tok_d), torch.empty_like(exp_d)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            ct.moe_align_tile_size_device(ids_d, tile_m, E, tok_g, exp_g, stream=side)
            assert ct.last_variant() == "moe_align_device_1wg"
    for _ in range(2):
        tok_g.fill_(-1); exp_g.fill_(-1)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(tok_g, tok_d) and torch.equal(exp_g, exp_d)


@pytest.mark.parametrize("num_tokens,E,topk,dtype", [(256, 32, 2, torch.float32), (48, 64, 8, torch.float32),
                                                     (7, 100, 5, torch.float16), (3, 512, 64, torch.float32),
                                                     (5, 6, 6, torch.bfloat16), (1, 1, 1, torch.float32),
                                                     (1000, 130, 4, torch.float32)])
def test_device_router_matches_oracle(ct, orc, num_tokens, E, topk, dtype):
    """mi_moe_route_topk against the oracle's router (stable argsort of the negated logits, softmax
    over the selected ones in float64): ids identical, weights within 1e-6 relative in f32 (one
    exp and one division in fp32) or one rounding step of the 16-bit output type."""
    rng = np.random.default_rng(num_tokens * 7 + E)
    logits = torch.from_numpy(rng.standard_normal((num_tokens, E)).astype(np.float32)).to(dtype)
    w_ref, ids_ref = orc.route_top2(logits.float().numpy().astype(np.float64), topk)
    w, ids = ct.moe_route_topk(logits.t().contiguous().cuda(), topk)            # torch (E, tokens) = Julia (tokens, E)
    assert ids.shape == (topk, num_tokens) and ids.dtype == torch.int64 and w.dtype == dtype
    assert np.array_equal(ids.cpu().numpy().T, ids_ref)
    tol = 1e-6 if dtype == torch.float32 else (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7)
    np.testing.assert_allclose(w.float().cpu().numpy().T, w_ref, rtol=tol, atol=1e-30 if dtype == torch.float32 else 1e-7)
    # f32 weights from 16-bit logits, and a strided (token-major) logits view
    w32, ids2 = ct.moe_route_topk(logits.cuda().t(), topk, weight_dtype=torch.float32)
    assert np.array_equal(ids2.cpu().numpy().T, ids_ref)
    np.testing.assert_allclose(w32.cpu().numpy().T, w_ref, rtol=1e-6)
    np.testing.assert_allclose(w32.sum(dim=0).cpu().numpy(), 1.0, rtol=1e-6)


def test_device_router_ties_and_nan(ct, orc):
    """Equal logits go to the lower expert id (the stable sort of the oracle); NaN logits are never
    preferred to numbers."""
    rng = np.random.default_rng(3)
    logits = rng.integers(-2, 3, size=(64, 40)).astype(np.float32)               # many ties
    w_ref, ids_ref = orc.route_top2(logits.astype(np.float64), 6)
    w, ids = ct.moe_route_topk(torch.from_numpy(logits).t().contiguous().cuda(), 6)
    assert np.array_equal(ids.cpu().numpy().T, ids_ref)
    np.testing.assert_allclose(w.cpu().numpy().T, w_ref, rtol=1e-6)
    logits = rng.standard_normal((16, 12)).astype(np.float32)
    logits[:, [1, 5, 7]] = np.nan
    clean = np.where(np.isnan(logits), -1e30, logits)
    _, ids_ref = orc.route_top2(clean.astype(np.float64), 4)
    _, ids = ct.moe_route_topk(torch.from_numpy(logits).t().contiguous().cuda(), 4)
    assert np.array_equal(ids.cpu().numpy().T, ids_ref)


def test_moe_routed_on_device_end_to_end(ct, orc):
    """Router, sort, GEMMs, activation and combine all on the GPU: the measured configuration from
    logits to output equals the run whose routing was prepared on the host."""
    d = moe.prepare(benchmark=True, topk=2, router="top2_logits")
    w, ids = ct.moe_route_topk(d.logits.t().contiguous(), 2, weight_dtype=d.topk_weights.dtype)
    assert torch.equal(ids, d.topk_ids)
    a = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, device_align=True)
    b = moe.cutile_moe(d.hidden_states, d.w1, d.w2, w, ids, 128, 128, 64, device_align=True)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(w), J(ids), dtype=np.float32)
    check(J(b), ref.astype(np.float64))
    assert (a.float() - b.float()).abs().max().item() <= 2e-3 * a.float().abs().max().item()  # weights differ by <= 1 f16 step


def test_moe_end_to_end_with_device_align(orc):
    """cutile_moe with the sort on the GPU equals the version that sorts on the host, bit for bit
    (the extra, unused blocks change nothing)."""
    d = moe.prepare(benchmark=True, topk=2, router="top2_logits")
    a = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, device_align=False, fuse_silu=False)
    b = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, device_align=True, fuse_silu=False)
    c = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64)   # defaults: device sort, fused SiLU
    assert torch.equal(a, b) and torch.equal(a, c)
    d = moe.prepare(num_tokens=33, hidden_size=256, num_experts=7, intermediate_size=128, topk=3)
    a = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 16, 128, 64, device_align=False, fuse_silu=False)
    b = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 16, 128, 64, device_align=True, fuse_silu=False)
    assert torch.equal(a, b)


@pytest.mark.parametrize("shape", [dict(benchmark=True, topk=2, router="top2_logits"),
                                   dict(num_tokens=33, hidden_size=256, num_experts=7, intermediate_size=128, topk=3),
                                   dict(num_tokens=20, hidden_size=512, num_experts=5, intermediate_size=80, topk=2),
                                   dict(num_tokens=64, hidden_size=384, num_experts=4, intermediate_size=1000, topk=1)])
def test_gemm_with_fused_silu_epilogue(ct, orc, shape):
    """mi_fused_moe_silu_kernel against mi_fused_moe_kernel followed by mi_silu_and_mul_kernel: both
    products are rounded to the activation type before SiLU, as the separate kernels do, so the
    results are bit-identical whenever the separate GEMM runs the same 128-lane-wide mainloop; when it
    picks its K-split shape (small problems) the fp32 sums are ordered differently and the outputs
    may differ by rounding (bar: the f16 tolerance of this file against the float64 oracle).
    Includes intermediate sizes that are not multiples of the 64-channel strips."""
    d = moe.prepare(**shape)
    tile_m = 128 if shape.get("benchmark") else 16
    a = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, tile_m, 128, 64, device_align=True)
    variants = set()
    inter, total = d.intermediate_size, d.num_tokens * d.topk
    tok, exp = ct.moe_align_tile_size_device(d.topk_ids, tile_m, d.num_experts)
    c1 = torch.zeros(total, 2 * inter, dtype=d.hidden_states.dtype, device="cuda")
    moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c1, d.topk_weights, tok, exp, mul_routed_weight=False,
                                num_token_replicas=d.topk, tile_m=tile_m, tile_n=128, tile_k=64)
    variants.add(ct.last_variant())
    b = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, tile_m, 128, 64, device_align=True,
                       fuse_silu=True)
    if variants == {"fused_moe_t32_n128_k128"}:
        assert torch.equal(a, b)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(b), ref)


def test_dense_routing_two_slot_tiles_per_workgroup(ct, orc):
    """More than 32 tokens per expert on average (the reference's own benchmark routing: 256 tokens, top-8 of 32
    experts, moe.jl:311-344): a workgroup then multiplies two 32-slot tiles with the same weight tile.  The wide,
    and the fused-SiLU mainloops have that variant (dense routing always takes wide strips); every element is accumulated in the same order
    as with one tile per workgroup, so fused and separate paths still agree bit for bit, and the result is checked
    against the float64 oracle.  Includes a small problem with unequal expert loads.  (These are the
    streaming kernels' shapes for dense routing; they serve blocks smaller than 128 slots and e4m3 weights, and are
    kept on here by the knob.)"""
    with _dense_knob("0"):
        _two_slot_tiles_body(ct, orc)


def _two_slot_tiles_body(ct, orc):
    d = moe.prepare(benchmark=True, topk=8)
    tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 128, d.num_experts)
    c1 = torch.zeros(d.num_tokens * 8, 2 * d.intermediate_size, dtype=torch.float16, device="cuda")
    moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c1, d.topk_weights, tok, exp, mul_routed_weight=False,
                                num_token_replicas=8, tile_m=128, tile_n=128, tile_k=64)
    assert ct.last_variant() == "fused_moe_t64_n128_k128"
    c2 = torch.zeros(d.num_tokens * 8, d.intermediate_size, dtype=torch.float16, device="cuda")
    moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c2, d.topk_weights, tok, exp, mul_routed_weight=False,
                                num_token_replicas=8, tile_m=128, tile_n=128, tile_k=64, fuse_silu=True)
    assert ct.last_variant() == "fused_moe_silu_t64_n64x2_k128"
    c3 = torch.zeros(d.num_tokens * 8, d.hidden_size, dtype=torch.float16, device="cuda")
    moe.invoke_fused_moe_kernel(c2, d.w2, c3, d.topk_weights, tok, exp, mul_routed_weight=True,
                                num_token_replicas=1, tile_m=128, tile_n=128, tile_k=64)
    assert ct.last_variant() == "fused_moe_t64_n128_k128"
    a = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, device_align=True, fuse_silu=False)
    b = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, device_align=True, fuse_silu=True)
    h = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, device_align=False,
                       fuse_silu=False)      # host sort: exact block count; the reference's launch sequence
    assert torch.equal(a, b) and torch.equal(a, h)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float32)
    check(J(a), ref.astype(np.float64))
    q = moe.quantize_weights(d)
    f = moe.cutile_moe(d.hidden_states, q.w1, q.w2, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=q.w1_scale,
                       w2_scale=q.w2_scale, device_align=True, fuse_silu=True)
    g = moe.cutile_moe(d.hidden_states, q.w1, q.w2, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=q.w1_scale,
                       w2_scale=q.w2_scale, device_align=True, fuse_silu=False)
    assert torch.equal(f, g)
    w1d = orc.e4m3fn_decode(J(q.w1.view(torch.uint8))) * J(q.w1_scale)[None]
    w2d = orc.e4m3fn_decode(J(q.w2.view(torch.uint8))) * J(q.w2_scale)[None]
    check(J(f), orc.ref_moe(J(d.hidden_states), w1d, w2d, J(d.topk_weights), J(d.topk_ids), dtype=np.float32).astype(np.float64))
    # small and uneven: 3 experts, 70 tokens, top-2 (about 47 tokens per expert, some tiles half empty)
    d = moe.prepare(num_tokens=70, hidden_size=256, num_experts=3, intermediate_size=192, topk=2)
    a = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, device_align=True, fuse_silu=False)
    b = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 64, 128, 64, device_align=False, fuse_silu=True)
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(a), ref)
    check(J(b), ref)


def test_fused_silu_epilogue_bf16_and_fp8_weights(orc):
    d = moe.prepare(num_tokens=40, hidden_size=256, num_experts=6, intermediate_size=192, topk=2, T=torch.bfloat16)
    a = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 32, 128, 64, device_align=False, fuse_silu=False)
    b = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 32, 128, 64, device_align=False, fuse_silu=True)
    assert torch.equal(a, b)
    d = moe.prepare(benchmark=True, topk=2, router="top2_logits")
    q = moe.quantize_weights(d)
    a = moe.cutile_moe(d.hidden_states, q.w1, q.w2, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=q.w1_scale,
                       w2_scale=q.w2_scale, device_align=True, fuse_silu=False)
    b = moe.cutile_moe(d.hidden_states, q.w1, q.w2, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=q.w1_scale,
                       w2_scale=q.w2_scale, device_align=True, fuse_silu=True)
    assert torch.equal(a, b)
    # the measured e4m3 configuration at full size (top-2) against ref_moe on the dequantised weights
    J = orc.to_julia
    w1d = orc.e4m3fn_decode(J(q.w1.view(torch.uint8))) * J(q.w1_scale)[None]
    w2d = orc.e4m3fn_decode(J(q.w2.view(torch.uint8))) * J(q.w2_scale)[None]
    ref = orc.ref_moe(J(d.hidden_states), w1d, w2d, J(d.topk_weights), J(d.topk_ids), dtype=np.float32).astype(np.float64)
    check(J(b), ref)
    assert orc.isapprox(J(b).astype(np.float64), ref, rtol=1e-2, atol=1e-2)


def test_product_quantizer_matches_oracle_codec(orc):
    """examples.moe.quantize_weights (torch, on the GPU) against the oracle's per-channel E4M3FN
    quantiser: scales equal to fp32 rounding of the division, codes equal except where that last
    bit of the scale moves a value across a rounding tie (then by one code step)."""
    d = moe.prepare(num_tokens=8, hidden_size=128, num_experts=3, intermediate_size=64, topk=1)
    q = moe.quantize_weights(d)
    J = orc.to_julia
    c1, s1 = orc.quantize_e4m3fn_per_channel(J(d.w1).astype(np.float32))
    np.testing.assert_allclose(J(q.w1_scale), s1, rtol=2e-7)
    got = J(q.w1.view(torch.uint8)).astype(np.int32)
    diff = np.abs(got - c1.astype(np.int32))
    assert diff.max() <= 1 and (diff != 0).mean() < 1e-3


def test_fused_silu_entry_checks_shapes(ct):
    d = moe.prepare(num_tokens=8, hidden_size=128, num_experts=2, intermediate_size=64, topk=1)
    tok, exp = ct.moe_align_tile_size(d.topk_ids.cpu(), 16, 2)
    tok, exp = tok.cuda(), exp.cuda()
    wrong = torch.zeros(8, 128, dtype=torch.float16, device="cuda")          # must be (total, inter) = (8, 64)
    with pytest.raises(ct.MiError) as e:
        ct.fused_moe_silu_kernel(d.hidden_states, d.w1, wrong, d.topk_weights.reshape(-1), tok, exp, 1, False, 16, 128, 64)
    assert e.value.code == ct.MI_E_SHAPE


def test_silu_and_topk_sum_beyond_65535_columns(ct, orc):
    """Prefill sizes: tokens * topk above 65535 (the reference's flattened grids take 2^24 - 1 blocks,
    src/launch.jl:743).  Checked against the same kernels run on column slices."""
    rng = np.random.default_rng(4)
    inter, total = 64, 70_001
    AB = torch.from_numpy((rng.standard_normal((total, 2 * inter)) * 3).astype(np.float16)).cuda()
    C = torch.zeros((total, inter), dtype=torch.float16, device="cuda")
    moe.invoke_silu_and_mul_kernel(AB, C)
    for lo, hi in ((0, 3), (65_530, 65_545), (total - 4, total)):
        ref = orc.silu_and_mul(orc.to_julia(AB[lo:hi, :inter]), orc.to_julia(AB[lo:hi, inter:]))
        check(orc.to_julia(C[lo:hi]), ref, 2e-3)
    C2 = torch.zeros_like(C)
    moe.invoke_silu_and_mul_kernel(AB[:60_000], C2[:60_000]); moe.invoke_silu_and_mul_kernel(AB[60_000:], C2[60_000:])
    assert torch.equal(C, C2)
    x = torch.from_numpy(rng.standard_normal((total, 2, 64)).astype(np.float16)).cuda()   # Julia (64, 2, total)
    out = torch.empty((total, 64), dtype=torch.float16, device="cuda")
    ct.moe_sum_topk(x, out)
    assert torch.equal(out, x.float().sum(dim=1).to(torch.float16))


@pytest.mark.parametrize("tokens,hidden,experts,inter,topk,T,fp8", [
    (256, 1024, 32, 2048, 2, torch.float16, False), (256, 1024, 32, 2048, 2, torch.float16, True),
    (100, 256, 8, 192, 2, torch.bfloat16, False), (33, 128, 3, 64, 1, torch.float16, False),
    (300, 264, 2, 256, 2, torch.float16, False), (1, 64, 4, 64, 2, torch.bfloat16, True),
])
def test_down_projection_that_adds_into_the_output(ct, orc, tokens, hidden, experts, inter, topk, T, fp8):
    """fuse_sum: the sort launch zeroes the output and the down projection adds every replica's row into it with
    packed atomic adds (mi_fused_moe_accumulate_kernel) -- three launches, no cache3.  With one or two slots per token
    the sum does not depend on the order of arrival, and the atomic add rounds like the separate sum does: the result
    is the unfused one bit for bit, run after run, and is checked against the float64 oracle as well."""
    d = moe.prepare(num_tokens=tokens, hidden_size=hidden, num_experts=experts, intermediate_size=inter, topk=topk, T=T,
                    router="top2_logits" if topk == 2 and experts >= 2 else "randperm")
    kw = {}
    if fp8:
        q = moe.quantize_weights(d)
        w1, w2, kw = q.w1, q.w2, dict(w1_scale=q.w1_scale, w2_scale=q.w2_scale)
    else:
        w1, w2 = d.w1, d.w2
    plain = moe.cutile_moe(d.hidden_states, w1, w2, d.topk_weights, d.topk_ids, 128, 128, 64, fuse_sum=False, **kw)
    assert ct.last_variant().startswith("moe_sum_topk")
    for _ in range(3):
        fused = moe.cutile_moe(d.hidden_states, w1, w2, d.topk_weights, d.topk_ids, 128, 128, 64, fuse_sum=True, **kw)
        assert ct.last_variant().startswith(("fused_moe_t", "fused_moe_dense_acc"))          # the last launch is the GEMM itself
        assert torch.equal(fused, plain)
    default = moe.cutile_moe(d.hidden_states, w1, w2, d.topk_weights, d.topk_ids, 128, 128, 64, **kw)
    assert torch.equal(default, plain)
    if not fp8:
        J = orc.to_julia
        ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
        check(J(fused), ref, 2e-2 if T == torch.float16 else 5e-2)
    # more than two slots: the fused form is refused, the default falls back to the separate sum
    if experts >= 4:
        d4 = moe.prepare(num_tokens=tokens, hidden_size=hidden, num_experts=experts, intermediate_size=inter, topk=4, T=T)
        with pytest.raises(ValueError):
            moe.cutile_moe(d4.hidden_states, d4.w1, d4.w2, d4.topk_weights, d4.topk_ids, 128, 128, 64, fuse_sum=True)
        moe.cutile_moe(d4.hidden_states, d4.w1, d4.w2, d4.topk_weights, d4.topk_ids, 128, 128, 64)
        assert ct.last_variant().startswith("moe_sum_topk")


@pytest.mark.parametrize("topk", [2, 4])
def test_replicas_with_an_expert_id_out_of_range_contribute_nothing(orc, topk):
    """Expert ids outside 1..num_experts: the reference raises on them (moe_align_tile_size indexes its counters by
    the id, moe.jl:150-160); the device-side sort drops such replicas.  Whatever path the call then takes (two slots:
    the down projection adds into the zeroed output; more: cache3 + the top-k sum), a dropped replica has to
    contribute 0 -- not what an unwritten cache column happens to hold (the tests run with poisoned allocations).
    The expected output is the oracle's with the dropped replicas' routed weights set to 0."""
    d = moe.prepare(num_tokens=40, hidden_size=256, num_experts=6, intermediate_size=192, topk=topk)
    ids = d.topk_ids.clone()
    ids[0, 3] = 0
    ids[topk - 1, 17] = d.num_experts + 1
    ids[1, 29] = -5
    w_ref = d.topk_weights.clone()
    bad = (ids < 1) | (ids > d.num_experts)
    w_ref[bad] = 0
    ids_ref = torch.where(bad, torch.ones_like(ids), ids)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(w_ref), J(ids_ref), dtype=np.float64)
    for fuse_silu in (True, False):
        got = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, ids, 16, 128, 64, device_align=True, fuse_silu=fuse_silu)
        assert not torch.isnan(got.float()).any()
        check(J(got), ref)
    if topk <= 2:
        sep = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, ids, 16, 128, 64, device_align=True, fuse_sum=False)
        assert torch.equal(sep, got)


def _every_path(d, tile_m, **kw):
    """cutile_moe over its launch sequences: fused SiLU + accumulating down projection (where top-k allows), fused SiLU
    + separate sum, and the reference's kernel-by-kernel sequence."""
    outs = {}
    a = (d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, tile_m, 128, 64)
    if d.topk <= 2 and d.hidden_size % 8 == 0:
        outs["fused"] = moe.cutile_moe(*a, **kw)
    outs["fused_silu"] = moe.cutile_moe(*a, fuse_sum=False, **kw)
    outs["separate"] = moe.cutile_moe(*a, fuse_silu=False, fuse_sum=False, **kw)
    return outs


@pytest.mark.parametrize("shape", [
    dict(benchmark=True, topk=8),                                                                     # the reference example's routing
    dict(num_tokens=1024, hidden_size=1024, num_experts=32, intermediate_size=2048, topk=2, router="top2_logits"),
    dict(num_tokens=300, hidden_size=328, num_experts=3, intermediate_size=200, topk=2),               # K and N off the tile grid
    dict(num_tokens=700, hidden_size=264, num_experts=5, intermediate_size=96, topk=1),                # one slot per token
    dict(num_tokens=1024, hidden_size=256, num_experts=160, intermediate_size=128, topk=8),
    dict(num_tokens=2048, hidden_size=256, num_experts=256, intermediate_size=64, topk=8),
    dict(num_tokens=400, hidden_size=512, num_experts=4, intermediate_size=256, topk=2, T=torch.bfloat16),
    # K of both projections from 512 on and off the grid of the 64-k stages (chunks past K in the last groups of steps)
    dict(num_tokens=300, hidden_size=520, num_experts=3, intermediate_size=776, topk=2),
    dict(num_tokens=96, hidden_size=1000, num_experts=4, intermediate_size=584, topk=2, T=torch.bfloat16),
])
@pytest.mark.parametrize("J", ["2", "4", "2wide", "4wide", "2wide_nt", "4wide_nt"])
def test_dense_routing_ring_kernel_gives_the_streaming_kernels_bits(ct, orc, shape, J, monkeypatch):
    """The grouped GEMM for dense routing (128-slot x 128-channel tiles fed by a ring of LDS stages, persistent
    workgroups) against the streaming kernels on the same launches: every output element is accumulated over k in
    the same order by both, so plain, SiLU-fused and accumulating launches have to agree bit for bit; the result is
    also checked against the float64 oracle.  Shapes: the reference example's own routing (moe.jl:311-344), a prefill
    batch, sizes off the tile grid (K = 328 ends in a zero-padded group of steps, N = 400 in clipped strips), one slot
    per token, 160 and 256 experts, bf16.  Both tile widths of the ring kernel: 128 weight rows on a ring of four stages
    (J = 2) and 256 rows on a ring of three (J = 4, whose K walk is padded to whole groups of three steps); and both
    again with stages of 64 k (whole 128-byte lines per row and transfer; from K = 512 on), forced on for every launch
    of the "wide" cases and off for the others; "_nt": their weight transfers non-temporal, as for launches with one
    block per expert (forced on for every launch; off for "wide")."""
    wide = "wide" in J
    monkeypatch.setenv("MI_MOE_DENSE_STREAM", "1" if J.endswith("_nt") else "0")
    J = J[0]
    monkeypatch.setenv("MI_MOE_DENSE_J", J)
    monkeypatch.setenv("MI_MOE_DENSE_WIDE", "1" if wide else "0")
    d = moe.prepare(**shape)
    J = orc.to_julia
    with _dense_knob("0"):
        ref_outs = _every_path(d, 128)
    names = set()
    with _dense_knob("1"):
        outs = _every_path(d, 128)
        tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 128, d.num_experts)
        c1 = torch.empty(d.num_tokens * d.topk, 2 * d.intermediate_size, dtype=d.hidden_states.dtype, device="cuda")
        moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c1, d.topk_weights, tok, exp, mul_routed_weight=False,
                                    num_token_replicas=d.topk, tile_m=128, tile_n=128, tile_k=64)
        names.add(ct.last_variant())
        c2 = torch.empty(d.num_tokens * d.topk, d.intermediate_size, dtype=d.hidden_states.dtype, device="cuda")
        moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c2, d.topk_weights, tok, exp, mul_routed_weight=False,
                                    num_token_replicas=d.topk, tile_m=128, tile_n=128, tile_k=64, fuse_silu=True)
        names.add(ct.last_variant())
    k = "k64" if wide and d.hidden_size >= 512 else "k32"
    assert names in ({f"fused_moe_dense_t128_n128_{k}_ring4", f"fused_moe_dense_silu_t128_n64x2_{k}_ring4"},
                     {f"fused_moe_dense_t128_n256_{k}_ring3", f"fused_moe_dense_silu_t128_n128x2_{k}_ring3"}), names
    for k in outs:
        assert not torch.isnan(outs[k].float()).any(), k
        assert torch.equal(outs[k], ref_outs[k]), k
        assert torch.equal(outs[k], outs["separate"]), k
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(outs["separate"]), ref, 5e-2 if d.hidden_states.dtype == torch.bfloat16 else 2e-2)


def test_dense_ring_kernel_other_block_sizes_sorts_and_output_layouts(ct, orc):
    """TILE_M = 256 (two 128-slot tiles per block, the second often empty), the host-side sort (exact block count),
    and an output whose rows are not whole 16-byte pieces (element-wise stores instead of 16-byte ones)."""
    d = moe.prepare(num_tokens=600, hidden_size=384, num_experts=6, intermediate_size=320, topk=2)
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    with _dense_knob("0"):
        want = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64, fuse_sum=False)
    with _dense_knob("1"):
        for tile_m, device_align in ((256, True), (256, False), (128, False), (512, True)):
            got = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, tile_m, 128, 64,
                                 device_align=device_align, fuse_sum=False)
            assert torch.equal(got, want), (tile_m, device_align)
            if device_align:
                acc = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, tile_m, 128, 64)
                assert torch.equal(acc, want), tile_m
        check(J(want), ref)
        # rows of C that start off a 16-byte boundary: leading dimension 2 * inter + 4 elements
        total, inter = d.num_tokens * d.topk, d.intermediate_size
        tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 128, d.num_experts)
        wide = torch.full((total, 2 * inter + 4), 7.0, dtype=torch.float16, device="cuda")
        dense_c1 = torch.empty(total, 2 * inter, dtype=torch.float16, device="cuda")
        for c in (wide[:, :2 * inter], dense_c1):
            moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c, d.topk_weights, tok, exp, mul_routed_weight=False,
                                        num_token_replicas=d.topk, tile_m=128, tile_n=128, tile_k=64)
            assert ct.last_variant().startswith("fused_moe_dense_t128_")
        assert torch.equal(wide[:, :2 * inter], dense_c1)
        assert bool((wide[:, 2 * inter:] == 7.0).all()), "the kernel wrote past the rows of its output"
    # 128-slot tiles need TILE_M to be a multiple of 128: smaller blocks stay on the streaming kernels
    with _dense_knob("1"):
        moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 64, 128, 64, fuse_sum=False)
        assert "dense" not in ct.last_variant()


@pytest.mark.parametrize("shape,T", [
    (dict(num_tokens=1024, hidden_size=1024, num_experts=32, intermediate_size=2048, topk=2, router="top2_logits"), torch.float16),
    (dict(benchmark=True, topk=8), torch.float16),
    (dict(num_tokens=300, hidden_size=528, num_experts=3, intermediate_size=560, topk=2), torch.bfloat16),   # K = 528, 560: zero-padded last steps
    (dict(num_tokens=500, hidden_size=512, num_experts=5, intermediate_size=544, topk=1), torch.float16),
])
def test_fp8_activations_times_fp8_weights_on_the_matrix_cores(ct, orc, shape, T):
    """E4M3FN activations x E4M3FN weights (the operand pairing of ext/DLFP8TypesExt.jl:15-19) in both grouped GEMMs of
    the MoE, fp32 accumulation, per-channel weight scales and per-tensor activation scales.  Oracle (the last row of the
    fp8 parity plan): ``ref_moe`` in float64 over the dequantised weights and the dequantised activations, with the
    intermediate rounded to the storage type and quantised exactly as the product does it between the projections
    (its own codec, pinned by the reference's vectors and by torch's fp8 dtype).  Only the accumulation order differs."""
    d = moe.prepare(T=T, **shape)
    q = moe.quantize_weights(d)
    J = orc.to_julia
    outs = []
    for kw in (dict(), dict(fuse_sum=False)):
        outs.append(moe.cutile_moe(d.hidden_states, q.w1, q.w2, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=q.w1_scale,
                                   w2_scale=q.w2_scale, fp8_activations=True, **kw))
        assert not torch.isnan(outs[-1].float()).any()
    assert "w8a8" in ct.last_variant() or ct.last_variant().startswith("moe_sum_topk")
    if d.topk <= 2:
        assert torch.equal(outs[0], outs[1])   # the accumulating down projection against cache3 + sum
    # the oracle's view of the same computation
    h8, a_scale = moe.quantize_activations(d.hidden_states)
    hs = orc.e4m3fn_decode(J(h8.view(torch.uint8))) * float(a_scale)
    # the library's quantiser against the oracle's codec: scale = max |x| / 448 and the quotient x / scale in fp32
    # (IEEE division), codes = round-to-nearest-even of that quotient.  (With bf16 data many quotients sit exactly on a
    # rounding boundary, so the quotient has to be formed in the same precision to compare codes one for one.)
    x32 = J(d.hidden_states).astype(np.float32)
    assert float(a_scale) == float(np.float32(np.abs(x32).max()) / np.float32(448.0))
    want = orc.e4m3fn_encode((x32 / np.float32(float(a_scale))).astype(np.float64))
    assert np.array_equal(want, J(h8.view(torch.uint8)))
    w1d = orc.e4m3fn_decode(J(q.w1.view(torch.uint8))) * J(q.w1_scale)[None]
    w2d = orc.e4m3fn_decode(J(q.w2.view(torch.uint8))) * J(q.w2_scale)[None]
    # the product's cache2: the first projection alone, then its quantisation
    tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 128, d.num_experts)
    c2 = torch.empty(d.num_tokens * d.topk, d.intermediate_size, dtype=T, device="cuda")
    moe.invoke_fused_moe_kernel(h8, q.w1, c2, d.topk_weights, tok, exp, mul_routed_weight=False, num_token_replicas=d.topk,
                                tile_m=128, tile_n=128, tile_k=64, b_scale=q.w1_scale * a_scale, fuse_silu=True)
    assert ct.last_variant() == "fused_moe_dense_silu_t128_n64x2_k64_ring4_w8a8"
    _, c_scale = moe.quantize_activations(c2)
    c_scale = float(c_scale)

    def mid(x):   # rounded to the storage type, then to e4m3 at the product's per-tensor scale
        x = orc.bf16_round(x.astype(np.float32)).astype(np.float64) if T == torch.bfloat16 else x.astype(np.float16).astype(np.float64)
        return orc.e4m3fn_decode(orc.e4m3fn_encode(x / c_scale)) * c_scale

    ref = orc.ref_moe(hs, w1d, w2d, J(d.topk_weights), J(d.topk_ids), dtype=np.float64, mid=mid)
    check(J(outs[1]), ref, 5e-2 if T == torch.bfloat16 else 2e-2)


def test_quantize_with_the_scale_folded_into_the_weight_scales(ct):
    """mi_quantize_e4m3fn_fold: the same codes and scale as mi_quantize_e4m3fn, and fold_out = fold_in * scale exactly
    (one fp32 multiply per element), for f16 and bf16, on a strided view of the activations."""
    g = torch.Generator(device="cuda"); g.manual_seed(3)
    for T in (torch.float16, torch.bfloat16):
        big = (torch.randn(300, 1040, device="cuda", generator=g) * 3).to(T)
        x = big[:, :1024]
        w_scale = torch.rand(33, 520, device="cuda", generator=g) + 0.5
        codes, scale = ct.quantize_e4m3fn(x)
        codes2, scale2, folded = ct.quantize_e4m3fn(x, fold=w_scale)
        assert torch.equal(codes.view(torch.uint8), codes2.view(torch.uint8)) and torch.equal(scale, scale2)
        assert torch.equal(folded, w_scale * scale)
    with pytest.raises(ct.MiError) as e:
        ct.quantize_e4m3fn(x, fold=w_scale, fold_out=torch.empty(5, device="cuda"))
    assert e.value.code == ct.MI_E_SHAPE


def test_fp8_activations_are_refused_where_no_kernel_takes_them(ct):
    d = moe.prepare(num_tokens=64, hidden_size=512, num_experts=4, intermediate_size=512, topk=2)
    q = moe.quantize_weights(d)
    h8, _ = moe.quantize_activations(d.hidden_states)
    tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 64, d.num_experts)
    c = torch.empty(d.num_tokens * 2, 2 * d.intermediate_size, dtype=torch.float16, device="cuda")
    with pytest.raises(ct.MiError) as e:    # blocks of 64 slots: only the 128-slot ring kernel multiplies fp8 by fp8
        moe.invoke_fused_moe_kernel(h8, q.w1, c, d.topk_weights, tok, exp, mul_routed_weight=False, num_token_replicas=2,
                                    tile_m=64, tile_n=128, tile_k=64, b_scale=q.w1_scale)
    assert e.value.code == ct.MI_E_UNSUPPORTED
    with pytest.raises(ct.MiError) as e:    # fp8 activations against 16-bit weights
        moe.invoke_fused_moe_kernel(h8, d.w1, c, d.topk_weights, tok, exp, mul_routed_weight=False, num_token_replicas=2,
                                    tile_m=128, tile_n=128, tile_k=64)
    assert e.value.code == ct.MI_E_DTYPE


def _routed(counts, topk=1, **kw):
    """moe.prepare with expert e taking counts[e] replicas (in shuffled order; topk slots of a token may name one expert twice)."""
    total = sum(counts)
    assert total % topk == 0
    d = moe.prepare(num_tokens=total // topk, num_experts=len(counts), topk=topk, **kw)
    ids = np.repeat(np.arange(1, len(counts) + 1), counts)
    np.random.default_rng(11).shuffle(ids)
    d.topk_ids = torch.from_numpy(ids.reshape(topk, -1).astype(np.int64)).cuda()
    return d


@pytest.mark.parametrize("rows", ["2", "4"])
@pytest.mark.parametrize("make", [
    # replicas per expert on the edges of 32-slot sub-tiles and of the tiles of 5 / 6 of them, none, and several tiles
    lambda: _routed([1, 31, 32, 33, 0, 127, 128, 160, 161, 192, 193, 700], hidden_size=256, intermediate_size=264),
    lambda: _routed([150, 170, 330, 250], topk=2, hidden_size=1000, intermediate_size=328, T=torch.bfloat16),   # K and N off 64 / 128 / 256
    lambda: moe.prepare(num_tokens=1024, hidden_size=256, num_experts=160, intermediate_size=256, topk=8),       # more runs than the table holds
    lambda: moe.prepare(num_tokens=2048, hidden_size=512, num_experts=8, intermediate_size=512, topk=2, router="top2_logits"),
], ids=["edges", "ragged", "many_runs", "prefill"])
def test_prefill_kernel_gives_the_streaming_kernels_bits(ct, orc, make, rows, monkeypatch):
    """The grouped GEMM whose transfers have waves of their own: k in the order of the streaming kernels, so the same bits on
    plain, SiLU-fused and accumulating launches, with both of its tiles (128 and 256 weight rows)."""
    d = make()
    with _dense_knob("0"):
        want = _every_path(d, 128)
    monkeypatch.setenv("MI_MOE_PREFILL", rows)
    with _dense_knob("1"):
        got = _every_path(d, 128)
        got256 = _every_path(d, 256)
        c = torch.full((d.num_tokens * d.topk, 2 * d.intermediate_size), float("nan"), dtype=d.hidden_states.dtype, device="cuda")
        tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 128, d.num_experts)
        moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c, d.topk_weights, tok, exp, mul_routed_weight=True,
                                    num_token_replicas=d.topk, tile_m=128, tile_n=128, tile_k=64)
        assert ct.last_variant() == ("fused_moe_dense_t128_to160_n256_k64_ring3" if rows == "4" else "fused_moe_dense_t128_to192_n128_k64_ring3")
        assert not torch.isnan(c.float()).any()
    for k in want:
        assert torch.equal(got[k], want[k]), k
        assert torch.equal(got256[k], want[k]), k
    J = orc.to_julia
    ref = orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float64)
    check(J(got["separate"]), ref, 5e-2 if d.hidden_states.dtype == torch.bfloat16 else 2e-2)


@pytest.mark.parametrize("counts,kw,names", [
    # (weight rows per tile as the launch picks them: gate / up 256 and down 256; 256 and 128; down 128 in one round; 256 and 256)
    ([256] * 32, dict(topk=2, hidden_size=1024, intermediate_size=2048), ("silu_", "acc_")),
    ([20, 150, 170, 200, 220, 250, 260, 270, 280, 290, 300, 330, 350, 380, 400, 226] * 2, dict(topk=2, hidden_size=1024, intermediate_size=2048), ("silu_", "acc_")),
    ([120, 344] * 8, dict(topk=1, hidden_size=1024, intermediate_size=2048, T=torch.bfloat16), ("", "acc_")),
    ([560, 1, 900, 219] * 8, dict(topk=2, hidden_size=512, intermediate_size=2048, T=torch.bfloat16), ("silu_", "acc_")),
    # where a few tiles more than CUs would be a round of their own: the ring kernel
    ([305] * 32, dict(topk=2, hidden_size=512, intermediate_size=512), ("", "")),
    ([314] * 16, dict(topk=1, hidden_size=1024, intermediate_size=512), ("", "")),
])
def test_prefill_kernel_picks_its_tiles_from_the_routing(ct, counts, kw, names):
    """Even and uneven routing through the rule as it stands: the streaming kernels' bits whichever tiles a launch picks."""
    d = _routed(counts, **kw)
    with _dense_knob("0"):
        want = _every_path(d, 128)
    got = _every_path(d, 128)
    for k in want:
        assert torch.equal(got[k], want[k]), k
    tok, exp = ct.moe_align_tile_size_device(d.topk_ids, 128, d.num_experts)
    c2 = torch.full((d.num_tokens * d.topk, d.intermediate_size), float("nan"), dtype=d.hidden_states.dtype, device="cuda")
    moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c2, d.topk_weights, tok, exp, mul_routed_weight=False, num_token_replicas=d.topk,
                                tile_m=128, tile_n=128, tile_k=64, fuse_silu=True)
    up = ct.last_variant()
    out = torch.zeros(d.num_tokens, d.hidden_size, dtype=d.hidden_states.dtype, device="cuda")
    ct.fused_moe_accumulate_kernel(c2, d.w2, out, d.topk_weights, tok, exp, 128, 128, 64)
    assert torch.equal(out, want["fused"])
    for name, part in zip((up, ct.last_variant()), names):
        assert ("_to160_" in name and "_or_to192_" in name and part in name) if part else "k32_ring" in name, name


@pytest.mark.parametrize("rows", ["2", "4"])
def test_prefill_kernel_on_arrays_that_no_sort_made(ct, rows, monkeypatch):
    """Slots without a token anywhere in a block, whole blocks without one, blocks of one expert apart from each other, blocks
    without an expert, and rows of C off 16 bytes: what the arrays name is computed, nothing else is written."""
    d = moe.prepare(num_tokens=1500, hidden_size=256, num_experts=5, intermediate_size=160, topk=1)
    rng = np.random.default_rng(3)
    exp = torch.from_numpy(np.array([2, 2, 0, 2, 5, 5, 5, 1, 4, 4, 9, 3, 2], dtype=np.int32)).cuda()
    ids = rng.permutation(1500)[:13 * 128 - 300].astype(np.int32) + 1
    ids = np.concatenate([ids, np.zeros(13 * 128 - ids.size, dtype=np.int32)])
    rng.shuffle(ids)
    ids[128:256] = 0                       # a run whose second block holds nothing
    ids[4 * 128 + 40:5 * 128] = 0          # a first block with one sub-tile and a part, followed by full ones
    ids[7 * 128 + 1:8 * 128] = 0           # a block with one token
    ids[11 * 128:11 * 128 + 100] = 0       # tokens in the last sub-tile only
    tok = torch.from_numpy(ids[:-3].copy()).cuda()   # (the last block ends early)
    def run(knob):
        c = torch.full((1500, 2 * 160 + 4), 7.0, dtype=torch.float16, device="cuda")
        with _dense_knob(knob):
            moe.invoke_fused_moe_kernel(d.hidden_states, d.w1, c[:, :2 * 160], d.topk_weights, tok, exp, mul_routed_weight=False,
                                        num_token_replicas=1, tile_m=128, tile_n=128, tile_k=64)
        return c, ct.last_variant()
    want, _ = run("0")
    monkeypatch.setenv("MI_MOE_PREFILL", rows)
    got, name = run("1")
    assert "_to1" in name
    assert torch.equal(got, want)
