"""The attention kernel for launches of few queries, whose waves share the keys of 32 queries (csrc/fmha_few.hip): stand-in for the
reference's examples/fmha.jl:20-139."""
import math

import pytest

torch = pytest.importorskip("torch")

from cutile_jl_amd.examples import fmha

pytestmark = pytest.mark.gpu


def _reference(Q, K, V, pos, causal):
    q, k, v = Q.double(), K.double(), V.double()
    g = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(q.shape[3])
    if causal:
        i, j = torch.arange(q.shape[2], device=q.device)[:, None], torch.arange(k.shape[2], device=q.device)[None]
        s.masked_fill_(j > i + pos, -math.inf)
    return torch.matmul(s.softmax(-1), v)


def _err(got, ref):
    return ((got.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("T", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,KVH,sq,skv,pos,causal", [
    # edges of the tiles of 32 queries and of the halves of 32 keys; fewer halves than waves; whole and part-filled last halves
    (1, 4, 4, 65, 65, 0, True), (2, 4, 2, 96, 96, 0, True), (1, 8, 2, 127, 127, 0, True), (1, 8, 8, 129, 129, 0, False),
    (3, 3, 1, 160, 160, 0, True), (1, 4, 4, 256, 256, 0, False), (2, 8, 2, 319, 319, 0, True), (1, 4, 1, 705, 705, 0, True),
    (1, 2, 2, 1023, 1023, 0, False),
    # more keys than queries (with and without an offset that hides some), fewer, and fewer than a half
    (1, 4, 4, 70, 200, 130, True), (1, 4, 2, 100, 333, 50, True), (2, 4, 4, 66, 33, 0, False), (1, 4, 4, 80, 40, 0, True),
])
def test_few_queries(ct, dim, T, B, H, KVH, sq, skv, pos, causal):
    """Against float64, no further off than the general kernel; views of a packed buffer with NaN around the rows that exist."""
    g = torch.Generator(device="cuda").manual_seed(sq + skv)
    def view(h, s):
        buf = torch.full((B, h, s + 2, dim + 8), float("nan"), dtype=T, device="cuda")
        v = buf[:, :, 1:s + 1, :dim]
        v.copy_(torch.empty(B, h, s, dim, device="cuda").normal_(0, 1.5, generator=g))
        return v
    Q, K, V = view(H, sq), view(KVH, skv), view(KVH, skv)
    ref = _reference(Q, K, V, pos, causal)
    got = fmha.cutile_fmha(Q, K, V, input_pos=pos, query_group_size=H // KVH, causal=causal)
    if skv >= 32:
        assert ct.last_variant().startswith(f"fmha_few_d{dim}_q32_keys"), ct.last_variant()
    assert not torch.isnan(got.float()).any()
    # (2^-9 of the weights and 2^-9 of the result at worst for bf16, 2^-12 for f16; weights of one sign add up to less)
    assert _err(got, ref) <= (2**-8 if T == torch.bfloat16 else 2**-11)


@pytest.mark.parametrize("dim,B,H,S,waves", [(64, 1, 4, 1408, 4), (64, 2, 32, 755, 2), (128, 1, 4, 1408, 4), (128, 6, 8, 576, 2)])
def test_few_queries_is_no_further_off_than_the_kernels_it_replaces(ct, monkeypatch, dim, B, H, S, waves):
    """Both numbers of waves, normal and peaked scores."""
    for std in (1.0, 3.0):
        g = torch.Generator(device="cuda").manual_seed(S)
        Q, K, V = (torch.empty(B, H, S, dim, device="cuda", dtype=torch.bfloat16).normal_(0, s, generator=g) for s in (std, 1.0, 1.0))
        got = fmha.cutile_fmha(Q, K, V, causal=True)
        assert ct.last_variant() == f"fmha_few_d{dim}_q32_keys{waves}", ct.last_variant()
        again = fmha.cutile_fmha(Q, K, V, causal=True)
        assert torch.equal(got, again)
        monkeypatch.setenv("MI_FMHA_FEW", "0")
        old = fmha.cutile_fmha(Q, K, V, causal=True)
        assert not ct.last_variant().startswith("fmha_few")
        monkeypatch.delenv("MI_FMHA_FEW")
        ref = _reference(Q, K, V, 0, True)
        assert _err(got, ref) <= (0.8 if dim == 64 else 1.0) * _err(old, ref)


@pytest.mark.parametrize("dim,B,H,sq,skv,few", [
    (64, 1, 4, 64, 640, False), (64, 1, 4, 65, 640, True), (64, 1, 1, 128, 5120, True), (64, 1, 1, 128, 5121, False),
    # the walk of a wave by itself against a split (2 heads, 5120 keys 24 us : 15.9), and the kernels that walk few keys
    (64, 1, 2, 128, 5120, False), (64, 1, 2, 128, 2700, True), (64, 1, 16, 512, 5120, True), (64, 1, 16, 512, 5121, False), (64, 4, 64, 331, 41, False), (128, 2, 8, 2375, 57, False),
    # not causal with other keys: two groups of waves, 59 us : 70
    (128, 1, 32, 838, 3111, False),
    (128, 1, 1, 128, 5121, False), (64, 8, 32, 1024, 1024, False), (128, 4, 32, 1024, 1024, False), (128, 1, 32, 1280, 1280, False),
    # walks of one length: 512 workgroups are one round, 576 leave a nearly empty second one
    (128, 1, 8, 2048, 1619, True), (128, 1, 8, 2282, 1619, False), (128, 1, 8, 136, 2396, False), (128, 1, 8, 136, 1000, True),
])
def test_both_sides_of_the_rule(ct, dim, B, H, sq, skv, few):
    g = torch.Generator(device="cuda").manual_seed(sq + skv)
    Q, K, V = (torch.empty(B, H, s, dim, device="cuda", dtype=torch.float16).normal_(0, 1, generator=g) for s in (sq, skv, skv))
    got = fmha.cutile_fmha(Q, K, V, causal=False)
    assert ct.last_variant().startswith("fmha_few") == few, ct.last_variant()
    assert _err(got[:1, :4], _reference(Q[:1, :4], K[:1, :4], V[:1, :4], 0, False)) <= 2**-10


@pytest.mark.parametrize("B,H,sq,skv,pos,few", [(1, 32, 1943, 555, 0, False), (16, 8, 268, 1612, 1344, False), (2, 4, 300, 555, 255, True)])
def test_both_sides_of_the_rule_causal_with_other_keys(ct, B, H, sq, skv, pos, few):
    """Heads of 128: walks of one length, which the pipelined kernel is ahead on."""
    g = torch.Generator(device="cuda").manual_seed(sq + skv)
    Q, K, V = (torch.empty(B, H, s, 128, device="cuda", dtype=torch.float16).normal_(0, 1, generator=g) for s in (sq, skv, skv))
    got = fmha.cutile_fmha(Q, K, V, input_pos=pos, causal=True)
    assert ct.last_variant().startswith("fmha_few" if few else "fmha_pipe_d128"), ct.last_variant()
    assert _err(got[:1, :4], _reference(Q[:1, :4], K[:1, :4], V[:1, :4], pos, True)) <= 2**-10


def test_few_queries_infinities_and_nan(ct):
    """A NaN in a key reaches the queries that see it and no others."""
    g = torch.Generator(device="cuda").manual_seed(3)
    Q, K, V = (torch.empty(1, 4, 200, 64, device="cuda", dtype=torch.float16).normal_(0, 1, generator=g) for _ in range(3))
    clean = fmha.cutile_fmha(Q, K, V, causal=True)
    assert ct.last_variant().startswith("fmha_few")
    K[0, 1, 70, 5] = float("nan")
    got = fmha.cutile_fmha(Q, K, V, causal=True)
    bad = torch.isnan(got.float()).any(-1)[0]
    assert bad[1, 70:].all() and not bad[1, :70].any() and not bad[[0, 2, 3]].any()
    assert torch.equal(got[0, 1, :70], clean[0, 1, :70])


@pytest.mark.parametrize("dim", [64, 128])
def test_few_queries_infinities_of_both_head_sizes(ct, dim):
    """A NaN or a score of either infinity reaches the queries that see it and no others, an infinite value likewise."""
    g = torch.Generator(device="cuda").manual_seed(3)
    Q, K, V = (torch.empty(1, 4, 200, dim, device="cuda", dtype=torch.float16).normal_(0, 1, generator=g) for _ in range(3))
    Q[..., 5] = Q[..., 5].abs() + 0.25
    def attend(K, V):
        got = fmha.cutile_fmha(Q, K, V, causal=True)
        assert ct.last_variant().startswith(f"fmha_few_d{dim}")
        return got
    clean = attend(K, V)
    for value in (float("nan"), float("inf")):
        k = K.clone(); k[0, 1, 70, 5] = value                       # (a score of +inf: inf - inf)
        got = attend(k, V)
        bad = torch.isnan(got.float()).any(-1)[0]
        assert bad[1, 70:].all() and not bad[1, :70].any() and not bad[[0, 2, 3]].any()
        assert torch.equal(got[0, 1, :70], clean[0, 1, :70])
    k = K.clone(); k[0, 1, 70, 5] = float("-inf")                   # a weight of zero
    got = attend(k, V)
    keep = [i for i in range(200) if i != 70]
    ref = _reference(Q[:, 1:2, 71:], K[:, 1:2, keep].contiguous(), V[:, 1:2, keep].contiguous(), 70, True)
    assert _err(got[:, 1:2, 71:], ref) <= 2**-11 and torch.equal(got[0, 1, :70], clean[0, 1, :70])
    v = V.clone(); v[0, 1, 70, 9] = float("inf")
    got = attend(K, v)
    assert (got[0, 1, 70:, 9] == float("inf")).all()
    got[0, 1, 64:, 9] = clean[0, 1, 64:, 9]                         # (queries that walk its half without seeing it: 0 * inf)
    assert torch.equal(got, clean)


@pytest.mark.parametrize("T", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,B,H,S,waves", [(64, 1, 4, 1408, 4), (64, 2, 32, 755, 2), (128, 1, 4, 1408, 4), (128, 6, 8, 576, 2)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("levels", [
    (0, 20, -30, 10, 25, -60, 24), (25, 0), (0, 25), (-40, -38, -36, -34, -32, -30, -28, -26), (24, 18, 12, 6, 0, -6, -12, -18),
    (20, -45, 20, -45), (3, -3),
], ids=["up_down_up", "down", "up", "rising", "falling", "every_second", "within_the_limit"])
def test_few_queries_scores_that_rise_and_fall_from_half_to_half(ct, dim, B, H, S, waves, T, causal, levels):
    """Each half of 32 keys has scores around a level of its own, the levels repeating along the keys (in units of log 2 up to 36 and
    -87 apart): what a wave's reference follows up, and heads of 128 down as far as 2^-8 of the largest weight."""
    g = torch.Generator(device="cuda").manual_seed(S)
    Q, K, V = (torch.empty(B, H, S, dim, device="cuda").normal_(0, 1, generator=g) for _ in range(3))
    Q[..., 0] = math.sqrt(dim)
    K[..., 0] = torch.tensor([float(levels[(k // 32) % len(levels)]) for k in range(S)], device="cuda")
    Q, K, V = (x.to(T) for x in (Q, K, V))
    got = fmha.cutile_fmha(Q, K, V, causal=causal)
    if causal:
        assert ct.last_variant() == f"fmha_few_d{dim}_q32_keys{waves}", ct.last_variant()
    # (the bounds of test_few_queries)
    assert _err(got, _reference(Q, K, V, 0, causal)) <= (2**-8 if T == torch.bfloat16 else 2**-11)
