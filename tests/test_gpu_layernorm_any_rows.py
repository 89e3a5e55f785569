"""LayerNorm on rows that are no multiple of four elements or lie off 16 bytes: forward and backward walk them in groups of
four like the others, and the group across the end is the row's last four elements less those that the group before has.
Lengths around the groups (4 elements), the kernels' borders (256, 512, 1024, 2048, 4096, 8192) and the smallest (4, and 3,
which stays element by element).

Tolerances.  Against float64: |got - ref| <= 1e-5 * (|ref| + max|ref|), as the other LayerNorm tests; sums of M rows of fp32
products err by at most about M * 2^-24 of the sum of magnitudes, far inside it at the M used here.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def close(got, ref, what):
    got, ref = got.double().cpu(), ref.double().cpu()
    bound = 1e-5 * (ref.abs() + ref.abs().max())
    assert bool(torch.all((got - ref).abs() <= bound)), f"{what}: worst {((got - ref).abs() / bound).max():.2f} of the bound"


def padded(M, N, lead, off, fill):
    """(M, N) rows with leading dimension `lead`, `off` elements into their memory; everything around them is `fill`."""
    base = torch.full((M * lead + off + 8,), fill, device="cuda")
    return base, base[off:off + M * lead].view(M, lead)[:, :N]


def untouched(base, view, fill):
    mask = torch.ones_like(base, dtype=torch.bool)
    mask.as_strided(view.shape, view.stride(), view.storage_offset()).fill_(False)
    rest = base[mask]
    return bool(torch.isnan(rest).all()) if fill != fill else bool((rest == fill).all())


@pytest.mark.parametrize("M,N,G,pad,off", [
    (3, 3, 2, 0, 0), (9, 4, 2, 1, 0), (17, 5, 4, 0, 0), (17, 6, 4, 1, 3), (33, 7, 1, 2, 1), (40, 8, 3, 0, 2),
    (64, 253, 8, 0, 0), (65, 255, 8, 0, 1), (70, 256, 8, 1, 0), (71, 257, 64, 0, 0), (300, 258, 8, 3, 2),
    (130, 510, 8, 0, 0), (131, 513, 2, 0, 3), (90, 1023, 64, 0, 0), (91, 1025, 8, 2, 0), (40, 1026, 4, 0, 1),
    (41, 2047, 2, 0, 0), (42, 2049, 8, 0, 0), (37, 2050, 1, 5, 0), (38, 4095, 4, 0, 0), (39, 4097, 2, 0, 2), (21, 4098, 8, 1, 0),
    (9, 8191, 2, 0, 0), (20, 8190, 1, 0, 1), (10, 8192, 2, 3, 1), (9, 8193, 2, 0, 0),
    (16384, 5, 64, 0, 0), (16390, 257, 64, 0, 0), (16385, 1022, 64, 1, 3), (3073, 2049, 64, 0, 0), (2050, 4099, 64, 0, 1),   # the forward kernels that walk
    (1025, 8195, 64, 2, 0), (3584, 8195, 64, 0, 1),   # over several rows
])
def test_rows_of_any_length_and_alignment(ct, M, N, G, pad, off):
    g = torch.Generator(device="cuda").manual_seed(M * 10007 + N)
    nan, eps, lead = float("nan"), 1e-5, N + pad
    xb, X = padded(M, N, lead, off, nan)          # NaN around what is read: an element too many shows
    dyb, DY = padded(M, N, lead, (off * 3) % 4, nan)
    yb, Y = padded(M, N, lead, off, 7.0)          # and 7 around what is written
    dxb, DX = padded(M, N, lead, (off + 1) % 4 if off else 0, 7.0)
    wb, W = padded(1, N, N, off, nan)
    bb, B = padded(1, N, N, off, nan)
    for t in (X, DY, W, B):
        t.copy_(torch.randn(t.shape, device="cuda", generator=g))
    W, B = W[0], B[0]
    X += 0.5
    Mean, Rstd = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    DWb, DW = padded(G, N, lead, 0, 0.0)
    DBb, DB = padded(G, N, lead, 0, 0.0)
    locks = torch.zeros(G, dtype=torch.int64, device="cuda")
    ct.layer_norm_fwd(X, W, B, Y, Mean, Rstd, eps, 1024)
    ct.layer_norm_bwd_dx_partial_dwdb(DX, DY, DW, DB, X, W, Mean, Rstd, locks, G, 1024)
    x, dy, w, b = (t.double().cpu() for t in (X, DY, W, B))
    mean = x.mean(1)
    rstd = 1 / ((x - mean[:, None]).square().mean(1) + eps).sqrt()
    xhat = (x - mean[:, None]) * rstd[:, None]
    assert ct.last_variant().startswith("ln_bwd_regs_b512_v") == (4 <= N <= 8192), ct.last_variant()
    close(Mean, mean, "mean")
    close(Rstd, rstd, "rstd")
    close(Y, xhat * w + b, "y")
    wdy = w * dy
    c1, c2 = (xhat * wdy).mean(1, keepdim=True), wdy.mean(1, keepdim=True)
    close(DX, (wdy - (xhat * c1 + c2)) * rstd[:, None], "dx")
    slot = torch.arange(M) % G
    close(DW, torch.zeros(G, N, dtype=torch.float64).index_add_(0, slot, dy * xhat), "partial dw")
    close(DB, torch.zeros(G, N, dtype=torch.float64).index_add_(0, slot, dy), "partial db")
    assert untouched(yb, Y, 7.0) and untouched(dxb, DX, 7.0) and untouched(DWb, DW, 0.0) and untouched(DBb, DB, 0.0)
    assert untouched(xb, X, nan) and untouched(dyb, DY, nan)


@pytest.mark.parametrize("M,N,G,kernel", [(256, 1001, 64, "v1_rg2"), (257, 1001, 64, "v4_rg8"), (8, 513, 4, "v1_rg2"), (17, 1023, 4, "v4_rg8"),
                                          (256, 511, 64, "v2_rg8"), (400, 1025, 64, "v2_rg2")])
def test_which_groups_walk_rows_off_16_bytes(ct, M, N, G, kernel):
    """513 to 1024 elements: a wave per group from five rows a slot on."""
    X, DY, DX = (torch.randn(M, N, device="cuda") for _ in range(3))
    W, mean, rstd = torch.randn(N, device="cuda"), X.mean(1), 1 / X.std(1)
    dw, db = torch.zeros(2, G, N, device="cuda")
    ct.layer_norm_bwd_dx_partial_dwdb(DX, DY, dw, db, X, W, mean, rstd, torch.zeros(G, dtype=torch.int64, device="cuda"), G, 1024)
    assert ct.last_variant() == "ln_bwd_regs_b512_" + kernel, ct.last_variant()
    close(db.sum(0), DY.double().sum(0), "db")
