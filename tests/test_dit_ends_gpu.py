"""GPU tests of the model's ends (csrc/dit_ends.hip) at the edges of their tiles.

The embedding's tiles are 64 video rows and 64 text rows; the output layer's
workgroups hold ceil(rows / CUs) rows in one or two blocks of 16 (two from
16 x 256 + 1 rows on, several rounds past 32 x 256).  References in fp64 from
the same bf16 operands.  Embedding bar: fp32 sums of up to 5120 terms, error
about sqrt(5120) 2^-24 = 4e-6 of the result, 1e-5.  Output layer: the
normalised row is rounded to bf16 after an fp32 scale that may differ from the
reference's by an ulp (2^-23), so about one value in 2^14 falls to the other
side of a rounding boundary, 2^-8 of itself away: sqrt(2^-14) 2^-8 = 3e-5 of
the result, bar 1e-4.
"""
import pytest

pytestmark = pytest.mark.gpu

DIM = 2560


def make_io(ctx, g):
    import torch
    r = lambda *s, scale=0.02: torch.randn(s, generator=g, device="cuda") * scale
    bf = torch.bfloat16
    w = {"vid_in_w": r(DIM, 132).to(bf), "vid_in_b": r(DIM), "txt_in_w": r(DIM, 5120).to(bf), "txt_in_b": r(DIM),
         "out_norm_w": 1 + r(DIM), "out_ada_shift": r(DIM), "out_ada_scale": 1 + r(DIM),
         "vid_out_w": r(64, DIM).to(bf), "vid_out_b": r(64)}
    return w, ctx.io_layers(w)


def rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("t,h,w,txt", [(1, 1, 1, 1), (1, 7, 9, 63), (2, 4, 8, 64), (1, 5, 13, 65), (3, 9, 11, 140)])
def test_embed_edges(ctx, t, h, w, txt):
    import torch
    g = torch.Generator(device="cuda").manual_seed(7 * h + txt)
    wts, io = make_io(ctx, g)
    grid = torch.randn((t, 2 * h, 2 * w, 33), generator=g, device="cuda")
    text = torch.randn((txt, 5120), generator=g, device="cuda")
    x = torch.full((t * h * w + txt + 1, DIM), 7.0, device="cuda")  # one guard row
    ctx.embed(io, grid, text, x=x)
    p = grid.reshape(t, h, 2, w, 2, 33).permute(0, 1, 3, 2, 4, 5).reshape(-1, 132).bfloat16().double()
    ref = torch.cat([p @ wts["vid_in_w"].double().T + wts["vid_in_b"].double(),
                     text.bfloat16().double() @ wts["txt_in_w"].double().T + wts["txt_in_b"].double()])
    assert rel(x[:-1], ref) <= 1e-5
    assert bool((x[-1] == 7.0).all())


@pytest.mark.parametrize("t,h,w", [(1, 1, 1), (1, 16, 17), (2, 3, 5), (1, 64, 64), (1, 17, 241), (1, 91, 91)])
def test_final_edges(ctx, t, h, w):
    """1 to 8281 rows: one row per workgroup, 16 (the last of the one-block form), 17 (4097 rows) and two rounds."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(h + w)
    wts, io = make_io(ctx, g)
    n = t * h * w
    x = torch.randn((n, DIM), generator=g, device="cuda")
    emb = torch.randn(6 * DIM, generator=g, device="cuda") * 0.02
    out = ctx.final(io, emb, x, t, 2 * h, 2 * w)
    d = x.double()
    y = d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5)
    sc = wts["out_norm_w"] * (emb[1::6] + wts["out_ada_scale"])
    y = (y * sc.double() + (emb[0::6] + wts["out_ada_shift"]).double()).bfloat16().double()
    y = y @ wts["vid_out_w"].double().T + wts["vid_out_b"].double()
    ref = y.reshape(t, h, w, 2, 2, 16).permute(0, 1, 3, 2, 4, 5).reshape(t, 2 * h, 2 * w, 16)
    assert rel(out, ref) <= 1e-4


@pytest.mark.parametrize("txt", [320, 321, 700])
def test_embed_long_text(ctx, txt):
    """Either side of the length from which the block's GEMM projects the text."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(txt)
    wts, io = make_io(ctx, g)
    grid = torch.randn((1, 6, 14, 33), generator=g, device="cuda")
    text = torch.randn((txt, 5120), generator=g, device="cuda")
    x = torch.full((21 + txt + 1, DIM), 7.0, device="cuda")  # one guard row
    ctx.embed(io, grid, text, x=x)
    p = grid.reshape(1, 3, 2, 7, 2, 33).permute(0, 1, 3, 2, 4, 5).reshape(-1, 132).bfloat16().double()
    ref = torch.cat([p @ wts["vid_in_w"].double().T + wts["vid_in_b"].double(),
                     text.bfloat16().double() @ wts["txt_in_w"].double().T + wts["txt_in_b"].double()])
    assert rel(x[:21], ref[:21]) <= 1e-5 and rel(x[21:-1], ref[21:]) <= 1e-5
    assert bool((x[-1] == 7.0).all())
