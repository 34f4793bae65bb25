"""Outputs that lie over inputs: the same bits as into buffers of their own.

The attention kernels read rows of vqkv and tqkv while other workgroups write
vattn, so those rows take another way then.
"""
import pytest

from conftest import seeded_awa_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("over", ["vqkv", "tqkv"])
@pytest.mark.parametrize("noalloc", [False, True])
def test_op_in_place(ctx, dtype, over, noalloc):
    import torch
    h, w, txt = 30, 41, 77
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    geom = ctx.build_geometry(1, h, w, (1, 4, 4), txt, 1)
    vqkv, tqkv, gains = seeded_awa_inputs(h * w, txt, 21)
    inputs = {"vqkv": torch.from_numpy(vqkv).cuda().to(dt), "tqkv": torch.from_numpy(tqkv).cuda().to(dt)}
    gains = [torch.from_numpy(g).cuda() for g in gains]
    ref = ctx.forward(geom, inputs["vqkv"], inputs["tqkv"], *gains, eps=1e-5, noalloc=noalloc)
    n, out = inputs[over].numel(), h * w * 2560
    buf = torch.empty(max(n, out), dtype=dt, device="cuda")
    buf[:n] = inputs[over].flatten()
    inputs[over] = buf[:n].view(-1, 7680)
    got = ctx.forward(geom, inputs["vqkv"], inputs["tqkv"], *gains, eps=1e-5, vattn=buf[:out].view(-1, 2560),
                      noalloc=noalloc)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    geom.close()


@pytest.mark.parametrize("over", ["grid", "txt"])
@pytest.mark.parametrize("txt", [90, 500])
def test_embed_in_place(ctx, over, txt):
    import torch
    from test_dit_ends_gpu import make_io
    g = torch.Generator(device="cuda").manual_seed(5)
    _, io = make_io(ctx, g)
    h, w = 40, 50
    inputs = {"grid": torch.randn((1, 2 * h, 2 * w, 33), generator=g, device="cuda"),
              "txt": torch.randn((txt, 5120), generator=g, device="cuda")}
    ref = ctx.embed(io, inputs["grid"], inputs["txt"])
    buf = torch.empty(ref.numel(), device="cuda")
    x, n = inputs[over], inputs[over].numel()
    buf[-n:] = x.flatten()  # under the last rows written
    inputs[over] = buf[-n:].view(x.shape)
    got = ctx.embed(io, inputs["grid"], inputs["txt"], x=buf.view(ref.shape))
    assert torch.equal(got, ref)


@pytest.mark.parametrize("over", ["x", "emb"])
def test_final_in_place(ctx, over):
    import torch
    from test_dit_ends_gpu import make_io
    g = torch.Generator(device="cuda").manual_seed(6)
    _, io = make_io(ctx, g)
    h, w = 40, 50
    x = torch.randn((h * w, 2560), generator=g, device="cuda")
    emb = torch.randn(6 * 2560, generator=g, device="cuda") * 0.02
    ref = ctx.final(io, emb, x, 1, 2 * h, 2 * w)
    n = ref.numel()
    if over == "x":
        out = x.view(-1)[-n:]
    else:
        buf = torch.empty(n, device="cuda")
        buf[n // 2:n // 2 + emb.numel()] = emb
        emb, out = buf[n // 2:n // 2 + emb.numel()], buf
    got = ctx.final(io, emb, x, 1, 2 * h, 2 * w, out=out.view(ref.shape))
    assert torch.equal(got, ref)
