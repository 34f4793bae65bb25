"""GPU tests of the fp32 op's split operands (csrc/awa_sdpa_f32.hip) where its
units, blocks and scales have edges.

Keys run in 32-row units, queries in 16-row blocks of one or two 64-row tiles,
and grids of at most one workgroup per CU split a window's units over two
halves.  Reference: the C oracle in fp32.  Bar 5e-6 (2-norm): both sides carry a
few 2^-24 of the scores' magnitude (up to about 16 in log2 units) into the
exponent, so each is about 1e-6 off, and the bar leaves a factor of two over
their sum.  Scaling V by a power of two scales every block's factor alike, so
the output scales exactly, bit for bit.
"""
import numpy as np
import pytest

from conftest import seeded_awa_inputs

pytestmark = pytest.mark.gpu


def run(ctx, geom, vqkv, tqkv, gains):
    import torch
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    va, ta = ctx.forward(geom, dev(vqkv), dev(tqkv), *[dev(g) for g in gains], eps=1e-5)
    torch.cuda.synchronize()
    return va.cpu().numpy(), ta.cpu().numpy()


def rel(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# one window of h x w rows: 1 unit, a full unit, one row into the next, whole and
# odd tiles; two windows per axis and enough of them for the unsplit form
@pytest.mark.parametrize("h,w,nw,txt", [(1, 1, (1, 1, 1), 1), (1, 31, (1, 1, 1), 32), (4, 8, (1, 1, 1), 33),
                                        (3, 11, (1, 1, 1), 64), (8, 16, (1, 1, 1), 65), (13, 5, (1, 1, 1), 31),
                                        (10, 29, (1, 2, 2), 58), (30, 41, (1, 4, 4), 77)])
@pytest.mark.parametrize("shifted", [0, 1])
def test_f32_edges(oracle, ctx, h, w, nw, txt, shifted):
    geom = ctx.build_geometry(1, h, w, nw, txt, shifted)
    og = oracle.Geometry(1, h, w, nw, txt, shifted)
    vqkv, tqkv, gains = seeded_awa_inputs(h * w, txt, 100 * h + w)
    ref = oracle.awa_forward(vqkv, tqkv, og, *gains, eps=1e-5)
    for a, b in zip(run(ctx, geom, vqkv, tqkv, gains), ref):
        assert rel(a, b) <= 5e-6
    geom.close()


@pytest.mark.parametrize("k", [-90, -20, 20, 90])
def test_v_scales_exactly(ctx, k):
    """Far outside fp16's range, V's scale only moves the blocks' exponents."""
    geom = ctx.build_geometry(1, 10, 29, (1, 2, 2), 58, 1)
    vqkv, tqkv, gains = seeded_awa_inputs(290, 58, 5)
    base = run(ctx, geom, vqkv, tqkv, gains)
    for x in (vqkv, tqkv):
        x[:, 5120:] *= np.float32(2.0 ** k)
    for a, b in zip(run(ctx, geom, vqkv, tqkv, gains), base):
        assert np.array_equal(a, b * np.float32(2.0 ** k))
    geom.close()


def test_mixed_scales(oracle, ctx):
    """Row blocks of V 2^24 apart, single values 2^12 above their block, all-zero
    rows of q, k and v, and gains far from 1."""
    h, w, txt = 9, 23, 40
    geom = ctx.build_geometry(1, h, w, (1, 1, 1), txt, 0)
    og = oracle.Geometry(1, h, w, (1, 1, 1), txt, 0)
    vqkv, tqkv, gains = seeded_awa_inputs(h * w, txt, 9)
    vqkv[40:60, 5120:] *= 2.0 ** 24
    vqkv[100, 5120::128] *= 2.0 ** 12
    vqkv[7] = 0
    tqkv[3] = 0
    # q and k gains of video and text together: scores keep their size (with one
    # of them alone text queries' scores reach 2^15, where the reference overflows)
    for i, e in enumerate((-15, 15, -15, 15)):
        gains[i] *= 2.0 ** e
    ref = oracle.awa_forward(vqkv, tqkv, og, *gains, eps=1e-5)
    for a, b in zip(run(ctx, geom, vqkv, tqkv, gains), ref):
        assert np.isfinite(a).all() and rel(a, b) <= 5e-6
    geom.close()


# one window (two halves of its units) and sixteen (the unsplit form); 40 and 77
# text rows leave a partly filled unit
SPLIT, UNSPLIT = (9, 23, (1, 1, 1), 40), (30, 41, (1, 4, 4), 77)


def both(oracle, ctx, shape, change, seed=11):
    """The op and the oracle on seeded inputs after change(vqkv, tqkv, gains)."""
    h, w, nw, txt = shape
    geom = ctx.build_geometry(1, h, w, nw, txt, 0)
    og = oracle.Geometry(1, h, w, nw, txt, 0)
    vqkv, tqkv, gains = seeded_awa_inputs(h * w, txt, seed)
    change(vqkv, tqkv, gains)
    got = run(ctx, geom, vqkv, tqkv, gains)
    geom.close()
    return got, oracle.awa_forward(vqkv, tqkv, og, *gains, eps=1e-5)


@pytest.mark.parametrize("shape", [SPLIT, UNSPLIT])
@pytest.mark.parametrize("zero", ["text_qk", "text", "video_qk", "video", "qk", "all"])
def test_zero_rows(oracle, ctx, shape, zero):
    """Whole blocks of zero queries and keys: equal weights, with masked keys at weight 0."""
    def change(vqkv, tqkv, gains):
        n = 5120 if zero.endswith("qk") else 7680
        if not zero.startswith("text"):
            vqkv[:, :n] = 0
        if not zero.startswith("video"):
            tqkv[:, :n] = 0
    for a, b in zip(*both(oracle, ctx, shape, change)):
        if zero == "all":
            assert not a.any()
        else:
            assert np.isfinite(a).all() and rel(a, b) <= 5e-6


def worst_channel(a, b):
    """Largest relative 2-norm error of one channel of one head over the rows."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    return float((np.linalg.norm(a - b, axis=0) / np.linalg.norm(b, axis=0)).max())


@pytest.mark.parametrize("shape", [SPLIT, UNSPLIT])
@pytest.mark.parametrize("e", [0, 6, 12, 24, 32, 60])
def test_one_large_v(oracle, ctx, shape, e):
    """Channels do not depend on each other: one element of V 2^e times as large
    leaves every other channel as accurate as before.  Bar 1e-5 per channel:
    the 5e-6 above, and a factor of two for the worst of 2,560 channels."""
    def change(vqkv, tqkv, gains):
        vqkv[101, 5120 + 128 * 3 + 17] *= np.float32(2.0 ** e)
    for a, b in zip(*both(oracle, ctx, shape, change)):
        assert worst_channel(a, b) <= 1e-5


@pytest.mark.parametrize("shape", [SPLIT, UNSPLIT])
def test_small_channels(oracle, ctx, shape):
    """Channels of V of very different sizes, side by side and from row to row."""
    def change(vqkv, tqkv, gains):
        for x in (vqkv, tqkv):
            x[:, 5120:] *= np.exp2(np.arange(2560) % 40 - 20).astype(np.float32)
        vqkv[150:170, 5120:] *= np.float32(2.0 ** -18)
    for a, b in zip(*both(oracle, ctx, shape, change)):
        assert worst_channel(a, b) <= 1e-5


@pytest.mark.parametrize("shape", [SPLIT, UNSPLIT])
def test_infinite_v(oracle, ctx, shape):
    """An infinity in V is an infinity in its channel of the rows that see it."""
    def change(vqkv, tqkv, gains):
        vqkv[101, 5120 + 17] = np.inf
        vqkv[33, 5120 + 128 * 7 + 90] = -np.inf
        tqkv[5, 5120 + 128 * 9 + 3] = np.inf
    for a, b in zip(*both(oracle, ctx, shape, change)):
        assert np.isinf(b).any() and np.array_equal(np.isinf(a), np.isinf(b)) and not np.isnan(a).any()
        fin = np.isfinite(b)
        assert np.array_equal(a[~fin], b[~fin]) and rel(a[fin], b[fin]) <= 5e-6


@pytest.mark.parametrize("shape", [SPLIT, UNSPLIT])
def test_opposite_gains(oracle, ctx, shape):
    """Gains of q and k that cancel channel by channel: the scores are as before."""
    def change(vqkv, tqkv, gains):
        s = np.exp2(4.0 * (np.arange(128) // 2 % 9 - 4)).astype(np.float32)
        for i in range(4):
            gains[i] = (gains[i] * (s if i % 2 == 0 else 1 / s)).astype(np.float32)
    for a, b in zip(*both(oracle, ctx, shape, change)):
        assert worst_channel(a, b) <= 1e-5


@pytest.mark.parametrize("shape", [SPLIT, UNSPLIT])
@pytest.mark.parametrize("small,large", [(-98, 0), (-110, 0), (-60, 60), (-112, -112)])
def test_ends_of_the_range(oracle, ctx, shape, small, large):
    """Channels of V near both ends of fp32's range, alone and side by side."""
    def change(vqkv, tqkv, gains):
        for x in (vqkv, tqkv):
            x[:, 5120::2] *= np.float32(2.0 ** small)
            x[:, 5121::2] *= np.float32(2.0 ** large)
    for a, b in zip(*both(oracle, ctx, shape, change)):
        assert worst_channel(a, b) <= 1e-5


@pytest.mark.parametrize("h,w,nw,txt", [(1, 1, (1, 1, 1), 1), (1, 31, (1, 1, 1), 32), (4, 8, (1, 1, 1), 33),
                                        (3, 11, (1, 1, 1), 64), (8, 16, (1, 1, 1), 65), (13, 5, (1, 1, 1), 31),
                                        (10, 29, (1, 2, 2), 58), (30, 41, (1, 4, 4), 77)])
@pytest.mark.parametrize("kind", ["wide", "full"])
def test_wide_edges(oracle, ctx, h, w, nw, txt, kind):
    """The paths of windows that the split does not hold, at the edges of their
    units and halves: channels of V 2^24 apart, and gains that cancel."""
    def change(vqkv, tqkv, gains):
        s = np.exp2(12.0 * (np.arange(128) // 2 % 3 - 1)).astype(np.float32)
        if kind == "wide":
            for x in (vqkv, tqkv):
                x[:, 5120:] *= np.tile(s, 20)
        else:
            for i in range(4):
                gains[i] = (gains[i] * (s if i % 2 == 0 else 1 / s)).astype(np.float32)
    for a, b in zip(*both(oracle, ctx, (h, w, nw, txt), change, seed=100 * h + w)):
        assert rel(a, b) <= 5e-6


@pytest.mark.parametrize("txt", [9, 77])
@pytest.mark.parametrize("kind", ["split", "wide", "full"])
def test_text_tables_per_window(oracle, ctx, txt, kind):
    """Windows with a text RoPE table (and so text tiles) of their own, one of them
    without video rows, on each path."""
    import types
    og = oracle.Geometry(1, 23, 27, (4, 3, 3), txt, 0)
    sl = np.insert(og.slices, 2, [0, 1, 5, 5, 0, 27], axis=0).astype(np.int32)
    nwin = og.nwin + 1
    tf = np.concatenate([og.txt_freq[:txt] * np.float32(1 + 0.25 * w) for w in range(nwin)])
    geo = types.SimpleNamespace(t=1, h=23, w=27, Lv=og.Lv, txt_len=txt, slices=sl, nwin=nwin, vid_freq=og.vid_freq,
                                txt_freq=np.ascontiguousarray(tf))
    g = ctx.geometry_from_win(1, 23, 27, sl, og.vid_freq, geo.txt_freq, txt)
    vqkv, tqkv, gains = seeded_awa_inputs(og.Lv, txt, 90 + txt)
    s = np.exp2(12.0 * (np.arange(128) // 2 % 3 - 1)).astype(np.float32)
    if kind == "wide":
        for x in (vqkv, tqkv):
            x[:, 5120:] *= np.tile(s, 20)
    elif kind == "full":
        for i in range(4):
            gains[i] = (gains[i] * (s if i % 2 == 0 else 1 / s)).astype(np.float32)
    ref = oracle.awa_forward(vqkv, tqkv, geo, *gains, eps=1e-5)
    for a, b in zip(run(ctx, g, vqkv, tqkv, gains), ref):
        assert np.isfinite(a).all() and rel(a, b) <= 5e-6
    g.close()


@pytest.mark.parametrize("shape", [SPLIT, UNSPLIT])
@pytest.mark.parametrize("e", [5, 12, 20, 28])
def test_large_rows_of_small_weight(oracle, ctx, shape, e):
    """Rows of V 2^e times the others, every eighth (so in every block), that all
    queries give a weight of about 2^-30: q and k agree in channel 126 (which no
    rotation touches), those rows' k has the other sign.  Scores of 15 in log2 units,
    rounded at 2^-20, leave up to 3e-5 in the worst channel of either side: bar 1e-4."""
    def change(vqkv, tqkv, gains):
        for x in (vqkv, tqkv):
            x[:, 126:2560:128] = 40
            x[:, 2560 + 126:5120:128] = 40
            x[::8, 2560 + 126:5120:128] = -40
            x[::8, 5120:] *= np.float32(2.0 ** e)
    for a, b in zip(*both(oracle, ctx, shape, change)):
        assert worst_channel(a, b) <= 1e-4


@pytest.mark.parametrize("gain", [1, 8, 48])
def test_large_gains(ctx, gain):
    """Gains far from 1 in every channel stay on the split operands.  Against the
    fp32 path, which an infinity in one V channel of every head takes (the oracle's
    exponentials overflow here): scores of up to 6 gain^2 in log2 units, off by a few
    2^-24 of that on both sides, in a softmax that few keys share."""
    h, w, nw, txt = SPLIT
    geom = ctx.build_geometry(1, h, w, nw, txt, 0)
    vqkv, tqkv, gains = seeded_awa_inputs(h * w, txt, 13)
    gains = [g * np.float32(gain) for g in gains]
    a = run(ctx, geom, vqkv, tqkv, gains)
    vqkv[101, 5120::128] = np.inf
    b = run(ctx, geom, vqkv, tqkv, gains)
    keep = np.arange(2560) % 128 != 0
    for x, y in zip(a, b):
        assert np.isfinite(x).all() and rel(x[:, keep], y[:, keep]) <= 2e-6 * gain
    geom.close()
