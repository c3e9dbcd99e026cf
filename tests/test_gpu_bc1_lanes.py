"""GPU parity of the two-pass BC1 Level8 encoder (bc1_classify_kernel +
bc1_search_kernel, 1 to 8 lanes per block over blocks bucketed by colour
count).

A context with the threshold at one block sends every image through it; the
checks are the same as for the one-pass encoder: the reference icbc's golden
blocks, the oracle on adversarial blocks and seeded images (byte for byte),
the per-block colour counts (n, m) against the oracle's, and the two
encoders against each other on larger images."""
import ctypes
import os

import numpy as np
import pytest

import blocks
import ntx_amd as N
from capture import Capture
from ntx_amd import synth

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")


@pytest.fixture(scope="module")
def lanes():
    ctx = N.Context(0)
    ctx.set_bc1_lanes_min(1)
    yield ctx
    ctx.close()


def _blocks_as_image(cols, wts):
    n = len(cols)
    img = np.zeros((4, 4, 4 * n), np.float32)
    for i in range(n):
        for t in range(16):
            y, x = divmod(t, 4)
            img[:3, y, 4 * i + x] = cols[i, t, :3]
            img[3, y, 4 * i + x] = wts[i, t]
    return img, 4 * n, 4


def _diff(a, b):
    return int(np.sum(np.any(a.reshape(-1, 8) != b.reshape(-1, 8), axis=1)))


def test_golden_blocks(lanes):
    """2048 blocks written by the reference's own icbc at Level8."""
    g = np.load(os.path.join(GOLD, "bc1_blocks.npz"))
    cws = g["color_weights"]
    bad = 0
    for key in {tuple(c) for c in cws}:
        sel = np.nonzero(np.all(cws == np.array(key, np.float32), axis=1))[0]
        img, w, h = _blocks_as_image(g["colors"][sel], g["weights"][sel])
        out = lanes.compress(N.FORMAT_BC1, img, w, h, alpha_mode=N.ALPHA_TRANSPARENCY,
                             color_weights=(key[0], key[1], key[2], 1.0))
        bad += _diff(out, g["expected"][sel])
    assert bad == 0, f"{bad} of {len(cws)} golden BC1 blocks differ"


@pytest.mark.parametrize("kind", range(len(blocks.KINDS)))
def test_adversarial_blocks(lanes, oracle, kind):
    rng = np.random.default_rng(300 + kind)
    n = 700  # several wavefronts per colour count, ragged tails
    cols = np.zeros((n, 16, 4), np.float32)
    wts = np.zeros((n, 16), np.float32)
    for i in range(n):
        cols[i], wts[i] = blocks.bc1_block(rng, blocks.KINDS[kind])
    img, w, h = _blocks_as_image(cols, wts)
    for mode in (N.ALPHA_TRANSPARENCY, N.ALPHA_NONE):
        for cw in ((1, 1, 1, 1), (0.5, 1.0, 0.25, 1.0)):
            a = lanes.compress(N.FORMAT_BC1, img, w, h, alpha_mode=mode, color_weights=cw)
            b = oracle.compress(N.FORMAT_BC1, img, w, h, alpha_mode=mode, cw=cw)
            assert np.array_equal(a, b), (blocks.KINDS[kind], mode, cw, _diff(a, b))


def test_mixed_kinds_in_one_image(lanes, oracle):
    """Every kind interleaved: waves of each colour count mix unit-weight,
    alpha-weighted and partial blocks."""
    rng = np.random.default_rng(77)
    n = 64 * 40
    cols = np.zeros((n, 16, 4), np.float32)
    wts = np.zeros((n, 16), np.float32)
    for i in range(n):
        cols[i], wts[i] = blocks.bc1_block(rng, blocks.KINDS[int(rng.integers(0, len(blocks.KINDS)))])
    img, w, h = _blocks_as_image(cols, wts)
    for mode in (N.ALPHA_TRANSPARENCY, N.ALPHA_NONE):
        a = lanes.compress(N.FORMAT_BC1, img, w, h, alpha_mode=mode)
        b = oracle.compress(N.FORMAT_BC1, img, w, h, alpha_mode=mode)
        assert np.array_equal(a, b), (mode, _diff(a, b))


@pytest.mark.parametrize("size", [(256, 256), (128, 64), (37, 23), (130, 66), (1, 1), (3, 5), (7, 1), (260, 9)])
@pytest.mark.parametrize("transparent", [False, True])
def test_images_match_oracle(lanes, oracle, size, transparent):
    w, h = size
    planar = synth.to_planar(synth.noise_rect_rgba(w, h, seed=41, transparent=transparent)).reshape(-1)
    for mode in (N.ALPHA_NONE, N.ALPHA_TRANSPARENCY):
        a = lanes.compress(N.FORMAT_BC1, planar, w, h, alpha_mode=mode)
        b = oracle.compress(N.FORMAT_BC1, planar, w, h, alpha_mode=mode)
        assert np.array_equal(a, b), (size, transparent, mode, _diff(a, b))


def test_dark_image(lanes, oracle):
    """Mostly black texels: skip_blacks drops clusters, the three-colour fit
    runs on a rebuilt table with its own count."""
    w, h = 192, 128
    img = synth.noise_rect_rgba(w, h, seed=5)
    img[:, :, :3] = (img[:, :, :3].astype(np.uint32) * 40 // 255).astype(np.uint8)
    planar = synth.to_planar(img).reshape(-1)
    a = lanes.compress(N.FORMAT_BC1, planar, w, h)
    b = oracle.compress(N.FORMAT_BC1, planar, w, h)
    assert np.array_equal(a, b), _diff(a, b)


def test_colour_counts_match_oracle(lanes, oracle):
    w, h = 160, 96
    planar = synth.to_planar(synth.noise_rect_rgba(w, h, seed=9)).reshape(-1)
    img = planar.astype(np.float32)
    d_in = lanes.alloc(img.nbytes).upload(img)
    nb = ((w + 3) // 4) * ((h + 3) // 4)
    d_out = lanes.alloc(nb * 8)
    d_nm = lanes.alloc(nb * 4)
    lanes.compress_bc1_stats_device(d_in, w, h, d_out, d_nm)
    got = d_out.download(np.uint8)
    nm = d_nm.download(np.int16).reshape(-1, 2)
    exp, exp_nm = oracle.compress_bc1_counts(planar, w, h)
    assert np.array_equal(got, exp)
    assert np.array_equal(nm, exp_nm)
    for b in (d_in, d_out, d_nm):
        b.free()


def test_two_encoders_agree_on_large_images(lanes, gpu):
    """1024^2 (65,536 blocks) and 2048x512, default context (one-pass below
    98,304 blocks) against the two-pass context."""
    for (w, h, seed) in ((1024, 1024, 3), (2048, 512, 4)):
        planar = synth.to_planar(synth.noise_rect_rgba(w, h, seed=seed, transparent=seed == 4)).reshape(-1)
        for mode in (N.ALPHA_NONE, N.ALPHA_TRANSPARENCY):
            a = lanes.compress(N.FORMAT_BC1, planar, w, h, alpha_mode=mode)
            b = gpu.compress(N.FORMAT_BC1, planar, w, h, alpha_mode=mode)
            assert np.array_equal(a, b), (w, h, mode, _diff(a, b))


def test_repeated_calls_reuse_cleared_tallies(lanes, oracle):
    """The search's last workgroup clears the per-count tallies: a second and
    a smaller third image on the same scratch give the same bytes."""
    res = []
    for (w, h) in ((96, 96), (96, 96), (40, 24)):
        planar = synth.to_planar(synth.noise_rect_rgba(w, h, seed=w + h)).reshape(-1)
        a = lanes.compress(N.FORMAT_BC1, planar, w, h)
        assert np.array_equal(a, oracle.compress(N.FORMAT_BC1, planar, w, h)), (w, h)
        res.append(a)
    assert np.array_equal(res[0], res[1])


def test_chain_and_image_set(lanes, oracle):
    """The chain entry point and the image scheduler (per-image scratch
    regions) through the two-pass encoder."""
    w = h = 128
    planar = synth.to_planar(synth.noise_rect_rgba(w, h, seed=8)).reshape(-1)
    levels = [planar]
    sizes = [(w, h)]
    while sizes[-1] != (1, 1):
        W, H = sizes[-1]
        levels.append(oracle.build_next_mipmap(N.FILTER_TRIANGLE, 1.0, None, N.WRAP_MIRROR, levels[-1], W, H))
        sizes.append((max(1, W // 2), max(1, H // 2)))
    d_lv = [lanes.alloc(4 * 4 * a * b) for (a, b) in sizes]
    d_lv[0].upload(planar)
    d_out = [lanes.alloc(N.compressed_size(N.FORMAT_BC1, a, b)) for (a, b) in sizes]
    lanes.compress_chain_device(N.FORMAT_BC1, N.FILTER_TRIANGLE, d_lv, w, h, d_out)
    for k, (a, b) in enumerate(sizes):
        exp = oracle.compress(N.FORMAT_BC1, levels[k], a, b)
        assert np.array_equal(d_out[k].download(np.uint8), exp), (a, b)
    for buf in d_lv + d_out:
        buf.free()


def _both_encoders(lanes, img, w, h, **kw):
    """The same image through the two-pass encoder and the one-pass one."""
    two = lanes.compress(N.FORMAT_BC1, img, w, h, **kw)
    lanes.set_bc1_lanes_min(1 << 30)
    try:
        one = lanes.compress(N.FORMAT_BC1, img, w, h, **kw)
    finally:
        lanes.set_bc1_lanes_min(1)
    return _diff(two, one)


@pytest.mark.parametrize("side", [60, 1024])  # four lanes a block, one lane a block (65,536 blocks)
@pytest.mark.parametrize("kind", ["units", "dark", "bright", "weights", "metric", "green", "specials"])
def test_search_forms_match_one_pass(lanes, side, kind):
    """The search's forms by how a candidate's terms come (from the table, as
    scalars, computed), its tie order on errors of both signs and of zero
    (dark blocks quantise to black), and the general path (values whose
    errors need not be finite, NaN among them)."""
    rng = np.random.default_rng(side + len(kind))
    base = synth.to_planar(synth.noise_rect_rgba(side, side, seed=5)).reshape(4, side, side)
    img, kw = base.copy(), {}
    noise = rng.random((3, side, side), dtype=np.float32)
    if kind == "units":
        img[:3, :, side // 2:] = noise[:, :, side // 2:]  # 16 clusters beside fewer
    elif kind == "dark":
        img[:3] = np.floor(noise * rng.integers(1, 9, (1, side, side))) / np.float32(255)
    elif kind == "bright":
        img[:3] = 1 - np.floor(noise * 6) / np.float32(255)
    elif kind == "weights":
        img[3] = rng.integers(0, 256, (side, side)) / np.float32(255)
        kw = dict(alpha_mode=N.ALPHA_TRANSPARENCY)
    elif kind == "metric":
        kw = dict(color_weights=(0.3, 0.59, 0.11, 1.0))
    elif kind == "green":
        kw = dict(color_weights=(0.0, 1.0, 0.0, 1.0))
    else:
        at = rng.integers(0, side * side, 200 + side)
        vals = np.array([np.nan, np.inf, -np.inf, 1e30, -1e30, 1e-30, 1e-42, 3e38, -0.0, 7.5], np.float32)
        img[:3].reshape(3, -1)[rng.integers(0, 3, at.size), at] = vals[rng.integers(0, len(vals), at.size)]
    w, h = side, side - (2 if kind == "units" else 0)  # a ragged last row: texels of weight 0 among the units
    assert _both_encoders(lanes, np.ascontiguousarray(img[:, :h]), w, h, **kw) == 0


@pytest.mark.parametrize("kind", ["random", "dark", "few", "both"])
@pytest.mark.parametrize("size", [(36, 28), (64, 64), (128, 64), (128, 68), (256, 128), (256, 132), (252, 260), (256, 256),
                                  (512, 132), (1024, 1024), (1448, 1452)])
def test_search_cuts_by_content(lanes, kind, size):
    """Lists that fill the grid's wavefronts exactly, by less, and by a block
    more (one list of 16 colours, with a few shorter ones; four colours a
    block; both): every block in exactly one wavefront, coarse or fine.  On
    the other side sixteen, four (from 513 blocks) and one (from 2,049) groups
    a block."""
    w, h = size
    rng = np.random.default_rng(w + h)
    img = np.ones((4, h, w), np.float32)
    img[:3] = rng.integers(0, 24 if kind == "dark" else 256, (3, h, w)) / np.float32(255)
    if kind in ("few", "both"):
        pal = (rng.integers(0, 256, (4, 3)) / 255).astype(np.float32)
        few = pal[rng.integers(0, 4, (h, w))].transpose(2, 0, 1)
        img[:3, :, w // 2 if kind == "both" else 0:] = few[:, :, w // 2 if kind == "both" else 0:]
    assert _both_encoders(lanes, img, w, h) == 0


@pytest.mark.parametrize("side", [60, 1024])
@pytest.mark.parametrize("scale, alpha", [(s, 1.0) for s in (1e8, 3e9, 1e10, 1e14, 9e17)] +
                         [(1.0, a) for a in (1e-12, 1e-16, 1e-20, 1e-30)] + [(1e10, 1e-20)])
def test_search_where_the_axis_overflows(lanes, oracle, side, scale, alpha):
    """Components and weights whose sums and errors are finite, but whose
    covariances have no finite squares, so that the projections that the
    clusters are sorted by are NaN: blocks of 2 to 16 colours, the reference's
    order (a NaN moves nothing) in both encoders."""
    rng = np.random.default_rng(int(np.log10(scale)) * 7 + side)
    nb = side // 4
    pal = rng.random((nb, nb, 16, 3), dtype=np.float32) * np.float32(scale)
    count = rng.integers(2, 17, (nb, nb, 1))
    pick = np.where(rng.random((nb, nb, 1)) < 0.3, np.arange(16), rng.integers(0, 16, (nb, nb, 16))) % count
    texels = np.take_along_axis(pal, pick[..., None], axis=2).reshape(nb, nb, 4, 4, 3)
    img = np.empty((4, side, side), np.float32)
    img[:3] = texels.transpose(4, 0, 2, 1, 3).reshape(3, side, side)
    img[3] = np.float32(alpha)
    kw = dict(alpha_mode=N.ALPHA_TRANSPARENCY)
    assert _both_encoders(lanes, img, side, side, **kw) == 0
    assert _diff(lanes.compress(N.FORMAT_BC1, img, side, side, **kw),
                 oracle.compress(N.FORMAT_BC1, img.reshape(-1), side, side, **kw)) == 0


def test_default_route_by_size_and_scratch():
    """A context as it is made: a set of 87,710 blocks, where the two-pass
    encoder is optional, with and without a scratch limit (which keeps it
    off), and an image of 57,500, below the line for one, give the one-pass
    encoder's bytes."""
    free, capped, one = N.Context(0), N.Context(0), N.Context(0)
    try:
        capped.lib.ntx_hip_set_scratch_limit(capped.handle, 1)
        one.set_bc1_lanes_min(1 << 30)
        sizes = [(1000, 917), (640, 480), (511, 333), (64, 64), (3, 2), (1, 1)]
        planes = [synth.to_planar(synth.noise_rect_rgba(w, h, seed=70 + k)).reshape(-1) for k, (w, h) in enumerate(sizes)]
        got = {}
        for name, ctx in (("free", free), ("capped", capped), ("one", one)):
            d = [ctx.alloc(p.nbytes).upload(p) for p in planes]
            single = ctx.alloc(N.compressed_size(N.FORMAT_BC1, *sizes[0]))
            ctx.compress_device(N.FORMAT_BC1, d[0], *sizes[0], single)
            outs = [ctx.alloc(N.compressed_size(N.FORMAT_BC1, w, h)) for w, h in sizes]
            ctx.profile(True)
            ctx.profile_read(reset=True)
            ctx.compress_images_device(N.FORMAT_BC1, d, sizes, outs)
            ran = ctx.profile_read(reset=True)
            # Both passes under their own names, once each, or neither.
            for kernel in ("bc1_classify_kernel", "bc1_search_kernel"):
                assert ran.get(kernel, (0, 0))[1] == (name == "free"), (kernel, ran)
            got[name] = [single.download(np.uint8)] + [o.download(np.uint8) for o in outs]
        for name in ("free", "capped"):
            for a, b in zip(got[name], got["one"]):
                assert np.array_equal(a, b)
    finally:
        for ctx in (free, capped, one):
            ctx.close()


def _input(ctx, w, h, seed):
    p = synth.to_planar(synth.noise_rect_rgba(w, h, seed=seed)).reshape(-1)
    return p, ctx.alloc(p.nbytes).upload(p)


def test_optional_scratch_is_off_a_later_limit():
    """Calls that took the two-pass encoder's optional scratch leave a limit
    that is set afterwards to the calls that need theirs."""
    with N.Context(0) as ctx:
        w, h = 1280, 1232  # 98,560 blocks
        _, d = _input(ctx, w, h, 81)
        _, d2 = _input(ctx, 640, 480, 82)
        out = [ctx.alloc(N.compressed_size(N.FORMAT_BC1, a, b)) for a, b in ((w, h), (640, 480))]
        ctx.compress_images_device(N.FORMAT_BC1, [d, d2], [(w, h), (640, 480)], out)
        ctx.compress_device(N.FORMAT_BC1, d, w, h, out[0])
        first = out[0].download(np.uint8)
        small = synth.to_planar(synth.noise_rect_rgba(64, 64, seed=83)).reshape(-1)
        ctx.lib.ntx_hip_set_scratch_limit(ctx.handle, small.nbytes + N.compressed_size(N.FORMAT_BC4, 64, 64))
        ctx.compress(N.FORMAT_BC4, small, 64, 64)
        for limit in (1, 0, 1 << 30, 0):  # without it, with it, and back
            ctx.lib.ntx_hip_set_scratch_limit(ctx.handle, limit)
            out[0].upload(np.zeros_like(first))
            ctx.compress_device(N.FORMAT_BC1, d, w, h, out[0])
            assert np.array_equal(out[0].download(np.uint8), first), limit


def test_optional_scratch_and_recorded_graphs():
    """A graph recorded over a call that needs the context's scratch, replayed
    after calls that took the optional one and between others; a scratch limit
    set while the context's stream records, and a call with the optional
    scratch while another stream does, which the recordings survive."""
    with N.Context(0) as ctx:
        w, h = 128, 96
        _, d = _input(ctx, w, h, 91)
        _, big = _input(ctx, 1280, 1232, 92)
        out = ctx.alloc(N.compressed_size(N.FORMAT_BC3, w, h))
        out_big = ctx.alloc(N.compressed_size(N.FORMAT_BC1, 1280, 1232))
        ctx.compress_device(N.FORMAT_BC3, d, w, h, out)  # its scratch is there before the recording
        want = out.download(np.uint8)
        ctx.compress_device(N.FORMAT_BC1, big, 1280, 1232, out_big)
        with Capture(ctx, ctx.lib.ntx_hip_stream(ctx.handle), 2) as g:
            ctx.compress_device(N.FORMAT_BC3, d, w, h, out)
            for limit in (1 << 30, 0):
                ctx.lib.ntx_hip_set_scratch_limit(ctx.handle, limit)
        ctx.lib.ntx_hip_set_scratch_limit(ctx.handle, 1 << 30)
        ctx.lib.ntx_hip_set_scratch_limit(ctx.handle, 0)
        other = ctypes.c_void_p()
        assert ctx.lib.hipStreamCreateWithFlags(ctypes.byref(other), 1) == 0
        recording = Capture(ctx, other.value, 0)
        results = []
        for k in range(4):
            if k == 1:
                with recording:
                    ctx.compress_device(N.FORMAT_BC1, big, 1280, 1232, out_big)
            elif k > 1:
                ctx.compress_device(N.FORMAT_BC1, big, 1280, 1232, out_big)
            if k:
                results.append(out_big.download(np.uint8))
            out.upload(np.zeros_like(want))
            g.launch()
            ctx.synchronize()
            assert np.array_equal(out.download(np.uint8), want), k
        ctx.set_bc1_lanes_min(1 << 30)
        ctx.compress_device(N.FORMAT_BC1, big, 1280, 1232, out_big)
        for r in results:
            assert np.array_equal(r, out_big.download(np.uint8))
        g.close()
        recording.close()
        assert ctx.lib.hipStreamDestroy(other) == 0
