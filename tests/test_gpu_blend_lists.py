"""Blends of hand-made tile lists through fgs_blend against the oracle's pair-by-pair walk: what a list may
hold beyond what fgs_preprocess makes."""
import numpy as np
import pytest

from flashgs_amd import cabi

pytestmark = pytest.mark.gpu

BLOCKS = [(16, 16), (32, 16), (32, 32)]


def column_of_tiles(lists, tiles):
    """Lists of (xy, conic_opacity, rgb) for tile 0, 1, ... of a frame one tile wide: (points_xy, rgb_depth,
    conic_opacity, values, ranges), the list positions shuffled over the Gaussian indices."""
    lengths = np.array([len(l[0]) for l in lists])
    ends = np.cumsum(lengths)
    ranges = np.zeros((tiles, 2), np.int32)
    ranges[:len(lists)] = np.stack([ends - lengths, ends], 1)
    xy, co, rgb = (np.concatenate([np.asarray(l[i], np.float64) for l in lists]) for i in range(3))
    n = len(xy)
    values = np.random.default_rng(n).permutation(n).astype(np.uint32)
    at = np.empty(n, np.int64)
    at[values] = np.arange(n)
    rgbd = np.concatenate([rgb, np.ones((n, 1))], 1)
    return tuple(np.ascontiguousarray(a[at], dtype=np.float32) for a in (xy, rgbd, co)) + (values, ranges)


def gpu_blend(block, W, H, arrays, bg, flags=None):
    """(float image, 8-bit image) of fgs_blend(_ex)."""
    import gpu_pipeline as gp
    import torch
    xy, rgbd, co, values, ranges = arrays
    d = [gp.dev(a) for a in (xy, rgbd, co, values.view(np.int32), ranges)]
    out = torch.full((H, W, 3), -1.0, device=gp.DEV, dtype=torch.float32)
    out_u8 = torch.full((H, W, 3), 77, device=gp.DEV, dtype=torch.uint8)
    cabi.blend(block[0], block[1], W, H, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), d[3].data_ptr(), d[4].data_ptr(),
               bg, out_u8.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream, flags=flags)
    torch.cuda.synchronize()
    return out.cpu().numpy(), out_u8.cpu().numpy()


def frame_height(block, W, ranked, lists):
    """(tiles, height) of a frame one tile wide with room for the lists, whose tiles are ranked by list length or are too many
    for that."""
    import gpu_pipeline  # noqa: F401  (torch before the library)
    tiles = lists if ranked else 8200
    H = tiles * block[1]
    assert ("tile_order_kernel" in cabi.blend_kernel_name(block[0], block[1], W, H)) == ranked
    return tiles, H


@pytest.mark.parametrize("ranked", [True, False])
@pytest.mark.parametrize("block", BLOCKS)
def test_last_of_an_odd_list_may_be_infinite(oracle, block, ranked):
    """A list ends behind its last Gaussian (render.cu:486-487), also where there is no second one of its pair: an infinite
    colour or weight of it stays infinite and does not meet a weight of zero.  The other colours: sums of weights
    that are exact to some 1e-6 each, over at most 65 Gaussians of colours up to 1."""
    rng = np.random.default_rng(5)
    lists = []
    for n in (1, 2, 3, 15, 16, 17, 31, 47, 63, 64, 65):
        for kind in ("colour", "negative colour", "weight", "colour in front"):
            c = rng.uniform(0, 16, (n, 2))
            c[:, 1] += block[1] * len(lists)
            co = np.stack([-rng.uniform(1e-4, 1e-3, n), np.zeros(n), -rng.uniform(1e-4, 1e-3, n), np.log2(rng.uniform(0.01, 0.05, n))], 1)
            rgb = rng.uniform(0, 1, (n, 3))
            if kind == "colour":
                rgb[-1, 0] = np.inf
            elif kind == "negative colour":
                rgb[-1, 1] = -np.inf
            elif kind == "colour in front":
                rgb[max(n - 2, 0), 2] = np.inf
            else:
                co[-1, 3] = 300.0
            lists.append((c, co, rgb))
    W = 7
    tiles, H = frame_height(block, W, ranked, len(lists))
    arrays = column_of_tiles(lists, tiles)
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    ref_u8, ref, _ = oracle.render(W, H, block[0], block[1], *arrays, bg)
    out, out_u8 = gpu_blend(block, W, H, arrays, bg)
    assert np.isinf(ref).any() and not np.isnan(ref).any()
    finite = np.isfinite(ref)
    assert np.array_equal(np.isfinite(out), finite) and np.array_equal(out[~finite], ref[~finite])
    assert np.abs(out[finite] - ref[finite]).max() <= 1e-4
    assert np.array_equal(out_u8[~finite], ref_u8[~finite])


@pytest.mark.parametrize("ranked", [True, False])
@pytest.mark.parametrize("flags", ["fp32", "f16"])
@pytest.mark.parametrize("block", BLOCKS)
def test_exponents_that_rise_steeply_along_a_column(oracle, block, flags, ranked):
    """Conics whose exponent starts below -126 at the first pixel of a strip of four and is near zero at another one of
    them: saddles (cx > 0, or cy^2 > 4 cx cz) with a curvature along the strip between -3 and 0, beside
    needles that are semidefinite to a rounding.  Frames one pixel wide, so that no column has weights
    above 1.  Bound: up to six terms of magnitude M < 2000, each rounded by M 2^-24, times ln 2 and a weight of
    up to 0.9, over lists whose weights sum to less than 2; 2^-10 of a colour more with f16 operands."""
    rng = np.random.default_rng(6)
    lists = []
    for i in range(48):
        n = (1, 2, 7, 16, 33, 64)[i % 6]
        rows = np.arange(block[1])
        cz = -rng.uniform(0.3, 3.0, n)
        dx = rng.uniform(2.0, 14.0, n) * rng.choice([-1, 1], n)
        if i % 3 == 0:
            cx, cy = rng.uniform(0.1, 1.0, n), np.zeros(n)
        elif i % 3 == 1:
            cx = -rng.uniform(0.1, 1.0, n)
            cy = rng.choice([-1, 1], n) * rng.uniform(2.5, 6.0, n) * np.sqrt(cx * cz)
        else:
            cx = -rng.uniform(0.1, 3.0, n)
            cy = rng.choice([-1, 1], n) * 2 * np.sqrt(cx * cz) * (1 + rng.uniform(-1e-6, 1e-6, n))
        dy0 = rng.uniform(-4, block[1] + 4, n)              # centre's row
        co = np.stack([cx, cy, cz, np.zeros(n)], 1)
        d = dy0[:, None] - rows
        peak = (cx * dx * dx)[:, None] + cz[:, None] * d * d + cy[:, None] * dx[:, None] * d
        # (an opacity that the form with f16 operands does not hold down)
        co[:, 3] = np.minimum(np.log2(rng.uniform(0.3, 0.9, n) / (1 if n < 3 else 0.5 * n)) - peak.max(1), 1.5)
        lists.append((np.stack([dx, dy0 + block[1] * i], 1), co, rng.uniform(0, 1, (n, 3))))
    W = 1
    tiles, H = frame_height(block, W, ranked, len(lists))
    arrays = column_of_tiles(lists, tiles)
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    _, ref, _ = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg, cabi.BLEND_FP32 if flags == "fp32" else cabi.BLEND_MATRIX_F16)
    err = np.abs(out - ref)
    assert np.isfinite(err).all()
    assert err.max() <= 6 * 2000 * 2.0 ** -24 * 0.69 * 2 + (2.0 ** -10 if flags == "f16" else 0.0), "max abs image error %g" % err.max()


def stops(T, squares, threshold):
    """Transmittances [pairs, pixels] of a tile behind every pair, and the square of every pixel: (the pair behind which all
    pixels have T < threshold, the last of the pairs behind which each square by itself first has)."""
    below = T < threshold
    first = [np.flatnonzero(b) for b in [below.all(1)] + [below[:, squares == s].all(1) for s in range(squares.max() + 1)]]
    first = [f[0] if len(f) else len(T) for f in first]
    return first[0], max(first[1:])


@pytest.mark.parametrize("flags", ["fp32", "f16"])
@pytest.mark.parametrize("block", [(32, 16), (32, 32)])
def test_a_wide_tile_stops_where_all_of_it_is_opaque_at_once(oracle, block, flags):
    """Weights above 1 (opacities up to 3) turn the sign of T, so a square of a wide tile that was opaque can be
    transparent again before the other squares are opaque: the tile goes on (render.cu:394-408).  Lists are drawn until
    some of them have such a history, none of it within a rounding of the threshold or with a product of weight and T that
    f16 operands cannot hold (4).  The bound: some 1e-6 per weight, times up to 3.5, a dozen weights of colours up to 1; with
    f16 operands 2^-10 of each weight's colour more."""
    rng = np.random.default_rng(8)
    y, x = np.mgrid[:block[1], :block[0]]
    squares = (x // 16 + (block[0] // 16) * (y // 16)).ravel()
    lists, late = [], 0
    while late < 12:
        n = int(rng.integers(6, 16))
        c = rng.uniform(-2, 34, (n, 2)) * (1, block[1] / 32)
        cx, cz = -rng.uniform(0.0002, 0.004, n), -rng.uniform(0.0002, 0.004, n)
        op = rng.choice([1.2, 1.6, 2.2, 3.0, 0.99], n)
        dx, dy = c[:, 0, None] - x.ravel(), c[:, 1, None] - y.ravel()
        alpha = op[:, None] * 2.0 ** (cx[:, None] * dx * dx + cz[:, None] * dy * dy)
        T = np.cumprod(1.0 - alpha, 0)
        heaviest = np.abs(alpha[1:] * T[:-1]).max()
        (together, alone), low, high = (stops(T[1::2], squares, t) for t in (1e-4, 0.95e-4, 1.05e-4))
        if heaviest > 3.5 or not low == high == (together, alone) or (together == alone and len(lists) - late > 12):
            continue
        late += together > alone
        c[:, 1] += block[1] * len(lists)
        lists.append((c, np.stack([cx, np.zeros(n), cz, np.log2(op)], 1), rng.uniform(0, 1, (n, 3))))
    W, H = block[0], block[1] * len(lists)
    arrays = column_of_tiles(lists, len(lists))
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    _, ref, _ = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg, cabi.BLEND_FP32 if flags == "fp32" else cabi.BLEND_MATRIX_F16)
    for i in range(len(lists)):
        rows = slice(i * block[1], (i + 1) * block[1])
        assert np.abs(out[rows] - ref[rows]).max() <= 1e-4 + (15 * 3.5 * 2.0 ** -10 if flags == "f16" else 0.0), i


@pytest.mark.parametrize("flags", ["fp32", "f16"])
@pytest.mark.parametrize("block", [(32, 16), (32, 32)])
def test_squares_of_a_wide_tile_walk_on_to_its_stop(oracle, block, flags):
    """One square of a tile is opaque (T < 1e-4) early, the tile late, and Gaussians of colour 1e4 lie between the two and
    behind the tile's stop: what lies between reaches the opaque square with up to 0.3, what lies behind reaches
    nothing.  Bound: relative errors of some 1e-6 of the weights, and of 1e-4 of a T that is a product of ten
    1 - 0.99; 2^-10 more with f16 operands."""
    rng = np.random.default_rng(9)
    lists, early = [], []
    for square in range(block[0] // 16 * (block[1] // 16)):
        for n_between in (2, 5, 18, 70):
            left, top = square % 2 * 16, square // 2 * 16
            head = [(left + 7.5, top + 7.5, -0.005, -0.005, 0.99, 1.0)] * 10
            between = [(16.0, 16.0, -1e-6, -1e-6, 0.3 if n_between < 10 else 0.02, 1e4)] * n_between
            close = [(16.0, 16.0, -1e-6, -1e-6, 0.99, 0.5)] * 12
            behind = [(16.0, 16.0, -1e-6, -1e-6, 0.9, 1e4)] * 4
            x, y, cx, cz, op, bright = np.array(head + between + close + behind).T
            n = len(x)
            early.append((len(lists) * block[1] + top, left, len(lists)))
            lists.append((np.stack([x, y + block[1] * len(lists)], 1), np.stack([cx, np.zeros(n), cz, np.log2(op)], 1),
                          bright[:, None] * rng.uniform(0.5, 1, (n, 3))))
    W, H = block[0], block[1] * len(lists)
    arrays = column_of_tiles(lists, len(lists))
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    _, ref, walked = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    _, short, _ = oracle.render(W, H, block[0], block[1], *column_of_tiles([[a[:10] for a in l] for l in lists], len(lists)),
                                bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg, cabi.BLEND_FP32 if flags == "fp32" else cabi.BLEND_MATRIX_F16)
    bound = 1e-3 + (1e-5 + (2.0 ** -9 if flags == "f16" else 0.0)) * np.abs(ref)
    for y, x, _ in early:
        assert np.abs(ref - short)[y:y + 16, x:x + 16].max() > 0.02     # the lists are what the test is about
    assert (np.abs(out - ref) <= bound).all(), np.abs(out - ref).max()


@pytest.mark.parametrize("block", BLOCKS)
def test_lists_that_end_with_the_last_pair_an_int_can_count(block):
    """Indices of later entries are fetched ahead of the walk: at the end of 2^31 - 1 pairs they are not to leave the int's
    range.  The same lists at the start of the pairs give the same bits."""
    import gpu_pipeline as gp
    import torch
    most = 2 ** 31 - 1
    if torch.cuda.mem_get_info()[0] < 4 * most + (1 << 30):
        pytest.skip("no memory for 2^31 - 1 values")
    rng = np.random.default_rng(10)
    lengths = [1500, 769, 300, 129, 128, 127, 65, 64, 63, 2, 1]
    lists = []
    for i, n in enumerate(lengths):
        c = rng.uniform(-4, 20, (n, 2)) + (0, block[1] * i)
        co = np.stack([-rng.uniform(0.005, 0.1, n), np.zeros(n), -rng.uniform(0.005, 0.1, n), np.log2(rng.uniform(0.0005, 0.01, n))], 1)
        lists.append((c, co, rng.uniform(0, 1, (n, 3))))
    W, H = 16, block[1] * len(lists)
    xy, rgbd, co, values, ranges = column_of_tiles(lists, len(lists))
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    expected, _ = gpu_blend(block, W, H, (xy, rgbd, co, values, ranges), bg)
    K = len(values)
    d = [gp.dev(a) for a in (xy, rgbd, co)]
    all_values = torch.empty(most, device=gp.DEV, dtype=torch.int32)
    all_values[most - K:] = gp.dev(values.view(np.int32))
    for last in range(len(lists)):          # every list in turn ends with the last pair
        there = ranges.astype(np.int64) + most - ranges[last, 1]
        there[last + 1:] = 0
        all_values[most - ranges[last, 1]:] = gp.dev(values[:ranges[last, 1]].view(np.int32))
        dr = gp.dev(there.astype(np.int32))
        out = torch.full((H, W, 3), -1.0, device=gp.DEV, dtype=torch.float32)
        cabi.blend(block[0], block[1], W, H, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), all_values.data_ptr(),
                   dr.data_ptr(), bg, 0, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        rows = (last + 1) * block[1]
        assert np.array_equal(out.cpu().numpy()[:rows], expected[:rows]), lengths[last]


@pytest.mark.parametrize("ranked", [True, False])
@pytest.mark.parametrize("flags", ["fp32", "f16"])
@pytest.mark.parametrize("block", BLOCKS)
def test_splats_sharper_than_a_pixel(oracle, block, flags, ranked):
    """Conics with a curvature along the strip beyond the recurrence's -3 (splats that were not widened by 0.3): up to -64,
    where exponents are summed up, and beyond, in lists around the chunk of 64, from the first Gaussian on, from later ones
    on, or in turn with others.  Bound: with a centre within 12 pixels the exponent's terms are below 64 * 144 + the
    like across, 18432, and are rounded three times, and slopes below 1536 up to three times each: 1.7e-3, times ln 2, on a
    weight of up to 0.6; beyond -64 every exponent is evaluated.  The 2^-10 of f16 operands on top."""
    rng = np.random.default_rng(11)
    lists = []
    for i in range(60):
        n = (1, 2, 15, 17, 63, 64, 65, 128, 131, 200)[i % 10]
        c = rng.uniform(-2, 18, (n, 2)) + (0, block[1] * i + rng.uniform(0, block[1] - 16))
        cx, cz = -rng.uniform(0.02, 0.5, n), -rng.uniform(0.02, 0.5, n)
        sharp = np.arange(n) >= (0, n // 2, 70)[i % 3] if i % 4 else np.arange(n) % 5 == 1
        cz[sharp] = -np.exp(rng.uniform(np.log(3.0), np.log(64.0 if i % 5 else 1000.0), sharp.sum()))
        cx[sharp] = -np.exp(rng.uniform(np.log(0.1), np.log(64.0), sharp.sum()))
        cy = rng.uniform(-0.95, 0.95, n) * 2 * np.sqrt(cx * cz)
        lists.append((c, np.stack([cx, cy, cz, np.log2(rng.uniform(0.05, 0.6, n))], 1), rng.uniform(0, 1, (n, 3))))
    W = 16
    tiles, H = frame_height(block, W, ranked, len(lists))
    arrays = column_of_tiles(lists, tiles)
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    _, ref, _ = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg, cabi.BLEND_FP32 if flags == "fp32" else cabi.BLEND_MATRIX_F16)
    err = np.abs(out - ref)
    assert np.isfinite(err).all()
    assert err.max() <= 0.6 * 0.69 * 1.7e-3 + (2.0 ** -10 if flags == "f16" else 0.0), "max abs image error %g" % err.max()


def exact_blend(block, W, H, arrays, bg):
    """The pair-by-pair walk of every tile's list in float64: (image, T of every pixel)."""
    xy, rgbd, co, values, ranges = arrays
    xy, rgbd, co = (a.astype(np.float64) for a in (xy, rgbd, co))
    gx = -(-W // block[0])
    out = np.zeros((-(-H // block[1]) * block[1], gx * block[0], 3))
    remaining = np.ones(out.shape[:2])
    for t, (lo, hi) in enumerate(ranges):
        y, x = np.mgrid[t // gx * block[1]:(t // gx + 1) * block[1], t % gx * block[0]:(t % gx + 1) * block[0]]
        g = values[lo:hi]
        dx, dy = xy[g, 0, None, None] - x, xy[g, 1, None, None] - y
        cx, cy, cz, w = (co[g, i, None, None] for i in range(4))
        alpha = np.exp2(w + cx * dx * dx + cz * dy * dy + cy * dx * dy)
        T = np.concatenate([np.ones((1,) + x.shape), np.cumprod(1.0 - alpha, 0)])
        stops = np.flatnonzero((T[2::2] < 1e-4).all((1, 2)))            # behind pair 0, 1, ...
        n = 2 * (stops[0] + 1) if len(stops) else hi - lo
        left = np.where(T[n] < 1e-4, 0.0, T[n])
        remaining[y, x] = T[n]
        out[y, x] = np.einsum("nyx,nc->yxc", alpha[:n] * T[:n], rgbd[g[:n], :3]) + left[..., None] * bg
    return out[:H, :W], remaining[:H, :W]


#: smallest and largest standard deviation of a splat along its axes in pixels, before it is widened by 0.3
SPLATS = {"small": (0.1, 2.0), "medium": (3.0, 20.0), "wide": (20.0, 300.0), "needles": (0.1, 100.0)}


@pytest.mark.parametrize("block", BLOCKS)
@pytest.mark.parametrize("splats", sorted(SPLATS))
def test_error_against_float64(oracle, block, splats):
    """The fp32 blend of conics as fgs_preprocess makes them against a float64 evaluation, beside an fp32 evaluation of
    render.cu:42-52 term by term (the oracle's).  Bound: half as much again as that, and twice as much at the
    worst pixel, for the other order of the sums; on top, for splats of a pixel, whose exponent is a sum of terms of up to
    2 * 2.4 * 12^2 = 700 where term by term it is small: two roundings of 700 * 2^-25 times ln 2 and a weight of up to 0.5, 1.4e-5 at
    the worst pixel, and a twentieth of it over all."""
    lo, hi = SPLATS[splats]
    rng = np.random.default_rng(12)
    lists = []
    for i in range(24):
        n = int(rng.integers(20, 250))
        sigma = np.exp(rng.uniform(np.log(lo), np.log(hi), (n, 2)))
        if splats == "needles":
            sigma = np.stack([np.exp(rng.uniform(np.log(30.0), np.log(hi), n)), rng.uniform(lo, 0.5, n)], 1)
        angle = rng.uniform(0, np.pi, n)
        c, s = np.cos(angle), np.sin(angle)
        a, b = sigma[:, 0] ** 2, sigma[:, 1] ** 2
        xx, yy, xy = a * c * c + b * s * s + 0.3, a * s * s + b * c * c + 0.3, (a - b) * c * s
        det = xx * yy - xy * xy
        half_log2e = 0.5 * 1.4426950408889634
        # a centre within two standard deviations of a pixel of the tile
        r = 2 * np.sqrt(rng.uniform(0, 1, n))
        phi = rng.uniform(0, 2 * np.pi, n)
        u, v = r * np.cos(phi) * sigma[:, 0], r * np.sin(phi) * sigma[:, 1]
        centre = rng.uniform(0, 1, (n, 2)) * block + np.stack([u * c - v * s, u * s + v * c], 1)
        lists.append((centre + (0, block[1] * i),
                      np.stack([-half_log2e * yy / det, 2 * half_log2e * xy / det, -half_log2e * xx / det,
                                np.log2(rng.uniform(0.02, 0.5, n))], 1), rng.uniform(0, 1, (n, 3))))
    W, H = block[0], block[1] * len(lists)
    arrays = column_of_tiles(lists, len(lists))
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    exact, T = exact_blend(block, W, H, arrays, bg.astype(np.float64))
    _, plain, _ = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg)
    scale = np.sqrt((exact ** 2).mean())
    same = np.abs(T / 1e-4 - 1) > 0.05        # where T is 1e-4 but for a rounding, the background stays or goes
    rms = [np.sqrt(((i - exact)[same] ** 2).mean()) / scale for i in (out, plain)]
    worst = [np.abs(i - exact)[same].max() for i in (out, plain)]
    print("%s %dx%d: rms error / rms value %.2e (term by term %.2e), largest error %.2e (%.2e)"
          % (splats, block[0], block[1], rms[0], rms[1], worst[0], worst[1]))
    assert same.mean() > 0.99
    assert rms[0] <= 1.5 * rms[1] + 7e-7 and worst[0] <= 2 * worst[1] + 1.4e-5


@pytest.mark.parametrize("flags", ["fp32", "f16"])
@pytest.mark.parametrize("tiles", [40, 300, 1100])
@pytest.mark.parametrize("block", BLOCKS)
def test_lists_shared_by_the_teams_of_a_workgroup(oracle, block, tiles, flags):
    """Lists around the lengths where they are shared out and where rounds and runs end, odd ones among them, with opaque content
    that ends the walk in the head, in one run or another, on a run's last pair, or never, and with weights above one in
    some runs; workgroups of 8, 4 and 2 teams, ranked, and the same bits from fgs_render_f32, which does not rank frames that are resident at once.  The walk ends behind the reference's pair, so the bound is the one of a
    whole walk: rounding of sums of up to 0.5 * 1500 weights of 1.5, some 1e-5, and twice that where weights above one turn T's sign."""
    rng = np.random.default_rng(tiles + block[0] * block[1])
    lengths = [1, 2, 63, 64, 65, 127, 128, 129, 191, 192, 193, 257, 319, 320, 321, 385, 511, 576, 577, 700, 832, 833, 1000, 1089, 1500, 1501]
    stops = [None, 10, 60, 66, 100, 127, 128, 160, 190, 250, 300, 319, 400, 500, 650, 900]
    lists = []
    for i in range(min(tiles, 40)):
        n = lengths[i % len(lengths)] if i < 30 else 1200
        top = block[1] * i
        xy = rng.uniform(0, 1, (n, 2)) * block + (0, top)
        cx, cz = -rng.uniform(0.005, 0.3, n), -rng.uniform(0.005, 0.3, n)
        w = np.log2(rng.uniform(0.002, 0.02, n))
        cy = rng.uniform(-0.9, 0.9, n) * 2 * np.sqrt(cx * cz)
        at = stops[(5 * i) % len(stops)]
        if at is not None and at + 30 <= n:          # opaque for every pixel: alpha of 0.9 and more
            o = slice(at, at + 30)
            cx[o] = cz[o] = -1e-5
            cy[o] = 0.0
            w[o] = np.log2(0.92)
            # (wide tiles: other squares stop at other pairs)
            o = slice(at, at + 8)
            cx[o] = cz[o] = -2e-2
        if i % 7 == 3 and n > 150:                   # weights of up to 1.4
            w[rng.integers(70, n, 3)] = 0.5
        lists.append((xy, np.stack([cx, cy, cz, w], 1), rng.uniform(0, 1, (n, 3))))
    W, H = block[0], block[1] * tiles
    arrays = column_of_tiles(lists, tiles)
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    _, ref, _ = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg, cabi.BLEND_FP32 if flags == "fp32" else cabi.BLEND_MATRIX_F16)
    err = np.abs(out - ref)
    assert err.max() <= (3e-5 if flags == "fp32" else 2.0 ** -10 * 1.5), "max abs image error %g at %r" % (err.max(), np.unravel_index(err.argmax(), err.shape))
    import gpu_pipeline as gp
    xy, rgbd, co, values, ranges = arrays
    keys = np.repeat(np.arange(tiles, dtype=np.uint64) << np.uint64(32), ranges[:, 1] - ranges[:, 0])
    found, _, same = gp.render(len(values), W, H, gp.dev(xy), gp.dev(rgbd), gp.dev(co), gp.dev(keys.view(np.int64)), gp.dev(values.view(np.int32)),
                               bg, block, flags=cabi.BLEND_FP32 if flags == "fp32" else cabi.BLEND_MATRIX_F16)
    assert np.array_equal(found.cpu().numpy(), ranges) and np.array_equal(same.cpu().numpy(), out)


@pytest.mark.parametrize("block, W, H, usual", [((32, 32), 640, 512, 22_000), ((32, 32), 512, 512, 27_000),
                                                ((32, 16), 640, 400, 27_000), ((16, 16), 400, 320, 54_000)])
def test_lists_of_tens_of_thousands_in_a_frame_of_few_tiles(oracle, block, W, H, usual):
    """The length from which lists are shared out is at its limit, which the ranking still tells apart: fgs_blend, which ranks the
    tiles, and fgs_render_f32, which does not rank so few, give the same bits.  Lists in front of, at and
    behind that limit, most of them of `usual` entries.  Three tiles against the oracle; bound: every weight and T carries a
    rounding for each entry in front of it, 2^-24 of a colour of at most 1 each."""
    import gpu_pipeline as gp
    import torch
    gx, gy = -(-W // block[0]), -(-H // block[1])
    tiles = gx * gy
    rng = np.random.default_rng(tiles)
    lengths = np.full(tiles, usual)
    lengths[::7] = np.resize([0, 1, 100, 5000, 8159, 8160, 8161, 9000, 30_000], len(lengths[::7]))
    K, squares = int(lengths.sum()), block[0] * block[1] // 256
    assert K * squares / 1024 * 3 / 8 > 8192 and tiles <= 512
    n = 60_000
    xy = rng.uniform(0, 1, (n, 2)) * (W, H)
    co = np.stack([np.full(n, -1e-6), np.zeros(n), np.full(n, -1e-6), np.log2(rng.uniform(0.1, 1.0, n) * 20.0 / usual)], 1)
    rgbd = np.concatenate([rng.uniform(0, 1, (n, 3)), np.ones((n, 1))], 1)
    xy, co, rgbd = (np.ascontiguousarray(a, dtype=np.float32) for a in (xy, co, rgbd))
    ends = np.cumsum(lengths)
    ranges = np.stack([ends - lengths, ends], 1).astype(np.int32)
    ranges[lengths == 0] = 0
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    # tile t's list: Gaussians t, t + 1, ... in turn
    tile = np.repeat(np.arange(tiles), lengths)
    values = ((np.arange(K) - (ends - lengths)[tile] + tile) % n).astype(np.uint32)
    out, out_u8 = gpu_blend(block, W, H, (xy, rgbd, co, values, ranges), bg)
    keys = gp.dev((tile.astype(np.uint64) << np.uint64(32)).view(np.int64))
    found, ref_u8, ref = gp.render(K, W, H, *(gp.dev(a) for a in (xy, rgbd, co)), keys, gp.dev(values.view(np.int32)), bg, block)
    assert np.array_equal(found.cpu().numpy(), ranges)
    assert np.array_equal(out, ref.cpu().numpy()) and np.array_equal(out_u8, ref_u8.cpu().numpy())
    few = np.zeros_like(ranges)
    some = [1, 7 * 5, 7 * 8]                 # `usual`, 8160 and 30 000 entries
    few[some] = ranges[some]
    _, exact, _ = oracle.render(W, H, block[0], block[1], xy, rgbd, co, values, few, bg, want_u8=False)
    for t in some:
        y, x = t // gx * block[1], t % gx * block[0]
        err = np.abs(out - exact)[y:y + block[1], x:x + block[0]]
        assert lengths[t] >= 8160 and err.max() <= 30_000 * 2.0 ** -24, (t, err.max())


@pytest.mark.parametrize("kind", ["flat along y", "growing along x and y", "growing along x"])
@pytest.mark.parametrize("block", BLOCKS)
def test_stop_in_a_run_that_conics_of_another_kind_undo(oracle, block, kind):
    """A list that is shared out becomes opaque in a run (T of some 8e-5 everywhere), and behind that two Gaussians of that run,
    whose exponents grow away from the centre, have weights of some 3.5 and turn the sign of T twice: at the run's end
    T is above the stop.  The walk ends where the reference's does, and what lies behind, of colour 1e4, reaches nothing.  Bound:
    relative errors of some 1e-6 of weights and 1e-4 of a T that is a product of 1 - 0.9, on colours of up to 1."""
    rng = np.random.default_rng(13)
    n, lists = 700, []
    for at in (64, 70, 126, 128, 200, 254, 320, 500):
        xy = rng.uniform(0, 1, (n, 2)) * block
        co = np.stack([np.full(n, -1e-6), np.zeros(n), np.full(n, -1e-6), np.log2(rng.uniform(0.001, 0.002, n))], 1)
        rgb = rng.uniform(0, 1, (n, 3))
        co[10:13, 3] = np.log2(0.874)               # T 2e-3
        co[at, 3] = np.log2(0.96)
        rgb[at + 2:] = 1e4
        turns = slice(at + 2, at + 4)
        if kind == "flat along y":
            xy[turns] = 1000.0, 5.0
            co[turns] = 2.4e-6, 0.0, 0.0, -0.6
        elif kind == "growing along x and y":
            xy[turns] = 700.0, 700.0
            co[turns] = 2.4e-6, 0.0, 2.4e-6, -0.6
        else:                                       # (the one kind that the multiplied form tells by itself)
            xy[turns] = 1000.0, 5.0
            co[turns] = 2.4e-6, 0.0, -1e-6, -0.6
        lists.append((xy + (0, block[1] * len(lists)), co, rgb))
    W, H = block[0], block[1] * len(lists)
    arrays = column_of_tiles(lists, len(lists))
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    _, ref, _ = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg)
    brightest, err = float(ref.max()), float(np.abs(out - ref).max())
    assert 0.1 < brightest <= 1.0 and err <= 1e-4


@pytest.mark.parametrize("kind", ["above one", "negative"])
@pytest.mark.parametrize("block", BLOCKS)
def test_runs_behind_weights_that_turned_the_transmittance(oracle, block, kind):
    """Weights of 4 at one pixel leave T of that pixel above 1, or far below zero, in front of a later run of the list.
    Above one: the run is opaque (its own T below 1e-4), the pixel not yet, and what lies behind in the run counts.
    Negative: the run has the tile's stop, and a weight of 1.005 behind that turns the pixel's T to above 1e-4: the walk ends at the
    stop.  Bound: relative errors of 1e-4 of T on what colours of up to 1e4 the reference blends, a hundred times less than
    what they are, and 1e-4."""
    rng = np.random.default_rng(14)
    n, lists = 900, []
    for at in (140, 200, 330, 450, 640):
        xy = rng.uniform(0, 1, (n, 2)) * block
        co = np.stack([np.full(n, -1e-6), np.zeros(n), np.full(n, -1e-6), np.log2(rng.uniform(0.0005, 0.001, n))], 1)
        rgb = rng.uniform(0, 1, (n, 3)) * 0.5
        pixel = (5.0, 6.0)
        if kind == "above one":
            turned = slice(70, 72)                       # T 9
            co[at:at + 8, 3] = np.log2(0.7)              # 6.6e-5
            rgb[at + 8:] = 1e4
        else:
            co[10:13, 3] = np.log2(0.83)                 # T 5e-3 everywhere
            turned = slice(70, 77)                       # T -10
            co[at, 3] = np.log2(0.985)                   # the tile's stop
            xy[at + 2] = pixel
            co[at + 2] = -2.0, 0.0, -2.0, 0.0072
            rgb[at] = 0.0
            rgb[at + 2:] = 1e4
        xy[turned] = pixel
        co[turned] = -2.0, 0.0, -2.0, 2.0
        rgb[turned] = 0.0
        lists.append((xy + (0, block[1] * len(lists)), co, rgb))
    W, H = block[0], block[1] * len(lists)
    arrays = column_of_tiles(lists, len(lists))
    bg = np.array([0.25, 0.5, 0.75], np.float32)
    _, ref, _ = oracle.render(W, H, block[0], block[1], *arrays, bg, want_u8=False)
    out, _ = gpu_blend(block, W, H, arrays, bg)
    err, dark = np.abs(out - ref), np.minimum(np.abs(ref), 1.0)
    assert (np.abs(ref) > 2.0).any() == (kind == "above one")
    worst = float((err - 0.01 * (np.abs(ref) - dark)).max())
    assert worst <= 1e-4
