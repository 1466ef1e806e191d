"""The work that a user of this framework has it do, as cases to be timed: frames of synthetic 3D Gaussian
scenes through ``flashgs_amd.rasterizer`` (one frame, or a batch of camera poses), through the operators of
``flash_gaussian_splatting.ops`` in the order of FlashGS's own driver, and through the C ABI with its opt-in
colour sums.

A scene has one of the four layouts of ``flashgs_amd.scenes`` (the distributions are the same, drawn on the
GPU so that millions of Gaussians take milliseconds), a number of Gaussians, a factor on the size of the
splats and a frame size.  Buffers have the sizes of ``render_scene``'s defaults.
"""
import math

import numpy as np
import torch

from flashgs_amd import cabi, scenes
from flashgs_amd.rasterizer import BatchRasterizer, Camera, Rasterizer, Scene, ops

DEVICE = "cuda:0"
MAX_NUM_RENDERED = 2 ** 27      # the defaults of flashgs_amd.rasterizer.render_scene
MAX_NUM_TILES = 2 ** 20


def case(name, via, scene, gaussians, width, height, tile="16x16", spread=1.0, extent=50.0, poses=1):
    """via: "forward" Rasterizer.forward, "batch" BatchRasterizer.render with two frames in flight, "ops" the
    operators one by one, "f16" the C ABI with the colour sums on the matrix unit.  spread: factor on the splat
    sizes.  extent: half side of the city.  poses: frames of one pass."""
    return {"name": name, "via": via, "scene": scene, "gaussians": gaussians, "width": width, "height": height,
            "tile": tile, "spread": spread, "extent": extent, "poses": poses}


def listed():
    return [
        # the smallest call: a thumbnail of a small object, where launches and host work are all there is
        case("thumbnail_2k", "forward", "box", 2_000, 256, 192),
        # a small scene in an interactive window
        case("window_100k_720p", "forward", "box", 100_000, 1280, 720),
        # an object-centred capture at full HD: few tiles, some of them with long lists
        case("clusters_1M_1080p", "forward", "clusters", 1_000_000, 1920, 1080),
        # the headline: a city block at 4K
        case("city_3M_4K", "forward", "city", 3_000_000, 3840, 2160),
        # a large city at 8K, two splats in a hundred much larger than the rest
        case("city_8M_8K", "forward", "city_big", 8_000_000, 7680, 4320, extent=200.0),
        # the same with splats five times as large: more than 100M pairs, the largest frame
        case("dense_8M_8K", "forward", "city_big", 8_000_000, 7680, 4320, spread=5.0, extent=200.0),
        # a camera inside the scene, close to thin 100:1 splats whose rectangles cover much of the screen
        case("needles_2M_4K", "forward", "orbit", 2_000_000, 3840, 2160),
        # the wide tile shapes, at sizes that are no multiple of a tile
        case("tiles_32x16_1599x901", "forward", "city", 500_000, 1599, 901, tile="32x16"),
        case("tiles_32x32_1440p", "forward", "clusters", 1_000_000, 2560, 1440, tile="32x32"),
        # a camera path rendered as one batch, two frames in flight
        case("path_2M_1080p_x6", "batch", "orbit", 2_000_000, 1920, 1080, poses=6),
        # FlashGS's own driver on the operators: blocking read of the pair count, a new image for every frame
        case("driver_700k_1080p", "ops", "clusters", 700_000, 1920, 1080),
        # the C ABI as a renderer without Python uses it, colour sums with f16 operands, 8-bit and float images
        case("cabi_f16_300k_odd", "f16", "city", 300_000, 1365, 767),
    ]


#: per layout: largest number of Gaussians, frame height and splat factor of a drawn case (all of them stay below
#: the pairs and the time of the dense 8K frame)
RANGES = {"box": (1_000_000, 2160, 2.0), "clusters": (3_000_000, 2160, 1.5), "city": (6_000_000, 4320, 2.0),
          "city_big": (8_000_000, 4320, 2.0), "orbit": (2_000_000, 2160, 1.0)}


def draw(rng):
    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    via = rng.choice(["forward", "forward", "forward", "ops", "batch", "f16"])
    scene = rng.choice(sorted(RANGES))
    most, tallest, widest = RANGES[scene]
    gaussians = int(log_uniform(2_000, most))
    height = int(log_uniform(192, tallest))
    width = int(height * rng.uniform(1.0, 1.78))
    poses = 1
    if via == "batch":
        poses = rng.randint(2, 6)
        gaussians, height = min(gaussians, 2_000_000), min(height, 1440)
        width = min(width, 2560)
    tile = "16x16" if via == "f16" else rng.choice(["16x16", "16x16", "16x16", "32x16", "32x32"])
    return {k: v for k, v in case("", via, scene, gaussians, width, height, tile, round(log_uniform(1.0, widest), 2),
                                  rng.choice([50.0, 200.0]), poses).items() if k != "name"}


# ---- scenes, on the GPU ---------------------------------------------------------------------------------------


class Draws:
    """Random tensors of one generator, in call order."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEVICE)

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=self.g, device=DEVICE)

    def index(self, below, n):
        return torch.randint(0, below, (n,), generator=self.g, device=DEVICE)


def covariances(scale, quat):
    """Upper triangles of R S^2 R^T, as ``scenes.cov3d_from_scale_rotation`` makes them."""
    r, x, y, z = (quat / quat.norm(dim=1, keepdim=True)).unbind(1)
    rows = [[1 - 2 * (y * y + z * z), 2 * (x * y - r * z), 2 * (x * z + r * y)],
            [2 * (x * y + r * z), 1 - 2 * (x * x + z * z), 2 * (y * z - r * x)],
            [2 * (x * z - r * y), 2 * (y * z + r * x), 1 - 2 * (x * x + y * y)]]
    m = [[rows[i][k] * scale[:, k] for k in range(3)] for i in range(3)]
    return torch.stack([m[a][0] * m[b][0] + m[a][1] * m[b][1] + m[a][2] * m[b][2]
                        for a, b in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))], dim=1)


def clusters(d, n):
    centres = d.uniform(-20.0, 20.0, 32, 3)
    return centres[d.index(32, n)] + 3.0 * d.normal(n, 3)


def city(d, n, extent):
    """Half of the points on a noisy ground plane, half on the walls and roofs of 200 boxes."""
    ground, build = n // 2, n - n // 2
    plane = torch.stack([d.uniform(-extent, extent, ground), 0.5 * d.normal(ground), d.uniform(-extent, extent, ground)], dim=1)
    s = extent / 50.0
    cx, cz = d.uniform(-0.9 * extent, 0.9 * extent, 200), d.uniform(-0.9 * extent, 0.9 * extent, 200)
    wx, wz, hy = d.uniform(2.0 * s, 8.0 * s, 200), d.uniform(2.0 * s, 8.0 * s, 200), d.uniform(3.0 * s, 25.0 * s, 200)
    areas = torch.stack([wz * hy, wz * hy, wx * hy, wx * hy, wx * wz], dim=1).reshape(-1)
    upto = torch.cumsum(areas, 0)
    pick = torch.searchsorted(upto, d.uniform(0.0, 1.0, build) * upto[-1]).clamp_(max=999)
    b, face = pick // 5, pick % 5
    u, v = d.uniform(-0.5, 0.5, build), d.uniform(0.0, 1.0, build)
    side = torch.where(face % 2 == 0, 0.5, -0.5)
    x = cx[b] + torch.where(face < 2, side, u) * wx[b]
    z = cz[b] + torch.where(face < 2, u, torch.where(face < 4, side, v - 0.5)) * wz[b]
    y = torch.where(face == 4, hy[b], v * hy[b])
    return torch.cat([plane, torch.stack([x, y, z], dim=1)])


def orbit_position(degrees):
    a = math.radians(degrees)
    return [30.0 * math.sin(a), 5.0, -30.0 * math.cos(a)]


def make_scene(c, seed):
    """(Scene on the GPU, list of Camera) of a case: layouts and distributions of flashgs_amd.scenes."""
    d, n, w, h = Draws(seed), c["gaussians"], c["width"], c["height"]
    turn = 6.0 * (seed % 60)                    # another seed looks from another side, where the layout has sides
    mean_op, sigma_op, target, fov = 0.0, 2.0, [0.0, 0.0, 0.0], 60.0
    if c["scene"] == "box":
        means, logs = d.uniform(-5.0, 5.0, n, 3), -4.0 + 0.5 * d.normal(n, 3)
        sigma_op, fov, places = 1.5, 50.0, [[0.0, 0.5 * k, -15.0] for k in range(c["poses"])]
    elif c["scene"] == "clusters":
        means, logs = clusters(d, n), -3.5 + 0.7 * d.normal(n, 3)
        turns = [math.radians(turn + 6.0 * k) for k in range(c["poses"])]
        places = [[37.6 * math.sin(a), 13.7, -37.6 * math.cos(a)] for a in turns]
    elif c["scene"] == "orbit":
        thin = n // 10
        ang, off = d.uniform(0.0, 2.0 * math.pi, thin), d.normal(thin, 3)
        off *= d.uniform(0.0, 1.0, thin, 1) ** (1.0 / 3.0) / off.norm(dim=1, keepdim=True)
        path = torch.stack([30.0 * torch.sin(ang), torch.full_like(ang, 5.0), -30.0 * torch.cos(ang)], dim=1)
        thin_logs = -4.5 + 0.5 * d.normal(thin, 1).expand(thin, 3).clone()
        thin_logs[:, 0] += math.log(100.0)
        place = torch.rand(n, generator=d.g, device=DEVICE).argsort()      # a random subset of the indices
        means = torch.cat([clusters(d, n - thin), path + off])[place]
        logs = torch.cat([-3.5 + 0.7 * d.normal(n - thin, 3), thin_logs])[place]
        places = [orbit_position(turn + 6.0 * k) for k in range(c["poses"])]
    else:
        means, logs = city(d, n, c["extent"]), -3.0 + 0.8 * d.normal(n, 3)
        logs[:, 2] -= 1.5                       # flat splats
        if c["scene"] == "city_big":
            logs[d.uniform(0.0, 1.0, n) < 0.02] += 2.0
            fov = 70.0
        mean_op = 0.5
        places = [[0.5 * k, 8.0, -0.9 * c["extent"]] for k in range(c["poses"])]
        target = None                           # straight ahead, 15 degrees down
    scene = Scene(torch.device(DEVICE))
    scene.num_vertex = n
    scene.position = means.contiguous()
    scene.shs = torch.cat([0.5 * d.normal(n, 3), 0.05 * d.normal(n, 45)], dim=1).contiguous()
    scene.opacity = torch.sigmoid(mean_op + sigma_op * d.normal(n)).contiguous()
    scene.cov3d = covariances(torch.exp(logs) * c["spread"], d.normal(n, 4)).contiguous()
    cameras = []
    for k, p in enumerate(places):
        at = target if target is not None else [p[0], p[1] + math.sin(math.radians(-15.0)), p[2] + math.cos(math.radians(-15.0))]
        cameras.append(Camera.from_synthetic(scenes.look_at(p, at, w, h, fov), k))
    return scene, cameras


# ---- what is timed --------------------------------------------------------------------------------------------


def prepare(c, seed):
    scene, cameras = make_scene(c, seed)
    state = {"case": c, "scene": scene, "cameras": cameras, "bg": torch.zeros(3, dtype=torch.float32)}
    tile = tuple(int(v) for v in c["tile"].split("x"))
    if c["via"] == "batch":
        state["batch"] = BatchRasterizer(scene, MAX_NUM_RENDERED, MAX_NUM_TILES, frames_in_flight=2, tile=tile)
    else:
        # the ops and C ABI cases use its buffers and not its forward()
        state["rasterizer"] = Rasterizer(scene, MAX_NUM_RENDERED, MAX_NUM_TILES, tile=tile)
    if c["via"] == "f16":
        cabi.load()
        state["pinned"] = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        state["u8"] = torch.zeros((c["height"], c["width"], 3), device=DEVICE, dtype=torch.uint8)
        state["f32"] = torch.zeros((c["height"], c["width"], 3), device=DEVICE, dtype=torch.float32)
    return state


def run(state):
    via = state["case"]["via"]
    if via == "forward":
        r = state["rasterizer"]
        image = r.forward(state["scene"], state["cameras"][0], state["bg"])
        return {"image": image, "pairs": r.num_rendered}
    if via == "batch":
        return {"images": state["batch"].render(state["scene"], state["cameras"], state["bg"])}
    return run_ops(state) if via == "ops" else run_cabi(state)


def run_ops(state):
    """FlashGS example.py:67-94 on the operators."""
    o, s, r, cam = ops(), state["scene"], state["rasterizer"], state["cameras"][0]
    bx, by = r.tile
    r.curr_offset.fill_(0)
    o.preprocess(s.position, s.shs, s.opacity, s.cov3d, cam.width, cam.height, bx, by, cam.position, cam.rotation,
                 cam.focal_x, cam.focal_y, cam.zFar, cam.zNear, r.points_xy, r.rgb_depth, r.conic_opacity,
                 r.gaussian_keys_unsorted, r.gaussian_values_unsorted, r.curr_offset)
    pairs = int(r.curr_offset.cpu()[0])
    o.sort_gaussian(pairs, cam.width, cam.height, bx, by, r.list_sorting_space, r.gaussian_keys_unsorted,
                    r.gaussian_values_unsorted, r.gaussian_keys_sorted, r.gaussian_values_sorted)
    image = torch.zeros((cam.height, cam.width, 3), device=DEVICE, dtype=torch.int8)
    render = {(16, 16): o.render_16x16, (32, 16): o.render_32x16, (32, 32): o.render_32x32}[r.tile]
    render(pairs, cam.width, cam.height, r.points_xy, r.rgb_depth, r.conic_opacity, r.gaussian_keys_sorted,
           r.gaussian_values_sorted, r.ranges, state["bg"], image)
    # with the operators the attribute rows, the tile ranges and the pair count are results too
    return {"image": image, "pairs": pairs, "points_xy": r.points_xy, "rgb_depth": r.rgb_depth, "conic_opacity": r.conic_opacity,
            "ranges": r.ranges[:((cam.width + bx - 1) // bx) * ((cam.height + by - 1) // by)]}


def run_cabi(state):
    """The frame through the C ABI on torch's memory and stream: f16 operands in the colour sums, float image too."""
    s, r, cam = state["scene"], state["rasterizer"], state["cameras"][0]
    stream = torch.cuda.current_stream().cuda_stream
    r.curr_offset.zero_()
    mirror = state["pinned"].data_ptr()
    cabi.preprocess(s.num_vertex, s.position.data_ptr(), s.shs.data_ptr(), s.opacity.data_ptr(), s.cov3d.data_ptr(),
                    cam.width, cam.height, 16, 16, cam.position.numpy(), cam.rotation.numpy(), cam.focal_x, cam.focal_y,
                    cam.zFar, cam.zNear, r.points_xy.data_ptr(), r.rgb_depth.data_ptr(), r.conic_opacity.data_ptr(),
                    r.gaussian_keys_unsorted.data_ptr(), r.gaussian_values_unsorted.data_ptr(), r.curr_offset.data_ptr(),
                    r.MAX_NUM_RENDERED, stream, count_mirror=mirror)
    pairs = cabi.wait_count(mirror)
    cabi.sort_gaussian(pairs, cam.width, cam.height, 16, 16, r.list_sorting_space.data_ptr(), r.SORT_BUFFER_SIZE,
                       r.gaussian_keys_unsorted.data_ptr(), r.gaussian_values_unsorted.data_ptr(),
                       r.gaussian_keys_sorted.data_ptr(), r.gaussian_values_sorted.data_ptr(), stream)
    cabi.render_f32(16, 16, pairs, cam.width, cam.height, r.points_xy.data_ptr(), r.rgb_depth.data_ptr(),
                    r.conic_opacity.data_ptr(), r.gaussian_keys_sorted.data_ptr(), r.gaussian_values_sorted.data_ptr(),
                    r.ranges.data_ptr(), np.zeros(3, np.float32), state["u8"].data_ptr(), state["f32"].data_ptr(), stream,
                    flags=cabi.BLEND_MATRIX_F16)
    return {"image": state["u8"], "colour": state["f32"]}


#: per layout: share of the Gaussians that is seen, Gaussians blended into a pixel on average, and the scene size at
#: which that many are (counted once on frames of the listed sizes; beyond it the pixels are opaque)
SEEN = {"box": (1.0, 56, 100_000), "clusters": (0.93, 222, 1_000_000), "city": (0.72, 180, 600_000),
        "city_big": (0.71, 80, 600_000), "orbit": (0.75, 46, 1_000_000)}


def work(c):
    """Every Gaussian's position, opacity and covariance and the seen ones' 48 coefficients read once, the image
    written once; 19 operations per Gaussian and pixel (two differences, the quadratic form, the product with the
    transmittance, three colour sums)."""
    seen, deep, full = SEEN[c["scene"]]
    deep *= min(1.0, c["gaussians"] * c["spread"] ** 2 / full)
    pixels = c["width"] * c["height"]
    frame = 40 * c["gaussians"] + 192 * seen * c["gaussians"] + 3 * pixels
    return {"bytes": c["poses"] * frame, "flops": c["poses"] * 19.0 * pixels * deep}


def tolerance(c):
    """The 8-bit encode truncates, so a value moves by one step where the fp32 rounding of the colour crosses a step.
    Against an evaluation of the same frames with the exponent's terms in another order 0.001 % to 0.034 % of the values
    move (most of them in the needles case); the attribute rows, ranges and pair counts do not move at all.  With f16
    operands the float image was 1.9e-4 (2-norm) and 8.2e-4 (largest) from the all-fp32 one, and 1 % of the 8-bit
    values differed."""
    if c["via"] == "f16":
        return {"rel": 8e-4, "max": 3.3e-3, "differ": 0.01}
    return {"rel": 0.0, "differ": 0.0014}
