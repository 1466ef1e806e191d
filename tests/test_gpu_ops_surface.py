"""The op surface on the GPU, used the way FlashGS's example.py uses it: ``Rasterizer.forward``
through ``flash_gaussian_splatting.ops`` against the oracle, and the error behaviour of the ops."""
import numpy as np
import pytest
import torch

from flashgs_amd import scenes
from flashgs_amd.rasterizer import Camera, Rasterizer, Scene, TooManyPairs, savePpm

pytestmark = pytest.mark.gpu


def _setup(n=40_000, cap=1 << 19, tile=(16, 16)):
    sc = scenes.config0(n=n)
    scene = Scene(torch.device("cuda:0")).from_arrays(sc.position, sc.shs, sc.opacity, sc.cov3d)
    return sc, scene, Camera.from_synthetic(sc.cameras[0]), Rasterizer(scene, cap, 1 << 14, tile=tile)


@pytest.mark.parametrize("tile", [(16, 16), (32, 16), (32, 32)])
def test_rasterizer_forward_matches_oracle(oracle, tile, tmp_path):
    sc, scene, cam, rast = _setup(tile=tile)
    c0 = sc.cameras[0]
    bg = torch.tensor([0.0, 0.2, 0.4])
    img = rast.forward(scene, cam, bg)
    img2 = rast.forward(scene, cam, bg).cpu().numpy()          # a second frame reuses every buffer
    K = rast.num_rendered
    pre = oracle.preprocess(sc.position, sc.shs, sc.opacity, sc.cov3d, c0.width, c0.height, tile[0], tile[1],
                            c0.position, c0.rotation, c0.focal_x, c0.focal_y, c0.zFar, c0.zNear, 1 << 19)
    assert pre["num_rendered"] == K
    ks, vs = oracle.sort(K, c0.width, c0.height, tile[0], tile[1], pre["keys"], pre["values"])
    assert np.array_equal(rast.gaussian_keys_sorted[:K].cpu().numpy().view(np.uint64), ks)
    assert np.array_equal(rast.gaussian_values_sorted[:K].cpu().numpy().view(np.uint32), vs)
    gx, gy = (c0.width + tile[0] - 1) // tile[0], (c0.height + tile[1] - 1) // tile[1]
    rg = oracle.ranges(K, ks, gx * gy)
    assert np.array_equal(rast.ranges[:gx * gy].cpu().numpy(), rg)
    u8, _, _ = oracle.render(c0.width, c0.height, tile[0], tile[1], pre["points_xy"], pre["rgb_depth"],
                             pre["conic_opacity"], vs, rg, bg.numpy(), want_f32=False)
    d = np.abs(img2.astype(np.int16) - u8.astype(np.int16))
    assert d.max() <= 1 and (d > 0).mean() < 0.02
    path = tmp_path / "frame.ppm"
    savePpm(img, str(path))
    data = path.read_bytes()
    assert data.startswith(b"P6\n%d %d\n255\n" % (c0.width, c0.height))


def test_int8_image_like_the_reference_driver():
    """example.py:89 allocates the image as int8; the op accepts any 1-byte dtype."""
    import flash_gaussian_splatting as fgs
    sc, scene, cam, rast = _setup(n=5000)
    bg = torch.zeros(3)
    ref = rast.forward(scene, cam, bg).clone()
    out = torch.zeros((cam.height, cam.width, 3), device="cuda:0", dtype=torch.int8)
    fgs.ops.render_16x16(rast.num_rendered, cam.width, cam.height, rast.points_xy, rast.rgb_depth, rast.conic_opacity,
                         rast.gaussian_keys_sorted, rast.gaussian_values_sorted, rast.ranges, bg, out)
    assert torch.equal(out.view(torch.uint8), ref)


def test_too_many_pairs_raises():
    sc, scene, cam, _ = _setup(n=40_000)
    small = Rasterizer(scene, 1000, 1 << 14)
    with pytest.raises(TooManyPairs):
        small.forward(scene, cam, torch.zeros(3))


def test_ops_errors_on_the_gpu():
    import flash_gaussian_splatting as fgs
    sc, scene, cam, rast = _setup(n=5000)
    rast.forward(scene, cam, torch.zeros(3))
    K = rast.num_rendered
    tiny = torch.zeros(64, device="cuda:0", dtype=torch.int8)
    with pytest.raises(RuntimeError, match="needed"):            # workspace too small
        fgs.ops.sort_gaussian(K, cam.width, cam.height, 16, 16, tiny, rast.gaussian_keys_unsorted,
                              rast.gaussian_values_unsorted, rast.gaussian_keys_sorted, rast.gaussian_values_sorted)
    with pytest.raises(RuntimeError, match="contiguous"):
        fgs.ops.preprocess(scene.position, scene.shs, scene.opacity, scene.cov3d, cam.width, cam.height, 16, 16,
                           cam.position, cam.rotation, cam.focal_x, cam.focal_y, cam.zFar, cam.zNear,
                           torch.zeros((scene.num_vertex, 4), device="cuda:0")[:, :2], rast.rgb_depth, rast.conic_opacity,
                           rast.gaussian_keys_unsorted, rast.gaussian_values_unsorted, rast.curr_offset)
    with pytest.raises(RuntimeError, match="dtype"):
        fgs.ops.preprocess(scene.position, scene.shs, scene.opacity, scene.cov3d, cam.width, cam.height, 16, 16,
                           cam.position, cam.rotation, cam.focal_x, cam.focal_y, cam.zFar, cam.zNear,
                           rast.points_xy, rast.rgb_depth, rast.conic_opacity,
                           rast.gaussian_keys_unsorted.to(torch.int32), rast.gaussian_values_unsorted, rast.curr_offset)
    with pytest.raises(RuntimeError, match="too small"):
        fgs.ops.render_16x16(K, cam.width, cam.height, rast.points_xy, rast.rgb_depth, rast.conic_opacity,
                             rast.gaussian_keys_sorted, rast.gaussian_values_sorted, rast.ranges[:10], torch.zeros(3),
                             torch.zeros((cam.height, cam.width, 3), device="cuda:0", dtype=torch.uint8))


def test_frames_start_from_the_offset_that_the_frame_before_cleared():
    """Frames of different pair counts in turn, a call of the operator on the rasterizer's offset and a tensor of the caller's
    between them: every count is the one of a rasterizer that has rendered nothing else, and is in curr_offset.  (Looked at after
    every frame; frames that nobody looks at are below.)"""
    import flash_gaussian_splatting as fgs
    sc, scene, cam, rast = _setup(n=5000)
    _, _, cam2, fresh = _setup(n=5000)
    cam2.width, cam2.height = cam.width // 2, cam.height // 2
    bg = torch.zeros(3)
    expected = []
    for c in (cam, cam2):
        _, _, _, once = _setup(n=5000)
        image = once.forward(scene, c, bg).clone()
        expected.append((once.num_rendered, image))
    assert expected[0][0] != expected[1][0]
    for i, c in enumerate((cam, cam2, cam2, cam, cam, cam2, cam)):
        if i == 3:              # as the reference's driver does it
            rast.curr_offset.fill_(0)
            fgs.ops.preprocess(scene.position, scene.shs, scene.opacity, scene.cov3d, cam.width, cam.height, 16, 16,
                               cam.position, cam.rotation, cam.focal_x, cam.focal_y, cam.zFar, cam.zNear,
                               rast.points_xy, rast.rgb_depth, rast.conic_opacity,
                               rast.gaussian_keys_unsorted, rast.gaussian_values_unsorted, rast.curr_offset)
            assert int(rast.curr_offset.cpu()[0]) == expected[0][0]
        if i == 5:
            rast.curr_offset = torch.full((1,), 99, device="cuda:0", dtype=torch.int32)
        image = rast.forward(scene, c, bg)
        count, ref = expected[c is cam2]
        assert rast.num_rendered == count == int(rast.curr_offset.cpu()[0])
        assert torch.equal(image, ref)


@pytest.mark.parametrize("looked_at", [None, 0, 1, 2, 3])
def test_a_caller_may_keep_the_word_of_the_pair_count(looked_at):
    """The rasterizer's offset taken once, before the first frame or after some, and counted in by the operator between frames:
    every frame's count and image are those of a rasterizer that has rendered nothing else, and the tensor holds the
    count of what ran last.  Nobody looks at it: the frames start from the words that the launches before them cleared."""
    import flash_gaussian_splatting as fgs
    sc, scene, cam, rast = _setup(n=5000)
    _, _, cam2, _ = _setup(n=5000)
    cam2.width, cam2.height = cam.width // 2, cam.height // 2
    bg = torch.zeros(3)
    expected = []
    for c in (cam, cam2):
        _, _, _, once = _setup(n=5000)
        image = once.forward(scene, c, bg).clone()
        expected.append((once.num_rendered, image))
    off = None
    for i, c in enumerate((cam, cam2, cam2, cam, cam, cam2, cam, cam2)):
        if i == looked_at:
            off = rast.curr_offset
            assert int(off.cpu()[0]) == rast.num_rendered
        if off is not None:
            off.fill_(0)
            fgs.ops.preprocess(scene.position, scene.shs, scene.opacity, scene.cov3d, cam.width, cam.height, 16, 16,
                               cam.position, cam.rotation, cam.focal_x, cam.focal_y, cam.zFar, cam.zNear,
                               rast.points_xy, rast.rgb_depth, rast.conic_opacity,
                               rast.gaussian_keys_unsorted, rast.gaussian_values_unsorted, off)
            assert int(off.cpu()[0]) == expected[0][0]
        image = rast.forward(scene, c, bg)
        count, ref = expected[c is cam2]
        assert rast.num_rendered == count and torch.equal(image, ref)
        assert off is None or (off is rast.curr_offset and int(off.cpu()[0]) == count)
    assert int(rast.curr_offset.cpu()[0]) == expected[1][0]


def test_the_next_offset_is_cleared_whatever_the_count():
    """preprocess_chained leaves zero in the other word: with Gaussians, without any, where the scan gives up and where an earlier one
    on the stream has."""
    import flash_gaussian_splatting as fgs
    from flashgs_amd import cabi
    sc, scene, cam, rast = _setup(n=5000)
    big = scenes.config0(n=1_200_000)           # more workgroups than the chip holds at once
    big_scene = Scene(torch.device("cuda:0")).from_arrays(big.position, big.shs, big.opacity, big.cov3d)
    big_rast = Rasterizer(big_scene, 1 << 22, 1 << 14)
    none = Scene(torch.device("cuda:0")).from_arrays(sc.position[:0], sc.shs[:0], sc.opacity[:0], sc.cov3d[:0])
    no_rast = Rasterizer(none, 1 << 10, 1 << 14)

    def count(r, s, start):
        off, other = (torch.full((1,), v, device="cuda:0", dtype=torch.int32) for v in (start, 77))
        fgs.ops.preprocess_chained(s.position, s.shs, s.opacity, s.cov3d, cam.width, cam.height, 16, 16,
                                   cam.position, cam.rotation, cam.focal_x, cam.focal_y, cam.zFar, cam.zNear,
                                   r.points_xy, r.rgb_depth, r.conic_opacity,
                                   r.gaussian_keys_unsorted, r.gaussian_values_unsorted, off, r._count, other)
        n = fgs.ops.wait_count(r._count, 60.0)
        torch.cuda.synchronize()
        assert int(other.cpu()[0]) == 0 and int(off.cpu()[0]) == n
        return n

    rast.forward(scene, cam, torch.zeros(3))
    assert count(rast, scene, 0) == rast.num_rendered and count(rast, scene, 5) == rast.num_rendered + 5
    assert count(no_rast, none, 0) == 0 and count(no_rast, none, 41) == 41
    previous = cabi.set_scan_spin_limit(0)
    try:
        assert count(big_rast, big_scene, 0) < 0
    finally:
        cabi.set_scan_spin_limit(previous)
    assert count(rast, scene, 0) < 0             # the scan status is marked
    fgs.ops.reset_scan(rast.ranges)
    assert count(rast, scene, 0) == rast.num_rendered
    image = no_rast.forward(none, cam, torch.zeros(3))
    for _ in range(3):
        assert no_rast.num_rendered == 0 and int(image.max()) == 0
        image = no_rast.forward(none, cam, torch.zeros(3))


@pytest.mark.parametrize("tile", [(16, 16), (32, 16), (32, 32)])
def test_a_frame_in_one_call_is_the_operators_one_by_one(tile):
    """forward against preprocess, sort_gaussian and render on buffers of their own; an image that is refused leaves no count pending, too many pairs
    are reported, and the next frame is whole either way."""
    import flash_gaussian_splatting as fgs
    from flashgs_amd.rasterizer import TooManyPairs
    sc, scene, cam, _ = _setup(n=5000)
    rast, apart = (Rasterizer(scene, 1 << 20, 1 << 14, tile=tile) for _ in range(2))
    bg = torch.tensor([0.1, 0.2, 0.3])
    fgs.ops.preprocess(scene.position, scene.shs, scene.opacity, scene.cov3d, cam.width, cam.height, *tile,
                       cam.position, cam.rotation, cam.focal_x, cam.focal_y, cam.zFar, cam.zNear,
                       apart.points_xy, apart.rgb_depth, apart.conic_opacity,
                       apart.gaussian_keys_unsorted, apart.gaussian_values_unsorted, apart.curr_offset)
    n = int(apart.curr_offset.cpu()[0])
    fgs.ops.sort_gaussian(n, cam.width, cam.height, *tile, apart.list_sorting_space, apart.gaussian_keys_unsorted, apart.gaussian_values_unsorted,
                          apart.gaussian_keys_sorted, apart.gaussian_values_sorted)
    expected = torch.zeros((cam.height, cam.width, 3), device="cuda:0", dtype=torch.uint8)
    getattr(fgs.ops, "render_%dx%d" % tile)(n, cam.width, cam.height, apart.points_xy, apart.rgb_depth, apart.conic_opacity,
                                            apart.gaussian_keys_sorted, apart.gaussian_values_sorted, apart.ranges, bg, expected)
    tiles = -(-cam.width // tile[0]) * -(-cam.height // tile[1])

    def whole():
        image = rast.forward(scene, cam, bg)
        assert rast.num_rendered == n and torch.equal(image, expected)
        for name in ("points_xy", "rgb_depth", "conic_opacity"):
            assert torch.equal(getattr(rast, name), getattr(apart, name))
        assert torch.equal(rast.gaussian_keys_sorted[:n], apart.gaussian_keys_sorted[:n])
        assert torch.equal(rast.gaussian_values_sorted[:n], apart.gaussian_values_sorted[:n])
        assert torch.equal(rast.ranges[:tiles], apart.ranges[:tiles])

    whole()
    for bad in (expected[:-1], expected.cpu(), expected[:, :, :2], expected.float()):
        with pytest.raises(RuntimeError, match="out_color"):
            rast.forward(scene, cam, bg, out=bad)
        whole()
    with pytest.raises(RuntimeError, match="bg_color"):
        rast.forward(scene, cam, bg[:2])
    whole()
    rast.MAX_NUM_RENDERED = n
    with pytest.raises(TooManyPairs, match="%d" % n):
        rast.forward(scene, cam, bg)
    rast.MAX_NUM_RENDERED = n + 1
    whole()


def _write_ply(path, recs):
    props = ["x", "y", "z", "nx", "ny", "nz"] + ["f_dc_%d" % i for i in range(3)] + ["f_rest_%d" % i for i in range(45)] \
        + ["opacity"] + ["scale_%d" % i for i in range(3)] + ["rot_%d" % i for i in range(4)]
    head = "ply\nformat binary_little_endian 1.0\nelement vertex %d\n" % len(recs)
    head += "".join("property float %s\n" % p for p in props) + "end_header\n"
    with open(path, "wb") as fh:
        fh.write(head.encode())
        fh.write(np.ascontiguousarray(recs, dtype="<f4").tobytes())


def test_render_scene_from_ply_and_cameras_json(oracle, tmp_path, capsys):
    """The file path of example.py:105-144: a 3DGS model directory (point_cloud.ply of 62-float
    records + cameras.json) goes through loadPly -> device -> preprocess -> sort -> render -> .ppm,
    and every image is the oracle's image of the same Gaussians (those loadPly returns)."""
    import json
    import flash_gaussian_splatting as fgs
    from flashgs_amd.rasterizer import render_scene
    rng = np.random.default_rng(21)
    n = 30_000
    recs = np.zeros((n, 62), np.float32)
    recs[:, 0:3] = rng.uniform(-5.0, 5.0, (n, 3))
    recs[:, 3:6] = rng.standard_normal((n, 3))                   # normals: ignored by the loader
    recs[:, 6:9] = 0.5 * rng.standard_normal((n, 3))             # f_dc
    recs[:, 9:54] = 0.05 * rng.standard_normal((n, 45))          # f_rest, planar
    recs[:, 54] = 1.5 * rng.standard_normal(n)                   # opacity logit
    recs[:, 55:58] = -3.2 + 0.6 * rng.standard_normal((n, 3))    # log-scales
    recs[:, 58:62] = rng.standard_normal((n, 4)) * 3.0           # quaternion, not normalised
    model = tmp_path / "model"
    ply_dir = model / "point_cloud" / "iteration_30000"
    ply_dir.mkdir(parents=True)
    _write_ply(str(ply_dir / "point_cloud.ply"), recs)
    cams = []
    for k, (w, h, pos) in enumerate([(1280, 720, [0.0, 0.0, -15.0]), (1000, 600, [1.0, -0.5, -13.0])]):
        c = scenes.look_at(pos, [0, 0, 0], w, h, 50.0)
        cams.append(dict(id=k, img_name="view_%d" % k, width=w, height=h, position=[float(v) for v in c.position],
                         rotation=[[float(v) for v in row] for row in c.rotation], fx=c.focal_x, fy=c.focal_y))
    (model / "cameras.json").write_text(json.dumps(cams))

    render_scene(str(model), test_performance=True, MAX_NUM_RENDERED=1 << 20, MAX_NUM_TILES=1 << 13, frames_in_flight=2)
    out = capsys.readouterr().out
    assert "num_vertex = %d" % n in out and "fps = " in out
    assert "batch of 1 cameras, 2 frames in flight" in out          # the second camera has another image size

    num, position, shs, opacity, cov3d = fgs.ops.loadPly(str(ply_dir / "point_cloud.ply"))
    assert num == n
    for cj in cams:
        w, h = cj["width"], cj["height"]
        pos = np.array(cj["position"], np.float32)
        rot = np.array(cj["rotation"], np.float32)
        pre = oracle.preprocess(position.numpy(), shs.numpy(), opacity.numpy(), cov3d.numpy(), w, h, 16, 16, pos, rot,
                                cj["fx"], cj["fy"], 100.0, 0.01, 1 << 20)
        K = pre["num_rendered"]
        assert K > 10_000
        ks, vs = oracle.sort(K, w, h, 16, 16, pre["keys"], pre["values"])
        rg = oracle.ranges(K, ks, ((w + 15) // 16) * ((h + 15) // 16))
        u8, _, _ = oracle.render(w, h, 16, 16, pre["points_xy"], pre["rgb_depth"], pre["conic_opacity"], vs, rg,
                                 np.zeros(3, np.float32), want_f32=False)
        data = (model / "test_out" / ("%s.ppm" % cj["img_name"])).read_bytes()
        head = b"P6\n%d %d\n255\n" % (w, h)
        assert data.startswith(head) and len(data) == len(head) + 3 * w * h
        img = np.frombuffer(data[len(head):], np.uint8).reshape(h, w, 3)
        d = np.abs(img.astype(np.int16) - u8.astype(np.int16))
        assert d.max() <= 1 and (d > 0).mean() < 0.02
        assert img.max() > 100          # not an empty frame


def test_two_rasterizers_on_two_streams_overlapping(oracle):
    """Two renderers with their own buffers on two streams of one device, frames enqueued back to
    back without any ordering between the streams: the library keeps its scratch per stream, so
    both produce exactly what each produces alone (and what the oracle produces)."""
    sc_a = scenes.config0(n=60_000)
    sc_b = scenes.make(1, n=150_000)
    dev = torch.device("cuda:0")
    jobs = []
    for sc in (sc_a, sc_b):
        scene = Scene(dev).from_arrays(sc.position, sc.shs, sc.opacity, sc.cov3d)
        cam = Camera.from_synthetic(sc.cameras[0])
        rast = Rasterizer(scene, 1 << 21, 1 << 14)
        jobs.append((sc, scene, cam, rast, torch.cuda.Stream()))
    bg = torch.tensor([0.1, 0.3, 0.5])
    alone = []
    for sc, scene, cam, rast, _ in jobs:
        alone.append(rast.forward(scene, cam, bg).clone())
        assert rast.num_rendered > 50_000
    torch.cuda.synchronize()
    # both frames are small enough to rank their tiles (the table the blend keeps per stream)
    outs = [[], []]
    for rep in range(6):
        for k, (sc, scene, cam, rast, stream) in enumerate(jobs):
            with torch.cuda.stream(stream):
                outs[k].append(rast.forward(scene, cam, bg).clone())
    torch.cuda.synchronize()
    for k in range(2):
        for img in outs[k]:
            assert torch.equal(img, alone[k])
    # and the image is the oracle's
    sc, scene, cam, rast, _ = jobs[0]
    c0 = sc.cameras[0]
    pre = oracle.preprocess(sc.position, sc.shs, sc.opacity, sc.cov3d, c0.width, c0.height, 16, 16,
                            c0.position, c0.rotation, c0.focal_x, c0.focal_y, c0.zFar, c0.zNear, 1 << 21)
    K = pre["num_rendered"]
    ks, vs = oracle.sort(K, c0.width, c0.height, 16, 16, pre["keys"], pre["values"])
    rg = oracle.ranges(K, ks, ((c0.width + 15) // 16) * ((c0.height + 15) // 16))
    u8, _, _ = oracle.render(c0.width, c0.height, 16, 16, pre["points_xy"], pre["rgb_depth"], pre["conic_opacity"], vs, rg,
                             bg.numpy(), want_f32=False)
    d = np.abs(alone[0].cpu().numpy().astype(np.int16) - u8.astype(np.int16))
    assert d.max() <= 1 and (d > 0).mean() < 0.02
