"""The two-level binning (gs_bin_tiles and its users) at the sizes where its
layout changes: one bin, one chunk and one more Gaussian, the largest view
with 4 x 4-tile bins and the next one, Gaussians over more bins than a lane
handles alone, and record buffers that the first guess does not fill."""
import numpy as np
import pytest
import torch

from oracle.oracle import _rects
from gs_scenes import RenderCfg, make_camera, random_small_scene, target_image
from helpers import assert_image_close

pytestmark = pytest.mark.gpu


def _pre(n, width, height, max_radius, seed):
    rng = np.random.default_rng(seed)
    pre = dict(means2D=rng.uniform(0, 1, (n, 2)) * (width + 40, height + 40) - 20,
               depths=rng.choice([0.5, 1.0, 2.0], n) + rng.integers(0, max(n // 4, 1), n) / max(n, 1),
               conics=np.ones((n, 3)), op2d=np.ones(n), rgb=np.ones((n, 3)))
    pre = {k: np.ascontiguousarray(v, np.float32) for k, v in pre.items()}
    r = np.exp(rng.uniform(0, np.log(max_radius), n)).astype(np.int32)
    r[rng.random(n) < 0.1] = 0  # culled
    pre["radii"] = r
    x0, y0, x1, y1 = _rects(pre["means2D"], r, width, height)
    pre["tiles"] = ((x1 - x0) * (y1 - y0) * (r > 0)).astype(np.int32)
    return pre


@pytest.mark.parametrize("n,width,height,max_radius", [
    (1, 16, 16, 30), (255, 64, 64, 40), (256, 65, 64, 40), (257, 80, 130, 100), (5000, 411, 307, 60),
    (2048, 200, 100, 20), (2049, 200, 100, 20), (16384, 300, 200, 10), (16385, 300, 200, 10),  # sort in one workgroup, or not
    (131_072, 500, 400, 8), (131_073, 500, 400, 8),  # digit counts scanned in the scatter, or in a launch
    (140_000, 500, 400, 12),            # 547 chunks of 256 Gaussians
    (140_000, 64, 64, 6), (140_001, 66, 20, 6),  # one bin and two: a group per chunk
    (262_143, 500, 400, 6), (262_144, 500, 400, 6), (262_657, 64, 64, 4),  # 128 chunks of 256, then of 512
    (3000, 2048, 2048, 300),            # 1024 bins of 4 x 4 tiles
    (3000, 2064, 2048, 300),            # bins of 8 x 8 tiles
    (500, 4080, 4080, 900),             # the largest view: 255 x 255 tiles
    (400, 1920, 1080, 4000),            # most Gaussians cover the view: the record buffer grows
])
def test_binning_equals_sorted_pairs(oracle, n, width, height, max_radius):
    from gs_hip import GsHip
    print("[case] binning", n, width, height, max_radius, flush=True)
    hip = GsHip(0)  # own context: its buffers start empty
    pre = _pre(n, width, height, max_radius, n + width)
    tiles = ((width + 15) // 16) * ((height + 15) // 16)
    keys, vals = oracle.duplicate(pre, n, width, height)
    ks, vs, ranges = oracle.sort_pairs(keys, vals, tiles)
    dev = {k: torch.tensor(v, device=hip.dev) for k, v in pre.items()}
    for _ in range(2):  # the second call finds the buffers grown
        got, rg, K = hip.bin_tiles(dev, width, height)
        assert K == len(vs)
        assert np.array_equal(got.cpu().numpy().view(np.uint32), vs)
        assert np.array_equal(rg.cpu().numpy().view(np.uint32), np.asarray(ranges).reshape(-1))
    assert not hip.check_overflow()


def _wide_scene():
    scene, _, _ = random_small_scene(600, 1, 17, logscale=(-0.6, 0.2), op=(-4.0, 0.5))
    return scene, make_camera((0.0, 0.0, -3.0), 1920, 1072, 60.0)


def test_trainer_redoes_when_records_outgrow_buffer(oracle):
    """A frame whose bin records outgrow the buffer that an earlier small view
    left (its pair count is then cut short too) is redone with larger ones."""
    from gs_hip import GsHip, GsTrainer
    print("[case] trainer record overflow", flush=True)
    hip = GsHip(0)
    scene, near = _wide_scene()
    far = make_camera((0.0, 0.0, -12.0), 64, 48, 60.0)
    cfg = RenderCfg(sh_degree=1, training=True)
    tr = GsTrainer(hip, scene)
    tr.render(far, cfg)
    K = tr.render(near, cfg)
    ref = oracle.forward(scene, near, cfg)
    assert K == len(ref["keys"])
    assert_image_close(tr.buffer("image", (near.height, near.width, 3)).cpu().numpy(), ref["img"])
    assert not hip.check_overflow()


def test_batch_grows_record_buffer(oracle):
    from gs_hip import GsBatch, GsHip, GsTrainer
    print("[case] batch record overflow", flush=True)
    hip = GsHip(0)
    scene, near = _wide_scene()
    small = make_camera((0.0, 0.0, -6.0), 50, 37, 60.0)
    cfg = RenderCfg(sh_degree=1, training=True)
    tr = GsTrainer(hip, scene)
    cams = [small, near]
    b = GsBatch(tr, cams, cfg, [target_image(c.width, c.height, 4) for c in cams])
    K = b.render()
    refs = [oracle.forward(scene, c, cfg) for c in cams]
    assert K == sum(len(r["keys"]) for r in refs)
    for img, r in zip(b.images(), refs):
        assert_image_close(img.cpu().numpy(), r["img"])


@pytest.mark.parametrize("n,width,height,max_radius", [(1, 16, 16, 5), (63, 300, 200, 80), (64, 300, 200, 80),
                                                       (65, 300, 200, 600), (5000, 411, 307, 60), (300, 4200, 300, 900)])
def test_duplicate_keys_equal_oracle(oracle, n, width, height, max_radius):
    """Waves of one, 63, 64 and 65 Gaussians, empty rectangles among them, and
    rectangles of the whole view; a capacity one short drops one pair and says so."""
    from gs_hip import GsHip
    print("[case] duplicate", n, width, height, flush=True)
    hip = GsHip(0)
    pre = _pre(n, width, height, max_radius, 3 * n + width)
    if n == 1:
        pre = dict(pre, radii=np.array([5], np.int32), means2D=np.array([[8.0, 8.0]], np.float32), tiles=np.array([1], np.int32))
    keys, vals = oracle.duplicate(pre, n, width, height)
    dev = {k: torch.tensor(v, device=hip.dev) for k, v in pre.items()}
    offsets, K = hip.scan_tiles(dev["tiles"])
    assert K == len(keys)
    k, v = hip.duplicate(dev, offsets, K, width, height)
    assert np.array_equal(k.cpu().numpy().view(np.uint64), keys)
    assert np.array_equal(v.cpu().numpy().view(np.uint32), vals)
    assert not hip.check_overflow()
    k, v = hip.duplicate(dev, offsets, K, width, height, capacity=K - 1)
    assert np.array_equal(k.cpu().numpy().view(np.uint64)[:K - 1], keys[:K - 1])
    assert hip.check_overflow()


def test_counted_binning_is_dropped_by_other_work(oracle):
    """gs_bin_tiles_place after another binning call on the context fails instead of placing its lists."""
    import ctypes
    from gs_hip import GsHip
    hip = GsHip(0)
    pre = _pre(300, 200, 100, 30, 9)
    dev = {k: torch.tensor(v, device=hip.dev) for k, v in pre.items()}
    K = ctypes.c_longlong()
    ps = hip._pre_struct(dev)
    hip._check(hip.lib.gs_bin_tiles_count(hip.ctx, 300, ctypes.byref(ps), 200, 100, ctypes.byref(K)), "count")
    hip.bin_sorted_words(dev, 200, 100)
    values = torch.empty(max(K.value, 1), dtype=torch.int32, device=hip.dev)
    ranges = torch.empty(2 * 13 * 7, dtype=torch.int32, device=hip.dev)
    assert hip.lib.gs_bin_tiles_place(hip.ctx, values.data_ptr(), values.numel(), ranges.data_ptr()) == 1


def _covering_scene(n, wide, corner=0.0):
    """n Gaussians, the first `wide` of them over all of a 1920 x 1024 view (480
    bins, 7680 tiles, each); the rest behind the camera, or (corner, a size in
    pixels) on the corners where four bins meet, two by two tiles over them."""
    cam = make_camera((0.0, 0.0, -3.0), 1920, 1024, 60.0)
    scene, _, _ = random_small_scene(n, 1, 5, op=(-4.0, 0.3))
    rng = np.random.default_rng(n)
    scene.pos[:] = rng.normal(0.0, 0.01, scene.pos.shape)
    scene.log_scale[:] = np.log(0.9)
    if corner:
        f = cam.width / (2.0 * cam.tan_fovx) / 3.0  # pixels per unit at the origin
        scene.pos[wide:, 0] = rng.integers(-14, 15, n - wide) * 64 / f
        scene.pos[wide:, 1] = rng.integers(-7, 8, n - wide) * 64 / f
        scene.pos[wide:, 2] = 0.0
        scene.log_scale[wide:] = np.log(corner / f)
    else:
        scene.pos[wide:, 2] = -5.0
    return scene, cam


def _batch(hip, scene, cam):
    from gs_hip import GsBatch, GsTrainer
    tr = GsTrainer(hip, scene)
    return tr, GsBatch(tr, [cam], RenderCfg(sh_degree=1, training=True), [target_image(cam.width, cam.height, 6)])


def test_batch_records_have_headroom():
    """A batch whose first measurement just fits the first guess of the record
    buffer (4 a Gaussian and 65536: 66104) takes steps on Gaussians that need a
    little more, as its pair buffer does."""
    from gs_hip import GsHip, train_cfg
    print("[case] batch record headroom", flush=True)
    hip = GsHip(0)
    scene, cam = _covering_scene(142, 137)  # 65760 records
    tr, b = _batch(hip, scene, cam)
    assert b.render() == 137 * 7680
    grown, _ = _covering_scene(142, 142)    # 68160 records
    tr.set_params(grown)
    for i in range(3):
        b.step(train_cfg(lr=1e-6), i)
    res, _ = b.result()
    assert res.pairs == 142 * 7680


@pytest.mark.parametrize("n,wide,grown_wide,corner,what", [(200_000, 1000, 1000, 1.0, "records only"),
                                                           (300, 20, 290, 0.0, "records and pairs"),
                                                           (300, 20, 30, 0.0, "neither")])
def test_batch_render_repeats_a_cut_render(n, wide, grown_wide, corner, what):
    """A render after the parameters changed, whose records or pairs outgrow the
    buffers that an earlier one sized: its count and image are the single
    view's, and the next step is applied."""
    from gs_hip import GsHip, GsTrainer, train_cfg
    print("[case] batch render outgrows", what, flush=True)
    hip = GsHip(0)
    scene, cam = _covering_scene(n, wide)
    tr, b = _batch(hip, scene, cam)
    b.render()
    grown, _ = _covering_scene(n, grown_wide, corner)
    tr.set_params(grown)
    K = b.render()
    single = GsTrainer(hip, grown)
    assert K == single.render(cam, RenderCfg(sh_degree=1, training=True))
    assert torch.equal(b.images()[0], single.buffer("image", (cam.height, cam.width, 3)))
    before = tr.params()[0].copy()
    b.step(train_cfg(lr=1e-3), 0)
    res, _ = b.result()
    assert res.pairs == K
    assert not np.array_equal(tr.params()[0], before)


def test_batch_render_leaves_suppressed_steps_to_their_result():
    """Steps that outgrew the buffers stay unapplied and reported after a render
    that repeats itself with larger ones."""
    from gs_hip import GsError, GsHip, train_cfg
    print("[case] batch render between overflowed steps and their result", flush=True)
    hip = GsHip(0)
    scene, cam = _covering_scene(300, 20)
    tr, b = _batch(hip, scene, cam)
    b.render()
    grown, _ = _covering_scene(300, 290)
    tr.set_params(grown)
    before = tr.params()[0].copy()
    b.step(train_cfg(lr=1e-3), 0)
    b.step(train_cfg(lr=1e-3), 1)
    assert b.render() == 290 * 7680
    with pytest.raises(GsError, match="2 step.s. were not applied"):
        b.result()
    assert np.array_equal(tr.params()[0], before)
    b.step(train_cfg(lr=1e-3), 0)
    b.result()
    assert not np.array_equal(tr.params()[0], before)


class _Array:
    def __init__(self, address, shape):
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(address, False), version=3)


def test_batch_result_measures_after_the_trainers_stream():
    """The result of an overflowed step sizes the buffers from the parameters as
    the work already queued on the trainer's stream leaves them, here behind a
    tenth of a second of matrix products: the redo then fits."""
    from gs_hip import GsError, GsHip, train_cfg
    print("[case] batch result behind queued parameter writes", flush=True)
    hip = GsHip(0)
    scene, cam = _covering_scene(300, 20)
    tr, b = _batch(hip, scene, cam)
    b.render()
    tr.set_params(_covering_scene(300, 100)[0])
    more = torch.tensor(_covering_scene(300, 290)[0].pos, device=hip.dev)
    pos = torch.as_tensor(_Array(tr.lib.gs_trainer_buffer(tr.tr, b"param_pos"), (300, 3)), device=hip.dev)
    a = torch.zeros((8192, 8192), dtype=torch.bfloat16, device=hip.dev)
    out = torch.empty_like(a)
    torch.mm(a, a, out=out)
    torch.cuda.synchronize()
    b.step(train_cfg(lr=1e-6), 0)
    for _ in range(100):
        torch.mm(a, a, out=out)
    pos.copy_(more)
    with pytest.raises(GsError, match="not applied"):
        b.result()
    b.step(train_cfg(lr=1e-6), 0)
    res, _ = b.result()
    assert res.pairs == 290 * 7680


@pytest.mark.parametrize("graph", [True, False])
def test_batch_step_whose_records_alone_outgrow_their_buffer(graph):
    """Steps (replayed from a graph, or not) whose records do not fit though their
    pairs would: parameters and moments stay, the error names the records, and
    the redo is the step of a batch that never overflowed."""
    from gs_hip import GsBatch, GsError, GsHip, GsTrainer, train_cfg
    print("[case] batch step outgrows its records", graph, flush=True)
    hip = GsHip(0)
    scene, cam = _covering_scene(200_000, 1000)
    cfg, gts, tc = RenderCfg(sh_degree=1, training=True), [target_image(cam.width, cam.height, 6)], train_cfg(lr=1e-3)
    tr = GsTrainer(hip, scene)
    b = GsBatch(tr, [cam], cfg, gts, use_graph=graph)
    b.render()
    grown, _ = _covering_scene(200_000, 1000, 1.0)
    tr.set_params(grown)

    def state(t):
        hip.sync()
        return {f"{a}_{k}": t.buffer(f"{a}_{k}", (t.n, w)).cpu().numpy() for a in ("param", "adam_m", "adam_v")
                for k, w in (("pos", 3), ("scale", 3), ("rot", 4), ("sh", 12), ("op", 1))}

    before = state(tr)
    b.step(tc, 0)
    b.step(tc, 1)
    with pytest.raises(GsError, match="bin records.* 2 step.s. were not applied"):
        b.result()
    for k, x in state(tr).items():
        assert np.array_equal(x, before[k]), k
    b.step(tc, 0)
    res, _ = b.result()
    clean = GsTrainer(hip, grown)
    bc = GsBatch(clean, [cam], cfg, gts, use_graph=graph)
    bc.step(tc, 0)
    ref, _ = bc.result()
    assert res.pairs == ref.pairs and res.loss == ref.loss
    want = state(clean)
    for k, x in state(tr).items():
        if k not in ("adam_m_rot", "adam_v_rot"):  # the scales are equal: no rotation gradient but rounding
            # float atomics in another order: 1e-3, as gradients between runs
            assert np.linalg.norm(x - want[k]) <= 1e-3 * np.linalg.norm(want[k]), k


@pytest.mark.parametrize("who", ["bin_tiles", "trainer"])
def test_growing_records_keep_the_overflow_flag(who):
    """Pairs that gs_duplicate_keys dropped are still reported after a binning
    whose bin records outgrew their buffer and were counted again."""
    from gs_hip import GsHip, GsTrainer
    print("[case] overflow flag kept", who, flush=True)
    hip = GsHip(0)
    small = {k: torch.tensor(v, device=hip.dev) for k, v in _pre(300, 200, 100, 30, 9).items()}
    # 48000 records, then 87600 for a first guess of 80000; the trainer's pairs keep fitting
    scene, cam = _covering_scene(10_000, 100)
    grown, _ = _covering_scene(10_000, 100, 1.0)
    cfg = RenderCfg(sh_degree=1, training=True)
    if who == "trainer":
        tr = GsTrainer(hip, scene)
        tr.render(cam, cfg)
        tr.set_params(grown)
    offsets, K = hip.scan_tiles(small["tiles"])
    hip.duplicate(small, offsets, K, 200, 100, capacity=K - 1)
    if who == "trainer":
        K = tr.render(cam, cfg)
    else:
        _, _, K = hip.bin_tiles(hip.preprocess(hip.upload_scene(grown), cam, cfg), cam.width, cam.height)
    assert K == 100 * 7680 + 9900 * 4
    assert hip.check_overflow()
    assert not hip.check_overflow()


def test_workspace_of_a_view_with_few_bins():
    """A Gaussian has one record per bin at most: a view of one bin reserves an
    eighth of the records that a view of eight or more does."""
    from gs_hip import GsHip
    print("[case] record workspace", flush=True)
    n = 1_000_000

    def used(width):
        dev = {k: torch.tensor(v, device="cuda") for k, v in _pre(n, width, 64, 3, 1).items()}
        hip = GsHip(0)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        hip.bin_tiles(dev, width, 64)
        torch.cuda.synchronize()
        got = free - torch.cuda.mem_get_info()[0]
        del hip, dev
        torch.cuda.empty_cache()
        return got

    used(64)  # code objects and torch's own pools
    assert used(512) - used(64) >= 7 * 8 * n
