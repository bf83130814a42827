"""GPU parity tests: every HIP stage against the CPU oracle on the same inputs,
and the whole GPU path against the reference's golden vectors.

Bars: binning/sort/tile ranges bit-exact given identical inputs; images and
per-Gaussian float outputs within 1e-4 max-abs; gradients within 1e-3 relative
(normalised by the largest entry of each array); Adam bit-exact.
"""
import sys

import numpy as np
import pytest
import torch

from gs_hip import GsError
from gs_scenes import (RenderCfg, gaussians_clusters, make_camera, make_workload, random_small_scene,
                       target_image)
from helpers import (IMAGE_TOL, assert_grad_close, assert_image_close, load_golden, rel_err, scene_dirs, u32)

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


def _np(t):
    return t.detach().cpu().numpy()


SMALL_CASES = [(n, deg, seed) for n, deg, seed in [(3, 0, 1), (40, 1, 2), (200, 2, 3), (500, 3, 4), (2000, 3, 5)]]


@pytest.mark.parametrize("n,deg,seed", SMALL_CASES)
def test_preprocess_matches_oracle(hip, oracle, n, deg, seed):
    _say("preprocess", n, deg, seed)
    scene, cam, gt = random_small_scene(n, deg, seed, width=96, height=72)
    cfg = RenderCfg(sh_degree=3, training=True)
    p = hip.upload_scene(scene)
    pre = hip.preprocess(p, cam, cfg)
    g = oracle.activate(scene)
    ref = oracle.preprocess(g, n, deg, scene.max_coeffs, cam, cfg, cache=False)
    assert np.array_equal(_np(pre["radii"]), ref["radii"])
    assert np.array_equal(_np(pre["tiles"]), ref["tiles"])
    for k in ["means2D", "depths", "conics", "op2d", "rgb"]:
        d = np.abs(_np(pre[k]) - ref[k]).max()
        assert d <= 1e-4, (k, d)


def test_activation_matches_oracle(hip, oracle):
    _say("activate")
    scene, cam, gt = random_small_scene(5000, 3, 11)
    p = hip.upload_scene(scene)
    a = hip.activate(p)
    ref = oracle.activate(scene)
    for k in ["pos", "rot", "sh"]:
        assert np.array_equal(_np(a[k]), ref[k].reshape(_np(a[k]).shape)), k
    # exp(scale) and the sigmoid use the device restatement of the CPU's expf
    for k in ["scale", "op"]:
        assert np.array_equal(_np(a[k]), ref[k].reshape(_np(a[k]).shape)), k


def test_exp_matches_cpu_expf_wide_range(hip, oracle):
    """The device exponential (exp(log-scale) and the opacity sigmoid of the
    activation) against the CPU path's expf, bit for bit, on 3 x 2^20 float
    bit patterns drawn uniformly over [-110, 95] plus the special values."""
    _say("exp wide range")
    from gs_scenes import RawScene
    rng = np.random.Generator(np.random.Philox(2024))
    lo, hi = np.float32(-110.0).view(np.uint32), np.float32(95.0).view(np.uint32)
    neg = rng.integers(np.float32(0.0).view(np.uint32) | 0x80000000, lo, size=1 << 20, dtype=np.uint64)
    pos = rng.integers(0, hi, size=1 << 20, dtype=np.uint64)
    vals = np.concatenate([neg.astype(np.uint32).view(np.float32), pos.astype(np.uint32).view(np.float32),
                           np.float32([np.inf, -np.inf, np.nan, 0.0, -0.0, 88.72283, 88.72284, -103.97208,
                                       -103.97209, -87.33655, 1e-45, -1e-45])])
    vals = np.resize(vals, (len(vals) // 3 + 1) * 3).astype(np.float32)
    n = len(vals) // 3
    scene = RawScene(pos=np.zeros((n, 3), np.float32), log_scale=vals.reshape(n, 3).copy(),
                     rot=np.tile(np.float32([1, 0, 0, 0]), (n, 1)), sh=np.zeros((n, 1, 3), np.float32),
                     opacity_logit=vals[:n].copy(), sh_degree=0)
    a = hip.activate(hip.upload_scene(scene))
    ref = oracle.activate(scene)
    for k in ["scale", "op"]:
        got, want = _np(a[k]).ravel(), ref[k].ravel()
        same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
        assert same.all(), (k, int((~same).sum()), got[~same][:4], want[~same][:4])


@pytest.mark.parametrize("n,deg,seed", SMALL_CASES[1:] + [(10000, 0, 0)])
def test_binning_and_sort_bitexact(hip, oracle, n, deg, seed):
    """Identical preprocess outputs in -> identical keys, values, ranges out."""
    _say("binning+sort", n, deg, seed)
    if n == 10000:
        scene, cams, _ = make_workload("10k_256")
        cam = cams[0]
    else:
        scene, cam, _ = random_small_scene(n, deg, seed, width=160, height=120)
    cfg = RenderCfg(sh_degree=3, training=True)
    g = oracle.activate(scene)
    ref = oracle.preprocess(g, scene.n, scene.sh_degree, scene.max_coeffs, cam, cfg, cache=False)
    keys_ref, vals_ref = oracle.duplicate(ref, scene.n, cam.width, cam.height)
    ks_ref, vs_ref, rg_ref = oracle.sort_pairs(keys_ref, vals_ref, cam.num_tiles)
    d = hip.dev
    pre = dict(means2D=torch.tensor(ref["means2D"], device=d), depths=torch.tensor(ref["depths"], device=d),
               radii=torch.tensor(ref["radii"], device=d), tiles=torch.tensor(ref["tiles"], device=d))
    offsets, K = hip.scan_tiles(pre["tiles"])
    assert K == len(keys_ref)
    assert np.array_equal(u32(offsets), np.cumsum(ref["tiles"]).astype(np.uint32))
    keys, vals = hip.duplicate(pre, offsets, K, cam.width, cam.height)
    assert np.array_equal(u32(keys), keys_ref)
    assert np.array_equal(u32(vals), vals_ref)
    ks, vs, ranges = hip.sort_pairs(keys, vals, cam.num_tiles)
    assert np.array_equal(u32(ks), ks_ref)
    assert np.array_equal(u32(vs), vs_ref)
    assert np.array_equal(u32(ranges), rg_ref)


@pytest.mark.parametrize("n,deg,seed", SMALL_CASES[1:] + [(10000, 0, 0)])
@pytest.mark.parametrize("radix_bits", [6, 8])
def test_depth_ordered_binning_bitexact(hip, oracle, n, deg, seed, radix_bits):
    """gs_bin_sorted_words: same per-tile Gaussian lists as the reference's
    duplicate-with-keys + stable 64-bit sort, bit for bit."""
    _say("depth-ordered binning", n, deg, seed, radix_bits)
    if n == 10000:
        scene, cams, _ = make_workload("10k_256")
        cam = cams[0]
    else:
        scene, cam, _ = random_small_scene(n, deg, seed, width=160, height=120)
    cfg = RenderCfg(sh_degree=3, training=True)
    g = oracle.activate(scene)
    ref = oracle.preprocess(g, scene.n, scene.sh_degree, scene.max_coeffs, cam, cfg, cache=False)
    if n == 200:  # force depth ties: equal depths must keep index order
        ref["depths"][::3] = ref["depths"][0]
    keys_ref, vals_ref = oracle.duplicate(ref, scene.n, cam.width, cam.height)
    ks_ref, vs_ref, rg_ref = oracle.sort_pairs(keys_ref, vals_ref, cam.num_tiles)
    pre = _to_dev(hip, {k: ref[k] for k in ["means2D", "depths", "conics", "op2d", "rgb", "radii", "tiles"]})
    hip.set_tuning(radix_bits=radix_bits)
    words, ranges, K = hip.bin_sorted_words(pre, cam.width, cam.height)
    hip.set_tuning(radix_bits=8)
    assert K == len(keys_ref)
    w = u32(words)
    assert np.array_equal((w & np.uint64(0xFFFFFFFF)).astype(np.uint32), vs_ref)
    assert np.array_equal((w >> np.uint64(32)).astype(np.uint32), (ks_ref >> np.uint64(32)).astype(np.uint32))
    assert np.array_equal(u32(ranges), rg_ref)


@pytest.mark.parametrize("n,deg,seed", SMALL_CASES[1:] + [(10000, 0, 0)])
def test_direct_binning_bitexact(hip, oracle, n, deg, seed):
    """gs_bin_tiles: values and ranges equal to the reference's
    duplicate-with-keys + stable 64-bit sort, bit for bit."""
    _say("direct binning", n, deg, seed)
    if n == 10000:
        scene, cams, _ = make_workload("10k_256")
        cam = cams[0]
    else:
        scene, cam, _ = random_small_scene(n, deg, seed, width=160, height=120)
    cfg = RenderCfg(sh_degree=3, training=True)
    g = oracle.activate(scene)
    ref = oracle.preprocess(g, scene.n, scene.sh_degree, scene.max_coeffs, cam, cfg, cache=False)
    if n == 200:  # force depth ties: equal depths must keep index order
        ref["depths"][::3] = ref["depths"][0]
    keys_ref, vals_ref = oracle.duplicate(ref, scene.n, cam.width, cam.height)
    ks_ref, vs_ref, rg_ref = oracle.sort_pairs(keys_ref, vals_ref, cam.num_tiles)
    pre = _to_dev(hip, {k: ref[k] for k in ["means2D", "depths", "conics", "op2d", "rgb", "radii", "tiles"]})
    vals, ranges, K = hip.bin_tiles(pre, cam.width, cam.height)
    assert K == len(keys_ref)
    assert np.array_equal(u32(vals), vs_ref)
    assert np.array_equal(u32(ranges), rg_ref)


@pytest.mark.parametrize("width,height", [(2080, 2080), (2032, 2032)])
def test_direct_binning_bitexact_large_view(hip, oracle, width, height):
    """Both bin sizes: 2032 x 2032 (127 x 127 tiles) has 1024 bins of 4 x 4
    tiles, 2080 x 2080 (130 x 130 tiles) would have more and takes bins of 8 x 8.
    Values and ranges equal the reference's duplicate + stable sort."""
    _say("direct binning large view", width, height)
    scene, cam, _ = random_small_scene(3000, 1, 23, width=width, height=height)
    cfg = RenderCfg(sh_degree=3, training=True)
    g = oracle.activate(scene)
    ref = oracle.preprocess(g, scene.n, scene.sh_degree, scene.max_coeffs, cam, cfg, cache=False)
    keys_ref, vals_ref = oracle.duplicate(ref, scene.n, cam.width, cam.height)
    ks_ref, vs_ref, rg_ref = oracle.sort_pairs(keys_ref, vals_ref, cam.num_tiles)
    assert len(keys_ref) > 10000
    pre = _to_dev(hip, {k: ref[k] for k in ["means2D", "depths", "conics", "op2d", "rgb", "radii", "tiles"]})
    vals, ranges, K = hip.bin_tiles(pre, cam.width, cam.height)
    assert K == len(keys_ref)
    assert np.array_equal(u32(vals), vs_ref)
    assert np.array_equal(u32(ranges), rg_ref)


def test_direct_binning_capacity_and_empty(hip, oracle):
    """Capacity errors report K without writing; an all-culled scene gives
    K = 0 and zero ranges."""
    _say("direct binning capacity/empty")
    scene, cam, _ = random_small_scene(500, 1, 88, width=96, height=80)
    cfg = RenderCfg(sh_degree=3, training=True)
    g = oracle.activate(scene)
    ref = oracle.preprocess(g, scene.n, scene.sh_degree, scene.max_coeffs, cam, cfg, cache=False)
    pre = _to_dev(hip, {k: ref[k] for k in ["means2D", "depths", "conics", "op2d", "rgb", "radii", "tiles"]})
    K_ref = int(ref["tiles"].astype(np.int64).sum())
    with pytest.raises(GsError):
        hip.bin_tiles(pre, cam.width, cam.height, capacity=max(K_ref - 1, 1))
    vals, ranges, K = hip.bin_tiles(pre, cam.width, cam.height, capacity=K_ref)
    assert K == K_ref
    culled = dict(ref)
    culled["radii"] = np.zeros_like(ref["radii"])
    culled["tiles"] = np.zeros_like(ref["tiles"])
    pre0 = _to_dev(hip, {k: culled[k] for k in ["means2D", "depths", "conics", "op2d", "rgb", "radii", "tiles"]})
    vals, ranges, K = hip.bin_tiles(pre0, cam.width, cam.height)
    assert K == 0
    assert not u32(ranges).any()


@pytest.mark.parametrize("radix_bits", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("count", [1, 63, 4096, 4097, 100_003])
def test_radix_sort_stable_random_keys(hip, count, radix_bits):
    """Random 64-bit keys with many ties: equal to numpy's stable argsort."""
    _say("radix", count, radix_bits)
    rng = np.random.default_rng(count * 10 + radix_bits)
    hi = rng.integers(0, 50, count, dtype=np.uint64)
    lo = rng.integers(0, 1 << 20, count, dtype=np.uint64) & np.uint64(0xFFFF0)  # ties
    keys = (hi << np.uint64(32)) | lo
    vals = np.arange(count, dtype=np.uint32)
    order = np.argsort(keys, kind="stable")
    kt = torch.tensor(keys.view(np.int64), device=hip.dev)
    vt = torch.tensor(vals.view(np.int32), device=hip.dev)
    ko, vo = hip.radix_sort(kt, vt, key_bits=38, radix_bits=radix_bits)
    assert np.array_equal(u32(ko), keys[order])
    assert np.array_equal(u32(vo), vals[order])


@pytest.mark.parametrize("radix_bits", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("key_bits", [32, 38])
def test_radix_sort_ignores_bits_above_key_bits(hip, key_bits, radix_bits):
    """Keys whose bits above key_bits are set (the depth-sort words carry the
    Gaussian index there): the order is numpy's stable argsort of the low
    key_bits, and whole keys travel.  A last digit that reads past key_bits
    breaks this whenever radix_bits does not divide key_bits."""
    _say("radix high bits", key_bits, radix_bits)
    count = 50_000
    rng = np.random.default_rng(key_bits * 10 + radix_bits)
    low = rng.integers(0, 1 << 12, count, dtype=np.uint64) << np.uint64(key_bits - 12)  # ties
    high = rng.integers(0, 1 << 20, count, dtype=np.uint64) << np.uint64(key_bits)
    keys = high | low
    vals = np.arange(count, dtype=np.uint32)
    order = np.argsort(keys & np.uint64((1 << key_bits) - 1), kind="stable")
    kt = torch.tensor(keys.view(np.int64), device=hip.dev)
    vt = torch.tensor(vals.view(np.int32), device=hip.dev)
    ko, vo = hip.radix_sort(kt, vt, key_bits=key_bits, radix_bits=radix_bits)
    assert np.array_equal(u32(ko), keys[order])
    assert np.array_equal(u32(vo), vals[order])


@pytest.mark.parametrize("radix_bits", [4, 5, 6, 7, 8])
def test_radix_sort_large_many_tiles(hip, radix_bits):
    """Above 4M keys (4096-key blocks, ~1300 of them) every digit width with at
    most eight passes runs the one-sweep passes, whose look-back crosses many
    blocks (4-bit digits need ten passes over 40 bits and keep the three-launch
    passes); 40-bit keys with heavy ties and a near-constant top digit, a count
    that is no multiple of the block size."""
    _say("radix large", radix_bits)
    rng = np.random.default_rng(11 + radix_bits)
    n = 5_300_001
    keys = (rng.integers(0, 1 << 20, n, dtype=np.uint64) << np.uint64(20)) | rng.integers(0, 3, n, dtype=np.uint64)
    keys[rng.integers(0, n, 1000)] |= np.uint64(1 << 39)
    vals = np.arange(n, dtype=np.uint32)
    order = np.argsort(keys, kind="stable")
    kt = torch.tensor(keys.view(np.int64), device=hip.dev)
    vt = torch.tensor(vals.view(np.int32), device=hip.dev)
    ko, vo = hip.radix_sort(kt, vt, key_bits=40, radix_bits=radix_bits)
    assert np.array_equal(u32(ko), keys[order])
    assert np.array_equal(u32(vo), vals[order])


def test_radix_sort_48m_pair_keys(hip):
    """A sort the size of the 1080p pair list (48M keys, 45-bit tile | depth
    keys as the duplicate step makes them, sorted twice in a row): equal to
    torch's stable sort on the device."""
    _say("radix 48m")
    n = 48_000_017
    g = torch.Generator(device=hip.dev).manual_seed(5)
    tile = torch.randint(0, 8160, (n,), device=hip.dev, generator=g, dtype=torch.int64)
    depth = torch.rand(n, device=hip.dev, generator=g) * 8.0 + 0.5
    keys = (tile << 32) | (depth.view(torch.int32).to(torch.int64) & 0xFFFFFFFF)
    keys[::97] = keys[5]  # ties
    vals = torch.arange(n, device=hip.dev, dtype=torch.int32)
    ref_k, ref_i = torch.sort(keys, stable=True)
    for _ in range(2):
        ko, vo = hip.radix_sort(keys, vals, key_bits=45, radix_bits=8)
        torch.cuda.synchronize()
        assert torch.equal(ko, ref_k)
        assert torch.equal(vo, ref_i.to(torch.int32))


def test_radix_sort_full_64bit(hip):
    _say("radix 64-bit")
    rng = np.random.default_rng(7)
    keys = rng.integers(0, np.iinfo(np.int64).max, 50_000, dtype=np.int64).view(np.uint64)
    keys[::7] = keys[3]  # ties
    keys[5] = np.uint64(0xFFFFFFFFFFFFFFFF)
    vals = np.arange(keys.size, dtype=np.uint32)
    order = np.argsort(keys, kind="stable")
    ko, vo = hip.radix_sort(torch.tensor(keys.view(np.int64), device=hip.dev),
                            torch.tensor(vals.view(np.int32), device=hip.dev), key_bits=64)
    assert np.array_equal(u32(ko), keys[order])
    assert np.array_equal(u32(vo), vals[order])


def test_sort_empty_and_tile_ranges_edge_cases(hip, oracle):
    _say("sort edge cases")
    # sorter_cpu known answers (test_sorter.cpp:6-102): empty, single, empty tile in the middle
    for keys, vals, tiles in [
        (np.array([], np.uint64), np.array([], np.uint32), 1),
        (np.array([42], np.uint64), np.array([7], np.uint32), 1),
        (np.array([(1 << 32) | 3, 1, 2], np.uint64), np.array([0, 1, 2], np.uint32), 2),
        (np.array([1, (2 << 32) | 2], np.uint64), np.array([0, 1], np.uint32), 3),
    ]:
        ks_ref, vs_ref, rg_ref = oracle.sort_pairs(keys, vals, tiles)
        ks, vs, rg = hip.sort_pairs(torch.tensor(keys.view(np.int64), device=hip.dev),
                                    torch.tensor(vals.view(np.int32), device=hip.dev), tiles)
        assert np.array_equal(u32(ks), ks_ref)
        assert np.array_equal(u32(vs), vs_ref)
        assert np.array_equal(u32(rg), rg_ref)


def _oracle_stage_inputs(oracle, scene, cam, cfg):
    f = oracle.forward(scene, cam, cfg)
    return f


def _to_dev(hip, pre):
    d = hip.dev
    out = {}
    for k, v in pre.items():
        out[k] = torch.tensor(np.ascontiguousarray(v), device=d)
    return out


@pytest.mark.parametrize("n,deg,seed,bg", [(40, 1, 2, (0, 0, 0)), (500, 3, 4, (0.2, 0.5, 1.0)), (2000, 3, 5, (0, 0, 0))])
@pytest.mark.parametrize("batch", [64, 256, 512])
def test_raster_fwd_matches_oracle(hip, oracle, n, deg, seed, bg, batch):
    _say("raster fwd", n, deg, seed, batch)
    scene, cam, gt = random_small_scene(n, deg, seed, width=100, height=75)
    cfg = RenderCfg(sh_degree=3, training=True, bg_color=bg)
    f = _oracle_stage_inputs(oracle, scene, cam, cfg)
    pre = _to_dev(hip, {k: f["pre"][k] for k in ["means2D", "conics", "op2d", "rgb", "radii"]})
    vs = torch.tensor(f["values_sorted"].view(np.int32), device=hip.dev)
    rg = torch.tensor(f["ranges"].view(np.int32), device=hip.dev)
    hip.set_tuning(raster_batch=batch)
    img, px = hip.raster_fwd(pre, vs, rg, cam.width, cam.height, bg)
    hip.set_tuning(raster_batch=256)
    assert_image_close(_np(img), f["img"])
    assert np.abs(_np(px["T_final"]) - f["T_final"]).max() <= 1e-5
    mism = int((_np(px["n_contrib"]) != f["n_contrib"]).sum())
    assert mism == 0, mism
    assert np.array_equal(u32(px["last_contrib"]), f["last_contrib"])


@pytest.mark.parametrize("n,deg,seed", [(500, 3, 4), (2000, 3, 5)])
def test_raster_inv_depth_matches_oracle(hip, oracle, n, deg, seed):
    """gs_raster_inv_depth (Rasterizer::rasterize's out_depth) from the
    forward's pixel state, against the oracle on the same stage inputs."""
    from oracle.oracle import inv_depth_oracle
    _say("inv depth", n, deg, seed)
    scene, cam, gt = random_small_scene(n, deg, seed, width=100, height=75)
    cfg = RenderCfg(sh_degree=3, training=True)
    f = _oracle_stage_inputs(oracle, scene, cam, cfg)
    pre = _to_dev(hip, {k: f["pre"][k] for k in ["means2D", "conics", "op2d", "rgb", "radii", "depths"]})
    vs = torch.tensor(f["values_sorted"].view(np.int32), device=hip.dev)
    rg = torch.tensor(f["ranges"].view(np.int32), device=hip.dev)
    img, px = hip.raster_fwd(pre, vs, rg, cam.width, cam.height)
    inv = _np(hip.raster_inv_depth(pre, vs, rg, cam.width, cam.height, px))
    ref = inv_depth_oracle(f["pre"], f["values_sorted"], f["ranges"], cam.width, cam.height)
    assert ref.max() > 0
    # The replay restates the reference's alpha (exact expf) and blend, so it is
    # bit-exact wherever the forward stopped at the reference's last
    # contributor; the forward's own alphas may differ by an ulp, which can move
    # its transmittance stop by one Gaussian (contributing alpha T < 1e-4).
    same = _np(px["last_contrib"]).astype(np.int64) == f["last_contrib"].astype(np.int64)
    assert same.mean() > 0.99, same.mean()
    np.testing.assert_array_equal(inv[same], ref[same])
    assert np.abs(inv - ref).max() <= IMAGE_TOL * max(1.0, float(ref.max()))


def test_l1_loss_fixtures(hip):
    """tests/test_data/l1_verify of the reference: bit-exact d_image, loss 1e-6 relative."""
    import json
    import os
    from helpers import GOLDEN
    base = os.path.join(GOLDEN, "l1_verify")
    for case in json.load(open(os.path.join(base, "manifest.json"))):
        _say("l1", case["name"])
        H, W = case["H"], case["W"]
        r = np.fromfile(os.path.join(base, case["name"] + "_rendered.bin"), np.float32).reshape(H, W, 3)
        g = np.fromfile(os.path.join(base, case["name"] + "_gt.bin"), np.float32).reshape(H, W, 3)
        d = np.fromfile(os.path.join(base, case["name"] + "_d_image.bin"), np.float32).reshape(H, W, 3)
        loss, d_img = hip.l1_loss(torch.tensor(r, device=hip.dev), torch.tensor(g, device=hip.dev))
        assert np.array_equal(_np(d_img), d)
        # loss.cpp:18-30: float difference, |.| accumulated in double
        exact = np.abs((r - g).astype(np.float64)).sum() / r.size
        assert abs(float(loss.item()) - exact) <= 1e-12 + 1e-9 * exact
        assert abs(float(loss.item()) - case["loss_serial"]) <= 1e-6


@pytest.mark.parametrize("n,deg,seed,bg", [(40, 1, 2, (0, 0, 0)), (500, 3, 4, (0.3, 0.1, 0.7)), (2000, 3, 5, (0, 0, 0))])
@pytest.mark.parametrize("batch", [64, 256])
def test_raster_bwd_matches_oracle(hip, oracle, n, deg, seed, bg, batch):
    _say("raster bwd", n, deg, seed, batch)
    scene, cam, gt = random_small_scene(n, deg, seed, width=100, height=75)
    cfg = RenderCfg(sh_degree=3, training=True, bg_color=bg)
    f = oracle.forward_backward(scene, cam, cfg, gt)
    pre = _to_dev(hip, {k: f["pre"][k] for k in ["means2D", "conics", "op2d", "rgb", "radii"]})
    vs = torch.tensor(f["values_sorted"].view(np.int32), device=hip.dev)
    rg = torch.tensor(f["ranges"].view(np.int32), device=hip.dev)
    px = dict(T_final=torch.tensor(f["T_final"], device=hip.dev),
              last_contrib=torch.tensor(f["last_contrib"].view(np.int32), device=hip.dev))
    d_img = torch.tensor(f["d_image"], device=hip.dev)
    hip.set_tuning(raster_bwd_batch=batch)
    g = hip.raster_bwd(pre, vs, rg, cam.width, cam.height, px, d_img, bg)
    hip.set_tuning(raster_bwd_batch=256)
    for k in ["d_means2D", "d_conics", "d_rgb", "d_op2d"]:
        assert_grad_close(_np(g[k]), f["rgrad"][k], k)


@pytest.mark.parametrize("n,deg,seed", [(40, 0, 2), (300, 1, 3), (300, 2, 6), (2000, 3, 5)])
def test_preprocess_bwd_matches_oracle(hip, oracle, n, deg, seed):
    _say("preprocess bwd", n, deg, seed)
    scene, cam, gt = random_small_scene(n, deg, seed, width=100, height=75)
    cfg = RenderCfg(sh_degree=3, training=True)
    f = oracle.forward_backward(scene, cam, cfg, gt)
    p = hip.upload_scene(scene)
    rg = _to_dev(hip, f["rgrad"])
    radii = torch.tensor(f["pre"]["radii"], device=hip.dev)
    out = hip.preprocess_bwd(p, cam, cfg, radii, rg)
    for k in ["pos", "scale", "rot", "sh", "op"]:
        assert_grad_close(_np(out[k]), f["grads"][k], "grad_" + k)


def test_adam_bitexact(hip, oracle):
    _say("adam")
    rng = np.random.default_rng(3)
    n, kc = 1001, 16
    shapes = dict(pos=(n, 3), scale=(n, 3), rot=(n, 4), sh=(n, kc, 3), op=(n,))
    p = {k: rng.standard_normal(s).astype(np.float32) for k, s in shapes.items()}
    m = {k: np.zeros(s, np.float32) for k, s in shapes.items()}
    v = {k: np.zeros(s, np.float32) for k, s in shapes.items()}
    d = hip.dev
    pt = {k: torch.tensor(a, device=d) for k, a in p.items()}
    mt = {k: torch.zeros(s, device=d) for k, s in shapes.items()}
    vt = {k: torch.zeros(s, device=d) for k, s in shapes.items()}
    pt["n"], pt["max_coeffs"] = n, kc
    lrs = [oracle.lr_schedule(1.6e-4, 1.6e-6, 0, 30000), 5e-3, 1e-3, 2.5e-3, 2.5e-2]
    for step in range(1, 4):
        g = {k: rng.standard_normal(s).astype(np.float32) for k, s in shapes.items()}
        g["sh"][::3] = 0.0
        gt_ = {k: torch.tensor(a, device=d) for k, a in g.items()}
        hip.adam(pt, gt_, mt, vt, lrs, 0.9, 0.999, 1e-8, step)
        bc1, bc2 = oracle.bias_corrections(0.9, 0.999, step)
        for i, k in enumerate(["pos", "scale", "rot", "sh", "op"]):
            oracle.adam_update(p[k], g[k], m[k], v[k], lrs[i], 0.9, 0.999, 1e-8, bc1, bc2)
    for k in shapes:
        assert np.array_equal(_np(pt[k]), p[k]), k
        assert np.array_equal(_np(mt[k]), m[k]), k
        assert np.array_equal(_np(vt[k]), v[k]), k


# verify_forward is a forward-render fixture: its target image is the rendered
# image itself (max |rendered - target| = 2.4e-7, 653 of 768 values equal), so
# sign(rendered - target) in the L1 gradient is decided by last-bit rounding
# and its gradients say nothing about the path.  Only its image is compared.
GRADIENT_UNDEFINED = {"verify_forward"}


@pytest.mark.parametrize("name", scene_dirs())
def test_golden_scenes_full_path(hip, name):
    """The whole GPU path against the reference's own golden vectors
    (train/verify_grads_ext/*, train/verify_forward)."""
    _say("golden", name)
    scene, cam, cfg, gt, exp = load_golden(name)
    p = hip.upload_scene(scene)
    f = hip.forward_backward(p, cam, cfg, torch.tensor(gt, device=hip.dev))
    assert_image_close(_np(f["img"]), exp["img"])
    if "loss" in exp:
        assert abs(float(f["loss"].item()) - exp["loss"]) <= 1e-6
    if name in GRADIENT_UNDEFINED:
        return
    for k in ["pos", "scale", "rot", "sh", "op"]:
        if "grad_" + k in exp:
            assert_grad_close(_np(f["grads"][k]), exp["grad_" + k], "grad_" + k)


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("n,deg,seed", [(500, 3, 21), (3000, 3, 22), (3000, 1, 23)])
def test_full_path_matches_oracle(hip, oracle, n, deg, seed, fast):
    _say("full path", n, deg, seed, fast)
    scene, cam, gt = random_small_scene(n, deg, seed, width=128, height=96)
    cfg = RenderCfg(sh_degree=3, training=True)
    ref = oracle.forward_backward(scene, cam, cfg, gt)
    p = hip.upload_scene(scene)
    run = hip.forward_backward_fast if fast else hip.forward_backward
    f = run(p, cam, cfg, torch.tensor(gt, device=hip.dev))
    assert_image_close(_np(f["img"]), ref["img"])
    assert abs(float(f["loss"].item()) - ref["loss"]) <= 1e-6
    for k in ["pos", "scale", "rot", "sh", "op"]:
        assert_grad_close(_np(f["grads"][k]), ref["grads"][k], "grad_" + k)


def test_c1_workload_full_path(hip, oracle):
    """10k Gaussians, 256x256, SH0: the reference's own CPU-runnable workload."""
    _say("c1 workload")
    scene, cams, gts = make_workload("10k_256")
    cam, gt = cams[0], gts[0]
    cfg = RenderCfg(sh_degree=3, training=True)
    ref = oracle.forward_backward(scene, cam, cfg, gt)
    p = hip.upload_scene(scene)
    f = hip.forward_backward_fast(p, cam, cfg, torch.tensor(gt, device=hip.dev))
    img_err = np.abs(_np(f["img"]) - ref["img"]).max()
    assert f["K"] == len(ref["keys"])
    assert img_err <= IMAGE_TOL, img_err
    assert abs(float(f["loss"].item()) - ref["loss"]) <= 1e-6
    for k in ["pos", "scale", "rot", "sh", "op"]:
        assert_grad_close(_np(f["grads"][k]), ref["grads"][k], "grad_" + k)


@pytest.mark.parametrize("seed", [1, 3, 4])
def test_needle_gradients_against_64_bits(hip, oracle, oracle64, seed):
    """Needles and sheets of hundreds of pixels: their conic gradients are sums
    of thousands of partly cancelling terms, and the step from the conic back to
    scale and rotation amplifies each rounding, in the reference's 32-bit
    arithmetic as well.  The HIP gradients are no further from the 64-bit
    oracle than the 32-bit oracle's own, up to the spread of such errors over
    orders of summation (four times for all but the worst Gaussian in a hundred,
    ten times in the 2-norm, which a single Gaussian decides)."""
    _say("needle gradients", seed)
    scene = gaussians_clusters(300, seed, 1, clusters=8, sigma=0.3, extent=2.0, logscale=(-2.5, 1.6), op=(-2.0, 2.0))
    cam = make_camera((0.0, 0.0, -6.0), 640, 360, 60.0)
    gt = target_image(cam.width, cam.height, seed)
    cfg = RenderCfg(sh_degree=1, training=True)
    want = oracle64.forward_backward(scene, cam, cfg, gt)["grads"]
    ref = oracle.forward_backward(scene, cam, cfg, gt)["grads"]
    for _ in range(3):  # float atomics: another order every time
        f = hip.forward_backward_fast(hip.upload_scene(scene), cam, cfg, torch.tensor(gt, device=hip.dev))
        for k in ["pos", "scale", "rot", "sh", "op"]:
            w = want[k].reshape(scene.n, -1)
            e_hip = np.linalg.norm(_np(f["grads"][k]).reshape(scene.n, -1) - w, axis=1)
            e_ref = np.linalg.norm(ref[k].reshape(scene.n, -1) - w, axis=1)
            assert np.quantile(e_hip, 0.99) <= 4 * np.quantile(e_ref, 0.99), k
            assert np.linalg.norm(e_hip) <= 10 * np.linalg.norm(e_ref), k
