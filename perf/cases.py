"""The work that users of this library have it do, as measurable cases.

A case is a dict of plain values.  ``kind`` names the entry point:

- ``step``:   ``GsTrainer.step``, the single-view training step (native driver);
- ``batch``:  ``GsBatch.step``, the multi-view training step replayed as a graph;
- ``render``: ``GsTrainer.render`` and the image it leaves (a viewer's frame);
- ``frame``:  ``GsHip.forward_fast``, a frame from parameters held as tensors;
- ``stages``: ``GsHip.forward``, the stage chain with the 64-bit pair sort;
- ``grads``:  ``GsHip.forward_backward_fast``, loss and gradients of one view;
- ``eval3d``: ``GsHip.render_3d``, the eval_3D forward.

Scenes follow the distributions of the benchmark workloads (``scene``: "cube",
"normal" or "clusters"), drawn on the GPU from the seed.  ``exact`` is the 2D
path again in plain torch and 64 bits.
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aaags-claude_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from gs_hip import GsBatch, GsHip, GsTrainer, train_cfg  # noqa: E402
from gs_scenes import MIXED_RES, RawScene, RenderCfg, make_camera  # noqa: E402

NAMES = ("pos", "scale", "rot", "sh", "op")
# a late-schedule learning rate: thousands of timed steps leave the scene as it was
LR, BETA1, BETA2, EPS = 1e-6, 0.9, 0.999, 1e-8


def _case(name, kind, n, width, height, degree=3, scene="cube", **more):
    return dict(name=name, kind=kind, n=n, width=width, height=height, degree=degree, scene=scene, **more)


def listed():
    return [
        # the smallest training step (10k Gaussians, 256 x 256, colour only): latency and launches count
        _case("step_10k_256", "step", 10_000, 256, 256, degree=0, fused=False, sync=True),
        # an ordinary training step, gradients written, then Adam; no read-back between steps
        _case("step_200k_720p", "step", 200_000, 1280, 720, scene="normal", fused=False, sync=False),
        # the headline training step: Adam inside the backward
        _case("step_1m_1080p", "step", 1_000_000, 1920, 1080, fused=True, sync=False),
        # a few small ragged views trained together
        _case("batch_50k_4views", "batch", 50_000, 0, 0, degree=2, views=4),
        # the mixed-resolution batch: 16 views over one scene
        _case("batch_1m_16views", "batch", 1_000_000, 0, 0, views=16),
        # the largest batch: 6M Gaussians in clusters, eight 1080p views
        _case("batch_6m_8x1080p", "batch", 6_000_000, 1920, 1080, scene="clusters", views=8),
        # an interactive viewer: one frame at the headline size, its image fetched
        _case("render_1m_1080p", "render", 1_000_000, 1920, 1080),
        # a thumbnail of odd size from a small model
        _case("frame_50k_411x307", "frame", 50_000, 411, 307, degree=1),
        # a 4K frame
        _case("frame_1m_4k", "frame", 1_000_000, 3840, 2160),
        # the reference-compatible stage chain: scan, keys, pair sort, raster
        _case("stages_200k_720p", "stages", 200_000, 1280, 720, scene="normal"),
        # gradients of an antialiased view of odd size (a user's own optimizer)
        _case("grads_300k_1111x777_aa", "grads", 300_000, 1111, 777, degree=2, antialiasing=True),
        # the eval_3D forward
        _case("eval3d_1m_1080p", "eval3d", 1_000_000, 1920, 1080),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, hi=1920):
    w = _log(rng, 160, hi)
    return w, max(90, int(w * rng.uniform(0.5, 0.8)))


def draw(rng: random.Random):
    kind = rng.choice(("step", "step", "batch", "render", "frame", "stages", "grads", "eval3d"))
    n = _log(rng, 10_000, 1_000_000)
    w, h = _size(rng, 3840 if kind in ("render", "frame") else 1920)
    more = {}
    if kind == "step":
        more = dict(fused=rng.random() < 0.5, sync=rng.random() < 0.5)
    elif kind == "batch":
        more = dict(views=rng.randint(2, 12))
        w, h = (0, 0) if rng.random() < 0.5 else (w, h)
    elif kind == "grads":
        more = dict(antialiasing=rng.random() < 0.5)
    elif kind == "eval3d":
        n = _log(rng, 100_000, 1_000_000)
    case = _case("", kind, n, w, h, rng.choice((0, 1, 2, 3, 3)), rng.choice(("cube", "normal")), **more)
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs --
def _device():
    return torch.device("cuda", 0)


def _scene(case, seed):
    """Raw parameters on the GPU, in upload_scene's layout."""
    d = _device()
    g = torch.Generator(device=d).manual_seed(int(seed))
    n, deg = case["n"], case["degree"]

    def normal(shape, mean, sigma):
        return torch.randn(shape, generator=g, device=d) * sigma + mean

    if case["scene"] == "cube":
        pos = torch.rand((n, 3), generator=g, device=d) * 2.0 - 1.0
        ls, op = (-4.0, 0.5), (0.0, 1.0)
    elif case["scene"] == "normal":
        pos = normal((n, 3), 0.0, 1.5)
        ls, op = (-4.5, 0.7), (-1.0, 1.5)
    else:
        centres = torch.rand((32, 3), generator=g, device=d) * 6.0 - 3.0
        which = torch.randint(0, 32, (n,), generator=g, device=d)
        pos = centres[which] + normal((n, 3), 0.0, 0.3)
        ls, op = (-5.0, 0.8), (-2.0, 2.0)
    rot = normal((n, 4), 0.0, 1.0)
    rot = rot / rot.norm(dim=1, keepdim=True)
    k = (deg + 1) ** 2
    sh = normal((n, k, 3), 0.0, 0.05)
    sh[:, 0] *= 10.0
    return dict(pos=pos, scale=normal((n, 3), *ls), rot=rot, sh=sh, op=normal((n,), *op), sh_degree=deg, max_coeffs=k,
                n=n)


def _cameras(case, seed):
    """The case's pinhole cameras: looking at the scene from its own distance, directions from the seed."""
    r = random.Random(int(seed) + 1000)
    dist = {"cube": 3.0, "normal": 4.0, "clusters": 8.0}[case["scene"]]
    cams = []
    for v in range(case.get("views", 1)):
        z, phi = r.uniform(-0.6, 0.6), r.uniform(0.0, 2.0 * math.pi)
        c = math.sqrt(1.0 - z * z)
        eye = (dist * c * math.cos(phi), dist * z, dist * c * math.sin(phi))
        if case["width"]:
            w, h = case["width"], case["height"]
        else:
            w, h = MIXED_RES[v % len(MIXED_RES)]
            if case["n"] < 200_000:  # small models are trained on small ragged images
                w, h = w // 4 + 3 * v + 1, h // 4 + v
        cams.append(make_camera(eye, w, h, 60.0 if case["scene"] != "normal" else 50.0))
    return cams


def _cfg(case):
    return RenderCfg(sh_degree=case["degree"], antialiasing=bool(case.get("antialiasing", False)),
                     training=case["kind"] in ("step", "batch", "grads"))


def _target(cam, seed, v=0):
    g = torch.Generator(device=_device()).manual_seed(int(seed) + 2000 + v)
    return torch.rand((cam.height, cam.width, 3), generator=g, device=_device())


class _Array:
    """A device array that the trainer owns, for torch to look at in place."""

    def __init__(self, address, shape):
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(address, False), version=3)


def _buffers(tr, prefix):
    out = {}
    for k, shape in dict(pos=(tr.n, 3), scale=(tr.n, 3), rot=(tr.n, 4), sh=(tr.n, tr.k, 3), op=(tr.n,)).items():
        address = tr.lib.gs_trainer_buffer(tr.tr, f"{prefix}_{k}".encode())
        t = out[f"{prefix}_{k}"] = torch.as_tensor(_Array(address, shape), device=_device())
        t.owner = tr  # the trainer frees its arrays when it goes: it stays while they are looked at
    return out


def prepare(case, seed):
    p = _scene(case, seed)
    cams, cfg = _cameras(case, seed), _cfg(case)
    hip = GsHip(0)
    s = dict(kind=case["kind"], hip=hip, cam=cams[0], cfg=cfg)
    if case["kind"] in ("step", "batch", "render"):
        scene = RawScene(*(p[k].cpu().numpy() for k in NAMES), sh_degree=p["sh_degree"])
        tr = s["tr"] = GsTrainer(hip, scene)
        s["tc"] = train_cfg(lr=LR, beta1=BETA1, beta2=BETA2, eps=EPS)
        s["it"] = 0
        if case["kind"] == "step":
            tr.set_options(fused_adam=case["fused"])
            s["sync"] = case["sync"]
            s["gt"] = _target(cams[0], seed)
            s["out"] = {**_buffers(tr, "param"), **_buffers(tr, "adam_m"), **_buffers(tr, "adam_v")}
            if not case["fused"]:
                s["out"].update(_buffers(tr, "grad"))
        elif case["kind"] == "batch":
            gts = [_target(c, seed, v).cpu().numpy() for v, c in enumerate(cams)]
            s["batch"] = GsBatch(tr, cams, cfg, gts)
            s["out"] = {**_buffers(tr, "param"), **_buffers(tr, "adam_m"), **_buffers(tr, "adam_v")}
    else:
        s["p"] = p
        if case["kind"] == "grads":
            s["gt"] = _target(cams[0], seed)
    return s


def run(s):
    kind, cam, cfg = s["kind"], s["cam"], s["cfg"]
    if kind == "step":
        res = s["tr"].step(cam, cfg, s["gt"], s["tc"], s["it"], sync=s["sync"])
        s["it"] += 1
        return dict(s["out"], loss=res.loss) if s["sync"] else s["out"]
    if kind == "batch":
        s["batch"].step(s["tc"], s["it"])
        s["it"] += 1
        return s["out"]
    if kind == "render":
        pairs = s["tr"].render(cam, cfg)
        return dict(img=s["tr"].buffer("image", (cam.height, cam.width, 3)), pairs=pairs)
    if kind == "frame":
        f = s["hip"].forward_fast(s["p"], cam, cfg)
        return dict(img=f["img"], T=f["px"]["T_final"], contributors=f["px"]["n_contrib"], ranges=f["ranges"])
    if kind == "stages":
        f = s["hip"].forward(s["p"], cam, cfg)
        return dict(img=f["img"], T=f["px"]["T_final"], contributors=f["px"]["n_contrib"], ranges=f["ranges"])
    if kind == "grads":
        f = s["hip"].forward_backward_fast(s["p"], cam, cfg, s["gt"])
        return dict(f["grads"], img=f["img"], loss=f["loss"])
    f = s["hip"].render_3d(s["p"], cam, cfg, fast=True)
    return dict(img=f["img"], T=f["T_final"], contributors=f["n_contrib"], ranges=f["ranges"])


def work(case):
    """Bytes: inputs read once, outputs written once (236 B of raw parameters a
    Gaussian at SH degree 3).  Operations: about 64 contributors a pixel, as
    the headline view has, at 28 FP32 operations forward and 72 backward."""
    n, k = case["n"], (case["degree"] + 1) ** 2
    param = 4 * (11 + 3 * k) * n
    pixels = sum(c.width * c.height for c in _cameras(case, 0))
    forward, backward = 64 * 28 * pixels, 64 * 72 * pixels
    if case["kind"] in ("step", "batch"):  # parameters, m and v read and written; the target read
        return dict(bytes=6 * param + 12 * pixels, flops=forward + backward)
    if case["kind"] == "grads":
        return dict(bytes=2 * param + 24 * pixels, flops=forward + backward)
    return dict(bytes=param + 16 * pixels, flops=forward)


def tolerance(case):
    # Images: float sums over the contributors; an alpha's last bit can move a
    # pixel's stop by one contributor (64-bit images are 1e-5 off).
    # Gradients: the same, summed over the pixels by atomics in an order that
    # changes from run to run (7e-5), and a pixel whose L1 difference is a
    # rounding error of 0 can change its sign (64-bit gradients are 6e-4 off).
    # The clusters hold a few Gaussians of hundreds of pixels, whose thousands
    # of partly cancelling terms leave 1.5e-2 between two runs.
    if case["scene"] == "clusters":
        return dict(rel=0.03, max=0.99, differ=1e-4)
    if case["kind"] in ("step", "batch", "grads"):
        return dict(rel=2e-3, max=0.2, differ=1e-4)
    return dict(rel=5e-5, max=5e-3, differ=1e-4)


# ------------------------------------------------- the 2D path in 64 bits --
C0, C1 = 0.28209479177387814, 0.4886025119029199
C2 = (1.0925484305920792, -1.0925484305920792, 0.31539156525252005, -1.0925484305920792, 0.5462742152960396)
C3 = (-0.5900435899266435, 2.890611442640554, -0.4570457994644658, 0.3731763325901154, -0.4570457994644658,
      1.445305721320277, -0.5900435899266435)


def _basis(d, degree):
    x, y, z = d.unbind(1)
    b = [torch.full_like(x, C0)]
    if degree > 0:
        b += [-C1 * y, C1 * z, -C1 * x]
    if degree > 1:
        b += [C2[0] * x * y, C2[1] * y * z, C2[2] * (2 * z * z - x * x - y * y), C2[3] * x * z,
              C2[4] * (x * x - y * y)]
    if degree > 2:
        b += [C3[0] * y * (3 * x * x - y * y), C3[1] * x * y * z, C3[2] * y * (4 * z * z - x * x - y * y),
              C3[3] * z * (2 * z * z - 3 * x * x - 3 * y * y), C3[4] * x * (4 * z * z - x * x - y * y),
              C3[5] * z * (x * x - y * y), C3[6] * x * (x * x - 3 * y * y)]
    return torch.stack(b, 1)


def _project(q, cam, cfg):
    """Screen-space mean, conic, opacity and colour of every Gaussian, its depth and the tile rectangle."""
    d = q["pos"].device
    view = torch.tensor(cam.view.astype("float64"), device=d).view(4, 4)  # column-major: rows here are columns
    vp = torch.tensor(cam.viewproj.astype("float64"), device=d).view(4, 4)
    pos = q["pos"]
    hom = torch.cat([pos, torch.ones_like(pos[:, :1])], 1)
    pv, ph = hom @ view, hom @ vp
    w, h = cam.width, cam.height
    ndc = ph[:, :2] / (ph[:, 3:] + 1e-7)
    mean = torch.stack([((ndc[:, 0] + 1) * w - 1) * 0.5, ((ndc[:, 1] + 1) * h - 1) * 0.5], 1)
    r, x, y, z = (q["rot"] / q["rot"].norm(dim=1, keepdim=True)).unbind(1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y + r * z), 2 * (x * z - r * y),
                     2 * (x * y - r * z), 1 - 2 * (x * x + z * z), 2 * (y * z + r * x),
                     2 * (x * z + r * y), 2 * (y * z - r * x), 1 - 2 * (x * x + y * y)], 1).view(-1, 3, 3)
    M = q["scale"].exp()[:, :, None] * R
    tx, ty, tz = pv[:, 0], pv[:, 1], pv[:, 2]
    limx, limy = 1.3 * cam.tan_fovx, 1.3 * cam.tan_fovy
    # outside 1.3 times the frustum the projection is linearised at its edge; the backward holds that point
    tx = torch.where((tx / tz).abs() < limx, tx, (torch.sign(tx) * limx * tz).detach())
    ty = torch.where((ty / tz).abs() < limy, ty, (torch.sign(ty) * limy * tz).detach())
    fx, fy = w / (2.0 * cam.tan_fovx), h / (2.0 * cam.tan_fovy)
    W = view[:3, :3].T  # world to camera
    J0 = (fx / tz)[:, None] * W[0] - (fx * tx / (tz * tz))[:, None] * W[2]
    J1 = (fy / tz)[:, None] * W[1] - (fy * ty / (tz * tz))[:, None] * W[2]
    u0, u1 = (M * J0[:, None, :]).sum(2), (M * J1[:, None, :]).sum(2)
    a0, b, c0 = (u0 * u0).sum(1), (u0 * u1).sum(1), (u1 * u1).sum(1)
    a, c = a0 + 0.3, c0 + 0.3
    det = a * c - b * b
    op = torch.sigmoid(q["op"])
    if cfg.antialiasing:
        op = op * torch.sqrt(torch.clamp((a0 * c0 - b * b) / det, min=0.000025))
    conic = torch.stack([c / det, -b / det, a / det], 1)
    direction = pos - torch.tensor(cam.cam_pos.astype("float64"), device=d)
    direction = direction / direction.norm(dim=1, keepdim=True)
    raw = (_basis(direction, cfg.sh_degree)[:, :, None] * q["sh"]).sum(1) + 0.5
    rgb = torch.clamp(raw, min=0.0) if cfg.training else torch.clamp(raw, 0.0, 1.0)
    with torch.no_grad():
        mid = 0.5 * (a + c)
        rad = torch.ceil(3.0 * torch.sqrt(mid + torch.sqrt(torch.clamp(mid * mid - det, min=0.1))))
        gx, gy = (w + 15) // 16, (h + 15) // 16
        lo = torch.stack([((mean[:, i] - rad) / 16).trunc().clamp(0, g) for i, g in enumerate((gx, gy))], 1)
        hi = torch.stack([((mean[:, i] + rad + 15) / 16).trunc().clamp(0, g) for i, g in enumerate((gx, gy))], 1)
        seen = (pv[:, 2] > 0.2) & (rad <= max(w, h)) & (hi > lo).all(1)
        rect = torch.cat([lo, hi], 1).nan_to_num().long() * seen[:, None]
    return dict(mean=mean, conic=conic, op=op, rgb=rgb, depth=pv[:, 2].detach(), rect=rect)


def _lists(s, cam):
    """Every tile's Gaussians in depth order: (indices, first, count)."""
    order = torch.sort(s["depth"].float(), stable=True).indices
    x0, y0, x1, y1 = s["rect"][order].unbind(1)
    nx = x1 - x0
    count = nx * (y1 - y0)
    at = torch.repeat_interleave(torch.arange(len(order), device=order.device), count)
    k = torch.arange(len(at), device=order.device) - (torch.cumsum(count, 0) - count)[at]
    gx, gy = (cam.width + 15) // 16, (cam.height + 15) // 16
    tile = ((y0[at] + k // nx[at]) * gx + x0[at] + k % nx[at]).int()
    del k
    tile, by = torch.sort(tile, stable=True)
    per = torch.bincount(tile, minlength=gx * gy)
    return order[at[by]], torch.cumsum(per, 0) - per, per


def _blend(s, lists, cam, final=None, d_image=None):
    """The tiles' blending, 32 list entries of every open tile at a time.  With
    (final, d_image): the gradients of the screen-space values too."""
    ids, first, per = lists
    d = ids.device
    gx, tiles = (cam.width + 15) // 16, len(first)
    lane = torch.arange(256, device=d)
    t = torch.arange(tiles, device=d)
    px = ((t % gx) * 16)[:, None] + (lane % 16)[None]
    py = ((t // gx) * 16)[:, None] + (lane // 16)[None]
    inside = (px < cam.width) & (py < cam.height)
    pix = (py * cam.width + px).clamp(max=cam.width * cam.height - 1)
    T = inside.double()
    stop = ~inside
    colour = torch.zeros((tiles, 256, 3), dtype=torch.float64, device=d)
    if d_image is not None:
        dC = d_image.view(-1, 3)[pix] * inside[..., None]
        total = (final.view(-1, 3)[pix] * dC).sum(2)
        out = {k: torch.zeros_like(s[k]) for k in ("mean", "conic", "op", "rgb")}
    base = 0
    step = max(4, min(32, (1 << 28) // (tiles * 256 * 8) * 4))
    while True:
        live = torch.nonzero((per > base) & ~stop.all(1)).flatten()
        if len(live) == 0:
            break
        j = base + torch.arange(step, device=d)
        ok = j[None] < per[live, None]
        g = ids[torch.where(ok, first[live, None] + j[None], 0)]
        m, co, o, rgb = s["mean"][g], s["conic"][g], s["op"][g] * ok, s["rgb"][g]
        dx = m[..., 0, None] - px[live, None].double()
        dy = m[..., 1, None] - py[live, None].double()
        power = -0.5 * (co[..., 0, None] * dx * dx + co[..., 2, None] * dy * dy) - co[..., 1, None] * dx * dy
        G = power.exp()
        alpha = (o[..., None] * G).clamp(max=0.99)
        use = (power <= 0) & (alpha >= 1.0 / 255.0) & ~stop[live, None]
        after = T[live, None] * torch.cumprod(torch.where(use, 1 - alpha, 1.0), 1)
        take = use & (after >= 1e-4)
        before = torch.cat([T[live, None], after[:, :-1]], 1)
        weight = torch.where(take, alpha * before, 0.0)
        if d_image is not None:
            dc = dC[live]
            cd = rgb @ dc.transpose(1, 2)  # [tile, entry, pixel]
            sofar = (colour[live] * dc).sum(2)[:, None] + torch.cumsum(weight * cd, 1)
            dal = torch.where(take, before * cd - (total[live, None] - sofar) / (1 - alpha), 0.0)
            dop = torch.where(alpha < 0.99, dal * G, 0.0)
            dp = dop * o[..., None]
            flat = g.flatten()
            add = lambda k, v: out[k].index_add_(0, flat, v.reshape(len(flat), -1).view(len(flat), *out[k].shape[1:]))  # noqa: E731
            sx, sy = (dp * dx).sum(2), (dp * dy).sum(2)
            add("mean", torch.stack([-co[..., 0] * sx - co[..., 1] * sy, -co[..., 2] * sy - co[..., 1] * sx], 2))
            add("conic", torch.stack([-0.5 * (dp * dx * dx).sum(2), -(dp * dx * dy).sum(2),
                                      -0.5 * (dp * dy * dy).sum(2)], 2))
            add("op", dop.sum(2))
            add("rgb", weight @ dc)
        colour[live] += weight.transpose(1, 2) @ rgb
        T[live] = torch.where(take, after, torch.inf).amin(1).minimum(T[live])
        stop[live] |= (use & ~take).any(1)
        base += step
    if d_image is not None:
        return out
    image = torch.zeros((cam.width * cam.height, 3), dtype=torch.float64, device=d)
    image[pix[inside]] = colour[inside]  # the background is black
    rest = torch.zeros(cam.width * cam.height, dtype=torch.float64, device=d)
    rest[pix[inside]] = T[inside]
    return image.view(cam.height, cam.width, 3), rest.view(cam.height, cam.width)


def _gradients(q, cam, cfg, gt):
    leaves = {k: q[k].clone().requires_grad_(True) for k in NAMES}
    s = _project(leaves, cam, cfg)
    flat = {k: v.detach() for k, v in s.items()}
    lists = _lists(flat, cam)
    img, _ = _blend(flat, lists, cam)
    diff = img - gt.double()
    back = _blend(flat, lists, cam, img, torch.sign(diff) / diff.numel())
    seen = (flat["rect"][:, 2] > flat["rect"][:, 0])
    keys = ("mean", "conic", "op", "rgb")
    upstream = [torch.where(seen.view(-1, *[1] * (back[k].dim() - 1)), back[k], 0.0) for k in keys]
    grads = torch.autograd.grad([s[k] for k in keys], [leaves[k] for k in NAMES], upstream, allow_unused=True)
    got = {k: torch.zeros_like(q[k]) if v is None else v.nan_to_num() for k, v in zip(NAMES, grads)}
    return got, img, diff.abs().mean()


def exact(case, seed):
    views = case.get("views", 1)
    # the k-buffer of eval_3D is a sequence over every tile's whole list; large batches take minutes
    if case["kind"] == "eval3d" or case["n"] * views > 1_500_000:
        return None
    p = _scene(case, seed)
    q = {k: p[k].double() for k in NAMES}
    cams, cfg = _cameras(case, seed), _cfg(case)
    if case["kind"] in ("step", "batch", "grads"):
        grads, loss, img = {k: torch.zeros_like(q[k]) for k in NAMES}, None, None
        for v, cam in enumerate(cams):
            g, img, loss = _gradients(q, cam, cfg, _target(cam, seed, v))
            for k in NAMES:
                grads[k] += g[k]
        if case["kind"] == "grads":
            return dict(grads, img=img, loss=loss.view(1))
        out = {}
        for k in NAMES:
            g = grads[k]
            out[f"adam_m_{k}"], out[f"adam_v_{k}"] = (1 - BETA1) * g, (1 - BETA2) * g * g
            out[f"param_{k}"] = q[k] - LR * g / (g.abs() + EPS)
            if case["kind"] == "step" and not case["fused"]:
                out[f"grad_{k}"] = g
        if case["kind"] == "step" and case["sync"]:
            out["loss"] = float(loss)
        return out
    cam = cams[0]
    s = _project(q, cam, cfg)
    img, T = _blend(s, _lists(s, cam), cam)
    if case["kind"] == "render":
        return dict(img=img, pairs=None)
    return dict(img=img, T=T, contributors=None, ranges=None)
