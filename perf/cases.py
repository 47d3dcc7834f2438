"""Performance cases: the work a user of the framework has it do, through its
public entry points, and a plain float64 restatement of what comes out.

  step     one training step on the model layer: render, fused L1 + SSIM loss,
           backward with the Adam step of every parameter inside it
  grads    render, fused loss and backward, the gradients kept (a caller with
           an optimiser of its own, and the densification statistics)
  dropin   the drop-in rasteriser under autograd, forward and backward
  view     a forward render of a resident scene (viewer, evaluation, serving)
  solve    pose solves of new frames, replayed from a HIP graph
  knn      distCUDA2 over a cloud
  ingest   a depth map and its 8-bit image to local Gaussians, one per pixel
  loss     the fused loss and its gradient on two images

``listed`` holds the fixed cases, ``draw`` makes others of the same ranges.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "cf-3dgs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from diff_gaussian_rasterization import GaussianRasterizer  # noqa: E402
from gs_hip import camera as gcam  # noqa: E402
from gs_hip import ingest, pose, scenes, serve  # noqa: E402
from gs_hip.batch import BatchedPoseSolver  # noqa: E402
from gs_hip.loss import fused_photometric_loss  # noqa: E402
from gs_hip.model import GaussianParams, render  # noqa: E402
from simple_knn._C import distCUDA2  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"


def listed():
    return [
        # the headline training step: a full scene at the benchmark's size
        dict(name="step_500k_960x540", kind="step", P=500_000, W=960, H=540, deg=3),
        # a scene that is still growing, at the small frame size and an odd
        # width, with its gradients kept for an optimiser outside
        dict(name="grads_60k_479x270", kind="grads", P=60_000, W=479, H=270, deg=3),
        # the smallest training call: latency and launches
        dict(name="dropin_10k_256", kind="dropin", P=10_000, W=256, H=256, deg=3, depth=False, white=False,
             colors=False),
        # every output in the loss, a background, a ragged image, a count that fills no block
        dict(name="dropin_100003_613x347_depth", kind="dropin", P=100_003, W=613, H=347, deg=1, depth=True,
             white=True, colors=False),
        # evaluation of a large scene at full HD
        dict(name="view_1200k_1920x1080", kind="view", P=1_200_000, W=1920, H=1080, deg=3),
        # an interactive view of a small one
        dict(name="view_100k_480x270", kind="view", P=100_000, W=480, H=270, deg=3),
        # a batch of new frames of mixed sizes, ten iterations (one graph)
        dict(name="solve_16_mixed", kind="solve", n=16, lo=20_000, hi=200_000, iters=10),
        # one new frame on its own, a Gaussian per pixel
        dict(name="solve_1_480x270", kind="solve", n=1, lo=129_600, hi=129_600, iters=10),
        # initial scales of one frame's cloud, and of a whole scene's
        dict(name="knn_frame_129600", kind="knn", n=129_600, cloud="frame"),
        dict(name="knn_scene_2M", kind="knn", n=2_000_000, cloud="scene"),
        # a new frame at full size, a Gaussian per pixel, as the pose solves take it
        dict(name="ingest_960x540", kind="ingest", W=960, H=540, deg=0),
        # the loss on its own
        dict(name="loss_960x540", kind="loss", W=960, H=540),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "grads", "dropin", "dropin", "view", "solve", "knn", "ingest", "loss"])
    W = rng.randint(200, 960)
    H = max(120, int(W * rng.uniform(0.5, 0.75)))
    if kind in ("step", "grads"):
        return dict(kind=kind, P=_log(rng, 10_000, 500_000), W=W, H=H, deg=rng.choice([0, 1, 2, 3, 3]))
    if kind == "dropin":
        return dict(kind=kind, P=_log(rng, 2_000, 250_000), W=W, H=H, deg=rng.choice([0, 1, 2, 3]),
                    depth=rng.random() < 0.4, white=rng.random() < 0.4, colors=rng.random() < 0.25)
    if kind == "view":
        W = rng.randint(300, 1920)
        return dict(kind=kind, P=_log(rng, 50_000, 1_200_000), W=W, H=int(W * 9 / 16) + rng.randint(0, 9), deg=3)
    if kind == "solve":
        return dict(kind=kind, n=_log(rng, 1, 16), lo=20_000, hi=_log(rng, 40_000, 200_000), iters=10)
    if kind == "knn":
        cloud = rng.choice(["frame", "scene"])
        return dict(kind=kind, n=_log(rng, 5_000, 300_000 if cloud == "frame" else 2_000_000), cloud=cloud)
    if kind == "ingest":
        return dict(kind=kind, W=W, H=H, deg=rng.choice([0, 3]))
    return dict(kind=kind, W=W, H=H)


# ---- inputs -----------------------------------------------------------------

# frame sizes of the pose solves, as the benchmark's batch draws them
_FRAMES = [(320, 180), (480, 270), (640, 360), (960, 540)]


def _scene(c, seed):
    """Raw parameters, camera and target of a training or viewing case (CPU)."""
    if c["kind"] == "dropin":
        sc = scenes.plain_scene(seed=seed, P=c["P"], W=c["W"], H=c["H"], target_seed=seed + 1)
        g = torch.Generator().manual_seed(seed + 2)
        sc["bg"] = torch.ones(3) if c["white"] else torch.zeros(3)
        sc["colors"] = torch.rand((c["P"], 3), generator=g) if c["colors"] else None
        sc["depth_target"] = 3.0 + torch.rand((1, c["H"], c["W"]), generator=g)
        # Gaussians whose screen size keeps the overlap of the 10,000 at 256 x 256
        sc["scales"] = sc["scales"] * (10_000 / c["P"]) ** 0.5 if c["P"] > 10_000 else sc["scales"]
        return sc
    sc = scenes.training_scene(seed=seed, P=c["P"], W=c["W"], H=c["H"], target_seed=seed + 1)
    sc["sh_degree"] = c["deg"]
    if c["kind"] == "view":
        sc["cam"] = serve.sphere_camera(seed, c["W"], c["H"], device="cpu")
    return sc


def _cloud(c, seed):
    g = torch.Generator().manual_seed(seed)
    n = c["n"]
    if c["cloud"] == "frame":  # every pixel of a lifted frame, shuffled
        H = int(math.sqrt(n / 480 * 270)) + 1
        W = -(-n // H)
        return pose.lift_points(seed, W, H, n)[0]
    centres = torch.rand((32, 3), generator=g) * 6 - 3
    return centres[torch.randint(0, 32, (n,), generator=g)] + torch.randn((n, 3), generator=g) * 0.3


def _images(c, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.rand((3, c["H"], c["W"]), generator=g)
    return (a + 0.2 * torch.randn((3, c["H"], c["W"]), generator=g)), a


def prepare(case, seed):
    c, dev = case, DEV
    kind = c["kind"]
    if kind in ("step", "grads", "view"):
        sc = _scene(c, seed)
        gp = GaussianParams(sc["xyz"], sc["features_dc"], sc["features_rest"], sc["scaling"], sc["rotation"],
                            sc["opacity"], c["deg"], device=dev)
        s = dict(kind=kind, g=gp, cam=sc["cam"].to(dev), bg=sc["bg"].to(dev), target=sc["target"].to(dev))
        if kind == "step":
            # learning rates of late training (decayed a hundredfold), so that
            # a state stepped many times keeps its character
            gp.training_setup(position_lr_init=1.6e-6, feature_lr=2.5e-5, opacity_lr=5e-4, scaling_lr=5e-5,
                              rotation_lr=1e-5)
        return s
    if kind == "dropin":
        sc = _scene(c, seed)
        leaves = {k: sc[k].to(dev).requires_grad_(True) for k in ("means", "opacities", "scales", "rotations")}
        col = "colors" if c["colors"] else "shs"
        leaves[col] = sc[col].to(dev).requires_grad_(True)
        rs = gcam.raster_settings(sc["cam"].to(dev), sc["bg"].to(dev), c["deg"])
        return dict(kind=kind, leaves=leaves, target=sc["target"].to(dev), depth_target=sc["depth_target"].to(dev),
                    depth=c["depth"], rast=GaussianRasterizer(raster_settings=rs, return_alpha=c["depth"]))
    if kind == "solve":
        rng = np.random.default_rng(seed)
        insts = []
        for i in range(c["n"]):
            if c["lo"] == c["hi"]:
                W, H, P = 480, 270, c["lo"]
            else:
                W, H = _FRAMES[int(rng.integers(len(_FRAMES)))]
                P = min(int(rng.integers(c["lo"], c["hi"] + 1)), 4 * W * H)
            insts.append(pose.build_instance(seed * 100 + i, W, H, P, device=dev))
        few = c["n"] < 4
        solver = BatchedPoseSolver(insts, iters=c["iters"], streams=1 if few else 2, iters_per_graph=10,
                                   groups=1 if few else 2, shared_sort=True)
        return dict(kind=kind, solver=solver)
    if kind == "knn":
        return dict(kind=kind, points=_cloud(c, seed).to(dev))
    if kind == "ingest":
        d, rgb, K, _ = pose.frame_payload(seed, c["W"], c["H"])
        return dict(kind=kind, depth=d.to(dev), image=(rgb * 255).to(torch.uint8).to(dev), K=K, deg=c["deg"])
    if kind == "loss":
        x, y = _images(c, seed)
        return dict(kind=kind, x=x.to(dev).requires_grad_(True), y=y.to(dev))
    raise ValueError(kind)


# ---- one pass ---------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "step":
        g = s["g"]
        out = render(g, s["cam"], s["bg"], clamp=False, adam_in_backward=True)
        loss, _ = fused_photometric_loss(out["image"], s["target"], clamp01=True)
        loss.backward()
        g.optimizer.step()
        g.optimizer.zero_grad(set_to_none=True)
        return dict(loss=loss.detach(), image=out["image"].detach(), xyz=g._xyz.detach(),
                    features=g._features.detach(), scaling=g._scaling.detach(), rotation=g._rotation.detach(),
                    opacity=g._opacity.detach())
    if kind == "grads":
        g = s["g"]
        params = (g._xyz, g._features, g._scaling, g._rotation, g._opacity)
        for p in params:
            p.grad = None
        out = render(g, s["cam"], s["bg"], clamp=False)
        loss, _ = fused_photometric_loss(out["image"], s["target"], clamp01=True)
        loss.backward()
        return dict(loss=loss.detach(), image=out["image"].detach(), radii=out["radii"],
                    screen=out["viewspace_points"].grad, xyz=params[0].grad, features=params[1].grad,
                    scaling=params[2].grad, rotation=params[3].grad, opacity=params[4].grad)
    if kind == "dropin":
        v = s["leaves"]
        for p in v.values():
            p.grad = None
        screen = torch.zeros_like(v["means"], requires_grad=True)
        got = s["rast"](means3D=v["means"], means2D=screen, opacities=v["opacities"], shs=v.get("shs"),
                        colors_precomp=v.get("colors"), scales=v["scales"], rotations=v["rotations"])
        color, radii, depth = got[:3]
        loss = (color - s["target"]).abs().mean()
        if s["depth"]:
            loss = loss + 0.1 * (depth - s["depth_target"]).square().mean() + 0.01 * got[3].mean()
        loss.backward()
        out = dict(color=color.detach(), depth=depth.detach(), radii=radii, screen=screen.grad)
        out.update({"d_" + k: p.grad for k, p in v.items()})
        return out
    if kind == "view":
        with torch.no_grad():
            out = render(s["g"], s["cam"], s["bg"])
        return dict(image=out["image"], depth=out["depth"], radii=out["radii"])
    if kind == "solve":
        poses, losses = s["solver"].run()
        return dict(poses=poses, losses=losses)
    if kind == "knn":
        return distCUDA2(s["points"])
    if kind == "ingest":
        return ingest.ingest_frame(s["depth"], s["image"], s["K"], voxel_size=None, max_sh_degree=s["deg"],
                                   channels_first=False)
    s["x"].grad = None
    loss, _ = fused_photometric_loss(s["x"], s["y"], clamp01=True)
    loss.backward()
    return dict(loss=loss.detach(), grad=s["x"].grad)


# ---- the work a pass cannot do without --------------------------------------

# A pixel of these scenes blends 20 to 50 splats before it is opaque or its
# list ends; 40 operations for the weight and the blend of one, 80 more for
# its gradient terms.
_PAIRS = 40
_FWD, _BWD = 40, 80


def work(case):
    c = case
    kind = c["kind"]
    if kind == "solve":
        n, P = c["n"], 0.5 * (c["lo"] + c["hi"])
        px = 129_600 if c["lo"] == c["hi"] else 230_400  # mean of the frame sizes
        return dict(bytes=c["iters"] * n * (P * 56 + px * 24.0), flops=c["iters"] * n * px * _PAIRS * (_FWD + _BWD))
    if kind == "knn":
        return dict(bytes=16.0 * c["n"], flops=8.0 * 27 * c["n"])
    if kind == "ingest":
        px = c["W"] * c["H"]
        return dict(bytes=7.0 * px + 4.0 * px * (3 + 3 * (c["deg"] + 1) ** 2 + 3 + 4 + 1 + 7), flops=8.0 * 27 * px)
    px = c["W"] * c["H"]
    if kind == "loss":
        return dict(bytes=12.0 * 3 * px, flops=3.0 * px * (11 * 2 * 2 * 8))
    P = c["P"]
    stored = 4 * (3 + 48 + 3 + 4 + 1)
    read = 4 * (3 + 3 * (c["deg"] + 1) ** 2 + 3 + 4 + 1)
    fwd = dict(bytes=float(P * (read + 4) + 16 * px), flops=float(px * _PAIRS * _FWD + 300 * P))
    if kind == "view":
        return fwd
    extra = 5 * stored if kind == "step" else stored + 12  # Adam state and weights, or the gradients
    return dict(bytes=fwd["bytes"] + float(P * extra + 28 * px),
                flops=fwd["flops"] + float(px * _PAIRS * _BWD + 1000 * P))


# ---- float64 restatement ----------------------------------------------------

_C0 = 0.28209479177387814
_C1 = 0.4886025119029199
_C2 = (1.0925484305920792, -1.0925484305920792, 0.31539156525252005, -1.0925484305920792, 0.5462742152960396)
_C3 = (-0.5900435899266435, 2.890611442640554, -0.4570457994644658, 0.3731763325901154, -0.4570457994644658,
       1.445305721320277, -0.5900435899266435)


def _sh_color(deg, sh, d):
    x, y, z = d[:, 0:1], d[:, 1:2], d[:, 2:3]
    b = [torch.full_like(x, _C0)]
    if deg > 0:
        b += [-_C1 * y, _C1 * z, -_C1 * x]
    if deg > 1:
        b += [_C2[0] * x * y, _C2[1] * y * z, _C2[2] * (2 * z * z - x * x - y * y), _C2[3] * x * z,
              _C2[4] * (x * x - y * y)]
    if deg > 2:
        b += [_C3[0] * y * (3 * x * x - y * y), _C3[1] * x * y * z, _C3[2] * y * (4 * z * z - x * x - y * y),
              _C3[3] * z * (2 * z * z - 3 * x * x - 3 * y * y), _C3[4] * x * (4 * z * z - x * x - y * y),
              _C3[5] * z * (x * x - y * y), _C3[6] * x * (x * x - 3 * y * y)]
    return sum(bk * sh[:, k] for k, bk in enumerate(b)) + 0.5


def _screen64(v, cam, deg, ndc_shift):
    """Per-Gaussian screen quantities in float64: rows (x, y, conic a, b, c,
    opacity, r, g, b, depth), and the integer tile rects."""
    W, H = cam.image_width, cam.image_height
    V = cam.world_view_transform.double().to(DEV)
    Pm = cam.full_proj_transform.double().to(DEV)
    m = v["means"]
    hom = torch.cat([m, torch.ones_like(m[:, :1])], 1)
    t = hom @ V[:, :3]
    ph = hom @ Pm
    pw = 1.0 / (ph[:, 3] + 1e-7)
    ndc = ph[:, :2] * pw[:, None] + ndc_shift[:, :2]
    size = torch.tensor([W, H], dtype=torch.float64, device=DEV)
    xy = ((ndc + 1) * size - 1) * 0.5
    q, sc = v["rotations"], v["scales"]
    r, x, y, z = q.unbind(1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - r * z), 2 * (x * z + r * y),
                     2 * (x * y + r * z), 1 - 2 * (x * x + z * z), 2 * (y * z - r * x),
                     2 * (x * z - r * y), 2 * (y * z + r * x), 1 - 2 * (x * x + y * y)], 1).view(-1, 3, 3)
    L = R * sc[:, None, :]
    S = L @ L.transpose(1, 2).contiguous()
    fx, fy = W / (2 * cam.tanfovx), H / (2 * cam.tanfovy)
    lx, ly = 1.3 * cam.tanfovx, 1.3 * cam.tanfovy
    tz = t[:, 2]

    def clamped(u, lim):  # the clamp's own dependence on the depth carries no gradient
        q = u / tz
        return torch.where((q < -lim) | (q > lim), (q.clamp(-lim, lim) * tz).detach(), u)

    tx, ty = clamped(t[:, 0], lx), clamped(t[:, 1], ly)
    zero = torch.zeros_like(tz)
    J = torch.stack([fx / tz, zero, -fx * tx / tz ** 2, zero, fy / tz, -fy * ty / tz ** 2], 1).view(-1, 2, 3)
    T = J @ V[:3, :3].T.contiguous()
    C = T @ S @ T.transpose(1, 2).contiguous()
    ca, cb, cc = C[:, 0, 0] + 0.3, C[:, 0, 1], C[:, 1, 1] + 0.3
    det = (ca * cc - cb * cb).detach()
    k = det ** 2 / (det ** 2 + 1e-7)  # the rasteriser's guarded inverse of det^2 in the gradient
    ca, cb, cc = (u * k + (u - u * k).detach() for u in (ca, cb, cc))
    det = ca * cc - cb * cb
    con = torch.stack([cc / det, -cb / det, ca / det], 1)
    with torch.no_grad():
        mid = 0.5 * (ca + cc)
        rad = torch.ceil(3 * torch.sqrt(mid + torch.sqrt((mid * mid - det).clamp_min(0.1))))
        rad = torch.where(tz > 0.2, rad, torch.zeros_like(rad))
        g = torch.tensor([(W + 15) // 16, (H + 15) // 16], dtype=torch.float64, device=DEV)
        lo = torch.minimum(((xy - rad[:, None]) / 16).trunc().clamp_min(0), g).long()
        hi = torch.minimum(((xy + rad[:, None] + 15) / 16).trunc().clamp_min(0), g).long()
        n = (hi - lo).clamp_min(0).prod(1) * (tz > 0.2)
    if v.get("colors") is not None:
        rgb = v["colors"]
    else:
        d = m - cam.camera_center.double().to(DEV)
        rgb = _sh_color(deg, v["shs"], d / d.norm(dim=1, keepdim=True)).clamp_min(0)
    rows = torch.cat([xy, con, v["opacities"].view(-1, 1), rgb, tz[:, None]], 1)
    return rows, lo, hi, n


def _tile_lists(rows, lo, hi, n, gx, gy):
    """Gaussian ids of every tile in depth order: (ids, first position of each tile)."""
    order = torch.argsort(rows[:, 9], stable=True)
    order = order[n[order] > 0]
    cnt = n[order]
    ids = torch.repeat_interleave(order, cnt)
    first = torch.repeat_interleave(torch.cumsum(cnt, 0) - cnt, cnt)
    j = torch.arange(ids.numel(), device=DEV) - first
    w = (hi - lo)[ids, 0]
    tile = (lo[ids, 1] + j // w) * gx + lo[ids, 0] + j % w
    tile, o = torch.sort(tile, stable=True)
    return ids[o], torch.searchsorted(tile, torch.arange(gx * gy + 1, device=DEV)).tolist()


def _blend64(d, px, py, bg):
    dx, dy = d[:, 0:1] - px, d[:, 1:2] - py
    power = -0.5 * (d[:, 2:3] * dx * dx + d[:, 4:5] * dy * dy) - d[:, 3:4] * dx * dy
    og = d[:, 5:6] * torch.exp(power.clamp_max(0))
    alpha = og + (og.clamp_max(0.99) - og).detach()
    alpha = torch.where((power <= 0) & (alpha >= 1.0 / 255.0), alpha, torch.zeros_like(alpha))
    Ti = torch.cumprod(1 - alpha, 0)
    Te = torch.cat([torch.ones_like(Ti[:1]), Ti[:-1]])
    w = torch.where(Ti >= 1e-4, alpha * Te, torch.zeros_like(alpha))
    acc = w.sum(0)
    color = d[:, 6:9].T.contiguous() @ w + bg[:, None] * (1 - acc)
    return torch.cat([color, (d[:, 9:10] * w).sum(0, keepdim=True), acc[None]])


def _raster64(v, cam, deg, bg, loss_fn=None):
    """(color, depth, alpha) of float64 leaves, and, with a loss of the three
    images, its gradients by autograd: left in the leaves' .grad."""
    W, H = cam.image_width, cam.image_height
    gx, gy = (W + 15) // 16, (H + 15) // 16
    shift = torch.zeros_like(v["means"]).requires_grad_(loss_fn is not None)
    with torch.set_grad_enabled(loss_fn is not None):
        rows, lo, hi, n = _screen64(v, cam, deg, shift)
    data = rows.detach()
    bg = bg.double().to(DEV)
    ids, first = _tile_lists(data, lo, hi, n, gx, gy)
    img = torch.zeros((5, H, W), dtype=torch.float64, device=DEV)

    def tiles():
        for t in range(gx * gy):
            x0, y0 = t % gx * 16, t // gx * 16
            yield ids[first[t]:first[t + 1]], x0, y0, min(x0 + 16, W), min(y0 + 16, H)

    def pixels(x0, y0, x1, y1):
        py, px = torch.meshgrid(torch.arange(y0, y1, device=DEV, dtype=torch.float64),
                                torch.arange(x0, x1, device=DEV, dtype=torch.float64), indexing="ij")
        return px.reshape(1, -1), py.reshape(1, -1)

    for i, x0, y0, x1, y1 in tiles():
        px, py = pixels(x0, y0, x1, y1)
        out = _blend64(data[i], px, py, bg) if i.numel() else torch.cat([bg, bg.new_zeros(2)])[:, None].expand(
            5, px.numel())
        img[:, y0:y1, x0:x1] = out.reshape(5, y1 - y0, x1 - x0)
    if loss_fn is None:
        return img[:3], img[3:4], img[4:5], None, None
    leaf = img.clone().requires_grad_(True)
    loss = loss_fn(leaf[:3], leaf[3:4], leaf[4:5])
    loss.backward()
    grads = torch.zeros_like(data)
    for i, x0, y0, x1, y1 in tiles():
        if not i.numel():
            continue
        d = data[i].requires_grad_(True)
        out = _blend64(d, *pixels(x0, y0, x1, y1), bg)
        out.backward(leaf.grad[:, y0:y1, x0:x1].reshape(5, -1))
        grads.index_add_(0, i, d.grad)
    vis = n > 0
    rows[vis].backward(grads[vis])
    return img[:3], img[3:4], img[4:5], loss.detach(), shift.grad


def _loss64(x, y):
    x = x.clamp(0, 1)
    g = torch.tensor([math.exp(-(k - 5) ** 2 / 4.5) for k in range(11)], dtype=torch.float64, device=x.device)
    g = (g / g.sum()).float().double()
    w = (g[:, None] * g[None]).expand(3, 1, 11, 11).contiguous()

    def conv(a):
        return F.conv2d(a[None], w, padding=5, groups=3)[0]

    m1, m2 = conv(x), conv(y)
    s1, s2, s12 = conv(x * x) - m1 * m1, conv(y * y) - m2 * m2, conv(x * y) - m1 * m2
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    ssim = ((2 * m1 * m2 + c1) * (2 * s12 + c2)) / ((m1 * m1 + m2 * m2 + c1) * (s1 + s2 + c2))
    return 0.8 * (x - y).abs().mean() + 0.2 * (1 - ssim.mean())


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "loss":
        x, y = (t.double().to(DEV) for t in _images(c, seed))
        x.requires_grad_(True)
        loss = _loss64(x, y)
        loss.backward()
        return dict(loss=loss.detach(), grad=x.grad)
    if kind == "knn":
        if c["n"] > 150_000:
            return None  # a brute-force search would take minutes
        p = _cloud(c, seed).double().to(DEV)
        out = []
        for a in p.split(1024):
            d = sum((a[:, k:k + 1] - p[None, :, k]) ** 2 for k in range(3))
            out.append(torch.topk(d, 4, dim=1, largest=False).values[:, 1:].sum(1) / 3)
        return torch.cat(out)
    if kind in ("step", "solve", "ingest"):
        return None  # updates that follow from earlier ones; a search too large by brute force
    sc = _scene(c, seed)
    if kind == "view":
        v = dict(means=sc["xyz"], shs=torch.cat([sc["features_dc"], sc["features_rest"]], 1),
                 scales=torch.exp(sc["scaling"].double()), rotations=F.normalize(sc["rotation"].double()),
                 opacities=torch.sigmoid(sc["opacity"].double()))
        v = {k: t.double().to(DEV) for k, t in v.items()}
        color, depth, _, _, _ = _raster64(v, sc["cam"], c["deg"], sc["bg"])
        return dict(image=color.clamp(0, 1), depth=depth, radii=None)
    if kind == "grads":
        raw = {k: t.double().to(DEV).requires_grad_(True) for k, t in dict(
            xyz=sc["xyz"], features=torch.cat([sc["features_dc"], sc["features_rest"]], 1), scaling=sc["scaling"],
            rotation=sc["rotation"], opacity=sc["opacity"]).items()}
        v = dict(means=raw["xyz"], shs=raw["features"], scales=torch.exp(raw["scaling"]),
                 rotations=F.normalize(raw["rotation"]), opacities=torch.sigmoid(raw["opacity"]))
        y = sc["target"].double().to(DEV)
        color, _, _, loss, screen = _raster64(v, sc["cam"], c["deg"], sc["bg"], lambda i, d, a: _loss64(i, y))
        return dict(loss=loss, image=color, radii=None, screen=screen, **{k: t.grad for k, t in raw.items()})
    names = ("means", "opacities", "scales", "rotations", "colors" if c["colors"] else "shs")
    v = {k: sc[k].double().to(DEV).requires_grad_(True) for k in names}
    y, z = sc["target"].double().to(DEV), sc["depth_target"].double().to(DEV)

    def loss_fn(i, d, a):
        loss = (i - y).abs().mean()
        return loss + 0.1 * (d - z).square().mean() + 0.01 * a.mean() if c["depth"] else loss

    color, depth, _, _, screen = _raster64(v, sc["cam"], c["deg"], sc["bg"], loss_fn)
    return dict(color=color, depth=depth, radii=None, screen=screen, **{"d_" + k: t.grad for k, t in v.items()})
