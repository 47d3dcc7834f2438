"""Gradients of one long, thin splat at tilts where the sheared second moments
of the render backward differ most (along an axis, a degree beside it, between
the axes), against the same formulas in float64.

Tolerance: with k = the ratio of the 2-D covariance's eigenvalues and u =
2^-24, the exponent's terms are up to k times their sum, so it and the conic
are off by up to 9 u k |power|, on average over the weights twice that (|power|
averages 2); the covariance adds 8 u k and its inverse as much again at most:
34 u k in all, of the pixels' absolute contributions to a gradient."""
import math

import pytest
import torch

from diff_gaussian_rasterization import GaussianRasterizer
from gs_hip import camera as gcam
from gs_hip import scenes

pytestmark = pytest.mark.gpu


def _image64(v, cam, active):
    V, Pm = cam.world_view_transform.double(), cam.full_proj_transform.double()
    W, H = cam.image_width, cam.image_height
    p = v["means"][0]
    t = p @ V[:3, :3] + V[3, :3]
    h = torch.cat([p, p.new_ones(1)]) @ Pm
    ndc = h[:2] / (h[3] + 1e-7)
    x, y = ((ndc[0] + 1) * W - 1) / 2, ((ndc[1] + 1) * H - 1) / 2
    r, i, j, k = v["rotations"][0]
    R = torch.stack([1 - 2 * (j * j + k * k), 2 * (i * j - r * k), 2 * (i * k + r * j),
                     2 * (i * j + r * k), 1 - 2 * (i * i + k * k), 2 * (j * k - r * i),
                     2 * (i * k - r * j), 2 * (j * k + r * i), 1 - 2 * (i * i + j * j)]).reshape(3, 3)
    M = R * v["scales"][0]
    fx, fy = W / (2 * math.tan(cam.FoVx / 2)), H / (2 * math.tan(cam.FoVy / 2))
    z = t[2]
    J = torch.stack([torch.stack([fx / z, 0 * z, -fx * t[0] / z ** 2]),
                     torch.stack([0 * z, fy / z, -fy * t[1] / z ** 2])])
    T = J @ V[:3, :3].T
    cov = T @ M @ M.T @ T.T + 0.3 * torch.eye(2, dtype=torch.float64)
    A = torch.linalg.inv(cov)
    gy, gx = torch.meshgrid(torch.arange(H, dtype=torch.float64), torch.arange(W, dtype=torch.float64), indexing="ij")
    dx, dy = x - gx, y - gy
    power = -0.5 * (A[0, 0] * dx * dx + A[1, 1] * dy * dy) - A[0, 1] * dx * dy
    e = torch.linalg.eigvalsh(cov.detach())
    return torch.where(active, v["opacities"][0] * torch.exp(power), torch.zeros_like(power)) * v["colors"][0][:, None, None], float(e[1] / e[0])


@pytest.mark.parametrize("length", [0.05, 0.4])
@pytest.mark.parametrize("tilt", [0, 1, 30, 45, 89, 90, 135, 179])
def test_thin_splat(tilt, length):
    print("thin splat", tilt, length, flush=True)
    cam = scenes.plain_scene(seed=3, P=1, W=150, H=131)["cam"]
    V = cam.world_view_transform.double()
    # a point near the optical axis, three units in front; in-plane tilt about the view axis
    pc = torch.tensor([0.07, -0.05, 3.0], dtype=torch.float64)
    pw = (pc - V[3, :3]) @ torch.linalg.inv(V[:3, :3])
    a = math.radians(tilt)
    axis = torch.tensor([0.0, 0.0, 1.0], dtype=torch.float64) @ V[:3, :3].T
    q = torch.cat([torch.tensor([math.cos(a / 2)], dtype=torch.float64), math.sin(a / 2) * axis / axis.norm()])
    raw = dict(means=pw.reshape(1, 3), scales=torch.tensor([[length, 0.001, 0.0015]], dtype=torch.float64),
               rotations=q.reshape(1, 4), opacities=torch.tensor([[0.6]], dtype=torch.float64),
               colors=torch.tensor([[0.9, 0.4, 0.7]], dtype=torch.float64))
    raw = {k: t.float() for k, t in raw.items()}
    wgt = torch.rand((3, cam.image_height, cam.image_width), generator=torch.Generator().manual_seed(tilt))

    g = {k: t.cuda().requires_grad_(True) for k, t in raw.items()}
    rs = gcam.raster_settings(cam.to("cuda"), torch.zeros(3, device="cuda"), 0)
    color = GaussianRasterizer(raster_settings=rs)(
        means3D=g["means"], means2D=torch.zeros_like(g["means"]), opacities=g["opacities"],
        colors_precomp=g["colors"], scales=g["scales"], rotations=g["rotations"])[0]
    (color * wgt.cuda()).sum().backward()

    v = {k: t.double().requires_grad_(True) for k, t in raw.items()}
    active = color.detach()[0].cpu() != 0
    assert int(active.sum()) > 8
    image, k = _image64(v, cam, active)
    pixels = (image * wgt.double()).sum(0)[active]
    tol = 34 * 2.0 ** -24 * k
    each = [torch.autograd.grad(x, list(v.values()), retain_graph=True) for x in pixels]
    for n, name in enumerate(v):
        terms = torch.stack([e[n] for e in each])
        err = float((g[name].grad.cpu().double() - terms.sum(0)).norm())
        assert err <= tol * float(terms.abs().sum(0).norm()), (name, err, tol)
