"""A splat of an infinite colour among the list entries that the blend carries
from one 64-entry window to the next: the pixels it misses stay finite, bit for
bit the oracle's image, on 4 x 4-pixel blocks and on 8 x 8 ones."""
import math

import numpy as np
import pytest
import torch

from gpu_helpers import np_, run_gpu, run_oracle
from gs_hip import scenes
from gs_hip.camera import make_camera

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tall", [False, True], ids=["4x4", "8x8"])
@pytest.mark.parametrize("n", [65, 100, 150])
@pytest.mark.parametrize("rank", [60, 61, 62, 63])
def test_infinite_colour_carried(rank, n, tall):
    """Wide faint splats that reach every pixel of the tile, in depth order, but
    for one of the first window that reaches its far corner only: a block then
    keeps 63 entries of the window and carries 15 (4 x 4, groups of 16) or 3 (8 x
    8, groups of 4).  `rank` is the infinite one's place; it covers a few pixels."""
    print("carried", rank, n, "8x8" if tall else "4x4", flush=True)
    W, H = (32, 16 * 513) if tall else (32, 16)  # more than 1024 tiles, or 2
    focal = 27.0
    cam = make_camera(np.eye(3), np.zeros(3), 2 * math.atan(W / (2 * focal)), 2 * math.atan(H / (2 * focal)), W, H)
    y0 = H // 32 * 16 if tall else 0  # the tile row on the optical axis
    g = torch.Generator().manual_seed(rank)
    z = torch.linspace(3.0, 5.0, n)
    px = torch.rand((n, 2), generator=g) * 16
    size = torch.full((n,), 30.0)  # pixels
    opacity = 0.01 + 0.01 * torch.rand((n, 1), generator=g)
    for k, at, o in ((5, (14.6, 14.6), 0.02), (rank, (6.0, 6.0), 0.9)):
        px[k] = torch.tensor(at)
        size[k] = 0.01
        opacity[k] = o
    sc = scenes.plain_scene(seed=8, P=n, W=W, H=H)
    sc["cam"], sc["bg"], sc["opacities"] = cam, torch.tensor([0.2, 0.0, 0.7]), opacity
    sc["means"] = torch.stack([(px[:, 0] - (W - 1) / 2) * z / focal, (px[:, 1] + y0 - (H - 1) / 2) * z / focal, z], 1)
    sc["scales"] = (size * z / focal)[:, None].repeat(1, 3)
    sc["shs"][rank, 0, 1] = float("inf")
    g = run_gpu(sc, 0)
    _, _, o = run_oracle(sc, 0)
    assert 0 < int((~np.isfinite(o["color"][1])).sum()) < 64
    for k in ("color", "depth", "alpha"):
        np.testing.assert_array_equal(np_(g[k]), o[k], err_msg=k)
    np.testing.assert_array_equal(np_(g["views"]["n_contrib"]), o["n_contrib"])
