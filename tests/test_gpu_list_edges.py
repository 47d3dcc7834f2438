"""Tile lists whose lengths fall on the edges of the blend's and the render
backward's steps (16-entry groups, 256-entry chunks), on an image whose last
tiles are cut off: images bit for bit and every gradient against the fp32
oracle, with atomics and in the fixed-order mode.  Tolerances are those of
test_gpu_forward.py and test_gpu_backward.py."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_, run_gpu, run_oracle
from gs_hip import scenes
from test_gpu_backward import _check

pytestmark = pytest.mark.gpu


def _stack(n, small):
    """n faint Gaussians in front of a 21 x 18 image: wide ones that reach
    every cell of every tile, or small ones that reach a few cells each."""
    sc = scenes.plain_scene(seed=50 + n, P=n, W=21, H=18)
    g = torch.Generator().manual_seed(n)
    sc["means"] = torch.cat([(torch.rand((n, 2), generator=g) - 0.5) * 2.0, 2.0 + 2.0 * torch.rand((n, 1), generator=g)], 1)
    sc["scales"] = torch.full((n, 3), 0.1 if small else 1.5) * (0.5 + torch.rand((n, 3), generator=g))
    sc["opacities"] = 0.01 + 0.01 * torch.rand((n, 1), generator=g)
    sc["bg"] = torch.tensor([0.2, 0.0, 0.7])
    return sc


@pytest.mark.parametrize("small", [False, True], ids=["wide", "small"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 255, 256, 257, 512, 529])
def test_list_lengths(n, small):
    print("list length", n, "small" if small else "wide", flush=True)
    sc = _stack(n, small)
    g = run_gpu(sc, 1)
    _, _, o = run_oracle(sc, 1)
    if not small:
        assert o["num_rendered"] == 4 * n
    np.testing.assert_array_equal(np_(g["views"]["n_contrib"]), o["n_contrib"])
    np.testing.assert_array_equal(np_(g["views"]["final_T"]), o["final_T"])
    for k in ("color", "depth", "alpha"):
        np.testing.assert_array_equal(np_(g[k]), o[k], err_msg=k)
    _check(sc, 1, seed=n)
    _check(sc, 1, seed=n, deterministic=True)


@pytest.mark.parametrize("tall", [False, True], ids=["4x4", "8x8"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 64, 65, 127, 300])
def test_blend_blocks(n, tall):
    """Both of the blend's blocks (2 x 2 tiles, or 2 x 513 with the splats
    spread over the first of them) where lists end inside a group, pixels
    saturate and one colour is infinite: the pixels it misses stay finite."""
    print("blend blocks", n, "tall" if tall else "small", flush=True)
    sc = _stack(n, True)
    if tall:
        tall_sc = scenes.plain_scene(seed=50 + n, P=n, W=21, H=16 * 512 + 3)
        for k in ("means", "scales", "bg"):
            tall_sc[k] = sc[k]
        sc = tall_sc
    sc["opacities"] = torch.linspace(0.004, 1.0, n).reshape(n, 1)[torch.randperm(n, generator=torch.Generator().manual_seed(n))]
    sc["shs"][n // 2, 0, 1] = float("inf")
    g = run_gpu(sc, 1)
    _, _, o = run_oracle(sc, 1)
    np.testing.assert_array_equal(np_(g["views"]["n_contrib"]), o["n_contrib"])
    np.testing.assert_array_equal(np_(g["views"]["final_T"]), o["final_T"])
    for k in ("color", "depth", "alpha"):
        np.testing.assert_array_equal(np_(g[k]), o[k], err_msg=k)
    assert np.isfinite(o["color"][[0, 2]]).all()


@pytest.mark.parametrize("n", [8, 9, 255, 256, 257, 700])
def test_runs_split_by_entry(n):
    """Gaussians that cover all 510 tiles among ones that cover few: up to 4096
    entries per 256 Gaussians the lists are expanded by Gaussian, past that by
    entry.  The lists against the oracle's."""
    print("runs", n, flush=True)
    sc = scenes.plain_scene(seed=70 + n, P=n, W=479, H=270)
    m = max(n // 3, min(n, 9))  # 9 x 510 entries are past 4096
    sc["scales"][:m] = 3.0
    sc["means"][:m] = torch.tensor([0.0, 0.0, 3.0])
    sc["opacities"] = torch.full((n, 1), 0.02)
    g = run_gpu(sc, 1)
    _, _, o = run_oracle(sc, 1)
    assert g["st"].num_rendered == o["num_rendered"]
    for k in ("color", "depth", "alpha"):
        np.testing.assert_array_equal(np_(g[k]), o[k], err_msg=k)
    np.testing.assert_array_equal(np_(g["views"]["n_contrib"]), o["n_contrib"])


@pytest.mark.parametrize("big", [0, 40], ids=["even", "uneven"])
@pytest.mark.parametrize("n", [1024 * 256, 1024 * 256 + 1])
def test_block_prefix(n, big):
    """1024 blocks of 256 Gaussians, whose prefix the duplicate forms itself, and
    1025, which have a launch for it; by Gaussian, and by entry (40 Gaussians
    that cover all 130 tiles)."""
    print("block prefix", n, big, flush=True)
    sc = scenes.plain_scene(seed=9, P=n, W=200, H=150)
    sc["scales"] *= 0.05
    sc["scales"][:big] = 3.0
    sc["means"][:big] = torch.tensor([0.0, 0.0, 3.0])
    sc["opacities"] *= 0.05
    g = run_gpu(sc, 1)
    _, _, o = run_oracle(sc, 1)
    assert g["st"].num_rendered == o["num_rendered"]
    for k in ("color", "depth", "alpha"):
        np.testing.assert_array_equal(np_(g[k]), o[k], err_msg=k)
    np.testing.assert_array_equal(np_(g["views"]["n_contrib"]), o["n_contrib"])
