"""The radix sort at the limits where its plan changes: 128 workgroups of 1024
keys, up to which the scatter of a plain sort adds the counts up itself, and list
capacities of 2^21, up to which lists of 257 to 1024 tiles take one digit."""
import numpy as np
import pytest

from gpu_helpers import np_, run_gpu, run_oracle
from gs_hip import _lib, raster, scenes
from test_gpu_sort_u32 import test_sort_pairs_u32_stable as _pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("end_bit", [9, 32])
@pytest.mark.parametrize("n", [128 * 1024 - 1, 128 * 1024, 128 * 1024 + 1])
def test_pairs_at_the_direct_limit(n, end_bit):
    print("pairs", n, end_bit, flush=True)
    _pairs(n, end_bit, 1 << end_bit)


@pytest.mark.parametrize("over", [0, 1], ids=["2^21", "past 2^21"])
@pytest.mark.parametrize("P", [4200, 7700])
def test_lists_at_the_wide_limit(P, over):
    """272 tiles, every splat on all of them: 1.1M entries, and 2 094 400, whose
    one-digit sort has the most workgroups it can have (512)."""
    W, H, cap = 257, 256, (1 << 21) + over * raster._CAPACITY_QUANTUM
    print("lists", P, cap, flush=True)
    sc = scenes.plain_scene(seed=P, P=P, W=W, H=H)
    sc["scales"][:] = 3.0
    _, _, o = run_oracle(sc, 1)
    assert o["num_rendered"] == 272 * P
    mode = _lib.BINNING_DEPTH_FIRST
    raster._LAST_CAPACITY[(P, W, H, mode)] = cap
    g = run_gpu(sc, 1, binning=mode)
    assert g["st"].num_rendered == 272 * P and g["st"].capacity == cap
    assert _lib.binning_layout(cap, P, W, H, mode).sort_passes == 1 + over
    np.testing.assert_array_equal(np_(g["views"]["vals"]).astype(np.int64), o["vals"].astype(np.int64))
    for k in ("color", "depth", "alpha"):
        np.testing.assert_array_equal(np_(g[k]), o[k], err_msg=k)
    np.testing.assert_array_equal(np_(g["views"]["n_contrib"]), o["n_contrib"])
    np.testing.assert_array_equal(np_(g["views"]["ranges"]).reshape(-1, 2), o["ranges"].reshape(-1, 2))
