"""The radix sort's plans at their edges: counts added up by the scatter (up to
32 workgroups of 1024 keys), digits of unequal width, 4096 keys a workgroup past
2^24; and lists of 257 to 1024 tiles, which take one digit of 10 bits."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_, run_gpu, run_oracle
from gs_hip import scenes
from test_gpu_sort_u32 import test_sort_pairs_u32_stable as _pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,end_bit", [(1023, 32), (1025, 32), (32 * 1024, 32), (32 * 1024 + 1, 32), (32 * 1024 + 1, 9),
                                       (50_000, 17), ((1 << 24) + 4097, 13)])
def test_pair_plans(n, end_bit):
    print("pairs", n, end_bit, flush=True)
    _pairs(n, end_bit, 1 << end_bit)


@pytest.mark.parametrize("W,H", [(257, 16 * 16), (512, 512), (513, 512)], ids=["272", "1024", "1056"])
@pytest.mark.parametrize("n", [3, 40, 4000])
def test_list_plans(W, H, n):
    """Lists of 272 and 1024 tiles (one pass) and of 1056 (two): the tiles' ranges
    and lists against the oracle's."""
    print("lists", W, H, n, flush=True)
    sc = scenes.plain_scene(seed=n, P=n, W=W, H=H)
    sc["scales"][::7] *= 6.0
    g = run_gpu(sc, 1)
    _, _, o = run_oracle(sc, 1)
    assert g["st"].num_rendered == o["num_rendered"]
    np.testing.assert_array_equal(np_(g["views"]["n_contrib"]), o["n_contrib"])
    for k in ("color", "depth", "alpha"):
        np.testing.assert_array_equal(np_(g[k]), o[k], err_msg=k)
    r, e = np_(g["views"]["ranges"]).reshape(-1, 2), o["ranges"].reshape(-1, 2)
    np.testing.assert_array_equal(r[:, 1] - r[:, 0], e[:, 1] - e[:, 0])
    np.testing.assert_array_equal(r[e[:, 1] > e[:, 0]], e[e[:, 1] > e[:, 0]])
