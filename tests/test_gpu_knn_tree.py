"""The k-nearest search's hierarchy at its edges: leaves, nodes and tops that
are partly filled, both curve lengths, coincident points, points far from the
rest and coordinates that are not finite.  Bit for bit against a search over
all points (the same operations in the same order, the three smallest summed
smallest first), for up to 1500 of the points."""
import pytest
import torch

from gpu_helpers import DEV
from gs_hip import raster

pytestmark = pytest.mark.gpu


def _points(n, kind):
    g = torch.Generator().manual_seed(n)
    p = torch.randn((n, 3), generator=g)
    if kind == "surface":
        p[:, 2] = torch.sin(3 * p[:, 0]) * 0.3
    elif kind == "clusters":
        p = p * 0.01 + torch.randint(0, 3, (n, 3), generator=g)
        p[:: 7] = p[0]  # coincident
    elif kind == "outlier":
        p[n // 2] = 1e4  # the rest falls into a few cells of the curve
        p[n // 3, 1] = float("nan")
        p[n // 4, 0] = float("inf")
    return p


@pytest.mark.parametrize("kind", ["surface", "clusters", "outlier"])
@pytest.mark.parametrize("n", [15, 16, 17, 63, 64, 65, 1023, 1025, 4097, 65_536, 65_600, 262_144, 262_145])
def test_knn_tree(n, kind):
    print("knn", n, kind, flush=True)
    p = _points(n, kind).to(DEV)
    got = raster.knn3_meandist(p)
    g = torch.Generator().manual_seed(1)
    rows = torch.randperm(n, generator=g)[:1500]
    rows = torch.cat([rows, torch.tensor([n // 2, n // 3, n // 4, 0, n - 1])]).unique().to(DEV)
    ref = torch.empty(len(rows), device=DEV)
    for a in range(0, len(rows), 256):
        r = rows[a:a + 256]
        dx, dy, dz = (p[r, k, None] - p[None, :, k] for k in range(3))
        d = (dx * dx + dy * dy) + dz * dz
        d[torch.arange(len(r), device=DEV), r] = float("inf")
        # as the oracle: a distance that is not below the largest float is none
        d = torch.where(d < torch.finfo(torch.float32).max, d, torch.finfo(torch.float32).max)
        b = torch.sort(torch.topk(d, 3, dim=1, largest=False).values, dim=1).values
        ref[a:a + 256] = ((b[:, 0] + b[:, 1]) + b[:, 2]) / torch.tensor(3.0, device=DEV)
    torch.cuda.synchronize()
    assert torch.equal(got[rows], ref)
