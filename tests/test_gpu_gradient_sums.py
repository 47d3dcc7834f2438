"""The render backward's sums, where another grouping or a value that is not
finite shows.

* Scenes whose rotation gradients are decided by the rounding of one thin,
  tilted splat's second moments: in the fixed-order mode that splat's gradients
  are the recorded ones of the reference formula summed pixel by pixel (the
  same operations in the same order, so to the bit; 1e-6 of the row's norm is
  allowed for another compiler's contractions).  Sums by 4 x 4-pixel cells differ
  from them by 5e-5 to 2e-4.
* A splat that no pixel blends has no influence on any gradient, whatever its
  colour."""
import random

import pytest
import torch

from gpu_helpers import DEV, np_
from gs_hip import camera as gcam
from gs_hip import raster, scenes

pytestmark = pytest.mark.gpu

# scene number: its thinnest splat's index, d loss / d rotation, d loss / d scale
_ROWS = {
    32: (1287, ("0x1.37f9ccp+2", "-0x1.fc5588p+2", "-0x1.e96ea6p+4", "0x1.e3ce08p+3"),
         ("-0x1.aa817cp+5", "-0x1.85aba4p+0", "-0x1.46e7d0p+2")),
    236: (1738, ("0x1.1f3038p+2", "-0x1.ae43b2p+4", "-0x1.4510d4p+2", "-0x1.cd870ap+4"),
          ("-0x1.52f3c8p+1", "-0x1.31c406p+2", "-0x1.025172p+5")),
    51: (909, ("-0x1.93ffdep+1", "-0x1.376c84p+1", "0x1.1ef078p-1", "0x1.d0efa4p-3"),
         ("-0x1.07fb84p+5", "-0x1.5db1e2p-2", "0x1.5164f8p+2")),
    249: (679, ("-0x1.a4f11cp-3", "-0x1.af5b26p+3", "0x1.4f411cp+0", "-0x1.b4eeb8p+2"),
          ("0x1.f15dc2p-1", "0x1.1ae630p+3", "0x1.907a96p+0")),
}


@pytest.mark.parametrize("i", sorted(_ROWS))
def test_thin_splat_of_a_scene(i):
    r = random.Random(i)
    P, W, H = r.choice([1500, 2500, 4000]), r.choice([640, 800]), r.choice([360, 480])
    print("thin splat of scene", i, P, W, H, flush=True)
    sc = scenes.plain_scene(seed=3000 + i, P=P, W=W, H=H)
    v = {k: sc[k].to(DEV) for k in ("means", "opacities", "scales", "rotations", "shs")}
    rs = gcam.raster_settings(sc["cam"].to(DEV), torch.zeros(3, device=DEV), 0)
    args = (v["means"], v["shs"], None, v["opacities"], v["scales"], v["rotations"], None)
    st = raster.forward(rs, *args)[4]
    dc = (torch.rand((3, H, W), generator=torch.Generator().manual_seed(i)) - 0.5).to(DEV)
    g = raster.backward(rs, st, *args, None, dc, None, None, deterministic=True)
    row, rot, scale = _ROWS[i]
    for name, want in (("rotations", rot), ("scales", scale)):
        want = torch.tensor([float.fromhex(x) for x in want], dtype=torch.float64)
        err = float((g[name][row].cpu().double() - want).norm() / want.norm())
        assert err <= 1e-6, (name, err)


@pytest.mark.parametrize("posed", [False, True], ids=["no pose", "pose"])
@pytest.mark.parametrize("det", [False, True], ids=["atomic", "fixed order"])
def test_a_splat_that_no_pixel_blends(det, posed):
    """The last splat's alpha is 1/255 only within 0.4 pixels of its centre, which
    lies half a pixel off the next ones: the reach test lets it pass, no pixel
    takes it.  A finite colour and an infinite one give the same gradients."""
    print("splat that no pixel blends", det, posed, flush=True)
    n, W, H = 40, 21, 18
    sc = scenes.plain_scene(seed=5, P=n + 1, W=W, H=H)
    g = torch.Generator().manual_seed(6)
    sc["means"][:n] = torch.cat([(torch.rand((n, 2), generator=g) - 0.5) * 2, 2 + torch.rand((n, 1), generator=g)], 1)
    sc["scales"][:n] = 0.3
    sc["opacities"][:n] = 0.05
    fx = W / (2 * sc["cam"].tanfovx)
    sc["means"][n] = torch.tensor([0.5 * 2.5 / fx, 0.0, 2.5])  # column 10.5, row 8.5, between the others
    sc["scales"][n] = 25.0 / fx  # 10 pixels
    sc["opacities"][n] = 1.0005 / 255.0
    v = {k: sc[k].to(DEV) for k in ("means", "opacities", "scales", "rotations")}
    pose = torch.tensor([0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1.0], device=DEV) if posed else None
    rs = gcam.raster_settings(sc["cam"].to(DEV), torch.zeros(3, device=DEV), 0)
    dc = (torch.rand((3, H, W), generator=g) - 0.5).to(DEV)
    got = []
    for last in (0.5, float("inf")):
        colors = torch.rand((n + 1, 3), generator=torch.Generator().manual_seed(7)).to(DEV)
        colors[n] = last
        args = (v["means"], None, colors, v["opacities"], v["scales"], v["rotations"], None)
        color, radii, _, _, st = raster.forward(rs, *args, pose=pose)
        assert int(radii[n]) > 0 and bool(torch.isfinite(color).all())
        b = raster.backward(rs, st, *args, pose, dc, None, None, deterministic=det)
        assert not np_(b["colors"][n]).any()  # no pixel took it
        got.append({k: t for k, t in b.items() if t is not None})
    for k, t in got[0].items():
        assert bool(torch.isfinite(got[1][k]).all()), k
        if det:
            assert torch.equal(t, got[1][k]), k
