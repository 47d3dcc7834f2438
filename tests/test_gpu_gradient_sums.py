"""The render backward's sums, where another grouping shows.

* Scenes whose rotation gradients are decided by the rounding of one thin,
  tilted splat's second moments: in the fixed-order mode that splat's gradients
  are the recorded ones of the reference formula summed pixel by pixel (the
  same operations in the same order, so to the bit; 1e-6 of the row's norm is
  allowed for another compiler's contractions).  Sums by 4 x 4-pixel cells differ
  from them by 5e-5 to 2e-4."""
import random

import pytest
import torch

from gpu_helpers import DEV
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
