"""gs_se3_adam for more poses than one round of its workgroup takes (24): every
pose as when stepped alone, bit for bit, and the pose of its own tangent."""
import pytest
import torch

from gpu_helpers import DEV
from gs_hip.pose import SE3Adam, se3_retract

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 23, 24, 25, 49])
def test_se3_adam_lanes(n):
    print("se3 adam", n, flush=True)
    g = torch.Generator().manual_seed(n)
    x0 = se3_retract((torch.randn((n, 6), generator=g) * 0.3).to(DEV))
    grads = torch.randn((4, n, 7), generator=g).to(DEV)
    opt = SE3Adam(n, DEV, lr=1e-2, X0=x0)
    one = [SE3Adam(1, DEV, lr=1e-2, X0=x0[i]) for i in sorted({0, n // 2, n - 1})]
    for it in range(4):
        opt.grad.copy_(grads[it])
        opt.step()
        for i, o in zip(sorted({0, n // 2, n - 1}), one):
            o.grad.copy_(grads[it, i:i + 1])
            o.step()
            assert torch.equal(o.xi[0], opt.xi[i]) and torch.equal(o.pose[0], opt.pose[i])
    assert torch.equal(se3_retract(opt.xi, x0), opt.pose)
    assert int(opt.step_count.item()) == 4
