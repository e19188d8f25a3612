"""What a program may do to a UNet's parameters and read from it between the
passes of a training step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(chans=(4, 8, 8), N=2, H=32, W=64, seed=3):
    import torch
    from imexlb.surrogate import UNet
    net = UNet(4, 3, list(chans), N, H, W, seed=seed)
    g = torch.Generator("cuda")
    g.manual_seed(seed + 1)
    for b in net.b:
        b.copy_(0.1 * torch.randn(b.shape, generator=g, device="cuda"))
    x = torch.randn((N, 4, H, W), generator=g, device="cuda")
    return net, x, torch.tanh(x[:, :3]).contiguous()


def _step(net, x, y):
    net.loss(net.forward(x), y)
    net.backward(net.grad_out)
    net.adam(3e-3)


@pytest.mark.parametrize("which", ["w", "b", "dw", "db", "mw", "vw", "mb", "vb"])
def test_replaced_tensors_take_part_in_training(which):
    """A parameter, gradient or moment replaced by another tensor trains as
    one whose values were set in place does."""
    import torch
    print(f"[unet] replaced {which}", flush=True)
    ends = []
    for replace in (False, True):
        net, x, y = _net()
        _step(net, x, y)
        held = getattr(net, which)
        new = held[2].abs() + 0.25
        before = new.cpu().numpy()
        if replace:
            held[2] = new
        else:
            held[2].copy_(new)
        for _ in range(3):
            _step(net, x, y)
        ends.append([v.cpu().numpy() for v in net.w + net.b])
        if which in "wb":
            assert not np.array_equal(getattr(net, which)[2].cpu().numpy(), before)  # it trained
    for k, (a, b) in enumerate(zip(*ends)):
        assert (a == b).all(), k
