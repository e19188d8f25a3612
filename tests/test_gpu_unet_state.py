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


def _conv_t(dz, w):
    """Data gradient of a 3x3 convolution in 64 bits (dz, w: FP64)."""
    import torch
    N, co, H, W = dz.shape
    p = torch.nn.functional.pad(dz, (1, 1, 1, 1))
    y = 0.0
    for k in range(9):
        part = p[:, :, 2 - k // 3:2 - k // 3 + H, 2 - k % 3:2 - k % 3 + W].reshape(N, co, -1)
        y = y + torch.matmul(w[:, :, k // 3, k % 3].t().contiguous(), part)
    return y.view(N, -1, H, W)


def test_input_gradients_are_those_of_the_last_backward_pass():
    """dx[k] does not change with the weights, the loss or the output
    gradient's buffer afterwards, also for replaced weights."""
    import torch
    for replace in (False, True):
        net, x, y = _net()
        if replace:
            net.w[1] = net.w[1] * 1.5
        net.loss(net.forward(x), y)
        net.backward(net.grad_out)
        then = [v.cpu().numpy() for v in net.dx]
        w1 = net.w[1].double().cpu()
        dz1 = net.dz[1].double().cpu()
        assert len(then) == len(net.dx) == len(net.shapes)
        net.adam(0.5)
        net.loss(net.forward(x), -y)
        net.grad_out.fill_(7.0)
        for k, a in enumerate(then):
            assert (net.dx[k].cpu().numpy() == a).all(), (replace, k)
        assert (net.dx[-1].cpu().numpy() == then[-1]).all()
        ref = _conv_t(dz1, w1)
        bound = 9 * 4 * 2.0 ** -24 * _conv_t(dz1.abs(), w1.abs()) + 1e-30
        assert bool((torch.tensor(then[1]).double() - ref).abs().le(bound).all())
        with pytest.raises(IndexError):
            net.dx[len(net.shapes)]


def test_backward_stores_the_joined_gradients_at_full_size():
    """What a backward pass at the network's real size (4 levels, 32 to 256
    channels, 128 x 512) leaves in its buffers, each from the buffers it was
    made from: every convolution's data gradient, gated by the ReLU before
    it, within the error bound of an FP32 sum of 9 CO terms; the upsampled,
    pooled and skip gradients, a few exact or once-rounded operations, bit
    for bit."""
    import torch
    chans = [32, 64, 128, 256]
    L = len(chans)
    net, x, y = _net(chans, 2, 128, 512)
    net.loss(net.forward(x), y)
    net.backward(net.grad_out)
    u = 2.0 ** -24
    last = len(net.shapes) - 1

    def check(k, got, gate):
        dz = (net.dz[k] if k < last else net.grad_out).double()
        w = net.w[k].double()
        ref, size = _conv_t(dz, w), _conv_t(dz.abs(), w.abs())
        if gate is not None:
            on = net.out[gate] > 0
            assert bool((got[~on] == 0).all()), ("gate", k)
            ref, size = ref * on, size * on
        assert bool((got.double() - ref).abs().le(9 * net.shapes[k][0] * u * size + 1e-30).all()), ("dgrad", k)

    print("[unet] stored gradients at full size", flush=True)
    check(last, net.dz[last - 1], last - 1)
    k = last
    for l in range(L - 1):
        k -= 2
        check(k + 1, net.dz[k], k)
        check(k, net.dcat[l], None)
        up = net.dcat[l][:, :chans[l + 1]]
        s = (up[:, :, ::2, ::2] + up[:, :, ::2, 1::2]) + (up[:, :, 1::2, ::2] + up[:, :, 1::2, 1::2])
        assert torch.equal(net.dz[k - 1], torch.where(net.out[k - 1] > 0, s, torch.zeros_like(s))), ("up", l)
    for l in range(L - 1, -1, -1):
        k -= 2
        check(k + 1, net.dz[k], k)
        if l == 0:
            break
        check(k, net.dpool[l], None)
        g = 0.25 * net.dpool[l].repeat_interleave(2, 2).repeat_interleave(2, 3) + net.dcat[l - 1][:, chans[l]:]
        assert torch.equal(net.dz[k - 1], torch.where(net.out[k - 1] > 0, g, torch.zeros_like(g))), ("pool", l)
    assert k == 0
