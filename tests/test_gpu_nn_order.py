"""The FP32 convolution and its weight gradient on the matrix instructions give
the sums of the plain loops (tests/nn_chain.c), bit for bit: products added one
after another, each as a fused multiply-add, subnormal values included."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import test_gpu_nn_kernels as K

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not available")]


@pytest.fixture(scope="module")
def chain(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("chain") / "nn_chain.so")
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "nn_chain.c")
    fma = ["-mfma"] if " fma " in open("/proc/cpuinfo").read() else []
    subprocess.run(["gcc", "-O2", "-std=c11", "-ffp-contract=off", "-fopenmp", "-fPIC", "-shared", *fma, src, "-lm", "-o",
                    so], check=True)
    return C.CDLL(so)


def _p(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


def _values(rng, shape, tiny):
    """Normal values of many magnitudes; tiny: products about the smallest
    normal number and below."""
    v = rng.normal(0, 1, shape) * np.exp2(rng.integers(-12, 12, shape))
    return (v * (2.0 ** -76 if tiny else 1.0)).astype(np.float32)


# the 16-column tile, 4 x 32, 8 x 32 and 8 x 32 for 64 channels; one to six
# input channels, whole and ragged chunks
SHAPES = [(1, 1, 1, 1, 1), (2, 3, 5, 9, 7), (1, 15, 31, 8, 16), (2, 17, 33, 5, 33), (1, 6, 40, 30, 70), (3, 8, 3, 2, 70),
          (20, 5, 31, 61, 97), (20, 9, 20, 61, 97), (9, 17, 65, 121, 64)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("tiny", [False, True])
def test_convolution_is_the_loop_s_sum(chain, shape, tiny):
    import torch
    N, ci, co, H, W = shape
    print(f"[order] conv {shape} tiny {tiny}", flush=True)
    rng = np.random.default_rng(23)
    x, w = _values(rng, (N, ci, H, W), tiny), _values(rng, (co, ci, 3, 3), tiny)
    b = (_values(rng, co, tiny) * np.float32(2.0 ** -70 if tiny else 1.0)).astype(np.float32)
    ref = np.empty((N, co, H, W), np.float32)
    chain.conv_chain(_p(x), _p(w), _p(b), _p(ref), N, ci, co, H, W)
    out = torch.empty(N, co, H, W, device="cuda")
    xd, wd, bd = (torch.tensor(v, device="cuda") for v in (x, w, b))
    K._call("conv3x3", xd, wd, bd, out, N, ci, co, H, W, 0)
    got = out.cpu().numpy()
    assert (got == ref).all(), int((got != ref).sum())
    if tiny and ref.size > 100:
        assert ((ref != 0) & (np.abs(ref) < 2.0 ** -126)).any()  # subnormal sums among them


@pytest.mark.parametrize("shape", [(1, 1, 1, 1, 1), (2, 3, 5, 9, 7), (3, 16, 17, 16, 16), (2, 40, 24, 35, 33),
                                   (2, 33, 20, 200, 300), (1, 20, 33, 200, 300), (2, 17, 33, 200, 300)])
@pytest.mark.parametrize("tiny", [False, True])
def test_weight_gradient_is_the_loop_s_sum(chain, shape, tiny):
    import torch

    from imexlb._lib import lib
    N, ci, co, H, W = shape
    print(f"[order] dw {shape} tiny {tiny}", flush=True)
    rng = np.random.default_rng(29)
    x, g = _values(rng, (N, ci, H, W), tiny), _values(rng, (N, co, H, W), tiny)
    ref = np.empty((co, ci, 3, 3), np.float32)
    chain.dw_chain(_p(x), _p(g), _p(ref), N, ci, co, H, W)
    n = int(lib().imexlb_nn_conv3x3_dw_work(ci, co, H, W))
    dw, work = torch.zeros(co, ci, 3, 3, device="cuda"), torch.empty(n, device="cuda")
    xd, gd = torch.tensor(x, device="cuda"), torch.tensor(g, device="cuda")
    K._call("conv3x3_dw_ordered", xd, gd, dw, work, n, N, ci, co, H, W)
    got = dw.cpu().numpy()
    assert (got == ref).all(), int((got != ref).sum())
    if tiny and ref.size > 100:
        assert ((ref != 0) & (np.abs(ref) < 2.0 ** -126)).any()
