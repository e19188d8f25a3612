"""The network's kernels on fields of few columns: the same results, and no
slower per value than on wide ones."""
import ctypes as C

import pytest

import test_gpu_nn_kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 3, 7, 2), (3, 5, 11, 4), (2, 7, 3, 6), (1, 2, 300, 1), (2, 2, 2, 128),
                                   (5, 3, 2, 130), (1, 1, 70, 3)])
@pytest.mark.parametrize("shift", [0, 1])
def test_pooling_and_upsampling_of_narrow_fields(shape, shift):
    K.test_pooling_and_upsampling(shape, shift)


def _time(f, repeat=20):
    import torch
    for _ in range(3):
        f()
    best = 1e9
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(repeat):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) / repeat)
    return best


@pytest.mark.parametrize("call", ["pool2", "pool2_bwd", "up2", "up2_bwd"])
def test_narrow_fields_take_the_time_of_wide_ones(call):
    """40 x 256 fields of 64 x 4 and of 4 x 64 pixels, the same values: up to
    19 times slower where a wave took a row."""
    import torch
    from imexlb._lib import lib
    ms = []
    for h, w in ((4, 64), (64, 4)):
        low = torch.zeros((40, 256, h, w), device="cuda")
        high = torch.zeros((40, 256, 2 * h, 2 * w), device="cuda")
        a, b = (high, low) if call in ("pool2", "up2_bwd") else (low, high)
        args = (40, 256, h, w) + ((256, 0) if call.startswith("up2") else ())
        f = getattr(lib(), "imexlb_nn_" + call)
        ms.append(_time(lambda: f(C.c_void_p(a.data_ptr()), C.c_void_p(b.data_ptr()), *args, None)))
    print(f"[narrow] {call}: {ms[0] * 1e3:.1f} us wide, {ms[1] * 1e3:.1f} us narrow", flush=True)
    assert ms[1] < 3.0 * ms[0], ms


# one block a CU and fewer (three chunks ahead), somewhat more with many input
# channels, more with few (plain); rows of more than 16 pixels with one chunk
@pytest.mark.parametrize("shape", [(20, 32, 70, 40, 8), (20, 128, 70, 40, 8), (20, 16, 70, 41, 5), (40, 32, 16, 64, 24),
                                   (7, 64, 40, 61, 33)])
def test_bf16_convolution_of_narrow_fields(shape):
    """Against the exact sums, and every image equal to itself alone, which
    few blocks compute: the tile does not change the sums."""
    import torch
    K.test_bf16_convolution_at_tile_edges(shape)
    N, ci, co, H, W = shape
    g = torch.Generator("cuda").manual_seed(17)
    x = torch.randn(N, H, W, ci, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(co, ci, 3, 3, generator=g, device="cuda")
    cop = 32 * -(-co // 32)
    wp = torch.empty(ci * 9 * cop, dtype=torch.bfloat16, device="cuda")
    K._call("pack_weights_bf16", w, wp, ci, co, ci, cop)
    out = torch.empty(N, co, H, W, device="cuda")
    K._call("conv3x3_bf16", x, wp, torch.zeros(co, device="cuda"), out, N, ci, co, cop, H, W, 0, 0, 1, 1)
    one = torch.empty(1, co, H, W, device="cuda")
    for k in (0, N - 1):
        K._call("conv3x3_bf16", x[k].contiguous(), wp, torch.zeros(co, device="cuda"), one, 1, ci, co, cop, H, W, 0, 0, 1, 1)
        assert torch.equal(one[0], out[k]), k


# output channels and place in a wider buffer: 16-byte, 4-byte and 2-byte
# accesses; tiles of 16 and 32 columns, one and two blocks of channels, the
# look-ahead form
@pytest.mark.parametrize("co,extra,off", [(8, 0, 0), (64, 8, 8), (64, 2, 2), (30, 0, 0), (58, 4, 2), (10, 1, 0), (6, 2, 1),
                                          (33, 0, 0), (31, 1, 1), (229, 0, 0), (12, 3, 3)])
@pytest.mark.parametrize("shape", [(3, 32, 9, 13), (2, 16, 18, 70), (24, 32, 61, 97), (20, 16, 40, 8)])
def test_bf16_output_of_any_channel_count(shape, co, extra, off):
    """The bf16 output is the FP32 output rounded, in its channels only."""
    import torch
    N, ci, H, W = shape
    g = torch.Generator("cuda").manual_seed(19)
    x = torch.randn(N, H, W, ci, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(co, ci, 3, 3, generator=g, device="cuda")
    b = torch.randn(co, generator=g, device="cuda")
    cop = 32 * -(-co // 32)
    wp = torch.empty(ci * 9 * cop, dtype=torch.bfloat16, device="cuda")
    K._call("pack_weights_bf16", w, wp, ci, co, ci, cop)
    f32 = torch.empty(N, co, H, W, device="cuda")
    out = torch.full((N, H, W, co + extra), 7.0, dtype=torch.bfloat16, device="cuda")
    K._call("conv3x3_bf16", x, wp, b, f32, N, ci, co, cop, H, W, 0, 0, 1, 1)
    K._call("conv3x3_bf16", x, wp, b, out, N, ci, co, cop, H, W, co + extra, off, 1, 0)
    assert torch.equal(out[..., off:off + co], f32.permute(0, 2, 3, 1).to(torch.bfloat16))
    rest = torch.cat([out[..., :off], out[..., off + co:]], 3)
    assert bool((rest == 7.0).all())
