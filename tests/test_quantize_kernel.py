"""The quantisation kernel against the tensor operations it stands for: the
same words and scales, bit for bit (no tolerance: both round the same fp32
quotients)."""
from __future__ import annotations

import pytest
import torch

import nibblegemm_amd as ng
from nibblegemm_amd import quant

pytestmark = pytest.mark.gpu


def _same(W, g):
    got, want = ng.quantize_device(W, g), quant._quantize_ops(W, g)
    assert quant._kernel_quantizes(W, g)
    assert torch.equal(got.qweight, want.qweight)
    assert torch.equal(got.scales.view(torch.int16), want.scales.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,N,g", [(128, 8, 128), (64, 128, 64), (512, 1000, 128), (192, 130, 64),
                                   (256, 1, 32), (1024, 127, 512), (8, 3, 8), (4096, 1024, 128)])
def test_words_and_scales(K, N, g, dtype):
    gen = torch.Generator(device="cuda").manual_seed(K + N + g)
    _same((torch.randn((K, N), generator=gen, device="cuda") * 0.02).to(dtype), g)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_halfway_quotients(dtype):
    """Quotients on and next to every half: the group's largest value is 7 s,
    the others (n + 1/2) s, exactly and one ulp to either side."""
    s = 0.125
    W = torch.zeros((128, 64), dtype=dtype, device="cuda")
    W[0] = 7 * s
    halves = (torch.arange(-7, 7, device="cuda").to(dtype) + 0.5) * s
    W[1:15] = halves[:, None]
    up, down = torch.full_like(halves, 100.0), torch.full_like(halves, -100.0)
    W[15:29] = torch.nextafter(halves, up)[:, None]
    W[29:43] = torch.nextafter(halves, down)[:, None]
    W[0, 1::2] = 7 * s * 1.5  # and a scale that is no power of two
    _same(W, 128)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_zeros_infinities_nans_and_extremes(dtype):
    gen = torch.Generator(device="cuda").manual_seed(9)
    W = torch.randn((256, 64), generator=gen, device="cuda").to(dtype)
    W[:128, 0] = 0.0
    W[5, 1] = float("inf")
    W[6, 2] = -float("inf")
    W[7, 3] = float("nan")
    W[:, 4] = torch.finfo(dtype).tiny
    W[:, 5] = torch.finfo(dtype).max
    W[3, 6] = torch.finfo(dtype).max
    W[:, 7] = -0.0
    W[:, 8] *= torch.finfo(dtype).tiny
    W[:, 9] = W[:, 9].abs() * (torch.finfo(dtype).max / 8)
    _same(W, 128)


def test_views_and_other_dtypes_take_the_operations():
    W = torch.randn((256, 200), device="cuda")
    for V in (W[:, :100], W.t()[:128].t().t(), W.double()):
        assert not quant._kernel_quantizes(V, 64)
        got = ng.quantize_device(V, 64) if V.shape[0] % 64 == 0 else None
        if got is not None:
            assert torch.equal(got.qweight, quant._quantize_ops(V.contiguous().float(), 64).qweight)
    negated = torch._neg_view(W)  # contiguous; its memory holds -values
    assert not quant._kernel_quantizes(negated, 64)
    want = ng.quantize_device(-W, 64)
    assert torch.equal(ng.quantize_device(negated, 64).qweight, want.qweight)
    offset = torch.randn(128 * 64 + 1, device="cuda")[1:].view(128, 64)  # 4-byte aligned rows
    _same(offset, 128)


def test_quantises_in_a_graph_and_on_a_side_stream():
    W = torch.randn((512, 256), device="cuda").half()
    want = quant._quantize_ops(W, 128)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = ng.quantize_device(W, 128)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got.qweight, want.qweight)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ng.quantize_device(W, 128)
    for _ in range(3):
        out.qweight.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.qweight, want.qweight) and torch.equal(out.scales, want.scales)
