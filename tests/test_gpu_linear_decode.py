"""A decode step's W8A8 Linear in one launch (mtrt_linear_w8a8_decode): rows 1 to 16, row lengths off whole slices and groups
and with fewer slices than waves, columns off whole and half tiles, the largest M * K it takes and the first it does not.
The sums are exact integers, so every result is checked bit for bit."""
import importlib

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(1, 128, 1), (1, 129, 16), (1, 4096, 4096), (1, 16384, 31), (2, 8192, 33), (3, 130, 17), (4, 4096, 48), (5, 4096, 48),
                                   (5, 1031, 40), (16, 1024, 80), (16, 1025, 80), (15, 255, 100), (16, 136, 16), (1, 16385, 20), (17, 256, 20), (7, 2049, 1000)])
@pytest.mark.parametrize("bias", [False, True])
def test_one_launch_is_exact(pkg, M, K, N, bias):
    import torch
    tp = importlib.import_module(pkg.__name__ + ".tp")
    g = torch.Generator().manual_seed(M * 1000 + K)
    lin = tp.Linear(K, N, bias=bias, dtype=tp.float16, quant_dtype=tp.int8, weight_quant_dim=0)
    lin.weight = tp.Tensor((torch.randn((N, K), generator=g) * 0.3).half())
    lin.weight_scale = tp.Tensor((lin.weight.torch().float().abs().amax(1) / 127 + 1e-3).half())
    lin.input_scale = tp.Tensor(torch.tensor(3.0 / 127).half())
    if bias:
        lin.bias = tp.Tensor(torch.randn(N, generator=g).half())
    flat = torch.zeros(M * K + 1, dtype=torch.float16, device="cuda")     # x off 16-byte alignment: rows start on any element
    flat[1:] = torch.randn(M * K, generator=g).half().cuda()
    x = tp.Tensor(flat[1:].view(M, K))
    y = lin(x).torch()
    assert lin.route() == "w8a8"
    Kp = (K + 127) // 128 * 128
    if M <= 16 and M * Kp <= 16384:
        assert pkg.last_kernel() == "mtrt_linear_w8a8_decode"
    else:
        assert pkg.last_kernel() != "mtrt_linear_w8a8_decode"
    xq = tp.quantize(x, lin.input_scale, tp.int8).torch().cpu().double()
    wq = tp.quantize(lin.weight, lin.weight_scale, tp.int8, 0).torch().cpu().double()
    acc = (xq @ wq.T).float()                                       # below 2^24 or rounded once, as the conversion of the sum is
    ref = ((acc * lin.input_scale.torch().float().cpu()) * lin.weight_scale.torch().float().cpu()).half()
    if bias:
        ref = (ref.float() + lin.bias.torch().float().cpu()).half()
    assert torch.equal(y.cpu(), ref)
