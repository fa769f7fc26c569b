"""tp.Linear modules of 8 Mi float8 weights and more, whose prepared weights are the codes, with their values beside them up to a size: the bits of the dequantized
weights' products, in the kernels of either, with the input quantized or plain, scales per tensor or output channel, and where the values find no room."""
import ctypes
import importlib

import pytest

from test_gpu_linear_codes import Plan

pytestmark = pytest.mark.gpu

SMALL = (2048, 4100)                                                 # K, N: 8.4 Mi weights
BOTH_UP_TO = {"float16": 32 << 20, "bfloat16": 40 << 20}


@pytest.fixture(scope="module")
def tp(pkg):
    return importlib.import_module(pkg.__name__ + ".tp")


def _module(tp, K, N, dname, per_channel, x_scale):
    import torch
    td = getattr(torch, dname)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    lin = tp.Linear(K, N, dtype=getattr(tp, dname), quant_dtype=tp.float8, weight_quant_dim=0 if per_channel else None)
    w = (torch.randn((N, K), generator=g, device="cuda") * 0.3).to(td)
    lin.weight, lin.bias = tp.Tensor(w), tp.Tensor(torch.randn(N, generator=g, device="cuda").to(td))
    lin.weight_scale = tp.Tensor(((w.float().abs().amax(1) if per_channel else w.float().abs().amax()) / 448).to(td).cpu())
    if x_scale:
        lin.input_scale = tp.Tensor(torch.tensor(4.0 / 448).to(td))
    return lin, g


class Dequantized:
    """The product of the module's dequantized weights, through the C ABI."""

    def __init__(self, pkg, tp, lin, code):
        import torch
        self.pkg, self.lin = pkg, lin
        self.N, self.K = lin.weight.shape
        dim = lin.weight_quant_dim
        w = tp.dequantize(tp.quantize(lin.weight, lin.weight_scale, tp.float8, dim), lin.weight_scale, lin.dtype, dim).device_data().contiguous()
        self.frag = torch.empty(pkg.lib().mtrt_hip_linear_fragments_bytes(code, self.K, self.N), dtype=torch.int8, device="cuda")
        pkg.check(pkg.lib().mtrt_hip_linear_prepack_fragments(None, w.data_ptr(), code, self.frag.data_ptr(), self.K, self.N))
        self.scale = None if lin.input_scale is None else lin.input_scale.torch().float().reshape(1).cuda()
        self.plan = Plan(route=2, dtype=code, q_dtype=-1 if self.scale is None else pkg.F8E4M3FN, K=self.K, N=self.N, w_frag=self.frag.data_ptr(),
                         x_scale=None if self.scale is None else self.scale.data_ptr(), bias=lin.bias.device_data().data_ptr())
        torch.cuda.synchronize()

    def __call__(self, x):
        import torch
        L, M = self.pkg.lib(), x.shape[0]
        need = L.mtrt_hip_linear_workspace(ctypes.byref(self.plan), M)
        ws, y = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda"), torch.full((M, self.N), 7.0, dtype=x.dtype, device="cuda")
        stream = torch.cuda.current_stream().cuda_stream
        self.pkg.check(L.mtrt_hip_linear(stream, ctypes.byref(self.plan), x.data_ptr(), y.data_ptr(), M, ws.data_ptr(), need))
        torch.cuda.synchronize()
        return y


def _compare(pkg, tp, lin, g, dname, kernels):
    """kernels: whether those of more than 16 rows are the codes'"""
    import torch
    code, xn = {"float16": (pkg.F16, "f16"), "bfloat16": (pkg.BF16, "bf16")}[dname]
    want = Dequantized(pkg, tp, lin, code)
    for M in (5, 16, 17, 300):
        x = torch.randn((M, want.K), generator=g, device="cuda").to(getattr(torch, dname))
        y = lin(tp.Tensor(x)).torch()
        name = pkg.last_kernel()
        assert tp._native().tp_linear(lin, tp.Tensor(x)) is not NotImplemented
        assert torch.equal(y.view(torch.int16), want(x).view(torch.int16)), (M, want.K, want.N, name)
        if M > 16:
            assert name.startswith("mtrt_gemm_dense_frag_%s_" % xn) and name.startswith("mtrt_gemm_dense_frag_%s_f8_" % xn) == kernels, (M, name)


@pytest.mark.parametrize("per_channel,x_scale", [(True, True), (False, True), (True, False), (False, False)])
@pytest.mark.parametrize("dname", ["float16", "bfloat16"])
def test_modules_of_every_size(pkg, tp, dname, per_channel, x_scale):
    # ragged K only where the input is quantized: otherwise the [N, K] kernels serve small products
    for K, N in (SMALL, (4096, 8450), (4096, 11008)) + (((2050, 4100),) if x_scale else ()):
        lin, g = _module(tp, K, N, dname, per_channel, x_scale)
        lin(tp.Tensor(lin.weight.device_data()[:1]))
        plan = lin._prepared()
        assert "codes_frag" in plan and "weight" not in plan and ("values_frag" in plan) == (K * N < BOTH_UP_TO[dname])
        _compare(pkg, tp, lin, g, dname, K * N >= BOTH_UP_TO[dname])


@pytest.mark.parametrize("why", ["little memory", "no dequantized matrix", "no fragments"])
def test_values_that_find_no_room(pkg, tp, monkeypatch, why):
    """The codes alone serve every call: also where memory that was said to be there is not."""
    import torch
    lin, g = _module(tp, *SMALL, "bfloat16", True, True)
    with monkeypatch.context() as m:
        def full(*args):
            raise torch.OutOfMemoryError("no room")
        if why == "little memory":
            total = torch.cuda.mem_get_info()[1]
            m.setattr(torch.cuda, "mem_get_info", lambda *a: (total // 8, total))
        elif why == "no fragments":
            fragments = tp.Linear._fragments
            m.setattr(tp.Linear, "_fragments", staticmethod(lambda w, *code: fragments(w, *code) if code else full()))
        else:
            m.setattr(tp, "dequantize", full)
        plan = lin._prepared()
    assert "codes_frag" in plan and "values_frag" not in plan
    _compare(pkg, tp, lin, g, "bfloat16", True)


@pytest.mark.parametrize("dname", ["float16", "bfloat16"])
def test_a_plain_input_of_a_ragged_length(pkg, dname):
    """Through the C ABI, whatever K: the bits of dequantized fragments without their [N, K]."""
    import torch
    L, td, code = pkg.lib(), getattr(torch, dname), {"float16": pkg.F16, "bfloat16": pkg.BF16}[dname]
    for M, K, N in ((3, 65, 33), (16, 1000, 100), (17, 1000, 640), (300, 2049, 1000)):
        g = torch.Generator(device="cuda").manual_seed(M + K + N)
        codes = torch.randint(0, 127, (N, K), generator=g, device="cuda", dtype=torch.uint8)
        scale = (torch.rand(N, generator=g, device="cuda") * 0.01 + 0.001).to(td).float()
        w = torch.empty((N, K), dtype=td, device="cuda")
        pkg.check(L.mtrt_hip_dequantize(None, codes.data_ptr(), pkg.F8E4M3FN, w.data_ptr(), code, scale.data_ptr(), pkg.SCALE_ROW, N, K, N))
        x = torch.randn((M, K), generator=g, device="cuda").to(td)
        out = []
        for route, weights, dtype in ((2, w, code), (3, codes, pkg.F8E4M3FN)):
            frag = torch.empty(L.mtrt_hip_linear_fragments_bytes(dtype, K, N), dtype=torch.int8, device="cuda")
            pkg.check(L.mtrt_hip_linear_prepack_fragments(None, weights.data_ptr(), dtype, frag.data_ptr(), K, N))
            p = Plan(route=route, dtype=code, q_dtype=-1, K=K, N=N, w_frag=frag.data_ptr(), w_scale=scale.data_ptr() if route == 3 else None)
            need = L.mtrt_hip_linear_workspace(ctypes.byref(p), M)
            ws, y = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda"), torch.full((M, N), 7.0, dtype=td, device="cuda")
            pkg.check(L.mtrt_hip_linear(None, ctypes.byref(p), x.data_ptr(), y.data_ptr(), M, ws.data_ptr(), need))
            torch.cuda.synchronize()
            out.append(y)
        assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16)), (M, K, N, pkg.last_kernel())
