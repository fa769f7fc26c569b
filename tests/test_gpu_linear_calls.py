"""tp.Linear in one native call (mtrt_hip_linear): the activation pass and the GEMMs on re-laid weights at the sizes where
they can go wrong - rows around the tile heights, columns off whole tiles, row lengths off whole slices and groups, split
K - for every route, element type and activation type."""
import importlib

import pytest

pytestmark = pytest.mark.gpu

UNIT = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


@pytest.fixture(scope="module")
def tp(pkg):
    return importlib.import_module(pkg.__name__ + ".tp")


def _module(tp, seed, K, N, dname, qname, bias, x_scale):
    import torch
    g = torch.Generator().manual_seed(seed)
    td = getattr(torch, dname)
    lin = tp.Linear(K, N, bias=bias, dtype=getattr(tp, dname), quant_dtype=None if qname is None else getattr(tp, qname), weight_quant_dim=0 if qname else None)
    lin.weight = tp.Tensor((torch.randn((N, K), generator=g) * 0.3).to(td))
    if bias:
        lin.bias = tp.Tensor(torch.randn(N, generator=g).to(td))
    if qname:
        top = {"int8": 127.0, "int4": 7.0, "float8": 448.0}[qname]
        lin.weight_scale = tp.Tensor((lin.weight.torch().float().abs().amax(1) / top).to(td))
        if x_scale:
            lin.input_scale = tp.Tensor(torch.tensor(4.0 / top).to(td))
    return lin, g


def _operands(tp, lin, x):
    """What the fake-quant product multiplies: float64 x', W'."""
    w = lin.weight
    if lin.quant_dtype is not None:
        w = tp.dequantize(tp.quantize(w, lin.weight_scale, lin.quant_dtype, 0), lin.weight_scale, lin.dtype, 0)
        if lin.input_scale is not None:
            x = tp.dequantize(tp.quantize(x, lin.input_scale, lin.quant_dtype), lin.input_scale, lin.dtype)
    return x.device_data().double(), w.device_data().double()


SHAPES = [(1, 64, 32), (16, 4096, 100), (32, 10496, 384), (33, 2048, 40), (64, 128, 31), (65, 1152, 129), (100, 11520, 300), (129, 192, 257),
          (300, 4096, 1001), (1000, 1024, 1000), (1100, 2048, 3000), (2100, 256, 770),
          (3, 65, 33), (17, 71, 640), (40, 1031, 260), (300, 2049, 1000), (900, 1023, 1030)]


@pytest.mark.parametrize("qname,x_scale", [(None, False), ("float8", True), ("int8", True), ("int4", True), ("int8", False), ("int4", False)])
@pytest.mark.parametrize("dname", ["float16", "bfloat16", "float32"])
def test_linear_against_float64(tp, dname, qname, x_scale):
    import torch
    u = UNIT[dname]
    for i, (M, K, N) in enumerate(SHAPES):
        lin, g = _module(tp, 5 * i + 1, K, N, dname, qname, i % 3 != 1, x_scale)
        x = tp.Tensor(torch.randn((M, K), generator=g).to(getattr(torch, dname)).cuda())
        lin(x)
        assert tp._native().tp_linear(lin, x) is not NotImplemented, (M, K, N)
        y = lin(x).torch().double()
        if lin.route() == "w8a8":                      # the codes' product times both scales, nothing rounded in between
            xd = tp.quantize(x, lin.input_scale, tp.int8).torch().double() * float(lin.input_scale.torch())
            wd = tp.quantize(lin.weight, lin.weight_scale, tp.int8, 0).torch().double() * lin.weight_scale.device_data().double()[:, None]
        else:
            xd, wd = _operands(tp, lin, x)
        b = lin.bias.device_data().double() if lin.bias is not None else 0.0
        ref, mass = xd @ wd.T + b, xd.abs() @ wd.abs().T + (b.abs() if lin.bias is not None else 0.0)
        assert qname != "int4" or x_scale or dname != "float16" or K % 64 or lin.route() == "w4a16"
        if lin.route() == "w8a8":
            # exact integer sums; two f32 products, a rounding to f16, the sum with the bias rounded once more
            core = ref - b
            tol = (3 * 2.0 ** -24 + u) * core.abs() + u * (ref.abs() + u * core.abs()) + 2.0 ** -24
        elif lin.route() == "w4a16":                   # f32 sums rounded to f16, the sum with the bias rounded once more
            core = ref - b
            tol = u * core.abs() + (1 + u) * (K + 2) * 2.0 ** -24 * mass + u * ref.abs() * (1 + u) + 2.0 ** -24
        else:
            # f32 accumulation in any order (K additions, the products exact for 16-bit operands), one rounding
            tol = u * ref.abs() + (1 + u) * (K + 2) * 2.0 ** -24 * mass + 2.0 ** -24
        bad = ((y - ref).abs() > tol).sum().item()
        assert y.shape == (M, N) and bad == 0, (M, K, N, bad, float(((y - ref).abs() / tol).max()))


@pytest.mark.parametrize("dname,qname", [("float16", "int8"), ("float16", None), ("bfloat16", "float8"), ("float16", "int4")])
def test_the_general_path_gives_the_same(tp, dname, qname):
    """Strided rows, host operands and leading axes reach the same kernels; a parameter that changes is noticed."""
    import torch
    td = getattr(torch, dname)
    K, N = 192, 72
    lin, g = _module(tp, 3, K, N, dname, qname, True, qname not in (None, "int4"))
    host = torch.randn((2, 3, K), generator=g).to(td)
    y = lin(tp.Tensor(host))
    assert y.shape == (2, 3, N) and y.dtype is lin.dtype
    wide = torch.zeros((2, 3, K + 1), dtype=td, device="cuda")
    wide[:, :, 1:] = host.cuda()
    assert torch.equal(lin(tp.Tensor(wide[:, :, 1:])).torch(), y.torch())
    flat = torch.empty(6 * K + 1, dtype=td, device="cuda")           # contiguous, off 16-byte alignment
    flat[1:] = host.cuda().reshape(-1)
    assert torch.equal(lin(tp.Tensor(flat[1:].view(2, 3, K))).torch(), y.torch())
    assert lin(tp.Tensor(host[:, :0])).shape == (2, 0, N)
    with torch.no_grad():
        lin.bias.device_data().zero_()
    zero = lin(tp.Tensor(host.cuda())).torch()
    assert not torch.equal(zero, y.torch())
    lin.bias = None
    assert torch.equal(lin(tp.Tensor(host.cuda())).torch(), zero)
    lin.weight.device_data().neg_()                                  # in place: the version says so
    assert torch.allclose(lin(tp.Tensor(host.cuda())).torch().float(), -zero.float(), atol=0.06 if qname == "int4" else 0.03)


@pytest.mark.parametrize("dname,qname", [("float16", "int8"), ("float16", None), ("bfloat16", "float8"), ("float16", "int4")])
def test_in_place_updates_of_a_subclass_parameter_are_noticed(tp, dname, qname):
    """The prepared weights follow torch's own in-place updates of the weight, of whichever Tensor class it is."""
    import torch

    class Parameter(tp.Tensor):
        pass
    K, N = 192, 72
    lin, g = _module(tp, 4, K, N, dname, qname, False, qname not in (None, "int4"))
    lin.weight = Parameter(lin.weight.torch().cuda())
    x = tp.Tensor(torch.randn((5, K), generator=g).to(getattr(torch, dname)).cuda())
    y = lin(x).torch()
    assert tp._native().tp_linear(lin, x) is not NotImplemented      # the plan is current
    lin.weight.torch().zero_()
    assert tp._native().tp_linear(lin, x) is NotImplemented
    assert bool((lin(x).torch() == 0).all()) and bool((y != 0).any())


@pytest.mark.parametrize("dname,qname,x_scale", [("float16", "int8", False), ("bfloat16", "float8", True), ("float16", None, False)])
def test_a_strided_bias_prepares_the_weights_once(tp, monkeypatch, dname, qname, x_scale):
    """A bias that is not contiguous takes the general path, which quantizes the weights on its first call only; the
    results are those of the same bias laid out densely."""
    import torch
    K, N = 192, 72
    lin, g = _module(tp, 8, K, N, dname, qname, True, x_scale)
    x = tp.Tensor(torch.randn((5, K), generator=g).to(getattr(torch, dname)).cuda())
    dense = lin(x).torch()
    wide = torch.zeros((N, 2), dtype=dense.dtype, device="cuda")
    wide[:, 0] = lin.bias.device_data()
    lin.bias = tp.Tensor(wide[:, 0])
    assert tp._native().tp_linear(lin, x) is NotImplemented
    first = lin(x).torch()
    quantize, of_weights = tp.quantize, []

    def counted(t, *rest):
        if t is lin.weight:
            of_weights.append(t)
        return quantize(t, *rest)
    monkeypatch.setattr(tp, "quantize", counted)
    assert torch.equal(lin(x).torch(), first) and not of_weights
    assert torch.allclose(first.float(), dense.float(), rtol=4 * UNIT[dname], atol=1e-4)
    lin.weight.device_data().zero_()                                 # a kept matrix goes with the plan
    assert torch.equal(lin(x).torch(), lin.bias.torch().expand(5, N)) and bool(of_weights) == (qname is not None)
    del of_weights[:]
    assert torch.equal(lin(x).torch(), lin.bias.torch().expand(5, N)) and not of_weights


@pytest.mark.parametrize("why", ["little memory", "none"])
def test_weights_that_do_not_fit_twice(tp, pkg, monkeypatch, why):
    """Without room for the fragments a plain 16-bit Linear runs on its parameter as it is, with the same result up to the
    order of its sums."""
    import torch
    lin, g = _module(tp, 9, 4096, 200, "float16", None, True, False)
    x = tp.Tensor(torch.randn((5, 4096), generator=g).half().cuda())
    y = lin(x).torch()
    assert pkg.last_kernel().startswith("mtrt_gemm_dense_frag_f16_")
    total = torch.cuda.mem_get_info()[1]
    if why == "none":
        def full(w):
            raise torch.OutOfMemoryError("no room")
        monkeypatch.setattr(tp.Linear, "_fragments", staticmethod(full))
    else:
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (total // 8, total))
    lin.invalidate()
    again = lin(x).torch()
    assert pkg.last_kernel() == "mtrt_gemm_dense_rows32_f16"
    xd, wd = _operands(tp, lin, x)
    tol = 2 * (UNIT["float16"] * y.double().abs() + 4100 * 2.0 ** -24 * (xd.abs() @ wd.abs().T) + 2.0 ** -24)
    assert bool(((again.double() - y.double()).abs() <= tol).all())


def test_a_first_call_that_is_recorded(tp):
    """A plain Linear whose first call is recorded into a graph: eager calls before and after a replay give its result."""
    import torch
    lin, g = _module(tp, 10, 256, 200, "float16", None, True, False)
    lin.weight, lin.bias = tp.Tensor(lin.weight.torch().cuda()), tp.Tensor(lin.bias.torch().cuda())
    x = tp.Tensor(torch.randn((5, 256), generator=g).half().cuda())
    xd, wd = _operands(tp, lin, x)
    ref = xd @ wd.T + lin.bias.torch().double()
    tol = UNIT["float16"] * ref.abs() + 260 * 2.0 ** -24 * (xd.abs() @ wd.abs().T + 8) + 2.0 ** -24
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = lin(x).torch()
    assert bool(((lin(x).torch().double() - ref).abs() <= tol).all())
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert bool(((y.double() - ref).abs() <= tol).all())
        assert torch.equal(lin(x).torch(), y)


def test_arguments_of_the_c_call(pkg):
    import ctypes
    L = pkg.lib()

    class Plan(ctypes.Structure):
        _fields_ = [(n, ctypes.c_int32) for n in ("route", "dtype", "q_dtype", "reserved")] + [("K", ctypes.c_int64), ("N", ctypes.c_int64)] + \
                   [(n, ctypes.c_void_p) for n in ("w", "w_frag", "w_scale", "x_scale", "bias")]

    def status(**k):
        v = dict(route=2, dtype=pkg.F16, q_dtype=-1, K=64, N=32, w_frag=256)
        M = k.pop("M", 4)
        v.update(k)
        return L.mtrt_hip_linear(None, ctypes.byref(Plan(**v)), 256, 256, M, None, 0)
    assert status(M=0) == 0
    for bad in (dict(route=3), dict(dtype=pkg.I8), dict(K=0), dict(N=-1), dict(M=-1), dict(w_frag=None), dict(q_dtype=pkg.I8),
                dict(q_dtype=pkg.I8, x_scale=256), dict(route=0), dict(route=1, dtype=pkg.BF16), dict(w_frag=8), dict(bias=1)):
        assert status(**bad) == 1, bad
    assert L.mtrt_hip_linear(None, None, 256, 256, 4, None, 0) == 1
    assert L.mtrt_hip_linear_workspace(None, 4) == 0
    assert L.mtrt_hip_linear_fragments_bytes(pkg.I8, 130, 33) == 64 * 256 and L.mtrt_hip_linear_fragments_bytes(pkg.BF16, 64, 1) == 32 * 128
    assert L.mtrt_hip_linear_fragments_bytes(pkg.F32, 64, 32) == 0
