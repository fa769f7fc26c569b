"""A 16-bit Linear of up to 16 rows in one launch: row lengths around whole slices and what eight waves share, element counts around
the two limits, columns around what a workgroup owns, for plain inputs and inputs that go through each kind of code."""
import importlib

import pytest

pytestmark = pytest.mark.gpu

TOP = {"int8": 127.0, "int4": 7.0, "float8": 448.0}
CODE = {"int8": "i8", "int4": "i4", "float8": "f8"}
SHORT = {"float16": "f16", "bfloat16": "bf16"}
UNIT = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


@pytest.fixture(scope="module")
def tp(pkg):
    return importlib.import_module(pkg.__name__ + ".tp")


@pytest.mark.parametrize("dname,qname", [("float16", None), ("bfloat16", None), ("float16", "float8"), ("bfloat16", "float8"), ("bfloat16", "int8"),
                                         ("bfloat16", "int4"), ("float16", "int4")])
def test_against_float64(tp, pkg, dname, qname):
    import torch
    td, u = getattr(torch, dname), UNIT[dname]
    units = torch.cuda.get_device_properties(0).multi_processor_count
    # (rows, K, N): the last two with weights of more than 48 MB
    shapes = [(1, 64, 15), (1, 192, 16), (2, 448, 17), (16, 512, 33), (3, 576, 1000), (16, 1024, 31), (15, 1088, 48), (16, 1088, 4097), (1, 8192, 40),
              (1, 16384, 70), (2, 8256, 300), (8, 4096, 16), (16, 2048, 4096), (16, 2112, 100), (5, 1984, 16 * units + 1), (7, 3008, 16 * units), (4, 2560, 9999),
              (17, 512, 100), (3, 2048, 12800)]
    if qname:
        shapes += [(2, 70, 20), (3, 65, 33), (5, 129, 640), (16, 1000, 257), (2, 1864, 2663), (4, 1001, 25000), (1, 32705, 64)]
    forms = set()
    for i, (M, K, N) in enumerate(shapes):
        g = torch.Generator(device="cuda").manual_seed(7 * i + 1)
        lin = tp.Linear(K, N, bias=i % 3 != 1, dtype=getattr(tp, dname), quant_dtype=None if qname is None else getattr(tp, qname), weight_quant_dim=0 if qname else None)
        w = (torch.randn((N, K), generator=g, device="cuda") * 0.3).to(td)
        lin.weight = tp.Tensor(w)
        if lin.bias is not None:
            lin.bias = tp.Tensor(torch.randn(N, generator=g, device="cuda").to(td))
        x = torch.randn((M, K), generator=g, device="cuda").to(td)
        wd, xd = w, x
        if qname:
            lin.weight_scale = tp.Tensor((w.float().abs().amax(1) / TOP[qname]).to(td).cpu())
            lin.input_scale = tp.Tensor(torch.tensor(4.0 / TOP[qname]).to(td))
            wd = tp.dequantize(tp.quantize(tp.Tensor(w), lin.weight_scale, lin.quant_dtype, 0), lin.weight_scale, lin.dtype, 0).torch()
            xd = tp.dequantize(tp.quantize(tp.Tensor(x), lin.input_scale, lin.quant_dtype), lin.input_scale, lin.dtype).torch()
        y = lin(tp.Tensor(x)).torch().double()
        padded = (K + 63) // 64 * 64
        # which products take one launch is measured; that its registers and LDS hold their rows is not
        kernel = pkg.last_kernel()
        form = "long" if "_rows16_long" in kernel else "short" if "_rows16" in kernel else "other"
        forms.add(form)
        if form != "other":
            assert kernel == "mtrt_gemm_dense_frag_%s_rows16%s%s" % (SHORT[dname], "_long" if form == "long" else "", "_" + CODE[qname] if qname else ""), (M, K, N)
            assert M <= 16 and M * padded <= (32768 if form == "long" else 16384), (M, K, N)
        b = lin.bias.device_data().double() if lin.bias is not None else torch.zeros(N, dtype=torch.float64, device="cuda")
        ref, mass = xd.double() @ wd.double().T + b, xd.double().abs() @ wd.double().abs().T + b.abs()
        # the products are exact, f32 accumulation in any order, one rounding
        tol = u * ref.abs() + (1 + u) * (K + 2) * 2.0 ** -24 * mass + 2.0 ** -24
        bad = int(((y - ref).abs() <= tol).logical_not().sum())
        assert y.shape == (M, N) and bad == 0, (M, K, N, bad)
    assert forms == {"short", "long", "other"}
