"""Dynamic per-tensor quantization of small tensors, whose workgroups take the maximum of all by themselves or meet the others, and around each
number of vectors that a lane holds: against amax and the fused pass as two calls, bit for bit, with the maximum in any workgroup and in place;
and amax where groups of its arrival tree have one member."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("code", ["I8", "F8E4M3FN"])
def test_small_tensors(pkg, dname, code):
    import torch
    td, code = getattr(torch, dname), getattr(pkg, code)
    group, qmax = 16 // td.itemsize, 127.0 if code == pkg.I8 else 448.0
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for nvec in (1, 1023, 1025, 4095, 4096, 4097, 8191, 8192, 8193, 12289):
        n = nvec * group
        for at in (0, n // 2, n - 1):
            x = torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(nvec), device="cuda").to(td)
            x[at] = -40.0
            amax, scale = pkg.amax(x, qmax)
            q, y = pkg.quantize_dequantize(x, scale.reshape(1), code)
            for _ in range(2):
                gq, gy, gamax, gscale = pkg.dynamic_quantize_dequantize(x, code, qmax)
                assert "mtrt_dynqdq_" in pkg.last_kernel()
                assert float(gamax) == float(amax) == 40.0 and float(gscale) == float(scale)
                assert torch.equal(gq.view(torch.uint8), q.view(torch.uint8)) and torch.equal(gy, y)
            z, q2, sc = x.clone(), torch.empty(n, dtype=torch.uint8, device="cuda"), torch.empty(1, device="cuda")
            rc = pkg.lib().mtrt_hip_dynamic_quantize_dequantize(st, z.data_ptr(), {"float32": pkg.F32, "float16": pkg.F16, "bfloat16": pkg.BF16}[dname],
                                                                q2.data_ptr(), code, z.data_ptr(), n, qmax, None, sc.data_ptr(), 0)
            assert rc == 0 and torch.equal(z, y) and torch.equal(q2, q.view(torch.uint8).flatten())


@pytest.mark.parametrize("dname,code", [("float32", "I8"), ("bfloat16", "I8"), ("float16", "F8E4M3FN")])
def test_tensors_around_each_number_of_vectors_a_lane(pkg, dname, code):
    """One to five vectors a lane on 256 compute units: the last tensor of each number, the first of the next, the maximum in the first and
    in the last vector."""
    import torch
    td, code = getattr(torch, dname), getattr(pkg, code)
    group, qmax = 16 // td.itemsize, 127.0 if code == pkg.I8 else 448.0
    for nvec in (131072, 131073, 393216, 393217, 589824, 589825, 1048576, 1048577, 1310720, 1310721):
        x = torch.randn(nvec * group, generator=torch.Generator(device="cuda").manual_seed(nvec), device="cuda").to(td)
        for at, most in ((0, 40.0), (-1, 41.0)):
            x[at] = -most
            amax, scale = pkg.amax(x, qmax)
            q, y = pkg.quantize_dequantize(x, scale.reshape(1), code)
            gq, gy, gamax, gscale = pkg.dynamic_quantize_dequantize(x, code, qmax)
            assert float(gamax) == float(amax) == most and float(gscale) == float(scale)
            assert torch.equal(gq.view(torch.uint8), q.view(torch.uint8)) and torch.equal(gy, y)
            only, none, _, _ = pkg.dynamic_quantize_dequantize(x, code, qmax, dequantize=False)
            assert none is None and torch.equal(only.view(torch.uint8), gq.view(torch.uint8))


@pytest.mark.parametrize("dname", ["float32", "bfloat16"])
def test_amax_of_few_workgroups(pkg, dname):
    import torch
    td = getattr(torch, dname)
    piece = 32768 // td.itemsize                               # what a workgroup takes
    for groups in (1, 2, 31, 32, 33, 63, 64, 65, 97):
        n = groups * piece - 5
        x = torch.rand(n, device="cuda").to(td)
        for turn, at in enumerate((0, n - 1, n // 2, (groups // 2) * piece, n - 7)):
            x[at] = -3.0 - turn
            amax, scale = pkg.amax(x, 2.0)
            assert float(amax) == 3.0 + turn and float(scale) == (3.0 + turn) / 2
