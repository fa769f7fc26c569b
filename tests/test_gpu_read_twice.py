"""Passes over a tensor that another pass has just read: the amax pass takes it in pieces of 32 KiB from its end, the passes behind
it forwards in the same pieces.  Sizes around a piece, around the number of workgroups, around the groups of pieces that are dealt to
the XCDs together, on both sides of the size beyond which they are dealt singly, and where the kernel of the fused pass changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIECE = 32 * 1024                                      # bytes of x


def _x(torch, n, dname):
    g = torch.Generator(device="cuda").manual_seed(n % 1000003)
    return torch.randn(n, generator=g, device="cuda").to(getattr(torch, dname))


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("off", [0, 1])
def test_amax_finds_the_maximum_wherever_it_is(pkg, dname, off):
    import torch
    per = PIECE // (4 if dname == "float32" else 2)
    for n in (1, 7, per // 2 + 3, per - 1, per, per + 1, 9 * per + 5, 511 * per + 9, 512 * per, 513 * per + per // 2 + 1, 1025 * per + 11):
        x = _x(torch, n + off, dname)[off:]            # one element off alignment: a head in front of the first vector
        for at in sorted({0, n // 2, n - 1, max(0, n - 9), min(n - 1, per - 1), min(n - 1, per), n // per * per - 1 if n > per else 0}):
            old = x[at].item()
            x[at] = -1000.0 - at % 7
            amax, scale = pkg.amax(x, 127.0)
            assert amax.item() == float(x[at].abs()) and scale.item() == np.float32(amax.item()) / np.float32(127.0), (n, at)
            x[at] = old


@pytest.mark.parametrize("dname,code", [("float32", "I8"), ("float16", "F8E4M3FN"), ("bfloat16", "F8E4M3FN"), ("bfloat16", "I8")])
def test_from_the_end_is_the_same_as_in_parts(pkg, dname, code):
    """Every element is taken once whatever the order: the codes and values of a tensor are those of its parts, each too short for
    any piece to change its place."""
    import torch
    q_dtype = getattr(pkg, code)
    scale = torch.tensor([0.037], device="cuda")
    block = 4096                                       # elements of a workgroup
    per = 8 // (4 if dname == "float32" else 2) * 8    # workgroups that are turned round together
    for n in (block * (per - 1), block * per, block * per + 8, block * (3 * per + 5) + 24, block * 8 * per + 1):
        x = _x(torch, n, dname)
        q, y = pkg.quantize_dequantize(x, scale, q_dtype)
        only = pkg.quantize(x, scale, q_dtype)
        part = block * 4
        qs, ys = zip(*(pkg.quantize_dequantize(x[i:i + part], scale, q_dtype) for i in range(0, n, part)))
        assert torch.equal(q, torch.cat(qs)) and torch.equal(only, q), n
        assert torch.equal(y.view(torch.uint8), torch.cat(ys).view(torch.uint8)), n


@pytest.mark.parametrize("dname,code", [("float32", "I8"), ("bfloat16", "F8E4M3FN")])
def test_both_sides_of_the_largest_size_that_is_turned_round(pkg, dname, code):
    import torch
    q_dtype, qmax = getattr(pkg, code), {"I8": 127.0, "F8E4M3FN": 448.0}[code]
    size = 4 if dname == "float32" else 2
    for n in ((192 << 20) // size - 4096 * 40, (192 << 20) // size + 4096 * 40):
        x = _x(torch, n, dname)
        x[n - 5] = 50.0
        q, y, amax, scale = pkg.dynamic_quantize_dequantize(x, q_dtype, qmax)
        assert amax.item() == 50.0
        for i in (0, n // 2 // 8 * 8, n - 65536):
            qs, ys = pkg.quantize_dequantize(x[i:i + 65536].clone(), scale.reshape(1), q_dtype)
            assert torch.equal(q[i:i + 65536], qs) and torch.equal(y[i:i + 65536].view(torch.uint8), ys.view(torch.uint8)), (n, i)


@pytest.mark.parametrize("shape", [(32, 256), (240, 1040), (1040, 1264), (2048, 1040)])
@pytest.mark.parametrize("dname", ["float32", "bfloat16"])
def test_nvfp4_from_the_end_is_the_same_as_in_parts(pkg, shape, dname):
    import torch
    x = _x(torch, shape[0] * shape[1], dname).view(shape)
    amax = x.float().abs().max().reshape(())
    for axis in (-1, -2):
        q, s = pkg.nvfp4_quantize(x, amax, axis=axis)
        y = pkg.nvfp4_dequantize(q, s, amax, x.dtype, x.shape, axis=axis)
        parts = [pkg.nvfp4_quantize(x[i:i + 16], amax, axis=axis) for i in range(0, shape[0], 16)]
        assert torch.equal(q.reshape(-1), torch.cat([p[0].reshape(-1) for p in parts])), axis
        assert torch.equal(s.reshape(-1), torch.cat([p[1].reshape(-1) for p in parts])), axis
        ys = [pkg.nvfp4_dequantize(p[0], p[1], amax, x.dtype, (16, shape[1]), axis=axis).reshape(-1) for p in parts]
        assert torch.equal(y.reshape(-1), torch.cat(ys)), axis


@pytest.mark.parametrize("dname,code", [("float32", "I8"), ("float32", "I4"), ("float32", "F8E4M3FN"), ("float16", "I8"), ("float16", "F8E4M3FN"), ("float16", "I4"),
                                        ("bfloat16", "I8"), ("bfloat16", "F8E4M3FN"), ("bfloat16", "I4")])
def test_both_kernels_of_the_fused_pass_are_a_quantize_and_a_dequantize(pkg, dname, code):
    """From 4 to 9 Mi elements (3, to float8) the fused pass has a kernel of its own but for f32 to float8; whole groups or not."""
    import torch
    q_dtype, m = getattr(pkg, code), 1 << 20
    scale = torch.tensor([0.037], device="cuda")
    for n, other in ((3 * m, False), (3 * m + 1, code == "F8E4M3FN"), (4 * m, code == "F8E4M3FN"), (4 * m + 1, True), (4 * m + 4096, True), (5 * m - 3, True), (9 * m - 1, True), (9 * m, False)):
        x = _x(torch, n, dname)
        q, y = pkg.quantize_dequantize(x, scale, q_dtype)
        assert pkg.last_kernel().endswith("s") == (other and (dname, code) != ("float32", "F8E4M3FN")), (n, pkg.last_kernel())
        only = pkg.quantize(x, scale, q_dtype)
        assert torch.equal(only, q), n
        assert torch.equal(pkg.dequantize(only, scale, q_dtype, x.dtype, x.shape).view(torch.uint8), y.view(torch.uint8)), n
