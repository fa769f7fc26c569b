"""Softmax rows cut at cache lines: every place of a row in a line, x and y off the same and off different 16-byte boundaries, rows that fill their lanes (no
room for a shift) and rows just past a kernel's vectors, against float64; nothing is written around the rows, and equal rows give equal bits wherever they lie."""
import pytest

pytestmark = pytest.mark.gpu

EPS = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
def test_softmax_rows_at_every_place_in_a_line(pkg, dname):
    import torch
    td = getattr(torch, dname)
    e = 16 // td.itemsize
    # (vectors, elements beyond): three, four, eight and sixteen vectors a lane, a wave's and a workgroup's, half full to full
    lengths = [v * e + t for v in (130, 187, 248, 249, 255, 256, 505, 512, 700, 1023, 1024, 1125, 2041, 2048, 4090, 5395, 8192) for t in (0, 1, e - 1)]
    for d in lengths:
        rows = 128 // td.itemsize + 1                                # neighbouring rows start at every place that a row of this length can have
        g = torch.Generator(device="cuda").manual_seed(d)
        one = (torch.randn(d, generator=g, device="cuda") * 2).to(td)
        one[d // 3] = float("-inf")
        ref = torch.softmax(one.double(), dim=-1)
        # the exponential's argument (up to 80 off by half an ulp), the instruction, the sum's narrowing and additions, the product and the narrowing
        tol = ref * (EPS[dname] + (80 + 16 + 32) * 2.0 ** -24) + (2.0 ** -25 if dname == "float16" else 2.0 ** -126)
        bits = torch.int32 if dname == "float32" else torch.int16
        for xo, yo in ((0, 0), (3, 3), (1, 2), (5, 5 + 64)):         # elements in front of x and y
            x, y = torch.zeros(xo + rows * d, dtype=td, device="cuda"), torch.full((yo + rows * d + 64,), 7.0, dtype=td, device="cuda")
            x[xo:] = one.repeat(rows)
            pkg.check(pkg.lib().mtrt_hip_softmax(0, x[xo:].data_ptr(), y[yo:].data_ptr(), {"float32": pkg.F32, "float16": pkg.F16, "bfloat16": pkg.BF16}[dname], rows, d))
            torch.cuda.synchronize()
            got = y[yo:yo + rows * d].view(rows, d)
            case = (d, xo, yo, pkg.last_kernel())
            assert bool(((got[0].double() - ref).abs() <= tol).all()), case
            assert torch.equal(got.view(bits), got[:1].view(bits).expand(rows, d)), case
            assert bool((y[:yo] == 7.0).all()) and bool((y[yo + rows * d:] == 7.0).all()), case


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
def test_cut_and_uncut_rows_of_whole_vectors_have_the_same_bits(pkg, dname):
    """Tensors on either side of the line, also rows of whole lines that start off one; x off a line, y on one and off it."""
    import torch
    td, code = getattr(torch, dname), {"float32": pkg.F32, "float16": pkg.F16, "bfloat16": pkg.BF16}[dname]
    e = 16 // td.itemsize
    for nvec in (33, 63, 64, 65, 121, 128, 187, 250, 256, 313, 505, 512, 600, 1017, 1023, 1024):
        d = nvec * e
        rows = -(-(14 << 20) // (16 * nvec))
        g = torch.Generator(device="cuda").manual_seed(nvec)
        for xo, yo in ((0, 0), (3 * e, 3 * e), (e, 0), (0, 5 * e)):
            x, y = (torch.randn(xo + rows * d, generator=g, device="cuda") * 2).to(td), torch.full((yo + rows * d + 64,), 7.0, dtype=td, device="cuda")
            x[xo + d:xo + d + d // 2] = float("-inf")
            pkg.check(pkg.lib().mtrt_hip_softmax(None, x[xo:].data_ptr(), y[yo:].data_ptr(), code, rows, d))
            name = pkg.last_kernel()
            assert name.endswith("c") == (nvec % 8 != 0 or xo != 0), (name, nvec, xo)
            few = torch.empty_like(y)
            for r0 in range(0, rows, rows // 2):
                n = min(rows // 2, rows - r0)
                pkg.check(pkg.lib().mtrt_hip_softmax(None, x[xo + r0 * d:].data_ptr(), few[yo + r0 * d:].data_ptr(), code, n, d))
                assert not pkg.last_kernel().endswith("c")
            torch.cuda.synchronize()
            bits = torch.int32 if td.itemsize == 4 else torch.int16
            assert torch.equal(y[yo:yo + rows * d].view(bits), few[yo:yo + rows * d].view(bits)), (nvec, xo, yo, name)
            assert bool((y[:yo] == 7.0).all()) and bool((y[yo + rows * d:] == 7.0).all())
            for r in (0, 1, rows - 1):
                row = x[xo + r * d:xo + (r + 1) * d].double()
                ref = torch.softmax(row, -1)
                tol = ref * (EPS[dname] + (40 + 16 + 32) * 2.0 ** -24) + (2.0 ** -25 if dname == "float16" else 2.0 ** -126)
                assert bool(((y[yo + r * d:yo + (r + 1) * d].double() - ref).abs() <= tol).all()), (nvec, r, name)
