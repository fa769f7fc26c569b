"""Softmax kernels of two long 16-bit rows to a compute unit: the bits of the kernels that few rows take, rows just above a form's vectors, at the line between the
forms and full, whole vectors and ragged, x and y off the same 16-byte boundary, read past the caches and through them; and float64."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dname", ["float16", "bfloat16"])
@pytest.mark.parametrize("d", [32776, 32769 + 8, 40000, 43165, 52424, 52432, 60001, 65528, 65535, 65536])
def test_the_bits_of_few_rows(pkg, dname, d):
    import torch
    td, code = getattr(torch, dname), {"float16": pkg.F16, "bfloat16": pkg.BF16}[dname]
    units = torch.cuda.get_device_properties(0).multi_processor_count
    g = torch.Generator(device="cuda").manual_seed(d)
    for rows, off in ((units + 1, 0), (units + 44, 3), (5 * units // 2, 0)):
        x = (torch.randn(off + rows * d, generator=g, device="cuda") * 2).to(td)
        x[off + d:off + d + d // 2] = float("-inf")
        y = torch.full((off + rows * d + 64,), 7.0, dtype=td, device="cuda")
        pkg.check(pkg.lib().mtrt_hip_softmax(None, x[off:].data_ptr(), y[off:].data_ptr(), code, rows, d))
        name = pkg.last_kernel()
        assert ("1024v8ra" if d % 8 == 0 and not off and d > 52428 else "1024v8r") in name, name
        few = torch.empty_like(y)
        for r0 in range(0, rows, 100):
            n, at = min(100, rows - r0), off + r0 * d
            pkg.check(pkg.lib().mtrt_hip_softmax(None, x[at:].data_ptr(), few[at:].data_ptr(), code, n, d))
            assert "1024v8r" not in pkg.last_kernel()
        torch.cuda.synchronize()
        assert torch.equal(y[off:off + rows * d].view(torch.int16), few[off:off + rows * d].view(torch.int16)), (rows, off, name)
        assert bool((y[:off] == 7.0).all()) and bool((y[off + rows * d:] == 7.0).all())
        for r in (0, 1, rows - 1):
            ref = torch.softmax(x[off + r * d:off + (r + 1) * d].double(), -1)
            u = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[dname]
            # the exponential's argument (up to 40 off by half an ulp), the instruction, the sum's additions, the product and the narrowing
            tol = ref * (u + (40 + 16 + 96) * 2.0 ** -24) + (2.0 ** -25 if dname == "float16" else 2.0 ** -126)
            assert bool(((y[off + r * d:off + (r + 1) * d].double() - ref).abs() <= tol).all()), (rows, off, r, name)
