"""Reductions over the lanes of a wave and of its groups of 2 to 32: one element of a row counts for everything, in every place of the row, so that
each lane's value has to arrive, once."""
import pytest

pytestmark = pytest.mark.gpu

EPS = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("vectors", [8, 16, 32, 64, 128, 256, 65, 256 * 4])
def test_rows(pkg, dname, vectors):
    """Groups of 8, 16 and 32 lanes, a wave with one, two and four vectors a lane, with ragged ends, and several waves to a row."""
    import torch
    td = getattr(torch, dname)
    e = 16 // td.itemsize
    d = vectors * e + (3 if vectors == 65 else 0)
    at = torch.arange(0, d, e, device="cuda")
    rows = torch.arange(at.numel(), device="cuda")
    x = torch.full((at.numel(), d), -120.0, dtype=td, device="cuda")
    x[rows, at] = 0.0                                          # exp(-120) is no f32: the place alone has probability 1
    one_hot = torch.zeros(x.shape, dtype=td, device="cuda")
    one_hot[rows, at] = 1.0
    assert torch.equal(pkg.softmax(x), one_hot), pkg.last_kernel()
    even = pkg.softmax(torch.zeros_like(x)).double()
    assert bool(((even * d - 1).abs() <= EPS[dname] + 16 * 2.0 ** -24).all())
    y = pkg.layernorm(one_hot, torch.ones(d, dtype=td, device="cuda"), torch.zeros(d, dtype=td, device="cuda"), 1e-5).double()
    ref = torch.nn.functional.layer_norm(one_hot.double(), (d,), eps=1e-5)
    assert bool(((y - ref).abs() <= ref.abs() * (EPS[dname] + 2e-5) + 2.0 ** -25).all()), pkg.last_kernel()


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
def test_amax(pkg, dname):
    import torch
    td = getattr(torch, dname)
    e = 16 // td.itemsize
    x = torch.zeros((64, 64 * e), dtype=td, device="cuda")
    at = torch.arange(64, device="cuda") * e
    x[torch.arange(64, device="cuda"), at] = -torch.arange(1, 65, device="cuda").to(td)
    want = torch.arange(1, 65, device="cuda", dtype=torch.float32)
    for r in range(64):
        amax, scale = pkg.amax(x[r].contiguous(), 127.0)
        assert float(amax) == r + 1, (r, pkg.last_kernel())
        _, _, amax, _ = pkg.dynamic_quantize_dequantize(x[r].contiguous(), pkg.I8, 127.0)
        assert float(amax) == r + 1, (r, pkg.last_kernel())
    got = pkg.dynamic_quantize_rows(x, pkg.I8, 127.0)
    assert any(isinstance(t, torch.Tensor) and t.dtype == torch.float32 and t.numel() == 64 and torch.equal(t.flatten(), want) for t in got), pkg.last_kernel()


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
def test_nvfp4_blocks(pkg, dname):
    """The largest of a block of 16 in each of its places: its scale is as if it stood first, the code 6 (7) moves with it."""
    import torch
    td = getattr(torch, dname)
    n = 16 * 64
    x = torch.zeros((16, n), dtype=td, device="cuda")
    for r in range(16):
        x[r, r::16] = 1.5 * (1 + torch.arange(64, device="cuda") % 7).to(td)
    q, s = pkg.nvfp4_quantize(x, torch.full((), 10.5, device="cuda"))
    q, s = q.view(torch.uint8).reshape(16, 64, 8), s.view(torch.uint8).reshape(16, 64)
    assert bool((s == s[0]).all()) and s[0].unique().numel() == 7
    for r in range(16):
        want = torch.zeros(8, dtype=torch.uint8, device="cuda")
        want[r // 2] = 7 << 4 * (r % 2)
        assert bool((q[r] == want).all()), r
