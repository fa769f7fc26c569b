"""Rows held by a workgroup (and, LayerNorm, by a wave) whose last vectors end inside, at and just past a wave's share, so that whole
waves have none of some step's vectors: softmax and LayerNorm against float64, with infinities in the row."""
import pytest

pytestmark = pytest.mark.gpu

EPS = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


def _lengths(e):
    vecs = [65, 129, 1025, 1088, 1089, 1279, 1281, 2047, 2049, 2112, 2305, 3000, 4095, 4097, 4160, 5120, 5121, 8191, 8193, 9217, 9280, 16383]
    return [v * e for v in vecs] + [v * e + e - 1 for v in vecs]


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
def test_softmax(pkg, dname):
    import torch
    td = getattr(torch, dname)
    for d in _lengths(16 // td.itemsize):
        g = torch.Generator(device="cuda").manual_seed(d)
        x = (torch.randn((7, d), generator=g, device="cuda") * 2).to(td)
        x[1, -1], x[2, d // 2:] = 60.0, float("-inf")
        x[3, :-1] = float("-inf")
        x[4], x[5, 3], x[6, 0] = float("-inf"), float("nan"), float("inf")
        y = pkg.softmax(x).double()
        ref = torch.softmax(x[:4].double(), dim=-1)
        # the f32 exponential's argument (up to 80 off by half an ulp), the instruction, the sum's additions, the product and the narrowing
        tol = ref * (EPS[dname] + (80 + 16 + 32) * 2.0 ** -24) + (2.0 ** -25 if dname == "float16" else 2.0 ** -126)
        assert bool(((y[:4] - ref).abs() <= tol).all()), (d, pkg.last_kernel())
        assert bool(torch.isnan(y[4:]).all()), d                  # as the reference operations give: -inf + inf, a NaN, inf - inf in the sum


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
def test_layernorm(pkg, dname):
    import torch
    td = getattr(torch, dname)
    for d in _lengths(16 // td.itemsize):
        g = torch.Generator(device="cuda").manual_seed(d)
        x = torch.randn((5, d), generator=g, device="cuda").to(td)
        x[1, -1] = 30.0
        gamma, beta = (torch.rand(d, generator=g, device="cuda") + 0.5).to(td), torch.randn(d, generator=g, device="cuda").to(td)
        y = pkg.layernorm(x, gamma, beta, 1e-5).double()
        xd = x.double()
        dev = xd - xd.mean(-1, keepdim=True)
        ref = dev / torch.sqrt((dev * dev).mean(-1, keepdim=True) + 1e-5) * gamma.double() + beta.double()
        # tree sums of up to 64 steps in f32, then six roundings, in units of the largest term
        tol = EPS[dname] * ref.abs() + (64 + 6) * 2.0 ** -24 * ((ref - beta.double()).abs() + beta.double().abs() + 1.0)
        assert bool(((y - ref).abs() <= tol).all()), (d, pkg.last_kernel())


@pytest.mark.parametrize("dname,op,forms", [
    ("float16", "layernorm", "g256v8e g256v16e u64v4e u64v8e u64v16e u256v8e u256v16e g1024v8a g1024v16a"), ("bfloat16", "layernorm", "g256v8e g256v16e u64v4e u64v8e u64v16e u256v8e u256v16e g1024v8a g1024v16a"),
    ("float32", "layernorm", "g256v8e g1024v8a"), ("float16", "softmax", "g256v8e g256v16e u256v8e u256v16e g1024v8a g1024v16a"),
    ("bfloat16", "softmax", "g256v8e g256v16e u256v8e u256v16e g1024v8a g1024v16a"), ("float32", "softmax", "g1024v8a g1024v16a u1024v8a u1024v16a")])
def test_both_forms_of_a_kernel_give_the_same_bits(pkg, dname, op, forms):
    """How many rows there are, and how much of its vectors a row fills, chooses the form; a row's bits depend on neither."""
    import torch
    td = getattr(torch, dname)
    bits = torch.int32 if dname == "float32" else torch.int16
    e, seen = 16 // td.itemsize, set()
    for vecs in (140, 200, 300, 500, 600, 1000, 1100, 1500, 1900, 2048, 2200, 3000, 3900, 4095, 4300, 6000, 8100, 8400, 12000, 16000, 16384):
        for tail in (0, e - 1):
            d = vecs * e + tail
            if vecs < 1025 and not tail or vecs in (2048, 16384) and tail:
                continue
            g = torch.Generator(device="cuda").manual_seed(d)
            x = torch.randn((7, d), generator=g, device="cuda").to(td)
            x[1, -1] = 30.0
            if op == "softmax":
                x[2, d // 2:] = float("-inf")
                call = pkg.softmax
            else:
                gamma, beta = (torch.rand(d, generator=g, device="cuda") + 0.5).to(td), torch.randn(d, generator=g, device="cuda").to(td)
                call = lambda t: pkg.layernorm(t, gamma, beta, 1e-5)
            ref = call(x)
            seen.add(pkg.last_kernel().rsplit("_", 1)[1])
            for rows in (8, 300, 700, 1100, 1400, 1600):
                if vecs > 4096 and rows > 300:
                    continue
                out = call(x.repeat((rows + 6) // 7, 1)[:rows].contiguous())
                seen.add(pkg.last_kernel().rsplit("_", 1)[1])
                want = ref.repeat((rows + 6) // 7, 1)[:rows]
                assert torch.equal(out.view(bits), want.view(bits)), (d, rows, pkg.last_kernel())
    assert set(forms.split()) <= seen, seen
