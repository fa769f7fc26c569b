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
