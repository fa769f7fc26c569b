"""Dense products whose rows are no whole 128-byte slices of K, at the row lengths where the last slice holds one element, one less
than a vector, one more and all but one, with rows around the tile heights, columns off whole tiles and operands at any element."""
import pytest

pytestmark = pytest.mark.gpu

EPS = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}


def _inside(torch, t, lead):
    """`t` as a contiguous view that starts `lead` elements into a buffer of NaN and ends as far before its end."""
    buf = torch.full((t.numel() + 2 * lead,), float("nan"), dtype=t.dtype, device=t.device)
    view = buf[lead:lead + t.numel()].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("M,N", [(1, 1), (5, 300), (31, 33), (33, 31), (64, 1000), (130, 8209), (300, 1000), (1500, 4100)])
def test_ragged_rows(pkg, M, N, dname):
    import torch
    td = getattr(torch, dname)
    slice_, vec = 128 // td.itemsize, 16 // td.itemsize
    lengths = [1, vec - 1, vec, vec + 1, slice_ - 1, slice_ + 1] + [s * slice_ + e for s, e in ((1, vec), (2, -1), (4, 1), (7, vec + 1), (8, 3), (9, -vec), (17, 1))]
    for i, K in enumerate(lengths):
        g = torch.Generator(device="cuda").manual_seed(1000 * M + i)
        x = _inside(torch, torch.randn((M, K), generator=g, device="cuda").to(td), i % 5)
        w = _inside(torch, (torch.randn((N, K), generator=g, device="cuda") * 0.3).to(td), (3 * i) % 7)
        b = torch.randn(N, generator=g, device="cuda").to(td) if i % 2 else None
        out = torch.full((M * N + 128,), 7.0, dtype=td, device="cuda")
        y = pkg.linear_dense(x, w, b, out[64:64 + M * N].view(M, N))
        assert pkg.last_kernel() == "mtrt_gemm_dense_edge_" + {"float32": "f32", "float16": "f16", "bfloat16": "bf16"}[dname]
        xd, wd = x.double(), w.double()
        bd = b.double() if b is not None else torch.zeros(N, dtype=torch.float64, device="cuda")
        ref, mass = xd @ wd.T + bd, xd.abs() @ wd.abs().T + bd.abs()
        # f32 sums of K products and the bias in any order, one rounding to the output's type
        tol = EPS[dname] * ref.abs() + (1 + EPS[dname]) * (K + 2) * 2.0 ** -24 * mass + 2.0 ** -24
        bad = int(((y.double() - ref).abs() <= tol).logical_not().sum())
        assert bad == 0, (M, K, N, bad)
        assert bool((out[:64] == 7).all()) and bool((out[64 + M * N:] == 7).all())


@pytest.mark.parametrize("dname", ["float32", "float16"])
def test_infinities_stay_in_their_row(pkg, dname):
    import torch
    td = getattr(torch, dname)
    for M, K, N in ((40, 70, 50), (9, 1031, 300)):
        x, w = torch.ones((M, K), dtype=td, device="cuda"), torch.ones((N, K), dtype=td, device="cuda")
        x[3, K - 1], x[5, 0], w[7, K - 1] = float("inf"), float("nan"), float("-inf")
        y = pkg.linear_dense(x, w).float()
        ref = torch.full((M, N), float(K), dtype=td, device="cuda").float()
        ref[3], ref[:, 7], ref[3, 7], ref[5] = float("inf"), float("-inf"), float("-inf"), float("nan")
        assert torch.equal(torch.nan_to_num(y, nan=-1.0), torch.nan_to_num(ref, nan=-1.0)), (M, K, N)
