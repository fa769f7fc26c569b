"""Dense products whose rows are no whole 128-byte slices of K, at the row lengths where the last slice holds one element, one less
than a vector, one more and all but one, with rows around the tile heights, columns off whole tiles and operands at any element."""
import pytest

pytestmark = pytest.mark.gpu

EPS = {"float32": 2.0 ** -24, "float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}
# (that these take every form of their kernels: test_dispatch.py)
RAGGED = [(1, 1), (5, 300), (31, 33), (33, 31), (64, 1000), (130, 8209), (300, 1000), (1500, 4100)]
WHOLE = ((32, 33), (64, 8193), (224, 31), (256, 1000), (288, 16385), (512, 8200), (1056, 2049), (4128, 65))


def ragged_lengths(item_bytes):
    slice_, vec = 128 // item_bytes, 16 // item_bytes
    return [1, vec - 1, vec, vec + 1, slice_ - 1, slice_ + 1] + [s * slice_ + e for s, e in ((1, vec), (2, -1), (4, 1), (7, vec + 1), (8, 3), (9, -vec), (17, 1))]


def _inside(torch, t, lead):
    """`t` as a contiguous view that starts `lead` elements into a buffer of NaN and ends as far before its end."""
    buf = torch.full((t.numel() + 2 * lead,), float("nan"), dtype=t.dtype, device=t.device)
    view = buf[lead:lead + t.numel()].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("M,N", RAGGED)
def test_ragged_rows(pkg, M, N, dname):
    import torch
    td = getattr(torch, dname)
    for i, K in enumerate(ragged_lengths(td.itemsize)):
        g = torch.Generator(device="cuda").manual_seed(1000 * M + i)
        x = _inside(torch, torch.randn((M, K), generator=g, device="cuda").to(td), i % 5)
        w = _inside(torch, (torch.randn((N, K), generator=g, device="cuda") * 0.3).to(td), (3 * i) % 7)
        b = torch.randn(N, generator=g, device="cuda").to(td) if i % 2 else None
        out = torch.full((M * N + 128,), 7.0, dtype=td, device="cuda")
        y = pkg.linear_dense(x, w, b, out[64:64 + M * N].view(M, N))
        if dname != "float32" or M > 32 or K * N < 16384:      # few rows of float32: below
            assert pkg.last_kernel() == "mtrt_gemm_dense_edge_" + {"float32": "f32", "float16": "f16", "bfloat16": "bf16"}[dname]
        xd, wd = x.double(), w.double()
        bd = b.double() if b is not None else torch.zeros(N, dtype=torch.float64, device="cuda")
        ref, mass = xd @ wd.T + bd, xd.abs() @ wd.abs().T + bd.abs()
        # f32 sums of K products and the bias in any order, one rounding to the output's type
        tol = EPS[dname] * ref.abs() + (1 + EPS[dname]) * (K + 2) * 2.0 ** -24 * mass + 2.0 ** -24
        bad = int(((y.double() - ref).abs() <= tol).logical_not().sum())
        assert bad == 0, (M, K, N, bad)
        assert bool((out[:64] == 7).all()) and bool((out[64 + M * N:] == 7).all())


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32])
def test_few_rows_of_float32(pkg, M):
    """K around whole steps of 256 and of the four waves that share them, columns around what a wave and a workgroup take, weights
    read through and past the caches."""
    import torch
    kernels = set()
    for i, (K, N) in enumerate(((4, 4099), (5, 8200), (255, 1001), (256, 300), (257, 70), (513, 4097), (772, 8192), (1023, 16), (1280, 1), (1535, 5000),
                                (1536, 33), (1539, 4100), (2048, 2047), (4095, 515), (4097, 66), (3071, 4200), (7681, 129))):
        g = torch.Generator(device="cuda").manual_seed(100 * M + i)
        x = _inside(torch, torch.randn((M, K), generator=g, device="cuda"), i % 4)
        w = _inside(torch, torch.randn((N, K), generator=g, device="cuda") * 0.3, (3 * i) % 7)
        b = torch.randn(N, generator=g, device="cuda") if i % 2 else None
        out = torch.full((M * N + 128,), 7.0, device="cuda")
        y = pkg.linear_dense(x, w, b, out[64:64 + M * N].view(M, N))
        kernels.add(pkg.last_kernel())
        xd, wd = x.double(), w.double()
        bd = b.double() if b is not None else torch.zeros(N, dtype=torch.float64, device="cuda")
        ref, mass = xd @ wd.T + bd, xd.abs() @ wd.abs().T + bd.abs()
        bad = int(((y.double() - ref).abs() <= (K + 2) * 2.0 ** -24 * mass).logical_not().sum())
        assert bad == 0, (M, K, N, bad)
        assert bool((out[:64] == 7).all()) and bool((out[64 + M * N:] == 7).all())
    rows = 1 if M == 1 else 2 if M == 2 else 4 if M <= 4 else 8
    assert "mtrt_gemm_dense_rows%d_f32" % rows in kernels
    assert M not in (5, 8) or "mtrt_gemm_dense_rows8_wide_f32" in kernels
    if M in (1, 8):                                            # (4100 x 3073: 50 MB)
        x, w = torch.randn((M, 3073), device="cuda"), torch.randn((4100, 3073), device="cuda") * 0.3
        ref, mass = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        assert bool(((pkg.linear_dense(x, w).double() - ref).abs() <= 3075 * 2.0 ** -24 * mass).all())


@pytest.mark.parametrize("dname", ["float32", "float16"])
def test_infinities_stay_in_their_row(pkg, dname):
    import torch
    td = getattr(torch, dname)
    for M, K, N in ((40, 70, 50), (9, 1031, 300), (9, 1025, 4100)):
        x, w = torch.ones((M, K), dtype=td, device="cuda"), torch.ones((N, K), dtype=td, device="cuda")
        x[3, K - 1], x[5, 0], w[7, K - 1] = float("inf"), float("nan"), float("-inf")
        y = pkg.linear_dense(x, w).float()
        ref = torch.full((M, N), float(K), dtype=td, device="cuda").float()
        ref[3], ref[:, 7], ref[3, 7], ref[5] = float("inf"), float("-inf"), float("-inf"), float("nan")
        assert torch.equal(torch.nan_to_num(y, nan=-1.0), torch.nan_to_num(ref, nan=-1.0)), (M, K, N)


@pytest.mark.parametrize("M", [9, 32, 33, 64, 65, 128, 129, 257])
def test_whole_slices_of_float32(pkg, M):
    """K in whole 128-byte slices, fewer and more of them than the waves that share them; columns around tiles; products whose
    tiles are fewer and more than the compute units, and whose columns alone are (the form that takes all rows at once)."""
    import torch
    kernels = set()
    for i, (K, N) in enumerate(WHOLE):
        g = torch.Generator(device="cuda").manual_seed(100 * M + i)
        x = torch.randn((M, K), generator=g, device="cuda")
        w = torch.randn((N, K), generator=g, device="cuda") * 0.3
        b = torch.randn(N, generator=g, device="cuda") if i % 2 else None
        out = torch.full((M * N + 128,), 7.0, device="cuda")
        y = pkg.linear_dense(x, w, b, out[64:64 + M * N].view(M, N))
        kernels.add(pkg.last_kernel())
        xd, wd = x.double(), w.double()
        bd = b.double() if b is not None else torch.zeros(N, dtype=torch.float64, device="cuda")
        ref, mass = xd @ wd.T + bd, xd.abs() @ wd.abs().T + bd.abs()
        bad = int(((y.double() - ref).abs() <= (K + 2) * 2.0 ** -24 * mass).logical_not().sum())
        assert bad == 0, (M, K, N, bad)
        assert bool((out[:64] == 7).all()) and bool((out[64 + M * N:] == 7).all())
    if M <= 32:
        assert kernels == {"mtrt_gemm_dense_rows32_f32"}
    elif M <= 128:
        rows = "mtrt_gemm_dense_rows%d" % (64 if M <= 64 else 128)
        assert {rows + "_f32", rows + "_tall_f32"} <= kernels
    else:
        assert kernels == {"mtrt_gemm_dense_rows128_f32", "mtrt_gemm_dense_mfma_f32"}


@pytest.mark.parametrize("M,K,N,kernel", [(1024, 32, 4097, "t128x128"), (129, 96, 30001, "t128x128"), (2001, 160, 3968, "t128x128"), (3970, 1056, 1023, "t128x128"),
                                          (2047, 1664, 3999, "t256x128"), (1793, 2080, 4096, "t256x128"), (3841, 1760, 1921, "t256x128")])
def test_large_tiles_of_float32(pkg, M, K, N, kernel):
    """Products of whole slices that fill the chip with larger tiles: the last tiles of rows and of columns hold one of them, all but one, half; fewer slices
    than parts of their sum, slices that the parts do not divide."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn((M, K), generator=g, device="cuda")
    w = torch.randn((N, K), generator=g, device="cuda") * 0.3
    for bias in (True, False):
        b = torch.randn(N, generator=g, device="cuda") if bias else None
        out = torch.full((M * N + 128,), 7.0, device="cuda")
        y = pkg.linear_dense(x, w, b, out[64:64 + M * N].view(M, N))
        assert pkg.last_kernel() == "mtrt_gemm_dense_%s_f32" % kernel
        ref, mass = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        if bias:
            ref, mass = ref + b.double(), mass + b.double().abs()
        bad = int(((y.double() - ref).abs() <= (K + 2) * 2.0 ** -24 * mass).logical_not().sum())
        assert bad == 0, bad
        assert bool((out[:64] == 7).all()) and bool((out[64 + M * N:] == 7).all())
        # the error of all sums together, in 2^-24 of the result: a chain of n random terms errs by 0.29 sqrt(n) (measured, K = 4096: 19), four
        # chains of n / 4 by half of that; the rounding of a result by 0.3 to 0.6
        chain = (K + 127) // 128 * 32
        assert float((y.double() - ref).norm() / ref.norm()) < 2.0 ** -24 * (0.6 + 0.36 * chain ** 0.5)
