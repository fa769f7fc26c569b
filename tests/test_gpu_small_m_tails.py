"""The small-M GEMM kernels at K ranges that leave their waves every number of slices modulo the pipeline's depth, at the row counts
where they change the form of their activation loads, and at tile counts around one, two and three per workgroup."""
import pytest

pytestmark = pytest.mark.gpu


def _w4(torch, pkg, M, K, N, block, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randint(-8, 8, (K, N), generator=g, device="cuda")
    flat = (w & 15).to(torch.uint8).reshape(-1)
    if flat.numel() % 2:
        flat = torch.cat([flat, flat.new_zeros(1)])
    packed = (flat[0::2] | (flat[1::2] << 4)).contiguous()
    a = torch.randn((M, K), generator=g, device="cuda").half()
    scale = (torch.rand((K // block, N), generator=g, device="cuda") * 0.015 + 0.005).half()
    y = pkg.gemm_w4a16(a, scale, K, N, block, w_prepacked=pkg.gemm_w4a16_prepack(packed, K, N))
    wd = (w.float() * scale.float().repeat_interleave(block, 0)).half().double()     # exact product, one rounding
    ref, mass = a.double() @ wd, a.double().abs() @ wd.abs()
    # f32 sums in any order, one rounding to f16
    tol = 2.0 ** -11 * ref.abs() + (1 + 2.0 ** -11) * (K + 2) * 2.0 ** -24 * mass + 2.0 ** -24
    bad = int(((y.double() - ref).abs() > tol).sum())
    assert bad == 0, (M, K, N, block, bad)


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
def test_w4a16_strips(pkg, M, block):
    import torch
    for i, slices in enumerate((2, 4, 5, 6, 7, 8, 11, 13, 18, 28)):
        K, N = slices * 256, (16, 40, 300, 1000, 4096, 4100, 8209)[i % 7]
        _w4(torch, pkg, M, K, N, block, 100 * M + i)
        expect = "mtrt_gemm_w4a16_strips16" + ("_b64" if block == 64 else "")
        assert pkg.last_kernel() == expect, (K, N)
    _w4(torch, pkg, M, 1536, 16 * 769, block, M)         # more than three tiles to each of 256 compute units


@pytest.mark.parametrize("M", [1, 9, 16, 17, 25, 32])
def test_w4a16_skinny(pkg, M):
    import torch
    for i, slices in enumerate((1, 2, 3, 4, 5, 6, 7, 9, 13, 17, 22, 31)):
        # (17 to 32 rows by few columns take the strips where K is a multiple of 128)
        K, N = slices * 64, (16, 40, 300, 1000, 8224)[i % 5] if M <= 16 or slices % 2 else 8224
        _w4(torch, pkg, M, K, N, 64, 100 * M + i)
        if M > 16 or K < 512 or K % 128:
            assert pkg.last_kernel().startswith("mtrt_gemm_w4a16_skinny"), (K, N)


@pytest.mark.parametrize("M", [1, 8, 9, 16])
def test_w8a8_small(pkg, M):
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    for i, slices in enumerate((1, 2, 3, 4, 5, 6, 7, 9, 12, 13, 15, 18, 23)):
        K, N = slices * 128, (4128, 5000, 8200)[i % 3]   # more than half as many 32-column tiles as compute units
        a = torch.randint(-128, 128, (M, K), generator=g, device="cuda", dtype=torch.int8)
        w = torch.randint(-128, 128, (K, N), generator=g, device="cuda", dtype=torch.int8)
        sa, sw = torch.rand(M, generator=g, device="cuda") * 0.01, torch.rand(N, generator=g, device="cuda") * 0.001
        y = pkg.gemm_w8a8_fragments(a, pkg.gemm_w8a8_prepack_fragments(w), sa, sw, N)
        assert pkg.last_kernel() == "mtrt_gemm_w8a8_small16"
        acc = (a.double() @ w.double()).float()          # exact: below 2^53, and 2^24 here
        assert torch.equal(y, ((acc * sa[:, None]) * sw[None, :]).half()), (M, K, N)


@pytest.mark.parametrize("M", [1, 8, 9, 16])
def test_w8a8_small_of_few_columns(pkg, M):
    """32-column tiles for half of the compute units, down to one, and one more; weights on both sides of the lines between loads past the caches and
    through them."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    for K, N in ((128, 1), (256, 32), (640, 33), (1152, 300), (2560, 1281), (2688, 4096), (2688, 4097), (4096, 2047), (4096, 2048), (16384, 4096), (16512, 4095)):
        a = torch.randint(-128, 128, (M, K), generator=g, device="cuda", dtype=torch.int8)
        w = torch.randint(-128, 128, (K, N), generator=g, device="cuda", dtype=torch.int8)
        sa, sw = torch.rand(M, generator=g, device="cuda") * 0.01, torch.rand(N, generator=g, device="cuda") * 0.001
        y = pkg.gemm_w8a8_fragments(a, pkg.gemm_w8a8_prepack_fragments(w), sa, sw, N)
        assert pkg.last_kernel() == "mtrt_gemm_w8a8_small16"
        acc = (a.double() @ w.double()).to(torch.int64).float()   # exact sums, one rounding to f32
        assert torch.equal(y, ((acc * sa[:, None]) * sw[None, :]).half()), (M, K, N)


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("M", [17, 20, 21, 24, 25, 32, 33, 63, 64, 65, 100, 256, 497, 512])
def test_w4a16_strips_in_groups_of_rows(pkg, M, block):
    """A last group of every form, one, two and three tiles to a workgroup, ragged last tiles, waves with every number of slices modulo four."""
    import torch
    units, groups = 256, (M + 15) // 16
    for i, (K, tiles) in enumerate(((2048, 1), (2048, units // groups), (2560, units // groups + 1), (2304, 2 * (units // groups)), (2560, 3 * (units // groups)))):
        N = 16 * tiles - (0, 7, 15, 0, 1)[i]
        if N > 0:
            _w4(torch, pkg, M, K, N, block, 10 * M + i)
            if torch.cuda.get_device_properties(0).multi_processor_count == units and (M > 32 or i < 4):
                assert pkg.last_kernel() == "mtrt_gemm_w4a16_strips16" + ("_b64" if block == 64 else ""), (K, N)


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("M", [17, 31, 33, 64, 100, 512])
def test_w4a16_strips_of_few_slices(pkg, M, block):
    """Fewer slices of 128 k than waves, as many, and one more; one, two and three tiles to a workgroup from where the rule takes them."""
    import torch
    groups = (M + 15) // 16
    for i, (K, each) in enumerate(((128, 1), (256, 1), (384, 1), (512, 1), (640, 1), (1024, 1), (256, 2), (512, 2), (1024, 2), (512, 3), (896, 3))):
        if M <= 32 and (each == 3 or (each == 2 and K < 1024)):
            continue
        N = 16 * ((256 // groups) * (each - 1) + 1) - (0, 9)[i % 2]
        _w4(torch, pkg, M, K, N, block, 10 * M + i)
        if torch.cuda.get_device_properties(0).multi_processor_count == 256:
            assert pkg.last_kernel() == "mtrt_gemm_w4a16_strips16" + ("_b64" if block == 64 else ""), (K, N)


@pytest.mark.parametrize("M,K,N,block", [(4, 4096, 5120, 128), (4, 4096, 5121, 64), (1, 4096, 5137, 128), (8, 4096, 24577, 128), (16, 4096, 24576, 64),
                                         (16, 4096, 24609, 128), (25, 4096, 24576, 64), (25, 4096, 24577, 64), (9, 4160, 24577, 64)])
def test_w4a16_weights_of_10_and_48_mib(pkg, M, K, N, block):
    """The kernels that read the weights once, on more of them than the tests above, ragged last tiles among them."""
    import torch
    _w4(torch, pkg, M, K, N, block, M)
    assert pkg.last_kernel().startswith("mtrt_gemm_w4a16_strips16" if M <= 16 and K % 128 == 0 else "mtrt_gemm_w4a16_skinny")


@pytest.mark.parametrize("M,N", [(1, 12288), (9, 12288), (9, 12289), (16, 12353)])
def test_w8a8_weights_of_48_mib(pkg, M, N):
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    K = 4096
    a = torch.randint(-128, 128, (M, K), generator=g, device="cuda", dtype=torch.int8)
    w = torch.randint(-128, 128, (K, N), generator=g, device="cuda", dtype=torch.int8)
    sa, sw = torch.rand(M, generator=g, device="cuda") * 0.01, torch.rand(N, generator=g, device="cuda") * 0.001
    y = pkg.gemm_w8a8_fragments(a, pkg.gemm_w8a8_prepack_fragments(w), sa, sw, N)
    acc = (a.double() @ w.double()).to(torch.int64).float()       # exact sums, one rounding to f32
    assert torch.equal(y, ((acc * sa[:, None]) * sw[None, :]).half())


@pytest.mark.parametrize("M", [17, 24, 25, 32])
def test_w8a8_up_to_32_rows(pkg, M):
    """Waves with no slice and every number of slices modulo four, at tiles below and above a workgroup to a unit, one workgroup to two tiles
    and to one on both sides of its lines, more than two tiles to a unit, and weights on both sides of the lines between loads past the caches and through them."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    shapes = [(128 * s, (40, 4100, 8200, 11008, 16390)[i % 5]) for i, s in enumerate((1, 2, 3, 4, 5, 6, 7, 9, 12, 13, 15, 16, 18, 23))]
    shapes += [(4096, 2047), (4096, 2048), (3968, 4097), (4096, 4097), (4096, 16384), (4096, 16385), (2048, 10240), (2048, 10273), (4096, 12288), (4096, 12289), (8192, 16384), (8192, 16385), (4096, 24576), (4096, 24577)]
    for K, N in shapes:
        a = torch.randint(-128, 128, (M, K), generator=g, device="cuda", dtype=torch.int8)
        w = torch.randint(-128, 128, (K, N), generator=g, device="cuda", dtype=torch.int8)
        sa, sw = torch.rand(M, generator=g, device="cuda") * 0.01, torch.rand(N, generator=g, device="cuda") * 0.001
        y = pkg.gemm_w8a8_fragments(a, pkg.gemm_w8a8_prepack_fragments(w), sa, sw, N)
        assert pkg.last_kernel() == "mtrt_gemm_w8a8_frag_rows32"
        acc = (a.double() @ w.double()).to(torch.int64).float()   # exact sums, one rounding to f32
        assert torch.equal(y, ((acc * sa[:, None]) * sw[None, :]).half()), (M, K, N)
