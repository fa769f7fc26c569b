"""float32 Linears whose 32 x 32 tiles have their K shared by workgroups: every number of parts (test_linear_split_f32_plan.py has them on the CPU), rows and columns at
the ends of tiles, rows that are whole slices and rows that are not, against float64; the same bits from call to call, with the tickets back at zero, on two
streams and in a replayed graph; and beside the entry point that does not share."""
import ctypes
import importlib
import math

import pytest

from test_gpu_linear_codes import Plan

pytestmark = pytest.mark.gpu

# (M, K, N, parts)
SHAPES = [(33, 1024, 97, 4), (128, 1056, 512, 4), (300, 1536, 256, 3), (65, 3072, 95, 8), (64, 2048, 97, 8), (109, 3072, 448, 4), (257, 4096, 300, 2), (200, 2048, 180, 6), (33, 8192, 1024, 4), (231, 10496, 1318, 3),
          (34, 1025, 97, 4), (66, 4099, 65, 8), (150, 5449, 515, 3), (40, 2047, 300, 8)]


@pytest.fixture(scope="module")
def tp(pkg):
    return importlib.import_module(pkg.__name__ + ".tp")


@pytest.mark.parametrize("M,K,N,parts", SHAPES)
def test_parts_against_float64(tp, pkg, M, K, N, parts):
    import torch
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    w, b = torch.randn((N, K), generator=g, device="cuda") / math.sqrt(K), torch.randn(N, generator=g, device="cuda")
    lin = tp.Linear(K, N, dtype=tp.float32)
    lin.load_state_dict({"weight": tp.Tensor(w), "bias": tp.Tensor(b)})
    x = torch.randn((M, K), generator=g, device="cuda")
    y = lin(tp.Tensor(x)).torch()
    assert pkg.last_kernel() == "mtrt_gemm_dense_split%s_f32" % ("_ragged" if K % 32 else ""), (pkg.last_kernel(), parts)
    ref, mass = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    # K products and additions, the bias and one more rounding, each within half an ulp of what it rounds
    assert bool(((y.double() - ref).abs() <= (K + 3) * 2.0 ** -24 * mass).all())
    for _ in range(3):
        assert torch.equal(lin(tp.Tensor(x)).torch(), y)
    streams, out = [torch.cuda.Stream() for _ in range(2)], []
    torch.cuda.synchronize()
    for i in range(6):
        with torch.cuda.stream(streams[i % 2]):
            out.append(lin(tp.Tensor(x)).torch())
    torch.cuda.synchronize()
    assert all(torch.equal(o, y) for o in out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = lin(tp.Tensor(x)).torch()
    for _ in range(3):
        captured.fill_(7.0)
        graph.replay()
        assert torch.equal(lin(tp.Tensor(x)).torch(), y)
        torch.cuda.synchronize()
        assert torch.equal(captured, y)


@pytest.mark.parametrize("M,K,N,parts", SHAPES)
def test_beside_the_call_that_does_not_share(tp, pkg, M, K, N, parts):
    """mtrt_hip_linear without memory for the parts, mtrt_hip_linear_dense and a module whose bias is not contiguous: the same bits, which the shared sum
    agrees with up to the order of its terms."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    w, b = torch.randn((N, K), generator=g, device="cuda") / math.sqrt(K), torch.randn(N, generator=g, device="cuda")
    x = torch.randn((M, K), generator=g, device="cuda")
    L, stream = pkg.lib(), torch.cuda.current_stream().cuda_stream
    p = Plan(route=2, dtype=pkg.F32, q_dtype=-1, K=K, N=N, w=w.data_ptr(), bias=b.data_ptr())
    need, out = L.mtrt_hip_linear_workspace(ctypes.byref(p), M), []
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert need == (M + 31) // 32 * ((N + 31) // 32) * parts * 4096
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    for memory in (need, need - 1, 0):
        y = torch.full((M, N), 7.0, device="cuda")
        pkg.check(L.mtrt_hip_linear(stream, ctypes.byref(p), x.data_ptr(), y.data_ptr(), M, ws.data_ptr() if memory else None, memory))
        assert ("split" in pkg.last_kernel()) == (memory == need), pkg.last_kernel()
        out.append(y)
    shared, dense = out[0], pkg.linear_dense(x, w, b)
    assert torch.equal(out[1], dense) and torch.equal(out[2], dense)
    lin = tp.Linear(K, N, dtype=tp.float32)
    wide = torch.zeros((N, 2), device="cuda")
    wide[:, 0] = b
    lin.weight, lin.bias = tp.Tensor(w), tp.Tensor(wide[:, 0])
    assert torch.equal(lin(tp.Tensor(x)).torch(), dense)
    # each within (K + 3) half ulps of the sum of the terms' sizes, test_parts_against_float64
    mass = x.double().abs() @ w.double().abs().T + b.double().abs()
    assert bool(((shared.double() - dense.double()).abs() <= 2 * (K + 3) * 2.0 ** -24 * mass).all())


@pytest.mark.parametrize("M,K,N,quantized", [(257, 12288, 512, False), (33, 4096, 1024, True)])
def test_a_module_whose_parts_find_no_memory(tp, pkg, M, K, N, quantized):
    """Where the allocator has room for the result (and an x that is quantized) and none for the partial sums: unsplit, as a call that does not share."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x, wide = tp.Tensor(torch.randn((M, K), generator=g, device="cuda")), torch.zeros((N, 2), device="cuda")
    wide[:, 0] = torch.randn(N, generator=g, device="cuda")
    lin = tp.Linear(K, N, dtype=tp.float32, quant_dtype=tp.float8 if quantized else None)
    lin.weight = tp.Tensor(torch.randn((N, K), generator=g, device="cuda") / math.sqrt(K))
    if quantized:
        lin.weight_scale, lin.input_scale = tp.Tensor(torch.tensor(4.0 / math.sqrt(K) / 448)), tp.Tensor(torch.tensor(4.0 / 448))
    lin.bias = tp.Tensor(wide[:, 0])
    want = lin(x).torch()                                            # (a strided bias takes the general path, which does not share)
    assert "split" not in pkg.last_kernel()
    lin.bias = tp.Tensor(wide[:, 0].contiguous())
    shared = lin(x).torch()
    assert "split" in pkg.last_kernel()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held, mib, total = [], 1 << 20, torch.cuda.get_device_properties(0).total_memory
    try:
        # one byte more than a MiB is asked of the device in 20 MiB, anything up to that in 2
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 8 * mib) / total)
        with pytest.raises(torch.OutOfMemoryError):
            for _ in range(4096):
                held.append(torch.empty(mib + 512, dtype=torch.uint8, device="cuda"))
        y = lin(x).torch()
        name = pkg.last_kernel()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert "split" not in name and torch.equal(y, want), name
    assert torch.equal(lin(x).torch(), shared) and "split" in pkg.last_kernel()
