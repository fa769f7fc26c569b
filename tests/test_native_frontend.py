"""The native side of the Python calls (csrc/frontend/frontend.cpp): the steady-state path of each `tp` function gives what
its general path gives on the same values, for every scale addressing, type and rank it takes on; what it does not
take on (values still in host memory, other axes, views that are not dense) goes to the general path; preconditions
are reported as the package's functions always did."""
import importlib

import numpy as np
import pytest

from helpers import rng


@pytest.fixture(scope="module")
def tp(pkg):
    return importlib.import_module(pkg.__name__ + ".tp")


def test_preconditions_are_assertions(pkg):
    import torch
    x = torch.zeros((2, 16))
    for call in (lambda: pkg.amax(x, 127.0), lambda: pkg.softmax(x), lambda: pkg.quantize(x, x, pkg.I8),
                 lambda: pkg.layernorm(x, x[0], x[0], 1e-5), lambda: pkg.linear_dense(x, x), lambda: pkg.nvfp4_quantize(x, x[0, 0]),
                 lambda: pkg.dynamic_quantize_rows(x, pkg.I8, 127.0), lambda: pkg.gemm_w4a16(x, x, 16, 2, 16)):
        with pytest.raises(AssertionError):
            call()
    with pytest.raises(TypeError):
        pkg.softmax([1.0, 2.0])


@pytest.mark.gpu
@pytest.mark.parametrize("dname", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("shape,dim,qname", [((3, 5, 7), 1, "int8"), ((3, 5, 7), -1, "float8"), ((6, 33), 0, "int8"), ((17,), None, "int8"),
                                             ((256, 48), "block", "int4"), ((), None, "float8"), ((1, 1, 1), 2, "int4"), ((2, 3, 4, 5), 0, "int4")])
def test_steady_state_calls_equal_the_general_path(tp, dname, shape, dim, qname):
    import torch
    td, d, qd = getattr(torch, dname), getattr(tp, dname), getattr(tp, qname)
    r = rng(31 + len(shape))
    host = torch.from_numpy(np.asarray(r.standard_normal(shape) * 3, dtype=np.float32)).to(td)
    sshape = () if dim is None else (shape[0] // 64, shape[1]) if dim == "block" else (shape[dim],)
    scale = tp.Tensor(torch.from_numpy(np.asarray(r.uniform(0.02, 0.2, sshape), dtype=np.float32)).to(td))
    dim = None if dim == "block" else dim
    native = tp._native()
    general = tp.quantize(tp.Tensor(host), scale, qd, dim)           # values in host memory: the general path uploads them
    x = tp.Tensor(host.cuda())
    q = native.tp_quantize(x, scale, qd, dim)
    assert q is not NotImplemented and type(q) is tp.Tensor and q.dtype is qd and q.shape == tuple(shape) and not q.is_cpu_constant
    assert torch.equal(q.torch(), general.torch())
    y = native.tp_dequantize(q, scale, d, dim)
    assert y is not NotImplemented and y.dtype is d and y.shape == tuple(shape)
    scale2 = tp.Tensor(scale.torch())                                # not uploaded yet: the general path
    assert native.tp_dequantize(q, scale2, d, dim) is NotImplemented
    assert torch.equal(tp.dequantize(q, scale2, d, dim).torch(), y.torch())


@pytest.mark.gpu
def test_what_is_left_to_the_general_path(tp):
    import torch
    native = tp._native()
    x = torch.randn(4, 6, device="cuda")
    one = tp.Tensor(np.float32(1.0))
    tp.quantize(tp.Tensor(x), one, tp.int8)
    t = tp.Tensor(x.t())                                             # not dense
    assert native.tp_quantize(t, one, tp.int8, None) is NotImplemented
    assert torch.equal(tp.quantize(t, one, tp.int8).torch(), tp.quantize(tp.Tensor(x), one, tp.int8).torch().t())
    for args in ((tp.Tensor(x), 1.0, tp.int8, None), (tp.Tensor(x), one, tp.float16, None), (tp.Tensor(x), one, tp.int8, 0),
                 (tp.Tensor(x.half()), one, tp.int8, None), (x, one, tp.int8, None), (tp.Tensor(x[:0]), one, tp.int8, None)):
        assert native.tp_quantize(*args) is NotImplemented
    assert native.tp_softmax(tp.Tensor(x), 0) is NotImplemented and native.tp_softmax(tp.Tensor(x), None) is NotImplemented
    w = tp.Tensor(torch.ones(6, device="cuda"))
    b = tp.Tensor(torch.zeros(6, device="cuda"))
    assert native.tp_layernorm(tp.Tensor(x), w, tp.Tensor(torch.zeros(5, device="cuda")), 1e-5) is NotImplemented
    assert native.tp_layernorm(tp.Tensor(x[0].contiguous()), w, b, 1e-5) is NotImplemented
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):                                       # enqueued on the current stream, whichever it is
        torch.cuda._sleep(1000000)
        late = tp.Tensor(x * 2)
        y = native.tp_softmax(late, -1)
    s.synchronize()
    assert torch.allclose(y.torch(), torch.softmax(x * 2, -1), atol=1e-6)
    assert torch.allclose(native.tp_layernorm(tp.Tensor(x), w, b, 1e-5).torch(), torch.nn.functional.layer_norm(x, (6,)), atol=1e-5)


@pytest.mark.gpu
def test_in_place_updates_of_a_scale_are_noticed(tp):
    """The device copy of a constant scale belongs to the values it was made from, in both paths and in a Linear."""
    import torch
    x = tp.Tensor(torch.full((4, 64), 8.0, device="cuda"))
    scale = tp.Tensor(np.float32(1.0))
    q = tp.quantize(x, scale, tp.int8)
    assert tp._native().tp_quantize(x, scale, tp.int8, None) is not NotImplemented
    scale.torch().mul_(2)
    assert tp._native().tp_quantize(x, scale, tp.int8, None) is NotImplemented
    assert bool((q.torch() == 8).all()) and bool((tp.quantize(x, scale, tp.int8).torch() == 4).all())
    assert bool((tp.dequantize(q, scale, tp.float32).torch() == 16).all())
    with torch.inference_mode():                                     # a constant without a version counter
        fixed = tp.Tensor(torch.tensor(4.0))
        assert bool((tp.quantize(x, fixed, tp.int8).torch() == 2).all())
        assert bool((tp._native().tp_quantize(x, fixed, tp.int8, None).torch() == 2).all())
    lin = tp.Linear(64, 8, bias=False, quant_dtype=tp.float8)
    lin.load_state_dict({"weight": tp.Tensor(torch.ones(8, 64)), "weight_scale": tp.Tensor(np.float32(0.5)), "input_scale": tp.Tensor(np.float32(0.5))})
    assert bool((lin(x).torch() == 512).all())
    lin.input_scale.torch().fill_(2.0 ** -6)                         # 8 / 2^-6 is past the largest code: 448 * 2^-6 = 7
    assert bool((lin(x).torch() == 448).all())
    lin.weight_scale.torch().fill_(2.0 ** -9)                        # 448 * 2^-9 = 0.875
    assert bool((lin(x).torch() == 392).all())


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["amax", "dynamic"])
def test_amax_and_scale_are_tensors_of_their_own(pkg, call):
    """Each is a dense f32 scalar, in-place work on one leaves the other, either outlives the other, and both serve as the scale of
    another call; so under inference mode and on a stream that is not the default one."""
    import torch
    x = torch.from_numpy(rng(5).standard_normal((7, 96), dtype=np.float32)).cuda()

    def run():
        if call == "amax":
            return pkg.amax(x, 127.0)
        return pkg.dynamic_quantize_dequantize(x, pkg.I8, 127.0)[2:]
    want = float(x.abs().max())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for where in (torch.no_grad(), torch.inference_mode(), torch.cuda.stream(side)):
        with where:
            amax, scale = run()
            for t in (amax, scale):
                assert t.shape == () and t.dtype == torch.float32 and t.is_cuda and t.is_contiguous() and not t.requires_grad
            codes = pkg.quantize(x, scale.reshape(1), pkg.I8)
            torch.cuda.synchronize()
            assert float(amax) == want and float(scale) == float(np.float32(want) / np.float32(127.0))
            amax.zero_()
            assert float(scale) == float(np.float32(want) / np.float32(127.0))
            kept = scale
            del amax, scale
            others = [run() for _ in range(64)]
            assert float(kept) == float(np.float32(want) / np.float32(127.0)) and all(float(a) == want for a, _ in others)
            assert int(codes.abs().max()) == 127


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["amax", "dynamic"])
def test_amax_and_scale_have_storages_of_their_own(pkg, call):
    """A storage of one number each, where torch's allocator starts one: resized, saved or handed on by address without the other."""
    import io

    import torch
    x = torch.from_numpy(rng(6).standard_normal((7, 96), dtype=np.float32)).cuda()
    amax, scale = pkg.amax(x, 127.0) if call == "amax" else pkg.dynamic_quantize_dequantize(x, pkg.I8, 127.0)[2:]
    value = float(np.float32(float(x.abs().max())) / np.float32(127.0))
    for t in (amax, scale):
        assert t.untyped_storage().nbytes() == 4 and t.storage_offset() == 0 and t.data_ptr() % 256 == 0
    assert amax.untyped_storage().data_ptr() != scale.untyped_storage().data_ptr()
    saved = io.BytesIO()
    torch.save(scale, saved)
    saved.seek(0)
    assert torch.load(saved, weights_only=True).untyped_storage().nbytes() == 4
    amax.untyped_storage().resize_(0)
    assert float(scale) == value


@pytest.mark.gpu
def test_extents_that_no_tensor_has(pkg):
    import torch
    a, s = torch.zeros((2, 64), dtype=torch.float16, device="cuda"), torch.zeros((1, 8), dtype=torch.float16, device="cuda")
    w = torch.zeros(64 * 8 // 2, dtype=torch.uint8, device="cuda")
    for n in (-1, 1 << 61):
        with pytest.raises(RuntimeError):
            pkg.gemm_w4a16(a, s, 64, n, 64, w_kn_packed=w)
    q, scales, amax = torch.zeros(128, dtype=torch.uint8, device="cuda"), torch.zeros(16, dtype=torch.uint8, device="cuda"), torch.ones((), device="cuda")
    with pytest.raises(RuntimeError):
        pkg.nvfp4_dequantize(q, scales, amax, torch.float16, (-2, 128))
