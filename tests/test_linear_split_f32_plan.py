"""The host side of float32 Linears whose K workgroups share: a call that gets no memory for the parts runs unsplit."""
import ctypes

import pytest

import dispatch


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    folder = tmp_path_factory.mktemp("split_f32")
    return folder, dispatch.build(str(folder))


@pytest.fixture
def gpu(pkg, library, request):
    folder, path = library
    return dispatch.Dispatch(pkg, path, str(folder / (request.node.name.replace("/", "_") + ".so")))


def _call(gpu, pkg, M, K, N, workspace, nbytes, q_dtype=-1):
    """(status, the GEMM's (name, its Split's first three or None))"""
    p = dispatch.LinearPlan(route=2, dtype=pkg.F32, q_dtype=q_dtype, K=K, N=N, w=256, x_scale=256 if q_dtype >= 0 else None)
    status = gpu.lib.mtrt_hip_linear(8, ctypes.byref(p), 256, 256, M, workspace, nbytes)
    return status, gpu.launches[-1][0] if gpu.launches else None, gpu.launches[-1][2] if gpu.launches else None


@pytest.mark.parametrize("M,K,N", [(109, 3072, 448), (66, 4099, 65)])
def test_a_call_without_memory_for_its_parts_runs_unsplit(gpu, pkg, M, K, N):
    """As it did when these products asked for no memory: none at all, a byte too little, off its alignment; and with an x that is quantized
    on the way, memory for that alone, which stays what such a call cannot do without."""
    ragged = "_ragged" if K % 32 else ""
    for q_dtype in (-1, pkg.I8):
        p = dispatch.LinearPlan(route=2, dtype=pkg.F32, q_dtype=q_dtype, K=K, N=N, w=256, x_scale=256 if q_dtype >= 0 else None)
        need, x_bytes = gpu.lib.mtrt_hip_linear_workspace(ctypes.byref(p), M), (M * K * 4 + 255) // 256 * 256 if q_dtype >= 0 else 0
        status, name, split = _call(gpu, pkg, M, K, N, 4096, need, q_dtype)
        assert status == 0 and name == "mtrt_gemm_dense_split%s_f32" % ragged and split[2] == 4096 + x_bytes, name
        assert need == x_bytes + (M + 31) // 32 * ((N + 31) // 32) * split[0] * 4096
        few = [(4096, need - 1), (4096, x_bytes)] + ([(None, 0), (None, need), (4096 + 4, need)] if q_dtype < 0 else [])
        for workspace, nbytes in few:
            status, name, split = _call(gpu, pkg, M, K, N, workspace, nbytes, q_dtype)
            assert status == 0 and "split" not in name and name.startswith("mtrt_gemm_dense_") and name.endswith("_f32"), (workspace, nbytes, name)
        if q_dtype >= 0:
            before = len(gpu.sizes)
            for workspace, nbytes in ((None, need), (4096 + 4, need), (4096, x_bytes - 1)):
                assert _call(gpu, pkg, M, K, N, workspace, nbytes, q_dtype)[0] != 0
            assert len(gpu.sizes) == before


def _shares(gpu, pkg, M, K, N):
    """(parts, slices to a part) of a call, 1 part where none share; the workspace asked for, the grid and the Split are those of the parts."""
    p = dispatch.LinearPlan(route=2, dtype=pkg.F32, q_dtype=-1, K=K, N=N, w=256)
    need, tiles, slices = gpu.lib.mtrt_hip_linear_workspace(ctypes.byref(p), M), (M + 31) // 32 * ((N + 31) // 32), (K + 31) // 32
    status, name, split = _call(gpu, pkg, M, K, N, 4096 if need else None, need)
    assert status == 0
    if "split" not in name:
        assert need == 0 or need % (tiles * 4096) == 0               # (asked for, and another form is the faster one)
        return 1, slices
    assert name == "mtrt_gemm_dense_split%s_f32" % ("_ragged" if K % 32 else "")
    assert need == tiles * split[0] * 4096 and split[2] == 4096 and gpu.sizes[-1][1:] == ((tiles + 7) // 8 * 8 * split[0], 512)
    assert (split[0] - 1) * split[1] < slices <= split[0] * split[1]
    return split[0], split[1]


def test_the_parts_of_the_shapes_that_run(gpu, pkg):
    """Those of test_gpu_linear_split_f32.py: every number of parts is among them, in either kernel and with a shorter last part."""
    from test_gpu_linear_split_f32 import SHAPES
    seen = {(shape, _shares(gpu, pkg, *shape[:3])) for shape in SHAPES for _ in range(2)}
    assert len(seen) == len(SHAPES) and all(shape[3] == parts for shape, (parts, _) in seen), seen
    assert {parts for _, (parts, _) in seen} == {2, 3, 4, 6, 8}
    assert {parts for shape, (parts, _) in seen if shape[1] % 32} >= {3, 4, 8}
    assert any(parts * per != (shape[1] + 31) // 32 for shape, (parts, per) in seen)


def test_the_ends_of_the_rule(gpu, pkg):
    """More than 32 rows, sixteen slices, eight tiles, and a ticket for each of at most 512."""
    for inside, outside in (((33, 8192, 256), (32, 8192, 256)), ((33, 481, 128), (33, 480, 128)), ((64, 8192, 128), (33, 8192, 96)), ((64, 8192, 128), (224, 8192, 32)),
                            ((512, 8192, 1024), (512, 8192, 1025))):
        plans = [dispatch.LinearPlan(route=2, dtype=pkg.F32, q_dtype=-1, K=K, N=N, w=256) for _, K, N in (inside, outside)]
        needs = [gpu.lib.mtrt_hip_linear_workspace(ctypes.byref(p), shape[0]) for p, shape in zip(plans, (inside, outside))]
        assert needs[1] == 0 and _shares(gpu, pkg, *outside)[0] == 1, (outside, needs)
        if inside[1] == 8192 and inside[0] < 512:
            assert needs[0] > 0 and _shares(gpu, pkg, *inside)[0] > 1, (inside, needs)


def test_calls_in_turn_have_their_own_parts(gpu, pkg):
    """A thread keeps the last plan: the same extents in other places, and a call without memory in between, leave no trace."""
    shapes = [(109, 3072, 448), (448, 3072, 109), (64, 2048, 97), (97, 2048, 64), (33, 3072, 448)]
    alone = [_shares(gpu, pkg, *s) for s in shapes]
    for order in (shapes, shapes[::-1]):
        for s in order:
            assert _call(gpu, pkg, *s, None, 0)[0] == 0 and "split" not in gpu.launches[-1][0]
            assert _shares(gpu, pkg, *s) == alone[shapes.index(s)]


def test_a_call_without_tickets_runs_unsplit(gpu, pkg):
    """As the other families' (test_dispatch.py): the stream handle that names another stream in every thread has none."""
    M, K, N = 109, 3072, 448
    p = dispatch.LinearPlan(route=2, dtype=pkg.F32, q_dtype=-1, K=K, N=N, w=256)
    need = gpu.lib.mtrt_hip_linear_workspace(ctypes.byref(p), M)
    for stream, shared in ((8, True), (2, False), (8, True)):
        assert gpu.lib.mtrt_hip_linear(stream, ctypes.byref(p), 256, 256, M, 4096, need) == 0
        assert ("split" in gpu.launches[-1][0]) == shared
    gpu.capturing(8, True)
    recorded = set()
    for _ in range(3):
        assert gpu.lib.mtrt_hip_linear(8, ctypes.byref(p), 256, 256, M, 4096, need) == 0
        recorded.add(gpu.launches[-1][2][3])
    assert len(recorded) == 3                                        # a recorded launch's tickets are its own
    gpu.capturing(8, False)
