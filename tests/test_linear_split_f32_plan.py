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
