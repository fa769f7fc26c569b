"""The host side of a Linear whose weights are float8 codes: which activations it takes."""
import ctypes

import pytest

import dispatch


@pytest.fixture(scope="module")
def gpu(pkg, tmp_path_factory):
    folder = tmp_path_factory.mktemp("codes")
    return dispatch.Dispatch(pkg, dispatch.build(str(folder)), str(folder / "copy.so"))


@pytest.mark.parametrize("M", [1, 16, 17, 999])
@pytest.mark.parametrize("through", [None, "F8E4M3FN", "I8", "I4"])
def test_codes_are_read_by_kernels_that_know_them(gpu, pkg, through, M):
    """Up to 16 rows x is quantized in the kernel that takes the weights, and only those of a plain x and of float8 codes have the
    weights' scales: another would read the codes as 16-bit weights, past their end."""
    q_dtype = -1 if through is None else getattr(pkg, through)
    p = dispatch.LinearPlan(route=3, dtype=pkg.F16, q_dtype=q_dtype, K=1024, N=8192, w_frag=256, w_scale=256, x_scale=256 if through else None)
    before = len(gpu.sizes)
    need = gpu.lib.mtrt_hip_linear_workspace(ctypes.byref(p), M)
    status = gpu.lib.mtrt_hip_linear(8, ctypes.byref(p), 256, 256, M, 4096 if need else None, need)
    if through in (None, "F8E4M3FN"):
        assert status == 0
        name = gpu.sizes[-1][0]
        assert name.startswith("mtrt_gemm_dense_frag_f16_rows16" if M <= 16 else "mtrt_gemm_dense_frag_f16_f8_"), name
    else:
        assert status != 0 and need == 0 and len(gpu.sizes) == before
