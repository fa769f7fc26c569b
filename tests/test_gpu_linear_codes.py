"""A Linear whose weights are kept as float8 codes gives the bits of the one whose weights are dequantized beforehand: every kernel of either, rows and columns
at the ends of tiles, K of one slice, of an odd number and off whole slices, all code values, scales from the least to the largest that matter."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

# the kernels' names behind the type, each with the least product that takes it and others off whole tiles
SHAPES = {"rows16_f8": [(1, 64, 37), (16, 832, 100)], "rows16_long_f8": [(5, 3520, 32), (2, 8256, 70)], "rows32": [(22, 64, 32), (31, 2240, 4001)],
          "t32x128": [(35, 64, 47), (33, 2112, 32)], "t64x128": [(199, 64, 4658), (1414, 5568, 149)],
          "t128x128": [(1041, 64, 1948), (1648, 4224, 596)], "t128x256": [(387, 64, 10457), (208, 4288, 10519)], "t128x384": [(1097, 384, 8474), (999, 4096, 11008)],
          "t256x256": [(1228, 1152, 10724)], "t256x384": [(2018, 256, 9493), (2000, 320, 11000)]}
RAGGED = [(3, 65, 33), (17, 1000, 640), (300, 2049, 1000)]


class Plan(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int32) for n in ("route", "dtype", "q_dtype", "reserved")] + [("K", ctypes.c_int64), ("N", ctypes.c_int64)] + \
               [(n, ctypes.c_void_p) for n in ("w", "w_frag", "w_scale", "x_scale", "bias")]


@pytest.mark.parametrize("dname", ["float16", "bfloat16"])
def test_codes_give_the_bits_of_dequantized_weights(pkg, dname):
    import torch
    L, td = pkg.lib(), getattr(torch, dname)
    code = {"float16": pkg.F16, "bfloat16": pkg.BF16}[dname]
    xn = {"float16": "f16", "bfloat16": "bf16"}[dname]

    def fragments(t, dtype, K, N):
        f = torch.empty(L.mtrt_hip_linear_fragments_bytes(dtype, K, N), dtype=torch.int8, device="cuda")
        pkg.check(L.mtrt_hip_linear_prepack_fragments(None, t.data_ptr(), dtype, f.data_ptr(), K, N))
        return f

    def linear(x, M, **k):
        p = Plan(**k)
        need = L.mtrt_hip_linear_workspace(ctypes.byref(p), M)
        ws, y = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda"), torch.full((M, k["N"]), 7.0, dtype=td, device="cuda")
        pkg.check(L.mtrt_hip_linear(None, ctypes.byref(p), x.data_ptr(), y.data_ptr(), M, ws.data_ptr(), need))
        torch.cuda.synchronize()
        return y, pkg.last_kernel()

    seen = set()
    for M, K, N in [s for some in SHAPES.values() for s in some] + RAGGED:
        g = torch.Generator(device="cuda").manual_seed(M + K + N)
        codes = torch.randint(0, 256, (N, K), generator=g, device="cuda", dtype=torch.uint8)
        codes = torch.where((codes & 0x7F) == 0x7F, codes & 0x80, codes)             # (no NaN among them: their payloads are nobody's business)
        # down to where f16 results are subnormal
        scale = torch.exp2(torch.rand(N, generator=g, device="cuda") * 12 - 20).to(td).float()
        w = torch.empty((N, K), dtype=td, device="cuda")
        pkg.check(L.mtrt_hip_dequantize(None, codes.data_ptr(), pkg.F8E4M3FN, w.data_ptr(), code, scale.data_ptr(), pkg.SCALE_ROW, N, K, N))
        x = torch.randn((M, K), generator=g, device="cuda").to(td)
        bias = torch.randn(N, generator=g, device="cuda").to(td)
        x_scale = torch.full((1,), 4.0 / 448, device="cuda").to(td).float()
        f8, f16 = fragments(codes, pkg.F8E4M3FN, K, N), fragments(w, code, K, N)
        for quantized in ((True, False) if K % 64 == 0 else (True,)):
            k = dict(dtype=code, q_dtype=pkg.F8E4M3FN if quantized else -1, K=K, N=N, x_scale=x_scale.data_ptr() if quantized else None, bias=bias.data_ptr())
            want, _ = linear(x, M, route=2, w_frag=f16.data_ptr(), **k)
            got, got_name = linear(x, M, route=3, w_frag=f8.data_ptr(), w_scale=scale.data_ptr(), **k)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (M, K, N, quantized, got_name)
            both, name = linear(x, M, route=3, w=f16.data_ptr(), w_frag=f8.data_ptr(), w_scale=scale.data_ptr(), **k)
            assert torch.equal(both.view(torch.int16), want.view(torch.int16)), (M, K, N, quantized, name)
            assert "_%s_f8_" % xn not in name, name                  # (rows16 kernels take either)
            seen.add(got_name)
        # the kernels agree with each other; one of them against 64 bits
        ref = x.double() @ w.double().T + bias.double()
        if not quantized:
            mass = x.double().abs() @ w.double().abs().T + bias.double().abs()
            u = {"float16": 2.0 ** -11, "bfloat16": 2.0 ** -8}[dname]
            assert bool(((got.double() - ref).abs() <= u * ref.abs() + (1 + u) * (K + 2) * 2.0 ** -24 * mass + 2.0 ** -24).all()), (M, K, N, name)
    for name in SHAPES:
        assert any(s.startswith("mtrt_gemm_dense_frag_%s_%s" % (xn, name if name.startswith("rows16") else "f8_" + name)) for s in seen), (name, sorted(seen))
