"""The host side of the cluster layer without a GPU: the runtime's own sources over the stand-ins of native/fake_hip.cpp (256
compute units), so that what a call would launch, with which arguments, can be looked at on the CPU."""
import ctypes
import os
import shutil
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_vp, _i32, _i64, _u32 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64, ctypes.c_uint32
_CALLBACK = ctypes.CFUNCTYPE(None, ctypes.c_char_p, _u32, _u32, _vp, ctypes.POINTER(_vp))


class Split(ctypes.Structure):
    """gemm_frag::Split"""
    _fields_ = [("splits", _u32), ("per", _u32), ("partial", _vp), ("tickets", _vp)]


class LinearPlan(ctypes.Structure):
    """struct mtrt_hip_linear_plan"""
    _fields_ = [(n, _i32) for n in ("route", "dtype", "q_dtype", "reserved")] + [("K", _i64), ("N", _i64)] + \
               [(n, _vp) for n in ("w", "w_frag", "w_scale", "x_scale", "bias")]


def build(folder):
    """Compiles the library into `folder`; returns its path."""
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    runtime = os.path.join(ROOT, "tensorrt-incubator_amd", "csrc", "runtime")
    image = os.path.join(folder, "image")
    with open(image, "wb") as f:
        f.write(b"\x7fELF" + b"\0" * 60)
    path = os.path.join(folder, "dispatch.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__",
                    '-DMTRT_HSACO_PATH="%s"' % image, "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(rocm, "include"), "-I" + runtime] +
                   [os.path.join(runtime, f) for f in ("clusters.cpp", "device_state.cpp")] +
                   [os.path.join(ROOT, "tests", "native", "fake_hip.cpp"), "-o", path], check=True)
    return path


class Dispatch:
    """The library with a state of its own (a copy of the file: a loaded library's state is the process's).  `launches`
    collects (kernel, stream, its (splits, per, partial, tickets) or the address of its reduction block or None), `fills` the
    clears (address, words, stream), `sizes` every launch's (kernel, grid, block), `forms` the run-time arguments by which some kernels
    choose what they do."""

    _FORMS = {"mtrt_gemm_dense_rows32_f32": (7, 8), "mtrt_gemm_dense_edge_f32": (7,), "mtrt_gemm_dense_edge_f16": (7,), "mtrt_gemm_dense_edge_bf16": (7,),
              "mtrt_gemm_w8a8_small16": (10,), "mtrt_gemm_w8a8_frag_rows32": (10,), "mtrt_gemm_dense_frag_f16_rows16": (9,), "mtrt_gemm_dense_frag_bf16_rows16_f8": (9,)}

    def __init__(self, pkg, path, copy):
        shutil.copy(path, copy)
        self.lib = ctypes.CDLL(copy)
        for name, (restype, argtypes) in pkg.PROTOTYPES.items():
            if hasattr(self.lib, name):
                f = getattr(self.lib, name)
                f.restype, f.argtypes = restype, argtypes
        self.lib.mtrt_hip_linear.restype, self.lib.mtrt_hip_linear.argtypes = _i32, [_vp, _vp, _vp, _vp, _i64, _vp, _i64]
        self.lib.mtrt_hip_linear_workspace.restype, self.lib.mtrt_hip_linear_workspace.argtypes = _i64, [_vp, _i64]
        self.lib.fake_set_capturing.argtypes = [_vp, _i32]
        self.lib.fake_destroy_stream.argtypes = [_vp]
        self.launches = []
        self.fills = []
        self.sizes = []
        self.forms = []
        self._callback = _CALLBACK(self._launched)
        self.lib.fake_set_launch_callback(self._callback)
        assert self.lib.mtrt_hip_init() == 0

    @staticmethod
    def _split_argument(name):
        """Which argument of a kernel is its Split, or None."""
        if name.startswith("mtrt_gemm_w8a8_frag_t") and "t256x384" not in name:
            return 8
        if name.startswith("mtrt_gemm_w4a16_t") and "_t256" not in name:
            return 9
        if name.startswith("mtrt_gemm_dense_frag_") and "rows" not in name and "t256x384" not in name or name.startswith("mtrt_gemm_dense_split"):
            return 7
        return None

    def _launched(self, name, grid, block, stream, args):
        name = name.decode()
        self.sizes.append((name, grid, block))
        if name in self._FORMS:
            self.forms.append((name,) + tuple(ctypes.cast(args[i], ctypes.POINTER(_i32))[0] for i in self._FORMS[name]))
        if name == "mtrt_fill":
            self.fills.append((ctypes.cast(args[0], ctypes.POINTER(_vp))[0], ctypes.cast(args[1], ctypes.POINTER(_i64))[0], stream))
            return
        at = self._split_argument(name)
        split = None
        if name.startswith(("mtrt_amax_", "mtrt_dynqdq_")):
            split = ctypes.cast(args[5 if name.startswith("mtrt_amax_") else 7], ctypes.POINTER(_vp))[0]
        elif name.startswith("mtrt_nvfp4_dq_"):       # (codes, scales, values, vectors)
            split = tuple(ctypes.cast(args[i], ctypes.POINTER(_i64))[0] for i in (0, 1, 3, 4))
        elif at is not None:
            s = ctypes.cast(args[at], ctypes.POINTER(Split))[0]
            split = (s.splits, s.per, s.partial, s.tickets)
        self.launches.append((name, stream, split))

    def capturing(self, stream, on):
        self.lib.fake_set_capturing(stream, on)

    # One call of each family; operands are addresses that nobody reads.  Returns the launch.
    def w8a8(self, stream, M, K, N, scratch=True):
        need = self.lib.mtrt_hip_gemm_w8a8_fragments_workspace(M, K, N)
        assert self.lib.mtrt_hip_gemm_w8a8_fragments_ws(stream, 256, 256, 256, 256, 256, M, K, N, 4096 if scratch else None, need if scratch else 0) == 0
        return self.launches[-1]

    def w4a16(self, stream, M, K, N, block=128, scratch=True):
        need = self.lib.mtrt_hip_gemm_w4a16_workspace(M, K, N, block)
        assert self.lib.mtrt_hip_gemm_w4a16_ws(stream, 256, 256, 256, 256, 256, M, K, N, block, 4096 if scratch else None, need if scratch else 0) == 0
        return self.launches[-1]

    def linear(self, stream, M, K, N, dtype, route=2, q_dtype=-1):
        p = LinearPlan(route=route, dtype=dtype, q_dtype=q_dtype, K=K, N=N, w_frag=256, w_scale=256 if route < 2 else None,
                       x_scale=256 if q_dtype >= 0 else None)
        need = self.lib.mtrt_hip_linear_workspace(ctypes.byref(p), M)
        assert self.lib.mtrt_hip_linear(stream, ctypes.byref(p), 256, 256, M, 4096 if need else None, need) == 0
        return self.launches[-1]

    def amax(self, stream, dtype):
        assert self.lib.mtrt_hip_amax(stream, 256, dtype, 4096, 127.0, 256, 256) == 0
        return self.launches[-1]

    def dynamic(self, stream, dtype, code):
        assert self.lib.mtrt_hip_dynamic_quantize_dequantize(stream, 256, dtype, 256, code, 256, 1 << 20, 127.0, 256, 256, 0) == 0
        return self.launches[-1]
