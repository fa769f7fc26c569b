"""What the compiled kernels ask of the device, from the code object's own metadata: a one-launch dynamic quantization holds its part of the
tensor in registers, and private memory beside them means that some of it is written out and read back (16 vectors a lane, f32 of 14 Mi
elements: 20.9 us with none, 22.9 with 164 bytes)."""
import os
import re
import subprocess

import pytest


def metadata(pkg, tmp_path):
    llvm = "/opt/rocm/llvm/bin/"
    module = os.path.join(os.path.dirname(pkg.__file__), "lib", "mtrt_kernels.hsaco")
    try:
        targets = subprocess.run([llvm + "clang-offload-bundler", "--list", "--type=o", "--input=" + module], capture_output=True, text=True, check=True).stdout
        target = next(t for t in targets.split() if "gfx950" in t)
        out = str(tmp_path / "kernels.elf")
        subprocess.run([llvm + "clang-offload-bundler", "--unbundle", "--type=o", "--targets=" + target, "--input=" + module, "--output=" + out], check=True)
        return subprocess.run([llvm + "llvm-readelf", "--notes", out], capture_output=True, text=True, check=True).stdout
    except FileNotFoundError:
        pytest.skip("no LLVM tools beside the compiler")


def test_one_launch_dynamic_quantization_stays_in_registers(pkg, tmp_path):
    private = dict(re.findall(r"\.name:\s+(mtrt_dynqdq_\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", metadata(pkg, tmp_path)))
    assert len(private) == 10 and {name: size for name, size in private.items() if size != "0"} == {}


def test_the_resident_layernorm_and_the_tiles_spill_nothing(pkg, tmp_path):
    """The eight-vector LayerNorm held to 64 registers: none of an f32 row's in private memory (one 8-byte slot: [5500, 2048] 16.5 -> 17.3 us); bf16 has had some
    (32 bytes) and does not pay.  The GEMM tiles' loops likewise: only the wide W8A8 tile with a bias has a few bytes."""
    private = dict(re.findall(r"\.name:\s+(mtrt_\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", metadata(pkg, tmp_path)))
    names = [n for n in private if re.match(r"mtrt_layernorm_\S+_v8r$|mtrt_gemm_(w4a16|w8a8_frag|dense_frag_\S+)_t\d|mtrt_gemm_w4a16_strips", n)]
    assert len(names) > 35
    assert {n: int(private[n]) for n in names if int(private[n]) > {"mtrt_layernorm_bf16_v8r": 32, "mtrt_gemm_w8a8_frag_t256x384_linear": 44}.get(n, 0)} == {}


def test_row_kernels_spill_nothing(pkg, tmp_path):
    """LayerNorm and softmax hold a row in registers; but for the LayerNorm above."""
    private = dict(re.findall(r"\.name:\s+(mtrt_(?:layernorm|softmax)_\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", metadata(pkg, tmp_path)))
    assert len(private) > 130
    assert {n for n, size in private.items() if size != "0"} <= {"mtrt_layernorm_bf16_v8r"}


def test_softmax_keeps_the_masks_of_a_rows_end(pkg, tmp_path):
    """A workgroup's softmax that works on every vector asks three times which of them are the row's; the answers stay in scalar registers, two to a
    vector (worked out in each pass, f32 [300, 9001] takes 6.8 us instead of 5.9)."""
    scalars = dict(re.findall(r"\.name:\s+(mtrt_softmax_\w+?_[gu](?:256v\d+|1024v\d+a)t?)\n(?:.*\n)*?\s+\.sgpr_count:\s+(\d+)", metadata(pkg, tmp_path)))
    assert len(scalars) == 40
    assert {n: int(s) for n, s in scalars.items() if int(s) < 3 * int(re.search(r"v(\d+)a?t?$", n).group(1))} == {}
