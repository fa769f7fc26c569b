"""Which loads and stores of the compiled kernels go past the caches, from their instructions: results do not depend on it, so that a hint that the
compiler drops, or a line between two bodies that it folds into one, is seen nowhere else."""
import collections
import os
import re
import subprocess

import pytest


@pytest.fixture(scope="module")
def code(pkg, tmp_path_factory):
    """names(pattern) of the module's kernels, and accesses(names): kernel -> Counter of (mnemonic, past the caches)."""
    llvm, folder = "/opt/rocm/llvm/bin/", tmp_path_factory.mktemp("code")
    module, out = os.path.join(os.path.dirname(pkg.__file__), "lib", "mtrt_kernels.hsaco"), str(folder / "kernels.elf")
    if not os.path.exists(llvm + "llvm-objdump"):
        pytest.skip("no LLVM tools beside the compiler")

    def run(tool, *args):
        return subprocess.run([llvm + tool] + list(args), capture_output=True, text=True, check=True).stdout
    target = next(t for t in run("clang-offload-bundler", "--list", "--type=o", "--input=" + module).split() if "gfx950" in t)
    run("clang-offload-bundler", "--unbundle", "--type=o", "--targets=" + target, "--input=" + module, "--output=" + out)
    everything = sorted(set(re.findall(r"\bFUNC\s+\S+\s+\S+\s+\S+\s+(mtrt_\S+)", run("llvm-readelf", "-sW", out))))

    def names(pattern):
        return [n for n in everything if re.fullmatch(pattern, n)]

    def accesses(kernels):
        found, kernel = {}, None
        for line in run("llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(kernels), out).splitlines():
            head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if head:
                kernel = found.setdefault(head.group(1), collections.Counter())
            access = re.match(r"\s+(global_(?:load|store)_\w+)\s", line)
            if access:
                kernel[access.group(1), re.search(r"\snt\b", line.split("//")[0]) is not None] += 1
        assert sorted(found) == sorted(kernels)
        return found
    return names, accesses


def test_rows_held_in_registers_are_written_past_the_caches(code):
    names, accesses = code
    kernels = names(r"mtrt_(layernorm|softmax)_\w+_[vgu]\d+(v\d+)?[rea]?t?")
    assert len(kernels) > 130
    folded = {"mtrt_softmax_f32_v1", "mtrt_softmax_bf16_v1"}         # whole rows of up to 64 vectors: the compiler makes one store of two branches
    for kernel, found in accesses(kernels).items():
        assert found["global_store_dwordx4", True] > 0 and (found["global_store_dwordx4", False] == 0 or kernel in folded), kernel


def test_one_launch_dynamic_quantization_passes_the_caches_by(code):
    """The tensor, codes and dequantized values; what the workgroups tell each other is one word or two.  In the four-vector kernels a few workgroups
    each read the others' parts from the caches as well."""
    names, accesses = code
    kernels = names(r"mtrt_dynqdq_\w+")
    assert len(kernels) == 10
    for kernel, found in accesses(kernels).items():
        assert found["global_store_dwordx4", True] > 0 and found["global_store_dwordx4", False] == 0, kernel
        assert found["global_store_dwordx2" if "f16" in kernel else "global_store_dword", True] > 0, kernel
        assert found["global_load_dwordx4", True] > 0 and found["global_load_dwordx4", False] == (4 if kernel.endswith("_v4") else 0), kernel


def test_layernorm_reads_its_rows_past_the_caches(code):
    """As many vectors past the caches as it stores; through them only the two parameters' vectors."""
    names, accesses = code
    kernels = names(r"mtrt_layernorm_\w+_[vgu]\d+(v\d+)?[rea]?")
    assert len(kernels) > 60
    for kernel, found in accesses(kernels).items():
        past = found["global_load_dwordx4", True]
        assert past == found["global_store_dwordx4", True] > 0 and found["global_load_dwordx4", False] == 2 * past, kernel


def test_softmax_reads_its_rows_as_its_name_says(code):
    """Through the caches in the kernels that end in t, past them in the others, of which each has one."""
    names, accesses = code
    kernels = names(r"mtrt_softmax_\w+_[vgu]\d+(v\d+)?[ea]?t?")
    assert len(kernels) > 120 and all(k + "t" in kernels for k in kernels if not k.endswith("t"))
    for kernel, found in accesses(kernels).items():
        assert found["global_load_dwordx4", not kernel.endswith("t")] > 0 and found["global_load_dwordx4", kernel.endswith("t")] == 0, kernel


def test_cut_softmax_rows_pass_the_caches_by(code):
    names, accesses = code
    kernels = names(r"mtrt_softmax_\w+_v\d+c")
    assert len(kernels) == 15
    for kernel, found in accesses(kernels).items():
        for access in ("load", "store"):                             # (of one vector a lane: the stores of its two bodies folded, as above)
            past, through = found["global_%s_dwordx4" % access, True], found["global_%s_dwordx4" % access, False]
            assert past > 0 and (through == 0 or (access == "store" and kernel.endswith("_v1c"))), kernel


def test_few_rows_read_int8_and_int4_weights_past_the_caches(code):
    """But where several groups of rows read them (the strips' fourth body), and in the second of W8A8's two bodies."""
    names, accesses = code
    kernels = names(r"mtrt_gemm_w4a16_(skinny|strips)\w+|mtrt_gemm_w4a16_skinny|mtrt_gemm_w8a8_(small16|frag_rows32)")
    found = {kernel: (c["global_load_dwordx4", True], c["global_load_dwordx4", False]) for kernel, c in accesses(kernels).items()}
    assert set(found) == {"mtrt_gemm_w4a16_skinny", "mtrt_gemm_w4a16_skinny16", "mtrt_gemm_w4a16_strips16", "mtrt_gemm_w4a16_strips16_b64", "mtrt_gemm_w8a8_small16",
                          "mtrt_gemm_w8a8_frag_rows32"}
    for kernel, (past, through) in found.items():
        assert past > 0 and past == {"mtrt_gemm_w4a16_strips16": 3 * through, "mtrt_gemm_w4a16_strips16_b64": 3 * through, "mtrt_gemm_w8a8_frag_rows32": through, "mtrt_gemm_w8a8_small16": through}.get(kernel, past)
        assert (through == 0) == kernel.startswith("mtrt_gemm_w4a16_skinny"), kernel
