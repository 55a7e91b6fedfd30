"""The build of the HIP libraries: what it reads from the compiler's report, and that no kernel of
the libraries in the tree spills registers to memory (such a kernel passes every numerical test and
runs ten times slower)."""

from __future__ import annotations

import json
import subprocess

from mini_llm_runtime_amd.kernels import build


def test_spilled_registers_are_read_from_the_compiler_report(monkeypatch):
    report = "\n".join([
        "a.hip:10:1: remark: Function Name: _Zkernel_one [-Rpass-analysis=kernel-resource-usage]",
        "   10 | __global__ void kernel_one(int n) {",
        "      | ^",
        "a.hip:10:1: remark:     VGPRs: 128 [-Rpass-analysis=kernel-resource-usage]",
        "a.hip:10:1: remark:     VGPRs Spill: 301 [-Rpass-analysis=kernel-resource-usage]",
        "a.hip:90:1: remark: Function Name: _Zkernel_two [-Rpass-analysis=kernel-resource-usage]",
        "a.hip:90:1: remark:     SGPRs Spill: 0 [-Rpass-analysis=kernel-resource-usage]",
        "a.hip:90:1: remark:     VGPRs Spill: 0 [-Rpass-analysis=kernel-resource-usage]",
        # accumulators kept in memory are reported as scratch, not as spills: 704 bytes a lane are 176 registers
        "a.hip:95:1: remark: Function Name: _Zkernel_three [-Rpass-analysis=kernel-resource-usage]",
        "a.hip:95:1: remark:     ScratchSize [bytes/lane]: 704 [-Rpass-analysis=kernel-resource-usage]",
        "a.hip:95:1: remark:     VGPRs Spill: 0 [-Rpass-analysis=kernel-resource-usage]",
        "a.hip:5:3: warning: something else",
    ])
    logged = []
    monkeypatch.setattr(build, "log", logged.append)
    monkeypatch.setattr(
        subprocess, "run", lambda *a, **k: subprocess.CompletedProcess(a, 0, stdout=report, stderr=None)
    )
    assert build._run(["hipcc"], "compiling a.hip") == {"_Zkernel_one": 301, "_Zkernel_two": 0, "_Zkernel_three": 176}
    assert any("warning: something else" in line and "remark" not in line for line in logged)
    assert not any("__global__" in line or "| ^" in line for line in logged)
    assert any("_Zkernel_one spills 301" in line for line in logged)


def test_no_kernel_of_the_built_libraries_spills():
    """Read from what the last build of each library wrote beside it (a library built before the build
    kept count has nothing to say)."""
    folder = build.build_dir()
    for module in build.all_modules():
        stamp = build.library_path(module, folder).with_suffix(".json")
        if not stamp.exists():
            continue
        data = json.loads(stamp.read_text())
        if "kernels" not in data:
            continue
        assert data["kernels"] > 0, f"{stamp.name}: the compiler reported no kernel"
        assert data["spilling_kernels"] == {}, f"{stamp.name}: kernels that spill registers: {data['spilling_kernels']}"


def test_kernel_choice_for_the_benchmark_shapes():
    """The choice of a product kernel is host code and answers without a GPU: the shapes of the three
    benchmark models get the tilings that the measurements behind the estimates chose.  (The numbers are
    those of `mlr_gemm_bf16`'s `kernel` argument.)"""
    import ctypes

    path = build.library_path(build.CORE, build.build_dir())
    if not path.exists() or not build.is_current(build.CORE):
        import pytest

        pytest.skip("the core library is not built from the present sources")
    lib = ctypes.CDLL(str(path))
    for fn in (lib.mlr_gemm_bf16_kernel, lib.mlr_gemm_bf16_slices):
        fn.argtypes, fn.restype = [ctypes.c_int] * 4, ctypes.c_int
    chosen = lambda m, n, k, most: lib.mlr_gemm_bf16_kernel(m, n, k, lib.mlr_gemm_bf16_slices(m, n, k, most))
    # up to 64 tokens: the row-splitting kernel for the 0.5B products, tiles of 64 tokens whose width
    # makes one round over the compute units for the gate-up of the 7B (160 features) and 32B (224) shapes
    assert chosen(8, 9728, 896, 1) == 16 and chosen(8, 896, 4864, 8) == 16
    assert chosen(64, 37888, 3584, 1) == 65 and chosen(8, 37888, 3584, 1) == 65
    assert chosen(64, 55296, 5120, 1) == 67 and chosen(8, 55296, 5120, 1) == 67
    assert chosen(64, 9728, 896, 1) == 62 and chosen(8, 151936, 896, 1) == 14
    # a prompt of 2,048 tokens: tiles of 256 tokens, 320 features wide for the 0.5B gate-up (one round),
    # 160 for the 7B query/key/value width, square for the large products
    assert chosen(2048, 9728, 896, 1) == 48
    assert chosen(2048, 4608, 3584, 1) == 47
    assert chosen(2048, 37888, 3584, 1) == 45 and chosen(2048, 55296, 5120, 1) == 45
    assert lib.mlr_gemm_bf16_slices(2048, 3584, 18944, 4) == 2 and chosen(2048, 3584, 18944, 4) == 45
    # in between, tiles of 64 tokens for a large matrix cut along k, the staged ones for a small one
    assert chosen(128, 3584, 18944, 4) == 64 and chosen(192, 2048, 1536, 4) == 11
    # every answer is a kernel that exists, whatever the shape
    known = {16, 14, 11, 22, 23, 44, 45, 46, 47, 48, 62, 63, 64, 65, 66, 67, 68}
    for m in (1, 5, 16, 17, 33, 64, 65, 100, 257, 1000, 5000):
        for n, k in ((8, 8), (100, 40), (517, 96), (896, 896), (4608, 3584), (151936, 896), (59136, 8192)):
            for most in (1, 4, 16):
                assert chosen(m, n, k, most) in known


def test_kernel_choice_where_tiles_of_tokens_are_not_full():
    """Products whose last tile of tokens is mostly empty, and up to 256 tokens of a matrix that one round of few-token tiles streams:
    the tilings that measured fastest, by 10 to 30 % (7B and 1.5B gate-up, the 32B shape's down product)."""
    import ctypes

    path = build.library_path(build.CORE, build.build_dir())
    if not path.exists() or not build.is_current(build.CORE):
        import pytest

        pytest.skip("the core library is not built from the present sources")
    lib = ctypes.CDLL(str(path))
    for fn in (lib.mlr_gemm_bf16_kernel, lib.mlr_gemm_bf16_slices):
        fn.argtypes, fn.restype = [ctypes.c_int] * 4, ctypes.c_int
    assert [lib.mlr_gemm_bf16_kernel(m, 37888, 3584, 1) for m in (257, 288, 320, 384, 512)] == [48] * 5
    assert [lib.mlr_gemm_bf16_kernel(m, 17920, 1536, 1) for m in (65, 80, 96, 128)] == [65] * 4
    for m in (96, 128):
        slices = lib.mlr_gemm_bf16_slices(m, 5120, 27648, 8)
        assert slices == 4 and lib.mlr_gemm_bf16_kernel(m, 5120, 27648, slices) == 65


def test_second_group_of_wavefronts_where_it_has_room():
    """32-bit prompt attention has one group of wavefronts a workgroup or two, which take the room of two workgroups up to head size 64 and of three or four
    beyond: two while every workgroup can have a unit, and further only beside long prompts (host code, answers without a GPU)."""
    import ctypes

    import pytest

    if not all(build.is_current(build.attention_module(d)) for d in (16, 64, 80, 128)):
        pytest.skip("the attention libraries are not built from the present sources")
    groups = {d: ctypes.CDLL(str(build.library_path(build.attention_module(d)))).mlr_attention_prefill_f32_groups for d in (16, 64, 80, 128)}
    for d in groups:  # (tiles, the longest prompt's, heads, window, chunk)
        assert groups[d](16, 1, 16, 0, 0) == 2 and groups[d](1, 1, 14, 0, 0) == 2  # 256 workgroups and fewer
        assert groups[d](32, 1, 16, 0, 0) == 1, "32 prompts of one tile"
        assert groups[d](32, 8, 16, 64, 0) == 1 and groups[d](32, 8, 16, 0, 64) == 1, "a window or chunk of a tile: chains of two"
        assert groups[d](17, 0, 16, 0, 0) == 1, "not known how long"
        assert groups[d](32, 8, 16, 0, 0) == 2, "one prompt of 2,048 tokens"
    assert groups[64](24, 3, 16, 0, 0) == 2 and groups[128](24, 3, 16, 0, 0) == 1  # 8 prompts of 130 tokens
    assert groups[64](128, 8, 16, 0, 0) == 2 and groups[80](128, 12, 16, 0, 0) == groups[16](128, 8, 16, 0, 0) == 1  # beyond two places a unit
    assert groups[16](128, 12, 16, 0, 0) == 2
    assert groups[64](40, 5, 16, 0, 0) == 1


def test_few_tokens_stream_whole_lines_where_that_is_faster():
    """Up to 16 tokens of matrices of 20 MB and more: the kernel that streams whole lines or the tiles, by the regions that measured slower through it
    (rows that meet modulo 64 KB, rows off a line, more than 8 tokens of many rows), and 2 slices where the norm adds them up one after the other."""
    import ctypes

    import pytest

    if not build.is_current(build.CORE):
        pytest.skip("the core library is not built from the present sources")
    lib = ctypes.CDLL(str(build.library_path(build.CORE)))
    for fn in (lib.mlr_gemm_bf16_kernel, lib.mlr_gemm_bf16_slices):
        fn.argtypes, fn.restype = [ctypes.c_int] * 4, ctypes.c_int
    lines = lambda m, n, k, most=8: lib.mlr_gemm_bf16_kernel(m, n, k, lib.mlr_gemm_bf16_slices(m, n, k, most)) == 16  # noqa: E731
    for m in (1, 4, 8, 12, 16):
        assert not any(lines(m, n, k) for n in (4096, 6144, 8064) for k in (8192, 12288, 20480, 11008)), m
        assert not lines(m, 3584, 24576) and not lines(m, 3584, 8192) and not lines(m, 3000, 22016)
        assert all(lines(m, n, k) for n in (3584, 6144) for k in (3584, 8320, 11136)), m
        assert all(lines(m, n, k) for n, k in ((2048, 24576), (2048, 11008), (3584, 12288), (3584, 18944), (4096, 14336), (5120, 5120)))
        assert not lines(m, 16384, 5848, 1) and lines(m, 16384, 3592, 1) and lines(m, 16384, 5632, 1)
        assert not lines(m, 201088, 2048, 1)
        assert lib.mlr_gemm_bf16_slices(m, 10240, 2816, 8) == 2 and 2 <= lib.mlr_gemm_bf16_slices(m, 8192, 2816, 8) <= 8
    assert lines(8, 20480, 4096 + 512, 1) and not lines(9, 20480, 4096 + 512, 1)
    assert lines(4, 152064, 2048, 1) and lines(4, 37888, 3584, 1) and not lines(5, 37888, 3584, 1)


def test_query_key_value_tiles_of_whole_heads():
    """The staged 128 x 128 tiles of the query/key/value product: from 80 tiles (128 of a long k) to two a unit, head sizes that divide 128, pages of eights, eight steps of k."""
    import ctypes

    import pytest

    if not build.is_current(build.CORE):
        pytest.skip("the core library is not built from the present sources")
    staged = ctypes.CDLL(str(build.library_path(build.CORE))).mlr_qkv_bf16_staged
    staged.argtypes, staged.restype = [ctypes.c_int] * 5, ctypes.c_int
    assert [staged(m, 1152, 896, 64, 16) for m in (64, 1024, 1025, 7168, 7169)] == [0, 0, 1, 1, 0]  # 72, 81, 504 and 513 tiles
    assert [staged(m, 4608, 3584, 128, 16) for m in (384, 385, 1792, 1793)] == [0, 1, 1, 0]  # 108, 144, 504 and 540
    assert staged(2048, 1152, 896, 64, 0) == staged(2048, 1152, 896, 64, 8) == 1  # no cache write, pages of 8 tokens
    assert staged(2048, 1152, 896, 64, 12) == staged(2048, 1152, 896, 48, 16) == staged(2048, 1152, 504, 64, 16) == staged(2048, 1152, 900, 64, 16) == 0
