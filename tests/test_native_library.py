"""The layer that compiles and loads the HIP libraries (no GPU needed: hipcc cross-compiles, nothing is run).

What is checked here is how it fails and when it builds again: there is no other path than the compiled kernels, so a
missing compiler or a source that does not compile has to say so, at once and by name.
"""
import os
import re
import subprocess

import pytest

from nanohybrid_vlm_amd.native import library


@pytest.fixture
def sandbox(tmp_path, monkeypatch):
    """Sources and libraries in a temporary folder of their own."""
    csrc, lib_dir = tmp_path / "csrc", tmp_path / "lib"
    csrc.mkdir()
    lib_dir.mkdir()
    (csrc / "common.h").write_text("#pragma once\n#define ANSWER 42\n")
    (csrc / "good.hip").write_text('#include "common.h"\nextern "C" int answer() { return ANSWER; }\n')
    monkeypatch.setattr(library, "CSRC", str(csrc))
    monkeypatch.setattr(library, "LIB_DIR", str(lib_dir))
    monkeypatch.setattr(library, "_loaded", {})
    return csrc, lib_dir


def test_a_missing_compiler_is_named(sandbox, monkeypatch):
    monkeypatch.setattr(library.shutil, "which", lambda name: None)
    monkeypatch.setattr(library.os.path, "isfile", lambda path: False if path.endswith("hipcc") else os.path.exists(path))
    with pytest.raises(library.NativeBuildError, match="hipcc was not found"):
        library.build_library("probe", ["good.hip"])


def test_a_source_that_does_not_compile_shows_the_compiler_s_words(sandbox):
    csrc, lib_dir = sandbox
    (csrc / "bad.hip").write_text('extern "C" int broken() { return no_such_name; }\n')
    with pytest.raises(library.NativeBuildError) as err:
        library.build_library("probe", ["good.hip", "bad.hip"])
    assert "bad.hip" in str(err.value) and "no_such_name" in str(err.value)
    assert not [f for f in os.listdir(lib_dir) if f.endswith(".so")], "nothing half-built is left behind"
    assert not [f for f in os.listdir(lib_dir) if f.startswith("nhv_build_")], "the work folder is gone"


def test_built_once_and_again_when_a_source_or_a_header_changes(sandbox):
    csrc, lib_dir = sandbox
    first = library.build_library("probe", ["good.hip"])
    assert os.path.dirname(first) == str(lib_dir) and os.path.isfile(first)
    stamp = os.stat(first).st_mtime_ns
    assert library.build_library("probe", ["good.hip"]) == first and os.stat(first).st_mtime_ns == stamp, "found, not built again"
    # the same sources under another name and with another define (the attention kernels: a library per head size)
    other = library.build_library("probe_d2", ["good.hip"], ["-DOTHER=1"])
    assert other != first and os.path.isfile(first) and os.path.isfile(other)
    # a changed header means new libraries, and those of the old sources are cleared away
    (csrc / "common.h").write_text("#pragma once\n#define ANSWER 43\n")
    second = library.build_library("probe", ["good.hip"])
    assert second != first and os.path.isfile(second) and not os.path.exists(first) and os.path.isfile(other)
    lib = library.load_library("probe", ["good.hip"])
    assert lib.answer() == 43                       # host code only: nothing here touches a GPU
    assert library.load_library("probe", ["good.hip"]) is lib


def test_the_wait_for_x_has_the_loads_behind_it_that_it_counts(tmp_path):
    """The few-rows products wait for their rows of x by the number of loads asked for since (``wait_for_x``). The weights'
    pointer must be one whose loads cannot legally leave their place (no ``__restrict__``), and in what the compiler makes of each
    kernel so many loads must stand between the last one of x and the wait."""
    source = os.path.join(library.CSRC, "gemm_fewrows_bf16.hip")
    text = open(source).read()
    for kernel in ("gemm_fewrows_tile_kernel", "gemm_fewrows_walk_kernel"):
        arguments = re.search(r"void %s\((.*?)\{" % kernel, text, re.S)[1]
        assert re.search(r"const bf16_t\s*\*\s*w\b", arguments), arguments
    out = tmp_path / "fewrows.s"
    subprocess.run([library._hipcc(), *[f for f in library.HIPCC_FLAGS if f != "-fPIC"], "-I", library.CSRC, "--cuda-device-only", "-S",
                    source, "-o", str(out)], check=True, capture_output=True)
    listing, seen = out.read_text(), 0
    name = re.compile(r"^(\S*gemm_fewrows_(tile|walk)_kernelILi(\d+)ELb([01])ELb([01])\S*):", re.M)
    for m in name.finditer(listing):
        if m[2] == "tile" and m[5] == "0":
            continue                                     # (x does not lie in LDS: nothing to wait for)
        body = listing[m.end():listing.index(".Lfunc_end", m.end())].split("\n")
        ops = [" ".join(line.split(";")[0].split()) for line in body]
        last = max(i for i, op in enumerate(ops) if "global_load_lds" in op)
        barrier = next(i for i in range(last, len(ops)) if ops[i].startswith("s_barrier"))
        between = ops[last + 1:barrier]
        waits = [int(n) for op in between for n in re.findall(r"vmcnt\((\d+)\)", op)]
        loads = sum(op.startswith("global_load") for op in between)
        assert waits == [int(m[3]) * (2 if m[4] == "1" else 1)] and loads >= waits[0], (m[1], waits, loads)
        assert not any(op.startswith(("scratch", "buffer", "flat", "global_store")) for op in between), m[1]
        seen += 1
    assert seen >= 50, seen


@pytest.mark.parametrize("D,tiles,blocks", [(48, 2, 3), (64, 1, 4), (80, 1, 3), (96, 1, 3)])
def test_the_prompts_attention_leaves_registers_for_the_blocks_that_fit(tmp_path, D, tiles, blocks):
    """Where LDS has room for three or four blocks of four waves a compute unit, a SIMD's 512 registers a lane have room for as many
    waves, and nothing is kept in memory instead: heads of these sizes, so many row tiles a wave, without cap or bias."""
    source, out = os.path.join(library.CSRC, "attention_prefill_bf16.hip"), tmp_path / "attention.s"
    subprocess.run([library._hipcc(), *[f for f in library.HIPCC_FLAGS if f != "-fPIC"], f"-DNHV_HEAD_DIM={D}", "-I", library.CSRC,
                    "--cuda-device-only", "-S", source, "-o", str(out)], check=True, capture_output=True)
    text, seen = out.read_text(), 0
    for name, registers in re.findall(r"\.set (\S*prefill_attention_kernelILb[01]ELi%dELb[01]ELb0ELb0E\S*?)\.num_vgpr, (\d+)" % tiles, text):
        scratch = re.search(re.escape(name) + r"\.private_seg_size, (\d+)", text)
        assert int(registers) <= 512 // blocks // 8 * 8 and scratch[1] == "0", (name, registers, scratch[1])
        seen += 1
    assert seen == 4


def test_no_scalar_offset_of_the_gates_kernel_lies_behind_its_rows(tmp_path):
    """Of a tile that is cut off at the end, the rows behind it are kept out by the descriptor's size, with which the lane's offset is
    compared after the scalar offset has been taken from it: that one must not be the larger. In what the compiler makes of each kernel
    every load to LDS has a scalar offset that has just been cut off at the size in its own descriptor."""
    source, out = os.path.join(library.CSRC, "gemm_phases_bf16.hip"), tmp_path / "phases.s"
    subprocess.run([library._hipcc(), *[f for f in library.HIPCC_FLAGS if f != "-fPIC"], "-I", library.CSRC, "--cuda-device-only", "-S",
                    source, "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"^(\S*gemm_phases_kernel\S*):[^\n]*\n(.*?)^\.Lfunc_end", out.read_text(), re.M | re.S)
    assert len(kernels) == 6
    for name, body in kernels:
        ops = [op for op in (" ".join(line.split(";")[0].split()) for line in body.split("\n")) if op]
        copies, loads = {}, 0
        for i, op in enumerate(ops):
            if re.match(r"\S+:$", op):                    # (where ways meet, only what is true on both would count)
                copies = {}
            if move := re.match(r"s_mov_b32 (s\d+), (s\d+)$", op):
                copies[move[1]] = copies.get(move[2], move[2])
            elif written := re.match(r"s_\S+ s(\d+|\[\d+:\d+\]),", op):
                first, last = (re.findall(r"\d+", written[1]) * 2)[:2] if "[" not in written[1] else re.findall(r"\d+", written[1])
                for n in range(int(first), int(last) + 1):
                    copies = {k: v for k, v in copies.items() if f"s{n}" not in (k, v)}
            if op.startswith("buffer_load") and op.endswith("lds"):
                rows, offset = re.match(r"buffer_load_dwordx4 v\d+, s\[(\d+):\d+\], (s\d+) offen lds$", op).groups()
                cut = re.match(r"s_min_u32 (s\d+), (s\d+), (s\d+)$", ops[i - 1])
                assert cut and cut[1] == offset, (name, ops[i - 3:i + 1])
                size = f"s{int(rows) + 2}"
                assert size in (cut[3], copies.get(cut[3])) or copies.get(size, size) == copies.get(cut[3], cut[3]), (name, ops[i - 3:i + 1])
                loads += 1
        assert loads >= 32, (name, loads)


@pytest.mark.parametrize("blocks", [1, 8, 64, 184, 192, 200, 256, 264, 320, 352, 360, 416, 424, 512, 1024, 4096])
def test_no_block_of_the_decode_attention_takes_a_long_context_alone(blocks):
    """However long the longest context and however many blocks there are: the splits cover it, and no block's chain of keys is longer
    than 2,048, or 6,144 where the whole context is one split. A window's tokens are split by what they read."""
    from nanohybrid_vlm_amd.native.ops import decode_split_length
    for covered in (1, 31, 300, 448, 449, 672, 1000, 2048, 3072, 4096, 4097, 6144, 6145, 12288, 48000, 196608, 1000000):
        for span in {covered, max(1, covered * 2 // 3)}:
            for window in (0, 100, 1024, -1024, 8192):
                seen = min(span, abs(window) + 64) if window else span
                split = decode_split_length(blocks, seen, covered, window)
                n = -(-covered // split)
                assert split > 0 and split % 32 == 0 and n <= 65535
                read = min(covered, abs(window) + 64) if window else covered
                assert min(split, read) <= (2048 if n > 1 else 6144), (covered, span, window, split)
    assert decode_split_length(8, 1088, 48000, 1024) <= 256        # (one token of 8 key/value heads deep in a context)
