"""The wait states that inline assembly has to bring itself, checked in the disassembly of the built kernels.

A vector-memory instruction that reads a scalar register has to stay five wait states behind a vector instruction that
wrote it (v_readlane, v_readfirstlane, a compare).  The compiler keeps that distance for its own instructions; it does not
look into assembly statements, and a scalar that it had spilled to a vector lane comes back right in front of one."""
import os
import re
import shutil
import subprocess

import pytest

from flashoverlap_amd import _capi, build

OBJDUMP = os.path.join(os.path.dirname(os.path.dirname(build.HIPCC)), "llvm", "bin", "llvm-objdump")
STATES = 5


def scalars(text):
    """Scalar registers named in an operand list."""
    found = set()
    for a, b, single in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        found |= {int(single)} if single else set(range(int(a), int(b) + 1))
    return found


def too_close(lines):
    """(kernel, writer, reader) wherever a vector-memory instruction reads a scalar fewer than STATES wait states after
    a vector instruction wrote it."""
    kernel, recent, bad = "", [], []  # recent: (wait states since, scalars written by a vector instruction, text)
    for line in lines:
        line = line.split("//")[0].strip()
        if line.endswith(">:"):
            kernel = line.split("<")[1][:-2]
            recent = []
            continue
        op, _, rest = line.partition(" ")
        if not re.match(r"[a-z]+_[a-z0-9_]+$", op):
            continue
        if re.match(r"(buffer|global|flat|scratch)_", op):
            reads = scalars(rest)
            bad += [(kernel, text, line) for _, wrote, text in recent if wrote & reads]
        states = int(rest, 0) + 1 if op == "s_nop" else 1
        first = rest.split(",")[0]
        recent = [(since + states, wrote - scalars(first) if op.startswith("s_") else wrote, text)
                  for since, wrote, text in recent if since + states < STATES]
        if op.startswith("v_") and scalars(first):
            recent.append((0, scalars(first), line))
        if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
            recent = []
    return bad


def vectors(text):
    """Vector registers named in an operand list."""
    found = set()
    for a, b, single in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        found |= {int(single)} if single else set(range(int(a), int(b) + 1))
    return found


def used_in_flight(lines):
    """(kernels seen, loads seen, [(kernel, load, user)]) of the 256x256 kernel's loads of group sizes and slots, which are assembly: no
    instruction may name their registers in front of the fill's wait."""
    kernel, flying, kernels, loads, bad = "", None, 0, 0, []
    for line in lines:
        line = line.split("//")[0].strip()
        if line.endswith(">:"):
            kernel = line.split("<")[1][:-2]
            flying = {} if "fo_gemm256_kernel" in kernel else None
            kernels += flying is not None
        elif flying is None:
            continue
        elif re.match(r"s_waitcnt vmcnt\(16\)", line):
            flying = None
        else:
            op, _, rest = line.partition(" ")
            named = vectors(rest)
            bad += [(kernel, text, line) for register, text in flying.items() if register in named]
            load = re.match(r"global_load_dword v(\d+), v\[\d+:\d+\], off$", line)
            if load:
                flying[int(load.group(1))] = line
                loads += 1
    return kernels, loads, bad


def test_the_check_sees_a_register_used_in_flight():
    start, load, wait = "0 <fo_gemm256_kernel>:", "global_load_dword v7, v[2:3], off", "s_waitcnt vmcnt(16)"
    assert used_in_flight([start, load, "v_add_u32_e32 v1, v7, v2", wait])[2] == [("fo_gemm256_kernel", load, "v_add_u32_e32 v1, v7, v2")]
    assert used_in_flight([start, load, "ds_read_b128 v[4:7], v1", wait])[2] != []
    assert used_in_flight([start, load, "v_add_u32_e32 v1, v8, v2", wait, "v_add_u32_e32 v1, v7, v2"]) == (1, 1, [])


def test_the_check_sees_what_it_looks_for():
    write, read = "v_readlane_b32 s18, v93, 24", "buffer_load_dwordx4 v62, s[52:55], s18 offen lds"
    assert too_close([write, "s_mov_b32 m0, s75", "s_nop 0", read]) == [("", write, read)]
    assert too_close([write, "s_mov_b32 m0, s75", "s_nop 2", read]) == [("", write, read)]
    assert too_close([write, "s_mov_b32 m0, s75", "s_nop 3", read]) == []
    assert too_close([write, "s_add_u32 s18, s18, 4", read]) == []   # the vector instruction's value is gone
    assert too_close([write, "s_branch 12", read]) == []
    assert too_close(["v_readfirstlane_b32 s53, v1", read]) != []


def test_scalar_operands_of_vector_memory_instructions(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump beside hipcc")
    shutil.copy2(_capi.KERNEL_LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    parts = [p for p in sorted(os.listdir(tmp_path)) if p.endswith(build.ARCH)]
    assert parts
    loads, bad, kernels, requests = 0, [], 0, 0
    for part in parts:
        text = subprocess.run([OBJDUMP, "-d", part], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        loads += len(re.findall(r"buffer_load_dwordx4.* lds", text))
        bad += too_close(text.splitlines())
        found = used_in_flight(text.splitlines())
        kernels, requests, bad = kernels + found[0], requests + found[1], bad + found[2]
    assert loads > 1000  # the operand loads of the GEMM kernels
    assert kernels == 2 * 8 and requests >= 2 * 7 and bad == []
