"""The large products' matrix instructions are written in assembly, where the
compiler does not keep the two wait states between a vector instruction and a
matrix instruction that takes its result.  Here its output is looked over."""

import os
import re
import shutil
import subprocess

import pytest

from scaffold.ops import backend

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CSRC = os.path.join(backend._REPO_ROOT, "csrc")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("asm")
    with open(os.path.join(CSRC, "kernels", "big_gemm.hip")) as f:
        used = sorted(set(re.findall(r"launch<((?:true|false)[^>]*)>\(a", f.read())))
    assert used
    src = d / "k.hip"
    src.write_text(f'#include "{CSRC}/kernels/big_gemm.h"\n' + "".join(
        f"template __global__ void big::gemm_kernel<{t}>(BigArgs);\n" for t in used))
    out = d / "k.s"
    subprocess.run([HIPCC, *backend._HIPCC_FLAGS, "--cuda-device-only", "-S",
                    str(src), "-o", str(out)], check=True, capture_output=True)
    bodies = re.findall(r"^_ZN3big11gemm_kernel\w+:(.*?)^\.Lfunc_end",
                        out.read_text(), re.S | re.M)
    assert len(bodies) == len(used)
    return [[ln.split(";")[0].strip() for ln in b.splitlines()
             if re.match(r"\s+[a-z]", ln)] for b in bodies]


def _registers(text):
    """v1, v[2:5] -> their numbers"""
    out = set()
    for a, b, c in re.findall(r"\bv(?:(\d+)|\[(\d+):(\d+)\])", text):
        out |= {int(a)} if a else set(range(int(b), int(c) + 1))
    return out


def test_operands_are_not_fresh_from_vector_instructions(kernels):
    for body in kernels:
        seen = 0
        for i, ln in enumerate(body):
            if not ln.startswith("v_mfma"):
                continue
            seen += 1
            reads = _registers(ln.split(None, 1)[1])
            assert len(reads) == 8 and "a[" in ln          # sums lie in a[...]
            for back in (1, 2):
                before = body[i - back]
                if before.startswith("v_") and not before.startswith("v_mfma"):
                    to = before.split(None, 1)[1].split(",")[0]
                    assert not reads & _registers(to), (before, ln)
        assert seen >= 384


def test_sums_are_read_when_they_are_there(kernels):
    """18 wait states behind a matrix instruction, a jump's target counting as
    one that has not waited."""
    for body in kernels:
        since = 99
        for ln in body:
            if ln.startswith("v_mfma"):
                since = 0
            elif ln.startswith("s_nop"):
                since += int(ln.split()[1]) + 1
            else:
                if ln.startswith("v_accvgpr_read") or (
                        ln.startswith(("buffer_store", "ds_write")) and "a[" in ln):
                    assert since >= 18
                since += 1


def test_nothing_is_spilled(kernels):
    assert not any(ln.startswith("scratch_") for body in kernels for ln in body)
