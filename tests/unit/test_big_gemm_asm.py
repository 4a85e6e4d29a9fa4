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
    return [Body(b) for b in bodies]


class Body:
    """A kernel's instructions, and for each those that may come next."""

    def __init__(self, text):
        self.lines, labels = [], {}
        for ln in text.splitlines():
            ln = ln.split(";")[0].strip()
            if re.match(r"\.L\w+:", ln):
                labels[ln[:-1]] = len(self.lines)
            elif re.match(r"[a-z]", ln):
                self.lines.append(ln)
        self.next = []
        for i, ln in enumerate(self.lines):
            op, *to = ln.split()
            assert not re.match(r"s_(setpc|swappc|call|cbranch_[ig]_|rfe)", op), ln
            after = [labels[to[0]]] if re.match(r"s_c?branch", op) else []
            if op not in ("s_branch", "s_endpgm"):
                after.append(i + 1)
            self.next.append(after)

    def before(self, first, step, join):
        """What holds ahead of each instruction, over all ways there: first at
        the start, step(instruction, that) behind one, joined where ways meet."""
        held = {0: first}
        todo = [0]
        while todo:
            i = todo.pop()
            behind = step(self.lines[i], held[i])
            for n in self.next[i]:
                new = join(held[n], behind) if n in held else behind
                if n not in held or new != held[n]:
                    held[n] = new
                    todo.append(n)
        return [held.get(i) for i in range(len(self.lines))]


def _registers(text, kind="v"):
    """v1, v[2:5] -> their numbers"""
    out = set()
    for a, b, c in re.findall(rf"\b{kind}(?:(\d+)|\[(\d+):(\d+)\])", text):
        out |= {int(a)} if a else set(range(int(b), int(c) + 1))
    return out


def _states(ln):
    return int(ln.split()[1]) + 1 if ln.startswith("s_nop") else 1


def _written(ln):
    """The vector registers that a vector instruction, and no matrix one, writes."""
    if not ln.startswith("v_") or ln.startswith("v_mfma"):
        return set()
    # a swap writes both
    to = ln.split(None, 1)[1].split(",")[:2 if "swap" in ln else 1]
    return _registers(",".join(to))


def test_operands_are_not_fresh_from_vector_instructions(kernels):
    for body in kernels:
        def step(ln, fresh):                       # {(register, states since)}
            n = _states(ln)
            return (frozenset((r, s + n) for r, s in fresh if s + n < 2)
                    | frozenset((r, 0) for r in _written(ln)))

        held = body.before(frozenset(), step, lambda a, b: a | b)
        seen = 0
        for ln, fresh in zip(body.lines, held):
            if not ln.startswith("v_mfma") or fresh is None:
                continue
            seen += 1
            reads = _registers(ln.split(None, 1)[1])
            assert len(reads) == 8 and "a[" in ln          # sums lie in a[...]
            assert not reads & {r for r, _ in fresh}, ln
        assert seen >= 384


def test_sums_are_read_when_they_are_there(kernels):
    """Between a matrix instruction and whatever else names a sum's register lie
    18 wait states, on each way from one to the other, that are there for that:
    other instructions, which a compiler may move, are not counted."""
    for body in kernels:
        sums = set().union(*(_registers(ln.split(",")[0], "a") for ln in body.lines
                             if ln.startswith("v_mfma")))
        assert len(sums) >= 192

        def step(ln, waited):
            if ln.startswith("v_mfma"):
                return 0
            return min(99, waited + (_states(ln) if ln.startswith("s_nop") else 0))

        held, seen = body.before(99, step, min), 0
        for ln, waited in zip(body.lines, held):
            if waited is None or ln.startswith("v_mfma"):
                continue
            if _registers(ln.split(None, 1)[-1], "a") & sums:
                seen += 1
                assert waited >= 18, ln
        assert seen >= len(sums) / 4


def test_ways_are_followed():
    """Both ways to a jump's target count, and a loop's edge."""
    body = Body("""
        s_branch .LBB0_2
    .LBB0_1:
        s_nop 15
    .LBB0_2:
        v_mov_b32 v0, v1
        v_mfma_x a[0:3], v[0:3], v[4:7], a[0:3]
        s_cbranch_scc1 .LBB0_2
        s_cbranch_scc0 .LBB0_1
        s_endpgm
    """)
    held = body.before(99, lambda ln, n: 7 if "mfma" in ln else
                       min(99, n + 16 * ("nop" in ln)), min)
    assert held == [99, 7, 7, 7, 7, 7, 7]


def test_nothing_is_spilled(kernels):
    assert not any(ln.startswith("scratch_") for body in kernels for ln in body.lines)
