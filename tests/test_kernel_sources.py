"""Inline assembly of the kernels, read as text: what a memory request delivers goes to LDS, never to a register.

The compiler takes an asm block's outputs as ready when the block ends.  A register that a load fills later can be copied or reused in
between, which no test would reliably show; LDS is not touched behind the kernel's back, and the kernels wait for their copies
themselves."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton_amd", "csrc")
LOADS = re.compile(r"\b(?:(?:buffer|global|flat|scratch)_load|ds_read|ds_load)\w*[^\n\"]*")


def asm_blocks(text):
    """Every asm statement: what stands between its parentheses, comments taken out."""
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r"\basm\s+volatile\s*\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            if c == '"' and text[i - 1] != "\\":
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            i += 1
        yield text[m.end():i - 1].replace("\\n", "\n").replace("\\t", " ")


def loads_to_registers(text):
    return [load for block in asm_blocks(text) for load in LOADS.findall(block) if not load.rstrip().endswith(" lds")]


def test_the_check_finds_them():
    assert loads_to_registers('asm volatile("s_nop 4\\n\\tbuffer_load_dword %0, %1, %2, 0 offen" : "=v"(v) : "v"(a), "s"(r));')
    assert not loads_to_registers('asm volatile("s_mov_b32 m0, %0\\n\\tbuffer_load_dword %1, %2, %3 offen lds" : : "s"(f(x)), "v"(a));')


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))), ids=os.path.basename)
def test_requests_deliver_to_lds(path):
    with open(path) as f:
        text = f.read()
    assert loads_to_registers(text) == []
    assert not re.search(r"\basm\s*\((?!\s*\))", re.sub(r"//[^\n]*", "", text)), "asm that is not volatile"


def test_barriers_wait_for_lds():
    """Every barrier is sync_threads(), whose wait for the wave's LDS accesses the compiler cannot take out."""
    bare = re.compile(r"\b__syncthreads\s*\(|\bs_barrier\b|__builtin_amdgcn_s_barrier")
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path) as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        if os.path.basename(path) == "common.h":
            at = re.search(r"void sync_threads\(\) \{\s*asm volatile\(\"s_waitcnt lgkmcnt\(0\)\" ::: \"memory\"\);\s*__syncthreads\(\);\s*\}", text)
            assert at
            text = text[:at.start()] + text[at.end():]
        assert not bare.findall(text), path


def test_stores_of_a_kernel_are_all_of_its_variant():
    """A kernel whose stores are non-temporal or not by a parameter makes all of them by it, also where scales are outside the fast range."""
    with open(os.path.join(CSRC, "mxfp.hip")) as f:
        kernels = re.findall(r"template <int DT, int GT, bool ONCE>\n__global__.*?\n}\n", re.sub(r"//[^\n]*", "", f.read()), re.S)
    assert len(kernels) == 2
    assert all(not re.search(r"\b(?:store_once|store16)\s*\((?:p\b|base\b)", k) for k in kernels)
