"""No wave passes a workgroup barrier with LDS accesses of its own outstanding.

s_barrier waits for no memory access and on gfx950 the compiler adds no wait before the
builtin, so a hand-over through LDS needs its own s_waitcnt lgkmcnt(0).  A missing one shows
in no result as long as the timing hides it; here the compiler's device assembly is followed
along every path, counting the LDS operations that may be outstanding."""
from __future__ import annotations

import re
import subprocess
from pathlib import Path

import pytest

from conftest import PKG_DIR

HIPCC = Path("/opt/rocm/bin/hipcc")
pytestmark = pytest.mark.skipif(not HIPCC.exists(), reason="no device compiler")
# operations of the LDS counter that touch no LDS memory
NO_MEMORY = {"ds_bpermute_b32", "ds_permute_b32", "ds_swizzle_b32"}
CAP = 64  # outstanding operations told apart


def device_assembly(tmp_path, source: Path) -> str:
    """The source compiled for the device with the flags of its Makefile."""
    names = "$(HIPFLAGS)" if source.parent.name == "engine" else "$(DEVICE) $(NUMERIC) $(CXXFLAGS)"
    flags = subprocess.run(["make", "-s", "--no-print-directory", "-C", str(source.parent),
                            "--eval", f"flags: ; @echo '{names}'", "flags"],
                           capture_output=True, text=True, check=True).stdout.split()
    out = tmp_path / (source.stem + ".s")
    subprocess.run([str(HIPCC), *flags, "--cuda-device-only", "-S", source.name, "-o", str(out)], check=True,
                   cwd=source.parent, capture_output=True, timeout=300)
    return out.read_text()


def functions(text: str) -> dict[str, list[str]]:
    """Function name -> its instructions and .LBB labels."""
    found, current = {}, None
    for line in text.splitlines():
        label = re.match(r"([A-Za-z_.][\w.$]*):", line)
        if line.startswith(".Lfunc_end"):
            current = None
        elif label and not label[1].startswith("."):
            current = found.setdefault(label[1], [])
        elif current is not None:
            code = label[0] if label and label[1].startswith(".LBB") else line.split(";")[0].strip()
            if code and (code.startswith(".LBB") or not code.startswith(".")):
                current.append(code)
    return found


def advance(code: str, outstanding: int) -> int:
    op = code.split()[0]
    if (op.startswith("ds_") and op not in NO_MEMORY) or op.startswith("flat_"):
        return min(outstanding + 1, CAP)
    count = re.search(r"lgkmcnt\((\d+)\)", code) if op == "s_waitcnt" else None
    return min(outstanding, int(count[1])) if count else outstanding


def at_barriers(body: list[str]) -> list[int]:
    """For every s_barrier the most LDS operations outstanding at it on any path."""
    blocks, labels = [[]], {}
    for code in body:
        if code.startswith(".LBB"):
            blocks.append([])
            labels[code[:-1]] = len(blocks) - 1
            continue
        blocks[-1].append(code)
        if re.match(r"s_(c?branch|endpgm|setpc)", code):
            blocks.append([])

    def successors(b):
        last = blocks[b][-1] if blocks[b] else ""
        jump = re.match(r"s_c?branch\S*\s+(\S+)", last)
        if jump:
            yield labels[jump[1]]
        if not re.match(r"s_(branch|endpgm|setpc)", last) and b + 1 < len(blocks):
            yield b + 1

    entry = {0: 0}
    work = [0]
    while work:
        b = work.pop()
        n = entry[b]
        for code in blocks[b]:
            n = advance(code, n)
        for s in successors(b):
            if n > entry.get(s, -1):
                entry[s] = n
                work.append(s)
    seen = []
    for b, n in entry.items():
        for code in blocks[b]:
            if code.split()[0] == "s_barrier":
                seen.append(n)
            n = advance(code, n)
    return seen


def test_counting():
    """The count follows branches, loops and partial waits."""
    loop = ["ds_write_b32 v0, v1", "s_cbranch_scc1 .LBB0_1", "s_waitcnt lgkmcnt(0)", ".LBB0_1:", "s_barrier",
            "ds_read_b32 v0, v1", "ds_read_b32 v2, v1", "s_waitcnt vmcnt(0) lgkmcnt(1)", "s_cbranch_scc1 .LBB0_1",
            "s_endpgm"]
    assert at_barriers(loop) == [1]
    assert at_barriers(["ds_write_b32 v0, v1", "s_waitcnt lgkmcnt(0)", "ds_bpermute_b32 v0, v0, v1", "s_barrier"]) == [0]


# the sources that use the builtin, themselves or through a header (__syncthreads brings its waits)
SOURCES = ["csrc/bnn_gemm.hip", "csrc/bnn_fused.hip", "csrc/bnn_rows.hip", "csrc/bnn_chain.hip", "engine/resident.hip"]


@pytest.mark.parametrize("source", SOURCES)
def test_barriers(tmp_path, source):
    checked = 0
    for name, body in functions(device_assembly(tmp_path, PKG_DIR / source)).items():
        counts = at_barriers(body)
        assert not any(counts), (name, counts)
        checked += len(counts)
    assert checked


def test_every_source_is_checked():
    texts = {p.relative_to(PKG_DIR): p.read_text() for p in PKG_DIR.rglob("*.h*") if p.suffix in (".hip", ".h")}
    headers = {p.name for p, text in texts.items() if p.suffix == ".h" and "__builtin_amdgcn_s_barrier" in text}
    users = {str(p) for p, text in texts.items() if p.suffix == ".hip" and (
        "__builtin_amdgcn_s_barrier" in text or any(h in text and "lds_barrier" in text for h in headers))}
    assert users == set(SOURCES)
