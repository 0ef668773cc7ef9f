"""What the kernels' own LLVM IR shows without a GPU: which memory a path reads,
and that accesses which must stay in order are ordered for the compiler.  The
sources are compiled here with the library's flags (device pass, IR as text)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mono-qwen27_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

pytestmark = pytest.mark.skipif(not shutil.which(HIPCC), reason="needs hipcc")


def kernel_blocks(tmp_path, source, kernel):
    """{label: lines} of one kernel of `source`, the entry block first."""
    ir = tmp_path / "kernel.ll"
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", CSRC, "--offload-device-only", "-S", "-emit-llvm", str(source), "-o",
                    str(ir)], check=True, capture_output=True, timeout=600)
    body = re.search(r"^define [^\n]*@\w*" + kernel + r"\w*\(([^\n]*)\{\n(.*?)^\}", ir.read_text(), re.M | re.S).group(2)
    blocks, label = {"": []}, ""
    for line in body.splitlines():
        m = re.match(r"(\d+):", line)
        if m:
            label = m.group(1)
            blocks[label] = []
        elif line.strip():
            blocks[label].append(line.strip())
    return blocks


def test_greedy_sampling_reads_the_first_index_alone(tmp_path):
    """temperature <= 0 gives idx[0]: the candidates behind it, their values and
    u are not read (a greedy caller need not have filled them)."""
    blocks = kernel_blocks(tmp_path, os.path.join(CSRC, "m27q_topk.hip"), "8k_sample")
    hot, seen, todo, loads = {}, set(), [""], []  # arguments: %0 idx, %1 val, %2 k, %3 temperature, ...
    while todo:
        b = todo.pop()
        if b in seen:
            continue
        seen.add(b)
        for line in blocks[b]:
            m = re.match(r"(%\d+) = fcmp .*\b(ogt|ugt|ole|ule) float %3, 0\.0", line)
            if m:
                hot[m.group(1)] = m.group(2) in ("ogt", "ugt")
            if re.search(r"= load ", line):
                loads.append(re.search(r"load \w+, ptr addrspace\(1\) (%\d+)", line).group(1))
            m = re.match(r"br i1 (%\d+), label %(\d+), label %(\d+)", line)
            if m:  # the branch on the temperature: the side of temperature <= 0 alone
                todo += [m.group(2 + hot[m.group(1)])] if m.group(1) in hot else [m.group(2), m.group(3)]
            elif line.startswith("br label"):
                todo.append(re.match(r"br label %(\d+)", line).group(1))
    assert hot and loads == ["%0"], loads


@pytest.mark.parametrize("wt,nt,layout", [("WQ80", 1, 0), ("WQ4K<false>", 2, 1), ("WQ6K", 4, 0)])
def test_one_wave_slices_order_their_lds_accesses(tmp_path, wt, nt, layout):
    """Wide products with one wave per slice of K: lanes hand activations to each
    other through LDS without a barrier, so on every path a fence must stand
    between an LDS write and the next read, and between a read and the next
    write; otherwise the compiler may swap two whose own-lane addresses differ."""
    src = tmp_path / "few.hip"
    src.write_text('#include "m27q_wide.h"\nnamespace m27q {\nhipError_t one(const MatmulMultiParams &p, hipStream_t s) '
                   "{ return launch_wide_t<%s, %d, ShapeFew, %d>(p, 1, s); }\n}\n" % (wt, nt, layout))
    blocks = kernel_blocks(tmp_path, src, "13k_matmul_wide")
    state = {b: set() for b in blocks}  # the LDS accesses that may be the last ones at a block's entry
    state[""] = {""}
    todo, accesses, swaps = [""], 0, []
    while todo:
        b = todo.pop()
        now = set(state[b])
        for line in blocks[b]:
            if line.startswith("fence "):
                now = {""}
            elif "addrspace(3)" in line and re.match(r"(store|%\d+ = load) ", line):
                kind = "store" if line.startswith("store") else "load"
                accesses += 1
                if now - {"", kind}:
                    swaps.append((b, line))
                now = {kind}
        for t in re.findall(r"label %(\d+)", blocks[b][-1] if blocks[b][-1].startswith("br ") else ""):
            if not now <= state[t]:
                state[t] |= now
                todo.append(t)
    assert accesses > 20 and not swaps, swaps[:4]
