"""The compacted walks' lists: written as words, read by halves."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vlm_training_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


def _typed_halves(ir):
    """(16-bit reads of LDS, those that the compiler may move past a write of words: type-based aliasing calls them short)."""
    node = {m.group(1): m.group(2) for m in re.finditer(r"^!(\d+) = (.*)$", ir, re.M)}
    reads = re.findall(r"= load (?:volatile )?i16, ptr addrspace\(3\) [^\n]*", ir)
    tags = [re.search(r"!tbaa !(\d+)", r) for r in reads]
    typed = [t for t in tags if t and '"omnipotent char"' not in node[re.match(r"!\{!(\d+)", node[t.group(1)]).group(1)]]
    return len(reads), len(typed)


def test_checker_sees_a_typed_read():
    ir = '%1 = load i16, ptr addrspace(3) %0, align 2, !tbaa !{}\n!1 = !{{!2, !2, i64 0}}\n!2 = !{{!"short", !3, i64 0}}\n!3 = !{{!"omnipotent char", !4, i64 0}}\n!5 = !{{!3, !3, i64 0}}\n'
    assert _typed_halves(ir.format(1)) == (1, 1) and _typed_halves(ir.format(5)) == (1, 0)


@pytest.mark.parametrize("source", ["dsa_tile_sel.hip", "dsa_tile_selkv.hip"])
def test_halves_of_a_list_entry_are_read_behind_its_words(source, tmp_path):
    """An entry is stored whole: a read of its half typed `short` may be moved in front of that store."""
    ir = tmp_path / "walk.ll"
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only",
                    "-S", "-emit-llvm", os.path.join(CSRC, source), "-o", str(ir)], check=True, capture_output=True)
    reads, typed = _typed_halves(ir.read_text())
    assert reads > 0 and typed == 0, (reads, typed)
