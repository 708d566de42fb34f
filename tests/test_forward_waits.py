"""The compiled forward kernels: what has arrived in LDS in front of their first step."""
import os
import re
import shutil
import subprocess

from tests.test_key_side import OBJDUMP
from vlm_training_amd import _lib


def _meetings(code):
    """Of each barrier of a function, in program order: requests into LDS since the one before (16 bytes a lane), the wait in front of it."""
    met, loads, wait = [], 0, None
    for line in code:
        text = line.partition("//")[0].strip()
        if text.startswith("buffer_load_dwordx4") and text.endswith("lds"):
            loads += 1
        elif text.startswith("s_waitcnt") and "vmcnt" in text:
            wait = int(re.search(r"vmcnt\((\d+)\)", text).group(1))
        elif text.startswith("s_barrier"):
            met.append((loads, wait))
            loads, wait = 0, None
    return met


def _late_first_tiles(met):
    """A block that staged its rows of q requests V(0), V(1) and V(2) between its first two barriers.  Step 0 reads V(0) and the first operands of
    V(1): behind the second barrier V(2) alone may be on its way, a third of the requests."""
    loads, wait = met[1]
    return loads > 0 and (loads % 3 != 0 or wait is None or wait > loads // 3)


def test_checker_sees_a_first_step_that_does_not_wait_for_its_second_tile():
    head = ["buffer_load_dwordx4 v1, s[4:7], 0 offen lds"] * 4 + ["s_waitcnt vmcnt(4)", "s_barrier"] + ["buffer_load_dwordx4 v1, s[4:7], 0 offen lds"] * 6
    for wait, late in (("s_waitcnt vmcnt(4)", True), ("s_waitcnt lgkmcnt(0)", True), ("s_waitcnt vmcnt(2)", False), ("s_waitcnt vmcnt(0) lgkmcnt(0)", False)):
        assert _late_first_tiles(_meetings(head + [wait, "s_barrier"])) is late, wait


def test_first_tiles_of_the_forward_are_there_before_they_are_read(tmp_path):
    lib = shutil.copy(_lib.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    staged, late = 0, []
    for name in sorted(os.listdir(tmp_path)):
        path = tmp_path / name
        if not name.endswith("gfx950") or b"dsa_tile_fwd_kernel" not in path.read_bytes():
            continue
        listing = subprocess.run([OBJDUMP, "-d", str(path)], check=True, capture_output=True, text=True).stdout
        for function in re.split(r"\n(?=[0-9a-f]+ <_Z)", listing):
            kernel = re.match(r"[0-9a-f]+ <(_Z\w*dsa_tile_fwd_kernel\w*)>:", function)
            if kernel:
                met = _meetings(function.splitlines())
                staged += met[1][0] > 0
                if _late_first_tiles(met):
                    late.append((kernel.group(1), met[:3]))
    assert staged >= 12 and not late, (staged, late[:3])
