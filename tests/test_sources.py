"""The kernels' sources: what several of them share is written once."""
import glob
import os
import re
from collections import Counter

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vlm_training_amd", "csrc")


def test_a_struct_is_defined_once():
    """Launch functions pass structs between files with C linkage: two definitions that differ would compile, link and be read wrongly."""
    found = Counter()
    for path in glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.cpp")):
        with open(path) as f:
            found.update(re.findall(r"^\s*(?:template\s*<[^>]*>\s*)?struct\s+(\w+)\s*\{", f.read(), re.M))
    assert found["DqBeside"] == 1 and [name for name, n in found.items() if n > 1] == []
