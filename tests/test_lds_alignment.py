"""Dynamic LDS is read 16 bytes at a time: every kernel's declaration asks for that alignment, whatever static LDS a kernel may come to have before it."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sofie_amd", "csrc")


def test_dynamic_lds_is_aligned():
    found = [(os.path.basename(path), line.strip()) for path in glob.glob(os.path.join(CSRC, "*.h*")) for line in open(path) if re.search(r"\bextern __shared__\b", line)]
    assert len(found) > 8
    assert not [f for f in found if "aligned(16)" not in f[1]]
