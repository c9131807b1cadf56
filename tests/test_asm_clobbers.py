"""Inline assembly of the kernels names every register that it writes by name."""
import glob
import os
import re

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_m0_is_a_clobber_where_it_is_written():
    found = 0
    for path in glob.glob(os.path.join(REPO, "distributed-lb-ib_amd", "csrc", "*.h*")):
        for block in re.findall(r"\basm\s+volatile\s*\((.*?)\);", open(path).read(), re.S):
            if re.search(r"\bs_\w+\s+m0\b", block):
                found += 1
                assert re.search(r":[^:]*\"m0\"[^:]*$", block), (os.path.basename(path), block)
    assert found
