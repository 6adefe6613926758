"""What the kernels' sources must keep and no run shows: an ordering that the
compiler may drop without changing today's results."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cgdycore.jl_amd", "csrc")


@pytest.mark.parametrize("name,store,read", [
    ("cgd_pass2_body.inc", r"mt\[11 \* NN \+ node\] = ", r"-D122 \* w|\bD\d\d\d \* "),
    ("cgd_pass2r_body.inc", r"mt\[4 \* NN \+ node\] = ", r"= mt\[nodeC\]"),
])
def test_metric_table_is_fenced(name, store, read):
    """The per-node metric table in LDS is stored by one lane of a node and
    first read by the others before any barrier: the fence lies between."""
    with open(os.path.join(CSRC, name)) as f:
        src = f.read()
    s = re.search(store, src).end()
    r = s + re.search(read, src[s:]).start()
    assert "wave_lds_fence();" in src[s:r]
    assert "__syncthreads" not in src[s:r]
