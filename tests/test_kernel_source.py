"""What the kernels' sources must keep and no run shows: an ordering that the
compiler may drop without changing today's results, and the chunk heights that a
kernel's use of its registers allows."""
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


@pytest.mark.parametrize("kernel", ["k_tr2", "k_tr2_lim"])
def test_tracer_heights_are_bounded(kernel):
    """A lane's halo levels below and above share registers: a chunk of 3
    levels would have a lane with second neighbours outside on both sides."""
    with open(os.path.join(CSRC, "cgd_kernels.hip")) as f:
        src = f.read()
    body = src[re.search(rf"\n[^\n]*\b{kernel}\(KArgs", src).end():]
    lowest = int(re.search(r"static_assert\(NZT >= (\d+)", body[:body.index("\n}\n")]).group(1))
    assert not any(l < 2 and l + 2 >= z for z in range(lowest, 17) for l in range(z))
