"""What the library's host code launches and how it keeps its scratch, on a
HIP runtime that only records (fake_hip.cpp): no GPU, nothing computed."""
import pytest

import fakehip


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fakehip.build(tmp_path_factory.mktemp("fake_hip"))


def new_allocs(before, after):
    """Indices of the allocations that a step made."""
    return range(len(before["allocs"]), len(after["allocs"]))


# A graph captured after an eager call holds the scratch's addresses: a later
# call that needs more must not free it.  The argmax's pairs share their buffer
# with the tile GEMM's partial sums, so a prompt whose K is split grows it.
@pytest.mark.parametrize("grow", [["gemm", "q4_k", 5120, 17408, 64], ["gemm", "iq4_xs", 5120, 17408, 333],
                                  ["argmax", 248320, 64]], ids=lambda g: g[0] + "_" + str(g[1]))
def test_captured_argmax_keeps_its_scratch(fake, grow):
    r = fakehip.run(fake, [["norm", 64, 1, 0], ["argmax", 248320, 1], ["capture", 1], ["argmax", 248320, 1],
                           ["capture", 0], grow])
    assert [s["status"] for s in r] == [0] * len(r)
    held = new_allocs(r[0], r[1])
    assert len(held) == 2 and len(r[3]["allocs"]) == len(r[1]["allocs"])  # pairs, counters; nothing in the capture
    assert len(r[-1]["allocs"]) > len(r[1]["allocs"])                     # (it did grow)
    assert [r[-1]["allocs"][i][1] for i in held] == [0, 0]
