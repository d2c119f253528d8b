"""The work-queue loops of the persistent kernels in the machine code of the library's own build: test_queue_structure
checks a compilation with flags of its own, here the flags are those the library is built with (__graft_entry__), whose
passes could structure the loops otherwise."""
import os
import subprocess

import pytest

import __graft_entry__ as entry
from test_queue_structure import HIPCC, SRC, SRC_ADJ, block_loops, queue_loops

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not present")


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    flags = [f for f in entry.HIPCC_FLAGS if f != "-fPIC"] + ["-w", "--cuda-device-only", "-S"]
    d = tmp_path_factory.mktemp("asm")
    outs = {src: str(d / (os.path.basename(src) + ".s")) for src in (SRC, SRC_ADJ)}
    procs = [subprocess.Popen([HIPCC, *flags, "-o", out, src], stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL) for src, out in outs.items()]
    assert [p.wait() for p in procs] == [0] * len(procs)
    return {src: open(out).read() for src, out in outs.items()}


def test_transfer_pops_on_every_back_edge(asm):
    loops = queue_loops(asm[SRC])
    assert len(loops) == 20          # 5 populations x 2 precisions x cull on/off
    for name, w in loops.items():
        assert w.get("pop") and w.get("barrier") and w.get("read"), (name, w)
        assert w["pop"] == w["barrier"] == w["read"], (name, w)


def test_element_adjoints_pop_on_every_back_edge(asm):
    loops = block_loops(asm[SRC_ADJ], "ks_adj_splats")
    assert len(loops) == 14          # 7 population sets x 2 precisions
    for name, (pop, stores) in loops.items():
        assert pop is not None and pop[1] == 1, (name, pop)
        assert stores and stores == {pop}, (name, pop, stores)
