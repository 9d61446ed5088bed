"""The barrier between the workgroups that share a pair or a sequence, in the
gfx950 assembly of the kernels that have one: the thread that writes the L2
back and counts the workgroup's arrival does so after a workgroup barrier, and
every wave has to wait for its own stores (vmcnt(0)) before that barrier.
s_barrier does not wait for them, and neither does a fence of workgroup scope:
without the wait another wave's store could follow the write-back.  Compiles
the kernels for gfx950; runs on the CPU."""
import os
import re
import subprocess

import pytest

from locarna_amd import build

KERNELS = {  # kernel: places with such a barrier
    "align_kernels": {"lcg_fill_band": 1, "lcg_fill_band_tab": 1},
    "pf_kernels": {"lcg_pf_pairs": 4},
    "fold_kernels": {"lcg_fold_seqs": 3},
}


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("asm")
    jobs = {f: subprocess.Popen([build.HIPCC] + build.HIP_FLAGS +
                                ["--cuda-device-only", "-S", "-o", str(tmp / f),
                                 os.path.join(build.CSRC, f + ".hip")], stderr=subprocess.DEVNULL) for f in KERNELS}
    assert [j.wait() for j in jobs.values()] == [0] * len(jobs)
    return {f: (tmp / f).read_text() for f in jobs}


def release_points(asm, kernel):
    """Per L2 write-back of the kernel, the lines before it, the nearest first."""
    body = re.split(r"\n%s:" % kernel, asm)[1].split("s_endpgm")[0]
    lines = [l.split(";")[0].strip() for l in body.split("\n")]
    lines = [l for l in lines if l and (not l.startswith(".") or l.endswith(":"))]
    return [lines[:k][::-1] for k, l in enumerate(lines) if l.startswith("buffer_wbl2")]


@pytest.mark.parametrize("source", KERNELS)
def test_waves_wait_for_their_stores(assembly, source):
    for kernel, places in KERNELS[source].items():
        points = release_points(assembly[source], kernel)
        assert len(points) == places, kernel
        for before in points:
            bar = before.index("s_barrier")
            assert not any(re.search("_store_|_atomic_", l) for l in before[:bar]), kernel
            # the wait stands in the barrier's own basic block, no store after it
            wait = next(k for k, l in enumerate(before) if k > bar and re.search(r"s_waitcnt.*vmcnt\(0\)", l))
            assert not any(re.search(r":$|branch|_store_|_atomic_", l) for l in before[bar:wait]), kernel
