"""The barrier between the workgroups that share a pair or a sequence, in the
gfx950 assembly of the kernels that have one: the thread that writes the L2
back and counts the workgroup's arrival does so after a workgroup barrier, and
every wave has to wait for its own stores (vmcnt(0)) before that barrier.
s_barrier does not wait for them, and neither does a fence of workgroup scope:
without the wait another wave's store could follow the write-back.  And the
counting of arrivals (arrive_and_wait) with expired waits, on the host.  Compiles
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


SHIM = """
#pragma once
#define __device__
#define __forceinline__ inline
static int polls_made = 0;
inline int atomicAdd(int *p, int v) { polls_made += v == 0; int x = *p; *p += v; return x; }
inline int atomicOr(int *p, int v) { int x = *p; *p |= v; return x; }
inline void __threadfence() {}
inline void __threadfence_block() {}
inline void __syncthreads() {}
inline void __builtin_amdgcn_s_sleep(int) {}
inline void __builtin_amdgcn_fence(int, const char *) {}
static struct { int x; } threadIdx;
"""

MAIN = """
#include "member_barrier.h"
#include <cstdio>
int main() {
    // three members, two barriers; the third comes after the others gave up
    int c = 0;
    const bool a1 = arrive_and_wait(&c, 3, 5), b1 = arrive_and_wait(&c, 3, 5);
    const int first = polls_made;
    const bool a2 = arrive_and_wait(&c, 6, 1000000), b2 = arrive_and_wait(&c, 6, 1000000);
    const bool l1 = arrive_and_wait(&c, 3, 5), l2 = arrive_and_wait(&c, 6, 5);
    std::printf("%d %d %d %d %d %d %d %d ", a1, b1, a2, b2, l1, l2, first, polls_made - first);
    // all there; no waiting at all; alone
    int d = 2, e = 2, f = 0;
    polls_made = 0;
    const bool last = arrive_and_wait(&d, 3, 5), none = arrive_and_wait(&e, 3, -1), one = arrive_and_wait(&f, 1, 0);
    std::printf("%d %d %d %d\\n", last, none, one, polls_made);
}
"""


def test_expired_wait_is_seen_by_all(tmp_path):
    """Members that come late learn that a wait has expired, and nobody waits
    for its bound again."""
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(SHIM)
    (tmp_path / "m.cpp").write_text(MAIN)
    exe = str(tmp_path / "m")
    subprocess.run([build.CXX, "-std=c++17", "-I" + str(tmp_path), "-I" + build.CSRC, "-o", exe, str(tmp_path / "m.cpp")],
                   check=True)
    out = [int(x) for x in subprocess.run([exe], check=True, stdout=subprocess.PIPE, text=True).stdout.split()]
    assert out[:6] == [0] * 6  # every wait reports it
    assert 0 < out[6] <= 8 and out[7] == 0  # one wait up to its bound, none after it
    assert out[8:] == [1, 0, 1, 0]
