"""Stores that one workgroup hands to another inside a launch.

The dense solves' workgroups publish tiles and vectors behind a release fence
(an L2 write-back) and a flag or counter.  What the hand-over needs is read from
the gfx950 assembly of the two kernels, since a missing wait shows in results
only when the timing is bad.
"""
import os
import re
import subprocess

import pytest

from psba_amd import build

LABEL = re.compile(r"^\.?\w+:|^BB\d+")
STORE = re.compile(r"^(global|flat|buffer)_(store|atomic)|^scratch_store")


def assembly(source, folder):
    out = os.path.join(str(folder), source + ".s")
    build._run([build.HIPCC] + build.HIP_FLAGS + ["--cuda-device-only", "-S", os.path.join(build.CSRC, source),
                                                  "-o", out])
    with open(out) as f:
        lines = [line.split(";")[0].strip() for line in f]
    return [x for x in lines if x and (not x.startswith(".") or LABEL.match(x))]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    folder = tmp_path_factory.mktemp("asm")
    return {s: assembly(s, folder) for s in ("k_chol.hip", "k_dense.hip")}


def workgroup_releases(code):
    """Write-backs that follow a workgroup barrier with no store between: their
    wave publishes what the whole workgroup stored.  Yields the barrier's place."""
    for at, line in enumerate(code):
        if not line.startswith("buffer_wbl2"):
            continue
        for k in range(at - 1, -1, -1):
            if STORE.match(code[k]) or code[k].startswith(("s_swappc", "s_setpc")):
                break
            if code[k].startswith("s_barrier"):
                yield k
                break


@pytest.mark.parametrize("source,least", [("k_chol.hip", 10), ("k_dense.hip", 2)])
def test_every_wave_drains_its_stores_before_the_barrier_of_a_release(kernels, source, least):
    code = kernels[source]
    found = list(workgroup_releases(code))
    assert len(found) >= least
    for barrier in found:
        for k in range(barrier - 1, -1, -1):
            assert not STORE.match(code[k]), "stores still on their way at the barrier: %s" % code[k:barrier + 1]
            if code[k].startswith("s_waitcnt") and "vmcnt(0)" in code[k]:
                break


@pytest.mark.parametrize("source,least", [("k_chol.hip", 10), ("k_dense.hip", 4)])
def test_a_release_waits_for_its_write_back(kernels, source, least):
    """The wave's next access (the flag) only once the write-back has ended."""
    code = kernels[source]
    found = [k for k, line in enumerate(code) if line.startswith("buffer_wbl2")]
    assert len(found) >= least
    for at in found:
        for line in code[at + 1:]:
            assert not re.match(r"(global|flat|buffer)_", line), "no wait between write-back and %s" % line
            if line.startswith("s_waitcnt") and "vmcnt(0)" in line:
                break
