"""Workgroups that count themselves as finished with a pass (csrc/hist_quantile.hip): in the compiled code every wave waits for its
adds to the shared histogram before the barrier behind which the arrival is counted.  Read from the assembly, which needs no GPU."""

import os
import re
import shutil
import subprocess

import pytest

import build_native


def unwaited_arrivals(body):
    """Lines of ``body`` (one function's instructions) at which an arrival is counted — an atomic add that returns its value — although
    between the last vector-memory write or atomic and the barrier in front of it no wave waits for ``vmcnt(0)``."""
    bad = []
    for i, line in enumerate(body):
        if not re.match(r"global_atomic_add\b.*\bsc0\b", line):
            continue
        barrier = max((j for j in range(i) if body[j] == "s_barrier"), default=0)
        writes = [j for j in range(barrier) if re.match(r"(global|buffer|flat)_(atomic|store)", body[j])]
        if writes and not any(re.match(r"s_waitcnt.*\bvmcnt\(0\)", body[j]) for j in range(writes[-1], barrier)):
            bad.append(i)
    return bad


def test_the_check_itself():
    add, barrier, arrive = "global_atomic_add v[2:3], v1, off", "s_barrier", "global_atomic_add v1, v1, v2, s[10:11] sc0"
    assert unwaited_arrivals([add, "s_waitcnt lgkmcnt(0)", barrier, arrive]) == [3]
    assert unwaited_arrivals([add, "s_waitcnt lgkmcnt(0)", barrier, "s_waitcnt vmcnt(0)", arrive]) == [4]  # (one wave's wait: too late)
    assert unwaited_arrivals([add, "s_waitcnt vmcnt(0)", "s_waitcnt lgkmcnt(0)", barrier, arrive]) == []
    assert unwaited_arrivals([add, "s_waitcnt vmcnt(0) lgkmcnt(0)", barrier, arrive]) == []


@pytest.mark.skipif(shutil.which(build_native.HIPCC) is None, reason="no hipcc")
def test_every_wave_waits_before_the_arrival_is_counted(tmp_path):
    asm = tmp_path / "hist_quantile.s"
    subprocess.run([build_native.HIPCC, f"--offload-arch={build_native.ARCH}", *build_native.DEVICE_FLAGS, "-O3", "-std=c++17", "-S", "--cuda-device-only",
                    str(build_native.CSRC / "hist_quantile.hip"), "-o", os.fspath(asm)], check=True, capture_output=True)
    bodies, name = {}, None
    for line in asm.read_text().splitlines():
        label = re.match(r"(_Z\w+):", line)
        if label:
            name = label.group(1)
            bodies[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name and line.startswith("\t") and line.strip()[:1] not in (".", ";"):
            bodies[name].append(line.split(";")[0].strip())
    picking = {n: b for n, b in bodies.items() if "select_pass_kernel" in n and any(re.match(r"global_atomic_add\b.*\bsc0\b", l) for l in b)}
    assert len(picking) == 2  # of floats, of doubles
    assert {n: unwaited_arrivals(b) for n, b in picking.items()} == {n: [] for n in picking}
