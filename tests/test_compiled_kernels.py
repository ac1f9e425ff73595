"""What the compiled kernels must have and no run shows reliably — waits, registers, spills — read from the assembly, which needs no GPU."""

import os
import re
import shutil
import subprocess

import pytest

import build_native

pytestmark = pytest.mark.skipif(shutil.which(build_native.HIPCC) is None, reason="no hipcc")


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


def assembly(tmp_path, source):
    asm = tmp_path / "kernels.s"
    subprocess.run([build_native.HIPCC, f"--offload-arch={build_native.ARCH}", *build_native.DEVICE_FLAGS, "-O3", "-std=c++17", *build_native.SOURCE_FLAGS.get(source, []), "-S", "--cuda-device-only",
                    str(build_native.CSRC / source), "-o", os.fspath(asm)], check=True, capture_output=True)
    return asm.read_text()


def resources(text):
    """{mangled name: (registers, spilled registers, LDS bytes)} of an assembly's kernels."""
    found = {}
    for entry in re.split(r"\n  - (?=\.agpr_count)", text[text.index("amdhsa.kernels:") :])[1:]:
        field = lambda name: re.search(rf"\.{name}:\s+(\S+)", entry).group(1)  # noqa: B023, E731
        found[field("name")] = (int(field("vgpr_count")), int(field("vgpr_spill_count")), int(field("group_segment_fixed_size")))
    return found


def test_every_wave_waits_before_the_arrival_is_counted(tmp_path):
    """Workgroups that count themselves as finished with a pass of the exact quantiles: every wave waits for its adds to the shared histogram before
    the barrier behind which the arrival is counted."""
    bodies, name = {}, None
    for line in assembly(tmp_path, "hist_quantile.hip").splitlines():
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


def test_the_delta_chain_keeps_its_workgroups_on_a_compute_unit(tmp_path):
    """Kernels of one column tile have the registers of one (a SIMD has 512, a workgroup of four waves one on each): 4, 3 and 2 workgroups for keys of up
    to 64, 128 and 256 channels; the one that may take two tiles of many short portions has room for 3.  None spills."""
    kernels = {n: r for n, r in resources(assembly(tmp_path, "delta_rule.hip")).items() if "delta_chain_kernel" in n}
    want = {"Li1ELi0E": 4, "Li2ELi0E": 3, "Li4ELi0E": 2, "Li2ELi3E": 3, "Li2ELi2E": 2}
    assert len(kernels) == 2 * len(want)  # of bf16 and fp32 rows
    for name, (registers, spilled, lds) in kernels.items():
        workgroups = next(w for form, w in want.items() if form in name)
        assert min(512 // (-(-registers // 8) * 8), 160 * 1024 // lds) >= workgroups and spilled == 0, (name, registers, spilled, lds)
