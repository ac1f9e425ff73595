"""What the compiled kernels must have and no run shows reliably — waits, counts of operations in flight, registers — read from the
built library's gfx950 code, which needs no GPU."""

import os
import re
import shutil
import struct
import subprocess

import pytest

import build_native

TOOLS = os.path.join(build_native.ROCM, "llvm", "bin")
pytestmark = pytest.mark.skipif(shutil.which(os.path.join(TOOLS, "llvm-objdump")) is None or not build_native.ext_path().exists(), reason="no library or no tools to read it")


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """Files of the device code, one for each source."""
    data, files, folder = build_native.ext_path().read_bytes(), [], tmp_path_factory.mktemp("code")
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at, entry = bundle.start(), bundle.start() + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, name = struct.unpack_from("<QQQ", data, entry)
            entry += 24 + name
            if size:
                files.append(folder / f"{len(files)}.o")
                files[-1].write_bytes(data[at + offset : at + offset + size])
    return files


def read(tool, *args):
    return subprocess.run([os.path.join(TOOLS, tool), *map(os.fspath, args)], check=True, capture_output=True, text=True).stdout


@pytest.fixture(scope="module")
def functions(code_objects):
    """``functions(part)``: {mangled name: instructions} of the kernels whose names hold ``part``."""

    def of(part):
        found = {}
        for file in code_objects:
            names = [line.split()[-1] for line in read("llvm-objdump", "-t", file).splitlines() if " F .text" in line and part in line]
            body = None
            for line in read("llvm-objdump", "-d", "--no-show-raw-insn", f"--disassemble-symbols={','.join(names)}", file).splitlines() if names else ():
                label = re.match(r"[0-9a-f]+ <(\S+)>:", line)
                if label:
                    body = found.setdefault(label.group(1), [])
                elif line.startswith("\t"):
                    body.append(line.split("//")[0].strip())
        return found

    return of


@pytest.fixture(scope="module")
def resources(code_objects):
    """{mangled name: (registers, spilled registers, bytes of scratch, bytes of LDS)} of all kernels."""
    found = {}
    for file in code_objects:
        for entry in re.split(r"\n\s+- (?=\.agpr_count)", read("llvm-readelf", "--notes", file))[1:]:
            field = lambda name: re.search(rf"\.{name}:\s+(\S+)", entry).group(1)  # noqa: B023, E731
            found[field("name")] = tuple(int(field(n)) for n in ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size", "group_segment_fixed_size"))
    return found


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


def test_unwaited_arrivals_are_found():
    add, barrier, arrive = "global_atomic_add v[2:3], v1, off", "s_barrier", "global_atomic_add v1, v1, v2, s[10:11] sc0"
    assert unwaited_arrivals([add, "s_waitcnt lgkmcnt(0)", barrier, arrive]) == [3]
    assert unwaited_arrivals([add, "s_waitcnt lgkmcnt(0)", barrier, "s_waitcnt vmcnt(0)", arrive]) == [4]  # (one wave's wait: too late)
    assert unwaited_arrivals([add, "s_waitcnt vmcnt(0)", "s_waitcnt lgkmcnt(0)", barrier, arrive]) == []
    assert unwaited_arrivals([add, "s_waitcnt vmcnt(0) lgkmcnt(0)", barrier, arrive]) == []


def test_every_wave_waits_before_an_arrival_is_counted(functions):
    """Workgroups that count themselves as finished — with a pass of the exact quantiles, with their share of a decode step's keys, with their part of
    a split product: every wave waits for what it wrote or added before the barrier behind which the arrival is counted."""
    for part, least in (("select_pass_kernel", 2), ("select_collect_kernel", 2), ("decode_attention_fused_kernel", 8), ("stream_gemm", 1)):
        arriving = {n: b for n, b in functions(part).items() if any(re.match(r"global_atomic_add\b.*\bsc0\b", line) for line in b)}
        assert len(arriving) >= least, part
        assert {n: unwaited_arrivals(b) for n, b in arriving.items()} == {n: [] for n in arriving}


def test_the_delta_chain_keeps_its_workgroups_on_a_compute_unit(resources):
    """Kernels of one column tile have the registers of one (a SIMD has 512, a workgroup of four waves one on each): 4, 3 and 2 workgroups for keys of up
    to 64, 128 and 256 channels; the one that may take two tiles of many short portions has room for 3.  None spills."""
    kernels = {n: r for n, r in resources.items() if "delta_chain_kernel" in n}
    want = {"Li1ELi0E": 4, "Li2ELi0E": 3, "Li4ELi0E": 2, "Li2ELi3E": 3, "Li2ELi2E": 2}
    assert len(kernels) == 2 * len(want)  # of bf16 and fp32 rows
    for name, (registers, spilled, _scratch, lds) in kernels.items():
        workgroups = next(w for form, w in want.items() if form in name)
        assert min(512 // (-(-registers // 8) * 8), 160 * 1024 // lds) >= workgroups and spilled == 0, (name, registers, spilled, lds)


def test_split_decode_attention_has_the_waves_its_shares_are_made_for(resources):
    """Ranges are cut for 2048 resident waves, two on a SIMD, and for 1024 where groups of more than four heads take their scores from the vector unit."""
    seen = set()
    for name, (registers, *_rest) in resources.items():
        form = re.search(r"decode_attention_fused_kernelILi(\d+)ELi[48]ELb[01]ELb1ELb[01]ELb([01])E", name)
        if form:
            wide = int(form.group(1)) > 4 and form.group(2) == "0"
            assert registers <= (512 if wide else 256), name
            seen.add(wide)
    assert seen == {True, False}


def test_panels_have_in_flight_what_they_wait_for(functions):
    """The products by panels wait for a stage by the number of operations issued behind it.  In the loop of each height that is a count of its own, and
    from one barrier to the next exactly a stage's loads are issued: four of weights, and the pieces of rows."""
    loads = {14: 8, 22: 8, 26: 7, 33: 7, 28: 6, 23: 5, 20: 5}  # {operations that may be in flight: a stage's}, 256 rows to 32
    kernels = functions("panel_kernel")
    assert len(kernels) == 6
    for name, body in kernels.items():
        before, issued, seen = -1, 0, set()
        for i, line in enumerate(body):
            issued += line.startswith("buffer_load")
            if line.startswith(("s_branch", "s_cbranch")):
                before = -1  # (what follows in the text need not follow in the run)
            if line != "s_barrier":
                continue
            wait = re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)", body[i - 1])
            allowed = int(wait.group(1)) if wait else -1
            if allowed == before and allowed in loads:
                assert issued == loads[allowed], (name, allowed, issued)
                seen.add(allowed)
            before, issued = allowed, 0
        assert seen == set(loads), (name, seen)


def test_narrow_tiles_have_in_flight_what_they_wait_for(functions):
    """Narrow tiles wait for a stage's rows by the number of operations issued behind them too.  Rows are fetched nowhere without their weights (the compiler
    drops loads that nothing multiplies: stages behind the loop must fetch neither); in the loop, from one barrier to the next, exactly a stage's."""
    kernels = functions("narrow_tiles_kernel")
    assert len(kernels) == 10
    for name, body in kernels.items():
        behind = 1 if "ELi0EEEv" in name else 0  # of a stage's two loads of weights, in front of its barrier: one of bf16, else none
        loops, seen = {6 * (2 + px) + px + behind: 2 + px for px in (1, 2)}, set()
        stretch, stretches = [], []
        for line in body:
            stretch.append(line)
            if line.startswith(("s_branch", "s_cbranch", "s_endpgm")):
                stretches.append(stretch)
                stretch = []
        for lines in stretches:
            at = [i for i, line in enumerate(lines) if line == "s_barrier"]
            fetched = [i for i, line in enumerate(lines) if line.startswith("buffer_load")]
            rows = sum(lines[i].endswith("lds") for i in fetched)
            assert len(fetched) in (2 * rows, 3 * rows), (name, rows, len(fetched))  # (two or one pieces of rows a stage)
            before, last = -1, 0
            for i in at:
                wait = re.match(r"s_waitcnt vmcnt\((\d+)\)", lines[i - 1])
                allowed = int(wait.group(1)) if wait else -1
                if allowed in loops and allowed == before:
                    assert sum(last < f < i for f in fetched) == loops[allowed], (name, allowed)
                    seen.add(allowed)
                before, last = allowed, i
        assert seen == set(loops), (name, seen)


def registers_of(text):
    found = set()
    for many in re.finditer(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        found |= {int(many.group(3))} if many.group(3) else set(range(int(many.group(1)), int(many.group(2)) + 1))
    return found


def test_nothing_touches_a_transposed_read_in_flight(functions):
    """The prompt attention kernels issue LDS reads that the compiler takes as done at once: until a wait has answered them (the LDS answers in
    order) no instruction reads, moves or overwrites their registers."""
    for part in ("chunk_prefill_kernel", "latent_prefill_kernel"):
        reads = 0
        for name, body in functions(part).items():
            flying = []
            for line in body:
                if line.startswith("s_waitcnt"):
                    left = re.search(r"lgkmcnt\((\d+)\)", line)
                    if left:
                        flying = flying[max(0, len(flying) - int(left.group(1))) :]
                    continue
                if line.startswith(("s_endpgm", "s_branch")):
                    flying = []
                    continue
                used = registers_of(line)
                assert not any(used & target for target in flying), (name, line)
                if line.startswith("ds_read_b64_tr"):
                    flying.append(registers_of(line.split(None, 1)[1].split(",", 1)[0]))
                    reads += 1
                elif line.startswith(("ds_", "s_load", "s_buffer_load")):
                    flying.append(set())
        assert reads > 100, part
