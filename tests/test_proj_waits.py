"""The waits of the Q8 projection kernels, replayed on the CPU over the
instructions their source compiles to: a wave may pass the barrier that opens
stage s only when its own direct-to-LDS loads of stage s are done, since its
neighbours read the rows it loads."""
import pathlib
import re
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
pytestmark = pytest.mark.skipif(
    shutil.which("hipcc") is None and not pathlib.Path("/opt/rocm/bin/hipcc").exists(),
    reason="needs the compiler")


@pytest.fixture(scope="module")
def proj(tmp_path_factory):
    return device_assembly("csrc/k3_proj.hip", tmp_path_factory.mktemp("proj"))


def device_assembly(source, tmp_path):
    """gfx950 assembly of a source file of the library, with the library's own flags."""
    obj = f"_build/{pathlib.Path(source).stem}.o"
    lines = subprocess.run(["make", "-n", "-B", obj], cwd=ROOT / "moonshine_amd", check=True,
                           capture_output=True, text=True).stdout.splitlines()
    cmd = next(l for l in lines if "hipcc" in l).split()
    out = tmp_path / "kernel.s"
    cmd = [c for c in cmd if c != "-c"]
    cmd[cmd.index("-o") + 1] = str(out)
    subprocess.run(cmd + ["-S", "--cuda-device-only"], cwd=ROOT / "moonshine_amd", check=True,
                   capture_output=True)
    return out.read_text()


def kernel_lines(asm, name):
    body = re.search(rf"^_Z\w*{name}\w*:.*?^\.Lfunc_end", asm, re.M | re.S)
    assert body, name
    lines = (re.sub(r";.*", "", l).strip() for l in body.group(0).splitlines()[1:])
    return [l for l in lines if l]


def replay(lines, barriers):
    """Runs the straight path (forward branches not taken, backward ones taken)
    until `barriers` barriers have passed; per barrier the direct-to-LDS loads
    issued and those among them still in flight, as issue numbers."""
    label = {l[:-1]: i for i, l in enumerate(lines) if l.endswith(":")}
    flight, issued, seen, pc = [], 0, [], 0
    while len(seen) < barriers:
        assert pc < len(lines), f"the path ended after {len(seen)} barriers"
        l = lines[pc]
        op = l.split()[0]
        if op.startswith("global_load_lds"):
            flight.append(issued)
            issued += 1
        elif op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            flight.append(None)
        elif op == "s_waitcnt":
            n = re.search(r"vmcnt\((\d+)\)", l)
            if n:
                flight = flight[len(flight) - min(int(n.group(1)), len(flight)):]
        elif op == "s_barrier":
            seen.append((issued, [f for f in flight if f is not None]))
        elif op.startswith(("s_cbranch", "s_branch")):
            target = label[l.split()[1]]
            if target < pc or op == "s_branch":
                pc = target
        elif op == "s_endpgm":
            raise AssertionError(f"the path ended after {len(seen)} barriers")
        pc += 1
    return seen


def check(stage, need, flight):
    late = [f for f in flight if f < need]
    assert not late, f"stage {stage}: loads {late} still in flight behind its barrier"


# kernel, loads of a wave and stage, stages fetched ahead of the first barrier
@pytest.mark.parametrize("name,loads,ahead", [("proj_wide_kernel", 4, 2),
                                              ("proj_ring_kernelILi2ELi1ELi2ELi2E", 4, 1),
                                              ("proj_ring_kernelILi2ELi1ELi2ELi6E", 4, 5)])
def test_stage_loads_are_done_at_its_barrier(proj, name, loads, ahead):
    for stage, (issued, flight) in enumerate(replay(kernel_lines(proj, name), 8)):
        assert issued == loads * (stage + ahead)
        check(stage, loads * (stage + 1), flight)


@pytest.mark.parametrize("name,loads,ring,phases", [("proj_ring_kernelILi2ELi2ELi2ELi4E", 5, 4, 2),
                                                    ("proj_ring_kernelILi4ELi2ELi2ELi3E", 7, 3, 4)])
def test_alternating_halves_wait_a_barrier_early(proj, name, loads, ring, phases):
    """Half of the block runs one barrier behind: the loads of stage s + 1 are
    done before the last but one of stage s's barriers."""
    groups = {}
    for issued, flight in replay(kernel_lines(proj, name), 2 + 6 * phases):
        groups.setdefault(issued, []).append(flight)
    check(0, loads, groups.pop(loads * (ring - 1))[0])
    for stage in range(5):
        barriers = groups.pop(loads * (ring + stage))
        assert len(barriers) == phases
        check(stage + 1, loads * (stage + 2), barriers[-2])
