"""The waits of the 256 x 128 Q8 projection kernel (proj_wide_kernel), replayed
on the CPU over the instructions its source compiles to: a wave may pass the
barrier that opens stage s only when its own direct-to-LDS loads of stage s are
done, since its neighbours read the rows it loads."""
import pathlib
import re
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
LOADS = 4  # direct-to-LDS loads of a wave and stage


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


@pytest.mark.skipif(shutil.which("hipcc") is None and not pathlib.Path("/opt/rocm/bin/hipcc").exists(),
                    reason="needs the compiler")
def test_wide_stage_loads_are_done_at_its_barrier(tmp_path):
    lines = kernel_lines(device_assembly("csrc/k3_proj.hip", tmp_path), "proj_wide_kernel")
    for stage, (issued, flight) in enumerate(replay(lines, 8)):
        assert issued == LOADS * (stage + 2)  # two stages ahead
        late = [f for f in flight if f < LOADS * (stage + 1)]
        assert not late, f"stage {stage}: loads {late} still in flight behind its barrier"
