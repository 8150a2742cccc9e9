"""What the kernels rest on in the gfx950 code that the compiler makes of them.

The kernels that write their own workgroup barrier (inline `s_barrier` instead of
__syncthreads, so that loads in flight stay in flight): on every path, no LDS access of
the wave may still be outstanding when it arrives.  Another wave may overwrite that LDS
right after the barrier; that a load lands late is not an order.  The GEMM kernels: no
operand spills to scratch."""
import re
import subprocess

import pytest

from inferno_amd.build import COMMON_FLAGS, CSRC, hipcc

OWN_BARRIERS = sorted(p.name for p in CSRC.glob("*.hip")
                      if re.search(r"s_barrier|lds_barrier\(\)", p.read_text()))


def _functions(asm):
    """{name: [instruction or label, ...]} of the device code."""
    out, lines = {}, None
    for raw in asm.splitlines():
        line = raw.split(";")[0].strip()
        label = re.match(r"^([.\w$]+):$", line)
        if label and label.group(1).startswith("_Z"):
            lines = out.setdefault(label.group(1), [])
        elif lines is not None and line and (label or not line.startswith(".")):
            lines.append(line)
        if line.startswith(".Lfunc_end"):
            lines = None
    return out


def outstanding_at_barriers(lines):
    """(barriers, [(line, LDS accesses that may be outstanding there), ...]).  The
    state on a path is the lgkm operations since the last complete wait, newest
    last ("d": LDS, "s": scalar), and lgkmcnt(n) leaves the newest n."""
    at = {l[:-1]: i for i, l in enumerate(lines) if l.endswith(":")}
    seen = [set() for _ in range(len(lines) + 1)]
    todo, found = [(0, "")], {}
    while todo:
        i, pending = todo.pop()
        while i < len(lines) and pending not in seen[i]:
            seen[i].add(pending)
            op, _, args = lines[i].partition(" ")
            i += 1
            if op.startswith("ds_"):
                pending = (pending + "d")[-16:]
            elif re.match(r"s_(buffer_|scratch_)?load_", op):
                pending = (pending + "s")[-16:]
            elif op == "s_waitcnt" and "lgkmcnt" in args:
                n = int(re.search(r"lgkmcnt\((\d+)\)", args).group(1))
                if n == 0:
                    pending = ""
                elif "s" not in pending:  # scalar loads return in any order
                    pending = pending[-n:]
            elif op == "s_barrier":
                found[i - 1] = max(found.get(i - 1, 0), pending.count("d"))
            elif op == "s_branch":
                i = at[args.strip()]
            elif op.startswith("s_cbranch"):
                todo.append((at[args.strip()], pending))
            elif op == "s_endpgm":
                break
    return len(found), [(lines[i], n) for i, n in sorted(found.items()) if n]


def test_the_scan_sees_reads_behind_waits_and_round_loops():
    lines = ["ds_read_b128 v[0:3], v9", "ds_read_b128 v[4:7], v9", "s_waitcnt lgkmcnt(1)", "s_barrier"]
    assert outstanding_at_barriers(lines) == (1, [("s_barrier", 1)])
    lines[2] = "s_waitcnt vmcnt(0) lgkmcnt(0)"
    assert outstanding_at_barriers(lines) == (1, [])
    loop = [".L1:", "s_barrier", "ds_write_b32 v0, v1", "s_cbranch_scc1 .L1", "s_endpgm"]
    assert outstanding_at_barriers(loop) == (1, [("s_barrier", 16)])


def _device_code(source, tmp_path):
    asm = tmp_path / "device.s"
    res = subprocess.run([hipcc(), *COMMON_FLAGS, "--cuda-device-only", "-S", str(CSRC / source),
                          "-o", str(asm)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return asm.read_text()


@pytest.mark.parametrize("source", OWN_BARRIERS)
def test_no_lds_access_outstanding_at_a_barrier(source, tmp_path):
    barriers, faults = 0, {}
    for name, lines in _functions(_device_code(source, tmp_path)).items():
        n, late = outstanding_at_barriers(lines)
        barriers += n
        if late:
            faults[name] = late
    assert barriers > 0
    assert not faults, faults


def test_gemm_kernels_keep_their_operands_in_registers(tmp_path):
    asm = _device_code("gemm.hip", tmp_path)
    sizes = re.findall(r"\.amdhsa_kernel (\S+).*?\.amdhsa_private_segment_fixed_size (\d+)", asm, re.S)
    assert sizes and all(int(n) == 0 for _, n in sizes), [k for k, n in sizes if int(n)]
