"""Waits that a kernel counts by hand, followed through the code the compiler makes of them: no GPU."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cyb_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _blocks(lines):
    """The kernel's code as blocks: label -> (events, successors); an event is 'c' (copy to LDS), 'w' (any other vector memory access),
    a number (wait until so many are left) or 'b' (barrier)."""
    blocks, label, events, nexts = {}, "entry", [], []
    for line in lines:
        s = line.split(";")[0].strip()
        m = re.match(r"(\.LBB\w+):", s)
        if m:
            blocks[label] = (events, nexts + [m.group(1)])
            label, events, nexts = m.group(1), [], []
            continue
        op = s.split(" ")[0]
        if op.startswith("global_load_lds"):
            events.append("c")
        elif op.startswith(("global_", "buffer_load", "buffer_store", "flat_", "scratch_")):
            events.append("w")
        elif op == "s_waitcnt":
            m = re.search(r"vmcnt\((\d+)\)", s)
            if m:
                events.append(int(m.group(1)))
        elif op == "s_barrier":
            events.append("b")
        elif op in ("s_branch", "s_endpgm") or op.startswith("s_cbranch"):
            if op != "s_endpgm":
                nexts.append(s.split()[1])
            after = f"behind {len(blocks)}"
            blocks[label] = (events, nexts + [after] if op.startswith("s_cbranch") else nexts)
            label, events, nexts = after, [], []
    blocks[label] = (events, nexts)
    return blocks


def _most_copies_in_flight_at_a_barrier(blocks):
    """Over every path through the blocks.  Accesses retire in the order of issue."""
    worst, seen, todo = 0, set(), [("entry", "")]
    while todo:
        label, queue = todo.pop()
        if (label, queue) in seen:
            continue
        seen.add((label, queue))
        events, nexts = blocks[label]
        for e in events:
            if e == "b":
                worst = max(worst, queue.count("c"))
            elif isinstance(e, int):
                queue = queue[len(queue) - e:] if e < len(queue) else queue
            else:
                queue += e
        assert len(queue) < 400, "copies without a wait"
        todo += [(n, queue) for n in nexts]
    return worst


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_the_copies_of_the_next_step_are_there_behind_every_barrier(tmp_path):
    """gemm_rows_pair_kernel copies X of a step (2 * MF copies per wave) RING - 1 steps ahead and waits, ahead of the barrier in front of a step,
    for all but the RING - 2 newest: no path may pass a barrier with more copies on their way, whatever the compiler made of the
    weight loads that the waits count (a load that nobody reads is not there)."""
    flags = subprocess.run(["make", "-s", "-C", CSRC, "flags"], capture_output=True, text=True, check=True).stdout.split()
    out = str(tmp_path / "gemm_rows.s")
    cc = subprocess.run([HIPCC, *flags, "--offload-device-only", "-S", os.path.join(CSRC, "gemm_rows.hip"), "-o", out], capture_output=True, text=True)
    assert cc.returncode == 0, cc.stderr[-3000:]
    with open(out) as f:
        text = f.read()
    kernels = re.findall(r"^(_ZN\S*gemm_rows_pair_kernelILi(\d)ELi(\d)ELi(\d)ELi(\d)E\S*):[^\n]*\n(.*?)^\.Lfunc_end", text, re.M | re.S)
    assert len(kernels) == 6
    for name, bits, mf, depth, ring, body in kernels:
        blocks = _blocks(body.split("\n"))
        assert sum(e == "b" for events, _ in blocks.values() for e in events) > int(depth)
        in_flight = _most_copies_in_flight_at_a_barrier(blocks)
        assert in_flight <= (int(ring) - 2) * 2 * int(mf), (bits, mf, depth, ring, in_flight)
