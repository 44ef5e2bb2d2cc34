"""LDS reads and the loads that overwrite what they read, in the built gfx950
code: a load with an LDS destination is not ordered behind the wave's earlier
LDS reads, so before it goes out to a slot the reads of that slot have to have
returned (s_waitcnt lgkmcnt). Read from the disassembly of the library, since
no run can show a wait that is missing but seldom needed. LDS reads of a wave
return in order, so a wait for at most n leaves the n youngest. Needs no GPU."""
import os
import re
import subprocess

import pytest

import q3vl_int8 as q

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

pytestmark = pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """{kernel symbol: [(address, instruction)]} of the library's device code."""
    d = tmp_path_factory.mktemp("code")
    os.symlink(q.LIB_PATH, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    out = {}
    for f in sorted(os.listdir(d)):
        if "gfx950" not in f:
            continue
        asm = subprocess.run([OBJDUMP, "-d", f], cwd=d, check=True, capture_output=True, text=True).stdout
        cur = None
        for line in asm.splitlines():
            m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
            if m:
                cur = out.setdefault(m.group(1), [])
            elif cur is not None:
                m = re.match(r"^\s+(\S.*?)\s*// ([0-9A-F]+):", line)
                if m:
                    cur.append((int(m.group(2), 16), m.group(1)))
    return out


def loops(ins):
    """Bodies (instruction texts) of the innermost backward branches."""
    at = {a: i for i, (a, _) in enumerate(ins)}
    found = []
    for i, (a, t) in enumerate(ins):
        m = re.match(r"s_c?branch\S* (\d+)", t)
        if m:
            to = at.get(a + 4 + 4 * ((int(m.group(1)) ^ 0x8000) - 0x8000))
            if to is not None and to <= i:
                found.append((to, i))
    return [[t for _, t in ins[a:b + 1]] for a, b in found
            if not any((c, d) != (a, b) and a <= c and d <= b for c, d in found)]


def outstanding(body, is_load):
    """Two turns of the body: for each load of the second turn that is_load
    picks, how many LDS reads of the first turn may still be under way."""
    queue, worst = [], []
    for turn in (0, 1):
        for t in body:
            if t.startswith("ds_read"):
                queue.append(turn)
            elif t.startswith("ds_"):
                queue.append(None)
            elif t.startswith("s_waitcnt"):
                m = re.search(r"lgkmcnt\((\d+)\)", t)
                if m:
                    queue = queue[max(0, len(queue) - int(m.group(1))):]
            elif turn and is_load(t):
                worst.append(sum(x == 0 for x in queue))
    return worst


def test_fragment_gemm_rereads_no_weight_scale_slot(code):
    """gemm_t16_kernel: a loop body ends by reading the next body's weight
    scales, and the next body's single-dword loads refill that slot."""
    seen = 0
    for name, ins in code.items():
        if "gemm_t16_kernel" not in name:
            continue
        bodies = [b for b in loops(ins) if any("v_mfma" in t for t in b) and
                  any(re.match(r"buffer_load_dword\b.* lds", t) for t in b)]
        assert len(bodies) == 1, name
        worst = outstanding(bodies[0], lambda t: re.match(r"buffer_load_dword\b.* lds", t))
        assert worst and max(worst) == 0, f"{name}: {worst} reads not waited for"
        seen += 1
    assert seen >= 30


def test_wide_gemm_reloads_read_slots_only(code):
    """gemm_wide_kernel: a pair's reads have returned before its ring slot
    takes the next one (the weights and scales are read first in the loop)."""
    seen = 0
    for name, ins in code.items():
        if "gemm_wide_kernel" not in name:
            continue
        bodies = [b for b in loops(ins) if any("v_mfma" in t for t in b)]
        assert len(bodies) == 1, name
        n, bad, first = 0, None, False
        for t in bodies[0]:
            if t.startswith("ds_"):
                n += 1
            m = re.match(r"s_waitcnt.*lgkmcnt\((\d+)\)", t)
            if m:
                n = min(n, int(m.group(1)))
            if re.match(r"buffer_load_dwordx4.* nt lds", t) and not first:
                first, bad = True, n
        assert first and bad == 0, f"{name}: {bad} reads under way at the first reload"
        seen += 1
    assert seen == 9
