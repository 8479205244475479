"""The compiled order of memory operations where a hand-written wait counts on it (no GPU needed).

k_tile_wide waits with vmcnt(8) for its direct copies to LDS: correct only while at least eight younger
memory operations follow the copies on every path to the wait.  The source pins that order; this reads
the assembly that the build's own flags give for gfx950.
"""
import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
VMEM = re.compile(r"^(buffer|global|flat)_(load|store|atomic)")


def _build():
    spec = importlib.util.spec_from_file_location("stacr_build_flags", os.path.join(ROOT, "stac-r_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    mod = _build()
    if not os.path.exists(mod.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("isa") / "tiles.s")
    res = subprocess.run([mod.HIPCC, *mod.FLAGS, "--offload-device-only", "-S", "-o", out,
                          os.path.join(mod.CSRC, "weight_grad_tiles.hip")], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stderr[-2000:]
    with open(out) as f:
        return f.read()


def _kernels(text, name):
    found = re.findall(rf"^(_ZN\S*{name}\S*):(.*?)^.Lfunc_end", text, re.M | re.S)
    return {n: [ln.split(";")[0].strip() for ln in body.splitlines() if ln.split(";")[0].strip()] for n, body in found}


def _fewest_younger(lines, wait):
    """The fewest memory operations between a copy to LDS and the wait at lines[wait], over all paths back
    from it (a path that drains the counter on the way is fine and not followed)."""
    label = {ln[:-1]: i for i, ln in enumerate(lines) if ln.endswith(":")}
    before = [[] for _ in lines]
    for i, ln in enumerate(lines):
        m = re.match(r"s_(c?branch)\S*\s+(\S+)", ln)
        if m:
            before[label[m.group(2)]].append(i)
        if i + 1 < len(lines) and not ln.startswith("s_branch"):
            before[i + 1].append(i)
    best, todo, seen = None, [(wait, 0)], {}
    while todo:
        at, n = todo.pop()
        if seen.get(at, 1 << 30) <= n:
            continue
        seen[at] = n
        for i in before[at]:
            ln = lines[i]
            if re.match(r"s_waitcnt\b.*vmcnt\(0\)", ln):
                continue
            if VMEM.match(ln) and ln.endswith(" lds"):
                best = n if best is None else min(best, n)
            elif n < 64:
                todo.append((i, n + bool(VMEM.match(ln))))
    return best


def test_wide_weight_gradient_waits_for_its_copies(assembly):
    kernels = _kernels(assembly, "k_tile_wide")
    assert len(kernels) == 4  # two types, two widths
    for name, lines in kernels.items():
        # the wait before the block's barrier: the last vmcnt(8) in front of it
        barriers = [i for i, ln in enumerate(lines) if ln == "s_barrier"]
        waits = [i for i, ln in enumerate(lines) if re.match(r"s_waitcnt\b.*vmcnt\(8\)", ln) and
                 any(b - 4 <= i < b for b in barriers)]
        assert waits, f"{name}: no vmcnt(8) in front of a barrier"
        for w in waits:
            fewest = _fewest_younger(lines, w)
            assert fewest is not None and fewest >= 8, f"{name}: {fewest} memory operations younger than a copy"
            # (and with one of those loads in front of the copies, planted in the text, it would be seen)
            copy = max(i for i in range(w) if lines[i].endswith(" lds") and VMEM.match(lines[i]))
            load = next(i for i in range(copy + 1, w) if VMEM.match(lines[i]))
            assert _fewest_younger(lines[:load] + ["s_nop 0"] + lines[load + 1:], w) == fewest - 1
