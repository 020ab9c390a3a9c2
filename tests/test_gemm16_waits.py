"""The fp16-plane GEMM's waits, read from its machine code (CPU-only).

k_q16 stages its activation tiles with loads straight into LDS and, before each
step's workgroup barrier, waits only until its loads of that step have landed:
the count of younger loads that may stay in flight is written in the source
(gemm16.hip, sync_loads) and holds as long as the compiler issues the loads in
the order, and in the number, that it assumes.  A load too few, and a wave
passes the barrier with a tile another wave reads still on its way: wrong
results now and then.  So this follows every path through the built kernels and
checks, at each step's barrier, that no load of that step is outstanding, and
that the wave's reads of the previous step's tile have returned (the loads that
follow the barrier write over it).
"""
import os
import re
import shutil
import subprocess

import pytest

from mojollama_amd import kernels

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects of a HIP shared library (offload bundles: magic, count, then offset, size, name)."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        u64 = lambda o: int.from_bytes(data[o:o + 8], "little")  # noqa: E731, B023
        n, o = u64(at + 24), at + 32
        for _ in range(n):
            off, size, name = u64(o), u64(o + 8), u64(o + 16)
            if b"gfx950" in data[o + 24:o + 24 + name]:
                yield data[at + off:at + off + size]
            o += 24 + name
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    if not os.path.exists(kernels.LIB_PATH):
        kernels.build()
    obj = [c for c in code_objects(kernels.LIB_PATH) if b"k_q16I" in c]
    assert len(obj) == 1
    f = tmp_path_factory.mktemp("co") / "gemm16.co"
    f.write_bytes(obj[0])
    return subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], capture_output=True, text=True,
                          check=True).stdout


def kernel_events(listing):
    """kernel -> (events, position by address): 'D' a load into LDS, 'V' another vector memory access, ('w', n) a
    wait for all but the youngest n, 'R' an LDS access, 'L' a wait for all of them, 'B' a workgroup barrier,
    ('c' / 'j', target) a branch, 'E' the end."""
    out = {}
    for name, body in re.findall(r"^[0-9a-f]+ <(_Z\S*5k_q16I\S*?)>:\n(.*?)(?=^\S|\Z)", listing, re.M | re.S):
        ev, at, base = [], {}, None
        for line in body.splitlines():
            m = re.match(r"\s+(\S+)(.*?)//\s*([0-9A-F]+)", line)
            if not m:
                continue
            op, arg, adr = m.group(1), m.group(2).split(), int(m.group(3), 16)
            base = adr if base is None else base
            at[adr - base] = len(ev)
            if "lds" in arg or "load_lds" in op:
                ev.append("D")
            elif re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", op):
                ev.append("V")
            elif op.startswith("ds_"):
                ev.append("R")
            elif op == "s_waitcnt":
                if "lgkmcnt(0)" in arg:
                    ev.append("L")
                n = re.search(r"vmcnt\((\d+)\)", " ".join(arg))
                if n:
                    ev.append(("w", int(n.group(1))))
            elif op == "s_barrier":
                ev.append("B")
            elif op == "s_endpgm":
                ev.append("E")
            elif op == "s_branch" or op.startswith("s_cbranch"):
                t = re.search(r"<\S+?(?:\+0x([0-9a-f]+))?>", line)
                ev.append(("j" if op == "s_branch" else "c", int(t.group(1) or "0", 16)))
        out[name] = (ev, at)
    return out


def only_loads(ev, i, t):
    return t > i and all(e == "D" for e in ev[i:t])


def faults(ev, at):
    """The barriers (0: the first step's, 1: the second's, 2: a later one's; with the loads a step and the steps
    ahead) that some path reaches with a load of their step outstanding; "reads": a barrier of the main loop that
    some path reaches with LDS reads outstanding.

    A state is a place in the code, the accesses that may be outstanding from the oldest load into LDS on, and how
    far the path is: the loads are numbered from 0, and from the second barrier on, which shows how many a step has,
    from the current step's first.  Only paths count that a workgroup can take: it runs one form of the main loop, so
    every interval holds the same number of loads, entry blocks (1, 2 or 4) times planes (1 or 2), and the first one
    or three times that; a wave issues its loads in every step or in none."""
    bad, seen = set(), set()
    # place, outstanding, loads issued, barriers passed, loads a step (before the second barrier: at the first),
    # loads ahead (before it: the oldest outstanding at the first), faults not yet counted, LDS reads outstanding
    todo = [(0, (), 0, 0, 0, -1, (), False)]
    while todo:
        st = todo.pop()
        while st not in seen:
            seen.add(st)
            i, q, n, nb, per, low, f, r = st
            e, i = ev[i], i + 1
            if e == "D":
                q, n = q + (n,), n + 1
            elif e == "V":
                q = q + ("V",) if q else q
            elif e == "R" or e == "L":
                r = e == "R"
            elif e == "E":
                break
            elif e == "B":
                low_now = min([k for k in q if k != "V"], default=n)
                if nb == 0 and n:
                    nb, per, low = 1, n, low_now
                elif nb == 1:
                    ahead, per = per, n - per
                    if per <= 0 or per & (per - 1) or ahead not in (per, 3 * per):
                        break
                    f = tuple((k, per, ahead // per) for k, o in enumerate((low, low_now)) if o < (k + 1) * per)
                    q, n, nb = tuple(k if k == "V" else k - 2 * per for k in q), n - 2 * per, 2
                    low = n
                elif nb == 2:
                    if n - per != low:
                        break
                    bad |= set(f) | ({(2, per, low // per + 1)} if low_now < per else set())
                    bad |= {"reads"} if r else set()
                    q, n = tuple(k if k == "V" else k - per for k in q), n - per
                    f = ()
            elif e[0] == "w":
                q = q[len(q) - e[1]:] if len(q) > e[1] else q
                while q and q[0] == "V":
                    q = q[1:]
            elif e[0] == "j":
                i = at[e[1]]
            else:
                # a branch around loads into LDS alone: waves whose rows the tile does not reach skip
                # them in every step; those that issue them have something to wait for
                t = at[e[1]]
                if not only_loads(ev, i, t):
                    todo.append((t, q, n, nb, per, low, f, r))
            st = (i, q, n, nb, per, low, f, r)
    return bad


def test_every_step_waits_for_its_tiles(listing):
    found = {k: faults(*v) for k, v in kernel_events(listing).items()}
    assert len(found) >= 20 and any("D" in v[0] for v in kernel_events(listing).values())
    assert not any(found.values()), {k: v for k, v in found.items() if v}
