"""Every workgroup barrier of the built kernels is reached with no LDS access of
the wave outstanding, on every path: a wave that has passed a barrier may read
or overwrite what another one stores or reads before it. The compiler (ROCm 7.2,
gfx950) has left this wait out on the way back to a barrier at the head of a
loop. Checked over the library's own gfx950 code, with a count of outstanding
LDS accesses (they complete in order) followed through every branch."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "vcp3d_open_amd", "libvcp3d_amd.so")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects():
    """The gfx950 code objects of the library."""
    data = open(LIB, "rb").read()
    at, out = data.find(MAGIC), []
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + length]:
                out.append(data[at + offset:at + offset + size])
            entry += 24 + length
        at = data.find(MAGIC, at + 1)
    return out


EVENT = re.compile(r"^\s+(ds_\w+|flat_\w+|s_waitcnt|s_barrier|s_c?branch\w*|s_endpgm|s_setpc\w*)\b([^/]*)//\s*([0-9A-F]+):")


def functions(text):
    name, events = None, []
    for line in text.splitlines():
        if line.endswith(">:"):
            if events:
                yield name, events
            name, events = line.split("<", 1)[1][:-2], []
        elif m := EVENT.match(line):
            events.append((m.group(1), m.group(2).strip(), int(m.group(3), 16)))
    if events:
        yield name, events


def outstanding_at_barriers(events):
    """Addresses of the barriers that a path reaches with an LDS access outstanding."""
    addresses = [a for _, _, a in events]
    first_at = {}
    for i, (op, arg, a) in enumerate(events):
        if op.startswith(("s_branch", "s_cbranch")):
            offset = int(arg.split()[0])
            target = a + 4 + 4 * (offset - 65536 if offset >= 32768 else offset)
            # the first event at or behind the target
            lo, hi = 0, len(addresses)
            while lo < hi:
                mid = (lo + hi) // 2
                lo, hi = (mid + 1, hi) if addresses[mid] < target else (lo, mid)
            first_at[i] = lo
    most = {0: 0}                      # event -> most accesses outstanding before it
    todo, bad = [0], set()
    while todo:
        i = todo.pop()
        n = most[i]
        while i < len(events):
            op, arg, a = events[i]
            if op.startswith(("ds_", "flat_")):
                n = min(n + 1, 64)
            elif op == "s_waitcnt":
                if m := re.search(r"lgkmcnt\((\d+)\)", arg):
                    n = min(n, int(m.group(1)))
            elif op == "s_barrier" and n:
                bad.add(a)
            elif op.startswith(("s_endpgm", "s_setpc")):
                break
            follow = [first_at[i]] if i in first_at else []
            if not op.startswith("s_branch"):
                follow.append(i + 1)
            for j in follow[:-1]:
                if most.get(j, -1) < n:
                    most[j] = n
                    todo.append(j)
            i = follow[-1]
            if most.get(i, -1) >= n:
                break
            most[i] = n
    return bad


def test_the_count_follows_branches():
    """A store behind which a loop branches back to its barrier is found, with
    the wait in the loop's head alone as well as at its end."""
    loop = [("s_waitcnt", "lgkmcnt(0)", 0), ("s_barrier", "", 4), ("ds_read_b64", "", 8), ("ds_write_b64", "", 16),
            ("s_cbranch_scc1", "65531", 20), ("s_endpgm", "", 24)]
    assert outstanding_at_barriers(loop) == {4}              # back to the barrier itself
    loop[4] = ("s_cbranch_scc1", "65530", 20)
    assert outstanding_at_barriers(loop) == set()            # back to the wait
    loop[3:5] = [("ds_write_b64", "", 12), ("s_waitcnt", "lgkmcnt(0)", 16), ("s_cbranch_scc1", "65531", 20)]
    assert outstanding_at_barriers(loop) == set()


@pytest.mark.slow
def test_no_access_outstanding_at_a_barrier(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and ROCm's llvm-objdump")
    found, barriers = {}, 0
    for i, code in enumerate(code_objects()):
        path = str(tmp_path / f"{i}.elf")
        with open(path, "wb") as f:
            f.write(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", path], capture_output=True, text=True,
                              check=True).stdout
        for name, events in functions(text):
            barriers += sum(op == "s_barrier" for op, _, _ in events)
            if bad := outstanding_at_barriers(events):
                found[name] = len(bad)
    assert barriers > 100
    assert not found, found
