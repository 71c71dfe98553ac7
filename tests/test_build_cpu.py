"""How the library is built: what its kernels are bundled in, and what a changed
header rebuilds."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mechafm_amd", "csrc")
LIB = os.path.join(ROOT, "mechafm_amd", "lib", "libmafm.so")


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_kernels_are_loaded_in_small_parts():
    """The runtime loads all kernels of a source file when the first one is
    launched, 2 ms a MB, so a program's first scan pays for its whole file."""
    data = open(LIB, "rb").read()
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)]
    assert len(starts) > 10
    sizes = []
    for s in starts:           # magic, number of entries, then offset, size and name length of each
        at, total = s + 24, 0
        n = int.from_bytes(data[at:at + 8], "little")
        at += 8
        for _ in range(n):
            off, size, length = (int.from_bytes(data[at + 8 * k:at + 8 * k + 8], "little") for k in range(3))
            total = max(total, off + size)
            at += 24 + length
        sizes.append(total)
    assert max(sizes) <= 2.5e6, sorted(sizes)[-3:]


def _includes(path, seen):
    """Local headers a source includes, directly or through others."""
    with open(path) as f:
        for name in re.findall(r'^#include "([^"]+)"', f.read(), re.M):
            p = os.path.normpath(os.path.join(os.path.dirname(path), name))
            if p not in seen:
                seen.add(p)
                _includes(p, seen)
    return seen


def test_objects_depend_on_every_header_they_include():
    """A changed header rebuilds each object that includes it (a stale one would be
    tested and timed with the old code)."""
    base = subprocess.run(["make", "-p", "-n", "all"], cwd=CSRC, capture_output=True, text=True, timeout=60).stdout
    rules = {}
    for m in re.finditer(r"^(\.\./lib/obj/\w+\.o):(?!=)(.*)$", base, re.M):
        deps = [os.path.normpath(os.path.join(CSRC, d)) for d in m.group(2).replace("|", " ").split()]
        rules.setdefault(os.path.basename(m.group(1)), set()).update(deps)
    assert len(rules) > 12
    missing = {}
    for obj, deps in rules.items():
        source = [d for d in deps if d.endswith((".hip", ".cpp"))]
        assert len(source) == 1, (obj, source)
        gone = _includes(source[0], set()) - deps
        if gone:
            missing[obj] = sorted(os.path.relpath(g, CSRC) for g in gone)
    assert not missing, missing
