"""The halo finder's peaks on different workgroups pass each other tags and done
flags by agent-scope atomics alone, in an order that gfx950 guarantees: no other
access to these words is written, and no other target is compiled."""
import os
import re
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cube_nufluid_amd", "csrc", "halo.hip")
INC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include")
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")


def code():
    return re.sub(r"//[^\n]*", "", open(SRC).read())


def function(name):
    text = code()
    at = text.index(name + "(", text.index("namespace {"))
    depth, i = 0, text.index("{", at)
    start = i
    while True:
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        if depth == 0:
            return text[start:i + 1]
        i += 1


def test_tags_and_flags_only_through_agent_scope_atomics():
    body = function("k_halo_process")
    uses = re.findall(r"([\w:]+)\(\s*(?:tag|done) \+", body)
    assert sorted(uses) == ["peak_finish", "peak_mark", "peak_word", "peak_word"]
    assert len(re.findall(r"\b(?:tag|done)\b", body)) == len(uses)
    for name in ("peak_word", "peak_mark", "peak_finish"):
        assert re.search(r"__hip_atomic_\w+\(.*__HIP_MEMORY_SCOPE_AGENT\)", function(name))


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
@pytest.mark.parametrize("arch,ok", [("gfx950", True), ("gfx942", False)])
def test_only_gfx950_compiles(arch, ok):
    r = subprocess.run([HIPCC, "-E", "--offload-device-only", "--offload-arch=" + arch, "-I" + INC, SRC], stdout=subprocess.DEVNULL,
                       stderr=subprocess.PIPE, text=True, timeout=300)
    assert (r.returncode == 0) == ok, r.stderr[-2000:]
    assert ok or "gfx950 guarantees" in r.stderr
