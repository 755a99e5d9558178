"""The Makefile's prerequisites: an object is rebuilt when a file that its
source includes, directly or through a header, has changed (CPU)."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "agdeblend_amd", "csrc")
INCLUDE = os.path.join(CSRC, "..", "..", "include")
SOURCES = sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".c")))


def _included(path, seen):
    with open(path) as f:
        for name in re.findall(r'^\s*#include "([^"]+)"', f.read(), re.M):
            for d in (CSRC, INCLUDE):
                p = os.path.normpath(os.path.join(d, name))
                if os.path.exists(p) and p not in seen:
                    seen.add(p)
                    _included(p, seen)
    return seen


@pytest.mark.parametrize("source", SOURCES)
def test_object_depends_on_every_included_file(source, tmp_path):
    obj = os.path.join(str(tmp_path), os.path.splitext(source)[0] + ".o")
    files = sorted(_included(os.path.join(CSRC, source), set()))
    assert files
    open(obj, "w").close()
    os.utime(obj, (2 ** 31, 2 ** 31))  # newer than its sources

    def rebuilt(changed):
        cmd = ["make", "-n", "-C", CSRC, "OBJ=" + str(tmp_path), obj] + changed
        out = subprocess.run(cmd, capture_output=True, text=True, check=True).stdout
        return " -c " in out

    assert not rebuilt([])
    for f in files:
        assert rebuilt(["-W", os.path.relpath(f, CSRC)]), "%s does not depend on %s" % (source, f)
