"""Every object of the library depends on the headers its source includes, so that a
build after a change to a header leaves no stale object."""
import os
import re
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cnn-crf-stereo_amd")


def headers(path, seen=None):
    """The .hpp files beside it that a source includes, directly or not."""
    seen = set() if seen is None else seen
    with open(path) as f:
        for name in re.findall(r'^#include "([\w.]+\.hpp)"', f.read(), re.M):
            if name not in seen:
                seen.add(name)
                headers(os.path.join(os.path.dirname(path), name), seen)
    return seen


def prerequisites():
    """Object -> prerequisites, as make reads the rules."""
    out = subprocess.run(["make", "-C", PKG, "-pnB", "libccs.so"], capture_output=True, text=True, check=True).stdout
    return {m.group(1): set(m.group(2).split()) for m in re.finditer(r"^_build/(\w+)\.o: (.*)$", out, re.M)}


@pytest.mark.parametrize("source", sorted(f for f in os.listdir(os.path.join(PKG, "csrc")) if f.endswith(".hip")))
def test_object_depends_on_its_headers(source):
    deps = prerequisites()[source[:-4]]
    assert not {h for h in headers(os.path.join(PKG, "csrc", source)) if "csrc/" + h not in deps}
