"""The native build compiles a translation unit again when a header that it includes has changed."""
import os
import re

import pytest

from symmetry_amd import _build

KERNELS = os.path.join(_build.CSRC, "kernels")


def _reached(path):
    """Names of the headers that a source includes, itself or through another header."""
    names, todo = set(), [path]
    while todo:
        for name in re.findall(r'#include "([^"]+)"', open(todo.pop()).read()):
            if name not in names and os.path.exists(os.path.join(KERNELS, name)):
                names.add(name)
                todo.append(os.path.join(KERNELS, name))
    return names


@pytest.mark.parametrize("header", sorted(n for n in os.listdir(KERNELS) if n.endswith(".h")))
def test_a_changed_header_reaches_its_units(header, monkeypatch):
    ran = []
    monkeypatch.setattr(_build, "_newer", lambda target, deps: header in [os.path.basename(d) for d in deps])
    monkeypatch.setattr(_build, "_run", lambda cmd, verbose: ran.append(cmd))
    monkeypatch.setattr(_build.os, "replace", lambda *a: None)
    for build in (_build.build_kernels, _build.build_latent, _build.build_hybrid):
        build()
    units = {os.path.basename(cmd[2]) for cmd in ran if cmd[1] == "-c"}
    folders = (KERNELS, os.path.join(_build.CSRC, "bindings"))
    sources = [os.path.join(d, n) for d in folders for n in os.listdir(d) if n.endswith((".hip", ".cpp"))]
    missed = {os.path.basename(s) for s in sources if header in _reached(s)} - units
    assert not missed
