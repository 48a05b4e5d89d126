"""The libraries of one design's sources load by themselves: whatever of this project their sources call, they define."""

import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from ohara_amd import build

NAMES = sorted(set().union(*build.SERVING.values()))


@pytest.fixture(scope="module")
def symbols(tmp_path_factory):
    """Source -> (what it defines, what it needs), from its host code."""
    nm = shutil.which("nm") or "/opt/rocm/llvm/bin/llvm-nm"
    if not os.path.exists(build.HIPCC) or not os.path.exists(nm):
        pytest.skip("no compiler here")
    out = tmp_path_factory.mktemp("host")

    def one(name):
        obj = str(out / f"{name}.o")
        build._run([build.HIPCC, *build.FLAGS, "-O0", "--cuda-host-only", "-c", os.path.join(build.CSRC, f"{name}.hip"), "-o", obj])
        listed = lambda what: {line.split()[-1] for line in subprocess.run([nm, what, obj], capture_output=True, text=True, check=True).stdout.splitlines()}  # noqa: E731
        return listed("--defined-only"), {s for s in listed("--undefined-only") if "ohara_" in s}

    with ThreadPoolExecutor(8) as pool:
        return dict(zip(NAMES, pool.map(one, NAMES)))


@pytest.mark.parametrize("design", sorted(build.SERVING))
def test_nothing_is_missing(symbols, design):
    parts = [symbols[name] for name in build.SERVING[design]]
    defined, needed = (set().union(*(p[i] for p in parts)) for i in range(2))
    assert needed, "the sources call each other"
    assert needed <= defined, sorted(needed - defined)
