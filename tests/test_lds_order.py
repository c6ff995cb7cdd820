"""Data that lanes or waves pass to each other in LDS without __syncthreads is ordered in the source
(no GPU needed): a wave barrier alone constrains scheduling and not memory, so it appears only inside
nmx_lds_wave_sync, between its two fences; and a loop that waits for another wave's progress is
followed by an acquire fence before anything it guards."""
from __future__ import annotations

import re
from pathlib import Path

import pytest

HIP = sorted((Path(__file__).resolve().parent.parent / "nibblemac_amd" / "csrc" / "hip").glob("nmx_*"))


def code(path: Path) -> str:
    return re.sub(r"//[^\n]*|/\*.*?\*/", "", path.read_text(), flags=re.S)


@pytest.mark.parametrize("path", HIP, ids=lambda p: p.name)
def test_wave_barriers_are_fenced(path):
    text = code(path)
    sync = re.compile(r'__builtin_amdgcn_fence\(__ATOMIC_RELEASE, "wavefront", "local"\);\s*'
                      r"__builtin_amdgcn_wave_barrier\(\);\s*"
                      r'__builtin_amdgcn_fence\(__ATOMIC_ACQUIRE, "wavefront", "local"\);')
    assert text.count("__builtin_amdgcn_wave_barrier") == len(sync.findall(text))


@pytest.mark.parametrize("path", HIP, ids=lambda p: p.name)
def test_waits_acquire(path):
    """Empty-bodied loops on an atomic load, named or through a lambda of one."""
    text = code(path)
    polls = ["__hip_atomic_load"] + re.findall(r"auto (\w+) = \[&\]\([^)]*\) \{\s*return __hip_atomic_load", text)
    for m in re.finditer(r"while \((?:%s)\([^{}]*\) \{\s*\}" % "|".join(polls), text):
        assert re.match(r"\s*__builtin_amdgcn_fence\(__ATOMIC_ACQUIRE,", text[m.end():]), \
            f"{path.name}: no acquire fence after `{m.group(0).split(chr(10))[0]}`"
