"""Values that the lanes of one wavefront exchange through LDS.

The hardware keeps one wavefront's LDS operations in order, so no run shows a
missing fence; without one the compiler may move one lane's load ahead of
another lane's store.  The source is what can be checked: between the stores
and the loads of the panel's transposition stands the wavefront's fence.
"""
from __future__ import annotations

import os
import re

from conftest import REPO


def test_panel_transposition_is_fenced():
    src = open(os.path.join(REPO, "falcon-dns_amd", "csrc", "fdns_kernels.hip")).read()
    body = src[src.index("void k_lu_small("):src.index("constexpr size_t lu_small_lds(")]
    store = re.search(r"Ln\[\(16 \* t \+ 4 \* r \+ lk\) \* P \+ li\] = C\[r\];", body)
    load = re.search(r"act\[q\] \? Ln\[\(lane \+ 64 \* q\) \* P \+ c\]", body)
    assert store and load and store.end() < load.start()
    assert "wave_lds_sync();" in body[store.end():load.start()]


def test_wavefront_fence():
    src = open(os.path.join(REPO, "falcon-dns_amd", "csrc", "fdns_kernels.hip")).read()
    f = src[src.index("void wave_lds_sync()"):]
    f = f[:f.index("\n}")]
    i = [f.index(s) for s in ('__ATOMIC_RELEASE, "wavefront"', "__builtin_amdgcn_wave_barrier()",
                              '__ATOMIC_ACQUIRE, "wavefront"')]
    assert i == sorted(i)
