"""Device code hands data between lanes and wavefronts only through the two helpers that also bind the
compiler: a bare wave barrier or wait leaves it free to move the accesses around it."""
import os
import re

import pytest

from conftest import PKG_DIR

CSRC = os.path.join(PKG_DIR, "csrc")
SOURCES = sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".h", ".cpp")))


def _helper(text, name):
    m = re.search(r"__device__ __forceinline__ void %s\(\) \{\n(.*?)\n\}" % name, text, re.S)
    assert m, name
    return m.group(1)


def test_the_helpers_fence():
    text = open(os.path.join(CSRC, "np_internal.h")).read()
    lds, stores = _helper(text, "wave_lds_order"), _helper(text, "stores_done")
    assert "__builtin_amdgcn_fence" in lds and "__builtin_amdgcn_wave_barrier" in lds
    wait = stores.index("__builtin_amdgcn_s_waitcnt(0)")
    assert stores.index("__ATOMIC_RELEASE") < wait < stores.index("__ATOMIC_ACQUIRE")


@pytest.mark.parametrize("name", SOURCES)
def test_no_bare_barrier_or_wait(name):
    text = open(os.path.join(CSRC, name)).read()
    if name == "np_internal.h":
        for helper in ("wave_lds_order", "stores_done"):
            text = text.replace(_helper(text, helper), "")
    for call in ("__builtin_amdgcn_wave_barrier", "__builtin_amdgcn_s_waitcnt"):
        assert call not in text, (name, call)
