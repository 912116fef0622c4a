"""What no run of a built kernel shows: properties of the kernels' sources and of the code that was built from them."""

import os
import re

import pytest

from kllm_amd.csrc import build

SOURCES = [f for f in build.sources() if "global_load_lds" in open(os.path.join(build.HERE, f)).read()]


@pytest.mark.parametrize("name", SOURCES)
def test_loads_into_lds_are_waited_for_in_front_of_a_barrier(name):
    """A barrier waits for no load from memory, and what another wave reads behind it has to be in LDS: between a load that goes there by itself
    and the next barrier in the text there is a wait for it, written out (where the barrier is a function's or a loop's, in that text)."""
    text = open(os.path.join(build.HERE, name)).read()
    for load in re.finditer(r"__builtin_amdgcn_global_load_lds", text):
        rest = text[load.end():]
        barrier = re.search(r"__syncthreads\(\)|_barrier\(\)", rest)
        assert barrier is None or not barrier.group().startswith("__sync") or "s_waitcnt" in rest[:barrier.start()], \
            text[:load.start()].count("\n") + 1
