"""The stack of edge-tree nodes that the lanes of a wave share in the selection
kernel: its top in LDS and the blocks of 64 entries below it in private memory
must behave exactly like a plain array stack (no reference counterpart;
self-checks on the device).  dr_test_tree_stack drives both with the same random
pushes and pops of sets of lanes, deep enough to spill and reload many blocks, half
the waves with the entries of the learned mixture (6 words), half with the plain
ones (4); dr_test_tree_walk expands trees as the selection does, up to the rule
that keeps a nearly full stack from overflowing, and past it."""
import ctypes

import pytest

from delta_ray_amd import _abi

pytestmark = pytest.mark.gpu


def test_lds_stack_matches_array_stack(gpu):
    lib = _abi.load_library()
    out = (ctypes.c_int64 * 2)()
    _abi.check(lib, lib.dr_test_tree_stack(4000, 17, out, None), "dr_test_tree_stack")
    assert out[0] == 0, "%d pops differ" % out[0]
    # the stack is filled to its capacity (32 entries a lane), far past the 2 in LDS
    assert out[1] == 32, out[1]


# 28 levels stay below the rule's line (1880 entries), 29 cross it, 31 is the deepest
# tree the builder accepts
@pytest.mark.parametrize("levels", [0, 1, 3, 28, 29, 30, 31])
def test_nearly_full_stack_loses_nothing(gpu, levels):
    lib = _abi.load_library()
    out = (ctypes.c_int64 * 4)()
    _abi.check(lib, lib.dr_test_tree_walk(levels, 1, out, None), "dr_test_tree_walk")
    assert list(out)[:3] == [0, 32 * 64 * (2 * levels + 1), 0], list(out)
    assert out[3] <= 2048, out[3]
    assert levels < 29 or out[3] > 1880, out[3]


def test_full_stack_is_counted(gpu):
    """without the rule, a chain deeper than the stack finds it full: what it cannot
    push is counted, and what it holds stays right"""
    lib = _abi.load_library()
    out = (ctypes.c_int64 * 4)()
    _abi.check(lib, lib.dr_test_tree_walk(100, 0, out, None), "dr_test_tree_walk")
    assert out[0] == 0 and out[2] > 0 and out[3] <= 2048, list(out)
    assert out[1] + out[2] == 32 * 64 * 201, list(out)
