"""A device allocation that fails (here: for want of a device) is reported once, by the call that
needed it, and leaves no error in the runtime for a later call to report."""

import ctypes

import pytest

from mnrt_amd import native as N


def test_failed_allocation_leaves_no_error():
    L = N.load()
    hip = ctypes.CDLL("libamdhip64.so")
    count = ctypes.c_int(0)
    if hip.hipGetDeviceCount(ctypes.byref(count)) == 0 and count.value > 0:
        pytest.skip("needs a machine without a device")
    hip.hipGetLastError()
    t = N.Tree()
    t.kind, t.num_nodes, t.d_nodes = N.KIND_POINT, 4, 64  # the address is not looked at: the allocation comes first
    assert L.mnrt_tree_collapse(ctypes.byref(t), 16, None) == -3
    assert not t.d_qnodes and not t.owns_qnodes
    assert hip.hipGetLastError() == 0
