"""Workspace queries: host functions, no GPU needed."""
import ctypes as C

import pytest

from fitre_amd import lib as L
from helpers import conv_shape


@pytest.mark.parametrize("k", [3, 5])
@pytest.mark.parametrize("a,b", [(0, 8), (8, 0), (65536, 65536), (1 << 30, 4), (-1, 1)])
def test_shapes_that_are_no_map(k, a, b):
    """A query does not know yet whether the shape is one (the call that uses the workspace says so): it returns."""
    s = conv_shape(4, 32, 32, a, b, k, 1, k // 2)
    for query in (L.hip.fitre_hip_conv_forward_workspace, L.hip.fitre_hip_conv_weight_grad_workspace, L.hip.fitre_hip_conv_input_grad_workspace,
                  L.hip.fitre_hip_conv_input_grad_prepared_bytes):
        query(C.byref(s))
