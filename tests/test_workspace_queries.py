"""Workspace queries: host functions, no GPU needed."""
import ctypes as C
import time

import pytest

from fitre_amd import lib as L
from fitre_amd import structs as S
from helpers import conv_shape


@pytest.mark.parametrize("k", [3, 5])
@pytest.mark.parametrize("a,b", [(0, 8), (8, 0), (65536, 65536), (1 << 30, 4), (-1, 1)])
def test_shapes_that_are_no_map(k, a, b):
    """A query does not know yet whether the shape is one (the call that uses the workspace says so): it returns."""
    s = conv_shape(4, 32, 32, a, b, k, 1, k // 2)
    for query in (L.hip.fitre_hip_conv_forward_workspace, L.hip.fitre_hip_conv_weight_grad_workspace, L.hip.fitre_hip_conv_input_grad_workspace,
                  L.hip.fitre_hip_conv_input_grad_prepared_bytes):
        query(C.byref(s))


def test_plans_of_a_network_are_searched_once():
    """The passes ask for their workspaces on every call: from the second time on without a search."""
    model = S.CNN_MODEL()
    L.cnn.readVGG16(C.byref(model), 123, 32, 32, 10, 3, 1, 1, S.CIFAR10)  # (a batch of no other test)

    def queries():
        start = time.perf_counter()
        for query in (L.cnn.cnnForwardMemRequired, L.cnn.cnnBackwardMemRequired, L.cnn.cnnHvMemRequired):
            query(C.byref(model))
        return time.perf_counter() - start

    first = queries()
    assert min(queries() for _ in range(20)) < first / 4
