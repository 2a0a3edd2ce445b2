"""Backward pass of small layers: input gradients whose waves share output channels."""
import ctypes as C

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from fitre_amd import lib as L
from fitre_amd.structs import fitre_conv_shape

pytestmark = pytest.mark.gpu
hip = L.hip


def ok(rc):
    assert rc == 0, hip.fitre_hip_last_error().decode()


# images, channels in and out, map, window, padding.  Tasks of a workgroup: one (four shares), two, three, several; fewer channels than shares;
# rows that are no whole groups
@pytest.mark.parametrize("n,ci,co,a,k,pad", [(16, 6, 16, 14, 5, 0), (128, 6, 16, 14, 5, 0), (300, 2, 3, 9, 3, 1), (7, 3, 1, 11, 5, 2), (200, 3, 2, 13, 7, 3),
                                             (5, 1, 31, 10, 3, 0), (170, 6, 7, 15, 5, 2), (600, 3, 5, 32, 5, 0)])
def test_input_gradient(dev, n, ci, co, a, k, pad):
    o = a + 2 * pad - k + 1
    s = fitre_conv_shape(n, ci, co, a, a, o, o, k, 1, pad)
    rng = np.random.default_rng(n)
    d, w = rng.standard_normal((co, n, o, o)).astype(np.float32), rng.standard_normal((co, ci, k, k)).astype(np.float32)
    nb = hip.fitre_hip_conv_input_grad_workspace(C.byref(s))
    ws, out = dev.alloc(max(nb, 4)), dev.upload(np.full(ci * n * a * a + 4, 7, np.float32))
    ok(hip.fitre_hip_conv_input_grad(C.byref(s), dev.upload(d.reshape(-1)), dev.upload(w.reshape(-1)), out, ws, nb))
    back = lambda x, y: F.conv_transpose2d(torch.from_numpy(x).double().transpose(0, 1), torch.from_numpy(y).double(), padding=pad).transpose(0, 1).numpy().reshape(-1)
    got, want, size = dev.download(out, ci * n * a * a + 4), back(d, w), back(abs(d), abs(w))
    assert (got[-4:] == 7).all()
    # one rounding per term and sum: error at most (terms + 3) u times the terms' sizes
    assert (abs(got[:-4] - want) <= (co * k * k + 3) * 2.0**-24 * 1.01 * size).all()
