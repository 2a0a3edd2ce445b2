"""A small network's forward pass in one launch (fitre_hip_thin_net_forward) against torch in float64 on the same float32 numbers."""
import ctypes as C

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from fitre_amd import lib as L
from fitre_amd import structs as S

pytestmark = pytest.mark.gpu
hip = L.hip

# images; convolutions (channels out, window, padding) on (channels, A, B); linear layers.  LeNet; one channel, odd numbers of channels
# and short rows; three layers with borders, the sixteenth channel and one pooled column; no linear layer; more linear parts than inputs
NETS = [(5, (3, 32, 32), [(6, 5, 0), (16, 5, 0)], [120, 84, 10]), (1, (1, 8, 12), [(5, 3, 1)], [7]),
        (3, (1, 28, 20), [(4, 3, 1), (9, 5, 1), (16, 3, 1)], [33, 3]), (2, (2, 6, 10), [(3, 5, 1)], []), (260, (1, 6, 6), [(2, 3, 0)], [2, 64])]
ACTS = [S.CNN_ACT_RELU, S.CNN_ACT_SWISH, S.ACT_TANH, S.CNN_ACT_NONE]


def activate(act, x):
    return {S.CNN_ACT_RELU: torch.relu, S.CNN_ACT_SWISH: lambda t: t * torch.sigmoid(t), S.ACT_TANH: torch.tanh, S.CNN_ACT_NONE: lambda t: t}[act](x)


@pytest.mark.parametrize("average", [0, 1])
@pytest.mark.parametrize("bias", [0, 1])
@pytest.mark.parametrize("n,image,convs,linears", NETS)
def test_forward(dev, n, image, convs, linears, average, bias):
    rng = np.random.default_rng(n + len(convs) + 10 * average + bias)
    rand = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    up = lambda a: dev.upload(np.ascontiguousarray(a).reshape(-1))
    c, a, b = image
    x = rand(c, n, a, b)
    h, want, got, terms = torch.from_numpy(x).double().transpose(0, 1), [], [], 1
    layers = (S.fitre_thin_net_layer * len(convs))()
    for i, (out, k, pad) in enumerate(convs):
        w, bw, act = rand(out, c, k, k) / np.float32(np.sqrt(c * k * k)), rand(out), ACTS[i % 3]
        oa, ob = a + 2 * pad - k + 1, b + 2 * pad - k + 1
        y = F.conv2d(h, torch.from_numpy(w).double(), torch.from_numpy(bw).double() if bias else None, padding=pad)
        z = activate(act, y)
        h = (F.avg_pool2d if average else F.max_pool2d)(z, 2)
        buf = [dev.upload(np.full(t.numel() + 4, 7, np.float32)) for t in (y, z, h)]
        layers[i] = S.fitre_thin_net_layer(S.fitre_conv_shape(n, c, out, a, b, oa, ob, k, 1, pad), act, average, up(w), up(bw) if bias else None, *buf)
        pooled = h.transpose(0, 1) if i + 1 < len(convs) else h.transpose(2, 3)  # the last one [n][c][b][a]
        want += [y.transpose(0, 1), z.transpose(0, 1), pooled]
        got += buf
        terms += c * k * k
        c, a, b = out, oa // 2, ob // 2
    f = h.transpose(2, 3).reshape(n, -1)
    rest = (S.fitre_fc_forward_layer * max(len(linears), 1))()
    for i, out in enumerate(linears):
        w, bw, act = rand(f.shape[1], out) / np.float32(np.sqrt(f.shape[1])), rand(out), ACTS[(i + 1) % 4]
        pre = f @ torch.from_numpy(w).double() + (torch.from_numpy(bw).double() if bias else 0)
        buf = [dev.upload(np.full(n * out + 4, 7, np.float32)) for _ in range(2)]
        rest[i] = S.fitre_fc_forward_layer(f.shape[1], out, act, up(w), up(bw) if bias else None, *buf)
        terms += f.shape[1]
        f = activate(act, pre)
        want += [pre, f]
        got += buf
    classes = f.shape[1]
    labels = rng.integers(1, classes + 1, n).astype(np.float32)
    labels[0] = classes + 1  # no class
    probs, errors, loss = dev.zeros(n * classes), dev.zeros(n * classes), C.c_float()
    assert hip.fitre_hip_thin_net_forward_fits(len(convs), layers, len(linears), rest, n, classes)
    rc = hip.fitre_hip_thin_net_forward(len(convs), layers, len(linears), rest, n, up(x), up(labels), classes, probs, errors, C.byref(loss))
    assert rc == 0, hip.fitre_hip_last_error().decode()
    # a sum of K terms in any order is off by K 2^-24 of the sum of their sizes at most; here they are normal and pass through few layers
    tol = terms * 2.0 ** -24
    for ptr, t in zip(got, want):
        v = dev.download(ptr, t.numel() + 4)
        np.testing.assert_array_equal(v[-4:], 7)
        t = t.reshape(-1).numpy()
        assert np.abs(v[:-4] - t).max() <= tol * max(1.0, np.abs(t).max())
    p = torch.softmax(f, 1).numpy() + 1e-10
    e, nll = p.copy(), np.zeros(n)
    for r in range(1, n):
        e[r, int(labels[r]) - 1] -= 1
        nll[r] = -np.log(p[r, int(labels[r]) - 1])
    assert np.abs(dev.download(probs, n * classes) - p.reshape(-1)).max() <= 4 * tol
    assert np.abs(dev.download(errors, n * classes) - e.reshape(-1) / n).max() <= 4 * tol / n
    assert abs(loss.value - nll.mean()) <= 16 * tol * max(1.0, nll.mean())


def test_other_networks_do_not_fit():
    layer = lambda n=4, ci=3, co=6, a=32, k=5, stride=1, pad=0, oa=28: S.fitre_thin_net_layer(S.fitre_conv_shape(n, ci, co, a, a, oa, oa, k, stride, pad), S.CNN_ACT_RELU, 0)
    fc = S.fitre_fc_forward_layer(6 * 14 * 14, 10, S.CNN_ACT_NONE)
    fits = lambda l, n=4, classes=10, rest=fc, linears=1: hip.fitre_hip_thin_net_forward_fits(1, C.byref(l), linears, C.byref(rest), n, classes)
    assert fits(layer())
    assert not fits(layer(co=17)) and not fits(layer(stride=2)) and not fits(layer(k=4, oa=29)) and not fits(layer(a=31, oa=27)) and not fits(layer(), classes=9)
    assert not fits(layer(n=3)) and not fits(layer(), linears=5) and not fits(layer(n=100000), n=100000) and not fits(layer(), rest=S.fitre_fc_forward_layer(77, 10, 0))
