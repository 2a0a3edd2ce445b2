"""Backward pass of small layers: input gradients whose waves share output channels or go on through a pool, weight gradients made together."""
import ctypes as C

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from fitre_amd import lib as L
from fitre_amd.structs import ACT_TANH, AVG_POOL, CNN_ACT_NONE, CNN_ACT_RELU, CNN_ACT_SWISH, MAX_POOL, fitre_conv_shape, fitre_fc_tail_layer

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


@pytest.mark.parametrize("n", [1, 13, 512, 700])
def test_weight_gradients_together(dev, n):
    """Held back with the linear layers' above and made in one launch (a fifth layer makes the first four's): the bits of the calls alone,
    and nothing written before."""
    rng = np.random.default_rng(n)
    up = lambda size: dev.upload(rng.standard_normal(size).astype(np.float32))
    full = lambda size: dev.upload(np.full(size, 7, np.float32))
    shapes = [fitre_conv_shape(n, ci, co, a, b, a + 2 * p - k + 1, b + 2 * p - k + 1, k, 1, p)
              for ci, co, a, b, k, p in [(3, 6, 32, 32, 5, 0), (6, 16, 14, 14, 5, 0), (2, 1, 7, 12, 3, 1), (1, 8, 9, 9, 5, 2), (4, 9, 10, 11, 3, 0)]]
    convs = [(s, up(s.inChannels * n * s.inA * s.inB), up(s.outChannels * n * s.outA * s.outB)) for s in shapes]
    dims = [(65, 33), (33, 31), (31, 2)]
    W, zin, top = [up(i * o) for i, o in dims], [up(n * i) for i, _ in dims], up(2 * n)

    def run(held):
        bufs, outs = [], []
        tail = (fitre_fc_tail_layer * 3)()
        for t, (i, o) in enumerate(dims):
            slot, dW, db = full(n * o), full(i * o), full(o)
            tail[t] = fitre_fc_tail_layer(i, o, CNN_ACT_NONE, W[t].value, None, None, zin[t].value, slot.value, dW.value, db.value)
            outs += [(dW, i * o), (db, o)]
            bufs.append(slot)
        if held:
            ok(hip.fitre_hip_weight_grads_defer())
        nb = hip.fitre_hip_fc_tail_workspace(3, tail, n)
        ok(hip.fitre_hip_fc_tail_backward(3, tail, n, top, 0, 0, full(n * 65), dev.alloc(max(nb, 4)), nb))
        for s, x, d in convs:
            assert hip.fitre_hip_thin_reduce_bytes(C.byref(s)) > 0
            nb = max(hip.fitre_hip_conv_weight_bias_grad_workspace(C.byref(s)), hip.fitre_hip_thin_reduce_bytes(C.byref(s)))
            size = s.outChannels * s.inChannels * s.ksize**2
            dW, db = full(size), full(s.outChannels)
            ok(hip.fitre_hip_conv_weight_bias_grad(C.byref(s), x, d, dW, db, dev.alloc(nb), nb))
            outs += [(dW, size), (db, s.outChannels)]
        if held:
            assert all((dev.download(*o) == 7).all() for o in outs[-2:])
            ok(hip.fitre_hip_thin_reduce_defer(0))
        return [dev.download(*o).view(np.uint32) for o in outs]

    for alone, together in zip(run(False), run(True)):
        np.testing.assert_array_equal(together, alone)


@pytest.mark.parametrize("pool", [MAX_POOL, AVG_POOL])
@pytest.mark.parametrize("act", [CNN_ACT_NONE, CNN_ACT_RELU, CNN_ACT_SWISH, ACT_TANH])
@pytest.mark.parametrize("n,ci,co,a,b,k", [(16, 6, 16, 14, 14, 5), (3, 5, 7, 6, 10, 3), (130, 2, 3, 5, 7, 3)])
def test_through_a_pool(dev, n, ci, co, a, b, k, act, pool):
    """An input gradient and a linear tail's delta taken on through the pool and activation below: the bits of the steps of their own."""
    s = fitre_conv_shape(n, ci, co, a, b, a - k + 1, b - k + 1, k, 1, 0)
    rng = np.random.default_rng(n + act)
    up = lambda size: dev.upload(rng.standard_normal(size).astype(np.float32))
    full = lambda size: dev.upload(np.full(size, 7, np.float32))
    cells = ci * n * a * b
    d, w, zi, za = up(co * n * s.outA * s.outB), up(co * ci * k * k), up(4 * cells), up(4 * cells)
    nb = hip.fitre_hip_conv_input_grad_workspace(C.byref(s))
    ws = dev.alloc(max(nb, 4))
    got, want = [[full(cells), full(4 * cells), full(4 * cells)] for _ in range(2)]
    ok(hip.fitre_hip_conv_input_grad_pool_type_act(C.byref(s), d, w, got[0], pool, act, zi, za, got[1], got[2], ws, nb))
    ok(hip.fitre_hip_conv_input_grad(C.byref(s), d, w, want[0], ws, nb))
    behind = lambda t: ok(hip.fitre_hip_pool_act_backward(pool, act, t[0], zi, za, ci, n, 2 * a, 2 * b, 2, 2, 0, a, b, t[1], t[2]))
    behind(want)

    dims, tops = [(ci * a * b, 30), (30, 4)], up(4 * n)
    W, zin = [up(i * o) for i, o in dims], [up(n * i) for i, _ in dims]

    def tail(call):
        layers = (fitre_fc_tail_layer * 2)(*[fitre_fc_tail_layer(i, o, CNN_ACT_NONE, W[t].value, None, None, zin[t].value, full(n * o).value, full(i * o).value,
                                                                 full(o).value) for t, (i, o) in enumerate(dims)])
        size = hip.fitre_hip_fc_tail_workspace(2, layers, n)
        ok(call(layers, dev.alloc(max(size, 4)), size))

    if hip.fitre_hip_fc_tail_fits(2, (fitre_fc_tail_layer * 2)(*[fitre_fc_tail_layer(i, o, CNN_ACT_NONE) for i, o in dims]), n):
        x, y = [[full(cells), full(4 * cells), full(4 * cells)] for _ in range(2)]
        tail(lambda l, v, size: hip.fitre_hip_fc_tail_backward_pool_type_act(2, l, n, tops, a, b, x[0], pool, act, zi, za, x[1], x[2], v, size))
        tail(lambda l, v, size: hip.fitre_hip_fc_tail_backward(2, l, n, tops, a, b, y[0], v, size))
        behind(y)
        got, want = got + x, want + y
    for i, (u, v) in enumerate(zip(got, want)):
        size = 4 * cells if i % 3 else cells
        np.testing.assert_array_equal(dev.download(u, size), dev.download(v, size))
    assert hip.fitre_hip_conv_input_grad_pool_type_act(C.byref(s), d, w, got[0], 77, act, zi, za, got[1], got[2], ws, nb) != 0


def test_work_held_back_ends_with_the_device_layer(dev):
    """Neither what was held back before a shutdown nor the request to hold more reaches the layer that is set up after it."""
    n, ci, co = 13, 6, 16
    s = fitre_conv_shape(n, ci, co, 14, 14, 10, 10, 5, 1, 0)
    rng = np.random.default_rng(4)
    x, d = (dev.upload(rng.standard_normal(size).astype(np.float32)) for size in (ci * n * 196, co * n * 100))
    dims, size = [(65, 33), (33, 4)], co * ci * 25
    W, zin = [dev.zeros(i * o) for i, o in dims], [dev.zeros(n * i) for i, _ in dims]
    dW, db, nb = dev.zeros(size), dev.zeros(co), hip.fitre_hip_conv_weight_bias_grad_workspace(C.byref(s))
    ws = dev.alloc(nb)
    tail = (fitre_fc_tail_layer * 2)(*[fitre_fc_tail_layer(i, o, CNN_ACT_NONE, W[t].value, None, None, zin[t].value, dev.zeros(n * o).value,
                                                           dev.zeros(i * o).value, dev.zeros(o).value) for t, (i, o) in enumerate(dims)])
    tail_nb = hip.fitre_hip_fc_tail_workspace(2, tail, n)
    grads = lambda: ok(hip.fitre_hip_conv_weight_bias_grad(C.byref(s), x, d, dW, db, ws, nb))

    def made():  # weight gradients and reductions of partial sums; the linear products are in the first
        out = []
        for kernel_class in (0, 3, 4):
            count, ms, work = C.c_long(), C.c_double(), C.c_double()
            ok(hip.fitre_hip_profile_read(kernel_class, C.byref(count), C.byref(ms), C.byref(work)))
            out.append(count.value)
        return out

    ok(hip.fitre_hip_weight_grads_defer())
    ok(hip.fitre_hip_fc_tail_backward(2, tail, n, dev.zeros(4 * n), 0, 0, dev.zeros(n * 65), dev.alloc(max(tail_nb, 4)), tail_nb))
    grads()
    ok(hip.fitre_hip_shutdown())
    ok(hip.fitre_hip_init(0))
    ok(hip.fitre_hip_profile_enable(1))
    ok(hip.fitre_hip_thin_reduce_flush())
    assert made() == [0, 0, 0]
    grads()
    assert made() == [1, 0, 1]
    ok(hip.fitre_hip_profile_enable(0))
    assert dev.download(dW, size).any()
