"""Weight copies made for several layers at once, and a sweep without waits: the bits of the steps they replace."""
import ctypes as C

import numpy as np
import pytest

from fitre_amd import lib as L
from fitre_amd.structs import CNN_ACT_RELU, MAX_POOL, NO_POOL, fitre_conv_shape

pytestmark = pytest.mark.gpu
hip = L.hip


def ok(rc):
    assert rc == 0, hip.fitre_hip_last_error().decode()


# samples, channels in and out, map, window: both windows, ragged groups of channels, the cell form, the dense form
LAYERS = [(96, 64, 130, 13, 3), (64, 64, 192, 15, 5), (300, 256, 512, 4, 3), (130, 512, 64, 2, 3), (128, 96, 300, 8, 3), (132, 64, 68, 2, 3)]


def layer(n, ci, co, a, k):
    return fitre_conv_shape(n, ci, co, a, a, a, a, k, 1, k // 2)


@pytest.mark.parametrize("grad", [0, 1])
def test_copies_of_several_layers(dev, grad):
    """One call for all of them leaves in every buffer what a call for the layer alone does."""
    shapes = [layer(*g) for g in LAYERS]
    query = hip.fitre_hip_conv_input_grad_prepared_bytes if grad else hip.fitre_hip_conv_forward_prepared_bytes
    shapes = [s for s in shapes if query(C.byref(s))] * 5  # more than one launch holds
    assert len(shapes) > 16
    rng = np.random.default_rng(1)
    w = [dev.upload(rng.standard_normal(s.inChannels * s.outChannels * s.ksize ** 2).astype(np.float32)) for s in shapes]
    size = [query(C.byref(s)) for s in shapes]
    one, all_ = ([dev.upload(np.full(b // 4 + 4, 7, np.float32)) for b in size] for _ in range(2))
    for s, a, o in zip(shapes, w, one):
        ok(hip.fitre_hip_conv_prepare_weights(1, C.byref(s), C.byref(C.c_void_p(a.value)), C.byref(C.c_void_p(o.value)), grad))
        if grad:
            ok(hip.fitre_hip_conv_input_grad_prepare(C.byref(s), a, o, query(C.byref(s))))
    n = len(shapes)
    ok(hip.fitre_hip_conv_prepare_weights(n, (fitre_conv_shape * n)(*shapes), (C.c_void_p * n)(*[a.value for a in w]),
                                          (C.c_void_p * n)(*[a.value for a in all_]), grad))
    for b, x, y in zip(size, one, all_):
        got = dev.download(y, b // 4 + 4).view(np.uint32)
        np.testing.assert_array_equal(got, dev.download(x, b // 4 + 4).view(np.uint32))
        assert (got[-4:].view(np.float32) == 7).all()
    bad = layer(1, 3, 3, 5, 3)
    assert hip.fitre_hip_conv_prepare_weights(1, C.byref(bad), C.byref(C.c_void_p(w[0].value)), C.byref(C.c_void_p(one[0].value)), grad) != 0


def test_accounted_bytes_of_several_layers_copies(dev):
    """A launch's bytes are those of its own layers: both windows and, behind them, the dense form."""
    shapes = [layer(*LAYERS[i]) for i in (0, 1, 4, 5)]
    buf = lambda words: C.c_void_p(dev.zeros(words).value)
    w = [buf(s.inChannels * s.outChannels * s.ksize ** 2) for s in shapes]
    to = [buf(hip.fitre_hip_conv_forward_prepared_bytes(C.byref(s)) // 4 + 1) for s in shapes]

    def accounted(which):
        n = len(which)
        ok(hip.fitre_hip_profile_enable(1))
        ok(hip.fitre_hip_conv_prepare_weights(n, (fitre_conv_shape * n)(*[shapes[i] for i in which]), (C.c_void_p * n)(*[w[i].value for i in which]),
                                              (C.c_void_p * n)(*[to[i].value for i in which]), 0))
        count, kind, tile, ms, work = C.c_long(), C.c_int(), C.c_int(), C.c_double(), C.c_double()
        ok(hip.fitre_hip_profile_launch_count(C.byref(count)))
        out = []
        for i in range(count.value):
            ok(hip.fitre_hip_profile_read_launch(i, C.byref(kind), C.byref(tile), C.byref(ms), C.byref(work)))
            out.append(work.value)
        ok(hip.fitre_hip_profile_enable(0))
        return out

    (three,), (five,), (eight,), (dense,) = (accounted([i]) for i in range(4))
    assert min(three, five, eight, dense) > 0
    assert accounted([0, 1, 2, 3]) == [three + eight, five, dense]


@pytest.mark.parametrize("geom", LAYERS)
def test_forward_with_a_copy(dev, geom):
    """The same bits with the copy made beforehand as with the one made inside."""
    s = layer(*geom)
    n, ci, co, a, k = geom
    rng = np.random.default_rng(n)
    x, w = dev.upload(rng.standard_normal(ci * n * a * a).astype(np.float32)), dev.upload(rng.standard_normal(co * ci * k * k).astype(np.float32))
    bias, count, bytes_ = dev.upload(rng.standard_normal(co).astype(np.float32)), co * n * a * a, hip.fitre_hip_conv_forward_prepared_bytes(C.byref(s))
    assert bytes_ > 0
    copy = dev.alloc(bytes_)
    ok(hip.fitre_hip_conv_prepare_weights(1, C.byref(s), C.byref(C.c_void_p(w.value)), C.byref(C.c_void_p(copy.value)), 0))
    nb = hip.fitre_hip_conv_bn_act_pool_workspace(C.byref(s), 1)
    ws = dev.alloc(nb)
    pool = (MAX_POOL, 2, 2, 0, a // 2, a // 2) if a % 2 == 0 else (NO_POOL, 0, 0, 0, a, a)
    results = []
    for prepared in (None, copy):
        bufs = [dev.zeros(count), dev.zeros(count), dev.zeros(co), dev.zeros(co), dev.zeros(co), dev.zeros(co), dev.zeros(count), dev.zeros(count)]
        y, zhat, mean, var, rmean, rvar, act, top = bufs
        ok(hip.fitre_hip_conv_bn_act_pool_forward_prepared(C.byref(s), x, w, prepared, bias, y, zhat, mean, var, rmean, rvar, 1e-5, 0.9, 1, CNN_ACT_RELU, act,
                                                           *pool, top if pool[0] != NO_POOL else None, 0, ws, nb))
        results.append([dev.download(b, m) for b, m in zip(bufs, (count, count, co, co, co, co, count, count))])
    for u, v in zip(*results):
        np.testing.assert_array_equal(u, v)


def test_totals_of_a_sweep(dev):
    """Losses and hits added on the device are those a host adds up in floats, batch by batch."""
    rng = np.random.default_rng(3)
    loss, hits, last = (C.c_float() for _ in range(3))
    want_loss, want_hits = np.float32(0), np.float32(0)
    ok(hip.fitre_hip_totals_begin())
    for rows, classes in ((256, 10), (1, 10), (77, 3), (1000, 65)):
        logits, labels = dev.upload(rng.standard_normal((rows, classes)).astype(np.float32)), dev.upload(rng.integers(1, classes + 1, rows).astype(np.float32))
        probs, errors, h, dot = dev.zeros(rows * classes), dev.zeros(rows * classes), dev.zeros(rows), C.c_float()
        ok(hip.fitre_hip_softmax_cross_entropy_add(logits, labels, rows, classes, probs, errors))
        ok(hip.fitre_hip_accuracy_add(probs, labels, rows, classes, h))
        one = C.c_float()
        ok(hip.fitre_hip_softmax_cross_entropy(logits, labels, rows, classes, probs, errors, C.byref(one)))
        ok(hip.fitre_hip_accuracy_hits(probs, labels, rows, classes, h))
        ok(hip.fitre_hip_dot(rows, h, h, C.byref(dot)))
        want_loss = np.float32(want_loss + np.float32(np.float32(one.value) * np.float32(rows)))
        want_hits = np.float32(want_hits + np.float32(dot.value))
    ok(hip.fitre_hip_totals_end(C.byref(loss), C.byref(hits), C.byref(last)))
    assert (loss.value, hits.value, last.value) == (want_loss, want_hits, dot.value)
    ok(hip.fitre_hip_totals_begin())
    ok(hip.fitre_hip_totals_end(C.byref(loss), C.byref(hits), None))
    assert (loss.value, hits.value) == (0, 0)


@pytest.mark.parametrize("rows", [1, 77, 1024, 1025, 5000])
def test_mean_loss(dev, rows):
    """Up to 1024 rows the host takes the mean of the terms, above a kernel does; labels out of range add nothing."""
    rng = np.random.default_rng(rows)
    logits, labels = rng.standard_normal((rows, 10)).astype(np.float32), rng.integers(0, 13, rows)
    labels[-1] = 10
    loss, probs = C.c_float(), dev.zeros(rows * 10)
    ok(hip.fitre_hip_softmax_cross_entropy(dev.upload(logits), dev.upload(labels.astype(np.float32)), rows, 10, probs, dev.zeros(rows * 10), C.byref(loss)))
    p = dev.download(probs, rows * 10).reshape(rows, 10).astype(np.float64)
    kept = (labels >= 1) & (labels <= 10)
    want = -np.log(p[kept, labels[kept] - 1]).sum() / rows
    assert abs(loss.value - want) <= 4 * 2.0**-23 * want  # a logarithm's last place and one rounding of the mean
