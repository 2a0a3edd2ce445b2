"""The fused steps of the forward pass (include/fitre_hip.h) against float64 numpy on the same float32 operands."""
import ctypes as C

import numpy as np
import pytest
import torch

from fitre_amd import lib as L
from fitre_amd.structs import (ACT_LINEAR, ACT_LOGISTIC, ACT_TANH, AVG_POOL, CNN_ACT_ELU, CNN_ACT_NONE, CNN_ACT_RELU,
                               CNN_ACT_SOFTPLUS, CNN_ACT_SWISH, MAX_POOL, NO_POOL)

pytestmark = pytest.mark.gpu
hip = L.hip


def ok(rc):
    assert rc == 0, hip.fitre_hip_last_error().decode()


def act64(act, x):
    with np.errstate(over="ignore"):
        sig = 1.0 / (1.0 + np.exp(-x))
        return {CNN_ACT_RELU: np.maximum(x, 0), CNN_ACT_ELU: np.where(x < 0, np.expm1(np.minimum(x, 0)), x), CNN_ACT_SOFTPLUS: np.logaddexp(0, x),
                CNN_ACT_SWISH: x * sig, ACT_LOGISTIC: sig, ACT_TANH: np.tanh(x)}.get(act, x)


# (widths from the lowest layer's inputs up, samples, activations): the sample groups of four and their remainders, widths at
# and around powers of two, the widest layers that fit, one layer and four
RUNS = [((400, 120, 84, 10), 128, (CNN_ACT_RELU, CNN_ACT_RELU, CNN_ACT_NONE)), ((512, 10), 77, (CNN_ACT_NONE,)),
        ((1, 1), 1, (ACT_LOGISTIC,)), ((2048, 48), 3, (CNN_ACT_SWISH,)), ((95, 1024), 6, (CNN_ACT_SOFTPLUS,)),
        ((33, 64, 65, 127, 128), 9, (CNN_ACT_ELU, ACT_TANH, ACT_LINEAR, CNN_ACT_SWISH)), ((384, 192, 10), 1025, (CNN_ACT_SWISH, CNN_ACT_NONE))]


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("dims,n,acts", RUNS)
def test_run_of_small_layers_in_one_launch(dev, dims, n, acts, bias):
    from fitre_amd.structs import fitre_fc_forward_layer
    rng = np.random.default_rng(sum(dims) + n)
    layers = len(dims) - 1
    x = rng.standard_normal((n, dims[0])).astype(np.float32)
    ws = [(rng.standard_normal((dims[f], dims[f + 1])) / np.sqrt(dims[f])).astype(np.float32) for f in range(layers)]
    bs = [rng.standard_normal(dims[f + 1]).astype(np.float32) for f in range(layers)]
    arr = (fitre_fc_forward_layer * layers)()
    outs = []
    px = dev.upload(x.reshape(-1))
    for f in range(layers):
        size = dims[f + 1] * n
        outs.append((dev.upload(np.full(size + 8, 7.0, np.float32)), dev.upload(np.full(size + 8, 7.0, np.float32))))
        arr[f] = fitre_fc_forward_layer(dims[f], dims[f + 1], acts[f], dev.upload(ws[f].reshape(-1)).value,
                                        dev.upload(bs[f]).value if bias else None, outs[f][0].value, outs[f][1].value)
    assert hip.fitre_hip_fc_tail_forward_fits(layers, arr, n) == 1
    ok(hip.fitre_hip_fc_tail_forward(layers, arr, n, px))
    z, bound = x.astype(np.float64), 0.0
    for f in range(layers):
        pre = z @ ws[f].astype(np.float64) + (bs[f] if bias else 0.0)
        # rounding of a float32 sum of dims[f] terms, 2^-24 a step, and what the layers below carry in (their gain is about 1)
        bound = 4 * bound + (dims[f] + 16) * 2.0 ** -24
        z = act64(acts[f], pre)
        for want, p in ((pre, outs[f][0]), (z, outs[f][1])):
            got = dev.download(p, dims[f + 1] * n + 8)
            assert np.abs(got[:-8].reshape(n, -1) - want).max() <= bound * max(1.0, np.abs(pre).max())
            np.testing.assert_array_equal(got[-8:], 7.0)


def test_what_a_run_of_layers_refuses(dev):
    from fitre_amd.structs import fitre_fc_forward_layer

    def fits(dims, n=8):
        arr = (fitre_fc_forward_layer * 5)(*[fitre_fc_forward_layer(a, b, CNN_ACT_NONE, None, None, None, None) for a, b in dims])
        return hip.fitre_hip_fc_tail_forward_fits(len(dims), arr, n)
    assert fits([(2048, 48)]) and not fits([(2049, 40)]) and not fits([(8, 1025)]) and not fits([(2048, 49)])
    assert not fits([(8, 8), (9, 8)]) and not fits([(4, 4)] * 5) and not fits([(8, 8)], 0) and not fits([(512, 128)], 4096)


# channels, samples, A, B, window, stride, padding, kind: pooled cells (2 x 2 maps, rows of ten, one cell only), patches, windows
# that are pooled apart, no pool, and counts that are no multiple of four
LAST = [(16, 77, 2, 2, 2, 2, 0, MAX_POOL), (16, 33, 10, 10, 2, 2, 0, MAX_POOL), (5, 9, 6, 10, 2, 2, 0, AVG_POOL), (1, 1, 2, 2, 2, 2, 0, AVG_POOL),
        (6, 5, 4, 8, 2, 2, 0, MAX_POOL), (6, 4, 4, 8, 2, 2, 0, AVG_POOL), (4, 8, 7, 7, 3, 2, 0, MAX_POOL), (4, 8, 8, 8, 3, 2, 1, MAX_POOL),
        (3, 7, 4, 6, 0, 0, 0, NO_POOL), (3, 7, 3, 5, 0, 0, 0, NO_POOL), (3, 3, 5, 7, 2, 2, 0, MAX_POOL)]


@pytest.mark.parametrize("act", [CNN_ACT_RELU, CNN_ACT_SWISH])
@pytest.mark.parametrize("bn,train", [(True, 1), (True, 0), (False, 1)])
@pytest.mark.parametrize("geom", LAST)
def test_last_layer_in_the_linear_layers_order(dev, geom, bn, train, act):
    """fitre_hip_bn_act_pool_forward_fc and the plain form against normalisation, activation, pooling and permutation as
    launches of their own: the same bits where the statistics are (one workgroup's share of a channel here)."""
    c, n, a, b, k, s, p, kind = geom
    oa, ob = ((a + 2 * p - k) // s + 1, (b + 2 * p - k) // s + 1) if kind != NO_POOL else (a, b)
    per, count, pooled = n * a * b, c * n * a * b, c * n * oa * ob
    rng = np.random.default_rng(count + kind)
    px = dev.upload((3 * rng.standard_normal(count) + 1).astype(np.float32))
    nb = max(hip.fitre_hip_batch_norm_workspace(c, per), 4 * max(count, pooled))
    ws = dev.alloc(nb)

    def buffers():
        return [dev.upload(np.full(size, 0.5, np.float32)) for size in (count, count, pooled, c, c, c, c)]

    def fetch(bufs, order):
        got = [dev.download(q, size) for q, size in zip(bufs, (count, count, pooled, c, c, c, c))]
        return [got[i] for i in order]

    sep = buffers()
    src = px
    if bn:
        ok(hip.fitre_hip_batch_norm_forward(px, c, per, sep[0], *sep[3:], 1e-5, 0.9, train, ws, nb))
        src = sep[0]
    ok(hip.fitre_hip_activation_forward(act, src, sep[1], count))
    if kind != NO_POOL:
        ok(hip.fitre_hip_pool_forward(kind, sep[1], c, n, a, b, k, s, p, oa, ob, sep[2]))
    fc = dev.upload(np.zeros(pooled, np.float32))
    ok(hip.fitre_hip_conv_to_fc(sep[1] if kind == NO_POOL else sep[2], c, n, oa, ob, fc))
    for call, permuted in ((hip.fitre_hip_bn_act_pool_forward, False), (hip.fitre_hip_bn_act_pool_forward_fc, True)):
        one = buffers()
        ok(call(px, c, n, a, b, one[0] if bn else None, *(one[3:] if bn else [None] * 4), 1e-5, 0.9, train, act, one[1], kind, k, s, p, oa,
                ob, one[2] if kind != NO_POOL else None, ws, nb))
        for i in (0, 3, 4, 5, 6):
            np.testing.assert_array_equal(dev.download(one[i], count if i == 0 else c), dev.download(sep[i], count if i == 0 else c))
        last = 1 if kind == NO_POOL else 2
        for i, size in ((1, count), (2, pooled)):
            want = fc if permuted and i == last else sep[i]
            np.testing.assert_array_equal(dev.download(one[i], size), dev.download(want, size))


# samples, cin, cout, A, B, window, padding: LeNet's two layers (with and without border, images that share a workgroup and a
# remainder of them, one channel of a wave and two; the other channel groups are VARIANTS below), odd rows and columns, one channel, sixteen of each, 3 x 3
# windows without a border, and shapes that stay on the tile engine (more channels, seven-wide windows)
THIN = [(7, 3, 6, 32, 32, 5, 0), (130, 6, 16, 14, 14, 5, 0), (2100, 6, 16, 14, 14, 5, 0), (9, 3, 6, 28, 28, 5, 2), (5, 1, 1, 6, 6, 5, 0),
        (6, 16, 16, 7, 11, 5, 2), (11, 5, 7, 9, 6, 3, 0), (3, 2, 3, 5, 5, 5, 1), (4, 4, 4, 30, 9, 5, 4), (3, 3, 20, 12, 12, 5, 0), (3, 2, 4, 14, 14, 7, 0)]


@pytest.mark.parametrize("act", [CNN_ACT_RELU, CNN_ACT_SWISH])
@pytest.mark.parametrize("kind,to_fc", [(MAX_POOL, 1), (AVG_POOL, 0), (NO_POOL, 0)])
@pytest.mark.parametrize("geom", THIN)
def test_thin_convolution_with_activation_and_pool(dev, geom, kind, to_fc, act):
    """fitre_hip_conv_act_pool_forward: the convolution against float64, then activation, pool and permutation as launches
    of their own on what it wrote, the same bits."""
    from fitre_amd.structs import fitre_conv_shape
    n, ci, co, a, b, k, pad = geom
    oa, ob = a + 2 * pad - k + 1, b + 2 * pad - k + 1
    pa, pb = (oa // 2, ob // 2) if kind != NO_POOL else (oa, ob)
    rng = np.random.default_rng(n + ci * co + a)
    x = rng.standard_normal((ci, n, a, b)).astype(np.float32)
    w = (rng.standard_normal((co, ci, k, k)) / np.sqrt(ci * k * k)).astype(np.float32)
    bias = rng.standard_normal(co).astype(np.float32)
    count, pooled = co * n * oa * ob, co * n * pa * pb
    shape = fitre_conv_shape(n, ci, co, a, b, oa, ob, k, 1, pad)
    nb = max(hip.fitre_hip_conv_forward_workspace(C.byref(shape)), 4 * count)
    ws = dev.alloc(nb)
    px, pw = dev.upload(x.reshape(-1)), dev.upload(w.reshape(-1))
    for with_bias in (True, False):
        y, ao, po = (dev.upload(np.full(size + 4, 7.0, np.float32)) for size in (count, count, pooled))
        ok(hip.fitre_hip_conv_act_pool_forward(C.byref(shape), px, pw, dev.upload(bias) if with_bias else None, y, act, ao, kind, 2, 2, 0,
                                               pa, pb, po if kind != NO_POOL else None, to_fc, ws, nb))
        got = dev.download(y, count + 4)
        np.testing.assert_array_equal(got[-4:], 7.0)
        want = torch.nn.functional.conv2d(torch.from_numpy(x).double().transpose(0, 1), torch.from_numpy(w).double(),
                                          torch.from_numpy(bias).double() if with_bias else None, padding=pad).transpose(0, 1).numpy()
        # a float32 sum of ci * k * k terms of size one over their root, 2^-24 a step
        assert np.abs(got[:-4] - want.reshape(-1)).max() <= (ci * k * k + 16) * 2.0 ** -24 * max(1.0, np.abs(want).max())
        ref, pref = dev.zeros(count), dev.zeros(pooled)
        ok(hip.fitre_hip_activation_forward(act, y, ref, count))
        last = ref
        if kind != NO_POOL:
            ok(hip.fitre_hip_pool_forward(kind, ref, co, n, oa, ob, 2, 2, 0, pa, pb, pref))
            last = pref
        np.testing.assert_array_equal(dev.download(ao, count), dev.download(ref, count))
        if to_fc:
            out = dev.zeros(pooled)
            ok(hip.fitre_hip_conv_to_fc(last, co, n, pa, pb, out))
            last = out
        if kind != NO_POOL:
            got = dev.download(po, pooled + 4)
            np.testing.assert_array_equal(got[:-4], dev.download(last, pooled))
            np.testing.assert_array_equal(got[-4:], 7.0)


# samples, cin, cout, A, B: one workgroup per channel (4 x 4 and 2 x 2 maps, the cell kernel and the nine-tap one, the most cells
# of one segment), a channel that is no whole number of segments, one that is no multiple of four cells and is not summed here
SPLIT = [(32, 256, 64, 4, 4), (21, 128, 64, 2, 2), (64, 128, 128, 8, 8), (52, 64, 96, 14, 12), (3, 64, 40, 7, 7), (16, 512, 32, 13, 13)]


@pytest.mark.parametrize("bn,train", [(True, 1), (True, 0), (False, 1)])
@pytest.mark.parametrize("kind,to_fc", [(MAX_POOL, 0), (MAX_POOL, 1), (NO_POOL, 0), (NO_POOL, 1)])
@pytest.mark.parametrize("geom", SPLIT)
def test_split_convolution_summed_by_the_pass_behind_it(dev, geom, kind, to_fc, bn, train):
    """fitre_hip_conv_bn_act_pool_forward against fitre_hip_conv_forward and fitre_hip_bn_act_pool_forward(_fc): the same
    partials summed in the same order, the same bits."""
    from fitre_amd.structs import fitre_conv_shape
    n, ci, co, a, b = geom
    k, s = (2, 2) if a % 2 == 0 and b % 2 == 0 else (3, 2)
    pa, pb = ((a - k) // s + 1, (b - k) // s + 1) if kind != NO_POOL else (a, b)
    rng = np.random.default_rng(n + ci * co + a)
    count, pooled = co * n * a * b, co * n * pa * pb
    px = dev.upload(rng.standard_normal(ci * n * a * b).astype(np.float32))
    pw = dev.upload((rng.standard_normal(co * ci * 9) / np.sqrt(ci * 9)).astype(np.float32))
    pbias = dev.upload(rng.standard_normal(co).astype(np.float32))
    shape = fitre_conv_shape(n, ci, co, a, b, a, b, 3, 1, 1)
    nb = 2 * max(hip.fitre_hip_conv_bn_act_pool_workspace(C.byref(shape), 1), 4 * count)
    ws = dev.alloc(nb)
    sizes = (count, count, count, pooled, co, co, co, co)

    def passes(whole):
        y, zhat, act, pool, *stats = bufs = [dev.upload(np.full(size, 0.5, np.float32)) for size in sizes]
        norm = [zhat, *stats] if bn else [None] * 5
        rest = (1e-5, 0.9, train, CNN_ACT_SWISH, act, kind, k, s, 0, pa, pb, pool if kind != NO_POOL else None)
        if whole:
            ok(hip.fitre_hip_conv_bn_act_pool_forward(C.byref(shape), px, pw, pbias, y, *norm, *rest, to_fc, ws, nb))
        else:
            ok(hip.fitre_hip_conv_forward(C.byref(shape), px, pw, pbias, y, ws, nb))
            ok((hip.fitre_hip_bn_act_pool_forward_fc if to_fc else hip.fitre_hip_bn_act_pool_forward)(y, co, n, a, b, *norm, *rest, ws, nb))
        return [dev.download(q, size) for q, size in zip(bufs, sizes)]

    for got, want in zip(passes(True), passes(False)):
        np.testing.assert_array_equal(got, want)


# samples, cin, cout on 2 x 2 maps: the smallest batch of the dense form, ragged samples and channels, two to eight ranges
# (an uncut reduction, and several segments of a channel, are among DENSE below)
@pytest.mark.parametrize("bn,train", [(True, 1), (False, 1)])
@pytest.mark.parametrize("n,ci,co", [(128, 64, 64), (131, 68, 70), (256, 256, 96), (700, 64, 512)])
def test_forward_on_two_by_two_maps_as_a_dense_product(dev, n, ci, co, bn, train):
    """The convolution against float64; normalisation, activation and pool against fitre_hip_bn_act_pool_forward on it."""
    from fitre_amd.structs import fitre_conv_shape
    rng = np.random.default_rng(n + ci + co)
    x = rng.standard_normal((ci, n, 2, 2)).astype(np.float32)
    w = (rng.standard_normal((co, ci, 3, 3)) / np.sqrt(4 * ci)).astype(np.float32)
    bias = rng.standard_normal(co).astype(np.float32)
    px, pw, pbias = dev.upload(x.reshape(-1)), dev.upload(w.reshape(-1)), dev.upload(bias)
    count, pooled = co * n * 4, co * n
    shape = fitre_conv_shape(n, ci, co, 2, 2, 2, 2, 3, 1, 1)
    nb = hip.fitre_hip_conv_bn_act_pool_workspace(C.byref(shape), 1) + 4096
    ws = dev.alloc(nb)
    sizes = (count, count, pooled, co, co, co, co)

    def rest(y, call, *head):
        zhat, act, pool, *stats = bufs = [dev.upload(np.full(size, 0.5, np.float32)) for size in sizes]
        norm = [zhat, *stats] if bn else [None] * 5
        tail = (0, ws, nb) if call is hip.fitre_hip_conv_bn_act_pool_forward else (ws, nb)
        ok(call(*head, *norm, 1e-5, 0.9, train, CNN_ACT_RELU, act, MAX_POOL, 2, 2, 0, 1, 1, pool, *tail))
        return [dev.download(q, size) for q, size in zip(bufs, sizes)]

    y = dev.upload(np.full(count + 4, 7.0, np.float32))
    got = rest(y, hip.fitre_hip_conv_bn_act_pool_forward, C.byref(shape), px, pw, pbias, y)
    out = dev.download(y, count + 4)
    np.testing.assert_array_equal(out[-4:], 7.0)
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double().transpose(0, 1), torch.from_numpy(w).double(),
                                      torch.from_numpy(bias).double(), padding=1).transpose(0, 1).numpy()
    # a float32 sum of 4 * ci terms of size one over their root, 2^-24 a step
    assert np.abs(out[:-4] - want.reshape(-1)).max() <= (4 * ci + 16) * 2.0 ** -24 * max(1.0, np.abs(want).max())
    for a, b in zip(got, rest(y, hip.fitre_hip_bn_act_pool_forward, y, co, n, 2, 2)):
        if bn:
            np.testing.assert_allclose(a, b, rtol=1e-5, atol=1e-6)
        else:
            np.testing.assert_array_equal(a, b)


CONV_FWD, SPLITK_REDUCE, DENSE_2X2, THIN_MATRIX = 2, 4, 6, 12  # classes and tile variants of include/fitre_hip.h


def launches(kernel_class, tile=None):
    """Accounted launches of a class (or of one tile variant of it) since the accounting was turned on."""
    count, ms, work = C.c_long(), C.c_double(), C.c_double()
    args = (C.byref(count), C.byref(ms), C.byref(work))
    ok(hip.fitre_hip_profile_read(kernel_class, *args) if tile is None else hip.fitre_hip_profile_read_tile(kernel_class, tile, *args))
    return count.value


def layer_passes(dev, n, ci, co, a, b, bn, seed=0):
    """(shape, run): run(fused, nb, kind, to_fc, train, act) makes a 3 x 3 layer's passes with a workspace of nb bytes and returns
    what they wrote and the launches (convolution, dense form of it, reductions of partials)."""
    from fitre_amd.structs import fitre_conv_shape
    rng = np.random.default_rng(n + ci * co + a + seed)
    px = dev.upload(rng.standard_normal(ci * n * a * b).astype(np.float32))
    pw = dev.upload((rng.standard_normal(co * ci * 9) / np.sqrt(ci * 9)).astype(np.float32))
    pbias = dev.upload(rng.standard_normal(co).astype(np.float32))
    shape = fitre_conv_shape(n, ci, co, a, b, a, b, 3, 1, 1)
    count = co * n * a * b

    def run(fused, nb, kind=NO_POOL, to_fc=0, train=1, act=CNN_ACT_SWISH, y=None):
        k, s = (2, 2) if a % 2 == 0 and b % 2 == 0 else (3, 2)
        pa, pb = ((a - k) // s + 1, (b - k) // s + 1) if kind != NO_POOL else (a, b)
        ws = dev.alloc(nb)
        sizes = (count, count, count, co * n * pa * pb, co, co, co, co)
        q = [dev.upload(np.full(size, 0.5, np.float32)) for size in sizes]
        if y is not None:
            q[0] = y
        norm = [q[1], *q[4:]] if bn else [None] * 5
        rest = (1e-5, 0.9, train, act, q[2], kind, k, s, 0, pa, pb, q[3] if kind != NO_POOL else None)
        ok(hip.fitre_hip_profile_enable(1))
        if fused:
            ok(hip.fitre_hip_conv_bn_act_pool_forward(C.byref(shape), px, pw, pbias, q[0], *norm, *rest, to_fc, ws, nb))
        else:
            if y is None:
                ok(hip.fitre_hip_conv_forward(C.byref(shape), px, pw, pbias, q[0], ws, nb))
            ok((hip.fitre_hip_bn_act_pool_forward_fc if to_fc else hip.fitre_hip_bn_act_pool_forward)(q[0], co, n, a, b, *norm, *rest, ws, nb))
        made = launches(CONV_FWD), launches(CONV_FWD, DENSE_2X2), launches(SPLITK_REDUCE)
        ok(hip.fitre_hip_profile_enable(0))
        out = [dev.download(p, size) for p, size in zip(q, sizes)]
        for p in ([ws] + q if y is None else [ws] + q[1:]):
            dev.free(p)
        return out, made
    return shape, run


def query(shape, bn):
    return hip.fitre_hip_conv_bn_act_pool_workspace(C.byref(shape), int(bn))


@pytest.mark.parametrize("bn", [True, False])
@pytest.mark.parametrize("n,ci,co", [(128, 64, 64), (131, 68, 70), (256, 512, 64), (128, 512, 512)])
def test_dense_form_runs_in_the_workspace_that_the_query_names(dev, n, ci, co, bn):
    shape, run = layer_passes(dev, n, ci, co, 2, 2, bn)
    _, made = run(True, query(shape, bn))
    assert made == (1, 1, 0)


# cells of one workgroup and of several segments, partials of less than a page, and layers whose partials are most of the room
ROOM = [(32, 256, 64, 4, 4), (21, 128, 64, 2, 2), (52, 64, 96, 14, 12), (1, 64, 8, 4, 4), (2, 128, 8, 2, 2)]


@pytest.mark.parametrize("bn", [True, False])
@pytest.mark.parametrize("geom", ROOM)
def test_split_convolution_in_the_workspace_that_the_query_names(dev, geom, bn):
    """No reduction launch with that size, and with less the ranges (and the bits) of fitre_hip_conv_forward in the same room."""
    shape, run = layer_passes(dev, *geom, bn)
    whole, sums = query(shape, bn), hip.fitre_hip_batch_norm_workspace(geom[2], geom[0] * geom[3] * geom[4]) if bn else 0
    conv = hip.fitre_hip_conv_forward_workspace(C.byref(shape))
    for nb in sorted({whole, max(conv, sums), max(whole - 256, sums), max(whole // 2, sums), max(sums, 16)}, reverse=True):
        got, made = run(True, nb)
        want, apart = run(False, nb)
        if nb == whole:
            assert apart == (1, 0, 1) and made == (1, 0, 0)
        for g, w in zip(got, want):
            np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("bn", [True, False])
@pytest.mark.parametrize("ranges,dense", [(11, 1), (10, 1), (6, 1), (5, 0), (0, 0)])
def test_dense_form_in_the_buffer_of_a_longer_batch(dev, ranges, dense, bn):
    """192 images, whose plan has eleven ranges: those that a smaller workspace holds, and nine taps below half of them.  Equal to
    the whole plan's result up to the order of its sums: 4 * 512 terms of size one over their root, 2^-24 a step, twice."""
    n, c = 192, 512
    shape, run = layer_passes(dev, n, c, c, 2, 2, bn)
    sums = hip.fitre_hip_batch_norm_workspace(c, 4 * n) if bn else 0
    nb = 64 * c * c + 16 * c * n * ranges + (sums + 255 & ~255)
    want, made = run(True, query(shape, bn))
    assert made == (1, 1, 0)
    got, made = run(True, nb)
    assert made[:2] == (1, dense)
    bound = 2 * (4 * c + 16) * 2.0 ** -24 * max(1.0, np.abs(want[0]).max())
    assert np.abs(got[0] - want[0]).max() <= bound
    if dense:  # the pass behind it reads the partials of the ranges that there are
        again, _ = run(False, nb, y=dev.upload(got[0]))
        for g, w in zip(got, again):
            np.testing.assert_array_equal(g, w)


# images, cin, cout, A, B: few channels (no partials at all), a split product, maps that are no whole 16-byte groups
TO_FC = [(5, 3, 6, 8, 8), (32, 256, 64, 4, 4), (3, 64, 40, 7, 7), (4, 8, 64, 8, 8)]


@pytest.mark.parametrize("kind", [MAX_POOL, NO_POOL])
@pytest.mark.parametrize("bn", [True, False])
@pytest.mark.parametrize("geom", TO_FC)
def test_permuted_output_in_the_workspace_that_the_query_names(dev, geom, bn, kind):
    n, ci, co, a, b = geom
    shape, run = layer_passes(dev, *geom, bn)
    pa, pb = (a, b) if kind == NO_POOL else ((a // 2, b // 2) if a % 2 == 0 else ((a - 3) // 2 + 1, (b - 3) // 2 + 1))
    nb = hip.fitre_hip_conv_bn_act_pool_fc_workspace(C.byref(shape), int(bn), pa, pb)
    got, _ = run(True, nb, kind, to_fc=1)
    want, _ = run(False, nb, kind, to_fc=1)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("geom", TO_FC)
def test_room_for_the_permutation_is_asked_for_where_it_is_used_and_before_anything_is_written(dev, geom):
    n, ci, co, a, b = geom
    _, run = layer_passes(dev, *geom, False)
    need = 4 * co * n * a * b
    with pytest.raises(AssertionError, match="workspace"):
        run(True, need - 4, NO_POOL, to_fc=1, y=(y := dev.upload(np.full(co * n * a * b, 7.0, np.float32))))
    np.testing.assert_array_equal(dev.download(y, co * n * a * b), 7.0)
    run(True, need, NO_POOL, to_fc=1)
    if a % 2 == 0:  # 2 x 2 pools are permuted on the way and need no room
        want, _ = run(True, need, MAX_POOL, to_fc=1)
        got, _ = run(True, 0, MAX_POOL, to_fc=1)
        if geom != (32, 256, 64, 4, 4):  # (a product that is cut where it has room)
            for g, w in zip(got, want):
                np.testing.assert_array_equal(g, w)


# small maps, of which a workgroup stages up to 64 at once, the last one with a remainder; long windows at few and at many images
@pytest.mark.parametrize("n,ci,co,a,b,k,pad,thin", [
    (4, 16, 16, 14, 14, 5, 0, 0), (64, 16, 6, 14, 14, 5, 0, 0), (256, 16, 16, 14, 14, 5, 0, 1), (16, 6, 16, 14, 14, 5, 0, 1),
    (1, 3, 6, 32, 32, 5, 0, 1), (64, 3, 5, 5, 5, 5, 0, 0),
    (64, 1, 4, 7, 7, 5, 0, 1), (257, 6, 16, 7, 7, 5, 0, 1), (33, 12, 9, 6, 7, 3, 1, 1), (1000, 1, 3, 4, 4, 3, 0, 1)])
def test_few_channels_take_the_shorter_of_two_chains(dev, n, ci, co, a, b, k, pad, thin):
    """Which kernel ran (the vector one has no tile, and from nine channels on it is the matrix form), and its result."""
    from fitre_amd.structs import fitre_conv_shape
    rng = np.random.default_rng(n + ci + co)
    x = rng.standard_normal((ci, n, a, b)).astype(np.float32)
    w = (rng.standard_normal((co, ci, k, k)) / np.sqrt(ci * k * k)).astype(np.float32)
    oa, ob = a + 2 * pad - k + 1, b + 2 * pad - k + 1
    shape = fitre_conv_shape(n, ci, co, a, b, oa, ob, k, 1, pad)
    count, nb = co * n * oa * ob, hip.fitre_hip_conv_forward_workspace(C.byref(shape))
    y, ws = dev.upload(np.full(count + 4, 7.0, np.float32)), dev.alloc(nb)
    ok(hip.fitre_hip_profile_enable(1))
    ok(hip.fitre_hip_conv_forward(C.byref(shape), dev.upload(x.reshape(-1)), dev.upload(w.reshape(-1)), None, y, ws, nb))
    assert launches(CONV_FWD, 0 if co < 9 else THIN_MATRIX) == thin and launches(CONV_FWD) == 1
    ok(hip.fitre_hip_profile_enable(0))
    got = dev.download(y, count + 4)
    np.testing.assert_array_equal(got[-4:], 7.0)
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double().transpose(0, 1), torch.from_numpy(w).double(), padding=pad).transpose(0, 1).numpy()
    # a float32 sum of ci * k * k terms of size one over their root, 2^-24 a step
    assert np.abs(got[:-4] - want.reshape(-1)).max() <= (ci * k * k + 16) * 2.0 ** -24 * max(1.0, np.abs(want).max())


# the split products of SPLIT (all but the one of 147 cells a channel), and channels of two and three segments
@pytest.mark.parametrize("train", [1, 0])
@pytest.mark.parametrize("bn", [True, False])
@pytest.mark.parametrize("geom", [g for g in SPLIT if g[0] * g[3] * g[4] % 4 == 0] + [(300, 64, 32, 4, 4), (40, 128, 96, 16, 16)])
def test_no_reduction_launch_where_the_pass_behind_sums(dev, geom, bn, train):
    """The product is cut, its partials are summed by the pass behind it, and the bits are those of the separate launches."""
    shape, run = layer_passes(dev, *geom, bn)
    nb = query(shape, bn)
    got, made = run(True, nb, train=train)
    want, apart = run(False, nb, train=train)
    assert made == (1, 0, 0) and apart == (1, 0, 1)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


# samples, cin, cout: one range whose only partial is handed on (64-deep slices, two segments of a channel), several ranges and
# segments, ragged channels
DENSE = [(1400, 64, 512), (1100, 256, 96), (131, 68, 70)]


@pytest.mark.parametrize("bn,train", [(True, 1), (True, 0), (False, 1)])
@pytest.mark.parametrize("kind,to_fc", [(MAX_POOL, 0), (MAX_POOL, 1), (NO_POOL, 1)])
@pytest.mark.parametrize("n,ci,co", DENSE)
def test_passes_behind_the_dense_form(dev, n, ci, co, kind, to_fc, bn, train):
    """Bit for bit what fitre_hip_bn_act_pool_forward(_fc) makes of the convolution that was written."""
    shape, run = layer_passes(dev, n, ci, co, 2, 2, bn)
    nb = hip.fitre_hip_conv_bn_act_pool_fc_workspace(C.byref(shape), int(bn), 2, 2)
    got, made = run(True, nb, kind, to_fc, train)
    assert made == (1, 1, 0)
    want, _ = run(False, nb, kind, to_fc, train, y=dev.upload(got[0]))
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("n,ci,co", DENSE)
def test_dense_form_against_float64(dev, n, ci, co):
    rng = np.random.default_rng(n + ci + co)
    x, w = rng.standard_normal((ci, n, 2, 2)).astype(np.float32), (rng.standard_normal((co, ci, 3, 3)) / np.sqrt(4 * ci)).astype(np.float32)
    from fitre_amd.structs import fitre_conv_shape
    shape = fitre_conv_shape(n, ci, co, 2, 2, 2, 2, 3, 1, 1)
    nb, count = query(shape, False), 4 * co * n
    y, act = dev.alloc(4 * count), dev.alloc(4 * count)
    ok(hip.fitre_hip_conv_bn_act_pool_forward(C.byref(shape), dev.upload(x.reshape(-1)), dev.upload(w.reshape(-1)), None, y, *[None] * 5, 0.0, 0.0, 0,
                                              CNN_ACT_NONE, act, NO_POOL, 2, 2, 0, 2, 2, None, 0, dev.alloc(nb), nb))
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double().transpose(0, 1), torch.from_numpy(w).double(), padding=1).transpose(0, 1).numpy()
    # a float32 sum of 4 * ci terms of size one over their root, 2^-24 a step
    assert np.abs(dev.download(y, count) - want.reshape(-1)).max() <= (4 * ci + 16) * 2.0 ** -24 * max(1.0, np.abs(want).max())


# geometry of THIN, and the channels that a wave of the vector kernel takes: two with an odd number of them, four, in both windows
VARIANTS = [((210, 2, 5, 36, 36, 5, 0), 2), ((210, 2, 7, 34, 34, 3, 0), 2), ((1024, 1, 8, 36, 36, 5, 0), 4), ((1024, 1, 8, 34, 34, 3, 0), 4),
            ((1025, 1, 8, 34, 33, 3, 0), 4)]


@pytest.mark.parametrize("kind,to_fc", [(MAX_POOL, 1), (NO_POOL, 0)])
@pytest.mark.parametrize("geom,channels", VARIANTS)
def test_channel_groups_of_the_vector_kernel(dev, geom, channels, kind, to_fc):
    n, ci, co, a, b, k, pad = geom
    oa, ob = a + 2 * pad - k + 1, b + 2 * pad - k + 1
    waves = n * -(-(-(-oa // 2) * -(-ob // 4)) // 64) * co  # of one channel each: one image a workgroup here
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert channels == (1 if waves <= 8 * cus else (4 if waves >= 64 * cus and co % 4 == 0 else 2))
    ok(hip.fitre_hip_profile_enable(1))
    test_thin_convolution_with_activation_and_pool(dev, geom, kind, to_fc, CNN_ACT_SWISH)
    assert launches(CONV_FWD, 0) == 2 and launches(CONV_FWD) == 2  # with and without a bias
    ok(hip.fitre_hip_profile_enable(0))


# nine and sixteen channels, bands of an image and several images a workgroup, both windows
@pytest.mark.parametrize("kind,to_fc", [(MAX_POOL, 1), (NO_POOL, 0)])
@pytest.mark.parametrize("geom", [(512, 1, 16, 36, 36, 5, 0), (512, 1, 16, 34, 34, 3, 0), (4, 3, 9, 28, 20, 5, 2), (1025, 12, 9, 6, 8, 3, 1), (2100, 6, 16, 14, 14, 5, 0)])
def test_matrix_form_of_nine_to_sixteen_channels(dev, geom, kind, to_fc):
    ok(hip.fitre_hip_profile_enable(1))
    test_thin_convolution_with_activation_and_pool(dev, geom, kind, to_fc, CNN_ACT_SWISH)
    assert launches(CONV_FWD, THIN_MATRIX) == 2 and launches(CONV_FWD) == 2  # with and without a bias
    ok(hip.fitre_hip_profile_enable(0))


def test_few_channels_on_unaligned_tensors_need_no_workspace(dev):
    """Where the tile engine would be the shorter way, but its activation, pool and permutation three launches and a workspace."""
    from helpers import at
    from fitre_amd.structs import fitre_conv_shape
    n, c, a, oa = 4, 16, 14, 10
    rng = np.random.default_rng(1)
    x, w = rng.standard_normal((c, n, a, a)).astype(np.float32), (rng.standard_normal((c, c, 5, 5)) / 20).astype(np.float32)
    shape, count, pooled = fitre_conv_shape(n, c, c, a, a, oa, oa, 5, 1, 0), c * n * oa * oa, c * n * 25
    y, act, pool = (dev.zeros(size + 4) for size in (count, count, pooled))
    ok(hip.fitre_hip_conv_bn_act_pool_forward(C.byref(shape), dev.upload(x.reshape(-1)), dev.upload(w.reshape(-1)), None, at(y, 1), *[None] * 5, 0.0,
                                              0.0, 0, CNN_ACT_RELU, at(act, 1), MAX_POOL, 2, 2, 0, 5, 5, at(pool, 1), 1, None, 0))
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double().transpose(0, 1), torch.from_numpy(w).double()).transpose(0, 1).numpy()
    got = dev.download(y, count, offset=1).reshape(c, n, oa, oa)
    assert np.abs(got - want).max() <= (25 * c + 16) * 2.0 ** -24 * max(1.0, np.abs(want).max())
    got = np.maximum(got, 0)
    np.testing.assert_array_equal(dev.download(act, count, offset=1).reshape(got.shape), got)
    top = got.reshape(c, n, 5, 2, 5, 2).max((3, 5))  # [C][N][a][b] -> [N][C][b][a]
    np.testing.assert_array_equal(dev.download(pool, pooled, offset=1).reshape(n, c, 5, 5), top.transpose(1, 0, 3, 2))


def test_few_channels_without_room_for_the_engines_ranges(dev):
    """The kernel of few channels, whose time needs no workspace, where the tile engine would have to run uncut."""
    from fitre_amd.structs import fitre_conv_shape
    shape = fitre_conv_shape(8, 16, 16, 14, 14, 10, 10, 5, 1, 0)
    nb = hip.fitre_hip_conv_forward_workspace(C.byref(shape))
    x, w, y, ws = dev.zeros(16 * 8 * 196), dev.zeros(16 * 400), dev.zeros(16 * 800), dev.alloc(nb)
    for room, thin in ((nb, 0), (nb // 4, 1), (0, 1)):
        ok(hip.fitre_hip_profile_enable(1))
        ok(hip.fitre_hip_conv_forward(C.byref(shape), x, w, None, y, ws if room else None, room))
        assert launches(CONV_FWD, THIN_MATRIX) == thin and launches(CONV_FWD) == 1
        ok(hip.fitre_hip_profile_enable(0))
