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
# remainder of them, the channel groups of one, two and four), odd rows and columns, one channel, sixteen of each, 3 x 3
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


# samples, cin, cout, A, B: one workgroup per channel (4 x 4 and 2 x 2 maps, the cell kernel and the nine-tap one), several
# segments of a channel, a channel of a multiple of four cells that is no whole number of segments, one that is none
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


# samples, cin, cout on 2 x 2 maps: the smallest batch of the dense form, ragged samples and channels, an uncut reduction
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
            np.testing.assert_allclose(a, b, rtol=1e-5, atol=1e-6)  # more than one segment of a channel from 1025 images on
        else:
            np.testing.assert_array_equal(a, b)
