"""The fused steps of the forward pass (include/fitre_hip.h) against float64 numpy on the same float32 operands."""
import numpy as np
import pytest

from fitre_amd import lib as L
from fitre_amd.structs import (ACT_LINEAR, ACT_LOGISTIC, ACT_TANH, CNN_ACT_ELU, CNN_ACT_NONE, CNN_ACT_RELU, CNN_ACT_SOFTPLUS,
                               CNN_ACT_SWISH)

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
