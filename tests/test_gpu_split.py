"""fp32 products on the bf16 matrix pipes (fitre_amd/csrc/hip/split_bf16.h): convolutions large enough to take them, against
float64.  A sum of K normal terms in fp32 multiply-adds is off by a random walk of K roundings, measured at 0.3 sqrt(K) 2^-24 of
its norm; these kernels round less often (0.1), and a product that drops one of its six parts is off by 2^-17 or more."""
import ctypes as C

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from fitre_amd import lib as L
from helpers import conv_shape

pytestmark = pytest.mark.gpu
hip = L.hip


def limit(terms, factor=0.3):
    return factor * np.sqrt(terms) * 2.0**-24


def far(got, want):
    return np.linalg.norm(got - want) / np.linalg.norm(want)


def tensors(case, seed=0):
    n, ci, co, a, b, k = case
    g = torch.Generator().manual_seed(seed + sum(case))
    x = torch.randn(n, ci, a, b, generator=g)
    w = torch.randn(co, ci, k, k, generator=g) / (ci * k * k) ** 0.5
    d = torch.randn(n, co, a, b, generator=g)
    return x, w, d


def flat(t):  # the library's order of a tensor [N][C][A][B]
    return t.transpose(0, 1).contiguous().numpy().ravel()


def conv(dev, case, which, source, w, second=None, bias=None, ws_bytes=None):
    n, ci, co, a, b, k = case
    shape = conv_shape(n, ci, co, a, b, k, 1, k // 2)
    out_channels = co if which == "fwd" else ci
    if second:
        nb = hip.fitre_hip_conv_pair_workspace(C.byref(shape), 0 if which == "fwd" else 1)
    else:
        nb = (hip.fitre_hip_conv_forward_workspace if which == "fwd" else hip.fitre_hip_conv_input_grad_workspace)(C.byref(shape))
    nb = nb if ws_bytes is None else ws_bytes(nb)
    ps, pw, ws, out = dev.upload(flat(source)), dev.upload(w.numpy().ravel()), dev.alloc(nb), dev.zeros(out_channels * n * a * b)
    bufs = [ps, pw, ws, out]
    if second:
        p2, w2 = dev.upload(flat(second[0])), dev.upload(second[1].numpy().ravel())
        bufs += [p2, w2]
    if which == "fwd":
        pb = dev.upload(bias.numpy()) if bias is not None else None
        if pb:
            bufs.append(pb)
        L.check(hip.fitre_hip_conv_forward_pair(C.byref(shape), ps, pw, p2, w2, pb, out, ws, nb) if second else
                hip.fitre_hip_conv_forward(C.byref(shape), ps, pw, pb, out, ws, nb))
    else:
        L.check(hip.fitre_hip_conv_input_grad_pair(C.byref(shape), ps, pw, p2, w2, out, ws, nb) if second else
                hip.fitre_hip_conv_input_grad(C.byref(shape), ps, pw, out, ws, nb))
    got = dev.download(out, out_channels * n * a * b).reshape(out_channels, n, a, b)
    for q in bufs:
        dev.free(q)
    return got


def reference(case, which, source, w):
    k = case[5]
    f = F.conv2d if which == "fwd" else F.conv_transpose2d
    return f(source.double(), w.double(), padding=k // 2).transpose(0, 1).numpy()


# N, Cin, Cout, A, B, window: every kernel of kConvSplitVariants, ragged tiles of positions and channels, split reductions
CASES = [
    (77, 128, 160, 8, 8, 3),   # 160 channels: a partial channel tile; 4928 positions: a partial position tile
    (77, 160, 128, 8, 8, 3),
    (96, 512, 512, 4, 4, 3),   # many images in a window, split reduction
    (45, 512, 512, 4, 2, 3),   # rectangular
    (40, 64, 192, 16, 16, 3),  # the input gradient has 64 channels: 256-position tiles
    (21, 64, 128, 32, 32, 3),  # rows of 32
    (7, 128, 144, 27, 64, 3),  # the widest row
    (150, 48, 272, 13, 5, 3),  # odd extents
    (40, 32, 48, 40, 24, 3),   # at most 64 channels each way
    (40, 64, 192, 13, 13, 5),  # 5 x 5 windows
    (11, 64, 192, 27, 27, 5),
    (30, 96, 80, 9, 14, 5),
]


@pytest.mark.parametrize("which", ["fwd", "dx"])
@pytest.mark.parametrize("case", CASES)
def test_convolution(dev, case, which):
    x, w, d = tensors(case)
    source = x if which == "fwd" else d
    bias = torch.linspace(-1, 1, case[2]) if which == "fwd" else None
    want = reference(case, which, source, w)
    if bias is not None:
        want = want + bias.double().numpy()[:, None, None, None]
    terms = source.shape[1] * case[5] ** 2
    assert far(conv(dev, case, which, source, w, bias=bias), want) < limit(terms)


@pytest.mark.parametrize("which", ["fwd", "dx"])
def test_a_pair_of_products(dev, which):
    case = (40, 128, 128, 8, 8, 3)
    (x, w, d), (x2, w2, d2) = tensors(case), tensors(case, 1)
    s, s2 = (x, x2) if which == "fwd" else (d, d2)
    got = conv(dev, case, which, s, w, second=(s2, w2))
    assert far(got, reference(case, which, s, w) + reference(case, which, s2, w2)) < limit(2 * 128 * 9)


def test_smaller_workspaces(dev):
    """Fewer reduction ranges, none, and (no room for the split weights) the fp32 kernel."""
    case = (40, 256, 256, 8, 8, 3)
    x, w, _ = tensors(case)
    want = reference(case, "fwd", x, w)
    weights = 6 * 9 * 256 * 256
    for ws_bytes in (lambda nb: nb, lambda nb: weights + 2 * 4 * 256 * 40 * 64 + 600, lambda nb: weights + 256, lambda nb: weights):
        assert far(conv(dev, case, "fwd", x, w, ws_bytes=ws_bytes), want) < limit(256 * 9)


def test_prepared_weights_give_the_same_bits(dev):
    from fitre_amd.structs import fitre_split_view
    case = (256, 128, 128, 8, 8, 3)
    n, ci, co, a, b, _ = case
    shape = conv_shape(n, ci, co, a, b, 3, 1, 1)
    _, w, d = tensors(case)
    prepared_bytes = hip.fitre_hip_conv_input_grad_prepared_bytes(C.byref(shape))
    assert prepared_bytes > 0
    nb = prepared_bytes + 256  # no room for partial results: one range
    pd, pw, ws, out, prepared = dev.upload(flat(d)), dev.upload(w.numpy().ravel()), dev.alloc(nb), dev.zeros(ci * n * a * b), dev.alloc(prepared_bytes)
    view = fitre_split_view()
    L.check(hip.fitre_hip_conv_input_grad_split(C.byref(shape), pd, pw, out, ws, nb, C.byref(view)))
    assert view.splits == 1
    first = dev.download(out, ci * n * a * b)
    L.check(hip.fitre_hip_conv_input_grad_prepare(C.byref(shape), pw, prepared, prepared_bytes))
    L.check(hip.fitre_hip_conv_input_grad_split_prepared(C.byref(shape), pd, pw, prepared, out, ws, nb, C.byref(view)))
    np.testing.assert_array_equal(dev.download(out, ci * n * a * b), first)
    for q in (pd, pw, ws, out, prepared):
        dev.free(q)


@pytest.mark.parametrize("which", ["fwd", "dx"])
def test_numbers_the_split_does_not_carry(dev, which):
    """Infinities, NaN, the largest floats (which round up to infinity in bf16) and tensors so small that the lower parts of
    their numbers are below the smallest bf16 number: what an fp32 chain gives."""
    case = (80, 128, 128, 8, 8, 3)
    x, w, d = tensors(case)
    source = x if which == "fwd" else d
    terms = 128 * 9
    plain = conv(dev, case, which, source, w)
    odd = source.clone()
    odd[3, 5, 0, 7], odd[40, 100, 4, 4], odd[79, 127, 7, 7] = float("inf"), float("nan"), float(np.finfo(np.float32).max)
    got, want = conv(dev, case, which, odd, w), reference(case, which, odd, w)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    huge = np.isfinite(want) & (np.abs(want) > 1e30)
    assert huge.any() and far(got[huge], want[huge]) < limit(terms)
    rest = np.isfinite(want) & ~huge
    assert far(got[rest], want[rest]) < limit(terms, 0.6)
    # tiles without such a number keep their bits
    far_off = slice(8, 30)  # images of tiles of their own (two images a tile)
    np.testing.assert_array_equal(got[:, far_off], plain[:, far_off])
    small = source * 2.0**-108
    assert far(conv(dev, case, which, small, w) * 2.0**108, reference(case, which, source, w)) < limit(terms, 0.6)
