"""fp32 products on the bf16 matrix pipes (fitre_amd/csrc/hip/split_bf16.h): convolutions large enough to take them, against
float64.  A sum of K normal terms in fp32 multiply-adds is off by a random walk of K roundings, measured at 0.3 sqrt(K) 2^-24 of
its norm; these kernels round less often (0.1), and a product that drops one of its six parts is off by 2^-17 or more.

Every call is made under the launch accounting, which says whether the kernel that the case is written for was the one that ran."""
import ctypes as C
from contextlib import contextmanager

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


CONV_DW, CONV_DX, CONV_FWD, FC_GEMM = 0, 1, 2, 3  # kernel classes and tile variants of include/fitre_hip.h
FP32, SPLIT, CELL = "fp32", 10, 11


@contextmanager
def taken(kernel_class, tile, launches=1):
    """The launches of a class made inside are of this variant (FP32: none of either split one)."""
    count, ms, work = C.c_long(), C.c_double(), C.c_double()
    L.check(hip.fitre_hip_profile_enable(1))
    try:
        yield
        made = {}
        for t in (SPLIT, CELL):
            L.check(hip.fitre_hip_profile_read_tile(kernel_class, t, C.byref(count), C.byref(ms), C.byref(work)))
            made[t] = count.value
    finally:
        L.check(hip.fitre_hip_profile_enable(0))
    assert made == {t: launches * (t == tile) for t in (SPLIT, CELL)}


def form(case, which, second=None):
    """The window form, or the cell form on 4 x 4 maps that fill its tiles of 32 images (no input gradient on its own)."""
    n, cell = case[0], case[3:] == (4, 4, 3) and (which == "fwd" or second)
    return CELL if cell and 100 * (-(-n // 32) * 32) < 137 * n else SPLIT


def flat(t):  # the library's order of a tensor [N][C][A][B]
    return t.transpose(0, 1).contiguous().numpy().ravel()


def conv(dev, case, which, source, w, second=None, bias=None, ws_bytes=None, tile=None):
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
    pb = dev.upload(bias.numpy()) if bias is not None else None
    if pb:
        bufs.append(pb)
    with taken(CONV_FWD if which == "fwd" else CONV_DX, tile or form(case, which, second)):
        if which == "fwd":
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
    (130, 256, 256, 4, 4, 3),  # many images in a window, split reduction; forward in the cell form, two images in the last tile
    (224, 256, 272, 4, 4, 3),  # whole tiles of images, a partial tile of channels
    (132, 512, 256, 4, 4, 3),
    (260, 256, 256, 4, 2, 3),  # rectangular
    (56, 64, 192, 16, 16, 3),  # the input gradient has 64 channels: 256-position tiles
    (21, 64, 128, 32, 32, 3),  # rows of 32
    (7, 128, 144, 27, 64, 3),  # the widest row
    (200, 48, 272, 13, 5, 3),  # odd extents
    (115, 32, 48, 40, 24, 3),  # at most 64 channels each way
    (40, 64, 192, 13, 13, 5),  # 5 x 5 windows
    (11, 64, 192, 27, 27, 5),
    (30, 96, 80, 9, 14, 5),
]


@pytest.mark.parametrize("case,which", [(case, which) for case in CASES for which in ("fwd", "dx")] + [
    ((66, 512, 256, 4, 4, 3), "fwd"),  # too little in the last tile of images for the cell form
])
def test_convolution(dev, case, which):
    x, w, d = tensors(case)
    source = x if which == "fwd" else d
    bias = torch.linspace(-1, 1, case[2]) if which == "fwd" else None
    want = reference(case, which, source, w)
    if bias is not None:
        want = want + bias.double().numpy()[:, None, None, None]
    terms = source.shape[1] * case[5] ** 2
    assert far(conv(dev, case, which, source, w, bias=bias), want) < limit(terms)


@pytest.mark.parametrize("case", [(40, 128, 128, 8, 8, 3), (130, 144, 176, 4, 4, 3)])
@pytest.mark.parametrize("which", ["fwd", "dx"])
def test_a_pair_of_products(dev, case, which):
    (x, w, d), (x2, w2, d2) = tensors(case), tensors(case, 1)
    s, s2 = (x, x2) if which == "fwd" else (d, d2)
    got = conv(dev, case, which, s, w, second=(s2, w2))
    assert far(got, reference(case, which, s, w) + reference(case, which, s2, w2)) < limit(2 * s.shape[1] * 9)


def test_smaller_workspaces(dev):
    """Fewer reduction ranges, none, and (no room for the split weights) the fp32 kernel."""
    case = (40, 256, 256, 8, 8, 3)
    x, w, _ = tensors(case)
    want = reference(case, "fwd", x, w)
    weights = 6 * 9 * 256 * 256
    for ws_bytes, tile in ((lambda nb: nb, SPLIT), (lambda nb: weights + 2 * 4 * 256 * 40 * 64 + 600, SPLIT), (lambda nb: weights + 256, SPLIT),
                           (lambda nb: weights, FP32)):
        assert far(conv(dev, case, "fwd", x, w, ws_bytes=ws_bytes, tile=tile), want) < limit(256 * 9)


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
    with taken(CONV_DX, SPLIT):
        L.check(hip.fitre_hip_conv_input_grad_split(C.byref(shape), pd, pw, out, ws, nb, C.byref(view)))
    assert view.splits == 1
    first = dev.download(out, ci * n * a * b)
    L.check(hip.fitre_hip_conv_input_grad_prepare(C.byref(shape), pw, prepared, prepared_bytes))
    with taken(CONV_DX, SPLIT):
        L.check(hip.fitre_hip_conv_input_grad_split_prepared(C.byref(shape), pd, pw, prepared, out, ws, nb, C.byref(view)))
    np.testing.assert_array_equal(dev.download(out, ci * n * a * b), first)
    for q in (pd, pw, ws, out, prepared):
        dev.free(q)


@pytest.mark.parametrize("case,copied", [((256, 128, 128, 8, 8, 3), True), ((8, 256, 512, 8, 8, 3), False), ((127, 512, 512, 4, 4, 3), False)])
def test_copies_are_asked_for_only_where_the_input_gradient_reads_them(dev, case, copied):
    """Below 2048 positions the fp32 kernels run: no copy, and none is made."""
    n, ci, co, a, b, _ = case
    shape = conv_shape(n, ci, co, a, b, 3, 1, 1)
    assert (hip.fitre_hip_conv_input_grad_prepared_bytes(C.byref(shape)) > 0) == copied
    w = dev.upload(np.zeros(ci * co * 9, np.float32))
    room = dev.alloc(6 * ci * 9 * co)
    assert (hip.fitre_hip_conv_input_grad_prepare(C.byref(shape), w, room, 6 * ci * 9 * co) == 0) == copied
    dev.free(w)
    dev.free(room)


@pytest.mark.parametrize("case,which", [((80, 128, 128, 8, 8, 3), "fwd"), ((80, 128, 128, 8, 8, 3), "dx"), ((159, 192, 208, 4, 4, 3), "fwd")])
def test_numbers_the_split_does_not_carry(dev, case, which):
    """Infinities, NaN, the largest floats (which round up to infinity in bf16) and tensors so small that the lower parts of
    their numbers are below the smallest bf16 number: what an fp32 chain gives."""
    x, w, d = tensors(case)
    source = x if which == "fwd" else d
    terms = source.shape[1] * 9
    plain = conv(dev, case, which, source, w)
    odd = source.clone()
    odd[3, 5, 0, 3], odd[40, 100, 2, 2], odd[-1, -1, -1, -1] = float("inf"), float("nan"), float(np.finfo(np.float32).max)
    got, want = conv(dev, case, which, odd, w), reference(case, which, odd, w)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    huge = np.isfinite(want) & (np.abs(want) > 1e30)
    assert huge.any() and far(got[huge], want[huge]) < limit(terms)
    rest = np.isfinite(want) & ~huge
    assert far(got[rest], want[rest]) < limit(terms, 0.6)
    # tiles without such a number keep their bits
    far_off = slice(8, 30) if case[3] == 8 else slice(64, 128)  # images of other tiles (two of 8 x 8, 32 of 4 x 4 a tile)
    np.testing.assert_array_equal(got[:, far_off], plain[:, far_off])
    small = source * 2.0**-108
    assert far(conv(dev, case, which, small, w) * 2.0**108, reference(case, which, source, w)) < limit(terms, 0.6)


def weight_grad(dev, case, x, d, second=None, ws_bytes=None, tile=SPLIT):
    n, ci, co, a, b, k = case
    shape = conv_shape(n, ci, co, a, b, k, 1, k // 2)
    nb = hip.fitre_hip_conv_pair_workspace(C.byref(shape), 2) if second else hip.fitre_hip_conv_weight_grad_workspace(C.byref(shape))
    nb = nb if ws_bytes is None else ws_bytes(nb)
    bufs = [dev.upload(flat(t)) for t in (x, d) + (second or ())] + [dev.alloc(nb), dev.zeros(co * ci * k * k)]
    ws, out = bufs[-2:]
    with taken(CONV_DW, tile):
        if second:
            L.check(hip.fitre_hip_conv_weight_grad_pair(C.byref(shape), *bufs[:4], out, ws, nb))
        else:
            L.check(hip.fitre_hip_conv_weight_grad(C.byref(shape), *bufs[:2], out, ws, nb))
    got = dev.download(out, co * ci * k * k).reshape(co, ci, k, k)
    for q in bufs:
        dev.free(q)
    return got


def weight_reference(case, x, d):
    k = case[5]
    return torch.nn.grad.conv2d_weight(x.double(), (case[2], case[1], k, k), d.double(), padding=k // 2).numpy()


# the three ways a row is cut into groups, one tile of channels and partial ones of either kind with each, and numbers of image rows
# that are no whole groups or stages
WEIGHT_CASES = [
    (130, 256, 272, 4, 4, 3),  # two rows a group
    (151, 200, 264, 5, 3, 3),  # rows of three cells, an odd number of rows
    (256, 64, 64, 4, 4, 3),    # one tile
    (33, 160, 144, 8, 8, 3),   # a row a group
    (130, 72, 130, 7, 6, 3),
    (512, 72, 130, 1, 8, 3),   # one image row: two of three tap rows are outside
    (112, 40, 48, 8, 8, 3),    # part of one tile
    (97, 130, 64, 9, 7, 3),
    (25, 64, 192, 13, 13, 3),  # two groups a row, the second five cells
    (9, 100, 70, 16, 16, 3),
    (10, 96, 64, 16, 16, 3),
    (6, 96, 128, 12, 32, 3),   # four groups a row
    (9, 64, 128, 27, 27, 3),
    (8, 128, 64, 11, 24, 3),   # three of four groups
    (13, 64, 192, 13, 13, 5),  # 5 x 5 windows
    (18, 80, 160, 15, 8, 5),
    (5, 64, 96, 20, 30, 5),
    (5, 64, 192, 27, 27, 5),
    (20, 72, 64, 15, 14, 5),   # at most 64 output channels
    (150, 48, 40, 8, 8, 5),
    (5, 96, 64, 27, 27, 5),
    (140, 64, 64, 2, 16, 5),   # fewer image rows than the window
    (280, 64, 64, 1, 16, 5),
]


@pytest.mark.parametrize("case", WEIGHT_CASES)
def test_weight_gradient(dev, case):
    x, _, d = tensors(case)
    assert far(weight_grad(dev, case, x, d), weight_reference(case, x, d)) < limit(case[0] * case[3] * case[4])


@pytest.mark.parametrize("case", [(256, 64, 128, 16, 16, 3), (256, 256, 256, 8, 8, 3), (256, 512, 256, 4, 4, 3), (64, 64, 64, 27, 27, 5)])
def test_weight_gradient_of_sparse_errors(dev, case):
    """Inputs behind a ReLU and one error in fifty not zero: a sum to which little is added is rounded rarely, by less than the one
    rounding of its result (3.7e-8 to 4.2e-8 of 2^-24 = 6.0e-8; the fp32 pipe has 5.2e-8 to 7.9e-8).  Were the small products of the
    split added to the large ones, every one of them would round the sum: 1.1e-7 to 1.4e-7."""
    x, _, d = tensors(case)
    x, d = x.relu(), d * (torch.rand(d.shape, generator=torch.Generator().manual_seed(1)) < 0.02)
    assert far(weight_grad(dev, case, x, d), weight_reference(case, x, d)) < 2.0**-24


def test_weight_gradient_of_a_pair(dev):
    case = (33, 128, 128, 8, 8, 3)
    (x, _, d), (x2, _, d2) = tensors(case), tensors(case, 1)
    got = weight_grad(dev, case, x, d, second=(x2, d2))
    assert far(got, weight_reference(case, x, d) + weight_reference(case, x2, d2)) < limit(2 * 33 * 64)


def test_weight_gradient_in_smaller_workspaces(dev):
    """Fewer reduction ranges, and (room for less than half of them) the fp32 kernels."""
    case = (64, 128, 128, 8, 8, 3)
    x, _, d = tensors(case)
    want, one = weight_reference(case, x, d), 4 * 128 * 128 * 9
    for ws_bytes, tile in ((lambda nb: nb - one, SPLIT), (lambda nb: nb * 3 // 4, SPLIT), (lambda nb: 3 * one, FP32), (lambda nb: 4, FP32)):
        assert far(weight_grad(dev, case, x, d, ws_bytes=ws_bytes, tile=tile), want) < limit(64 * 64)


@pytest.mark.parametrize("case", [(64, 128, 128, 8, 8, 3), (130, 128, 256, 4, 4, 3), (20, 64, 128, 16, 16, 3), (20, 64, 64, 15, 15, 5)])
def test_numbers_the_split_does_not_carry_in_a_weight_gradient(dev, case):
    x, _, d = tensors(case)
    terms = case[0] * case[3] * case[4]
    odd, odd_d = x.clone(), d.clone()
    odd[1, 5, 2, 2], odd[2, 9, 0, 3], odd_d[3, 7, 2, 1] = float("inf"), float(np.finfo(np.float32).max), float("nan")
    odd_d[2] *= 0.05  # no product with the largest float overflows
    got, want = weight_grad(dev, case, odd, odd_d), weight_reference(case, odd, odd_d)
    # (every tap at these cells is inside the image: what is multiplied with padding is not the question here)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    huge = np.isfinite(want) & (np.abs(want) > 1e30)
    rest = np.isfinite(want) & ~huge
    assert huge.any() and far(got[huge] * 1e-35, want[huge] * 1e-35) < limit(terms)
    assert far(got[rest], want[rest]) < limit(terms, 0.6)
    assert far(weight_grad(dev, case, x, d * 2.0**-108) * 2.0**108, weight_reference(case, x, d)) < limit(terms, 0.6)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(200, 130, 777), (64, 64, 2560), (131, 600, 520)])
def test_product(dev, M, N, K, ta, tb):
    """alpha, beta and a bias, and the numbers the split does not carry: in the middle, in a corner, at a ragged end of the
    reduction, and behind it (where a row of the matrix holds what is not part of the product)."""
    rng = np.random.default_rng(M + 3 * N + 7 * K + ta + 2 * tb)
    lda, ldb, ldc = (K if ta else M) + 5, (N if tb else K) + 3, M + 1
    A = rng.standard_normal((M if ta else K, lda)).astype(np.float32)
    B = rng.standard_normal((K if tb else N, ldb)).astype(np.float32)
    C0, bias = rng.standard_normal((N, ldc)).astype(np.float32), rng.standard_normal(M).astype(np.float32)
    A[:, K if ta else M:] = np.inf
    B[:, N if tb else K:] = np.nan
    nb = hip.fitre_hip_gemm_workspace(M, N, K)
    ws, pbias = dev.alloc(max(nb, 4)), dev.upload(bias)

    def run(a, b):
        pa, pb, pc = dev.upload(a.reshape(-1)), dev.upload(b.reshape(-1)), dev.upload(C0.reshape(-1))
        with taken(FC_GEMM, SPLIT):
            L.check(hip.fitre_hip_gemm(ta, tb, M, N, K, 0.5, pa, lda, pb, ldb, -2.0, pc, ldc, pbias, ws, nb))
        got = dev.download(pc, ldc * N).reshape(N, ldc)
        for q in (pa, pb, pc):
            dev.free(q)
        return got

    def op(a, b):
        return (a[:, :K].T if ta else a[:, :M]).astype(np.float64), (b[:, :N].T if tb else b[:, :K]).astype(np.float64)

    opA, opB = op(A, B)
    rest = bias.astype(np.float64) - 2.0 * C0[:, :M].astype(np.float64)
    got, want = run(A, B), 0.5 * opB @ opA + rest
    assert far(got[:, :M], want) < limit(K, 0.6)
    np.testing.assert_array_equal(got[:, M:], C0[:, M:])
    odd_a, odd_b = A.copy(), B.copy()
    opA, opB = op(odd_a, odd_b)
    views = (odd_a[:, :K].T if ta else odd_a[:, :M]), (odd_b[:, :N].T if tb else odd_b[:, :K])  # [K][M], [N][K] of the copies
    views[1][:, 3] *= 0.05
    views[0][3, 7], views[0][K - 1, M - 1], views[1][N - 1, 0] = np.finfo(np.float32).max, np.inf, np.nan
    with np.errstate(invalid="ignore"):
        opA, opB = op(odd_a, odd_b)
        got, want = run(odd_a, odd_b)[:, :M], 0.5 * np.array([[(opB[n] * opA[:, m]).sum() for m in range(M)] for n in range(N)]) + rest
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    huge = np.isfinite(want) & (np.abs(want) > 1e30)
    fine = np.isfinite(want) & ~huge
    assert far(got[huge] * 1e-35, want[huge] * 1e-35) < limit(K) and far(got[fine], want[fine]) < limit(K, 1.0)
    for q in (ws, pbias):
        dev.free(q)


@pytest.mark.parametrize("ta,tb,M,N,K,tile", [
    (0, 0, 32, 140_001, 64, FP32), (1, 0, 140_001, 32, 64, FP32), (1, 1, 32, 140_001, 64, FP32), (0, 0, 33, 140_001, 64, SPLIT),
    (1, 0, 32, 140_001, 65, SPLIT), (0, 1, 31, 140_001, 256, FP32), (0, 1, 31, 140_001, 257, SPLIT), (0, 1, 3001, 2999, 64, FP32),
    (0, 1, 3001, 2999, 65, SPLIT), (0, 1, 6000, 5001, 192, FP32), (0, 1, 6000, 5001, 193, SPLIT), (0, 0, 6000, 5001, 16, FP32),
    (1, 1, 6000, 5001, 17, SPLIT), (1, 0, 6000, 5001, 16, FP32)])
def test_products_bound_by_what_they_write(dev, ta, tb, M, N, K, tile):
    """Both sides of the lines up to which the fp32 engine has them."""
    rng = np.random.default_rng(M + N + K)
    A, B = rng.standard_normal((M, K) if ta else (K, M)).astype(np.float32), rng.standard_normal((K, N) if tb else (N, K)).astype(np.float32)
    nb = hip.fitre_hip_gemm_workspace(M, N, K)
    pa, pb, pc, ws = dev.upload(A.reshape(-1)), dev.upload(B.reshape(-1)), dev.zeros(M * N), dev.alloc(max(nb, 4))
    with taken(FC_GEMM, tile):
        L.check(hip.fitre_hip_gemm(ta, tb, M, N, K, 1.0, pa, A.shape[1], pb, B.shape[1], 0.0, pc, M, None, ws, nb))
    got = dev.download(pc, M * N).reshape(N, M)
    for q in (pa, pb, pc, ws):
        dev.free(q)
    opA, opB = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    for cols in (slice(0, 100), slice(N - 100, N)):
        assert far(got[cols], opB[cols] @ opA) < limit(K) + 2.0**-24


@pytest.mark.parametrize("tb,K,split", [(0, 17, 2), (1, 2, 1)])
def test_product_of_more_columns_than_a_grid_has(dev, tb, K, split):
    """In two launches; a large result of two terms a sum is one of the fp32 engine's."""
    M, N = 33, 65535 * 64 + 37
    rng = np.random.default_rng(tb)
    A, B = rng.standard_normal((K, M)).astype(np.float32), rng.standard_normal((K, N) if tb else (N, K)).astype(np.float32)
    nb = hip.fitre_hip_gemm_workspace(M, N, K)
    pa, pb, pc, ws = dev.upload(A.reshape(-1)), dev.upload(B.reshape(-1)), dev.zeros(M * N), dev.alloc(max(nb, 4))
    with taken(FC_GEMM, SPLIT, launches=split):
        L.check(hip.fitre_hip_gemm(0, tb, M, N, K, 1.0, pa, M, pb, N if tb else K, 0.0, pc, M, None, ws, nb))
    got = dev.download(pc, M * N).reshape(N, M)
    for q in (pa, pb, pc, ws):
        dev.free(q)
    edge = 65535 * 64
    for cols in (slice(0, 200), slice(edge - 130, N)):
        assert far(got[cols], (B[:, cols].T if tb else B[cols]).astype(np.float64) @ A.astype(np.float64)) < 3 * 2.0**-24  # few roundings


@pytest.mark.parametrize("ta,tb,M,N", [(0, 0, 2000, 4000), (1, 1, 4000, 2000)])
def test_product_of_a_short_reduction_with_a_large_leading_dimension(dev, ta, tb, M, N):
    """Seventeen reduction indices 35 million apart: the other fifteen of a slice lie past 2^32 bytes, where 32-bit offsets would come
    back into the first row; the other operand's rows are followed by numbers that are not part of the product."""
    K, far_apart, padded = 17, 35_000_000, 40
    rng = np.random.default_rng(M)
    near = rng.standard_normal((M if ta else N, padded)).astype(np.float32)
    rows = rng.standard_normal((K, N if tb else M)).astype(np.float32)
    first = np.ones(far_apart, np.float32)  # (and what follows the first row's numbers)
    first[:rows.shape[1]] = rows[0]
    apart = dev.zeros(K * far_apart)
    for k in range(K):
        row = first if k == 0 else rows[k]
        L.check(hip.fitre_hip_copy_h2d(C.c_void_p(apart.value + 4 * k * far_apart), row.ctypes.data_as(C.c_void_p), row.nbytes))
    nb = hip.fitre_hip_gemm_workspace(M, N, K)
    other, pc, ws = dev.upload(near.reshape(-1)), dev.zeros(M * N), dev.alloc(max(nb, 4))
    pa, lda, pb, ldb = (other, padded, apart, far_apart) if ta else (apart, far_apart, other, padded)
    with taken(FC_GEMM, SPLIT):
        L.check(hip.fitre_hip_gemm(ta, tb, M, N, K, 1.0, pa, lda, pb, ldb, 0.0, pc, M, None, ws, nb))
    got = dev.download(pc, M * N).reshape(N, M)
    for q in (apart, other, pc, ws):
        dev.free(q)
    a, b = (near[:, :K].T, rows.T) if ta else (rows, near[:, :K])
    assert far(got, b.astype(np.float64) @ a.astype(np.float64)) < 3 * 2.0**-24  # each accumulator and their sum are rounded a few times


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (1, 1)])
def test_product_of_padded_matrices(dev, ta, tb):
    """What lies between the rows of a matrix has no part in a sum, nor in how it is computed: the same bits whatever it is."""
    M, N, K = 200, 130, 777
    rng = np.random.default_rng(ta + 2 * tb)
    A = rng.standard_normal((M, K + 7) if ta else (K, M + 7)).astype(np.float32)
    B = rng.standard_normal((K, N + 7) if tb else (N, K + 7)).astype(np.float32)
    nb = hip.fitre_hip_gemm_workspace(M, N, K)
    got = []
    for between in (0.0, np.nan, np.inf):
        A[:, -7:] = B[:, -7:] = between
        pa, pb, pc, ws = dev.upload(A.reshape(-1)), dev.upload(B.reshape(-1)), dev.zeros(M * N), dev.alloc(max(nb, 4))
        with taken(FC_GEMM, SPLIT):
            L.check(hip.fitre_hip_gemm(ta, tb, M, N, K, 1.0, pa, A.shape[1], pb, B.shape[1], 0.0, pc, M, None, ws, nb))
        got.append(dev.download(pc, M * N))
        for q in (pa, pb, pc, ws):
            dev.free(q)
    np.testing.assert_array_equal(got[0], got[1])
    np.testing.assert_array_equal(got[0], got[2])


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("K", [777, 640])
def test_product_of_parts_of_larger_matrices(dev, ta, tb, K):
    """Columns cut out of larger matrices: the last one ends with its last number, at the end of the memory there is."""
    M, N, room = 330, 270, 1 << 20
    rng = np.random.default_rng(K + ta + 2 * tb)
    ends, views = [], []
    for rows, cols in ((M, K) if ta else (K, M)), ((K, N) if tb else (N, K)):
        ld = cols + 150
        whole = np.full(room, np.nan, np.float32)
        first = room - ((rows - 1) * ld + cols)
        part = np.lib.stride_tricks.as_strided(whole[first:], (rows, cols), (4 * ld, 4))
        part[:] = rng.standard_normal((rows, cols))
        ends.append((dev.upload(whole), first, ld))
        views.append(part.astype(np.float64))
    (pa, fa, lda), (pb, fb, ldb) = ends
    nb = hip.fitre_hip_gemm_workspace(M, N, K)
    pc, ws = dev.zeros(M * N), dev.alloc(max(nb, 4))
    with taken(FC_GEMM, SPLIT):
        L.check(hip.fitre_hip_gemm(ta, tb, M, N, K, 1.0, C.c_void_p(pa.value + 4 * fa), lda, C.c_void_p(pb.value + 4 * fb), ldb, 0.0, pc, M, None, ws, nb))
    got = dev.download(pc, M * N).reshape(N, M)
    for q in (pa, pb, pc, ws):
        dev.free(q)
    assert far(got, (views[1].T if tb else views[1]) @ (views[0].T if ta else views[0])) < limit(K)


def forward_2x2(dev, case, x, w):
    """The dense form of 3 x 3 windows on 2 x 2 maps (through the layer's pass, without normalisation, activation and pool)."""
    from fitre_amd.structs import CNN_ACT_NONE, NO_POOL
    n, ci, co = case[:3]
    shape = conv_shape(n, ci, co, 2, 2, 3, 1, 1)
    nb, size = hip.fitre_hip_conv_bn_act_pool_workspace(C.byref(shape), 0), co * n * 4
    px, pw, ws, y, act = dev.upload(flat(x)), dev.upload(w.numpy().ravel()), dev.alloc(nb), dev.zeros(size), dev.zeros(size)
    L.check(hip.fitre_hip_conv_bn_act_pool_forward(C.byref(shape), px, pw, None, y, None, None, None, None, None, 1e-5, 0.1, 1, CNN_ACT_NONE,
                                                   act, NO_POOL, 0, 0, 0, 0, 0, None, 0, ws, nb))
    got = dev.download(y, size).reshape(co, n, 2, 2)
    for q in (px, pw, ws, y, act):
        dev.free(q)
    return got


@pytest.mark.parametrize("n", [130, 200])
def test_forward_on_2x2_maps(dev, n):
    ci, co = 96, 132
    case = (n, ci, co, 2, 2, 3)
    x, w, _ = tensors(case)
    assert far(forward_2x2(dev, case, x, w), reference(case, "fwd", x, w)) < limit(ci * 4)
    odd = x.clone()
    odd[5, 3, 1, 0], odd[n - 1, 95, 0, 1] = float("inf"), float("nan")
    got, want = forward_2x2(dev, case, odd, w), reference(case, "fwd", odd, w)
    finite = np.isfinite(want)
    np.testing.assert_array_equal(np.isfinite(got), finite)
    assert far(got[finite], want[finite]) < limit(ci * 4, 0.6)
    assert far(forward_2x2(dev, case, x * 2.0**-108, w) * 2.0**108, reference(case, "fwd", x, w)) < limit(ci * 4, 0.6)


def product(dev, a, b):
    (K, M), N = a.shape, b.shape[0]
    nb = hip.fitre_hip_gemm_workspace(M, N, K)
    pa, pb, pc, ws = dev.upload(a.numpy().ravel()), dev.upload(b.numpy().ravel()), dev.zeros(M * N), dev.alloc(max(nb, 4))
    with taken(FC_GEMM, SPLIT):
        L.check(hip.fitre_hip_gemm(0, 0, M, N, K, 1.0, pa, M, pb, K, 0.0, pc, M, None, ws, nb))
    got = dev.download(pc, M * N).reshape(N, M)
    for q in (pa, pb, pc, ws):
        dev.free(q)
    return got


def one_of_each(kernel):
    """(factors, run(dev, factors), float64 result, terms of a sum) of a product on one of the kernels."""
    if kernel == "product":
        g = torch.Generator().manual_seed(1)
        factors = torch.randn(777, 200, generator=g), torch.randn(130, 777, generator=g)
        return factors, product, lambda a, b: (b.double() @ a.double()).numpy(), 777
    case = {"forward": (80, 128, 128, 8, 8, 3), "input gradient": (80, 128, 128, 8, 8, 3), "cell": (159, 192, 208, 4, 4, 3), "2x2": (130, 96, 132, 2, 2, 3),
            "weight gradient": (64, 128, 128, 8, 8, 3), "weight gradient 5x5": (20, 64, 64, 15, 15, 5)}[kernel]
    x, w, d = tensors(case)
    if kernel.startswith("weight"):
        return (x, d), lambda dev, x, d: weight_grad(dev, case, x, d), lambda x, d: weight_reference(case, x, d), case[0] * case[3] * case[4]
    which = "dx" if kernel == "input gradient" else "fwd"
    run = (lambda dev, s, w: forward_2x2(dev, case, s, w)) if kernel == "2x2" else (lambda dev, s, w: conv(dev, case, which, s, w))
    return (d if which == "dx" else x, w), run, lambda s, w: reference(case, which, s, w), case[1] * case[5] ** 2


@pytest.mark.parametrize("kernel", ["forward", "input gradient", "cell", "2x2", "weight gradient", "weight gradient 5x5", "product"])
def test_small_numbers(dev, kernel):
    """Factors of any size are carried, subnormal ones too: a power of two in front of a tensor changes no bit, a factor without its
    lower parts is not hidden by a large one beside it, and what is below the smallest normal result is rounded, not dropped."""
    (a, b), run, want, terms = one_of_each(kernel)
    plain = run(dev, a, b)
    np.testing.assert_array_equal(run(dev, a * 2.0**-100, b), plain * np.float32(2.0**-100))
    np.testing.assert_array_equal(run(dev, a, b * 2.0**-100), plain * np.float32(2.0**-100))
    for first, second in ((-124, 60), (-138, 100), (60, -124), (100, -138)):
        fa, fb = a * 2.0**first, b * 2.0**second  # from 2^-127 on rounded to the numbers there are
        back = 2.0 ** -(first + second)
        assert far(run(dev, fa, fb).astype(np.float64) * back, want(fa, fb) * back) < limit(terms)
    tiny = run(dev, a * 2.0**-70, b * 2.0**-70).astype(np.float64) - want(a * 2.0**-70, b * 2.0**-70)
    assert np.abs(tiny).max() < (terms / 16 + 1) * 2.0**-150  # every range of the reduction is rounded once, the shortest has sixteen terms
