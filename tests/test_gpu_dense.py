"""Products of the fully connected family with the step behind them (fitre_hip_dense_products) against float64 numpy on the same
float32 operands.  A sum is off by at most the split's accumulation, 0.1 sqrt(K) 2^-24 of its norm and a rounding: 1e-6 at K <= 4096."""
import ctypes as C

import numpy as np
import pytest

from fitre_amd import lib as L
from fitre_amd import structs as S
from helpers import rel_err

pytestmark = pytest.mark.gpu
hip = L.hip
TOL = 2e-6  # of the largest result, which bounds the activations and derivatives behind it too

# (M, N, K): around the tile of 64 rows x 32 (or 64) columns, the step of 16 and the eight waves of a workgroup; a grid past
# the compute units, whose tiles are twice as wide; rows that are no whole 16-byte groups; the longest reduction the family brings, twice that
# with a second pair
SHAPES = [(1, 1, 1), (63, 31, 15), (64, 32, 16), (65, 33, 17), (66, 64, 127), (64, 65, 128), (130, 100, 129), (33, 17, 784), (784, 1000, 40), (1001, 999, 33), (70, 40, 4095),
          (65, 33, 4096)]


def ok(rc):
    assert rc == 0, hip.fitre_hip_last_error().decode()


class Problem:
    def __init__(self, dev, M, N, K, transA, transB, pair, offset=0):
        rng = np.random.default_rng(M * 31 + N * 7 + K + 2 * transA + transB)
        self.dev, self.shape = dev, (M, N, K)
        self.p = S.fitre_dense_product(transA=transA, transB=transB, M=M, N=N, K=K, alpha=1.0)
        self.v = np.zeros((M, N))
        for a, b in (("A", "B"), ("A2", "B2"))[:1 + pair]:
            x, y = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
            setattr(self.p, a, self.up(x.T if transA else x, offset))
            setattr(self.p, b, self.up(y.T if transB else y, offset))
            self.v += x.astype(np.float64) @ y.astype(np.float64)
            if a == "A":
                self.rows = x.astype(np.float64).sum(1)
        self.rng, self.offset = rng, offset
        self.p.C = self.up(np.full((M, N), 7, np.float32), offset)

    def up(self, matrix, offset=0):
        """Device copy of a matrix, column-major, some floats behind an allocation's start."""
        return self.dev.upload(np.concatenate([np.zeros(offset, np.float32), np.ascontiguousarray(matrix.T, np.float32).reshape(-1)])).value + 4 * offset

    def random(self):
        x = self.rng.standard_normal(self.shape[:2]).astype(np.float32)
        return x.astype(np.float64), self.up(x, self.offset)

    def get(self, ptr):
        M, N, _ = self.shape
        return self.dev.download(C.c_void_p(ptr), M * N).reshape(N, M).T

    def sums(self):
        return self.dev.download(C.c_void_p(self.p.rowSums), self.shape[0])

    def run(self):
        ok(hip.fitre_hip_dense_products(C.byref(self.p), 1))


def sigmoid(x):
    return 1 / (1 + np.exp(-x))


@pytest.mark.parametrize("transA,transB", [(0, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("pair", [0, 1])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product(dev, M, N, K, transA, transB, pair):
    q = Problem(dev, M, N, K, transA, transB, pair)
    bias = q.rng.standard_normal(M).astype(np.float32)
    q.p.alpha, q.p.bias, q.p.rowSums = -0.5, dev.upload(bias), None if transA else dev.upload(np.full(M, 9, np.float32))
    q.run()
    assert rel_err(q.get(q.p.C), -0.5 * q.v + bias[:, None]) < TOL
    assert transA or rel_err(q.sums(), -0.5 * q.rows) < TOL


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("M,N,K", [(65, 33, 17), (784, 1000, 40)])
def test_steps_behind_a_product(dev, M, N, K, offset):
    q = Problem(dev, M, N, K, 0, 0, 0, offset)
    z, q.p.z = q.random()
    x, q.p.x = q.random()
    d, q.p.d = q.random()
    q.p.raw, q.p.also = q.random()[1], q.random()[1]
    for act, f, df, g in ((S.ACT_LOGISTIC, sigmoid, z * (1 - z), 1 - 2 * z), (S.ACT_TANH, np.tanh, 1 - z * z, -2 * z), (S.ACT_LINEAR, lambda v: v, 1 + 0 * z, 0 * z)):
        q.p.act = act
        for then, want in ((S.FITRE_DENSE_ACTIVATE, f(q.v)), (S.FITRE_DENSE_DERIVATIVE, df * q.v), (S.FITRE_DENSE_ROP_BACKWARD, df * q.v + x * g * d)):
            q.p.then = then
            q.run()
            assert rel_err(q.get(q.p.C), want) < TOL, (act, then)
            assert rel_err(q.get(q.p.raw), q.v) < TOL and np.array_equal(q.get(q.p.also), -q.get(q.p.C))


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (65, 33, 17), (784, 1000, 40)])
def test_heads(dev, M, N, K):
    q = Problem(dev, M, N, K, 0, 0, 0)
    y, q.p.d = q.random()
    q.p.also = q.random()[1]
    tiles = hip.fitre_hip_dense_product_tiles(M, N)
    q.p.headSums = dev.alloc(16 * tiles)
    a, b = C.c_float(), C.c_float()
    for then, out, scale, terms in ((S.FITRE_DENSE_LOGISTIC_HEAD, sigmoid(q.v), 1, y * q.v - np.logaddexp(0, q.v)), (S.FITRE_DENSE_LINEAR_HEAD, q.v, 2, (y - q.v) ** 2)):
        q.p.then = then
        q.run()
        ok(hip.fitre_hip_dense_head_sums(q.p.headSums, tiles, C.byref(a), C.byref(b)))
        assert rel_err(q.get(q.p.C), out) < TOL and rel_err(q.get(q.p.also), scale * (y - out)) < TOL
        assert abs(a.value - terms.sum()) < TOL * np.abs(terms).sum() and abs(b.value - ((y - out) ** 2).sum()) < TOL * ((y - out) ** 2).sum()


def test_several_in_one_launch(dev):
    """The weight gradients of a pass: each as it is by itself, bit for bit."""
    q = [Problem(dev, M, N, 300, 0, 1, pair) for M, N, pair in ((784, 512, 0), (64, 33, 1), (5, 7, 0))]
    for one in q:
        one.p.rowSums = dev.zeros(one.shape[0])
        one.run()
    alone = [(one.get(one.p.C), one.sums()) for one in q]
    for one in q:
        one.p.C, one.p.rowSums = one.up(np.zeros(one.shape[:2])), dev.zeros(one.shape[0])
    ok(hip.fitre_hip_dense_products((S.fitre_dense_product * 3)(*[one.p for one in q]), 3))
    for one, (c, rows) in zip(q, alone):
        assert np.array_equal(one.get(one.p.C), c) and np.array_equal(one.sums(), rows)


@pytest.mark.parametrize("transA,transB", [(0, 0), (1, 0), (0, 1)])
def test_numbers_the_split_does_not_carry(dev, transA, transB):
    """An infinity, a NaN and products past 2^96 reach the results they are part of, and no others."""
    q = Problem(dev, 70, 40, 37, transA, transB, 0)
    x, y = np.random.default_rng(1).standard_normal((70, 37)).astype(np.float32), np.random.default_rng(2).standard_normal((37, 40)).astype(np.float32)
    x[3, 36], x[5, 0], x[7], y[0, 39] = np.inf, np.nan, 1e30, 1e35
    q.p.A, q.p.B = q.up(x.T if transA else x), q.up(y.T if transB else y)
    q.run()
    with np.errstate(all="ignore"):
        want = x.astype(np.float64) @ y.astype(np.float64)
        want = np.where(np.abs(want) > np.finfo(np.float32).max, np.sign(want) * np.inf, want)
    got = q.get(q.p.C)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    assert np.abs(got[fine] - want[fine]).max() < TOL * np.abs(want[fine]).max()


def test_refusals(dev):
    q = Problem(dev, 8, 8, 8, 0, 0, 0)
    for change in (dict(A=None), dict(A2=q.p.A), dict(M=0), dict(transA=1, transB=1), dict(transA=1, rowSums=q.p.C), dict(then=9), dict(then=S.FITRE_DENSE_DERIVATIVE, act=S.ACT_LOGISTIC),
                   dict(then=S.FITRE_DENSE_LOGISTIC_HEAD, act=S.ACT_LOGISTIC), dict(then=S.FITRE_DENSE_ACTIVATE, act=S.ACT_SOFTMAX)):
        p = S.fitre_dense_product.from_buffer_copy(q.p)
        for k, v in change.items():
            setattr(p, k, v)
        assert hip.fitre_hip_dense_products(C.byref(p), 1) != 0, change
    assert hip.fitre_hip_dense_products(C.byref(q.p), 9) != 0
