"""The full-CI sigma on every shape its kernels are built for: each reduction depth with each
count of row tiles (and the row past full tiles) against the oracle, few and many beta strings
(list lengths, columns past the last tile, fewer than four strings of a spin, the last reduction
step partly or wholly moved back inside); against the table kernels, the rows too long to stage
and each tile edge of the same-spin product."""

import numpy as np
import pytest

from conftest import rand_vectors

pytestmark = pytest.mark.gpu

# FP64: sums of up to a few thousand products, 1e-12 of the result's scale as for every other
# FP64 sigma; FP32 2e-5
SHAPES = [
    (0, 1, 3), (1, 0, 1), (1, 1, 1), (1, 1, 2), (2, 2, 2), (1, 2, 3), (2, 1, 4), (2, 3, 5),   # depth 4
    (3, 2, 6), (3, 4, 7),                                       # 8
    (2, 4, 8), (4, 4, 8), (4, 1, 9), (4, 4, 9),                 # 12: 1 tile, 1 + a row, 2
    (1, 5, 10), (2, 3, 10), (3, 1, 10), (5, 2, 10),             # 16: 1, 1 + a row, 2
    (1, 4, 11), (3, 2, 11), (3, 1, 12), (4, 2, 12), (5, 1, 12), (6, 1, 12),   # 20: 1, 2, 2 + a row, 3
    (1, 6, 13), (2, 2, 13), (4, 1, 13),                         # 24
    (1, 7, 14), (2, 2, 14), (3, 1, 14), (6, 1, 14), (7, 1, 14),   # 28: 1, 2, 3, 3 + a row, 4
    (1, 2, 15), (2, 1, 15), (3, 1, 15), (5, 1, 15),             # 32
]


@pytest.mark.parametrize("na,nb,n", SHAPES)
def test_dense_sigma_shapes(J, orc, ctx, na, nb, n):
    m1, m2 = J.synth_integrals(n, 37)
    gs = J.Space(ctx, na, nb, n, 0, n, 0, 1)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    X = rand_vectors(gs.ndets, 3, 5)
    ref = orc.Space(na, nb, n, 0, n, 0, 1).sigma(m1, m2, X)
    scale = np.abs(ref).max()
    for k in (1, 3):
        e64 = np.abs(h.sigma(X[:k], method=J.SIGMA_GEMM64) - ref[:k]).max() / scale
        e32 = np.abs(h.sigma(X[:k], method=J.SIGMA_GEMM32) - ref[:k]).max() / scale
        assert e64 < 1e-12, (k, e64)
        assert e32 < 2e-5, (k, e32)
    h.close()
    gs.close()


@pytest.mark.parametrize("na,nb,n,nvec", [
    (2, 6, 15, 1), (3, 6, 15, 1), (5, 6, 15, 1),     # rows of 5005 strings, gathered from memory
    (4, 4, 12, 1),                                    # same-spin tiles of 32 (495 strings)
    (4, 5, 13, 3),                                    # of 64 (715 x 1287)
    (5, 5, 13, 2),                                    # of 128 (1287 x 1287)
])
def test_dense_sigma_large(J, ctx, na, nb, n, nvec):
    m1, m2 = J.synth_integrals(n, 41)
    gs = J.Space(ctx, na, nb, n, 0, n, 0, 1)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    X = rand_vectors(gs.ndets, nvec, 7)
    ref = h.sigma(X, method=J.SIGMA_FAST64)
    scale = np.abs(ref).max()
    assert np.abs(h.sigma(X, method=J.SIGMA_GEMM64) - ref).max() / scale < 1e-12
    assert np.abs(h.sigma(X, method=J.SIGMA_GEMM32) - ref).max() / scale < 2e-5
    h.close()
    gs.close()
