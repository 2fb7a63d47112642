"""The dense-string sigma of a vector does not depend on the vectors that go with it: alone, in a
block, in the passes of the allocation-free entry point and in a batch whose pool leaves room for
fewer of them, to the last bit."""
import numpy as np
import pytest

from conftest import rand_vectors
from test_zz_no_alloc import DevBuf, _entry_points, _hip

pytestmark = pytest.mark.gpu


# 495 x 924 and 715 x 715 strings of several vectors would tie between tiles of 64 and 128; 1287 x
# 1287 (two vectors) likewise; 2002 x 2002 takes 128 for any number
@pytest.mark.parametrize("na,nb,n,nvec", [(3, 3, 8, 8), (4, 4, 12, 7), (4, 6, 12, 7), (4, 4, 13, 6),
                                          (5, 5, 13, 2), (5, 5, 14, 2)])
def test_vectors_alone_and_together(J, ctx, na, nb, n, nvec):
    L, hip = _entry_points(J), _hip()
    m1, m2 = J.synth_integrals(n, 43)
    gs = J.Space(ctx, na, nb, n)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    N = gs.ndets
    X = rand_vectors(N, nvec, 8)
    bx, by = DevBuf(hip, 8 * N * nvec), DevBuf(hip, 8 * N * nvec)
    bx.put(np.ascontiguousarray(X.T))
    for method in (J.SIGMA_GEMM64, J.SIGMA_GEMM32):
        Y = h.sigma(X, method=method)
        for k in (0, nvec - 1):
            assert np.array_equal(Y[k], h.sigma(X[k], method=method)), (method, k)
        # what the scratch array has room for: all, and one vector a pass
        if n < 12 or ((na, nb, n) == (4, 6, 12) and method == J.SIGMA_GEMM32):
            by.fill(0x11)
            assert L.jci_sigma_dev_noalloc(h._h, method, nvec, bx.p, by.p) == 0, J.last_error()
            ctx.sync()
            assert np.array_equal(by.get((N, nvec)).T, Y), method
    bx.free()
    by.free()
    h.close()
    gs.close()


def test_batch_independent_of_pool(J, ctx):
    # 5a5b/13, two pending vectors: a pool for one vector's intermediate and one for all
    m1, m2 = J.synth_integrals(13, 44)
    gs = J.Space(ctx, 5, 5, 13)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    p = h.params(nroots=2, restol=1e-6, krymin=4, krymax=16, maxiter=6, refdim=64,
                 guess=J.GUESS_DIAG)
    out = []
    for pool in (600 << 20, 4 << 30):
        b = J.Batch(ctx, 2, 16, pool_bytes=pool)
        slot = b.add(h, p)
        b.run(6)
        out.append(b.result(slot)[0])
        b.close()
    assert np.array_equal(out[0], out[1])
    h.close()
    gs.close()
