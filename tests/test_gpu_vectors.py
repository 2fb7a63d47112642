"""The Davidson vector kernels: Gram products of every count of column tiles (and rows in whole
steps, with remainders and fewer than one) against numpy; solves of one to seven roots, whose
residuals and combinations are built per number of vectors, alone and in a batch, against dense
eigenvalues."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 63, 513, 70001])
def test_gram_tiles(J, ctx, n):
    rng = np.random.default_rng(n)
    X, Y = rng.standard_normal((64, n)), rng.standard_normal((64, n))
    for m in (2, 16, 31, 33, 50, 64):
        for w in (1, 18, 48, 49):
            G = ctx.gram(X[:m], Y[:w])
            np.testing.assert_allclose(G, X[:m] @ Y[:w].T, rtol=1e-12, atol=1e-12 * np.sqrt(n))


@pytest.mark.parametrize("nroots", [1, 2, 3, 4, 5, 6, 7])
def test_solve_roots(J, orc, ctx, nroots):
    m1, m2 = J.synth_integrals(7, 53)
    sp = J.Space(ctx, 3, 3, 7, 0, 7, 0, 1)
    h = J.Hamiltonian(sp, m1, m2, J.DIRECT_TABLES)
    w = np.linalg.eigvalsh(orc.Space(3, 3, 7, 0, 7, 0, 1).dense_h(m1, m2))[:nroots]
    kw = dict(nroots=nroots, restol=1e-7, krymin=nroots + 1, krymax=5 * nroots + 8, refdim=48)
    ev, _, st = h.solve(maxiter=400, **kw)
    np.testing.assert_allclose(ev, w, rtol=0, atol=1e-9)
    b = J.Batch(ctx, 1, 5 * nroots + 8, graphs=True)
    s = b.add(h, h.params(maxiter=400, **kw))
    b.run(400)
    ev, _, st = b.result(s)
    assert st["done"] == 1, st
    np.testing.assert_allclose(ev, w, rtol=0, atol=1e-9)
    b.release(s)
    b.close()
    h.close()
    sp.close()
