"""Truncated instances of a batch hold the table kernels' memory only: Hamiltonians created for one
(TABLE_KERNELS) from the start, others from admission on, unless the allocation-free entry point
has used their buffers; the form can be brought back."""
import numpy as np
import pytest

from conftest import rand_vectors
from test_zz_no_alloc import DevBuf, _entry_points, _hip

pytestmark = pytest.mark.gpu
SPEC = (4, 4, 10, 2, 4, 2, 1)


@pytest.fixture
def space(J, ctx):
    gs = J.Space(ctx, *SPEC)
    yield gs, J.synth_integrals(10, 97), rand_vectors(gs.ndets, 3, 17)
    gs.close()


def _energy(J, ctx, h):
    b = J.Batch(ctx, 2, 16)
    slot = b.add(h, h.params(nroots=1, restol=1e-8, krymin=4, krymax=16, refdim=32, guess=J.GUESS_DIAG))
    b.run(200)
    ev, _, st = b.result(slot)
    assert st["converged"]
    b.close()
    return ev[0]


def test_created_for_a_batch(J, ctx, space):
    gs, (m1, m2), X = space
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES | J.TABLE_KERNELS)
    d = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    assert h.contraction()[0] == 0 and h.contraction()[2] == 0
    assert d.contraction()[0] == 1 and d.contraction()[2] > 0
    want = d.sigma(X, method=J.SIGMA_FAST64)
    d.fast_split(2)
    assert np.array_equal(h.sigma(X, method=J.SIGMA_FAST64), d.sigma(X, method=J.SIGMA_FAST64))
    e = _energy(J, ctx, h)
    assert abs(e - d.solve(nroots=1, restol=1e-8)[0][0]) < 1e-10
    assert h.contraction()[2] == 0
    assert h.contraction(use=1)[0] == 1              # built where it was left out
    assert np.array_equal(h.sigma(X, method=J.SIGMA_FAST64), want)
    d.close()
    h.close()


def test_admission_gives_the_memory_back(J, ctx, space):
    gs, (m1, m2), X = space
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    want = h.sigma(X, method=J.SIGMA_FAST64)
    scale = np.abs(want).max()
    with pytest.raises(J.JciError):                  # refused: nothing changes
        J.Batch(ctx, 2, 8).add(h, h.params())
    assert h.contraction()[0] == 1 and np.array_equal(h.sigma(X, method=J.SIGMA_FAST64), want)
    e = _energy(J, ctx, h)
    assert h.contraction()[0] == 0 and h.contraction()[2] == 0
    assert np.abs(h.sigma(X, method=J.SIGMA_FAST64) - want).max() < 1e-12 * scale
    assert h.contraction(use=1)[0] == 1
    assert np.array_equal(h.sigma(X, method=J.SIGMA_FAST64), want)
    assert abs(_energy(J, ctx, h) - e) < 1e-12
    h.close()


def test_used_buffers_stay(J, ctx, space):
    gs, (m1, m2), X = space
    L, hip = _entry_points(J), _hip()
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    N = gs.ndets
    bx, by = DevBuf(hip, 8 * N), DevBuf(hip, 8 * N)
    bx.put(X[0])
    out = []
    for _ in range(2):
        by.fill(0x11)
        assert L.jci_sigma_dev_noalloc(h._h, J.SIGMA_FAST64, 1, bx.p, by.p) == 0, J.last_error()
        ctx.sync()
        out.append(by.get((N,)))
        held = h.contraction()[2]
        _energy(J, ctx, h)
        assert h.contraction()[0] == 1 and h.contraction()[2] == held > 0
    assert np.array_equal(out[0], out[1])
    bx.free()
    by.free()
    h.close()
