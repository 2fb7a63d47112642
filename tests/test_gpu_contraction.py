"""The contraction form of the truncated-space sigma (the default of the FAST methods on spaces
of several blocks) against the oracle, at the edges of its tiles: groups of fewer than 16
internal parts and none or many external ones, reductions of one and of several chunks, two
electrons of a spin (one pair), unequal spins, three excitation levels, spaces with one
electron of a spin (which keep the table kernels); against the table kernels on a space whose
intermediate takes several rounds; and the allocation-free entry point bit for bit."""

import numpy as np
import pytest

from conftest import rand_vectors
from test_zz_no_alloc import DevBuf, _entry_points, _hip

pytestmark = pytest.mark.gpu

# FP64: products of up to a few thousand terms, 1e-12 of the result's scale as for every other
# FP64 sigma; FP32 2e-5
SPACES = [
    (2, 2, 6, 1, 2, 2, 1),      # one pair per spin
    (3, 2, 8, 1, 2, 3, 0),      # three levels
    (2, 3, 9, 0, 3, 2, 0),      # no doubly occupied orbitals
    (6, 5, 8, 4, 3, 2, 1),      # one external orbital
    (4, 4, 7, 3, 4, 2, 1),      # none
    (3, 2, 19, 1, 3, 1, 1),     # single external part counts of 15
    (2, 2, 30, 1, 2, 1, 0),     # reduction of one full chunk
    (3, 3, 26, 1, 4, 2, 1),     # several chunks, more rows than a wave holds
    (5, 4, 12, 2, 5, 2, 1),
    (3, 1, 8, 1, 3, 2, 0),      # one electron of a spin: table kernels
]


@pytest.mark.parametrize("spec", SPACES)
def test_contraction_against_oracle(J, orc, ctx, spec):
    na, nb, n, nd, nact, xl, rule = spec
    m1, m2 = J.synth_integrals(n, 23)
    gs = J.Space(ctx, na, nb, n, nd, nact, xl, rule)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    X = rand_vectors(gs.ndets, 8, 3)
    ref = orc.Space(na, nb, n, nd, nact, xl, rule).sigma(m1, m2, X)
    scale = np.abs(ref).max()
    for k in (1, 3, 8):
        e64 = np.abs(h.sigma(X[:k], method=J.SIGMA_FAST64) - ref[:k]).max() / scale
        e32 = np.abs(h.sigma(X[:k], method=J.SIGMA_FAST32) - ref[:k]).max() / scale
        assert e64 < 1e-12, (spec, k, e64)
        assert e32 < 2e-5, (spec, k, e32)
    h.close()
    gs.close()


def test_contraction_rounds(J, ctx):
    # 7a6b, 3 doubly occupied + 6 active + 8 external: 696,563 determinants
    m1, m2 = J.synth_integrals(17, 29)
    gs = J.Space(ctx, 7, 6, 17, 3, 6, 2, 1)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    X = rand_vectors(gs.ndets, 2, 4)
    y64, y32 = h.sigma(X, method=J.SIGMA_FAST64), h.sigma(X, method=J.SIGMA_FAST32)
    assert h.fast_split(2) == 2                     # the table kernels from here on
    ref = h.sigma(X, method=J.SIGMA_FAST64)
    scale = np.abs(ref).max()
    assert np.abs(y64 - ref).max() / scale < 1e-12
    assert np.abs(y32 - ref).max() / scale < 2e-5
    h.close()
    gs.close()


def test_contraction_noalloc(J, ctx):
    L, hip = _entry_points(J), _hip()
    m1, m2 = J.synth_integrals(12, 31)
    gs = J.Space(ctx, 5, 4, 12, 2, 5, 2, 1)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    n = gs.ndets
    bx, by = DevBuf(hip, 8 * 3 * n), DevBuf(hip, 8 * 3 * n)
    for k in (1, 3):
        bx.put(np.ascontiguousarray(rand_vectors(n, k, 6).T))
        for method in (J.SIGMA_FAST64, J.SIGMA_FAST32):
            out = []
            for f in (L.jci_sigma_dev_noalloc, L.jci_sigma_dev):
                by.fill(0xFF)
                assert f(h._h, method, k, bx.p, by.p) == 0
                ctx.sync()
                out.append(by.get((n, k)) if k == 3 else by.get((3 * n,))[:n])
            assert np.array_equal(out[0], out[1]), (k, method)
    bx.free()
    by.free()
    h.close()
    gs.close()
