"""Truncated spaces of few internal orbitals, where the reordering of the vectors has about one
tile per determinant: more tiles than one launch has work-groups, more than a launch could have,
against the oracle (sampled rows where the space is large)."""
import numpy as np
import pytest

from conftest import rand_vectors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec,nvec", [((2, 2, 60, 1, 2, 2, 1), 2),      # 19,840 tiles
                                       ((4, 4, 60, 2, 4, 2, 1), 1)])     # 35,580
def test_many_tiles(J, orc, ctx, spec, nvec):
    m1, m2 = J.synth_integrals(spec[2], 73)
    gs = J.Space(ctx, *spec)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    assert h.contraction()[0] == 1
    X = rand_vectors(gs.ndets, nvec, 15)
    rows = np.unique(np.r_[0, gs.ndets - 1, np.random.default_rng(5).integers(0, gs.ndets, size=200)])
    osp = orc.Space(*spec)
    y64, y32 = h.sigma(X, method=J.SIGMA_FAST64), h.sigma(X, method=J.SIGMA_FAST32)
    for k in range(nvec):
        ref = osp.sigma_rows(m1, m2, X[k], rows)
        scale = np.abs(ref).max()
        assert np.abs(y64[k][rows] - ref).max() < 1e-12 * scale
        assert np.abs(y32[k][rows] - ref).max() < 2e-5 * scale
    h.close()
    gs.close()


@pytest.mark.slow
def test_tile_per_determinant(J, orc, ctx):
    # 3a3b in 34 orbitals, 2 active, six excitations: 35,808,256 determinants, 30.1M tiles
    spec = (3, 3, 34, 0, 2, 6, 0)
    m1, m2 = J.synth_integrals(34, 79)
    gs = J.Space(ctx, *spec)
    assert gs.ndets == 35808256
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    x = np.random.default_rng(6).standard_normal(gs.ndets)
    y = h.sigma(x, method=J.SIGMA_FAST64)
    rows = np.unique(np.r_[0, gs.ndets - 1, np.random.default_rng(7).integers(0, gs.ndets, size=14)])
    ref = orc.Space(*spec).sigma_rows(m1, m2, x, rows)
    np.testing.assert_allclose(y[rows], ref, rtol=1e-12, atol=1e-12 * np.abs(ref).max())
    h.close()
    gs.close()
