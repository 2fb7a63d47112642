"""The contraction form in many rounds against the oracle: every way of cutting the intermediate
(CUTS of test_contraction_plan.py: ranges of external parts, of column tiles, of first-spin strings,
of columns and of N - 2 electron strings, tasks one by one), several vectors, both precisions."""
import numpy as np
import pytest

from conftest import rand_vectors
from test_contraction_plan import CUTS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec,elems,cuts", CUTS)
def test_cut_rounds_against_oracle(J, orc, ctx, spec, elems, cuts):
    m1, m2 = J.synth_integrals(spec[2], 67)
    gs = J.Space(ctx, *spec)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    X = rand_vectors(gs.ndets, 3, 13)
    ref = orc.Space(*spec).sigma(m1, m2, X)
    scale = np.abs(ref).max()
    plan = J.contraction_plan(*spec, elems=elems)
    use, most, _, rounds = h.contraction(elems=elems)
    assert use == 1 and most == plan["elems"] and rounds == plan["rounds"]
    for k in (1, 3):
        # FP64: as for every other FP64 sigma, 1e-12 of the result's scale; FP32 2e-5
        e64 = np.abs(h.sigma(X[:k], method=J.SIGMA_FAST64) - ref[:k]).max() / scale
        e32 = np.abs(h.sigma(X[:k], method=J.SIGMA_FAST32) - ref[:k]).max() / scale
        assert e64 < 1e-12, (k, e64)
        assert e32 < 2e-5, (k, e32)
    h.close()
    gs.close()


def test_rounds_of_a_larger_space(J, ctx):
    # 7a6b/17: 34M and 27M elements, here in rounds of at most 2M; the default takes one a part
    m1, m2 = J.synth_integrals(17, 71)
    gs = J.Space(ctx, 7, 6, 17, 3, 6, 2, 1)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    X = rand_vectors(gs.ndets, 2, 14)
    assert h.contraction()[3] == (1, 1)
    ref = h.sigma(X, method=J.SIGMA_FAST64)
    scale = np.abs(ref).max()
    use, most, _, rounds = h.contraction(elems=2 << 20)
    assert most <= 2 << 20 and rounds[0] > 8 and rounds[1] > 8
    assert np.abs(h.sigma(X, method=J.SIGMA_FAST64) - ref).max() / scale < 1e-12
    assert np.abs(h.sigma(X, method=J.SIGMA_FAST32) - ref).max() / scale < 2e-5
    h.close()
    gs.close()
