"""An infinite vector element stays with the determinants it is connected to: the contraction
form of the truncated-space sigma gives every determinant more than two replacements away the
value it has with a zero in that place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec", [(2, 2, 6, 1, 2, 2, 1), (3, 2, 8, 1, 2, 3, 0), (3, 3, 8, 2, 2, 2, 1),
                                  (4, 3, 9, 1, 4, 2, 0)])
def test_infinite_element(J, ctx, spec):
    m1, m2 = J.synth_integrals(spec[2], 47)
    gs = J.Space(ctx, *spec)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    N = gs.ndets
    a, b = gs.dets()
    pop = np.array([bin(i).count("1") for i in range(1 << spec[2])])
    # the first determinants of every block (string 0 of a group among them) and a few others
    picks = sorted(set(range(0, 8)) | set(np.random.default_rng(3).integers(0, N, 24).tolist()) |
                   {i for i in range(1, N) if a[i] != a[i - 1] and i % 3 == 0})[:64]
    x = np.random.default_rng(4).standard_normal(N)
    for method, tol in ((J.SIGMA_FAST64, 1e-12), (J.SIGMA_FAST32, 2e-5)):
        for j0 in range(0, len(picks), 8):
            js = picks[j0:j0 + 8]
            X = np.tile(x, (len(js), 1))
            Z = X.copy()
            for k, j in enumerate(js):
                X[k, j], Z[k, j] = np.inf, 0.0
            Y, ref = h.sigma(X, method=method), h.sigma(Z, method=method)
            scale = np.abs(ref).max()
            for k, j in enumerate(js):
                far = (pop[(a ^ a[j]).astype(int)] + pop[(b ^ b[j]).astype(int)]) > 4
                assert np.isfinite(Y[k][far]).all(), (spec, method, j)
                assert np.abs(Y[k] - ref[k])[far].max(initial=0) <= tol * scale, (spec, method, j)
                assert not np.isfinite(Y[k][j])
    h.close()
    gs.close()
