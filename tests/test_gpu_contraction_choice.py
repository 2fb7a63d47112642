"""The form of the FAST methods on truncated spaces: a rejected table shape changes nothing, the
autotuner leaves the faster form (with the table kernels' tables gone where it built them), and the
caller can go back from the tables."""
import numpy as np
import pytest

from conftest import rand_vectors

pytestmark = pytest.mark.gpu


@pytest.fixture
def ham(J, ctx):
    m1, m2 = J.synth_integrals(10, 83)
    gs = J.Space(ctx, 4, 4, 10, 2, 4, 2, 1)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    yield h, rand_vectors(gs.ndets, 3, 16)
    h.close()
    gs.close()


def test_rejected_shapes_change_nothing(J, ham):
    h, X = ham
    want = [h.sigma(X, method=m) for m in (J.SIGMA_FAST64, J.SIGMA_FAST32)]
    for bad in (lambda: h.fast_tiles(width=100), lambda: h.fast_tiles(width=64, chunk=3),
                lambda: h.fast_tiles(chunk=16), lambda: h.fast_split(4), lambda: h.fast_xcd(5000),
                lambda: h.contraction(use=2)):
        with pytest.raises(J.JciError):
            bad()
        assert h.contraction()[0] == 1
        for m, y in zip((J.SIGMA_FAST64, J.SIGMA_FAST32), want):
            assert np.array_equal(h.sigma(X, method=m), y)


def test_autotune_and_back(J, ham):
    h, X = ham
    want = [h.sigma(X, method=m) for m in (J.SIGMA_FAST64, J.SIGMA_FAST32)]
    scale = np.abs(want[0]).max()
    h.autotune(nvec=1, reps=3)
    h.contraction(use=1)
    for m, y in zip((J.SIGMA_FAST64, J.SIGMA_FAST32), want):
        assert np.array_equal(h.sigma(X, method=m), y)
    for split in (1, 0, 2):                          # the tables, built again where they had gone
        assert h.fast_split(split) == split and h.contraction()[0] == 0
        assert np.abs(h.sigma(X, method=J.SIGMA_FAST64) - want[0]).max() < 1e-12 * scale
        assert np.abs(h.sigma(X, method=J.SIGMA_FAST32) - want[0]).max() < 2e-5 * scale
    h.autotune(nvec=3, reps=3)
    assert h.contraction(use=1)[0] == 1
    for m, y in zip((J.SIGMA_FAST64, J.SIGMA_FAST32), want):
        assert np.array_equal(h.sigma(X, method=m), y)


def test_no_form_to_go_back_to(J, ctx):
    m1, m2 = J.synth_integrals(8, 89)
    gs = J.Space(ctx, 3, 1, 8, 1, 3, 2, 0)           # one electron of a spin
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    assert h.contraction()[0] == 0
    with pytest.raises(J.JciError):
        h.contraction(use=1)
    h.close()
    gs.close()
