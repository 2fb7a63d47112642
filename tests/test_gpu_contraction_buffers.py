"""Buffers of the contraction form: those of the allocation-free entry point stay where a captured
graph found them, whatever other calls grow; calls whose vectors do not fit go in passes with the
same results; small spaces hold enough from creation on."""
import ctypes

import numpy as np
import pytest

from conftest import rand_vectors
from test_zz_no_alloc import DevBuf, _entry_points, _hip

pytestmark = pytest.mark.gpu


def test_captured_call_survives_growth(J, ctx):
    L, hip = _entry_points(J), _hip()
    m1, m2 = J.synth_integrals(17, 53)
    gs = J.Space(ctx, 7, 6, 17, 3, 6, 2, 1)         # one vector's buffers 294 MB
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    N = gs.ndets
    bx, by = DevBuf(hip, 16 * N), DevBuf(hip, 16 * N)
    bx.put(np.ascontiguousarray(rand_vectors(N, 2, 9).T))
    st = ctypes.c_void_p(ctx.stream)
    for method, k in ((J.SIGMA_FAST64, 1), (J.SIGMA_FAST32, 2)):
        assert L.jci_sigma_dev_noalloc(h._h, method, k, bx.p, by.p) == 0, J.last_error()
        ctx.sync()
        want = by.get((2 * N,))[:N * k]
        g, ex = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(st, 1) == 0
        rc = L.jci_sigma_dev_noalloc(h._h, method, k, bx.p, by.p)
        assert hip.hipStreamEndCapture(st, ctypes.byref(g)) == 0 and rc == 0
        assert hip.hipGraphInstantiate(ctypes.byref(ex), g, None, None, ctypes.c_size_t(0)) == 0
        for grow in (1, 2, 4):
            # up to more vectors than the kept buffers hold
            held = h.contraction()[2]
            X = rand_vectors(N, grow, 10)
            Y = h.sigma(X, method=J.SIGMA_FAST64)
            assert np.abs(Y).max() > 0
            if grow == 4 and method == J.SIGMA_FAST64:
                assert h.contraction()[2] > held
            by.fill(0x11)
            ctx.sync()
            assert hip.hipGraphLaunch(ex, st) == 0
            ctx.sync()
            assert np.array_equal(by.get((2 * N,))[:N * k], want), (method, grow)
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(g)
    for b in (bx, by):
        b.free()
    h.close()
    gs.close()


@pytest.mark.parametrize("spec", [(5, 4, 12, 2, 5, 2, 1), (6, 6, 14, 2, 8, 2, 1)])
def test_passes_give_the_same_results(J, ctx, spec):
    m1, m2 = J.synth_integrals(spec[2], 59)
    gs = J.Space(ctx, *spec)
    X = rand_vectors(gs.ndets, 8, 11)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    kept = h.contraction()[2]
    assert h.contraction(nbytes=1)[2] == kept       # nothing beyond what is kept
    out = {m: h.sigma(X, method=m) for m in (J.SIGMA_FAST64, J.SIGMA_FAST32)}
    assert h.contraction()[2] == kept
    cap = 3 * kept
    h.contraction(nbytes=cap)                       # a few vectors at a time
    for m in out:
        assert np.array_equal(h.sigma(X, method=m), out[m]), m
    assert h.contraction()[2] <= kept + cap
    h.contraction(nbytes=1 << 50)                   # all at once
    for m in out:
        assert np.array_equal(h.sigma(X, method=m), out[m]), m
        assert np.array_equal(h.sigma(X[5], method=m), out[m][5]), m
    h.close()
    gs.close()


def test_small_space_allocates_nothing_later(J, ctx):
    m1, m2 = J.synth_integrals(10, 61)
    gs = J.Space(ctx, 4, 4, 10, 2, 4, 2, 1)
    h = J.Hamiltonian(gs, m1, m2, J.DIRECT_TABLES)
    held = h.contraction()[2]
    assert 0 < held <= 64 << 20
    for m in (J.SIGMA_FAST64, J.SIGMA_FAST32):
        h.sigma(rand_vectors(gs.ndets, 8, 12), method=m)
    assert h.contraction()[2] == held
    h.close()
    gs.close()
