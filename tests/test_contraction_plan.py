"""Rounds of the truncated-space sigma's contraction form, planned on the host: no round's
intermediate exceeds the bound, however large the space, and small bounds force every way of
cutting one (the cases that the GPU runs against the oracle in test_gpu_contraction_cuts.py)."""
import pytest

BOUND = 256 << 20       # elements per vector, 2 GiB in FP64; the determinants where they are more


@pytest.mark.parametrize("spec,bound", [
    ((8, 8, 60, 4, 8, 2, 1), 603651972), ((8, 8, 40, 4, 8, 2, 1), BOUND),
    ((8, 8, 28, 4, 8, 2, 1), BOUND), ((10, 10, 30, 6, 8, 2, 1), BOUND),
    ((22, 22, 44, 20, 4, 2, 1), BOUND), ((18, 18, 40, 16, 4, 2, 1), BOUND),
    ((6, 6, 14, 2, 8, 2, 1), BOUND),
])
def test_rounds_within_bound(J, spec, bound):
    p = J.contraction_plan(*spec)
    assert p is not None and 0 < p["elems"] <= bound, p
    assert p["grid"] < 1 << 24
    # cut finer, as many elements in all
    q = J.contraction_plan(*spec, elems=BOUND // 16)
    assert q["elems"] <= BOUND // 16 and q["total"] == p["total"], q
    assert sum(q["rounds"]) > sum(p["rounds"])


# (space, bound) and whether it cuts by external parts, column tiles, strings JL, columns and N - 2
# electron strings
CUTS = [
    ((5, 4, 12, 2, 5, 2, 1), 100000, (1, 0, 0, 1, 1)),
    ((5, 4, 12, 2, 5, 2, 1), 30000, (1, 1, 1, 1, 1)),
    ((5, 4, 12, 2, 5, 2, 1), 3000, (1, 1, 1, 1, 1)),
    ((3, 3, 26, 1, 4, 2, 1), 200000, (1, 0, 1, 1, 0)),
    ((3, 3, 26, 1, 4, 2, 1), 20000, (1, 0, 1, 1, 1)),
    ((4, 3, 9, 1, 5, 2, 0), 6000, (1, 0, 1, 0, 1)),
    ((2, 2, 30, 1, 2, 1, 0), 5000, (1, 0, 1, 0, 0)),
]


@pytest.mark.parametrize("spec,elems,cuts", CUTS)
def test_cuts(J, spec, elems, cuts):
    p = J.contraction_plan(*spec, elems=elems)
    assert p["elems"] <= elems
    assert tuple(int(n > 0) for n in p["split"]) == cuts, p
    assert p["total"] == J.contraction_plan(*spec)["total"]


def test_lane_counts_the_planned_buffers(J):
    """The lane's memory estimate covers the buffers that the plan asks for, and block solves of
    the largest space fit the card (309 GB): three roots with the sigma's vectors at once, five
    with one at a time."""
    from jayci_amd import serve
    for spec in ((8, 8, 60, 4, 8, 2, 1), (22, 22, 44, 20, 4, 2, 1), (3, 3, 26, 1, 4, 2, 1)):
        d = dict(zip(("na", "nb", "norbs", "ndocc", "nactv", "xlvl", "rule"), spec), nroots=3)
        e = serve.sigma_elems(d, 10 ** 6)
        assert e >= J.contraction_plan(*spec)["elems"]
    N = 603651972
    d = dict(na=8, nb=8, norbs=60, ndocc=4, nactv=8, xlvl=2, rule=1)
    e = serve.sigma_elems(d, N)
    for nroots, at_once, krymax in ((3, None, 18), (5, 1, 15)):
        p = serve.lane_solve_params(dict(d, nroots=nroots), N, budget=300e9, kfac=6, at_once=at_once)
        nt = p["nroots"] + p["nbuffer"]
        assert p["krymax"] >= krymax
        # basis and sigma vectors, new directions and sigma input, buffers, diagonal
        need = 8 * N * (2 * p["krymax"] + 2 * nt + 1) + (at_once or nt) * (
            32 * N + 8 * J.contraction_plan(8, 8, 60, 4, 8, 2, 1)["elems"])
        assert need <= serve.lane_vector_bytes(N, p["krymax"], nt, e, at_once) <= 300e9
    # one block: the table kernels' transposed input and tables
    assert serve.sigma_elems(dict(d, ndocc=0, nactv=60, xlvl=0), 10 ** 6) == 0


@pytest.mark.parametrize("spec,taken", [
    # few internal orbitals, many excitations: the table kernels are faster
    ((2, 2, 60, 0, 2, 4, 0), False), ((2, 2, 50, 1, 0, 4, 0), False), ((3, 3, 34, 0, 2, 6, 0), False),
    ((4, 4, 20, 0, 2, 6, 0), False), ((4, 4, 16, 0, 4, 8, 0), False), ((4, 4, 30, 2, 1, 4, 0), False),
    ((5, 5, 18, 0, 4, 6, 0), False), ((3, 3, 26, 0, 2, 4, 0), False),
    # few internal orbitals, two excitations or few connections; and truncated CAS spaces
    ((2, 2, 60, 0, 2, 2, 0), True), ((8, 8, 60, 8, 0, 2, 1), True), ((4, 4, 24, 0, 4, 4, 0), True),
    ((3, 3, 16, 0, 2, 4, 0), True), ((2, 2, 6, 1, 2, 2, 1), True), ((4, 4, 10, 2, 4, 2, 1), True),
    ((7, 7, 14, 2, 10, 2, 1), True), ((6, 6, 16, 0, 12, 2, 0), True), ((8, 8, 60, 4, 8, 2, 1), True),
    # one electron of a spin; one block
    ((3, 1, 8, 1, 3, 2, 0), False), ((3, 3, 8, 0, 8, 0, 1), False),
])
def test_form_chosen(J, spec, taken):
    assert (J.contraction_plan(*spec) is not None) == taken
