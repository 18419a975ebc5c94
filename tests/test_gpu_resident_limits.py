"""Resident chains at every number of elements a thread holds, and where chains
run resident at all (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu

# 1, 2, 5 (just below 1 024, 2 048, 5 120 states), 3, 4, 8, 12 and 16 elements of 1024
# threads; one and several hopping values
SECTORS = [(lattice.ring(13), (1, 2)), (lattice.ring(10), (2, 2)), (lattice.ring(14), (1, 3)), (lattice.ring(9), (2, 3)),
           (lattice.ring(8), (3, 4)), (lattice.ring(9), (3, 3)), (lattice.disordered_rect(3, 3), (3, 3)),
           (lattice.square(3, 3), (4, 3)), (lattice.disordered_rect(2, 5), (3, 3)), (lattice.square(3, 3), (4, 4))]


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


def _route(capfd):
    return [x.split(": ")[1] for x in capfd.readouterr().err.splitlines() if x.startswith("[edl] chain steps: ")]


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("k", range(len(SECTORS)))
def test_elements_a_thread_vs_oracle(ed, orc, k, prec, monkeypatch, capfd):
    """Coefficients of a random seed against the oracle's recurrence, the first ten
    (fp64 1e-9; fp32 vectors and products 1e-4, ten steps of 2e-6 each)."""
    H, sec = SECTORS[k]
    m = orc.Model(H, [4.0])
    ed.set_hamiltonian(H, [4.0])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    monkeypatch.setenv("EDL_RESIDENT", "1")
    monkeypatch.setenv("EDL_VERBOSE", "1")
    seed = np.random.default_rng(k).standard_normal(dim)
    capfd.readouterr()
    a, b, n2 = ed.tridiag_Hv_sector(isec, seed, 12, prec)
    assert _route(capfd) == ["resident"]
    ao, bo, _ = orc.lanczos_tridiag(orc.hamiltonian_csr(m, *sec), seed, 12)
    tol = 1e-9 if prec == "fp64" else 1e-4
    assert abs(n2 - seed @ seed) < 1e-12 * n2
    np.testing.assert_allclose(a[:10], ao[:10], rtol=tol, atol=tol)
    np.testing.assert_allclose(b[1:10], bo[1:10], rtol=tol, atol=tol)


# (lattice, sector, precision, whether its ground state runs resident, chains a group, whether they do)
LIMITS = [(lattice.square(3, 3), (3, 3), "fp64", True, 2, True), (lattice.ring(11), (2, 3), "fp64", True, 2, True),
          (lattice.square(3, 3), (4, 3), "fp64", False, 2, True), (lattice.square(3, 3), (4, 4), "fp64", False, 2, False),
          (lattice.square(3, 3), (4, 4), "fp64", False, 128, True), (lattice.square(3, 3), (4, 4), "fp32", False, 32, True),
          (lattice.ring(10), (2, 5), "fp32", True, 2, True), (lattice.disordered_rect(3, 3), (3, 3), "fp64", True, 2, True),
          (lattice.disordered_rect(3, 3), (4, 3), "fp64", False, 2, False),
          (lattice.disordered_rect(3, 3), (4, 3), "fp64", False, 32, True),
          (lattice.disordered_rect(2, 5), (3, 3), "fp32", False, 2, False)]


@pytest.mark.parametrize("k", range(len(LIMITS)))
def test_limit(ed, orc, k, monkeypatch, capfd):
    """The form taken on both sides of the limits, and the same answers as from the
  other one: E0 (fp64 1e-10, fp32 1e-5) and a seed's leading coefficients (eight
    to 1e-9, four to 1e-4: a ground-state seed amplifies rounding about sevenfold a
    step)."""
    H, sec, prec, gs, n, seeds = LIMITS[k]
    ed.set_hamiltonian(H, [4.0])
    isec = ed.sector_index(*sec)
    ed.build_sector(isec)
    monkeypatch.setenv("EDL_VERBOSE", "1")
    sd = [("sz", 1, 1 + j % H.shape[1], 0) for j in range(n)]
    r, t = [], []
    for pin in (None, "0" if gs else "1"):
        if pin:
            monkeypatch.setenv("EDL_RESIDENT", pin)
        capfd.readouterr()
        r.append(ed.lanczos_eigh(isec, prec, niter=120))
        assert (_route(capfd) == ["resident"]) == (gs if pin is None else not gs)
    monkeypatch.setenv("EDL_RESIDENT", "0")
    ed.lanczos_eigh(isec, "fp64", niter=120)  # one state for both groups
    for pin in (None, "0" if seeds else "1"):
        if pin:
            monkeypatch.setenv("EDL_RESIDENT", pin)
        else:
            monkeypatch.delenv("EDL_RESIDENT")
        capfd.readouterr()
        t.append(ed.tridiag_batched(sd, 20, prec))
        assert (_route(capfd) == ["resident"]) == (seeds if pin is None else not seeds)
    assert abs(r[0]["e0"] - r[1]["e0"]) < (1e-10 if prec == "fp64" else 1e-5) * abs(r[0]["e0"])
    c, tol = (8, 1e-9) if prec == "fp64" else (4, 1e-4)
    for key in ("alpha", "beta"):
        np.testing.assert_allclose(t[0][key][:, :c], t[1][key][:, :c], rtol=tol, atol=tol)
