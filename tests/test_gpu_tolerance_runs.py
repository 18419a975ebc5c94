"""Ground-state runs whose Ritz value is checked on the way (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu

# a resident chain, two-launch steps (one and several hopping values)
CASES = [(lattice.ring(8), (4, 4)), (lattice.square(3, 4), (6, 5)), (lattice.disordered_rect(3, 4), (5, 6))]


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_checks_do_not_change_the_recurrence(ed, k, prec, monkeypatch):
    """A tolerance that no step meets (checks every five steps of an unconverged
    run) gives the bits of the run without one: coefficients, energy, vector.
    With the eigenvector from the second run of the chain too, so that that run
    repeats the first one's recurrence."""
    H, sec = CASES[k]
    ed.set_hamiltonian(H, [6.0])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    print(f"tolerance run {prec} sector {sec} dim {dim}", flush=True)
    for basis in ("1", "0"):
        monkeypatch.setenv("EDL_LANCZOS_BASIS", basis)
        free = ed.lanczos_eigh(isec, prec, niter=33, want_vector=True)
        chk = ed.lanczos_eigh(isec, prec, niter=33, tol=1e-300, want_vector=True)
        assert chk["nsteps"] == free["nsteps"] == 33
        np.testing.assert_array_equal(chk["alpha"], free["alpha"])
        np.testing.assert_array_equal(chk["beta"], free["beta"])
        assert chk["e0"] == free["e0"]
        np.testing.assert_array_equal(chk["gs"], free["gs"])


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_vector_from_basis_and_from_second_run(ed, k, prec, monkeypatch):
    """A run ended by its tolerance: the same coefficients and the same vector
    from the stored basis and from the second run of the chain.  The two add the
    same terms in the same order, with weights rounded once and twice: 1e-12."""
    H, sec = CASES[k]
    ed.set_hamiltonian(H, [6.0])
    isec = ed.sector_index(*sec)
    ed.build_sector(isec)
    print(f"basis and second run {prec} sector {sec}", flush=True)
    r = []
    for basis in ("1", "0"):
        monkeypatch.setenv("EDL_LANCZOS_BASIS", basis)
        r.append(ed.lanczos_eigh(isec, prec, niter=150, tol=1e-12, want_vector=True))
    if prec == "fp64":
        np.testing.assert_array_equal(r[0]["alpha"], r[1]["alpha"])
        assert r[0]["e0"] == r[1]["e0"]
    assert np.max(np.abs(r[0]["gs"] - r[1]["gs"])) < 1e-12
