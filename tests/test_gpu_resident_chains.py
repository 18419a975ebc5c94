"""Lanczos chains of small sectors run whole by one block, against the
step-by-step kernels and the oracle (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu

# sectors around the edges of the elements a thread holds (1, 2, 4, 5, 8, 16 of
# 1024 threads), the smallest, one string of a spin, one and several hopping values
SECTORS = [(lattice.ring(2), 2.0, (1, 1)), (lattice.ring(6), 4.0, (1, 0)), (lattice.ring(6), 4.0, (3, 3)),
           (lattice.disordered_rect(2, 3), 3.0, (3, 2)), (lattice.ring(8), 4.0, (2, 4)), (lattice.ring(8), 4.0, (4, 4)),
           (lattice.ring(7), 4.0, (3, 4)), (lattice.disordered_rect(3, 3), 4.0, (4, 3)),
           (lattice.square(3, 3), 5.0, (4, 5)), (lattice.disordered_rect(3, 3), 4.0, (4, 4))]


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("k", range(len(SECTORS)))
def test_resident_tridiag_vs_oracle(ed, orc, k, prec):
    """Coefficients of a random seed against the oracle's recurrence: the
    first ten, where rounding is not yet amplified (fp64 1e-9; fp32 vectors
    and products 1e-4, ten steps of 2e-6 each)."""
    H, U, sec = SECTORS[k]
    m = orc.Model(H, [U])
    ed.set_hamiltonian(H, [U])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    print(f"resident chain {prec} sector {sec} dim {dim}", flush=True)
    seed = np.random.default_rng(k).standard_normal(dim)
    a, b, n2 = ed.tridiag_Hv_sector(isec, seed, 12, prec)
    ao, bo, _ = orc.lanczos_tridiag(orc.hamiltonian_csr(m, *sec), seed, 12)
    tol = 1e-9 if prec == "fp64" else 1e-4
    assert abs(n2 - seed @ seed) < 1e-12 * n2
    n = min(10, len(ao), max(1, dim // 2))
    np.testing.assert_allclose(a[:n], ao[:n], rtol=tol, atol=tol)
    np.testing.assert_allclose(b[1:n], bo[1:n], rtol=tol, atol=tol)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("k", [1, 3, 5, 9])
def test_resident_ground_state_vs_dense(ed, orc, k, prec):
    """E0 and the state against dense diagonalisation, with a tolerance that
    ends the run (several launches) and without."""
    H, U, sec = SECTORS[k]
    m = orc.Model(H, [U])
    ed.set_hamiltonian(H, [U])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    print(f"resident ground state {prec} sector {sec} dim {dim}", flush=True)
    Hc = orc.hamiltonian_csr(m, *sec)
    for tol in (0.0, 1e-13):
        r = ed.lanczos_eigh(isec, prec, niter=200, tol=tol, want_vector=True)
        x = r["gs"]
        assert abs(np.linalg.norm(x) - 1.0) < 1e-12
        res = np.linalg.norm(Hc @ x - r["e0"] * x)
        assert res < 1e-4 * max(1.0, abs(r["e0"])), res  # |dE| <= res^2 / gap: 1e-8 in the energy
        if dim <= 5000:
            e0 = np.linalg.eigvalsh(Hc.toarray())[0]
            assert abs(r["e0"] - e0) < 1e-10 * abs(e0)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_resident_seeds_equal_tiles(ed, prec, monkeypatch):
    """Every kind of seed, in groups of all and of one, on the ring and a
    disordered cluster: norms to 1e-12 and the leading coefficients against the
    tile kernels (fp64: ten to 1e-9; fp32: four to 1e-4, a recurrence from a
    ground-state seed amplifies rounding about sevenfold a step, so that the
    tenth of any fp32 kernel is off its fp64 value in the first digits)."""
    for H, U, sec in ((lattice.ring(8), 4.0, (4, 4)), (lattice.disordered_rect(2, 4, seed=11), 4.0, (4, 3))):
        ed.set_hamiltonian(H, [U])
        isec = ed.sector_index(*sec)
        ed.lanczos_eigh(isec, "fp64", niter=100)
        seeds = [("cdg", 1, 1, 0), ("c", 1, 2, 5), ("cdg", 2, 3, 0), ("c", 2, 4, 6), ("sz", 1, 3, 0), ("sz", 1, 2, 7),
                 ("j", 0, 1, 0)]
        monkeypatch.delenv("EDL_BATCHED_KERNELS", raising=False)
        r = ed.tridiag_batched(seeds, 30, prec)
        r1 = ed.tridiag_batched(seeds, 30, prec, group=1)
        monkeypatch.setenv("EDL_BATCHED_KERNELS", "tiles")
        t = ed.tridiag_batched(seeds, 30, prec)
        tol = 1e-9 if prec == "fp64" else 1e-4
        np.testing.assert_array_equal(r["alpha"], r1["alpha"])
        np.testing.assert_array_equal(r["nsteps"], t["nsteps"])
        np.testing.assert_array_equal(r["isector"], t["isector"])
        np.testing.assert_allclose(r["norm2"], t["norm2"], rtol=1e-12, atol=1e-14)
        n = 10 if prec == "fp64" else 4
        np.testing.assert_allclose(r["alpha"][:, :n], t["alpha"][:, :n], rtol=tol, atol=tol)
        np.testing.assert_allclose(r["beta"][:, :n], t["beta"][:, :n], rtol=tol, atol=tol)
