"""Lanczos steps of two launches against the oracle (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


@pytest.mark.parametrize("clean", [True, False])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_two_launch_steps_vs_oracle(ed, orc, prec, clean, monkeypatch):
    """Ground states and seed chains whose steps run in two launches: E0 within
    1e-10 of the oracle with and without a tolerance that ends the run, the
    vector from the stored basis and from the second run of the chain to 1e-12
    (the same sums), and the first ten coefficients of a seed to 1e-9."""
    H, U, sec = (lattice.square(3, 4) if clean else lattice.disordered_rect(3, 4)), 6.0, (6, 5)
    m = orc.Model(H, [U])
    ed.set_hamiltonian(H, [U])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    Hc = orc.hamiltonian_csr(m, *sec)
    e0, _, _ = orc.lanczos_ground_state(Hc, lattice.splitmix_vector(dim, 0x5EED), 200, want_vector=False)
    r = ed.lanczos_eigh(isec, prec, niter=200, want_vector=True)
    assert abs(r["e0"] - e0) < 1e-10 * abs(e0)
    rt = ed.lanczos_eigh(isec, prec, niter=200, tol=1e-13)
    assert abs(rt["e0"] - e0) < 1e-10 * abs(e0)
    monkeypatch.setenv("EDL_LANCZOS_BASIS", "0")
    r0 = ed.lanczos_eigh(isec, "fp64", niter=120, want_vector=True)
    monkeypatch.delenv("EDL_LANCZOS_BASIS")
    r1 = ed.lanczos_eigh(isec, "fp64", niter=120, want_vector=True)
    assert r0["e0"] == r1["e0"] and np.max(np.abs(r0["gs"] - r1["gs"])) < 1e-12
    monkeypatch.setenv("EDL_BATCHED_KERNELS", "chain")
    seed = np.random.default_rng(1).standard_normal(dim)
    a, b, n2 = ed.tridiag_Hv_sector(isec, seed, 12, "fp64")
    ao, bo, _ = orc.lanczos_tridiag(Hc, seed, 12)
    assert abs(n2 - seed @ seed) < 1e-12 * n2
    np.testing.assert_allclose(a[:10], ao[:10], rtol=1e-9, atol=1e-9)
    np.testing.assert_allclose(b[1:10], bo[1:10], rtol=1e-9, atol=1e-9)
