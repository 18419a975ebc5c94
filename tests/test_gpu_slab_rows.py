"""Down tiles of the batched chains with 16 bytes of rows a lane (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


# slab heights on both sides of 16 bytes a column; 1, 9, 84 and 126 up strings
# (one row, remainders of 32 and of every height), fewer columns than a wave
# and more; table words and two hops to a word
@pytest.mark.parametrize("rows", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("H,sec", [(lattice.ring(6), (0, 3)), (lattice.ring(9), (1, 4)), (lattice.square(3, 3), (6, 2)),
                                   (lattice.disordered_rect(3, 3), (5, 4))])
def test_slab_rows_vs_oracle(ed, orc, H, sec, prec, rows, monkeypatch):
    """Coefficients of a random seed against the oracle's recurrence: the first
    ten, where rounding is not yet amplified (fp64 1e-9; fp32 vectors and
    products 1e-4, ten steps of 2e-6 each)."""
    monkeypatch.setenv("EDL_BATCHED_KERNELS", "tiles")
    monkeypatch.setenv("EDL_BATCHED_SLAB_ROWS", str(rows))
    m = orc.Model(H, [4.0])
    ed.set_hamiltonian(H, [4.0])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    print(f"slab rows {rows} {prec} sector {sec} dim {dim}", flush=True)
    seed = np.random.default_rng(rows).standard_normal(dim)
    a, b, n2 = ed.tridiag_Hv_sector(isec, seed, 12, prec)
    Hc = orc.hamiltonian_csr(m, *sec)
    ao, bo, _ = orc.lanczos_tridiag(Hc, seed, 12)
    tol = 1e-9 if prec == "fp64" else 1e-4
    assert abs(n2 - seed @ seed) < 1e-12 * n2
    n = min(10, len(ao), max(1, dim // 2))
    if dim < 100:  # the recurrence ends, or runs on rounding, after as many steps as H has levels
        n = min(n, len(np.unique(np.round(np.linalg.eigvalsh(Hc.toarray()), 9))) - 1)
    np.testing.assert_allclose(a[:n], ao[:n], rtol=tol, atol=tol)
    np.testing.assert_allclose(b[1:n], bo[1:n], rtol=tol, atol=tol)
