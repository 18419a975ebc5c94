"""Seeds of a batched group built by one launch (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


# one string of a spin in a target, a stride of many padding rows, one block and
# several blocks a seed, target sectors of unlike sizes in one group
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("H,sec", [(lattice.ring(6), (1, 5)), (lattice.disordered_rect(2, 4), (4, 3)),
                                   (lattice.square(3, 3), (5, 2)), (lattice.ring(10), (5, 4))])
def test_seed_group_norms_and_groups(ed, H, sec, prec, monkeypatch):
    """Seed norms against the state's densities and spin correlations (1e-12:
    sums of at most 6e4 squares in fp64), with the same bits whether a seed is
    built in the group or by itself (the coefficients' last bits follow the tile
    shapes, which are tuned for the number of chains)."""
    monkeypatch.setenv("EDL_BATCHED_KERNELS", "tiles")
    ed.set_hamiltonian(H, [4.0])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    print(f"seed group {prec} sector {sec} dim {dim}", flush=True)
    ed.lanczos_eigh(isec, "fp64", niter=100)
    o, sz2 = ed.observables(), ed.correlations()["sz2"]
    seeds, want = [], []
    for i in (1, 3, H.shape[1]):
        seeds += [("cdg", 1, i, 0), ("c", 1, i, 0), ("cdg", 2, i, 0), ("c", 2, i, 0), ("sz", 1, i, 0)]
        want += [1 - o["dens_up"][i - 1], o["dens_up"][i - 1], 1 - o["dens_dw"][i - 1], o["dens_dw"][i - 1],
                 sz2[i - 1, i - 1]]
    seeds += [("sz", 1, 1, 2), ("j", 0, 1, 0)]
    r = ed.tridiag_batched(seeds, 6, prec)
    np.testing.assert_allclose(r["norm2"][:15], want, rtol=0, atol=1e-12)
    pair = sz2[0, 0] + sz2[1, 1] + 2 * sz2[0, 1]
    np.testing.assert_allclose(r["norm2"][15], pair, rtol=0, atol=1e-12)
    for g in (1, 4):
        r1 = ed.tridiag_batched(seeds, 6, prec, group=g)
        np.testing.assert_array_equal(r["norm2"], r1["norm2"])
        np.testing.assert_array_equal(r["nsteps"], r1["nsteps"])
