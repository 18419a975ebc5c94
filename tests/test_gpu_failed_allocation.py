"""A call after one that failed for memory (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu


def test_call_after_failed_allocation(orc):
    """More than the device has is an error; the next call runs and is right (the
    operator's 1e-13)."""
    H = lattice.ring(8)
    m = orc.Model(H, [4.0])
    with EDLattice(0) as ed:
        ed.set_hamiltonian(H, [4.0])
        isec = ed.sector_index(4, 3)
        dim, _, _ = ed.build_sector(isec)
        ed.lanczos_eigh(isec, "fp64", niter=20)  # buffers kept, given back by the failing call
        with pytest.raises(Exception, match="memory"):
            ed.alloc(1 << 45)
        v = np.random.default_rng(1).standard_normal(dim)
        hv = ed.direct_matvec(isec, v, "fp64")
        ref = orc.matvec(m, 4, 3, v).real
        assert np.max(np.abs(hv - ref)) < 1e-13 * np.max(np.abs(ref))
        r = ed.lanczos_eigh(isec, "fp64", niter=20)
        assert r["nsteps"] == 20
