"""The one-launch H x v over column panels, forced wherever the panels fit,
against the oracle (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_one_launch_hxv_vs_oracle(ed, orc, prec, monkeypatch):
    """Natural layout on device vectors and the engine's padded layout (host
    vectors); one and several hopping values, one string of a spin, odd and
    even DimUp, DimUp over 1024; the operator's tolerances (1e-13, 2e-6)."""
    monkeypatch.setenv("EDL_ONE_PASS", "1")
    t = np.float64 if prec == "fp64" else np.float32
    tol = 1e-13 if prec == "fp64" else 2e-6
    rng = np.random.default_rng(9)
    for H, U, sec in [(lattice.ring(8), 4.0, (4, 4)), (lattice.ring(8), 4.0, (8, 4)), (lattice.ring(8), 4.0, (4, 0)),
                      (lattice.ring(7), 3.0, (3, 4)), (lattice.disordered_rect(3, 4), 4.0, (6, 5)),
                      (lattice.square(3, 4), 6.0, (5, 6)), (lattice.ring(13), 4.0, (6, 2))]:
        m = orc.Model(H, [U])
        ed.set_hamiltonian(H, [U])
        isec = ed.sector_index(*sec)
        dim, du, _ = ed.build_sector(isec)
        print(f"one launch {prec} sector {sec} DimUp {du}", flush=True)
        v = rng.standard_normal(dim).astype(t)
        ref = orc.matvec(m, *sec, v.astype(np.float64), nthreads=8).real
        src, dst = ed.alloc(v.nbytes), ed.alloc(v.nbytes)
        ed._ck(ed.lib.edl_copy_h2d(ed.h, src, v.ctypes.data, v.nbytes))
        ed.hxv_device(isec, prec, src, dst)
        out = ed.copy_to_host(dst, np.empty_like(v))
        assert np.max(np.abs(out - ref)) < tol * max(np.max(np.abs(ref)), 1e-300)
        assert ed.bench_passes(isec, prec, 1)[2]["two_pass"] == 0
        host = ed.direct_matvec(isec, v.astype(np.float64), prec)
        assert np.max(np.abs(host - ref)) < tol * max(np.max(np.abs(ref)), 1e-300)
