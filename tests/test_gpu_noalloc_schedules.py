"""Schedules of the allocation-free operator call: what earlier calls on the
sector tuned, for any of the layouts it ran on (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, _lib, lattice

pytestmark = pytest.mark.gpu

# sectors of lattices no other test runs (the schedules are the process's):
# (lattice, sector, the call before, where the schedule comes from)
CASES = [(lattice.ring(11), (5, 3), "solve", "the chain"), (lattice.ring(11), (3, 5), "host", "the padded stride"),
         (lattice.ring(11), (4, 6), "device", "this stride"), (lattice.ring(11), (2, 2), "solve", "none, one launch"),
         (lattice.ring(11), (5, 6), None, "none, one launch"), (lattice.ring(13), (7, 6), None, "none, two passes"),
         (lattice.disordered_rect(1, 11), (6, 4), "solve", "the chain")]


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_noalloc_schedule(orc, k, prec, monkeypatch, capfd):
    """Where the schedule comes from, and the product against the oracle (the
    operator's 1e-13 and 2e-6)."""
    H, sec, before, want = CASES[k]
    if k == 5 and prec == "fp32":
        want = "none, one launch"  # 12 MB: within the one-launch form's size
    t = np.float64 if prec == "fp64" else np.float32
    m = orc.Model(H, [4.0])
    monkeypatch.setenv("EDL_VERBOSE", "1")
    with EDLattice(0) as ed:
        ed.set_hamiltonian(H, [4.0])
        isec = ed.sector_index(*sec)
        dim, du, _ = ed.build_sector(isec)
        assert du % 32 != 0  # the padded stride is another
        v = np.random.default_rng(k).standard_normal(dim).astype(t)
        src, dst = ed.alloc(v.nbytes), ed.alloc(v.nbytes)
        ed._ck(ed.lib.edl_copy_h2d(ed.h, src, v.ctypes.data, v.nbytes))
        if before == "solve":
            ed.lanczos_eigh(isec, prec, niter=10)
        elif before == "host":
            ed.direct_matvec(isec, v.astype(np.float64), prec)
        elif before == "device":
            ed.hxv_device(isec, prec, src, dst)
        capfd.readouterr()
        ed._ck(ed.lib.edl_hxv_noalloc(ed.h, isec, getattr(_lib, "EDL_" + prec.upper()), src, dst))
        assert f"noalloc schedule tuned for: {want}\n" in capfd.readouterr().err
        out = ed.copy_to_host(dst, np.empty_like(v))
    ref = orc.matvec(m, *sec, v.astype(np.float64), nthreads=8).real
    assert np.max(np.abs(out - ref)) < (1e-13 if prec == "fp64" else 2e-6) * np.max(np.abs(ref))
