"""Which chains run steps of two launches, and that both forms of the step agree
on one schedule (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu

# vector-gather down pass in the locality order of columns, which pins the chain's
# down pass too (32, 64 and 128 rows, more and fewer blocks)
PINS = ["1,512,256,64,256,64,2,4,1,16,1,0,0,1", "1,512,256,128,256,17,1,2,1,16,1,0,0,1",
        "1,1024,256,32,512,300,2,2,1,16,1,0,0,1"]


@pytest.fixture(scope="module")
def ed():
    e = EDLattice(0)
    yield e
    e.close()


def _route(capfd):
    return [x.split(": ")[1] for x in capfd.readouterr().err.splitlines() if x.startswith("[edl] chain steps: ")]


@pytest.mark.parametrize("clean", [True, False])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("pin", PINS)
def test_both_forms_of_a_step(ed, orc, pin, prec, clean, monkeypatch, capfd):
    """The same kernels' sums, added up in another order: ten coefficients of the
    chain to 1e-9 (fp32 four to 1e-4), E0 against the oracle (1e-10, fp32 1e-5)."""
    H, sec = (lattice.square(3, 4) if clean else lattice.disordered_rect(3, 4)), (5, 5)
    m = orc.Model(H, [6.0])
    ed.set_hamiltonian(H, [6.0])
    isec = ed.sector_index(*sec)
    dim, _, _ = ed.build_sector(isec)
    monkeypatch.setenv("EDL_TWO_PASS_CFG_" + ("F64" if prec == "fp64" else "F32"), pin)
    monkeypatch.setenv("EDL_VERBOSE", "1")
    r = []
    for two, name in (("1", "two launches"), ("0", "more than two launches")):
        monkeypatch.setenv("EDL_TWO_LAUNCH", two)
        capfd.readouterr()
        r.append(ed.lanczos_eigh(isec, prec, niter=200, seed=3))
        assert _route(capfd) == [name]
    Hc = orc.hamiltonian_csr(m, *sec)
    e0, _, _ = orc.lanczos_ground_state(Hc, lattice.splitmix_vector(dim, 3), 200, want_vector=False)
    n, tol, te = (10, 1e-9, 1e-10) if prec == "fp64" else (4, 1e-4, 1e-5)
    for key in ("alpha", "beta"):
        np.testing.assert_allclose(r[0][key][:n], r[1][key][:n], rtol=tol, atol=tol)
    for x in r:
        assert abs(x["e0"] - e0) < te * abs(e0)


def test_forced_two_launch_steps_of_a_segmented_sector(ed, monkeypatch):
    """No such form: an error, not another route."""
    H = lattice.ring(10)
    ed.set_hamiltonian(H, [4.0])
    isec = ed.sector_index(5, 5)
    ed.build_sector(isec)
    monkeypatch.setenv("EDL_UP_SEGMENT_ROWS", "100")
    monkeypatch.setenv("EDL_TWO_LAUNCH", "1")
    with pytest.raises(Exception, match="EDL_TWO_LAUNCH"):
        ed.lanczos_eigh(isec, "fp64", niter=20)
    monkeypatch.delenv("EDL_TWO_LAUNCH")
    ed.lanczos_eigh(isec, "fp64", niter=20)
