"""H x v on device vectors in the reference's own layout (column stride
DimUp), where the vector-gather down pass reads row segments of any
alignment: odd and even DimUp, columns of fewer rows than a lane takes,
buffers off by one element, against the oracle (GPU)."""
import numpy as np
import pytest

from ed_lattice_amd import EDLattice, lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("R", [16, 64, 128, 256])
def test_hxv_natural_layout_vector_gathers_vs_oracle(orc, R, prec, monkeypatch):
    """Tolerances as for the host-vector operator: rounding of a sum of the
    diagonal and at most 33 hops, 1e-13 in fp64 and 2e-6 in fp32."""
    rows = min(R, 128) if prec == "fp64" else R  # 256-row panels are fp32 only
    tail = f"{rows},256,1,2,2,1,8,1"
    monkeypatch.setenv("EDL_TWO_PASS_CFG_F32", "3,1024,256," + tail)
    monkeypatch.setenv("EDL_TWO_PASS_CFG_F64", "1,512,512," + tail)
    t = np.float64 if prec == "fp64" else np.float32
    rng = np.random.default_rng(5)
    with EDLattice(0) as ed:
        for H, U, sec in [(lattice.ring(7), 3.0, (3, 3)), (lattice.ring(8), 4.0, (1, 7)), (lattice.ring(8), 4.0, (8, 4)),
                          (lattice.ring(3), 2.0, (1, 1)), (lattice.disordered_rect(3, 3), 4.0, (4, 5)),
                          (lattice.square(3, 4), 6.0, (5, 6))]:
            m = orc.Model(H, [U])
            ed.set_hamiltonian(H, [U])
            isec = ed.sector_index(*sec)
            dim, du, _ = ed.build_sector(isec)
            v = rng.standard_normal(dim).astype(t)
            ref = orc.matvec(m, *sec, v.astype(np.float64), nthreads=8).real
            for shift in (0, 1):  # elements
                print(f"natural layout {prec} R {rows} sector {sec} DimUp {du} shift {shift}", flush=True)
                n = (dim + 2) * v.itemsize
                src, dst = ed.alloc(n), ed.alloc(n)
                edge = np.full(dim + 2, -7.0, t)  # guard elements around the output
                ed._ck(ed.lib.edl_copy_h2d(ed.h, dst, edge.ctypes.data, n))
                ed._ck(ed.lib.edl_copy_h2d(ed.h, src + shift * v.itemsize, v.ctypes.data, v.nbytes))
                ed.hxv_device(isec, prec, src + shift * v.itemsize, dst + shift * v.itemsize)
                out = ed.copy_to_host(dst, edge)
                tol = 1e-13 if prec == "fp64" else 2e-6
                assert np.max(np.abs(out[shift:shift + dim] - ref)) < tol * np.max(np.abs(ref))
                assert np.all(out[:shift] == -7.0) and np.all(out[shift + dim:] == -7.0)
