"""FP32 nonlocal energy and forces: the sums over a sphere are FP64.

With table values that FP32 holds exactly and no Bloch phase, every input is the
same number in either precision and a product of two FP32 values is exact in
FP64, so the FP32 entry point differs from the FP64 one by the order of FP64 sums
only: at most (number of voxels) 2^-52 of the sums of magnitudes, below 1e-10 of
the largest component here.  Bands of one sign make the gradient sums cancel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("one_sign", [False, True])
@pytest.mark.parametrize("lmax,nradial,rc,ncomp,nb", [(1, 1, 1.5, 1, 33), (2, 1, 2.5, 1, 40), (2, 1, 2.0, 2, 9),
                                                      (3, 1, 2.2, 2, 17), (3, 2, 2.5, 2, 24)])
def test_f32_forces_sum_in_fp64(qm, torch_cuda, lmax, nradial, rc, ncomp, nb, one_sign):
    torch = torch_cuda
    print(f"case f32 forces l {lmax} x {nradial} rc {rc} ncomp {ncomp} {nb} bands one sign {one_sign}", flush=True)
    s = qm.system.small_system(n=32, L=6.0, natoms=4, lmax=lmax, nradial=nradial, rc=rc, nbands=nb, ncomp=ncomp)
    s.table = s.table.astype(np.float32).astype(np.float64)
    s.dtable = s.dtable.astype(np.float32).astype(np.float64)
    H = qm.hamiltonian.Hamiltonian(s)
    g = torch.Generator(device="cuda").manual_seed(nb)
    x = torch.rand((nb * ncomp, s.ng), device="cuda", generator=g) + (0.5 if one_sign else -0.5)
    occ = np.linspace(2.0, 0.1, nb)
    e32, f32 = H.nonlocal_forces(x, occ)
    e64, f64 = H.nonlocal_forces(x.double(), occ)
    scale = max(abs(e64), np.abs(f64).max())
    assert abs(e32 - e64) <= 1e-10 * scale
    assert np.abs(f32 - f64).max() <= 1e-10 * scale
    H.close()
