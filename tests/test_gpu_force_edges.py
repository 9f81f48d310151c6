"""Nonlocal forces and band density at the edges of their kernels' tiles.

Forces: projector counts on both sides of each MFMA row-tile count (1, 4, 9,
16, 18, 32 per atom: 1, 1, 3, 4, 8, 8 tiles of 16 rows for the four tables),
spheres shorter and longer than a 64-voxel sub-chunk and a 512-voxel work item,
band counts that fill no 16-column group or need a second band slice (128).
Density: band counts that are no multiple of 4 and beyond one launch's 256.

Reference: the CPU FP64 oracle.  Tolerances as for the parity tests of the same
entry points: FP64 <= 1e-12 of the largest component (sums of a few thousand
products in another order), FP32 <= 1e-5 for forces; densities sum exact FP64
squares of the inputs, so <= 1e-13 in either precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # lmax, nradial, rc, ncomp, k, bands
    (0, 1, 0.6, 1, (0, 0, 0), 1),
    (0, 1, 1.4, 2, (0.25, 0, 0), 17),
    (1, 1, 0.9, 2, (0, 0, 0), 8),
    (2, 1, 1.9, 1, (0, 0, 0), 130),
    (2, 1, 1.2, 2, (0.5, 0.25, -0.125), 9),
    (3, 1, 1.4, 1, (0, 0, 0), 15),
    (2, 2, 1.4, 2, (0.25, 0.25, 0.25), 65),
    (3, 2, 1.9, 2, (0.25, 0, 0), 129),
    (3, 2, 1.0, 1, (0, 0, 0), 16),
]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("lmax,nradial,rc,ncomp,k,nb", SHAPES)
def test_forces_at_tile_edges(qm, orc, torch_cuda, lmax, nradial, rc, ncomp, k, nb, prec):
    torch = torch_cuda
    s = qm.system.small_system(n=13, L=4.2, natoms=3, lmax=lmax, nradial=nradial, rc=rc, nbands=nb, ncomp=ncomp,
                               k_red=k)
    print(f"case forces l {lmax} x {nradial} rc {rc} ncomp {ncomp} {nb} bands {prec}", flush=True)
    H = qm.hamiltonian.Hamiltonian(s)
    rng = np.random.default_rng(11)
    psi = rng.uniform(-0.5, 0.5, (nb * ncomp, s.ng))
    if prec == "f32":
        psi = psi.astype(np.float32).astype(np.float64)
    occ = rng.uniform(0.0, 2.0, nb)
    x = torch.from_numpy(psi).to("cuda", torch.float64 if prec == "f64" else torch.float32)
    e, f = H.nonlocal_forces(x, occ)
    e0, f0 = orc.nonlocal_forces(s, psi, occ, k=s.kpoints[0])
    tol = 1e-12 if prec == "f64" else 1e-5
    assert abs(e - e0) <= tol * max(abs(e0), np.abs(f0).max())
    assert np.abs(f - f0).max() <= tol * max(np.abs(f0).max(), abs(e0))
    H.close()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("ncomp,nb", [(1, 1), (1, 6), (2, 3), (1, 257), (2, 260)])
def test_density_band_counts(qm, orc, torch_cuda, ncomp, nb, prec):
    torch = torch_cuda
    s = qm.system.small_system(n=11, L=4.0, natoms=1, nbands=nb, ncomp=ncomp)
    print(f"case density ncomp {ncomp} {nb} bands {prec}", flush=True)
    H = qm.hamiltonian.Hamiltonian(s)
    rng = np.random.default_rng(3)
    psi = rng.uniform(-0.5, 0.5, (nb * ncomp, s.ng))
    if prec == "f32":
        psi = psi.astype(np.float32).astype(np.float64)
    occ = rng.uniform(0.0, 2.0, nb)
    x = torch.from_numpy(psi).to("cuda", torch.float64 if prec == "f64" else torch.float32)
    rho = H.band_density(x, occ).cpu().numpy()
    want = orc.band_density(s, psi, occ)
    assert np.abs(rho - want).max() <= 1e-13 * np.abs(want).max()
    H.close()
