"""H.psi at the edges of the MFMA scatter's tiles.

Covered points below one tile of 64 and no multiple of 16, spheres wider than
the cell (an atom covers a point more than once), projector counts on both sides
of each K-step count (9, 16, 18, 32 per atom), column counts that fill no group
of 16 or 32, and wave counts on both sides of the point-tile rule.

Reference: the CPU FP64 oracle, tolerances as for the operator's parity tests:
FP64 1e-12, FP32 2e-6 of the largest value.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # n, lmax, nradial, rc, ncomp, k, bands
    (13, 0, 1, 0.5, 1, (0, 0, 0), 1),
    (13, 2, 1, 0.9, 1, (0, 0, 0), 17),
    (12, 2, 1, 2.9, 2, (0.5, 0.25, -0.125), 3),
    (13, 3, 1, 1.4, 1, (0, 0, 0), 33),
    (14, 3, 1, 1.7, 2, (0, 0, 0), 16),
    (12, 2, 2, 2.9, 2, (0.25, 0, 0), 9),
    (13, 3, 2, 0.5, 1, (0, 0, 0), 5),
    (13, 3, 2, 1.4, 2, (0.25, 0.25, 0.25), 65),
    (20, 3, 2, 1.9, 1, (0, 0, 0), 500),
    (20, 2, 1, 1.9, 2, (0.25, 0, 0), 251),
]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,lmax,nradial,rc,ncomp,k,nb", SHAPES)
def test_scatter_at_tile_edges(qm, orc, torch_cuda, n, lmax, nradial, rc, ncomp, k, nb, prec):
    torch = torch_cuda
    s = qm.system.small_system(n=n, L=4.2, natoms=3, lmax=lmax, nradial=nradial, rc=rc, nbands=nb, ncomp=ncomp,
                               k_red=k)
    print(f"case scatter {n}^3 l {lmax} x {nradial} rc {rc} ncomp {ncomp} {nb} bands {prec}", flush=True)
    H = qm.hamiltonian.Hamiltonian(s)
    psi = np.random.default_rng(5).uniform(-0.5, 0.5, (nb * ncomp, s.ng))
    if prec == "f32":
        psi = psi.astype(np.float32).astype(np.float64)
    x = torch.from_numpy(psi).to("cuda", torch.float64 if prec == "f64" else torch.float32)
    y = torch.full_like(x, float("nan"))  # every output element must be written
    H.apply(y, x)
    want = orc.hpsi(s, psi, k=s.kpoints[0])
    tol = 1e-12 if prec == "f64" else 2e-6
    assert np.abs(y.double().cpu().numpy() - want).max() <= tol * np.abs(want).max()
    H.close()
