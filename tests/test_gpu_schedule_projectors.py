"""The tuned form of a full H.psi apply follows the projector set: a set with more
than twice, or less than half, the voxels times table rows that it was tuned with
is tuned again; a moved set of the same size keeps it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_full_apply_retuned_for_another_set(qm, orc, torch_cuda):
    torch = torch_cuda

    def system(natoms, rc, seed):
        return qm.system.small_system(n=24, L=6.0, natoms=natoms, rc=rc, nbands=6, seed=seed)

    small, moved, heavy = system(1, 0.9, 1), system(1, 0.9, 2), system(6, 1.8, 3)
    H = qm.hamiltonian.Hamiltonian(small)
    psi = np.random.default_rng(5).uniform(-0.5, 0.5, (6, small.ng))
    x = torch.from_numpy(psi).cuda()

    def check(s):
        H.set_vloc(s.vloc)
        y = torch.empty_like(x)
        H.apply(y, x)
        want = orc.hpsi(s, psi, k=s.kpoints[0])
        assert np.abs(y.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()

    print("case schedule small", flush=True)
    assert H.stencil_choice(64, 6, full=True) == -1
    check(small)
    assert H.stencil_choice(64, 6, full=True) >= 0
    H.set_projectors(moved)
    assert H.stencil_choice(64, 6, full=True) >= 0
    check(moved)
    print("case schedule heavy", flush=True)
    H.set_projectors(heavy)
    assert H.stencil_choice(64, 6, full=True) == -1
    assert H.stencil_choice(64, 6) >= 0  # the local shape does not depend on the set
    check(heavy)
    assert H.stencil_choice(64, 6, full=True) >= 0
    print("case schedule back", flush=True)
    H.set_projectors(small)
    assert H.stencil_choice(64, 6, full=True) == -1
    check(small)
    H.close()
