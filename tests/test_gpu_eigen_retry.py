"""A tridiagonal divide and conquer that runs out of steps is redone by rocSOLVER.

The bound is forced from the host (0: every leaf and root runs out at once; 2: some
do), every kernel still ends.  qm_sygvd_f64 and qm_hegvd_z64 then give LAPACK's
results all the same, and qm_lobpcg_solve the energies of an undisturbed run, with
its redone solves counted.  Tolerances as for the same entry points' LAPACK parity
tests (1e-11 of the scale) and 1e-10 relative for 6 LOBPCG iterations, whose
subspace vectors come from another algorithm."""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu


@pytest.fixture
def limit(qm, request):
    qm.hamiltonian.dc_step_limit(request.param)
    yield request.param
    qm.hamiltonian.dc_step_limit(None)


@pytest.mark.parametrize("limit", [0, 2], indirect=True)
@pytest.mark.parametrize("n,nev", [(16, 5), (17, 17), (90, 30), (384, 128)])
@pytest.mark.parametrize("cplx", [False, True])
def test_eigensolves_redone(qm, torch_cuda, limit, n, nev, cplx):
    torch = torch_cuda
    print(f"case redone n {n} nev {nev} complex {cplx} limit {limit}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    rng = np.random.default_rng(n)

    def mat():
        return rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)

    a, b = mat(), mat()
    a, b = 0.5 * (a + a.conj().T), b @ b.conj().T / n + np.eye(n)
    w, z, _ = (H.hegvd if cplx else H.sygvd)(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), nev)
    w, z = w.cpu().numpy(), z.cpu().numpy()
    scale = max(1.0, np.abs(a).max() * n)
    assert np.abs(w - scipy.linalg.eigh(a, b, eigvals_only=True)).max() <= 1e-11 * scale
    assert np.abs(a @ z - (b @ z) * w[:nev]).max() <= 1e-11 * scale
    assert np.abs(z.conj().T @ b @ z - np.eye(nev)).max() <= 1e-11 * n
    H.close()


@pytest.mark.parametrize("ncomp,k", [(1, (0.0, 0.0, 0.0)), (2, (0.25, 0.25, 0.0))])
def test_lobpcg_redone(qm, torch_cuda, ncomp, k):
    torch = torch_cuda
    print(f"case lobpcg redone ncomp {ncomp}", flush=True)
    s = qm.system.small_system(n=16, L=4.0, natoms=2, nbands=10, ncomp=ncomp, k_red=k)
    H = qm.hamiltonian.Hamiltonian(s)
    x0 = torch.from_numpy(s.initial_bands()).cuda()
    got = []
    try:
        for limit in (None, 0):
            qm.hamiltonian.dc_step_limit(limit)
            solver = qm.lobpcg.LOBPCG(H, s.nbands, precision=64)
            x = x0.clone()
            ev, rn = solver.solve(x, 6, first_time=True)
            retries = solver.eigen_retries()[0]
            print(f"limit {limit}: redone {retries}, fallbacks {solver.lib.qm_lobpcg_fallbacks(solver.h)}", flush=True)
            assert solver.lib.qm_lobpcg_fallbacks(solver.h) == 0
            assert retries == (0 if limit is None else 6)
            got.append((ev, rn))
            solver.close()
    finally:
        qm.hamiltonian.dc_step_limit(None)
    (e0, r0), (e1, r1) = got
    assert np.abs(e0 - e1).max() <= 1e-10 * np.abs(e0).max()
    H.close()
