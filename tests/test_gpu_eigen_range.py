"""qm_sygvd_f64 at the ends of FP64's range.

Matrices with entries of 1e150 and 1e-150 (orders on both sides of the leaf size
and of a tile), and eigenvalues above 2^1023: a power of two is taken off the
tridiagonal matrix before it is solved, and put back.  Tolerances as for the
ordinary sizes: (64 + 8 n) eps of the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.3e-16


def _sygvd(qm, torch, H, a, b, nev):
    w, z, u = H.sygvd(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), nev)
    return w.cpu().numpy(), z.cpu().numpy()


@pytest.mark.parametrize("scale", [1e150, 1e-150])
@pytest.mark.parametrize("n", [15, 17, 63, 130])
def test_sygvd_scaled(qm, torch_cuda, n, scale):
    torch = torch_cuda
    print(f"case sygvd n {n} scale {scale:g}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    rng = np.random.default_rng(n)
    e = rng.standard_normal(n - 1)
    a = np.diag(rng.standard_normal(n)) + np.diag(e, 1) + np.diag(e, -1)
    w, z = _sygvd(qm, torch, H, a * scale, np.eye(n), n)
    tol = (64 + 8 * n) * EPS
    ref = np.linalg.eigvalsh(a)
    assert np.isfinite(w).all() and np.isfinite(z).all()
    assert np.abs(w / scale - ref).max() <= tol * np.abs(ref).max()
    assert np.abs(z.T @ z - np.eye(n)).max() <= tol
    assert np.abs(a @ z - z * (w / scale)).max() <= tol * np.abs(ref).max()
    H.close()


@pytest.mark.parametrize("n", [1, 2, 16, 17, 40])
def test_sygvd_largest_values(qm, torch_cuda, n):
    torch = torch_cuda
    print(f"case sygvd largest n {n}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    d = 1.5e308 * np.linspace(1.0, -1.0, n) if n > 1 else np.array([1.5e308])
    w, z = _sygvd(qm, torch, H, np.diag(d), np.eye(n), n)
    assert np.isfinite(w).all() and np.array_equal(w, np.sort(d))
    assert np.array_equal(np.abs(z), np.eye(n)[:, np.argsort(d)])
    H.close()
