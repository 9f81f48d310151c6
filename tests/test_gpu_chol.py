"""Blocked Cholesky factor with its inverse (csrc/chol.hip) through qm_sygvd_f64
and qm_hegvd_z64 at orders around its 32 x 32 blocks, and the order of the first
failing minor wherever it falls in a block.

U against numpy within 8 n eps cond-free (B has condition < 20, so U is computed
to a few n eps of its norm); A z = l B z residuals and B-orthonormality within
1e-11 as in test_gpu_eigen.py."""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu


def _pair(n, seed, cplx):
    rng = np.random.default_rng(seed)
    a, g = rng.standard_normal((2, n, n))
    if cplx:
        a, g = a + 1j * rng.standard_normal((n, n)), g + 1j * rng.standard_normal((n, n))
    g = g * (0.3 / np.sqrt(n))
    b = np.eye(n) + g @ g.conj().T
    return 0.5 * (a + a.conj().T), 0.5 * (b + b.conj().T)


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
def test_chol_orders(qm, torch_cuda, cplx):
    torch = torch_cuda
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    for n in (1, 2, 31, 32, 33, 63, 64, 65, 96, 97, 135, 384, 1000):
        print(f"case Cholesky n {n} complex {cplx}", flush=True)
        a, b = _pair(n, n, cplx)
        # only the upper triangles may be read
        au, bu = a.copy(), b.copy()
        low = np.tril_indices(n, -1)
        au[low] = bu[low] = np.nan
        nev = max(1, n // 3)
        w, z, u = (H.hegvd if cplx else H.sygvd)(torch.from_numpy(au).cuda(), torch.from_numpy(bu).cuda(), nev)
        w, z, u = w.cpu().numpy(), z.cpu().numpy()[:, :nev], np.triu(u.cpu().numpy())
        ref = np.linalg.cholesky(b).conj().T
        assert np.abs(u - ref).max() <= 8 * (n + 8) * 2.3e-16 * np.abs(ref).max(), n
        scale = max(1.0, np.abs(a).max() * n)
        assert np.abs(w - scipy.linalg.eigh(a, b, eigvals_only=True)).max() <= 1e-11 * scale, n
        assert np.abs(a @ z - (b @ z) * w[:nev]).max() <= 1e-11 * scale, n
        assert np.abs(z.conj().T @ b @ z - np.eye(nev)).max() <= 1e-11 * n, n
    H.close()


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("n,bad", [(1, 0), (33, 0), (33, 31), (33, 32), (100, 63), (100, 64), (100, 99)])
def test_chol_failing_minor(qm, torch_cuda, n, bad, cplx):
    torch = torch_cuda
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    print(f"case Cholesky failing minor n {n} at {bad} complex {cplx}", flush=True)
    a, b = _pair(n, n + bad, cplx)
    b[bad, bad] = -2.0
    if bad > 2:
        b[bad, bad] = np.nan if bad == 63 else -2.0
    with pytest.raises(qm._lib.QMError) as e:
        (H.hegvd if cplx else H.sygvd)(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), 1)
    assert f"leading minor {bad + 1})" in str(e.value)
    H.close()
