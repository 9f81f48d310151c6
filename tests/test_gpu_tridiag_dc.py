"""Divide and conquer of the subspace eigensolve (csrc/tridiag_dc.hip) through
qm_sygvd_f64 / qm_hegvd_z64 with B = 1, on tridiagonal matrices where it can go
wrong: orders around the leaf size and around tiles, everything deflating
(diagonal, zero couplings, Kronecker-like blocks), chains of close poles (glued
Wilkinson), graded and tiny couplings, all and one wanted vector.

Backward error: eigenvalues against numpy, residuals and orthogonality within
(64 + 8 n) eps (times the norm): the reduction, the merges (L levels of O(n eps))
and the back-transformation each contribute a small multiple of n eps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.3e-16


def _matrix(kind, n, rng):
    if kind == "toeplitz":
        return np.full(n, 2.0), np.full(n - 1, -1.0)
    if kind == "diagonal":
        return rng.standard_normal(n), np.zeros(n - 1)
    if kind == "identity":
        return np.ones(n), np.zeros(n - 1)
    if kind == "zero":
        return np.zeros(n), np.zeros(n - 1)
    if kind == "wilkinson":
        return np.abs(np.arange(n) - (n - 1) / 2.0), np.ones(n - 1)
    if kind == "glued":
        d, e = np.abs(np.arange(n) % 21 - 10.0), np.ones(n - 1)
        e[20::21] = 1e-10
        return d, e
    if kind == "graded":
        return 10.0 ** (-12.0 * np.arange(n) / n), 10.0 ** (-12.0 * np.arange(1, n) / n) * 0.5
    if kind == "blocks":
        d, e = np.tile([1.0, 2.0, 1.0, 2.0], n)[:n], np.full(n - 1, 0.5)
        e[3::4] = 0.0
        return d, e
    if kind == "large":
        return rng.standard_normal(n) * 1e150, rng.standard_normal(n - 1) * 1e150
    return rng.standard_normal(n), rng.standard_normal(n - 1)


KINDS = ["random", "toeplitz", "diagonal", "identity", "zero", "wilkinson", "glued", "graded", "blocks"]


def _check(a, w, z, tag):
    n, nev = a.shape[0], z.shape[1]
    tol = (64 + 8 * n) * EPS
    ref = np.linalg.eigvalsh(a)
    nrm = max(np.abs(ref).max(), 1e-300)
    assert np.isfinite(w).all() and np.isfinite(z).all(), tag
    assert np.abs(w - ref).max() <= tol * nrm, (tag, np.abs(w - ref).max() / nrm)
    assert np.abs(z.conj().T @ z - np.eye(nev)).max() <= tol, (tag, np.abs(z.conj().T @ z - np.eye(nev)).max())
    assert np.abs(a @ z - z * w[:nev]).max() <= tol * nrm, tag


@pytest.mark.parametrize("kind", KINDS)
def test_tridiag_dc_kinds(qm, torch_cuda, kind):
    torch = torch_cuda
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    rng = np.random.default_rng(11)
    for n in (2, 15, 16, 17, 32, 33, 48, 63, 65, 129, 250):
        print(f"case tridiag {kind} n {n}", flush=True)
        d, e = _matrix(kind, n, rng)
        a = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
        w, z, _ = H.sygvd(torch.from_numpy(a).cuda(), torch.eye(n, dtype=torch.float64, device="cuda"))
        _check(a, w.cpu().numpy(), z.cpu().numpy(), (kind, n))
    H.close()


@pytest.mark.parametrize("n,nev", [(1, 1), (16, 3), (17, 1), (100, 15), (100, 16), (384, 128), (513, 513), (1024, 40)])
def test_tridiag_dc_wanted(qm, torch_cuda, n, nev):
    """Dense random real and complex matrices, nev vectors."""
    torch = torch_cuda
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    rng = np.random.default_rng(n)
    for cplx in (False, True):
        print(f"case tridiag wanted n {n} nev {nev} complex {cplx}", flush=True)
        a = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)
        a = 0.5 * (a + a.conj().T)
        eye = torch.eye(n, dtype=torch.complex128 if cplx else torch.float64, device="cuda")
        w, z, _ = (H.hegvd if cplx else H.sygvd)(torch.from_numpy(a).cuda(), eye, nev=nev)
        _check(a, w.cpu().numpy(), z.cpu().numpy()[:, :nev], (n, nev, cplx))
    H.close()
