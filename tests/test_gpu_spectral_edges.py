"""Edges of the spectral kinetic kernels (csrc/spectral.hip): every radix (2, 3,
4, 5, 7, 8, 11, 13) as first, middle and last stage, an axis of one stage, odd
nz and a plane that no tile divides for real bands, odd band counts, planes in
the 512- and 1024-thread workgroups, and the grids that take the library
transforms instead (a prime factor of 17; a plane larger than the LDS).

Against the FP64 numpy oracle; tolerances as in test_gpu_fft.py: 1e-12 (FP64)
and 2e-6 (FP32) relative, max-norm."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(4, 4, 4), (8, 4, 5), (26, 22, 14), (15, 21, 35), (39, 33, 9), (13, 11, 7), (64, 12, 72), (90, 100, 10),
         (96, 96, 6), (34, 16, 8), (128, 110, 8)]


def _sys(qm, grid, ncomp):
    k = np.array([[0.25, 0.0, -0.4]]) if ncomp == 2 else np.zeros((1, 3))
    return qm.system.System("edge", *grid, tuple(0.25 * n for n in grid), np.array([[0.5, 0.5, 0.5]]),
                            np.array([0], np.int32), np.array([0.45]), 3, ncomp, k, 31).build()


@pytest.mark.parametrize("ncomp", [1, 2])
@pytest.mark.parametrize("grid", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_spectral_edges(qm, orc, torch_cuda, grid, ncomp):
    torch = torch_cuda
    s = _sys(qm, grid, ncomp)
    H = qm.hamiltonian.Hamiltonian(s)
    H.set_kinetic("fft")
    psi = s.initial_bands()
    for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 2e-6)):
        print(f"case spectral {grid} ncomp {ncomp} {dtype}", flush=True)
        x = torch.from_numpy(psi).to("cuda", dtype)
        y = torch.full_like(x, float("nan"))
        H.apply(y, x, part="local")
        torch.cuda.synchronize()
        want = orc.hpsi_fft(s, x.double().cpu().numpy(), k=s.kpoints[0], nonlocal_=False)
        err = float(np.abs(y.double().cpu().numpy() - want).max() / np.abs(want).max())
        assert err <= tol, (grid, ncomp, dtype, err)
    H.close()


@pytest.mark.parametrize("grid", [(12, 10, 14), (13, 8, 22), (34, 8, 6)], ids=["small radices", "11 and 13", "library"])
def test_spectral_step_edges(qm, torch_cuda, grid):
    """psi <- e^{-i dt |G + k|^2 / 2} psi in place against numpy's FFT in FP64."""
    torch = torch_cuda
    s = _sys(qm, grid, 2)
    H = qm.hamiltonian.Hamiltonian(s)
    psi, dt, k = s.initial_bands(), 0.13, s.kpoints[0]
    g2 = 0.0
    for ax, (n, q) in enumerate(zip(grid, k)):
        i = np.arange(n)
        g = np.where(2 * i > n, i - n, i) * 2 * np.pi / (0.25 * n) + q
        g2 = g2 + (g * g).reshape([-1 if 2 - ax == d else 1 for d in range(3)])
    z = (psi[0::2] + 1j * psi[1::2]).reshape(-1, grid[2], grid[1], grid[0])
    for dtype, name, tol in ((torch.float64, "f64", 1e-12), (torch.float32, "f32", 2e-6)):
        print(f"case spectral step {grid} {name}", flush=True)
        x = torch.from_numpy(psi).to("cuda", dtype)
        fn = getattr(H.lib, f"qm_td_kinetic_fft_{name}")
        assert fn(H.ctx, ctypes.c_void_p(x.data_ptr()), s.nbands, 0, ctypes.c_double(dt),
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
        want = np.fft.ifftn(np.exp(-0.5j * dt * g2) * np.fft.fftn(z, axes=(1, 2, 3)), axes=(1, 2, 3))
        got = x.double().cpu().numpy()
        got = (got[0::2] + 1j * got[1::2]).reshape(want.shape)
        err = float(np.abs(got - want).max() / np.abs(want).max())
        assert err <= tol, (grid, name, err)
    H.close()


@pytest.mark.parametrize("grid", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_poisson_edges(qm, torch_cuda, grid):
    """V_H = IFFT(4 pi / |G|^2 FFT rho) without G = 0 against numpy's FFT, 1e-12 relative."""
    torch = torch_cuda
    s = _sys(qm, grid, 1)
    H = qm.hamiltonian.Hamiltonian(s)
    print(f"case Poisson {grid}", flush=True)
    rho = np.random.default_rng(7).uniform(0.1, 1.0, s.ng)
    g2 = 0.0
    for ax, n in enumerate(grid):
        g = np.fft.fftfreq(n, 1.0 / n) * 2 * np.pi / (0.25 * n)
        g2 = g2 + (g * g).reshape([-1 if 2 - ax == d else 1 for d in range(3)])
    f = np.fft.fftn(rho.reshape(grid[2], grid[1], grid[0]))
    g2[0, 0, 0] = 1.0
    f *= 4 * np.pi / g2
    f[0, 0, 0] = 0.0
    want = np.fft.ifftn(f).real.reshape(-1)
    got = qm.scf.hartree(H, torch.from_numpy(rho).cuda()).cpu().numpy()
    assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
    H.close()
