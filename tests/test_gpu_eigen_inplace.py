"""qm_sygvd_f64 and qm_hegvd_z64 with the factor written over B (d_U = d_B, and a
d_U that begins inside B's array): the same results, bit for bit, as with arrays of
their own, on orders below, at and above the Cholesky's 32-column blocks.  Its
workgroups read B's first block rows while others write U's."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 8])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n", [5, 32, 33, 150, 400])
def test_factor_over_b(qm, torch_cuda, n, cplx, shift):
    torch = torch_cuda
    print(f"case factor over B n {n} complex {cplx} shift {shift}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system(n=8, L=4.0, natoms=1, nbands=1))
    rng = np.random.default_rng(n)

    def mat():
        return rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)

    a, b = mat(), mat()
    a, b = 0.5 * (a + a.conj().T), b @ b.conj().T / n + np.eye(n)
    dt = torch.complex128 if cplx else torch.float64
    fn = H.lib.qm_hegvd_z64 if cplx else H.lib.qm_sygvd_f64

    def solve(in_place):
        A = torch.from_numpy(a.T.copy()).cuda()
        room = torch.zeros(n * n + shift, dtype=dt, device="cuda")
        B = room[:n * n]
        B.copy_(torch.from_numpy(b.T.copy()).cuda().reshape(-1))
        U = room[shift:shift + n * n] if in_place else torch.zeros(n * n, dtype=dt, device="cuda")
        w = torch.empty(n, dtype=torch.float64, device="cuda")
        Z = torch.empty((n, n), dtype=dt, device="cuda")
        qm._lib.check(fn(H.ctx, n, *(ctypes.c_void_p(t.data_ptr()) for t in (A, B, w, Z, U)), n,
                         ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        return w, Z, torch.tril(U.reshape(n, n))  # rows of the buffer are U's columns

    for x, y in zip(solve(False), solve(True)):
        assert torch.equal(x, y)
    H.close()
