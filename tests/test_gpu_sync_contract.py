"""Calls that return finished work: qm_band_density_* and qm_nonlocal_forces_*
synchronise the stream they are given.

Each is called on a non-blocking stream behind products of about a tenth of a
second; when it returns, the stream has nothing left to do.  The forces also for
atoms without projectors, where there is nothing to sum."""
import types

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _idle_after(torch, call):
    """Whether `call`, made behind long work on a stream of its own, leaves that stream idle."""
    a = torch.rand((8192, 8192), device="cuda")
    b = torch.empty_like(a)
    torch.mm(a, a, out=b)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for _ in range(20):
            torch.mm(a, a, out=b)
        assert not stream.query()
        call()
        idle = stream.query()
    torch.cuda.synchronize()
    return idle


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_band_density_synchronises(qm, orc, torch_cuda, prec):
    torch = torch_cuda
    s = qm.system.small_system(n=11, L=4.0, natoms=1, nbands=5)
    print(f"case density behind long work {prec}", flush=True)
    H = qm.hamiltonian.Hamiltonian(s)
    rng = np.random.default_rng(4)
    psi = rng.uniform(-0.5, 0.5, (5, s.ng)).astype(np.float32).astype(np.float64)
    x = torch.from_numpy(psi).to("cuda", torch.float64 if prec == "f64" else torch.float32)
    rho = torch.zeros(s.ng, dtype=torch.float64, device="cuda")
    occ = np.linspace(2.0, 0.5, 5)
    assert _idle_after(torch, lambda: H.band_density(x, occ, rho=rho))
    want = orc.band_density(s, psi, occ)
    assert np.abs(rho.cpu().numpy() - want).max() <= 1e-13 * np.abs(want).max()
    H.close()

@pytest.mark.parametrize("projectors", [True, False])
def test_forces_synchronise(qm, torch_cuda, projectors):
    torch = torch_cuda
    s = qm.system.small_system(n=11, L=4.0, natoms=1, nbands=5)
    print(f"case forces behind long work, projectors {projectors}", flush=True)
    H = qm.hamiltonian.Hamiltonian(s)
    if not projectors:
        none = np.zeros(0)
        H.set_projectors(types.SimpleNamespace(
            natoms=1, nproj=[0], vox_off=[0, 4], vox_xyz=np.zeros((4, 3), np.int32), table=none,
            dtable=none, tab_off=[0, 0], energy=none, proj_off=[0, 0]))
    x = torch.rand((5, s.ng), dtype=torch.float64, device="cuda")
    out = []
    assert _idle_after(torch, lambda: out.append(H.nonlocal_forces(x, np.ones(5))))
    e, f = out[0]
    assert (np.abs(f).max() > 0.0 and e != 0.0) if projectors else (e == 0.0 and not f.any())
    H.close()
