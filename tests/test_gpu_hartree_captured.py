"""A Hartree solve on a context whose spectral apply a graph holds: the first
solve of the context allocates its spectrum although the graph pins the context
(no graph can hold a buffer that does not exist yet), on grids where the Poisson
solve runs on the own kernels (24^3) and where it takes the library transforms
while the FP32 apply does not (128 x 128 planes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(24, 24, 24), (128, 128, 4)])
def test_hartree_beside_a_captured_apply(qm, torch_cuda, n):
    torch = torch_cuda
    print(f"case hartree beside a graph {n}", flush=True)
    S = qm.system
    s = S.System("planes", *n, tuple(0.25 * m for m in n), np.full((1, 3), 0.4), np.zeros(1, np.int32),
                 np.full(1, 0.4), 4, 2, np.zeros((1, 3)), 1, 1).build()
    H = qm.hamiltonian.Hamiltonian(s)
    H.set_kinetic("fft")
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand((8, s.ng), device="cuda", generator=gen) - 0.5
    want, y = torch.empty_like(x), torch.empty_like(x)
    H.apply(want, x)
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph):
            H.apply(y, x)
    torch.cuda.current_stream().wait_stream(side)
    rho = torch.rand(s.ng, dtype=torch.float64, device="cuda", generator=gen)
    vh = torch.empty_like(rho)
    r = np.fft.fftn(rho.cpu().numpy().reshape(n[::-1]))
    g2 = 0.0
    for d in range(3):
        q = np.fft.fftfreq(n[d], d=1.0 / n[d]) * (2 * np.pi / s.cell[d])
        g2 = g2 + (q * q).reshape([-1 if 2 - e == d else 1 for e in range(3)])
    ref = np.fft.ifftn(r * np.where(g2 > 0, 4 * np.pi / np.where(g2 > 0, g2, 1.0), 0.0)).real.reshape(-1)
    for rep in range(3):
        print(f"case replay {rep}", flush=True)
        vh.fill_(float("nan"))
        y.fill_(float("nan"))
        qm.scf.hartree(H, rho, vh)
        graph.replay()
        torch.cuda.synchronize()
        assert np.abs(vh.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
        assert torch.equal(y, want)
    del graph
    H.lib.qm_release_captures(H.ctx)
    H.close()
