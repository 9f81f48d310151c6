"""Rounding of the FP32 update that no elementwise bound on well-scaled inputs shows.

No common sign: the bf16 matrix cores round their sums downward.  Left alone that
moves every output the same way, by 0.1 - 0.18 of the rms error from m = 1024 on;
accumulated with its sign turned for the middle half of K, what is left is the
unevenness of the growth of the sum (below a tenth of it), so the mean error over
all outputs stays below 1/32 of the rms error (the mean of 10^7 independent errors
is 3e-4 of it).

Tiny values beside ordinary ones: every output within (6 ceil(m / 16) + 2) units
of 2^-23 of its own sum of magnitudes, the bound of the well-scaled tests, where
an output consists of values down to FP32's smallest only.
"""
import math

import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -23


@pytest.mark.parametrize("kind", ["mixed", "one sign", "z one sign", "ramp"])
@pytest.mark.parametrize("m,n", [(1024, 256), (1536, 128), (3072, 256)])
def test_update_has_no_common_sign(qm, torch_cuda, m, n, kind):
    torch = torch_cuda
    print(f"case signed error {kind} {m} x {n}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system())
    g = torch.Generator(device="cuda").manual_seed(m + len(kind))
    z, u = (torch.rand(s, device="cuda", generator=g) for s in ((m, 60001), (m, n)))
    if kind == "mixed":
        z -= 0.5
    if kind in ("mixed", "z one sign"):
        u -= 0.5
    if kind == "ramp":
        u *= torch.linspace(0.01, 1.0, m, device="cuda")[:, None]
    err = H.update(z, u).double() - u.double().T @ z.double()
    rms, mean = float((err * err).mean().sqrt()), float(err.mean())
    print(f"mean / rms {mean / rms:+.4f}", flush=True)
    assert abs(mean) <= rms / 32
    H.close()

@pytest.mark.parametrize("size", [1e-30, 1e-34, 1e-36, 1e-38, 1e-42])
@pytest.mark.parametrize("where", ["z column", "z point", "u entry", "both"])
def test_update_tiny_beside_ordinary(qm, torch_cuda, where, size):
    torch = torch_cuda
    m = n = 160
    ng = 50001
    print(f"case tiny {where} {size:g}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system())
    g = torch.Generator(device="cuda").manual_seed(7)
    z = torch.rand((m, ng), device="cuda", generator=g) - 0.5
    u = torch.zeros((m, n), device="cuda")
    u[torch.randperm(m, device="cuda", generator=g)[:n], torch.arange(n, device="cuda")] = 1.0
    if where in ("z column", "both"):  # one column of Z, passed on by a permutation
        z[77] *= size
    if where in ("z point", "both"):   # one point of every column
        z[:, 33333] *= size
    if where == "u entry":             # one coefficient in a column that has no other at its points
        u[:, 5] = 0.0
        u[12, 5] = 0.7 * size
    zd, ud = z.double(), u.double()
    bound = (6 * math.ceil(m / 16) + 2) * EPS * (ud.abs().T @ zd.abs())
    # half a unit of the smallest subnormal for the store (and for each product of a tiny coefficient)
    err = (H.update(z, u).double() - ud.T @ zd).abs()
    assert bool((err <= bound + 2.0 ** -149).all())
    H.close()


@pytest.mark.parametrize("zs,us", [(1e10, 1e3), (1e10, 1e10), (1e30, 1e-20), (1e-25, 1e35), (3e37, 1e-5), (1.0, 3e37)])
def test_update_large_values(qm, torch_cuda, zs, us):
    """Scaled up or down against each other, on both sides of the split's upper end."""
    torch = torch_cuda
    m, n, ng = 160, 160, 50001
    print(f"case large {zs:g} {us:g}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system())
    g = torch.Generator(device="cuda").manual_seed(8)
    z, u = ((torch.rand(s, device="cuda", generator=g) - 0.5) * f for s, f in (((m, ng), zs), ((m, n), us)))
    zd, ud = z.double(), u.double()
    bound = (6 * math.ceil(m / 16) + 2) * EPS * (ud.abs().T @ zd.abs())
    assert bool(((H.update(z, u).double() - ud.T @ zd).abs() <= bound).all())
    H.close()
