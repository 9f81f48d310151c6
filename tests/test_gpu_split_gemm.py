"""The FP32 update on the bf16 matrix cores at the edges of its tiles.

Reference: float64 products.  Bound, elementwise, from the number of FP32
roundings of a sum, each at most one unit in the last place (2^-23) of the sum of
magnitudes: six per 16 K values, and 2^-22 for the three-way split and the store.

Values outside the split's range take the FP32 route: infinities give infinities
at the same places, values of 1e-33 keep the same relative bound.
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -23

SHAPES = [  # m, n, ng
    (1, 128, 49153),
    (15, 128, 49152),
    (128, 129, 50001),
    (257, 200, 49207),
    (270, 256, 60480),
    (300, 385, 33333),
    (512, 513, 20000),
]


def _check(H, z, u):
    """One update against float64; z, u on the device."""
    zd, ud = z.double(), u.double()
    bound = (6 * math.ceil(u.shape[0] / 16) + 2) * EPS * (ud.abs().T @ zd.abs())
    assert bool(((H.update(z, u).double() - ud.T @ zd).abs() <= bound).all())


@pytest.mark.parametrize("m,n,ng", SHAPES)
def test_split_update(qm, torch_cuda, m, n, ng):
    torch = torch_cuda
    print(f"case split {m} x {n} over {ng}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system())
    g = torch.Generator(device="cuda").manual_seed(m + n)
    z, u = (torch.rand(s, device="cuda", generator=g) - 0.5 for s in ((m, ng), (m, n)))
    _check(H, z, u)
    H.close()


@pytest.mark.parametrize("tiny", ["z", "u", "column"])
def test_split_tiny_values(qm, torch_cuda, tiny):
    torch = torch_cuda
    m, n, ng = 130, 140, 50001
    print(f"case split tiny {tiny}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system())
    g = torch.Generator(device="cuda").manual_seed(3)
    z, u = (torch.rand(s, device="cuda", generator=g) - 0.5 for s in ((m, ng), (m, n)))
    {"z": z, "u": u, "column": u[:, 77]}[tiny].mul_(1e-33)
    _check(H, z, u)
    H.close()


def test_split_infinities(qm, torch_cuda):
    torch = torch_cuda
    m, n, ng = 130, 140, 50001
    print("case split infinities", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system())
    g = torch.Generator(device="cuda").manual_seed(4)
    z, u = (torch.rand(s, device="cuda", generator=g) - 0.5 for s in ((m, ng), (m, n)))
    z[7, 1234], z[99, 50000], z[12, 300] = math.inf, -math.inf, math.nan
    got, want = H.update(z, u).cpu().numpy(), (u.double().T @ z.double()).cpu().numpy()
    assert np.isinf(want).any() and np.isnan(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    H.close()
