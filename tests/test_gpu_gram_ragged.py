"""Gram and update at sizes off the tiles: single columns, one past a tile, K with
and without a remainder of a panel, and blocks that start off a 16-byte boundary.

Reference: float64 products.  Bound, elementwise, of the sum of magnitudes: FP32
sums round at most 256 times before they go to FP64 (the Gram) and m times (the
update), at 2^-24 each; FP64 sums round at most once per term at 2^-53 (and the
reference the same): 2^-52 per term.
"""
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # m, n, ng
    (1, 1, 5),
    (3, 65, 16),
    (17, 33, 1000),
    (65, 66, 4096),
    (129, 64, 4097),
    (128, 128, 8192),
    (90, 129, 12345),
    (200, 300, 20001),
]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("m,n,ng", SHAPES)
def test_ragged_products(qm, torch_cuda, m, n, ng, prec, offset):
    torch = torch_cuda
    dt = torch.float64 if prec == "f64" else torch.float32
    print(f"case products {m} x {n} over {ng} {prec} offset {offset}", flush=True)
    H = qm.hamiltonian.Hamiltonian(qm.system.small_system())
    gen = torch.Generator(device="cuda").manual_seed(m * n + ng)

    def block(rows, cols):
        x = torch.rand(rows * cols + offset, device="cuda", dtype=dt, generator=gen) - 0.5
        return x[offset:].view(rows, cols)

    a, b, u = block(m, ng), block(n, ng), block(m, n)
    ad, bd, ud = a.double(), b.double(), u.double()
    per_gram = 2.0 ** -52 * (ng + 8) + (258 * 2.0 ** -24 if prec == "f32" else 0.0)
    bound = per_gram * (ad.abs() @ bd.abs().T)
    assert bool(((H.gram(a, b) - ad @ bd.T).abs() <= bound).all())
    per_upd = (m + 2) * (2.0 ** -24 if prec == "f32" else 2.0 ** -52)
    bound = per_upd * (ud.abs().T @ ad.abs())
    assert bool(((H.update(a, u).double() - ud.T @ ad).abs() <= bound).all())
    H.close()
