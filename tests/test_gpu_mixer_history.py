"""DIIS rings longer than one pass of the overlap kernel (9 fields), than the
order whose elimination runs in LDS (32) and the longest one (64), against the
oracle.  Every step's density is independent random, so the overlap matrix is
well conditioned (cond < 1e4) and both sides' coefficients agree to cond * eps
* (order) < 1e-9."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import scf_ref as S  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("history", [2, 8, 9, 10, 18, 31, 32, 64])
def test_mixer_long_history(qm, torch_cuda, history):
    torch = torch_cuda
    print(f"case DIIS history {history}", flush=True)
    s = qm.system.small_system(n=12, L=6.0, natoms=1, nbands=1)
    H = qm.hamiltonian.Hamiltonian(s)
    rng = np.random.default_rng(history)
    x0 = rng.uniform(0, 1, s.ng)
    m, o = qm.scf.Mixer(H, "diis", history, 0.3), S.MixDIIS(0.3, history)
    m.init(torch.from_numpy(x0.copy()).cuda())
    o.init(x0)
    for step in range(history + 2):
        out = rng.uniform(0, 1, s.ng)
        t = torch.from_numpy(out.copy()).cuda()
        dg = m.predict(t)
        xo, do = o.predict(out)
        assert abs(dg - do) <= 1e-9 * do, step
        assert np.abs(t.cpu().numpy() - xo).max() <= 1e-9 * np.abs(xo).max(), step
    m.close()
    H.close()
