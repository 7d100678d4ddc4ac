"""The chemistry adjoint's launch shapes (pairs of waves for small batches, four groups of 64
cells per block for large ones, single groups where nothing is recomputed): cells are independent
of each other, so a batch gives the same bits as its parts, and as any checkpoint interval. The
small shapes are held against the oracle in test_gpu_adjoint.py; one wave past the edge between
the shapes (2 x 256 waves) runs the large one here."""
import importlib.util
import os

import numpy as np
import pytest

import orc
from conftest import PKG

spec = importlib.util.spec_from_file_location("mvd_problems", os.path.join(PKG, "problems.py"))
problems = importlib.util.module_from_spec(spec)
spec.loader.exec_module(problems)

pytestmark = pytest.mark.gpu
NSTEPS, H = 5, 200.0


def run(mvd, torch, y0, yp, lamT, K):
    n = y0.size // 10
    ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
    ctx.chem_setup(orc.load_tables(), n)
    yd = torch.from_numpy(y0.copy()).to("cuda")
    ctx.chem_prepare(yd)
    yd.copy_(torch.from_numpy(yp))
    lt = torch.from_numpy(lamT).to("cuda")
    l0 = torch.full_like(lt, float("nan"))
    assert ctx.dirk_adjoint(yd, H, NSTEPS, K, lt, l0) == 0
    out = yd.cpu().numpy().reshape(n, 10), l0.cpu().numpy().reshape(n, 10)
    ctx.close()
    return out


@pytest.mark.parametrize("n,K", [(32769, 2), (32768, 2), (1000, 2), (65, 1), (63, NSTEPS)])
def test_batch_equals_parts(mvd, torch_gpu, n, K):
    torch = torch_gpu
    print(f"[adjoint shapes] n={n} K={K}", flush=True)
    y0, _ = problems.chem_cells(n, seed=81)
    rng = np.random.default_rng(82)
    yp = 1.0 + 0.3 * rng.uniform(-1, 1, 10 * n)
    lamT = rng.standard_normal(10 * n)
    y, lam = run(mvd, torch, y0, yp, lamT, K)
    assert np.isfinite(y).all() and np.isfinite(lam).all()
    for a, b in ((0, min(n, 61)), (max(n - 70, 0), n)):
        c = slice(10 * a, 10 * b)
        ys, ls = run(mvd, torch, y0[c], yp[c], lamT[c], 3)
        assert np.array_equal(ys, y[a:b]) and np.array_equal(ls, lam[a:b]), (a, b)
