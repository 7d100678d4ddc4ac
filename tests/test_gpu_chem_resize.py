"""The block solver when mvd_chem_setup is called again on its context with another number of
cells: factors of the earlier cells are refused (MVD_NOT_READY) and the next lsetup has room for
all of the new ones. Residual bound of the other solver tests, 1e-13 of |A||x|."""
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


# from 65 cells: the same number of waves, more of them, fewer cells, more again
@pytest.mark.parametrize("formed", [False, True])
def test_solver_follows_setup(mvd, torch_gpu, formed):
    torch = torch_gpu
    ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
    gamma = 435.8
    for k, n in enumerate((65, 128, 1000, 30, 5000)):
        print(f"[chem resize] n={n} formed={formed}", flush=True)
        y, _ = problems.chem_cells(n, seed=61 + k)
        ctx.chem_setup(orc.load_tables(), n)
        yd = torch.from_numpy(y.copy()).to("cuda")
        ctx.chem_prepare(yd)
        b = np.random.default_rng(k).standard_normal(10 * n)
        bd = torch.from_numpy(b).to("cuda")
        x = torch.empty_like(bd)
        if k:
            assert mvd.lib().mvd_chem_lsolve(ctx.h, mvd.dptr(bd), mvd.dptr(x)) == mvd.MVD_NOT_READY
        ctx.chem_rhs(yd, torch.empty_like(yd))
        J = torch.empty(100 * n, dtype=torch.float64, device="cuda")
        ctx.chem_jac(yd, J)
        A = np.eye(10)[None] - gamma * J.cpu().numpy().reshape(n, 10, 10).transpose(0, 2, 1)
        if formed:
            Ad = torch.from_numpy(np.ascontiguousarray(A.transpose(0, 2, 1)).reshape(-1)).to("cuda")
            assert mvd.lib().mvd_chem_lsetup_matrix(ctx.h, mvd.dptr(Ad)) == 0
        else:
            assert ctx.chem_lsetup(gamma, J) == 0
        ctx.chem_lsolve(bd, x)
        xs = x.cpu().numpy().reshape(n, 10)
        res = np.abs(np.matmul(A, xs[:, :, None])[:, :, 0] - b.reshape(n, 10)).max(axis=1)
        size = (np.abs(A) * np.abs(xs)[:, None, :]).sum(axis=2).max(axis=1)
        assert np.all(res <= 1e-13 * size)
    ctx.close()
