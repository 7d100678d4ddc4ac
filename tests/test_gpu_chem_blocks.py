"""The Jacobian and the block linear solver around the edges of a wave (64 cells) and of the
32 cells it moves through LDS at a time: every cell's Jacobian block against the oracle (1e-12
of the block's largest entry, the bound of the other Jacobian tests) with nothing written past
the last one, and the solve's residual (1e-13 of |A||x|, the bound of the other solver tests)
from the Jacobian and from a formed matrix at a 8-byte aligned address."""
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


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 97, 200])
def test_blocks(mvd, torch_gpu, n):
    torch = torch_gpu
    print(f"[chem blocks] n={n}", flush=True)
    y, _ = problems.chem_cells(n, seed=61)
    oc = orc.Chem(n)
    yo = y.copy()
    oc.prepare(yo)
    oc.extra()
    ref = oc.rhs(yo)
    refJ = oc.jac(yo).transpose(0, 2, 1).reshape(n, 100)     # column-major blocks
    ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
    ctx.chem_setup(orc.load_tables(), n)
    yd = torch.from_numpy(y.copy()).to("cuda")
    ctx.chem_prepare(yd)
    f = torch.empty_like(yd)
    ctx.chem_rhs(yd, f)
    assert np.isfinite(ref).all()
    buf = torch.full((100 * n + 65,), -7.25, dtype=torch.float64, device="cuda")
    J = buf[1:1 + 100 * n]                       # 8-byte, not 16-byte aligned
    ctx.chem_jac(yd, J)
    got = J.cpu().numpy().reshape(n, 100)
    scale = np.abs(refJ).max(axis=1, keepdims=True)
    assert np.all(np.abs(got - refJ) <= 1e-12 * scale)
    assert float(buf[0]) == -7.25 and bool((buf[1 + 100 * n:] == -7.25).all())
    gamma = 435.8
    A = np.eye(10)[None] - gamma * got.reshape(n, 10, 10).transpose(0, 2, 1)
    b = np.random.default_rng(3).standard_normal(10 * n)
    bd = torch.from_numpy(b).to("cuda")
    formed = torch.empty(100 * n + 1, dtype=torch.float64, device="cuda")[1:]
    formed.copy_(torch.from_numpy(np.ascontiguousarray(A.transpose(0, 2, 1)).reshape(-1)))
    for setup in ("jacobian", "matrix"):
        if setup == "jacobian":
            assert ctx.chem_lsetup(gamma, J) == 0
        else:
            assert mvd.lib().mvd_chem_lsetup_matrix(ctx.h, mvd.dptr(formed)) == 0
        x = torch.empty_like(bd)
        ctx.chem_lsolve(bd, x)
        xs = x.cpu().numpy().reshape(n, 10)
        res = np.abs(np.matmul(A, xs[:, :, None])[:, :, 0] - b.reshape(n, 10)).max(axis=1)
        size = (np.abs(A) * np.abs(xs)[:, None, :]).sum(axis=2).max(axis=1)
        assert np.all(res <= 1e-13 * size), setup
    # an exactly singular last block is counted
    formed[100 * (n - 1):] = 0.0
    assert mvd.lib().mvd_chem_lsetup_matrix(ctx.h, mvd.dptr(formed)) == 1
    ctx.close()
