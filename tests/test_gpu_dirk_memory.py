"""The batched chemistry step's LDS layouts (by the number of 64-cell waves: up to one per CU the
cells' table bins, up to two the long tables' stage derivatives, beyond that neither): cells are
independent of each other, so a batch gives the same bits as its parts. The sizes lie on both
sides of each edge of a 256-CU device; small batches are held against the oracle in
test_gpu_dirk.py."""
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


def run(mvd, torch, opts, y0, yp, force, h, nsteps):
    n = y0.size // 10
    ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
    ctx.chem_setup(orc.load_tables(), n)
    yd = torch.from_numpy(y0.copy()).to("cuda")
    ctx.chem_prepare(yd)
    yd.copy_(torch.from_numpy(yp))
    fd = torch.from_numpy(force).to("cuda") if force is not None else None
    failed, _ = ctx.dirk_steps(yd, h, nsteps, fd, opts)
    out = yd.cpu().numpy().reshape(n, 10)
    ctx.close()
    assert failed == 0
    return out


@pytest.mark.parametrize("table,forced", [("ark437", True), ("ark437", False), ("sdirk3", True)])
@pytest.mark.parametrize("n", [32769, 32768, 16385, 16384, 8193, 2049, 65])
def test_batch_equals_parts(mvd, torch_gpu, table, forced, n):
    torch = torch_gpu
    print(f"[dirk memory] {table} n={n}", flush=True)
    # short steps of a substepping solver, held factors between them
    opts = getattr(mvd, table)(newton_tol=1e-2, max_iters=10, max_steps_between_setups=2,
                               max_halvings=6)
    h, nsteps = 200.0, 3
    y0, _ = problems.chem_cells(n, seed=91)
    rng = np.random.default_rng(92)
    yp = 1.0 + 0.02 * rng.uniform(-1, 1, 10 * n)
    force = rng.standard_normal(10 * n) * 0.02 / (nsteps * h) if forced else None
    whole = run(mvd, torch, opts, y0, yp, force, h, nsteps)
    assert np.isfinite(whole).all()
    for a, b in ((0, min(n, 70)), (n // 2, min(n, n // 2 + 2100)), (max(n - 61, 0), n)):
        c = slice(10 * a, 10 * b)
        part = run(mvd, torch, opts, y0[c], yp[c], force[c] if forced else None, h, nsteps)
        assert np.array_equal(part, whole[a:b]), (a, b)


@pytest.mark.parametrize("table", ["ark437", "sdirk3"])
@pytest.mark.parametrize("n", [20000, 8193, 4096, 130])
def test_forced_steps_without_rejection(mvd, torch_gpu, table, n):
    """Without step rejection (a kernel variant of its own) the same bits as with it, where no
    step is rejected."""
    torch = torch_gpu
    print(f"[dirk memory, no rejection] {table} n={n}", flush=True)
    h, nsteps = 50.0, 3
    y0, _ = problems.chem_cells(n, seed=93)
    rng = np.random.default_rng(94)
    yp = 1.0 + 0.02 * rng.uniform(-1, 1, 10 * n)
    force = rng.standard_normal(10 * n) * 0.02 / (nsteps * h)
    got = [run(mvd, torch, getattr(mvd, table)(newton_tol=1e-2, max_iters=20, max_halvings=k),
               y0, yp, force, h, nsteps) for k in (0, 6)]
    assert np.isfinite(got[0]).all()
    assert np.array_equal(got[0], got[1])
