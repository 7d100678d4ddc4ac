"""The batched chemistry step's work queue in each of its kernel variants (table width, forcing,
step rejection, the three LDS layouts): 40000 cells on so few waves that waves take several
chunks, one by its index and the rest from the queue. The queue changes which wave solves a cell and nothing else, so the states, the
temperatures and the Newton work equal, bit for bit, those of the default shape, where every
chunk has a wave."""
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
N, H = 40000, 500.0


@pytest.mark.parametrize("table", ["sdirk3", "ark437"])
@pytest.mark.parametrize("forced", [False, True])
@pytest.mark.parametrize("halvings", [0, 3])
def test_queue_variants(mvd, torch_gpu, table, forced, halvings):
    torch = torch_gpu
    print(f"[dirk queue variants] {table} forced={forced} halvings={halvings}", flush=True)
    opts = getattr(mvd, table)(newton_tol=1e-2, max_iters=10, max_halvings=halvings)
    y0, _ = problems.chem_cells(N, seed=97)
    rng = np.random.default_rng(98)
    yp = 1.0 + 0.02 * rng.uniform(-1, 1, 10 * N)
    force = torch.from_numpy(rng.standard_normal(10 * N) * 0.02 / H).to("cuda") if forced else None
    ref = None
    # waves: the default, one per CU at most, two, more (625 chunks of 64 cells)
    for block, waves in ((256, 0), (64, 100), (128, 300), (256, 520)):
        ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
        ctx.chem_setup(orc.load_tables(), N)
        yd = torch.from_numpy(y0.copy()).to("cuda")
        ctx.chem_prepare(yd)
        yd.copy_(torch.from_numpy(yp))
        ctx.dirk_set_shape(block, waves)
        failed, st = ctx.dirk_steps(yd, H, 2, force, opts)
        got = (failed, st["newton_iters"], st["setups"], st["hist"], yd.cpu().numpy(),
               ctx.chem_state("Ts", torch).cpu().numpy())
        ctx.close()
        assert failed == 0 and np.isfinite(got[4]).all()
        ref = ref or got
        assert got[:4] == ref[:4], (block, waves)
        assert np.array_equal(got[4], ref[4]) and np.array_equal(got[5], ref[5]), (block, waves)
