"""The temperature and its slope as an implicit step leaves them, against the oracle's ten Newton
steps, for warm starts far from the root, 1% and 2e-8 away from it. The step is one backward
Euler stage of 1e-200 s: h f underflows next to the state, one Newton iteration accepts it
unchanged, and Ts and dTs_ge are those of the one right-hand side evaluated at it.

Tolerance: each side's T is the root of its own rounding of T kb nsum / (density mH) = ge, and
that expression has at most 16 roundings of 2^-53 (the density's sum, the monatomic sum, two
terms with 1 / (gamma - 1), the products), so both together 32 * 2^-53 = 3.6e-15 of T; the slope
has half as many more in its second term, 48 * 2^-53 = 5.3e-15 of dTs_ge."""
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


# 65 cells: the step's own solve; 5000: the one of the ordering pass; the plain path; the
# substepping variant, which solves again
@pytest.mark.parametrize("n,plain,halvings", [(65, False, 0), (5000, False, 0), (300, True, 0),
                                              (5000, False, 2)])
def test_step_temperature(mvd, torch_gpu, n, plain, halvings):
    torch = torch_gpu
    print(f"[step temperature] n={n} plain={plain} halvings={halvings}", flush=True)
    y, _ = problems.chem_cells(n, seed=71)
    oc = orc.Chem(n)
    yo = y.copy()
    oc.prepare(yo)
    oc.extra()
    yo *= np.exp(np.random.default_rng(5).normal(0.0, 0.02, 10 * n))
    ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
    ctx.chem_setup(orc.load_tables(), n)
    ctx.chem_prepare(torch.from_numpy(y.copy()).to("cuda"))
    o = mvd.set_table(mvd.sdirk3(max_halvings=halvings), [[1.0]])
    oc.array("Ts")[:] = 1000.0
    oc.rhs(yo)
    root = oc.array("Ts").copy()
    noise = np.random.default_rng(6).normal(0.0, 1.0, n)
    for T0 in (np.full(n, 1000.0), root * (1.0 + 1e-2 * noise), root * (1.0 + 2e-8 * noise)):
        oc.array("Ts")[:] = T0
        oc.rhs(yo)
        ctx.chem_state_set("Ts", torch.from_numpy(T0.copy()).to("cuda"))
        yd = torch.from_numpy(yo.copy()).to("cuda")
        failed, stats = ctx.dirk_step(yd, 1e-200, o, plain=plain)
        assert failed == 0 and stats["newton_iters"] == n
        assert np.array_equal(yd.cpu().numpy(), yo)
        for name, tol in (("Ts", 3.6e-15), ("dTs_ge", 5.3e-15)):
            got, ref = ctx.chem_state(name, torch).cpu().numpy(), oc.array(name)
            assert np.max(np.abs(got - ref) / np.abs(ref)) <= tol, name
    ctx.close()
