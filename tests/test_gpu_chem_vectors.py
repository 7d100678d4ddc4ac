"""The per-call chemistry kernels around the edges of a wave, whose vectors pass through LDS:
the RHS, its vector-Jacobian product and the RHS returned beside it for cell counts that leave
a wave's last lanes idle, at 8-byte aligned addresses, with nothing written past the last cell
and in place. Bounds: 1e-12 (RHS) and 1e-10 (product) of a component's largest magnitude, those
of the other tests of these kernels."""
import importlib.util
import os

import numpy as np
import pytest

import orc
from conftest import PKG, normwise_err

spec = importlib.util.spec_from_file_location("mvd_problems", os.path.join(PKG, "problems.py"))
problems = importlib.util.module_from_spec(spec)
spec.loader.exec_module(problems)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 130])
def test_vectors(mvd, torch_gpu, n):
    torch = torch_gpu
    print(f"[chem vectors] n={n}", flush=True)
    y, _ = problems.chem_cells(n, seed=71)
    oc = orc.Chem(n)
    yo = y.copy()
    oc.prepare(yo)
    oc.extra()
    rng = np.random.default_rng(72)
    yo *= 1.0 + 0.05 * rng.standard_normal(yo.size)
    ctx = mvd.Context(mvd.make_params(4, 4, 4, 10))
    ctx.chem_setup(orc.load_tables(), n)
    ctx.chem_prepare(torch.from_numpy(y.copy()).to("cuda"))

    def odd(a=None):                       # 8-byte, not 16-byte aligned, with a guard behind
        buf = torch.full((10 * n + 21,), -7.25, dtype=torch.float64, device="cuda")
        if a is not None:
            buf[1:1 + 10 * n] = torch.from_numpy(a).to("cuda")
        return buf, buf[1:1 + 10 * n]

    def clean(buf):
        return float(buf[0]) == -7.25 and bool((buf[1 + 10 * n:] == -7.25).all())

    _, yd = odd(yo)
    fbuf, f = odd()
    for _ in range(3):                     # converge both temperature warm starts
        rf = oc.rhs(yo)
        ctx.chem_rhs(yd, f)
    assert clean(fbuf)
    got, ref = f.cpu().numpy().reshape(n, 10), rf.reshape(n, 10)
    for s in range(10):
        assert normwise_err(got[:, s], ref[:, s]) <= 1e-12, s
    v = rng.standard_normal(10 * n)
    rv = oc.vjp(yo, v).reshape(n, 10)
    _, vd = odd(v)
    bbuf, yb = odd()
    gbuf, g = odd()
    ctx.chem_vjp(yd, vd, yb, g)
    assert clean(bbuf) and clean(gbuf)
    got = yb.cpu().numpy().reshape(n, 10)
    for s in range(10):
        assert normwise_err(got[:, s], rv[:, s]) <= 1e-10, s
        assert normwise_err(g.cpu().numpy().reshape(n, 10)[:, s], ref[:, s]) <= 1e-12, s
    ctx.chem_vjp(yd, vd, vd)               # in place, from the same temperatures
    for s in range(10):
        assert normwise_err(vd.cpu().numpy().reshape(n, 10)[:, s], rv[:, s]) <= 1e-10, s
    ctx.close()
