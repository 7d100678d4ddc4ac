"""fe() and its vector-Jacobian product in units where velocities are s and energies s^2 (densities
one): the acoustic reconstructions scale their eps with the squared sound speed, whose powers must
not underflow. fe() holds down to a squared sound speed of 3e-17, the product further.

The reference's eigenvectors hold the squared sound speed where the sound speed would stand, so
in such units the two parts of an acoustic value, K (s^3) and A (s^2), are 1/s apart, and what K
adds is left with 1/s times the rounding of the values. The bound is therefore 1e-12 / s of a
field's norm against the CPU oracle, a hundred times the difference that s = 1 leaves."""
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
MIXED = (0, 0, 1, 3, 3, 1)


def state(dims, nchem, s):
    w = problems.smooth_state(*dims, nchem=nchem, seed=13)
    return [w[0]] + [a * s for a in w[1:4]] + [w[4] * s * s, w[5]]


@pytest.mark.parametrize("dims,nchem", [((33, 17, 19), 2), ((70, 5, 6), 0)])
@pytest.mark.parametrize("s", [1e-8, 1e-10])
def test_vjp(mvd, torch_gpu, dims, nchem, s):
    torch = torch_gpu
    print(f"[fe vjp scales] dims={dims} nchem={nchem} s={s}", flush=True)
    w = state(dims, nchem, s)
    rng = np.random.default_rng(14)
    # cotangents in the inverse units, so that the fields' shares are as they are for s = 1
    v = [rng.standard_normal(a.size) / f for a, f in zip(w, (1.0, s, s, s, s * s, 1.0))]
    ref = orc.fe_vjp(orc.make_grid(*dims, nchem, MIXED), w, v)
    nf = 6 if nchem else 5
    ctx = mvd.Context(mvd.make_params(*dims, nchem, MIXED))
    dev = [[torch.from_numpy(a).to("cuda") for a in x[:nf]] + [None] * (6 - nf) for x in (w, v)]
    out = [torch.full_like(a, float("nan")) if a is not None else None for a in dev[0]]
    ctx.fe_vjp(dev[0], dev[1], out)
    for q in range(nf):
        assert np.isfinite(ref[q]).all()
        assert normwise_err(out[q].cpu().numpy(), ref[q]) <= 1e-12 / s, q
    ctx.close()


@pytest.mark.parametrize("dims,nchem", [((33, 17, 19), 2), ((70, 5, 6), 0)])
def test_fe(mvd, torch_gpu, dims, nchem):
    torch, s = torch_gpu, 1e-8
    print(f"[fe scales] dims={dims} nchem={nchem} s={s}", flush=True)
    w = state(dims, nchem, s)
    flag, ref = orc.fe(orc.make_grid(*dims, nchem, MIXED), w)
    assert flag == 0
    nf = 6 if nchem else 5
    ctx = mvd.Context(mvd.make_params(*dims, nchem, MIXED))
    wd = [torch.from_numpy(a).to("cuda") for a in w[:nf]] + [None] * (6 - nf)
    out = [torch.full_like(a, float("nan")) if a is not None else None for a in wd]
    for on in (0, 2):                      # the one-launch kernel, the face kernels
        assert mvd.lib().mvd_profile(ctx.h, on) == 0
        ctx.fe(wd, out)
        for q in range(nf):
            assert normwise_err(out[q].cpu().numpy(), ref[q]) <= 1e-12 / s, (on, q)
    ctx.close()
