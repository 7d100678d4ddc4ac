"""The legal-state flag from call to call: a call's result depends on its own state alone, whatever
the call before it found (its flag is cleared by a launch only where it may be set), with and
without waiting calls in between, for the one-launch and the multi-kernel fe()."""
import importlib.util
import os

import pytest

from conftest import PKG

spec = importlib.util.spec_from_file_location("mvd_problems", os.path.join(PKG, "problems.py"))
problems = importlib.util.module_from_spec(spec)
spec.loader.exec_module(problems)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,nchem", [((9, 8, 7), 0), ((9, 8, 7), 4), ((52, 50, 50), 0),
                                        ((66, 34, 33), 2)])
def test_flag_is_the_calls_own(mvd, torch_gpu, dims, nchem):
    torch = torch_gpu
    print(f"[state flag] dims={dims} nchem={nchem}", flush=True)
    w = problems.smooth_state(*dims, nchem=nchem, seed=41)
    good = [torch.from_numpy(a).to("cuda") if a is not None else None for a in w[:5 + (nchem > 0)]]
    good += [None] * (6 - len(good))
    bad = [a.clone() if a is not None else None for a in good]
    bad[0][3] = -1.0                                  # one cell's density
    out = [torch.empty_like(a) if a is not None else None for a in good]
    ctx = mvd.Context(mvd.make_params(*dims, nchem))
    illegal = mvd.MVD_ILLEGAL_STATE

    def check(state, expect):
        assert ctx.fe(state, out, allow_illegal=True) == expect
        assert (ctx.last_state_flags() != 0) == (expect != 0)

    for state, expect in ((good, 0), (good, 0), (bad, illegal), (bad, illegal), (good, 0),
                          (good, 0), (bad, illegal), (good, 0)):
        check(state, expect)
    ctx.fe_async(bad, out)
    assert ctx.last_state_flags() != 0
    check(good, 0)
    ctx.fe_async(good, out)
    check(bad, illegal)
    ctx.fe_async(good, out)
    assert ctx.last_state_flags() == 0
    check(good, 0)
    check(bad, illegal)
    ctx.close()
