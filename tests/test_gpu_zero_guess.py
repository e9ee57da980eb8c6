"""FP32 cycles that start from a zero guess they neither clear nor read: a
solver that has solved another problem before gives the bits of a fresh one --
nothing of the old correction is left -- for every way a cycle can begin (one
sweep a launch, a small finest level, pairs of sweeps, no pre-sweep, the first
and the further cycles of one preconditioner application)."""
import numpy as np
import pytest

import pamr_amrd_amd as pm
from pamr_amrd_amd import hierarchy as H

pytestmark = pytest.mark.gpu

BOX = (0.0, 1.0, 0.0, 1.0, 0.0, 1.0)


def solver(n, op, pre, pst, pairs):
    S = pm.Solver(n, op=op)
    S.set_params(pre=pre, pst=pst)
    if pairs:
        assert pm.lib().pmg_set_sweep_blocking(S.h, 1, 16) == 0
    shape = (n, n, n)
    if op == 1:
        S.upload(S.nlev, pm.PMG_F_A, H.lognormal_on(shape, BOX))
        S.upload(S.nlev, pm.PMG_F_C, H.uniform_on(shape, BOX))
    return S


def solve(S, n, seed, fgmres):
    shape = (n, n, n)
    rho = -H.gaussian_on(shape, BOX, seed=seed)
    rho[0], rho[-1] = 0, 0
    rho[:, 0], rho[:, -1], rho[:, :, 0], rho[:, :, -1] = 0, 0, 0, 0
    S.upload(S.nlev, pm.PMG_F_RHO, rho)
    S.init()
    S.zero_solution()
    r0, h = S.solve_fgmres(6, 1e-9, 12) if fgmres else S.solve_rel(1, 1e-9, 12)
    return S.download(S.nlev, pm.PMG_F_U), np.asarray(h) / r0


@pytest.mark.parametrize("n,op,pre,pst,pairs,fgmres,cycles", [
    (81, 0, 2, 2, False, False, 1), (81, 1, 2, 2, False, True, 2), (81, 0, 1, 2, False, False, 1),
    (33, 0, 2, 2, False, False, 1), (33, 0, 0, 2, False, False, 1), (81, 0, 0, 3, False, True, 1),
    (81, 0, 2, 2, True, False, 1)])
def test_second_solve_equals_fresh(torch_cuda, n, op, pre, pst, pairs, fgmres, cycles):
    print(f"case zero guess n={n} op={op} V({pre},{pst}) pairs={pairs} fgmres={fgmres} cycles={cycles}", flush=True)
    out = []
    for first in (None, 7):
        S = solver(n, op, pre, pst, pairs)
        if fgmres:
            S.set_fgmres_prec_cycles(cycles)
        if first is not None:
            solve(S, n, first, fgmres)
        out.append(solve(S, n, 1234, fgmres))
        S.close()
    (u0, h0), (u1, h1) = out
    assert h0[-1] < 1e-4
    assert np.array_equal(h0, h1)
    assert np.array_equal(u0, u1)
