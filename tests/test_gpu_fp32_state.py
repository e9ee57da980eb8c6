"""What calls between solves do to the FP32 arrays, and what the next solve
makes of it: solves start their FP32 cycles from zero, so a solver with values
in its FP32 correction gives a fresh one's bits.  81^3 points a level above
those whose legs are one launch, 33^3 one of them."""
import numpy as np
import pytest

import pamr_amrd_amd as pm
from pamr_amrd_amd import hierarchy as H

pytestmark = pytest.mark.gpu

BOX = (0.0, 1.0, 0.0, 1.0, 0.0, 1.0)


def solver(n, op):
    S = pm.Solver(n, op=op)
    shape = (n, n, n)
    S.upload(S.nlev, pm.PMG_F_RHO, -H.gaussian_on(shape, BOX))
    if op == 1:
        S.upload(S.nlev, pm.PMG_F_A, H.lognormal_on(shape, BOX))
        S.upload(S.nlev, pm.PMG_F_C, H.uniform_on(shape, BOX))
    S.set_params(pre=2, pst=2)
    S.init()
    return S


def solve(S, fgmres):
    S.zero_solution()
    r0, h = S.solve_fgmres(3, 1e-9, 6) if fgmres else S.solve_rel(1, 1e-9, 4)
    return S.download(S.nlev, pm.PMG_F_U), np.asarray(h) / r0


@pytest.mark.parametrize("n,op", [(33, 0), (81, 0), (81, 1)])
@pytest.mark.parametrize("fgmres", [False, True])
def test_uploaded_correction_is_not_a_guess(torch_cuda, n, op, fgmres):
    print(f"case uploaded u32 n={n} op={op} fgmres={fgmres}", flush=True)
    out = []
    for dirty in (False, True):
        S = solver(n, op)
        if dirty:
            S.upload32(S.nlev, 0, np.random.default_rng(n).standard_normal((n, n, n)))
        out.append(solve(S, fgmres))
        S.close()
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("n", [33, 81])
def test_correction_reads_as_zero_once_added(torch_cuda, n):
    """a mixed iteration's correction belongs to the FP64 u; what FGMRES's
    preconditioner returned last stays readable until the next cycle"""
    print(f"case u32 after solves n={n}", flush=True)
    S = solver(n, 0)
    solve(S, False)
    assert not S.download32(S.nlev, 0).any()
    solve(S, True)
    z = S.download32(S.nlev, 0)
    assert z.any()
    assert np.array_equal(S.download32(S.nlev, 0), z)
    S.close()


def test_set_params_leaves_the_correction(torch_cuda):
    print("case u32 after set_params", flush=True)
    S = solver(81, 0)
    solve(S, True)
    z = S.download32(S.nlev, 0)
    S.set_params(pre=2, pst=2)
    assert z.any() and np.array_equal(S.download32(S.nlev, 0), z)
    S.close()


@pytest.mark.parametrize("fgmres", [False, True])
@pytest.mark.parametrize("w0_i", [0.0, float("nan")])
def test_solve_after_weights_that_give_nan(torch_cuda, w0_i, fgmres):
    """faces of the correction are 0 / w0_i: what a solve with such a weight
    leaves there is gone when the weight is a number again"""
    print(f"case w0_i={w0_i} fgmres={fgmres}", flush=True)
    out = []
    for bad in (False, True):
        S = solver(81, 0)
        if bad:
            S.set_params(pre=2, pst=2, w0_i=w0_i)
            S.solve_rel(1, 1e-9, 2)
            S.set_params(pre=2, pst=2)
        out.append(solve(S, fgmres))
        S.close()
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0])
