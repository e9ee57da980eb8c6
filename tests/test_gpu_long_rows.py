"""Rows of more than 2^23 points, whose tiles do not fit 32-bit byte offsets:
an FP64 cycle and a mixed iteration on such a grid equal those of its last 2049
columns as a grid of their own, bit for bit away from the cut -- with four
sweeps on the coarsest level a point depends on no more than 40 columns
around it."""
import numpy as np
import pytest

import pamr_amrd_amd as pm

pytestmark = pytest.mark.gpu

NX, M = (1 << 23) + 1025, 2049


def _solver(nx, op, data):
    S = pm.Solver(0, bbox=(0.0, 0.25 * (nx - 1), 0.0, 1.0, 0.0, 1.0), min_cwidth=3, op=op, shape=(nx, 5, 5))
    assert S.nlev == 2
    S.set_params(max_citer=0)
    for k, v in data.items():
        S.upload(S.nlev, getattr(pm, "PMG_F_" + k), v)
    S.init()
    return S


@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("mixed", [False, True])
def test_long_rows(torch_cuda, op, mixed):
    print(f"case long rows op={op} mixed={mixed}", flush=True)
    rng = np.random.default_rng(op)
    names = ("U", "RHO") + (("A", "C") if op else ())
    # values that repeat after a prime number of points: no address repeats a row's
    data = {k: np.resize(rng.random(1000003) if k == "A" else rng.standard_normal(1000003), (5, 5, NX)) + (k == "A")
            for k in names}
    if op:
        data["C"] = -np.abs(data["C"])
    out = []
    for nx, d in ((NX, data), (M, {k: v[:, :, -M:] for k, v in data.items()})):
        S = _solver(nx, op, d)
        if mixed:
            S.solve_rel(1, 0.0, 1)
        else:
            S.vcycle()
        out.append(S.download(S.nlev, pm.PMG_F_U)[:, :, -(M - 100):])
        S.close()
    assert not np.array_equal(out[0], data["U"][:, :, -(M - 100):])
    assert np.array_equal(out[0], out[1])
