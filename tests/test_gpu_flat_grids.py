"""Grids with so many (x, y) tiles that a launch would need more blocks than the
norm workspace holds -- the residual's short marches on a flat one, the fused
residual + injection on a thin one: two cycles bit for bit against the oracle."""
import numpy as np
import pytest

import oracle as O
import pamr_amrd_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,bbox,op", [((9, 8209, 33), (0.0, 1.0, 0.0, 1026.0, 0.0, 4.0), 0),
                                           ((9, 8209, 33), (0.0, 1.0, 0.0, 1026.0, 0.0, 4.0), 1),
                                           ((1048577, 5, 5), (0.0, 262144.0, 0.0, 1.0, 0.0, 1.0), 0)])
def test_flat_grid_cycles(torch_cuda, shape, bbox, op):
    print(f"case flat grid {shape} op={op}", flush=True)
    rng = np.random.default_rng(op)
    m = O.UniformMG(0, bbox=bbox, mcw=3, op=op, shape=shape)
    S = pm.Solver(0, bbox=bbox, min_cwidth=3, op=op, shape=shape)
    assert m.nlev == S.nlev
    full = m.shape(m.nlev)
    data = {"RHO": rng.standard_normal(full), "U": rng.standard_normal(full)}
    if op == 1:
        data["A"] = np.exp(0.3 * rng.standard_normal(full))
        data["C"] = -rng.random(full)
    for k, v in data.items():
        m.field(m.nlev, getattr(O, "F_" + k))[:] = v
        S.upload(S.nlev, getattr(pm, "PMG_F_" + k), v)
    for x in (m, S):
        x.set_params(max_citer=4)
        x.init()
    for _ in range(2):
        rm, nm, cm = m.vcycle()
        rs, ns, cs = S.vcycle()
        assert abs(rs - rm) <= 1e-12 * rm and cs == cm
        assert np.allclose(ns, nm, rtol=1e-12, atol=0)
    assert np.array_equal(S.download(S.nlev, pm.PMG_F_U), m.field(m.nlev, O.F_U))
    S.close()
