"""The one-launch legs of small levels (8^3 tiles with their halo in LDS)
against the oracle where the tiles have remainders: sides of one tile and a
point, unequal sides, spacings that are no power of two, nonzero boundary
data, excision, weights and restriction kinds other than the default.  Two
cycles; u, f_rhs, f_lop and f_res of every level bit for bit."""
import numpy as np
import pytest

import oracle as O
import pamr_amrd_amd as pm
from pamr_amrd_amd import hierarchy as H

pytestmark = pytest.mark.gpu


def _problem(shape, bbox, op, ex, par):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx * 7 + ny * 3 + nz + op)
    m = O.UniformMG(0, bbox=bbox, op=op, do_ex=ex, ex=1.0, shape=shape)
    S = pm.Solver(0, bbox=bbox, op=op, do_ex=ex, ex=1.0, shape=shape)
    assert m.nlev == S.nlev
    full = m.shape(m.nlev)
    if ex:
        box = np.array(bbox).reshape(3, 2)
        mid = box.mean(axis=1)
        for lev in range(1, m.nlev + 1):
            ch = H.chr_on(m.shape(lev), bbox, [(mid, 0.22 * (box[:, 1] - box[:, 0]).min())])
            m.field(lev, O.F_CHR)[:] = ch
            S.set_chr(lev, ch)
    data = {"RHO": rng.standard_normal(full), "U": rng.standard_normal(full)}
    if op == 1:
        data["A"] = np.exp(0.3 * rng.standard_normal(full))
        data["C"] = -rng.random(full)
    for k, v in data.items():
        m.field(m.nlev, getattr(O, "F_" + k))[:] = v
        S.upload(S.nlev, getattr(pm, "PMG_F_" + k), v)
    for x in (m, S):
        x.set_params(**par)
        x.init()
    return m, S


@pytest.mark.parametrize("shape,bbox,op,ex,par", [
    ((33, 33, 33), (0, 1, 0, 1, 0, 1), 0, 0, {}),
    ((17, 33, 25), (0, 1.1, 0, 0.9, -0.3, 1), 0, 0, {}),
    ((41, 17, 49), (0, 1, 0, 1, 0, 1), 1, 0, {"w0_r": 0.9, "w0_i": 1.1}),
    ((33, 65, 17), (0, 1, 0, 2, 0, 0.5), 0, 0, {"rop_u": 1, "rop_res": 3}),
    ((25, 33, 41), (0, 1, 0, 1, 0, 1), 0, 1, {}),
    ((33, 25, 33), (0, 1, 0, 1, 0, 1.3), 1, 1, {}),
])
def test_legs_match_oracle(torch_cuda, shape, bbox, op, ex, par):
    print(f"case small levels {shape} op={op} ex={ex}", flush=True)
    bbox = tuple(float(v) for v in bbox)
    m, S = _problem(shape, bbox, op, ex, par)
    for cyc in range(2):
        rm, nm, cm = m.vcycle()
        rs, ns, cs = S.vcycle()
        assert abs(rs - rm) <= 1e-12 * rm and cs == cm, cyc
        # FP64 sums of squares over at most 10^5 points in another order
        assert np.allclose(ns, nm, rtol=1e-12, atol=0)
    for lev in range(1, m.nlev + 1):
        for k in ("U", "RHS", "LOP", "RES"):
            if lev == m.nlev and k in ("RHS", "LOP"):
                continue  # zero on the finest level; not stored there
            got, want = S.download(lev, getattr(pm, "PMG_F_" + k)), m.field(lev, getattr(O, "F_" + k))
            assert np.array_equal(got, want), (lev, k)
    S.close()


@pytest.mark.parametrize("op,ex", [(0, 0), (1, 0), (1, 1)])
def test_fp32_legs_match_separate_kernels(torch_cuda, op, ex):
    """mixed-precision iterations at 65^3 with the finest level's legs in one
    launch and (paired sweeps on) as separate kernels: the same u"""
    print(f"case small levels fp32 op={op} ex={ex}", flush=True)
    out = []
    for paired in (False, True):
        _, S = _problem((65, 65, 65), (0.0, 1.0, 0.0, 1.0, 0.0, 1.0), op, ex, {})
        S.set_sweep_blocking(paired)
        _, h = S.solve_rel(1, 0.0, 3)
        out.append((S.download(S.nlev, pm.PMG_F_U), h))
        S.close()
    assert np.array_equal(out[0][0], out[1][0])
    assert np.allclose(out[0][1], out[1][1], rtol=1e-12, atol=0)
