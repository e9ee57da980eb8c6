"""The one-launch legs of the levels below an AMR hierarchy's base, against the
multi-patch oracle: V(2,2) cycles (legs) before and after a V(3,2) cycle
(separate kernels), spacings whose squares are powers of two and others, with
and without refined levels -- u of every level bit for bit, the norms of every
level within their summation order, FP32 cycles of the mixed solve down to the
FP64 cycles' solution."""
import numpy as np
import pytest

import oracle as O
import pamr_amrd_amd as pm
from pamr_amrd_amd import hierarchy as H

pytestmark = pytest.mark.gpu

UNIT = (0.0, 1.0, 0.0, 1.0, 0.0, 1.0)
BOX = (0.0, 1.3, -0.2, 0.7, 0.1, 1.2)


def sources(x, op, put):
    for L in range(x.base, x.nlev + 1):
        for g in range(x.ngrids(L)):
            shape, bb = x.grid(L, g)
            put(L, g, "rho", -H.gaussian_on(shape, bb, seed=31))
            if op == 1:
                put(L, g, "a", H.lognormal_on(shape, bb))
                put(L, g, "c", H.uniform_on(shape, bb))


@pytest.mark.parametrize("base_n,bbox,refined,op", [(33, BOX, False, 0), (33, BOX, False, 1), (65, UNIT, False, 0),
                                                    (33, UNIT, True, 1)])
def test_legs_bit_exact(torch_cuda, base_n, bbox, refined, op):
    print(f"case amr legs base={base_n} box={bbox} refined={refined} op={op}", flush=True)
    levels = H.random_boxes(base_n=base_n, nref=1, nmin=3, nmax=4, smin=9, smax=17, seed=3) if refined else []
    m, a = O.AmrMG(base_n, levels, bbox=bbox, op=op), pm.Amr(base_n, levels, bbox=bbox, op=op)

    def put(L, g, which, v):
        m.field(L, g, {"rho": O.OA_RHO, "a": O.OA_A, "c": O.OA_C}[which])[:] = v
        a.upload(L, g, {"rho": pm.PMG_F_RHO, "a": pm.PMG_F_A, "c": pm.PMG_F_C}[which], v)

    sources(m, op, put)
    for x in (m, a):
        x.set_params()
        x.init()
    for cycle, pre in enumerate((2, 2, 3, 2)):
        for x in (m, a):
            x.set_params(pre=pre)
        rm, nm, cm = m.vcycle()
        ra, na, ca = a.vcycle()
        assert cm == ca and abs(ra - rm) <= 1e-12 * rm, (cycle, ra, rm)
        assert np.allclose(na, nm, rtol=1e-12, atol=0), (cycle, na, nm)
        for L in range(1, m.nlev + 1):
            for g in range(m.ngrids(L)):
                assert np.array_equal(a.download(L, g, pm.PMG_F_U), m.field(L, g, O.OA_U)), (cycle, L, g)
    a.close()


@pytest.mark.parametrize("op", [0, 1])
def test_legs_fp32(torch_cuda, op):
    """65^3 without refinement: the mixed solve's FP64 residual reaches 1e-10
    of the first, its solution the FP64 solve's to 1e-9 (both satisfy the same
    discrete equation; a residual of 1e-10 leaves an error of about that), in the
    FP64 solve's number of cycles and at most one more (FP32 rounding of a cycle
    is far below its contraction)"""
    print(f"case amr legs fp32 op={op}", flush=True)
    out = []
    for mode, rtol in ((0, 1e-12), (1, 1e-10)):
        a = pm.Amr(65, [], op=op)
        sources(a, op, lambda L, g, which, v: a.upload(L, g, {"rho": pm.PMG_F_RHO, "a": pm.PMG_F_A,
                                                              "c": pm.PMG_F_C}[which], v))
        a.set_params()
        a.init()
        r0, h = a.solve_rel(mode, rtol, 60)
        assert len(h) and h[-1] <= rtol * r0
        out.append((a.download(a.base, 0, pm.PMG_F_U), int(np.argmax(np.asarray(h) <= 1e-10 * r0)) + 1))
        a.close()
    (u64, n64), (u32, n32) = out
    assert n32 <= n64 + 1
    assert np.abs(u32 - u64).max() <= 1e-9 * np.abs(u64).max()
