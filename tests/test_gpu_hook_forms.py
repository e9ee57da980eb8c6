"""The application hooks over the grids where their index can go wrong: one
interior point, rows of one point, even and odd rows (the colours then hold
different counts), sizes around one block's places and around the change from
one to two places a thread, no point active -- grid functions bit for bit
against the oracle."""
import numpy as np
import pytest

import oracle as O
import pamr_amrd_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 3, 3), (3, 40, 3), (3, 3, 1030), (514, 3, 3), (515, 4, 3),
                                   (1027, 3, 4), (10, 66, 4), (67, 18, 34), (130, 66, 66),
                                   (263, 67, 66)])
@pytest.mark.parametrize("op,on", [(0, 1.0), (1, 0.7), (1, 0.0)])
def test_hook_forms(torch_cuda, shape, op, on):
    torch = torch_cuda
    nx, ny, nz = shape
    print(f"case hook form op={op} on={on} shape={shape}", flush=True)
    rng = np.random.default_rng(nx + 3 * ny + 7 * nz + op)
    f = {k: rng.standard_normal((nz, ny, nx)) for k in ("V", "rho", "rhs")}
    f["a"] = np.exp(0.5 * rng.standard_normal((nz, ny, nx)))
    f["c"] = rng.random((nz, ny, nx))
    f["cm"] = np.where(rng.random((nz, ny, nx)) < on, 1.0, 0.0)
    d = {k: torch.from_numpy(v).to("cuda") for k, v in f.items()}
    h = (1.0 / (nx - 1), 0.7 / (ny - 1), 1.3 / (nz - 1))
    tail = (2.0, nx, ny, nz, *h)
    ho = [O.P(f["rho"]), O.P(f["a"]) if op else None, O.P(f["c"]) if op else None, O.P(f["cm"]), None]
    de = [pm.tptr(d["rho"]), pm.tptr(d["a"]) if op else None, pm.tptr(d["c"]) if op else None, pm.tptr(d["cm"]), None]
    nrm = torch.zeros(2, dtype=torch.float64, device="cuda")
    n0, n1 = (pm.tptr(nrm[k:]) for k in (0, 1))
    res, lop = torch.full_like(d["V"], 5.0), torch.full_like(d["V"], 5.0)
    L, OL = pm.lib(), O.lib()
    assert L.pmg_hook_relax(op, pm.tptr(d["V"]), pm.tptr(d["rhs"]), *de, *tail, n0, None) == 0
    assert L.pmg_hook_residual(op, pm.tptr(res), pm.tptr(d["rhs"]), pm.tptr(d["V"]), *de, *tail, n1, None) == 0
    assert L.pmg_hook_lop(op, pm.tptr(lop), pm.tptr(d["V"]), *de, *tail, None) == 0
    torch.cuda.synchronize()
    V, r, l = f["V"].copy(), np.full((nz, ny, nx), 5.0), np.full((nz, ny, nx), 5.0)
    ref = [OL.or_relax(op, O.P(V), O.P(f["rhs"]), *ho, *tail), OL.or_residual(op, O.P(r), O.P(f["rhs"]), O.P(V), *ho, *tail)]
    OL.or_lop(op, O.P(l), O.P(V), *ho, *tail)
    assert np.array_equal(d["V"].cpu().numpy(), V)
    assert np.array_equal(res.cpu().numpy(), r)
    assert np.array_equal(lop.cpu().numpy(), l)
    # sums of n non-negative terms in different orders agree to n eps
    n = (nx - 2) * (ny - 2) * (nz - 2)
    for got, want in zip(nrm.tolist(), ref):
        if f["cm"][1:-1, 1:-1, 1:-1].any() or not np.isnan(want):
            assert abs(got - want) <= (n + 4) * 2.0 ** -52 * abs(want), (got, want)
        else:
            assert np.isnan(got)
