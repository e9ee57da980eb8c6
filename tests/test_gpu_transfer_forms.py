"""The one-thread-per-point transfer kernels over the forms their arguments
allow: segments inside larger arrays (pre-filled targets, anchors outside the
segment), ratios 1 to 4, unequal along the axes, strides other than 1, boxes
narrower than a thread row, one-line segments, dense excision masks -- bit for
bit against the oracle."""
import numpy as np
import pytest

import oracle as O
import pamr_amrd_amd as pm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dens", [0.0, 0.2, 0.7, 1.0])
@pytest.mark.parametrize("seg", [
    # (ni, nj, nk), coarse offset, fine offset, strides, ratios, extra
    ((5, 4, 6), (1, 1, 1), (1, 1, 1), (1, 1, 1), (2, 2, 2), 0),
    ((3, 2, 70), (5, 5, 5), (9, 9, 9), (1, 1, 1), (2, 2, 2), 7),
    ((70, 3, 2), (5, 5, 5), (13, 13, 13), (1, 1, 1), (3, 3, 3), 9),
    ((6, 5, 4), (5, 5, 5), (17, 13, 9), (1, 1, 1), (4, 3, 2), 12),
    ((4, 6, 5), (9, 9, 9), (9, 9, 9), (2, 2, 2), (2, 2, 2), 8),
    ((7, 1, 1), (5, 5, 5), (9, 9, 9), (1, 1, 1), (2, 2, 2), 6),
    ((6, 5, 1), (5, 5, 5), (9, 9, 9), (1, 1, 1), (2, 2, 2), 6),
    ((5, 5, 5), (5, 5, 5), (4, 4, 4), (1, 1, 1), (1, 1, 1), 3),
])
def test_trilinear_forms(torch_cuda, seg, dens):
    torch = torch_cuda
    n, o1, o2, st, rho, extra = seg
    print(f"case trilinear form {seg} density {dens}", flush=True)
    rng = np.random.default_rng(sum(n) * 31 + sum(rho) + int(100 * dens))
    # coarse arrays hold 4 more anchors past the segment, the reach of the
    # extrapolation (and of the reference's bounds check on n * stride)
    c = [max((o + m - 1) * s, o + (m + 3) * s) + 1 for o, m, s in zip(o1, n, st)]
    f = [o + (m - 1) * r + extra for o, m, r in zip(o2, n, rho)]
    u1, u2 = rng.standard_normal(c[::-1]), rng.standard_normal(f[::-1])
    chr_ = np.where(rng.random(c[::-1]) < dens, 1.0, 0.0)
    ex = int(dens > 0)
    args = [*c, *f, *o1, *o2, *n, *st, *rho, 2]
    ref = O.dminterp3d(u1.copy(), u2.copy(), args, chr1=chr_, ex=1.0, do_ex=ex)
    d1, d2, dc = (torch.from_numpy(a).cuda() for a in (u1, u2, chr_))
    assert pm.lib().pmg_dminterp3d(pm.tptr(d1), pm.tptr(d2), *args, pm.tptr(dc), 1.0, ex, None) == 0
    assert np.array_equal(d2.cpu().numpy(), ref)


@pytest.mark.parametrize("seg", [((3, 70, 2), (2, 3, 1), (1, 2, 3)), ((130, 2, 3), (1, 1, 1), (2, 1, 1)),
                                 ((1, 1, 5), (3, 2, 2), (1, 1, 1))])
@pytest.mark.parametrize("kind", ["copy", "fw", "hw", "fw_ex"])
def test_box_forms(torch_cuda, seg, kind):
    torch = torch_cuda
    n, o1, st2 = seg
    print(f"case box form {kind} {seg}", flush=True)
    rng = np.random.default_rng(sum(n) + len(kind))
    s1 = (2, 2, 2)
    a = [o + (m - 1) * 2 + 1 for o, m in zip(o1, n)]
    b = [2 + (m - 1) * s + 2 for m, s in zip(n, st2)]
    u1, u2 = rng.standard_normal(a[::-1]), rng.standard_normal(b[::-1])
    chr_ = np.where(rng.random(a[::-1]) < 0.3, 1.0, 0.0)
    args = [*a, *b, *o1, 2, 2, 2, *n, *s1, *st2]
    ref = u2.copy()
    d1, d2, dc = (torch.from_numpy(v).cuda() for v in (u1, u2, chr_))
    OL, L = O.lib(), pm.lib()
    if kind == "copy":
        OL.or_dmcopy3d(O.P(u1), O.P(ref), *args)
        rc = L.pmg_dmcopy3d(pm.tptr(d1), pm.tptr(d2), *args, None)
    else:
        ex, name = int(kind == "fw_ex"), "dm" + kind[:2] + "r3d"
        getattr(OL, "or_" + name)(O.P(u1), O.P(ref), *args, O.P(chr_), 1.0, ex)
        rc = getattr(L, "pmg_" + name)(pm.tptr(d1), pm.tptr(d2), *args, pm.tptr(dc), 1.0, ex, None)
    assert rc == 0 and np.array_equal(d2.cpu().numpy(), ref)
