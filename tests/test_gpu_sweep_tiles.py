"""The separate kernels of a cycle -- the sweep's tile variants, the fused
residual + injection -- where the cycle really launches them: V(3,2) cycles,
whose levels never take the one-launch legs, against the oracle; sweeps alone in
both precisions against the same operations in numpy; the FP32 sweep of a zero
guess against pairs of sweeps, which read the zeros.  All bit for bit, with the
variable coefficient (in the LDS ring where it fits and from memory where not),
excision, spacings that are and are not powers of two, sides that leave
remainders of every tile and marches of one plane, of a few and of all."""
from functools import lru_cache

import numpy as np
import pytest

import oracle as O
import pamr_amrd_amd as pm
from pamr_amrd_amd import hierarchy as H

pytestmark = pytest.mark.gpu

SHAPE = (145, 33, 41)  # two columns of the widest tile, 19 x 5 x 6 on the coarsest level
DYADIC, OTHER = (0.0, 4.5, 0.0, 1.0, 0.0, 1.25), (0.0, 1.0, -0.1, 0.4, 0.0, 0.3)
CYCLE = {"pre": 3, "pst": 2}


@lru_cache(maxsize=None)
def _data(op, shape=SHAPE):
    rng = np.random.default_rng(op)
    full = shape[::-1]
    d = {"RHO": rng.standard_normal(full), "U": rng.standard_normal(full)}
    if op:
        d["A"] = np.exp(0.3 * rng.standard_normal(full))
        d["C"] = -rng.random(full)
    return d


def _set(x, mod, op, ex, bbox, shape=SHAPE):
    box = np.array(bbox).reshape(3, 2)
    for lev in range(1, x.nlev + 1) if ex else ():
        ch = H.chr_on(x.shape(lev), bbox, [(box.mean(axis=1), 0.3 * (box[:, 1] - box[:, 0]).min())])
        if mod is O:
            x.field(lev, O.F_CHR)[:] = ch
        else:
            x.set_chr(lev, ch)
    for k, v in _data(op, shape).items():
        if mod is O:
            x.field(x.nlev, getattr(O, "F_" + k))[:] = v
        else:
            x.upload(x.nlev, getattr(pm, "PMG_F_" + k), v)
    x.set_params(**CYCLE)
    x.init()
    return x


def _solver(op, ex, bbox, shape=SHAPE):
    return _set(pm.Solver(0, bbox=bbox, op=op, do_ex=ex, ex=1.0, shape=shape), pm, op, ex, bbox, shape)


@lru_cache(maxsize=None)
def _oracle_cycle(op, ex, bbox, shape=SHAPE):
    """residual norm and, per level, u, rhs and res after one cycle"""
    m = _set(O.UniformMG(0, bbox=bbox, op=op, do_ex=ex, ex=1.0, shape=shape), O, op, ex, bbox, shape)
    r, _, _ = m.vcycle()
    names = ("U", "RHS", "RES")
    return r, [{k: np.array(m.field(lev, getattr(O, "F_" + k))) for k in names} for lev in range(1, m.nlev + 1)]


def _same(S, want):
    for lev in range(1, S.nlev + 1):
        for k, v in want[lev - 1].items():
            if lev < S.nlev or k == "U":
                assert np.array_equal(S.download(lev, getattr(pm, "PMG_F_" + k)), v), (lev, k)


@pytest.mark.parametrize("ex", [0, 1])
@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("variant", range(12))
def test_tile_variants_in_cycles(torch_cuda, variant, op, ex):
    for bbox, z in ((DYADIC, variant % 7 + 1), (OTHER, 16)):
        print(f"case sweep variant {variant} z={z} op={op} ex={ex} bbox={bbox}", flush=True)
        r, want = _oracle_cycle(op, ex, bbox)
        S = _solver(op, ex, bbox)
        S.set_sweep_config(variant, z)
        rs, _, _ = S.vcycle()
        assert abs(rs - r) <= 1e-12 * r
        _same(S, want)
        S.close()


def _relax(u, rho, rhs, a, c, upd, h, sweeps):
    """red-black sweeps with the kernels' operations in u's type"""
    t = u.dtype.type
    h = [t(v) for v in h]
    d2 = [v * v for v in h]
    jc = t(-2) / d2[0] - t(2) / d2[1] - t(2) / d2[2]
    k, j, i = np.indices(u.shape)

    def at(f, dx, dy, dz):
        n = f.shape
        return f[1 + dz:n[0] - 1 + dz, 1 + dy:n[1] - 1 + dy, 1 + dx:n[2] - 1 + dx]

    def nb(f):
        return [at(f, *o) for o in ((0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1))]

    u = u.copy()
    half, two = t(0.5), t(2)
    for _ in range(sweeps):
        for p in (0, 1):
            uc, ue, uw, un, us, ut, ub = nb(u)
            if a is None:
                x, y, z = ((ue - two * uc) + uw) / d2[0], ((un - two * uc) + us) / d2[1], ((ut - two * uc) + ub) / d2[2]
                res = (((x + y) + z) - at(rho, 0, 0, 0)) - at(rhs, 0, 0, 0)
                new = uc - res * (t(1) / jc) if t is np.float32 else uc - res / jc
            else:
                ac, ae, aw, an, as_, at_, ab = nb(a)
                cc = at(c, 0, 0, 0)
                fe, fw, fn, fs, ft, fb = (half * (ac + v) for v in (ae, aw, an, as_, at_, ab))
                x = (fe * (ue - uc) - fw * (uc - uw)) / d2[0]
                y = (fn * (un - uc) - fs * (uc - us)) / d2[1]
                z = (ft * (ut - uc) - fb * (uc - ub)) / d2[2]
                jac = ((-(fe + fw) / d2[0] - (fn + fs) / d2[1]) - (ft + fb) / d2[2]) + cc
                res = ((((x + y) + z) + cc * uc) - at(rho, 0, 0, 0)) - at(rhs, 0, 0, 0)
                new = uc - res / jac
            on = at(upd & ((i + j + k + p) % 2 == 1), 0, 0, 0)
            uc[on] = new[on]
    return u


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("ex", [0, 1])
@pytest.mark.parametrize("op", [0, 1])
def test_tile_variants_alone(torch_cuda, op, ex, prec):
    """two sweeps of the finest level (no rhs) and of the one below, whose rhs
    the cycle before has left"""
    for bbox in (DYADIC, OTHER):
        S = _solver(op, ex, bbox)
        S.solve_rel(1, 0.0, 1) if prec else S.vcycle()
        t = np.float32 if prec else np.float64
        box = np.array(bbox).reshape(3, 2)
        rng = np.random.default_rng(7)
        for lev in (S.nlev, S.nlev - 1):
            shape = S.shape(lev)
            fine = lev == S.nlev
            h = [(x0 + (x1 - x0) / (n - 1)) - x0 for (x0, x1), n in zip(box, shape[::-1])]
            upd = np.zeros(shape, dtype=bool)
            upd[1:-1, 1:-1, 1:-1] = True
            if ex:
                upd &= H.chr_on(shape, bbox, [(box.mean(axis=1), 0.3 * (box[:, 1] - box[:, 0]).min())]) != 1.0
            a, c = (S.download(lev, f).astype(t) for f in (pm.PMG_F_A, pm.PMG_F_C)) if op else (None, None)
            rhs = np.zeros(shape, t) if fine else S.download32(lev, 2) if prec else S.download(lev, pm.PMG_F_RHS)
            assert fine or rhs.any()
            u0, rho = (rng.standard_normal(shape).astype(t) for _ in range(2))
            if prec:  # corrections are 0 on the faces; an upload goes to one of the two buffers
                u0[[0, -1]], u0[:, [0, -1]], u0[:, :, [0, -1]] = 0, 0, 0
            want = _relax(u0, rho, rhs, a, c, upd, h, 2)
            for variant in range(12):
                for z in (1, variant % 5 + 2, 64):
                    print(f"case sweep alone op={op} ex={ex} prec={prec} level {lev} variant {variant} z={z}", flush=True)
                    S.set_sweep_config(variant, z)
                    if prec:
                        S.upload32(lev, 0, u0)
                        S.upload32(lev, 1, rho)
                    else:
                        S.upload(lev, pm.PMG_F_U, u0)
                        S.upload(lev, pm.PMG_F_RHO, rho)
                    S.time_kernel(0, lev, prec, 2)
                    got = S.download32(lev, 0) if prec else S.download(lev, pm.PMG_F_U)
                    assert np.array_equal(got, want), (variant, z)
        S.close()


@pytest.mark.parametrize("op,ex", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("variant", [1, 5, 6, 9, 11])
def test_zero_guess_sweeps(torch_cuda, variant, op, ex):
    """FP32 cycles whose first sweep takes its guess as zero, and whose first
    pair of sweeps reads the zeros: the same u after mixed iterations and after
    FGMRES with two cycles an application"""
    n = 81
    bbox = (0.0, 1.0, 0.0, 1.0, 0.0, 1.0)
    out = []
    for pairs in (False, True):
        print(f"case zero guess variant {variant} op={op} ex={ex} pairs={pairs}", flush=True)
        S = _solver(op, ex, bbox, (n, n, n))
        S.set_params(pre=2, pst=2)
        S.set_sweep_config(variant, 8)
        S.set_sweep_blocking(pairs, 16)
        S.set_fgmres_prec_cycles(2)
        S.solve_rel(1, 0.0, 2)
        u = S.download(S.nlev, pm.PMG_F_U)
        S.solve_fgmres(2, 1e-12, 2)
        out.append((u, S.download(S.nlev, pm.PMG_F_U)))
        S.close()
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("op", [0, 1])
@pytest.mark.parametrize("shape,bbox", [(SHAPE, DYADIC), ((33, 81, 65), OTHER)])
def test_residual_injection_kinds(torch_cuda, shape, bbox, op):
    """separate kernels, the residual planes in a ring, the restriction streamed
    with one and two planes in flight; FP32 by the u two mixed iterations give"""
    r, want = _oracle_cycle(op, 0, bbox, shape)
    mixed = []
    for kind in (0, 1, 2, 3):
        for cz in (1, 3, 16) if kind else (8,):
            print(f"case residual + injection kind {kind} cz={cz} {shape} op={op}", flush=True)
            S = _solver(op, 0, bbox, shape)
            S.set_restrict_fusion(kind)
            for prec in (0, 1):
                S.set_resid_restrict_zchunk(prec, cz)
            rs, _, _ = S.vcycle()
            assert abs(rs - r) <= 1e-12 * r
            _same(S, want)
            S.solve_rel(1, 0.0, 2)
            mixed.append(S.download(S.nlev, pm.PMG_F_U))
            S.close()
    assert all(np.array_equal(u, mixed[0]) for u in mixed)
