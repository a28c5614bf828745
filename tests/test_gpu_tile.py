"""The tile step against the strip step (chosen by a rows-per-segment
request) at the edges of its tiles: forward seismograms, gradients, misfits,
energy maps and pseudo-Hessian must be the same bits, and the gradient the
oracle's."""
import sys

import numpy as np
import pytest

from common import oracle, product

pytestmark = pytest.mark.gpu

FL = [6.25, 50.0, 12.0, 30.0]


def say(*a):
    print(*a)
    sys.stdout.flush()


def _inputs(nx, ny, shots, nt, seed):
    rng = np.random.default_rng(seed)
    vs = (120.0 + 200.0 * np.arange(ny)[:, None] / ny + 10.0 * rng.standard_normal((ny, nx))).astype(np.float32)
    rho = (1800.0 + 20.0 * rng.standard_normal((ny, nx))).astype(np.float32)
    qs = np.full((ny, nx), 20.0, np.float32)
    sig = (rng.standard_normal((shots, nt)) * 1e-2).astype(np.float32)
    # sources and receivers on both sides of the tile edges at columns 64 and rows 8 and 16
    cols = [c for c in (3, 62, 63, 64, 65, 66, nx // 2, nx - 2) if 1 <= c <= nx]
    rows = [r for r in (2, 7, 8, 9, 10, 16, 17, ny - 1) if 1 <= r <= ny]
    si = np.array([cols[s % len(cols)] for s in range(shots)], np.int32)
    sj = np.array([rows[(3 * s) % len(rows)] for s in range(shots)], np.int32)
    rec = [(c, r) for r in sorted(set(rows[1:6])) for c in sorted(set(cols))]
    ri, rj = np.array([c for c, _ in rec], np.int32), np.array([r for _, r in rec], np.int32)
    nts = np.array([nt - 5 * (s % 3) for s in range(shots)], np.int32)
    obs = (rng.standard_normal((shots, len(rec), nt)) * 1e-3).astype(np.float32)
    return vs, rho, qs, sig, si, sj, ri, rj, nts, obs


def _run(dn, par, inp, rows, multi):
    vs, rho, qs, sig, si, sj, ri, rj, nts, obs = inp
    ctx = dn.Context(par["nx"], par["ny"], fdorder=par["fdorder"], fw=par["fw"], free_surf=par["free_surf"], L=par["L"],
                     fl=FL[:par["L"]], dt=1e-4, dh=0.25, fpml=40.0, dtinv=par["dtinv"], snap_precision=par["snap"],
                     boundary=par["boundary"])
    ctx.set_batch(0, rows)
    ctx.set_model(vs, rho, qs if par["L"] else None)
    ctx.set_receivers(ri, rj)
    if multi:
        # two sources per shot
        off = np.arange(0, 2 * len(si) + 1, 2).astype(np.int32)
        ctx.set_shots_multi(off, np.repeat(si, 2) + np.tile([0, 1], len(si)).astype(np.int32) * (np.repeat(si, 2) < par["nx"]),
                            np.repeat(sj, 2), np.repeat(sig, 2, 0), nts)
    else:
        ctx.set_shots(si, sj, sig, nts)
    seis = ctx.forward()
    ctx.set_observed(obs)
    l2, en = ctx.gradient()
    out = [seis, np.array([l2, en])] + ctx.get_gradient() + list(ctx.energy_maps()) + list(ctx.pseudo_hessian())
    out += ctx.forward_fields(0, 30)
    ctx.close()
    return out


CONFIGS = [
    # nx, ny, fdorder, L, free_surf, boundary, shots, snap, dtinv, two sources per shot
    (64, 33, 8, 2, 1, 0, 2, 0, 2, False),
    (65, 40, 8, 2, 0, 0, 1, 1, 3, True),
    (63, 41, 12, 3, 0, 0, 3, 2, 4, False),
    (129, 47, 12, 4, 1, 0, 2, 0, 1, False),
    (130, 34, 2, 1, 0, 0, 1, 1, 2, True),
    (100, 48, 4, 0, 1, 0, 4, 0, 2, False),
    (190, 39, 6, 0, 0, 0, 1, 2, 2, False),
    (71, 36, 10, 2, 1, 0, 2, 0, 4, False),
    (128, 35, 8, 2, 1, 1, 2, 0, 2, False),     # periodic: the narrowest grid on tiles
    (133, 40, 12, 1, 0, 1, 1, 1, 2, True),
    (127, 40, 4, 0, 1, 1, 1, 0, 2, False),     # periodic: strips on both sides
    # more than 256 tiles of 16 rows: two rows per wave
    (140, 50, 8, 2, 0, 0, 24, 0, 4, False),
    (129, 65, 12, 3, 1, 0, 18, 1, 2, False),
    (66, 49, 2, 0, 0, 0, 33, 2, 3, False),
    (192, 40, 4, 1, 1, 1, 30, 0, 4, True),
]


@pytest.mark.parametrize("nx,ny,fdorder,L,free_surf,boundary,shots,snap,dtinv,multi", CONFIGS)
def test_tiles_equal_strips(nx, ny, fdorder, L, free_surf, boundary, shots, snap, dtinv, multi):
    say("tile step", nx, ny, "FDORDER", fdorder, "L", L, "shots", shots)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=free_surf, boundary=boundary, snap=snap, dtinv=dtinv, fw=8)
    inp = _inputs(nx, ny, shots, 90, seed=nx + ny)
    dn = product()
    a = _run(dn, par, inp, 0, multi)
    b = _run(dn, par, inp, 13, multi)
    assert np.abs(a[2]).max() > 0 and np.isfinite(a[2]).all()
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), "output %d differs" % k


@pytest.mark.parametrize("nx,ny,fdorder,L,shots", [(65, 49, 8, 2, 1), (130, 33, 4, 0, 30)])
def test_tiles_equal_oracle(nx, ny, fdorder, L, shots):
    from pyoracle import make_cfg
    say("tile step against the oracle", nx, ny)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=0, boundary=0, snap=0, dtinv=2, fw=8)
    vs, rho, qs, sig, si, sj, ri, rj, nts, obs = _inputs(nx, ny, shots, 60, seed=3)
    nts = np.full(shots, 60, np.int32)
    got = _run(product(), par, (vs, rho, qs, sig, si, sj, ri, rj, nts, obs), 0, False)
    cfg = make_cfg(nx, ny, fdorder=fdorder, fw=8, free_surf=0, L=L, nt=60, dtinv=2, dt=1e-4, dh=0.25, damping=300.0,
                   fpml=40.0, fl=FL[:L])
    ref = oracle("f32").gradient(cfg, vs, rho, qs if L else None, si, sj, sig, ri, rj, obs)
    assert np.array_equal(got[2], ref["grad_vs"]) and np.array_equal(got[3], ref["grad_rho"])


@pytest.mark.parametrize("nx,ny,fdorder,L,shots,dtinv", [
    (512, 33, 10, 0, 1, 2),     # one band of eight columns of tiles, one shot
    (513, 40, 8, 2, 3, 3),      # a band and one column, a pair of shots and one
    (600, 40, 8, 2, 4, 2),      # a band and two columns, two pairs
    (960, 35, 10, 1, 5, 4),     # a band and seven columns
    (1088, 60, 12, 2, 2, 3),    # two bands and one column
])
def test_order_of_tiles_equals_strips(nx, ny, fdorder, L, shots, dtinv):
    say("order of the tiles", nx, ny, "FDORDER", fdorder, "shots", shots)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=1, boundary=0, snap=0, dtinv=dtinv, fw=8)
    inp = _inputs(nx, ny, shots, 70, seed=nx + ny)
    dn = product()
    for x, y in zip(_run(dn, par, inp, 0, False), _run(dn, par, inp, 13, False)):
        assert np.array_equal(x, y)
