"""Several time steps per launch against the strip step (chosen by a
rows-per-segment request) at the edges of its tiles of 24 x 8 cells: forward
seismograms, gradients, misfits, energy maps, pseudo-Hessian and fields must
be the same bits, and the gradient the oracle's.  Records end at every place
inside a launch, and the longest replay captured launches."""
import numpy as np
import pytest

from common import oracle, product
from test_gpu_tile import FL, _inputs, _run, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,fdorder,free_surf,boundary,shots,snap,dtinv,two,nt", [
    (48, 24, 4, 0, 0, 1, 0, 1, False, 150),
    (47, 25, 4, 1, 0, 3, 0, 2, True, 149),
    (49, 23, 2, 0, 0, 2, 0, 3, False, 151),
    (97, 40, 4, 0, 0, 3, 0, 5, False, 162),
    (64, 41, 2, 1, 0, 4, 0, 4, True, 150),
    (128, 33, 4, 1, 1, 2, 0, 2, False, 150),   # periodic: the narrowest grid on tiles
    (130, 40, 2, 0, 1, 3, 0, 1, True, 149),
    (65, 39, 4, 0, 0, 2, 1, 2, False, 150),    # 16-bit snapshots: recording passes only
    (70, 24, 4, 1, 0, 1, 2, 2, False, 3),      # shorter than a launch
    (24, 24, 4, 0, 0, 1, 0, 1, False, 5),
    (576, 64, 4, 0, 0, 4, 0, 3, False, 40),    # 768 workgroups: the most for a gradient
    (577, 64, 4, 0, 0, 4, 0, 3, False, 40),    # 800: forward several steps, gradient tiles
    (1104, 88, 2, 0, 0, 4, 0, 2, False, 40),   # 2024 of FDORDER 2
])
def test_several_steps_equal_strips(nx, ny, fdorder, free_surf, boundary, shots, snap, dtinv, two, nt):
    say("several steps", nx, ny, "FDORDER", fdorder, "shots", shots, "steps", nt)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=0, free_surf=free_surf, boundary=boundary, snap=snap, dtinv=dtinv, fw=8)
    inp = list(_inputs(nx, ny, shots, nt, seed=nx + ny))
    inp[8] = np.maximum(1, nt - np.arange(shots)).astype(np.int32)
    dn = product()
    a = _run(dn, par, inp, 0, two)
    b = _run(dn, par, inp, 13, two)
    assert np.isfinite(a[2]).all() and (nt < 40 or np.abs(a[2]).max() > 0)
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), "output %d differs" % k


@pytest.mark.parametrize("nx,ny,fdorder", [(65, 33, 4), (40, 30, 2)])
def test_several_steps_equal_oracle(nx, ny, fdorder):
    from pyoracle import make_cfg
    say("several steps against the oracle", nx, ny)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=0, free_surf=0, boundary=0, snap=0, dtinv=2, fw=8)
    inp = list(_inputs(nx, ny, 2, 62, seed=3))
    inp[8] = np.full(2, 62, np.int32)
    vs, rho, _, sig, si, sj, ri, rj, _, obs = inp
    got = _run(product(), par, inp, 0, False)
    cfg = make_cfg(nx, ny, fdorder=fdorder, fw=8, free_surf=0, L=0, nt=62, dtinv=2, dt=1e-4, dh=0.25, damping=300.0,
                   fpml=40.0, fl=[])
    ref = oracle("f32").gradient(cfg, vs, rho, None, si, sj, sig, ri, rj, obs)
    assert np.array_equal(got[2], ref["grad_vs"]) and np.array_equal(got[3], ref["grad_rho"])


@pytest.mark.parametrize("nx,ny,fdorder,L,free_surf,boundary,shots,dtinv,two", [
    (48, 24, 4, 2, 0, 0, 1, 1, False),
    (49, 25, 2, 3, 1, 0, 3, 2, True),
    (97, 40, 6, 0, 0, 0, 3, 5, False),
    (63, 33, 6, 3, 0, 0, 2, 3, True),
    (71, 41, 8, 2, 0, 0, 2, 4, False),
    (72, 40, 8, 1, 1, 0, 1, 3, False),
    (130, 39, 8, 0, 0, 1, 2, 2, True),
    (128, 47, 4, 1, 1, 1, 4, 2, False),
    (24, 24, 8, 3, 0, 0, 1, 1, False),
])
def test_several_higher_order_and_viscoelastic_steps_equal_strips(nx, ny, fdorder, L, free_surf, boundary, shots, dtinv,
                                                                  two):
    say("several steps", nx, ny, "FDORDER", fdorder, "L", L, "shots", shots)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=free_surf, boundary=boundary, snap=0, dtinv=dtinv, fw=8)
    inp = list(_inputs(nx, ny, shots, 150, seed=nx + ny))
    inp[8] = (150 - np.arange(shots)).astype(np.int32)
    dn = product()
    a = _run(dn, par, inp, 0, two)
    b = _run(dn, par, inp, 13, two)
    assert np.isfinite(a[2]).all() and np.abs(a[2]).max() > 0
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), "output %d differs" % k


@pytest.mark.parametrize("nx,ny,fdorder,L", [(65, 33, 8, 2), (70, 41, 6, 1), (50, 30, 4, 3)])
def test_several_viscoelastic_steps_equal_oracle(nx, ny, fdorder, L):
    from pyoracle import make_cfg
    say("several steps against the oracle", nx, ny, "FDORDER", fdorder, "L", L)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=0, boundary=0, snap=0, dtinv=2, fw=8)
    inp = list(_inputs(nx, ny, 2, 62, seed=3))
    inp[8] = np.full(2, 62, np.int32)
    vs, rho, qs, sig, si, sj, ri, rj, _, obs = inp
    got = _run(product(), par, inp, 0, False)
    cfg = make_cfg(nx, ny, fdorder=fdorder, fw=8, free_surf=0, L=L, nt=62, dtinv=2, dt=1e-4, dh=0.25, damping=300.0,
                   fpml=40.0, fl=FL[:L])
    ref = oracle("f32").gradient(cfg, vs, rho, qs, si, sj, sig, ri, rj, obs)
    assert np.array_equal(got[2], ref["grad_vs"]) and np.array_equal(got[3], ref["grad_rho"])


# ny below 2 FW under a free surface: the bottom frame reaches rows that would
# belong to the top one if there were one
SHALLOW = [(64, 12, 4, 0), (64, 15, 4, 2), (49, 8, 2, 0), (70, 15, 8, 2), (65, 12, 6, 1), (47, 16, 8, 3), (130, 9, 2, 3)]


@pytest.mark.parametrize("nx,ny,fdorder,L", SHALLOW)
def test_several_steps_of_shallow_free_surface_grids_equal_strips(nx, ny, fdorder, L):
    say("several steps, shallow", nx, ny, "FDORDER", fdorder, "L", L)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=1, boundary=0, snap=0, dtinv=2, fw=8)
    inp = list(_inputs(nx, ny, 2, 90, seed=nx + ny))
    inp[8] = np.array([90, 89], np.int32)
    dn = product()
    a = _run(dn, par, inp, 0, False)
    b = _run(dn, par, inp, 13, False)
    assert np.isfinite(a[2]).all() and np.abs(a[2]).max() > 0
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), "output %d differs" % k


@pytest.mark.parametrize("nx,ny,fdorder,L", SHALLOW)
def test_several_steps_of_shallow_free_surface_grids_equal_oracle(nx, ny, fdorder, L):
    from pyoracle import make_cfg
    say("several steps against the oracle, shallow", nx, ny, "FDORDER", fdorder, "L", L)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=1, boundary=0, snap=0, dtinv=2, fw=8)
    inp = list(_inputs(nx, ny, 2, 62, seed=3))
    inp[8] = np.full(2, 62, np.int32)
    vs, rho, qs, sig, si, sj, ri, rj, _, obs = inp
    got = _run(product(), par, inp, 0, False)
    cfg = make_cfg(nx, ny, fdorder=fdorder, fw=8, free_surf=1, L=L, nt=62, dtinv=2, dt=1e-4, dh=0.25, damping=300.0,
                   fpml=40.0, fl=FL[:L])
    ref = oracle("f32").gradient(cfg, vs, rho, qs if L else None, si, sj, sig, ri, rj, obs)
    assert np.array_equal(got[2], ref["grad_vs"]) and np.array_equal(got[3], ref["grad_rho"])


@pytest.mark.parametrize("nx,ny,fdorder,L,shots", [
    (70, 40, 4, 2, 34),     # 15 workgroups a shot, 510 of 512: second halves for every shot
    (70, 40, 4, 2, 35),     # one shot more: tiles, and several steps for one shot alone
    (60, 24, 8, 3, 29),     # 9 workgroups a shot, 261 of 256
    (60, 24, 2, 0, 30),
])
def test_batches_around_the_second_halves_equal_strips(nx, ny, fdorder, L, shots):
    say("several steps, batch of", shots, nx, ny, "FDORDER", fdorder, "L", L)
    par = dict(nx=nx, ny=ny, fdorder=fdorder, L=L, free_surf=0, boundary=0, snap=0, dtinv=2, fw=8)
    inp = _inputs(nx, ny, shots, 60, seed=shots)
    dn = product()
    a = _run(dn, par, inp, 0, False)
    b = _run(dn, par, inp, 13, False)
    assert np.isfinite(a[2]).all() and np.abs(a[2]).max() > 0
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y), "output %d differs" % k
