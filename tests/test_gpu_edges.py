"""The chunked residual, smooth2 and Gaussian kernels at the edges of their
chunks, row groups and pair tables, bit for bit against the oracle."""
import sys

import numpy as np
import pytest

from common import oracle, product
from test_gpu_misfit import oracle_residual

pytestmark = pytest.mark.gpu

O32 = oracle("f32")


def say(*a):
    print(*a)
    sys.stdout.flush()


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("ntr,ns", [(1, 127), (15, 128), (16, 129), (17, 256), (33, 257), (50, 64), (2, 1000)])
def test_residual_chunks(ntr, ns):
    say("residual", ntr, ns)
    rng = np.random.default_rng(ntr + ns)
    syn = rng.standard_normal((ntr, ns)).astype(np.float32)
    obs = (syn + 0.3 * rng.standard_normal((ntr, ns))).astype(np.float32)
    diff, l2, en, ob = product().calc_res(syn, obs, 1e-4)
    rdiff, rl2, ren, rob = oracle_residual(syn, obs, float(np.float32(1e-4)))
    assert np.array_equal(diff, rdiff) and np.array_equal(ob, rob)
    # the sums of a trace run in sample order; only the order over traces differs
    assert abs(l2 - rl2) <= 1e-12 * abs(rl2) and abs(en - ren) <= 1e-12 * abs(ren)


@pytest.mark.parametrize("nx,ny", [(2, 3), (129, 17), (130, 18), (128, 16), (257, 34), (145, 66), (100, 97), (64, 98)])
def test_smooth2_chunks(nx, ny):
    say("smooth2", nx, ny)
    g = np.random.default_rng(nx * ny).standard_normal((ny, nx)).astype(np.float32)
    for wd in (1.5, 11.0):
        assert np.array_equal(bits(product().smooth2(g, wd)), bits(O32.smooth2(g, wd)))


@pytest.mark.parametrize("name,ny,nx,wd,wd1,fc,lo,hi", [
    ("a jump at every cell", 20, 130, 0.3, 0.25, 20.0, 60.0, 500.0),
    ("more pairs than the table takes", 70, 130, 1.1, 0.9, 5.0, 20.0, 600.0),
    ("one pair", 9, 65, 0.3, 0.3, 25.0, 200.0, 200.0),
])
def test_gauss_pairs(name, ny, nx, wd, wd1, fc, lo, hi):
    say("gauss_filt_var", name)
    rng = np.random.default_rng(4)
    vel = rng.uniform(lo, hi, (ny, nx)).astype(np.float32)
    g = rng.standard_normal((ny, nx)).astype(np.float32)
    got = product().gauss_filt_var(g, vel, 0.25, wd, wd1, fc)
    assert np.array_equal(bits(got), bits(O32.gauss_filt_var(g, vel, 0.25, wd, wd1, fc)))


def test_gauss_out_of_range_is_refused():
    dn = product()
    vel = np.full((20, 70), 200.0, np.float32)
    vel[7, 33] = np.nan
    with pytest.raises(dn.DeniseError):
        dn.gauss_filt_var(np.ones((20, 70), np.float32), vel, 0.25, 0.3, 0.3, 25.0)
    vel[7, 33] = 1e6
    with pytest.raises(dn.DeniseError):
        dn.gauss_filt_var(np.ones((20, 70), np.float32), vel, 0.25, 0.3, 0.3, 25.0)


@pytest.mark.parametrize("ntr,ns", [(1, 2), (3, 3), (5, 64), (9, 65), (16, 130), (17, 300), (2, 5000), (7, 9000), (1, 40000)])
def test_stf_passes(ntr, ns):
    """Transform lengths 2^3 to 2^18: one, two and three passes, the last of
    one to seven stages; trace counts around the eight read ahead.  The bound
    is the float rounding of the regulariser and the output, as for the
    record lengths of the other STF tests."""
    import stf_oracle
    say("stf", ntr, ns)
    rng = np.random.default_rng(ns)
    syn = rng.standard_normal((ntr, ns)).astype(np.float32)
    obs = (0.7 * syn + 0.3 * rng.standard_normal((ntr, ns))).astype(np.float32)
    sig = rng.standard_normal(ns).astype(np.float32)
    got = product().stf(obs, syn, sig, eps_stf=0.05)
    want = stf_oracle.stf(obs, syn, sig, eps_stf=0.05)
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("ntr,ns,normalize", [(33, 5000, 0), (64, 5000, 1), (65, 4100, 2), (3, 140000, 2)])
def test_stf_batches(ntr, ns, normalize):
    """32 traces of 2^15 points to a batch, or one of 2^20: remainders of one
    trace, none, and muted traces on both sides of a batch's edge.  The bound
    is test_stf_passes'."""
    import stf_oracle
    say("stf batches", ntr, ns, normalize)
    rng = np.random.default_rng(ns + ntr)
    syn = rng.standard_normal((ntr, ns)).astype(np.float32)
    obs = (0.7 * syn + 0.3 * rng.standard_normal((ntr, ns))).astype(np.float32)
    sig = rng.standard_normal(ns).astype(np.float32)
    mute = np.zeros(ntr, np.uint8)
    mute[[1, min(31, ntr - 1)]] = 1
    got = product().stf(obs, syn, sig, mute=mute, eps_stf=0.05, normalize=normalize)
    want = stf_oracle.stf(obs, syn, sig, mute=mute, eps_stf=0.05, normalize=normalize)
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("nx,ny", [
    # unknowns of a row: 511, 512, 513, 528, 1024, 1099 (chunks of 512; last
    # chunks of 511, 512, 1, 16, 512 and 75)
    (512, 18), (513, 5), (514, 17), (529, 34), (1025, 3), (1100, 20),
    # unknowns of a column: 127, 128, 129, 257 (chunks of 128)
    (70, 128), (65, 129), (66, 130), (129, 258),
])
def test_smooth2_carries_between_chunks(nx, ny):
    say("smooth2, several chunks", nx, ny)
    g = np.random.default_rng(nx * ny).standard_normal((ny, nx)).astype(np.float32)
    for wd in (1.5, 11.0):
        assert np.array_equal(bits(product().smooth2(g, wd)), bits(O32.smooth2(g, wd)))
