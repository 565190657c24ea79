"""Angles and phases of any size in the source, where the short sine and cosine
end (2^20 radians, 2^31 quarter turns, 2^50 radians): the tails of a beta
profile, a wide Gaussian, dither phases after many periods; against the CPU
oracle."""
import numpy as np
import pytest

from marx_amd import Photons, Tracer
from oracle.oracle import Oracle, stream_uniforms
from tests.parity import DIR_TOL, compare
from tests.test_gpu_batch import ON_AXIS

N = 20_000
ARCSEC = np.pi / (180.0 * 3600.0)
STAGE_SOURCE = 1


def _create(t):
    pg, po = Photons(N), Photons(N)
    assert t.create_photons(pg, N) == Oracle(t).create_photons(po, N) == N
    return pg.active.copy(), po.active.copy()


def _radius_draws(seed):
    """The uniform that a photon's off-axis angle is made from: the energy and
    the azimuth come first (zero, which is drawn again, is not among these)."""
    u = np.array([stream_uniforms(seed, tag, STAGE_SOURCE, 3)[2] for tag in range(N)])
    assert (u > 0.0).all()
    return u


@pytest.mark.gpu
@pytest.mark.parametrize("shape,par,angle", [
    ("BETA", {"S-BetaCoreRadius": 10.0, "S-BetaBeta": 0.55},
     lambda u: 10.0 * ARCSEC * np.sqrt(u ** (1.0 / (1.5 - 1.65)) - 1.0)),
    ("BETA", {"S-BetaCoreRadius": 10.0, "S-BetaBeta": 0.51},
     lambda u: 10.0 * ARCSEC * np.sqrt(u ** (1.0 / (1.5 - 1.53)) - 1.0)),
    ("GAUSS", {"S-GaussSigma": 1.0e12}, lambda u: 1.0e12 * ARCSEC * np.sqrt(-np.log(u)))])
def test_profiles(gpu, shape, par, angle):
    t = Tracer(seed=71, source=True, GratingType="NONE", DetectorType="NONE", SourceType=shape, SpectrumType="FLAT",
               MinEnergy=1.0, MaxEnergy=2.0, DitherModel="NONE", **par, **ON_AXIS)
    a, b = _create(t)
    theta = angle(_radius_draws(71))
    assert (theta > 2.0 ** 20).sum() > 10 and np.isfinite(theta).all()
    assert np.abs(np.linalg.norm(a["p"], axis=1) - 1.0).max() < 1e-14
    # pow, log and the square root round an angle by a few of its last bits on
    # either side, which turns the direction by as much
    bound = DIR_TOL + 16.0 * 2.0 ** -53 * theta
    dp = np.abs(a["p"] - b["p"]).max(axis=1)
    assert (dp <= bound).all(), (dp / bound).max()
    assert (bound < 1e-3).sum() > N // 2


@pytest.mark.gpu
@pytest.mark.parametrize("period", [1.0e-2, 1.0e-5, 1.0e-13, np.inf])
def test_dither_after_many_periods(gpu, period):
    t = Tracer(seed=72, source=True, GratingType="NONE", DetectorType="NONE", SpectrumType="FLAT", MinEnergy=0.4,
               MaxEnergy=8.0, DitherModel="INTERNAL", DitherAmp_RA=20.0, DitherAmp_Dec=10.0, DitherAmp_Roll=60.0,
               DitherPeriod_RA=period, DitherPeriod_Dec=0.7 * period, DitherPeriod_Roll=1.3 * period, DitherPhase_RA=1.0,
               **ON_AXIS)
    a, b = _create(t)
    compare(a, b, max_flips=0, check_pixels=False, label=f"period {period}")
    # the state is the float of an angle that two sines may round apart in its last bit
    d = np.abs(a["dither"].view(np.int32).astype(np.int64) - b["dither"].view(np.int32))
    assert np.isfinite(a["dither"]).all() and d.max() <= 1 and (d > 0).mean() < 1e-4
