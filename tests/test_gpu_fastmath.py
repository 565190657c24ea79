"""The stages' FP64 primitives (dev_math.h) where their shortcuts end: GPU
against the CPU oracle at the bars of tests/parity.py.

- surface tilts: the products with a surface's tilt matrices are left out
  when no shell tilts it; every surface, one of them, or none tilted;
- angles past the small-angle polynomials (2^-6 rad): mirror blurs of
  degrees, dither of degrees in every axis, a roll that varies;
- on-axis rays exactly along the axis, where the paraboloid's quadratic
  degenerates, and rays far off it;
- a source at a finite distance."""
import numpy as np
import pytest

from marx_amd import Photons, Tracer, offaxis_directions, on_axis_photons
from oracle.oracle import Oracle
from tests.parity import compare
from tests.test_cpu_pins_mirror import _rdb_with
from tests.test_gpu_source import ON_AXIS, _both

N = 60_000


def _reflect(t, rec, distance=0.0):
    pg, po = Photons(len(rec)), Photons(len(rec))
    for p in (pg, po):
        p.load(rec)
        p.pt.source_distance = distance
    t.reflect(pg)
    Oracle(t).reflect(po)
    return pg.active.copy(), po.active.copy()


@pytest.mark.gpu
@pytest.mark.parametrize("tilts", [{}, {"p3": (2.0e-3, -1.0e-3)}, {"h1": (-1.0e-3, 2.0e-3)},
                                   {f"{s}{n}": (3.0e-4 * k, -2.0e-4 * k) for s in "ph"
                                    for k, n in enumerate((1, 3, 4, 6), 1)}])
def test_tilted_surfaces(gpu, tmp_path, tilts):
    path = str(tmp_path / "geom.rdb")
    _rdb_with(path, tilts)
    t = Tracer(seed=3, GratingType="NONE", DetectorType="NONE", HRMA_Geometry_File=path)
    rec = on_axis_photons(N, 1.49, tag_start=77)
    a, b = _reflect(t, rec)
    compare(a, b, max_flips=2, label=f"tilts {tilts}")
    assert ((a["flags"] & 0xFF) == 0).mean() > 0.2


@pytest.mark.gpu
@pytest.mark.parametrize("blur", [0.0, 40.0, 20000.0])
def test_blur_of_any_size(gpu, blur):
    t = Tracer(seed=4, GratingType="NONE", DetectorType="NONE",
               **{f"{s}{n}Blur": blur for s in "PH" for n in (1, 3, 4, 6)})
    rec = on_axis_photons(N, 1.0)
    a, b = _reflect(t, rec)
    compare(a, b, max_flips=2, label=f"blur {blur}")


@pytest.mark.gpu
@pytest.mark.parametrize("arcmin", [0.0, 1.0e-6, 25.0, 120.0])
def test_rays_on_and_off_the_axis(gpu, arcmin):
    t = Tracer(seed=5, GratingType="NONE", DetectorType="NONE")
    rec = on_axis_photons(N, np.random.default_rng(1).uniform(0.1, 10.0, N))
    rec["p"] = offaxis_directions(np.full(N, np.radians(arcmin / 60.0)), np.linspace(0.0, 2.0 * np.pi, N))
    a, b = _reflect(t, rec)
    compare(a, b, max_flips=2, label=f"{arcmin} arcmin")


@pytest.mark.gpu
def test_source_at_a_finite_distance(gpu):
    t = Tracer(seed=6, GratingType="NONE", DetectorType="NONE")
    a, b = _reflect(t, on_axis_photons(N, 1.49), distance=5.3e5)
    compare(a, b, max_flips=2, label="finite distance")
    assert ((a["flags"] & 0xFF) == 0).any()


@pytest.mark.gpu
@pytest.mark.parametrize("amp", [0.0, 300.0, 20000.0])
def test_dither_of_any_size(gpu, amp):
    t = Tracer(seed=7, source=True, GratingType="NONE", DetectorType="NONE", SpectrumType="FLAT", MinEnergy=0.4,
               MaxEnergy=8.0, DitherModel="INTERNAL", DitherAmp_RA=amp, DitherAmp_Dec=0.7 * amp,
               DitherAmp_Roll=3.0 * amp, DitherPeriod_Roll=313.0, DitherPhase_RA=1.0, **ON_AXIS)
    pg, po = _both(t, N)
    compare(pg.active, po.active, max_flips=0, check_pixels=False, label=f"dither {amp}")
    assert np.array_equal(pg.active["arrival_time"], po.active["arrival_time"])
    # the state is the float of an angle that two sines may round apart in its last bit
    d = np.abs(pg.active["dither"].view(np.int32).astype(np.int64) - po.active["dither"].view(np.int32))
    assert d.max() <= 1 and (d > 0).mean() < 1e-5
