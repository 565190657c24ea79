"""Device-created traces and batches with an ACIS FEF file: the stage kernels
that hand their survivors on densely (the mirror to an LETG grating, a grating
to the detector) and make the photons fresh at the mirror's entry, which only a
run with a FEF file takes.  With the synthetic FEF of tests/fefgen.py:

- a trace against the stages on a host list (marx_create_photons and the three
  stage calls) and against the allocation-free trace, which use neither, record
  for record;
- a batch against the CPU oracle, and its graph launches against eager passes;
- the reflection at 2, 3 and 4 waves a SIMD on a host list, record for record."""
import numpy as np
import pytest

from marx_amd import Photons, Tracer, offaxis_directions, on_axis_photons
from tests.fefgen import write_fef
from tests.parity import compare
from tests.test_gpu_batch import ON_AXIS, _download, _oracle, assert_same_records, keep_schedule   # noqa: F401
from tests.test_gpu_passes import _same

RUNS = [("HETG", "ACIS-S", "POINT", "INTERNAL"), ("LETG", "ACIS-S", "DISK", "INTERNAL"), ("NONE", "ACIS-I", "POINT", "NONE"),
        ("HETG", "ACIS-I", "GAUSS", "NONE")]


def _tracer(tmp_path, grating, det, shape, dither):
    path = write_fef(str(tmp_path / "fef.fits"), range(0, 4) if det == "ACIS-I" else range(4, 10), split=256)
    par = {"DISK": {"S-DiskTheta0": 0.0, "S-DiskTheta1": 60.0}, "GAUSS": {"S-GaussSigma": 20.0}}.get(shape, {})
    t = Tracer(seed=61, GratingType=grating, DetectorType=det, SourceType=shape, SpectrumType="FLAT", MinEnergy=0.3,
               MaxEnergy=9.0, DitherModel=dither, ACISFEFFile=path, **par, **ON_AXIS)
    t.init_source(SourceFlux=60_000 / (1.0e4 * t.geometric_area))
    return t


@pytest.mark.gpu
@pytest.mark.parametrize("grating,det,shape,dither", RUNS)
@pytest.mark.parametrize("n,exposure", [(60_011, -1.0), (60_011, 4.0e3), (255, -1.0)])
def test_trace(gpu, tmp_path, grating, det, shape, dither, n, exposure):
    t = _tracer(tmp_path, grating, det, shape, dither)
    ncol, ndet, rec = _same(t, n, exposure=exposure, tag_start=3)
    assert t.pass_ms() == [0.0, 0.0, 0.0]          # the stages are kernels of their own
    p = Photons(n)
    p.pt.tag_start, p.pt.start_time = 3, 20.0
    assert t.create_photons(p, n, exposure if exposure > 0.0 else None) == ncol
    t.reflect(p)
    if grating != "NONE":
        t.diffract(p)
    t.detect(p)
    assert_same_records(rec, p.active[:ncol].copy(), f"{grating} + {det} with a FEF file")
    alive = (rec["flags"] & 0xFF) == 0
    assert alive.sum() == ndet
    assert n < 1000 or ((rec["pulse_height"][alive] > 100).any() and ndet > 100)


@pytest.mark.gpu
@pytest.mark.parametrize("grating,det,shape,dither", RUNS)
def test_batch(gpu, tmp_path, grating, det, shape, dither):
    t = _tracer(tmp_path, grating, det, shape, dither)
    rng = np.random.default_rng(8)
    dirs = offaxis_directions(np.radians(rng.uniform(0, 5, 30) / 60), rng.uniform(0, 2 * np.pi, 30))
    counts = rng.integers(0, 4000, 30).astype(np.uint32)
    n = int(counts.sum())
    for tag in (1000, 5):
        ndet, _ = t.trace_batch(dirs, counts, tag_start=tag, start_time=500.0, exposure=3.0e4, use_graph=False)
        got = _download(t, n)
        want = _oracle(t, dirs, counts, tag, 500.0, 3.0e4, grating)
        compare(got, want, max_flips=2, label=f"batch {grating} + {det} with a FEF file")
        same = got["flags"] == want["flags"]
        # two photons may take another component of the mixture (tests/test_gpu_fef.py)
        assert (got["pulse_height"][same] != want["pulse_height"][same]).sum() <= 2
        assert ndet == ((got["flags"] & 0xFF) == 0).sum()
        for replay in range(3):
            t.trace_batch(dirs, counts, tag_start=tag, start_time=500.0, exposure=3.0e4, use_graph=True)
            assert_same_records(_download(t, n), got, f"graph launch {replay}")


@pytest.mark.gpu
def test_waves_of_the_reflection(gpu, keep_schedule):   # noqa: F811
    t = Tracer(seed=62, GratingType="NONE", DetectorType="NONE")
    n = 50_021
    rec = on_axis_photons(n, np.random.default_rng(1).uniform(0.1, 10.0, n))
    out = []
    for waves in (4, 2, 3):
        t.set_schedule(reflect_waves=waves)
        p = Photons(n)
        p.load(rec)
        t.reflect(p)
        out.append(p.active.copy())
    assert_same_records(out[1], out[0], "2 waves")
    assert_same_records(out[2], out[0], "3 waves")
