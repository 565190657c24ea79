"""The device-created trace as chunk kernels (mxg_trace_device, mxg_trace_batch)
against the stage kernels (mxg_trace_device_noalloc) bit for bit, and against
the CPU oracle.

- lengths around the wavefront, the block and the scan tile, with an exposure
  cut inside the chunk and none;
- every grating and detector, extended and point sources, uniform times;
- draws the entry repeats (closed quadrants, a shell with none open), where
  the mirror's stream goes on elsewhere than usual;
- batches with empty sources and sources of one photon, which the wave's
  source search steps over."""
import ctypes

import numpy as np
import pytest

from marx_amd import Photons, Tracer, offaxis_directions
from tests.parity import compare
from tests.test_gpu_batch import _oracle, assert_same_records
from tests.test_gpu_source import ON_AXIS, _both
from tests.test_zz_no_alloc import _columns, _records


def _tracer(grating="HETG", det="ACIS-S", shape="POINT", uniform=0.0, n=1000, seed=5, **par):
    t = Tracer(seed=seed, GratingType=grating, DetectorType=det, SourceType=shape, SpectrumType="FLAT", MinEnergy=0.3,
               MaxEnergy=8.0, DitherModel="INTERNAL", **par, **ON_AXIS)
    t.init_source(uniform_times=uniform, SourceFlux=n / (1.0e4 * t.geometric_area))
    return t


def _same(t, n, exposure=-1.0, tag_start=3):
    """Both traces of a chunk: (collected, detected, records)."""
    ncol, ndet, _ = t.trace_device(n, tag_start=tag_start, start_time=20.0, exposure_time=exposure)
    counts = t.stage_counts()
    p = Photons(n)
    t.download(p)
    want = p.active.copy()
    cols, view = _columns(n)
    c, d = ctypes.c_uint(), ctypes.c_uint()
    assert 0 == t.lib.mxg_trace_device_noalloc(ctypes.byref(view), n, tag_start, 20.0, exposure, ctypes.byref(c),
                                               ctypes.byref(d)), t.lib.mxg_last_error()
    assert (ncol, ndet) == (c.value, d.value)
    assert_same_records(want, _records(cols, ncol), f"n={n} exposure={exposure}")
    assert counts[0] == ncol and counts[3] == ndet
    return ncol, ndet, want


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 2047, 2048, 2049, 100_003])
@pytest.mark.parametrize("cut", [False, True])
def test_lengths(gpu, n, cut):
    t = _tracer(n=n)
    ncol, _, _ = _same(t, n, exposure=6.0e3 if cut else -1.0)
    assert ncol == n if not cut or n < 3 else ncol <= n


@pytest.mark.gpu
@pytest.mark.parametrize("grating", ["NONE", "HETG", "LETG"])
@pytest.mark.parametrize("det", ["NONE", "ACIS-S", "ACIS-I", "HRC-S", "HRC-I"])
@pytest.mark.parametrize("shape,uniform", [("POINT", 500.0), ("DISK", 0.0)])
def test_modules(gpu, grating, det, shape, uniform):
    n = 30_011
    _, ndet, rec = _same(_tracer(grating, det, shape, uniform, n), n)
    assert ndet == ((rec["flags"] & 0xFF) == 0).sum()


@pytest.mark.gpu
@pytest.mark.parametrize("par", [dict(HRMA_Ideal="yes"), dict(Shutters1="0101", Shutters3="1000", Shutters4="1111"),
                                 dict(HRMA_Use_Blur="no"), dict(HRMA_Use_WFold="no"),
                                 dict(HRMA_Use_Struts="no", HRMA_Use_Scale_Factors="no")])
def test_mirror_options(gpu, par):
    n = 40_000
    t = _tracer("NONE", "NONE", n=n, **par)
    _, _, rec = _same(t, n)
    pg, po = _both(t, n)
    from oracle.oracle import Oracle
    Oracle(t).reflect(po)
    t.trace_device(n, tag_start=0)
    p = Photons(n)
    t.download(p)
    compare(p.active.copy(), po.active.copy(), max_flips=2, label=f"{par}")
    assert ((rec["flags"] & 0xFF) == 0).any()


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[1], [0, 0, 5, 0], [0] * 70 + [3] + [0] * 200 + [1] * 90 + [700, 0, 64, 0],
                                    [1, 0] * 150 + [257], [3000, 1, 0, 0, 0, 0, 0, 0, 2, 1000]])
@pytest.mark.parametrize("graph", [False, True])
def test_batches_with_small_and_empty_sources(gpu, counts, graph):
    t = _tracer("NONE", "ACIS-I")
    k = len(counts)
    rng = np.random.default_rng(k)
    dirs = offaxis_directions(np.radians(rng.uniform(0, 15, k) / 60), rng.uniform(0, 2 * np.pi, k))
    counts = np.array(counts, np.uint32)
    for tag in (11, 5000):
        ndet, _ = t.trace_batch(dirs, counts, tag_start=tag, start_time=7.0, exposure=2.0e4, use_graph=graph)
        p = Photons(int(counts.sum()))
        t.download(p)
        got = p.active.copy()
        compare(got, _oracle(t, dirs, counts, tag, 7.0, 2.0e4, "NONE"), max_flips=1, label=f"{k} sources, tag {tag}")
        assert ndet == ((got["flags"] & 0xFF) == 0).sum()


@pytest.mark.gpu
@pytest.mark.parametrize("grating", ["NONE", "HETG"])
def test_kernel_times_are_the_stages(gpu, grating):
    """The stages share the kernels' times; the source's has the scan besides."""
    t = _tracer(grating, "ACIS-S", n=200_000)
    _, _, ms = t.trace_device(200_000, timing=True)
    create, mirror, diffract = t.pass_ms()
    assert create > 0 and mirror > 0 and (diffract > 0) == (grating != "NONE")
    enter, reflect = t.kernel_stats()[0]
    assert mirror + diffract == pytest.approx(reflect + ms[3] + ms[4], rel=1e-5)
    assert create < ms[0] + enter < create + 1.0
