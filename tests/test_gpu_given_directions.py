"""Directions that the library did not make and that are not of length 1: the
rays of a USER plug-in (a ray file's go through the same kernel), a batch's
directions, a photon list.  The dither and the extended shapes make them unit
vectors, the mirror takes them as they are; against the CPU oracle at the bars
of tests/parity.py."""
import numpy as np
import pytest

from marx_amd import Photons, Tracer, offaxis_directions, on_axis_photons
from oracle.oracle import Oracle
from tests.parity import compare
from tests.test_gpu_batch import ON_AXIS, _batch, _download, _oracle

LENGTHS = (0.5, 1.1, 3.0 ** 0.5, 2.0)


@pytest.mark.gpu
@pytest.mark.parametrize("length", LENGTHS)
def test_user_rays(gpu, tmp_path, length):
    from tests.user_plugin import build
    path, plug = build(str(tmp_path))
    t = Tracer(seed=5, GratingType="NONE", DetectorType="NONE", SourceType="USER", SpectrumType="FLAT", MinEnergy=1.0,
               MaxEnergy=10.0, DitherModel="INTERNAL", UserSourceFile=path, UserSourceArgs=f"length={length}", **ON_AXIS)
    t.init_source(SourceFlux=20.0)
    n = 5000
    pg, po = Photons(n), Photons(n)
    assert t.create_photons(pg, n) == Oracle(t).create_user(po, n, plug) == n
    compare(pg.active, po.active, max_flips=0, check_pixels=False, label=f"rays of length {length}")
    assert np.abs(np.linalg.norm(pg.active["p"], axis=1) - 1.0).max() < 1e-15


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dither,par", [
    ("POINT", "INTERNAL", {}), ("POINT", "NONE", {}), ("DISK", "NONE", {"S-DiskTheta0": 5.0, "S-DiskTheta1": 40.0}),
    ("GAUSS", "INTERNAL", {"S-GaussSigma": 20.0}), ("LINE", "NONE", {"S-LineTheta": 300.0, "S-LinePhi": 60.0})])
@pytest.mark.parametrize("length", (0.5, 2.0))
def test_batch_directions(gpu, tmp_path, shape, dither, par, length):
    t, dirs, counts = _batch(tmp_path, 12, dither=dither, shape=shape, **par)
    dirs = length * dirs
    t.trace_batch(dirs, counts, tag_start=9, start_time=0.0, exposure=2.0e4, use_graph=False)
    compare(_download(t, int(counts.sum())), _oracle(t, dirs, counts, 9, 0.0, 2.0e4, "NONE"), max_flips=2,
            label=f"{shape} of length {length}")


@pytest.mark.gpu
@pytest.mark.parametrize("length", LENGTHS)
def test_lists_at_the_mirror(gpu, length):
    n = 60_000
    t = Tracer(seed=6, GratingType="NONE", DetectorType="NONE")
    rec = on_axis_photons(n, 1.49)
    rec["p"] = length * offaxis_directions(np.full(n, 2.0e-3), np.linspace(0.0, 2.0 * np.pi, n))
    pg, po = Photons(n), Photons(n)
    pg.load(rec)
    po.load(rec)
    t.reflect(pg)
    Oracle(t).reflect(po)
    compare(pg.active, po.active, max_flips=2, label=f"list of length {length}")
    assert ((pg.active["flags"] & 0xFF) == 0).any()
