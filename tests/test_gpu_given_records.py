"""Records of a photon list that no source makes, at the edges of the stages'
divisions: energies of 0 and infinity and next to them, rays along the shield's
plane at HRC-S; against the CPU oracle."""
import numpy as np
import pytest

from marx_amd import Photons, Tracer, on_axis_photons
from oracle.oracle import Oracle
from tests.parity import DIR_TOL, POS_TOL_MM

FIELDS = ("flags", "mirror_shell", "order", "support_orders", "ccd_num", "detector_region", "pulse_height")


def _pair(rec):
    pair = Photons(len(rec)), Photons(len(rec))
    for p in pair:
        p.load(rec)
    return pair


def _agree(a, b, label):
    for f in FIELDS:
        assert np.array_equal(a[f], b[f]), (label, f)
    alive = (b["flags"] & 0xFF) == 0
    for f, tol in (("x", POS_TOL_MM), ("p", DIR_TOL)):
        bad = ~(np.abs(a[f] - b[f]) <= tol) & ~(np.isnan(a[f]) & np.isnan(b[f]))
        assert not bad[alive].any(), (label, f)


@pytest.mark.gpu
@pytest.mark.parametrize("grating", ["HETG", "LETG"])
@pytest.mark.parametrize("energy", [0.0, 1e-320, 1e-306, 1e-300, 1e-30, 1e30, np.inf])
def test_energies_at_the_grating(gpu, grating, energy):
    t = Tracer(seed=81, GratingType=grating, DetectorType="NONE")
    n = 20_000
    start, _ = _pair(on_axis_photons(n, 1.5))
    t.reflect(start)
    rec = start.active.copy()
    rec["energy"] = energy
    pg, po = _pair(rec)
    t.diffract(pg)
    Oracle(t).diffract(po)
    _agree(pg.active, po.active, f"{grating} {energy}")


@pytest.mark.gpu
@pytest.mark.parametrize("energy", [0.0, 1e-320, 1e-300, 1e-30, 1e3, np.inf])
def test_energies_at_the_mirror(gpu, energy):
    t = Tracer(seed=83, GratingType="NONE", DetectorType="NONE")
    rec = on_axis_photons(20_000, energy)
    pg, po = _pair(rec)
    t.reflect(pg)
    Oracle(t).reflect(po)
    _agree(pg.active, po.active, f"mirror {energy}")


@pytest.mark.gpu
@pytest.mark.parametrize("det", ["ACIS-S", "HRC-S", "HRC-I"])
@pytest.mark.parametrize("energy", [0.0, 1e-320, 1e-30, 1e3, 1e30, np.inf])
def test_energies_at_the_detector(gpu, det, energy):
    t = Tracer(seed=84, GratingType="NONE", DetectorType=det)
    start, _ = _pair(on_axis_photons(20_000, 1.5))
    t.reflect(start)
    rec = start.active.copy()
    rec["energy"] = energy
    pg, po = _pair(rec)
    t.detect(pg)
    Oracle(t).detect(po)
    _agree(pg.active, po.active, f"{det} {energy}")


@pytest.mark.gpu
def test_rays_along_the_shield(gpu):
    t = Tracer(seed=82, GratingType="NONE", DetectorType="HRC-S")
    n = 20_000
    rec = on_axis_photons(n, 1.0)
    rng = np.random.default_rng(2)
    rec["x"] = rng.uniform((-0.5, -1.0, -8.0), (3.0, 1.0, 8.0), (n, 3))
    rec["p"] = 0.0
    rec["p"][:, 1] = np.where(rng.random(n) < 0.5, 1.0, -1.0)
    pg, po = _pair(rec)
    t.detect(pg)
    Oracle(t).detect(po)
    _agree(pg.active, po.active, "HRC-S")
    assert (po.active["flags"] != po.active["flags"][0]).any()
