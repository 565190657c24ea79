"""Passes after a module alone, or every one, is set up again: the tables that
the kernels stage in LDS are remade where their module changed and only there."""
import pytest

from marx_amd import Photons, Tracer
from tests.test_cpu_pins_mirror import _rdb_with
from tests.test_gpu_batch import ON_AXIS, assert_same_records

N = 20_011
PAR = dict(SpectrumType="FLAT", MinEnergy=0.3, MaxEnergy=8.0, DitherModel="INTERNAL", **ON_AXIS)


def _records(grating, det, **par):
    t = Tracer(seed=91, GratingType=grating, DetectorType=det, **par, **PAR)
    t.init_source(SourceFlux=N / (1.0e4 * t.geometric_area))
    out = []
    for again in range(2):
        if again:
            t.init_source(SourceFlux=N / (1.0e4 * t.geometric_area))     # a source set-up leaves the tables
        t.trace_device(N, tag_start=5)
        p = Photons(N)
        t.download(p)
        out.append(p.active.copy())
    assert_same_records(out[1], out[0], "the source set up again")
    return out[0]


@pytest.mark.gpu
def test_modules_set_up_in_turn(gpu, tmp_path):
    path = str(tmp_path / "geom.rdb")
    _rdb_with(path, {"p3": (2.0e-3, -1.0e-3)})
    first = {}
    for turn in range(2):
        for name, run in {"hetg": ("HETG", "ACIS-S", {}), "none": ("NONE", "ACIS-S", {}), "letg": ("LETG", "HRC-S", {}),
                          "tilted": ("HETG", "ACIS-S", dict(HRMA_Geometry_File=path)),
                          "shutters": ("HETG", "ACIS-S", dict(Shutters1="0101"))}.items():
            rec = _records(run[0], run[1], **run[2])
            assert_same_records(rec, first.setdefault(name, rec), f"{name}, turn {turn}")
    assert (first["hetg"]["x"] != first["tilted"]["x"]).any() and (first["hetg"]["x"] != first["shutters"]["x"]).any()
