"""The work that is timed: passes of the photon trace through its public entry points.

A case is one pass as a user's program makes it:

- ``trace``: a chunk created and traced in HBM (Tracer.trace_device), its
  records left in the resident columns (mxg_get_soa);
- ``batch``: many point sources in one pass (Tracer.trace_batch), graph
  launched as a loop over pointings or tag ranges does it;
- ``diff``: a gradient of an image loss by the 20 mirror misalignments
  (DiffMirror.image and backward), one step of an alignment fit;
- ``dropin``: the reference's call sequence on a host photon list
  (marx_create_photons, marx_mirror_reflect, marx_grating_diffract,
  marx_detect);
- ``events``: a traced chunk with its event coordinates (Tracer.event_coords)
  brought to the host, what an event file is written from.

Every random draw is keyed by (seed, tag), so a pass's records follow from
the case and the seed alone.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

from marx_amd import _lib
from marx_amd.diff import DiffMirror
from marx_amd.sim import Photons, Tracer, offaxis_directions
from marx_amd.spectra import write_power_law
from marx_amd.workloads import ON_AXIS

EXPOSURE = 50_000.0          # s, of every chunk of Poisson arrivals
ARCSEC = math.pi / (180.0 * 3600.0)
ROLL = math.radians(237.36968458476) - 2.0 * math.pi      # the parameter file's Roll_Nom, in (-pi, pi]


def _case(name, kind, n, grating="NONE", detector="NONE", source="POINT", spectrum="FLAT", emin=1.49, emax=1.49,
          dither=False, uniform=False, sources=0, tile=0, npix=0):
    return {"name": name, "kind": kind, "n": n, "grating": grating, "detector": detector, "source": source,
            "spectrum": spectrum, "emin": emin, "emax": emax, "dither": dither, "uniform": uniform,
            "sources": sources, "tile": tile, "npix": npix}


def listed():
    return [
        # the benchmark workload: a long HETG observation in one chunk
        _case("hetg acis-s 1e7", "trace", 10_000_000, "HETG", "ACIS-S", spectrum="FILE", emin=0.4, emax=8.0,
              dither=True),
        # an extended source through the grating with the most draws, the largest chunk
        _case("letg hrc-s disk 5e7", "trace", 50_000_000, "LETG", "HRC-S", "DISK", emin=0.07, emax=10.0, dither=True),
        # a monochromatic calibration source without grating or dither
        _case("plain acis-s 1e6", "trace", 1_000_000, detector="ACIS-S", uniform=True),
        # the parameter file's default iteration size (dNumRays)
        _case("hetg acis-s 1e5", "trace", 100_000, "HETG", "ACIS-S", spectrum="FILE", emin=0.4, emax=8.0, dither=True),
        # a few photons of a faint extended source: what a call costs by itself
        _case("hrc-i gauss 1009", "trace", 1_009, detector="HRC-I", source="GAUSS", emin=0.3, emax=9.0, dither=True),
        # a field of 4096 sources, under the library's default schedule and as one persistent launch
        _case("batch 4096 acis-i staged", "batch", 0, detector="ACIS-I", spectrum="FILE", emin=0.3, emax=10.0,
              sources=4096),
        _case("batch 4096 acis-i persistent", "batch", 0, detector="ACIS-I", spectrum="FILE", emin=0.3, emax=10.0,
              sources=4096, tile=2048),
        # a small field seen through the grating
        _case("batch 37 hetg acis-s", "batch", 0, "HETG", "ACIS-S", spectrum="FILE", emin=0.4, emax=8.0, dither=True,
              sources=37),
        # a step of an alignment fit at full photon number, and a coarse one
        _case("diff 1e7", "diff", 10_000_000, npix=256),
        _case("diff 30011", "diff", 30_011, npix=96),
        # marx's own loop over a host photon list, at the largest iteration it allows
        _case("drop-in hetg acis-s 1e6", "dropin", 1_000_000, "HETG", "ACIS-S", spectrum="FILE", emin=0.4, emax=8.0,
              dither=True),
        # a chunk with its sky and detector coordinates
        _case("events hetg acis-s 1e6", "events", 1_000_003, "HETG", "ACIS-S", spectrum="FILE", emin=0.4, emax=8.0,
              dither=True),
    ]


def _odd_log(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi], mostly no round one."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "trace", "batch", "diff", "dropin", "events"])
    if kind == "diff":
        return _unnamed("diff", _odd_log(rng, 5_000, 8_000_000), npix=rng.choice([64, 96, 129, 256, 300]))
    grating = rng.choice(["NONE", "HETG", "LETG"])
    detector = rng.choice(["ACIS-S", "ACIS-I", "HRC-S", "HRC-I"])
    emin = round(rng.uniform(0.1, 1.0), 3)
    emax = round(rng.uniform(4.0, 10.0), 3)
    common = dict(grating=grating, detector=detector, spectrum=rng.choice(["FLAT", "FILE"]), emin=emin, emax=emax,
                  dither=rng.random() < 0.6)
    if kind == "batch":
        return _unnamed("batch", 0, sources=_odd_log(rng, 8, 2000), tile=rng.choice([0, 0, 512, 1024, 2048]), **common)
    if kind == "dropin":
        return _unnamed("dropin", _odd_log(rng, 2_000, 1_000_000), source=rng.choice(["POINT", "DISK"]), **common)
    if kind == "events":
        common["detector"] = rng.choice(["ACIS-S", "ACIS-I"])
        return _unnamed("events", _odd_log(rng, 20_000, 3_000_000), **common)
    return _unnamed("trace", _odd_log(rng, 1_000, 20_000_000), source=rng.choice(["POINT", "DISK", "GAUSS", "LINE"]),
                    uniform=rng.random() < 0.25, **common)


def _unnamed(kind, n, **kw):
    c = _case("", kind, n, **kw)
    del c["name"]
    return c


# ---- inputs ---------------------------------------------------------------------

_default_schedule = None


def _schedule(tile):
    """The library's own schedule, or its persistent pass at `tile` photons."""
    global _default_schedule
    lib = _lib.load()
    if _default_schedule is None:
        _default_schedule = _lib.Schedule()
        _lib.check(lib.mxg_get_schedule(ctypes.byref(_default_schedule)), "mxg_get_schedule")
    s = _lib.Schedule.from_buffer_copy(_default_schedule)
    if tile:
        s.persistent_tile = tile
        s.persistent_blocks_per_cu = 4
    _lib.check(lib.mxg_set_schedule(ctypes.byref(s)), "mxg_set_schedule")


def _tracer(case, seed):
    par = dict(ON_AXIS, GratingType=case["grating"], DetectorType=case["detector"], SourceType=case["source"],
               SpectrumType=case["spectrum"], MinEnergy=case["emin"], MaxEnergy=case["emax"],
               DitherModel="INTERNAL" if case["dither"] else "NONE")
    if case["source"] == "DISK":
        par.update({"S-DiskTheta0": 0.0, "S-DiskTheta1": 120.0})
    elif case["source"] == "GAUSS":
        par["S-GaussSigma"] = 45.0
    elif case["source"] == "LINE":
        par.update({"S-LineTheta": 300.0, "S-LinePhi": 35.0})
    with tempfile.TemporaryDirectory() as d:
        if case["spectrum"] == "FILE":
            par["SpectrumFile"] = write_power_law(os.path.join(d, "powerlaw.dat"), gamma=2.0, emin=case["emin"],
                                                  emax=case["emax"])
        t = Tracer(seed=seed, **par)
        t.init_source(uniform_times=1.0e4 if case["uniform"] else 0.0,
                      SourceFlux=max(case["n"], 1) / (EXPOSURE * t.geometric_area))
    return t


def _layout(case):
    """The batch's source counts (log-uniform over 1e2-1e5 for a large field, 1e2-1e3 for a small one) and off-axis angles."""
    rng = np.random.default_rng(case["sources"])
    counts = np.round(10.0 ** rng.uniform(2.0, 5.0 if case["sources"] >= 1000 else 3.0, case["sources"]))
    theta = np.radians(rng.uniform(0.0, 15.0, case["sources"]) / 60.0)
    return counts.astype(np.uint32), theta


def _order(case, seed):
    """The batch's sources in an order, and at azimuths and a first tag, of the seed."""
    rng = np.random.default_rng(seed)
    counts, theta = _layout(case)
    order = rng.permutation(len(counts))
    return counts[order], theta[order], rng.uniform(0.0, 2.0 * np.pi, len(counts)), int(rng.integers(1 << 30))


def prepare(case, seed):
    kind = case["kind"]
    _schedule(case["tile"])
    if kind == "batch":
        # one library seed for the whole program: the fields differ by their layouts and tag ranges
        t = _tracer(case, 1)
        counts, theta, phi, tag = _order(case, seed)
        return {"kind": kind, "t": t, "dirs": offaxis_directions(theta, phi), "counts": counts, "tag": tag, "views": {}}
    t = _tracer(case, seed)
    state = {"kind": kind, "t": t, "n": case["n"], "seed": seed, "views": {}}
    if kind == "dropin":
        state["photons"] = Photons(case["n"])
        state["records"], state["index"] = _host_views(state["photons"])
    elif kind == "diff":
        rng = np.random.default_rng(seed)
        step = np.tile([1.0, 1.0, 0.01, 0.01, 0.01], 4)     # 1 arcsec tilts, 10 um shifts
        at = rng.normal(0.0, 1.0, 20) * step
        dm = DiffMirror(t, case["n"], npix=case["npix"], pixel_size=1.024 / case["npix"])
        target = torch.empty((case["npix"], case["npix"]), dtype=torch.float32, device="cuda")
        dm.forward_into(at + rng.normal(0.0, 1.0, 20) * step, target, tangents=False)
        state.update(dm=dm, target=target, params=torch.tensor(at, dtype=torch.float64, requires_grad=True))
    elif kind == "events":
        # the program's own rows, as an event file's writer keeps them
        state["capacity"] = case["n"] // 2
        state["events"] = {k: np.zeros(state["capacity"], dt) for k, dt in t.EVENT_COLUMNS}
        state["rows"] = _lib.EventColumns(*[a.ctypes.data for a in state["events"].values()])
        state["cfg"] = t.event_cfg(pix_adj="EDSER", seed=7)
    return state


# ---- the passes -----------------------------------------------------------------

class _Column:
    """One device column as the CUDA array interface shows it to torch."""

    def __init__(self, ptr, n, typestr):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _host_views(p):
    """The list's records and sorted_index as arrays that keep the list alive."""
    views = []
    for addr, dtype in ((p.pt.attributes, _lib.ATTR_DTYPE),
                        (ctypes.cast(p.pt.sorted_index, ctypes.c_void_p).value, np.dtype("<u4"))):
        buf = (ctypes.c_char * (p.capacity * dtype.itemsize)).from_address(addr)
        buf.owner = p
        views.append(np.frombuffer(buf, dtype=dtype))
    return views


def _columns(state, n):
    """The resident columns as tensors (no copy); made again when the store has moved."""
    v = _lib.SoaView()
    _lib.check(_lib.load().mxg_get_soa(ctypes.byref(v)), "mxg_get_soa")
    views = state["views"]
    if views.get("at") != (v.energy, v.tag, n):
        ptrs = {"energy": (v.energy, "<f8"), "arrival_time": (v.arrival_time, "<f8"), "flags": (v.flags, "<i4"),
                "y_pixel": (v.y_pixel, "<f4"), "z_pixel": (v.z_pixel, "<f4"), "u_pixel": (v.u_pixel, "<f4"),
                "v_pixel": (v.v_pixel, "<f4"), "pi": (v.pi, "<f4"), "pulse_height": (v.pulse_height, "<i2"),
                "mirror_shell": (v.mirror_shell, "|u1"), "ccd_num": (v.ccd_num, "|i1"),
                "detector_region": (v.detector_region, "|i1"), "order": (v.order, "|i1"), "tag": (v.tag, "<i4")}
        for k in range(3):
            ptrs["x%d" % k] = (v.x[k], "<f8")
            ptrs["p%d" % k] = (v.p[k], "<f8")
        for k in range(6):
            ptrs["dither%d" % k] = (v.dither[k], "<f4")
        for k in range(4):
            ptrs["support_order%d" % k] = (v.support_orders[k], "|i1")
        views["columns"] = {k: torch.as_tensor(_Column(p, n, s), device="cuda") for k, (p, s) in ptrs.items()}
        views["at"] = (v.energy, v.tag, n)
    return views["columns"]


def run(state):
    kind, t = state["kind"], state["t"]
    if kind == "batch":
        detected, _ = t.trace_batch(state["dirs"], state["counts"], tag_start=state["tag"], exposure=EXPOSURE,
                                    use_graph=True)
        return {"columns": _columns(state, int(t.stage_counts()[0])), "detected": detected}
    t.set_seed(state["seed"])
    if kind == "diff":
        params = state["params"]
        params.grad = None
        image = state["dm"].image(params)
        loss = ((image - state["target"]) ** 2).sum()
        loss.backward()
        return {"image": image.detach(), "gradient": params.grad, "weight": state["dm"].total_weight}
    if kind == "dropin":
        p = state["photons"]
        p.pt.tag_start, p.pt.start_time, p.pt.total_time = 0, 0.0, 0.0
        t.create_photons(p, state["n"])
        t.reflect(p)
        t.diffract(p)
        t.detect(p)
        a = state["records"][:p.pt.n_photons]
        state["index"][p.pt.num_sorted:] = 0       # past the photons alive: no list
        return {"records": {k: a[k] for k in a.dtype.names}, "sorted_index": state["index"]}
    created, detected, _ = t.trace_device(state["n"])
    if kind == "events":
        _lib.check(t.lib.mxg_event_coords(ctypes.byref(state["cfg"]), ctypes.byref(state["rows"]), state["capacity"],
                                          ctypes.byref(ctypes.c_uint())), "mxg_event_coords")
        return {"events": state["events"], "detected": detected}
    return {"columns": _columns(state, created), "detected": detected}


# ---- what a pass cannot do without -----------------------------------------------

RECORD = 126        # bytes of one photon's resident columns

# FP64 operations a photon of each stage, transcendental calls not counted
# (the operation-counting build of the CPU oracle), and the share of the
# created photons that enter the stage
SOURCE, ENTER, REFLECT, DETECT = 146.0, 130.3, 598.6 * 0.5, 200.1
GRATING = {"NONE": 0.0, "HETG": 249.3 * 0.3, "LETG": 1422.0 * 0.16}
DETECTED_IN = {"NONE": 0.3, "HETG": 0.06, "LETG": 0.03}


def work(case):
    if case["kind"] == "diff":
        # the image, its target and its gradient; the photons need not leave the chip
        return {"bytes": 4.0 * 4 * case["npix"] ** 2 + 2 * 8 * 20, "flops": (122.7 + 1681.5 + 42.7) * case["n"]}
    n = float(_layout(case)[0].sum()) if case["kind"] == "batch" else case["n"]
    flops = n * (SOURCE + ENTER + REFLECT + GRATING[case["grating"]]
                 + DETECT * DETECTED_IN[case["grating"]] * (case["detector"] != "NONE"))
    if case["kind"] == "dropin":
        # 136-byte host records: created, then into and out of each stage
        stages = 3 if case["grating"] != "NONE" else 2
        return {"bytes": 136.0 * n * (1 + 2 * stages), "flops": flops}
    if case["kind"] == "events":
        # the records, and a row of 50 bytes for each detected photon
        return {"bytes": n * (RECORD + 50.0 * 0.04), "flops": flops}
    return {"bytes": RECORD * n, "flops": flops}


def tolerance(case):
    """About four times what the passes were measured to differ by from the
    FP64 CPU oracle, which has its own transcendentals and order of sums."""
    if case["kind"] == "diff":
        # FP32 image sums in any order (2e-7, 4e-7 at most), in the image and,
        # through the loss, in the gradient
        return {"rel": 1e-6, "max": 5e-6}
    if case["kind"] == "events":
        # the sky pixels go through acos of numbers next to 1: up to 0.01 of 4096 pixels
        return {"rel": 1e-7, "max": 1e-5, "differ": 1e-6}
    # FP64 columns differ by 1e-15 (6e-14 at most), so an FP32 column by the
    # last bit of a value now and then: 1.2e-7 of it, 2e-9 of a thousand
    return {"rel": 5e-9, "max": 5e-7, "differ": 1e-6}


# ---- 64-bit values ----------------------------------------------------------------

def _philox(tag, stage, block, seed):
    """Four uniforms of each tag: Philox4x32-10 (Salmon et al., SC'11) of the
    counter (tag, stage, block, 0) and the 64-bit key `seed`, u32 / (2^32 - 1)."""
    mask = 0xFFFFFFFF
    c0 = tag.clone()
    c1 = torch.full_like(tag, stage)
    c2 = torch.full_like(tag, block)
    c3 = torch.zeros_like(tag)
    k0, k1 = seed & mask, (seed >> 32) & mask
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
        a, b = c0 * 0xD2511F53, c2 * 0xCD9E8D57      # the 64-bit products, wrapped
        c0, c1, c2, c3 = ((b >> 32) & mask) ^ c1 ^ k0, b & mask, ((a >> 32) & mask) ^ c3 ^ k1, a & mask
    return [c.double() / mask for c in (c0, c1, c2, c3)]


def _energies(case, u):
    if case["spectrum"] == "FLAT":
        return case["emin"] + (case["emax"] - case["emin"]) * u
    with tempfile.TemporaryDirectory() as d:
        e, f = np.loadtxt(write_power_law(os.path.join(d, "s"), gamma=2.0, emin=case["emin"], emax=case["emax"])).T
    cum = np.cumsum(f * np.diff(e, prepend=e[0]))
    e, cum = (torch.from_numpy(x).to(u.device) for x in (e, cum / cum[-1]))
    k = torch.searchsorted(cum, u).clamp(1, len(cum) - 1)
    return e[k - 1] + (e[k] - e[k - 1]) * (u - cum[k - 1]) / (cum[k] - cum[k - 1])


def exact(case, seed):
    """The values that follow from the draws alone: energies, arrival times
    and dither angles.  The rest follows from calibration tables as the
    library reads them, and the differentiable pass and the event
    coordinates (detector positions) from those: None."""
    kind = case["kind"]
    if kind in ("diff", "events"):
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "batch":
        counts, _, _, first = _order(case, seed)
        n, seed = int(counts.sum()), 1
    else:
        n, first = case["n"], 0
    tag = torch.arange(first, first + n, dtype=torch.int64, device=device)
    u = _philox(tag, 1, 0, seed)
    energy = _energies(case, u[0])
    # the energy, then the direction's draws, then the time's
    v = u[1 + {"POINT": 0, "LINE": 1, "DISK": 2, "GAUSS": 2}[case["source"]]]
    if kind == "batch":
        time = EXPOSURE * v
    elif case["uniform"]:
        time = 1.0e4 * v
    else:
        time = torch.cumsum(-torch.log(v), 0) * (EXPOSURE / n)
    angles = [torch.zeros_like(time) for _ in range(6)]
    if case["dither"]:
        angles[0] = 16.0 * ARCSEC * torch.sin(2.0 * math.pi * time / 1414.2)
        angles[1] = 16.0 * ARCSEC * torch.sin(2.0 * math.pi * time / 2000.0)
        angles[2] = torch.full_like(time, ROLL)
    if kind == "dropin":
        names = ("energy", "x", "p", "arrival_time", "flags", "y_pixel", "z_pixel", "u_pixel", "v_pixel", "dither",
                 "pi", "pulse_height", "mirror_shell", "ccd_num", "detector_region", "order", "support_orders", "tag")
        values = dict.fromkeys(names)
        values.update(energy=energy, arrival_time=time, dither=torch.stack(angles, 1))
        return {"records": values, "sorted_index": None}
    values = {"energy": energy, "arrival_time": time}
    values.update({"dither%d" % k: a for k, a in enumerate(angles)})
    return {"columns": values, "detected": None}
