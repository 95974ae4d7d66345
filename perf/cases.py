"""The work that is timed: what programs on this package run, through its public entry points.

Kinds of case (`kind`), each a call or a short sequence of calls that a program makes:

  diffraction   one aperture onto every bin, host arrays in and out (the tracer's per-beam call of its
                memory-saving mode)
  diff_main     both beam trees of one orientation, host arrays in and out (the Fortran drop-in's call)
  step          the drivers' loop body on device-resident records: far field of both trees, then the
                epilogue (Mueller matrices, phi and theta integrals, optional energy scaling)
  batch         the orientation-batched plan: Mueller sum, 1-D matrices, per-orientation integrals
  retrieval     one gradient step of the shape retrieval: apertures gathered from the particle's
                vertices, batched far field with amplitudes, loss, backward through the adjoint
  vis_batch     facet visibility of many beams over one facet topology, on the device
  vis_call      facet visibility of one beam, host arrays in and out

Beam sets are traced from seeded particles (a smooth or rough hexagonal column of random
orientation) or drawn as random facets ("facets", "polygons").  `exact` evaluates the closed form of
the diffracted amplitude (Kirchhoff aperture integral, Karczewski-Wolf polarisation) in plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from abt_amd import autograd as AG
from abt_amd import lib
from abt_amd import visibility as V
from abt_amd.beams import BeamSet
from abt_amd.workloads import (euler_matrix, grid, hex_column, hex_column_apertures, random_rotations, to_beamset,
                               trace_orientations)

LAM = 0.532
PI_R4 = float(np.float32(3.14159265358979))
EXT_FOV = PI_R4 / 2


def listed():
    return [
        # one aperture per call from the tracer's OpenMP threads, on the default 361 x 180 grid
        dict(name="diffraction_call", kind="diffraction", precision="fp64", ntheta=361, nphi=180),
        # the drop-in as the sequential driver calls it: the default column, one orientation
        dict(name="diff_main_column", kind="diff_main", precision="fp64", source="column", radius=5.0, length=10.0,
             nfhr=6, nfpl=12, sigma=0.0, rec=8, ntheta=361, nphi=180, fast_diff=False),
        # an unrefined crystal: a few many-sided facets on a fine grid, energies rescaled; the epilogue weighs most
        dict(name="step_few_polygons", kind="step", precision="fp64", source="polygons", nb=37, ne=8, ntheta=721,
             nphi=180, scaling=True, fast_diff=False),
        # many small apertures on the finest grid (the diffraction stress test, fewer apertures)
        dict(name="step_many_facets", kind="step", precision="fp64_fast", source="facets", nb=9001, ne=1000,
             ntheta=1801, nphi=360, scaling=False, fast_diff=False),
        # a quick look: few orientations, few reflections, a coarse grid; latency
        dict(name="average_coarse", kind="batch", precision="fp64_fast", norient=4, radius=10.0, length=20.0, nfhr=4,
             nfpl=7, sigma=0.3, rec=3, ntheta=37, nphi=36, fast_diff=False),
        # the orientation average on its usual grid (a share of the 1000 orientations)
        dict(name="average_fine", kind="batch", precision="fp64_fast", norient=24, radius=10.0, length=20.0, nfhr=8,
             nfpl=14, sigma=0.5, rec=10, ntheta=721, nphi=180, fast_diff=False),
        # the FP32 body, where speed matters more than the last digits
        dict(name="average_mixed", kind="batch", precision="mixed", norient=16, radius=10.0, length=20.0, nfhr=8,
             nfpl=14, sigma=0.5, rec=10, ntheta=361, nphi=180, fast_diff=False),
        # one orientation of a large column, beams confined to their field of view
        dict(name="one_orientation_large", kind="batch", precision="fp64_fast", norient=1, radius=50.0, length=100.0,
             nfhr=16, nfpl=32, sigma=0.0, rec=6, ntheta=451, nphi=360, fast_diff=True),
        # shape retrieval, the default precision
        dict(name="retrieval_mixed", kind="retrieval", precision="mixed", norient=8, nfhr=8, nfpl=14, sigma=0.5,
             rec=10, ntheta=361, nphi=90),
        # shape retrieval near its optimum, in FP64 throughout
        dict(name="retrieval_fp64", kind="retrieval", precision="fp64", norient=5, nfhr=6, nfpl=9, sigma=0.4, rec=6,
             ntheta=181, nphi=90),
        # one generation of internal beams of the tracer
        dict(name="vis_internal", kind="vis_batch", mode="int", nbeam=2048, nfhr=8, nfpl=14, sigma=0.5),
        # the incident beam, once per orientation, as the Fortran module calls it
        dict(name="vis_incident_call", kind="vis_call", mode="inc", nfhr=8, nfpl=14, sigma=0.5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["diffraction", "diff_main", "step", "step", "batch", "batch", "batch", "retrieval",
                       "vis_batch", "vis_call"])
    nth, nph = _log(rng, 33, 1201), _log(rng, 24, 360)
    if kind == "diffraction":
        return dict(kind=kind, precision=rng.choice(["fp64", "fp64", "fp64_fast", "mixed"]), ntheta=nth, nphi=nph)
    if kind == "vis_batch":
        return dict(kind=kind, mode=rng.choice(["int", "ext", "inc"]), nbeam=_log(rng, 3, 2500),
                    nfhr=rng.randint(1, 8), nfpl=rng.randint(1, 14), sigma=round(rng.uniform(0.0, 0.5), 3))
    if kind == "vis_call":
        return dict(kind=kind, mode=rng.choice(["int", "ext", "inc"]), nfhr=rng.randint(1, 9),
                    nfpl=rng.randint(1, 16), sigma=round(rng.uniform(0.0, 0.5), 3))
    nfhr, nfpl = rng.randint(2, 8), rng.randint(2, 14)
    per = 3 * (12 * nfhr * nfpl + 12 * nfhr * nfhr)      # about what a traced orientation has of beams
    if kind == "retrieval":
        nth, nph = _log(rng, 33, 361), _log(rng, 24, 120)
        most = max(1, int(8e8 / (per * nth * nph)))
        return dict(kind=kind, precision=rng.choice(["mixed", "fp64"]), norient=_log(rng, 1, max(2, min(12, most))),
                    nfhr=nfhr, nfpl=nfpl, sigma=round(rng.uniform(0.2, 0.5), 3), rec=rng.randint(2, 10), ntheta=nth,
                    nphi=nph)
    if kind == "batch":
        prec = rng.choice(["fp64_fast", "fp64_fast", "fp64_fast", "mixed", "fp64"])
        most = max(1, int((3e9 if prec == "fp64" else 8e9) / (per * nth * nph)))
        return dict(kind=kind, precision=prec, norient=_log(rng, 1, max(2, min(40, most))),
                    radius=round(rng.uniform(5.0, 30.0), 2), length=round(rng.uniform(10.0, 60.0), 2), nfhr=nfhr,
                    nfpl=nfpl, sigma=round(rng.uniform(0.1, 0.5), 3), rec=rng.randint(2, 10), ntheta=nth, nphi=nph,
                    fast_diff=rng.random() < 0.2)
    if kind == "diff_main":
        return dict(kind=kind, precision=rng.choice(["fp64", "fp64", "fp64_fast", "mixed"]), source="column",
                    radius=round(rng.uniform(3.0, 12.0), 2), length=round(rng.uniform(5.0, 25.0), 2), nfhr=nfhr,
                    nfpl=nfpl, sigma=round(rng.uniform(0.0, 0.3), 3), rec=rng.randint(2, 10), ntheta=min(nth, 721),
                    nphi=min(nph, 180), fast_diff=rng.random() < 0.2)
    source = rng.choice(["facets", "polygons"])
    nb = _log(rng, 5, 9000 if source == "facets" else 900)
    return dict(kind="step", precision=rng.choice(["fp64", "fp64_fast", "fp64_fast", "mixed"]), source=source, nb=nb,
                ne=max(1, nb // 7), ntheta=nth, nphi=nph, scaling=rng.random() < 0.4, fast_diff=rng.random() < 0.2)


# ---------------------------------------------------------------------------
# inputs

def _angles(case):
    """0 to 180 degrees in ntheta nodes, 0 to just below 360 in nphi nodes (uniform)."""
    nth, nph = case["ntheta"], case["nphi"]
    return grid((0, 180.0 / (nth - 1), 180.0), (0, 360.0 / nph, 360.0 - 360.0 / nph))


def _unit(a):
    return a / np.linalg.norm(a, axis=-1, keepdims=True)


def _facets(n, rng, polygons, ext, box=60.0):
    """n seeded facets in a cube: triangles (edges 0.3-5 um), or convex polygons of 3 to 6 vertices on a
    circle of 1-8 um; beams leave at 5-80 degrees from the facet's normal, amplitudes over six decades
    (ext: the incident direction (0, 0, -1), amplitudes of size one)."""
    c = rng.uniform(-box / 2, box / 2, (n, 3))
    nrm = _unit(rng.normal(size=(n, 3)))
    if ext:
        nrm[:, 2] = np.abs(nrm[:, 2]) + 0.1
        nrm[:, 0] += 0.15
        nrm = _unit(nrm)
    a = _unit(np.cross(nrm, rng.normal(size=(n, 3))))
    b = np.cross(nrm, a)
    if polygons:
        nv = rng.integers(3, 7, n)
        start, r = rng.uniform(0, 2 * np.pi, n), rng.uniform(1.0, 8.0, n)
        verts = []
        for i in range(n):
            t = start[i] + 2 * np.pi * (np.arange(nv[i]) + rng.uniform(-0.25, 0.25, nv[i])) / nv[i]
            verts.append(c[i] + r[i] * (np.cos(t)[:, None] * a[i] + np.sin(t)[:, None] * b[i]))
        verts = np.concatenate(verts)
    else:
        nv = np.full(n, 3)
        t1 = rng.uniform(0, 2 * np.pi, (n, 1))
        t2 = t1 + rng.uniform(0.3, np.pi - 0.3, (n, 1))
        l1, l2 = rng.uniform(0.3, 5.0, (n, 1)), rng.uniform(0.3, 5.0, (n, 1))
        e1, e2 = l1 * (np.cos(t1) * a + np.sin(t1) * b), l2 * (np.cos(t2) * a + np.sin(t2) * b)
        v0 = c - (e1 + e2) / 3
        verts = np.stack([v0, v0 + e1, v0 + e2], 1).reshape(-1, 3)
    if ext:
        prop = np.tile([0.0, 0.0, -1.0], (n, 1))
        ampl = rng.normal(size=(n, 8))
    else:
        tilt, az = np.deg2rad(rng.uniform(5, 80, (n, 1))), rng.uniform(0, 2 * np.pi, (n, 1))
        prop = np.cos(tilt) * nrm + np.sin(tilt) * (np.cos(az) * a + np.sin(az) * b)
        ampl = rng.normal(size=(n, 8)) * 10.0 ** rng.uniform(-6, 0, (n, 1))
    vk7 = _unit(np.cross(nrm, prop))
    fov = rng.uniform(0.5, np.pi / 2, n)
    return BeamSet(ampl, vk7, prop, fov, np.concatenate([[0], np.cumsum(nv)]), verts)


def _traced(case, seed, norient, device="cuda"):
    """Beams of `norient` random orientations of a seeded column (see trace_orientations)."""
    radius, length = case.get("radius", 10.0), case.get("length", 20.0)
    verts, faces = hex_column(radius, length, case["nfhr"], case["nfpl"], case["sigma"], seed=seed)
    if norient is None:      # one orientation given by Euler angles near the drop-in's default (0, 30, 0)
        a = np.random.default_rng(seed).uniform(-15, 15, 3) + np.array([0.0, 30.0, 0.0])
        rots = euler_matrix(*a)[None]
    else:
        rots = random_rotations(norient, seed + 1)
    m = 1.31 + (0.01j if radius >= 50 else 0j)
    t = trace_orientations(verts, faces, rots, la=LAM, m=m, rec=case["rec"], device=device)
    t["verts0"], t["faces"], t["rots"] = verts, faces, rots
    if case.get("fast_diff"):
        # fields of view of 20 to 90 degrees
        r = np.random.default_rng(seed + 5).uniform(np.deg2rad(20), np.pi / 2, t["beams"]["prop"].shape[0])
        t["beams"]["fov"] = torch.from_numpy(r).to(t["beams"]["prop"].device)
    return t


def _trees(case, seed):
    """(beams, ext, beam offsets, ext offsets) as host beam sets."""
    if case["kind"] == "diffraction":
        return _facets(8, np.random.default_rng(seed), False, False), None, None, None
    if case.get("source") in ("facets", "polygons"):
        rng = np.random.default_rng(seed)
        poly = case["source"] == "polygons"
        return _facets(case["nb"], rng, poly, False), _facets(case["ne"], rng, poly, True), None, None
    t = _traced(case, seed, case.get("norient"))
    return (to_beamset(t["beams"]), to_beamset(t["ext"]), t["beam_off"].cpu().numpy(), t["ext_off"].cpu().numpy())


def _energies(seed):
    return [float(x) for x in np.random.default_rng(seed + 9).uniform(50.0, 150.0, 2)]


def _vis_inputs(case, seed, nbeam):
    """Topology, rotation per beam, illuminating facets, incident height (as the tracer holds them)."""
    verts, faces, ap, apn = hex_column_apertures(10.0, 20.0, case["nfhr"], case["nfpl"], case["sigma"], seed=seed)
    topo = V.VisGeometry.from_mesh(verts, faces, ap, apn)
    rots = random_rotations(nbeam, seed + 7)
    rng = np.random.default_rng(seed + 11)
    apz = np.einsum("bj,aj->ba", rots[:, 2], topo.ap_n)
    off, fins = [0], []
    by_ap = [np.nonzero(topo.ap == a + 1)[0] + 1 for a in range(topo.na)]
    for b in range(nbeam):
        if case["mode"] == "inc":
            fin = np.zeros(0, np.int64)
        else:
            want = apz[b] > 0.01 if case["mode"] == "int" else apz[b] < -0.01
            fin = by_ap[rng.choice(np.nonzero(want)[0])]
        fins.append(fin)
        off.append(off[-1] + len(fin))
    bmz = np.einsum("bj,vj->bv", rots[:, 2], topo.v).max(1) + 1.0
    return topo, rots, np.array(off, np.int64), np.concatenate(fins).astype(np.int64), bmz


def _target(case, seed, device):
    """A smooth S11 and polarisation pattern with seeded ripple: the measured pattern of a retrieval."""
    th, ph = _angles(case)
    rng = np.random.default_rng(seed + 77)
    t = (2e4 / (1.0 + (th / 0.05) ** 2) + 40.0)[:, None] * np.exp(0.2 * rng.normal(size=(len(th), len(ph))))
    p = 0.3 * np.sin(th)[:, None] ** 2 + 0.05 * rng.normal(size=(len(th), len(ph)))
    g = lambda a: torch.from_numpy(a.reshape(-1)).to(device)
    return g(t), g(p), AG.solid_angle_weights(th, ph, device)


def _retrieval(case, seed, device):
    """A retrieval in progress: beams traced once from the case's particle (their facets, directions and
    orientations stay), and the iterate of this seed: vertices and amplitudes off those of the trace."""
    t = _traced(case, 0, case["norient"])
    rng = np.random.default_rng(seed + 33)
    v = t["verts0"] + rng.normal(scale=0.03, size=t["verts0"].shape)
    ampl = []
    for k in ("beams", "ext"):
        a = t[k]["ampl"].to(device)
        ampl.append((a * torch.from_numpy(1 + 0.1 * rng.normal(size=tuple(a.shape))).to(device)).requires_grad_(True))
    return t, torch.tensor(v, dtype=torch.float64, device=device, requires_grad=True), ampl


def prepare(case, seed):
    kind = case["kind"]
    dev = torch.device("cuda:0")
    f64 = dict(dtype=torch.float64, device=dev)
    s = dict(case)
    if kind in ("vis_batch", "vis_call"):
        topo, rots, off, fin, bmz = _vis_inputs(case, seed, case.get("nbeam", 1))
        if kind == "vis_call":
            s.update(geom=topo.rotated(rots[0]), fin=fin if len(fin) else None, bmz=float(bmz[0]))
            return s
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
        v, mid, nz, apnz = V.rotate_dev(t(rots), topo)
        s["batch"] = V.VisBatch(case["mode"], topo, v, mid, nz, apnz, t(off), t(fin) if len(fin) else None, t(bmz))
        return s
    th, ph = _angles(case)
    s.update(th=th, ph=ph)
    if kind == "retrieval":
        t, s["V"], s["ampl"] = _retrieval(case, seed, dev)
        g = lib.DeviceGrid(th, ph, LAM)
        tree = lambda k: {q: t[k][q] for q in ("prop", "vk7")}
        s["system"] = AG.FarFieldSystem(g, t["beam_off"].cpu().numpy(), t["ext_off"].cpu().numpy(), tree("beams"),
                                        tree("ext"), precision=case["precision"])
        faces = torch.as_tensor(t["faces"], device=dev)
        s["gather"] = [AG.ApertureGather(faces, t[k]["fi"], len(t["verts0"])) for k in ("beams", "ext")]
        s["orient"] = [t[k]["orient"] for k in ("beams", "ext")]
        s["rots"] = torch.as_tensor(t["rots"], **f64)
        s["target"] = _target(case, seed, dev)
        return s
    B, E, boff, eoff = _trees(case, seed)
    s.update(B=B, E=E)
    if kind == "diffraction":
        s["xyz"] = lib.make_far_field_bins(th, ph)
        s["i"] = seed % B.n
        return s
    if kind == "diff_main":
        return s
    g = s["g"] = lib.DeviceGrid(th, ph, LAM)
    rb, vb = lib.prepare_beams_host(B, LAM)
    re, ve = lib.prepare_beams_host(E, LAM, fov_value=EXT_FOV)
    t = lambda a: torch.from_numpy(a).to(dev)
    poly = case.get("source") == "polygons"
    s.update(rb=t(rb), re=t(re), vb=t(vb) if poly else None, ve=t(ve) if poly else None)
    n = g.nbins
    if kind == "batch":
        s["plan"] = lib.BatchPlan(g, boff, eoff, case["precision"], case["fast_diff"])
        s.update(m=torch.empty(16 * n, **f64), m1=torch.empty(16 * len(th), **f64),
                 integrals=torch.empty(6 * case["norient"], **f64))
        return s
    s.update(ab=torch.empty(8 * n, **f64), ae=torch.empty(8 * n, **f64), m=torch.empty(48 * n, **f64),
             m1=torch.empty(48 * len(th), **f64), par=torch.zeros(9, **f64), energies=_energies(seed))
    ws = max(lib.far_field_workspace(g, max(B.n, E.n), case["precision"]), 8)
    s["work"] = torch.empty(ws // 8 + 1, **f64)
    s["fwork"] = torch.empty(lib.load().abt_finalise_workspace(g.handle) // 8 + 1, **f64)
    return s


def run(s):
    kind = s["kind"]
    if kind == "diffraction":
        return lib.diffraction(s["th"], s["ph"], *s["xyz"], LAM, s["B"], s["i"], precision=s["precision"])
    if kind == "diff_main":
        b, e = lib.diff_main(s["th"], s["ph"], LAM, s["B"], s["E"], precision=s["precision"],
                             fast_diff=s["fast_diff"], raw=True)
        return {"beam": b, "ext": e}
    if kind == "step":
        p, fd = s["precision"], s["fast_diff"]
        lib.far_field_dev(s["g"], s["rb"], s["B"].n, s["ab"], s["vb"], p, fd, work=s["work"])
        lib.far_field_dev(s["g"], s["re"], s["E"].n, s["ae"], s["ve"], p, fd, work=s["work"])
        lib.finalise_dev(s["g"], s["ab"], s["ae"], s["m"], s["m1"], s["par"], s["scaling"], *s["energies"],
                         work=s["fwork"])
        return {"beam": s["ab"], "ext": s["ae"], "mueller": s["m"], "mueller_1d": s["m1"], "params": s["par"]}
    if kind == "batch":
        s["plan"].run(s["rb"], s["re"], s["m"], s["integrals"], s["m1"], s["vb"], s["ve"])
        return {"mueller": s["m"], "mueller_1d": s["m1"], "integrals": s["integrals"]}
    if kind == "retrieval":
        s["V"].grad = None
        for a in s["ampl"]:
            a.grad = None
        vb, ve = (s["gather"][q](s["V"], s["rots"], s["orient"][q]) for q in (0, 1))
        X = AG.far_field(s["system"], vb, s["ampl"][0], ve, s["ampl"][1])
        loss = AG.retrieval_loss(X, *s["target"])
        loss.backward()
        return {"loss": loss, "X": X, "grad_vertices": s["V"].grad, "grad_beam": s["ampl"][0].grad,
                "grad_ext": s["ampl"][1].grad}
    if kind == "vis_batch":
        s["batch"].run()
        return s["batch"].results()
    return V.find_vis(s["mode"], s["geom"], s["fin"], s["bmz"])


# ---------------------------------------------------------------------------
# the work a pass cannot do without

FLOP_BEAM_BIN = 250.0    # a triangular aperture on one bin: geometry, three phases, polarisation, 2 x 2 sum
BYTES_BEAM = 192.0       # amplitude, three directions, three vertices


def _per_orientation(case):
    """About how many beams and ext beams a traced orientation has (half of the facets are lit)."""
    nf = 12 * case["nfhr"] * case["nfpl"] + 12 * case["nfhr"] ** 2
    return (0.5 + 0.155 * case["rec"]) * nf, 0.5 * nf


def work(case):
    kind = case["kind"]
    if kind in ("vis_batch", "vis_call"):
        nf = 12 * case["nfhr"] * case["nfpl"] + 12 * case["nfhr"] ** 2
        nb = case.get("nbeam", 1)
        # per facet: coordinates, midpoint, normal in; five results out; a scan of the blockers over it
        return {"bytes": nb * nf * (12 + 24 + 8 + 19.0), "flops": nb * nf * 500.0}
    nbins = case["ntheta"] * case["nphi"]
    if kind == "diffraction":
        return {"bytes": 24.0 * nbins + 64.0 * nbins, "flops": FLOP_BEAM_BIN * nbins}
    if "nb" in case:
        beams = case["nb"] + case["ne"]
    else:
        beams = sum(_per_orientation(case)) * case.get("norient", 1)
    flops = FLOP_BEAM_BIN * beams * nbins
    if kind == "diff_main":
        return {"bytes": BYTES_BEAM * beams + 128.0 * nbins, "flops": flops}
    if kind == "step":
        return {"bytes": BYTES_BEAM * beams + (128.0 + 384.0) * nbins, "flops": flops + 300.0 * nbins}
    if kind == "batch":
        return {"bytes": BYTES_BEAM * beams + 128.0 * nbins, "flops": flops + 300.0 * nbins * case["norient"]}
    return {"bytes": 2 * BYTES_BEAM * beams + 128.0 * nbins * case["norient"], "flops": 3.0 * flops}


# ---------------------------------------------------------------------------
# the closed form in plain torch

K2CLAMP, FWD_DOT, ANTI = (float(np.float32(v)) for v in (0.999999, 0.999, 0.0001))


class _Bins:
    def __init__(self, th, ph):
        dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
        st, ct, sp, cp = np.sin(th), np.cos(th), np.sin(ph), np.cos(ph)
        r = 1e6
        x = np.stack([(r * st[:, None] * cp).ravel(), (r * st[:, None] * sp).ravel(),
                      np.repeat(-(r * ct), len(ph))])
        self.nth, self.nph, self.n = len(th), len(ph), x.shape[1]
        self.k = 2.0 * PI_R4 / LAM
        xl = x.astype(np.longdouble)
        rad = np.sqrt((xl * xl).sum(0))
        turns = np.longdouble(self.k) * rad / (2 * np.longdouble("3.14159265358979323846264338327950288"))
        turns = (turns - np.rint(turns)).astype(np.float64)
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
        self.x, self.rad, self.dev = t(x), t(rad.astype(np.float64)), dev
        phase = torch.from_numpy(2 * np.pi * turns).to(dev)
        self.phase = torch.complex(torch.cos(phase), torch.sin(phase))
        it = int(np.argmax(th > PI_R4 / 180)) if (th > PI_R4 / 180).any() else len(th) - 1
        self.xt = self.x.reshape(3, self.nth, self.nph)[:, it].repeat(1, self.nth)   # the theta_i bin of the same phi
        self.cphi, self.sphi = t(np.tile(cp, self.nth)), t(np.tile(sp, self.nth))


def _padded(b: BeamSet, dev):
    """Vertices (n, most, 3), the last one repeated, and the vertex counts."""
    nv = np.diff(b.vert_off)
    most = int(nv.max())
    idx = b.vert_off[:-1, None] + np.minimum(np.arange(most)[None], nv[:, None] - 1)
    return torch.from_numpy(b.verts[idx]).to(dev), torch.from_numpy(nv.astype(np.float64)).to(dev)


def _dot(a, b):
    return (a * b).sum(-1)


def _form_factor(qx, qy, X, Y, nv, amax):
    """int e^{i q.u} dA over the (clockwise) polygon with in-plane vertices X, Y (n, most)."""
    most = X.shape[1]
    q2 = qx * qx + qy * qy
    small = q2 * (amax * amax)[:, None] < 1.0
    safe = torch.where(small, torch.ones_like(q2), q2)
    sr, si = torch.zeros_like(q2), torch.zeros_like(q2)
    for j in range(most):
        jn = (j + 1) % most
        ex, ey = X[:, jn] - X[:, j], Y[:, jn] - Y[:, j]
        mx, my = 0.5 * (X[:, j] + X[:, jn]), 0.5 * (Y[:, j] + Y[:, jn])
        c = qx * ey[:, None] - qy * ex[:, None]
        t = c * torch.sinc((qx * ex[:, None] + qy * ey[:, None]) / (2 * math.pi))
        mu = qx * mx[:, None] + qy * my[:, None]
        sr = sr + t * torch.cos(mu)
        si = si + t * torch.sin(mu)
    Fr, Fi = -si / safe, sr / safe
    if bool(small.any()):
        b, i = torch.nonzero(small, as_tuple=True)
        px, py = qx[b, i], qy[b, i]
        fr, fi = torch.zeros_like(px), torch.zeros_like(px)
        for j in range(most):           # fan of triangles about the centre: phases 0, u, w
            jn = (j + 1) % most
            sa = -0.5 * (X[:, j] * Y[:, jn] - X[:, jn] * Y[:, j])[b]
            u, w = px * X[b, j] + py * Y[b, j], px * X[b, jn] + py * Y[b, jn]
            e1, e2 = u + w, u * w
            h1, h0 = e1, torch.ones_like(e1)      # h_n, h_{n-1}
            fr, f = fr + sa, 2.0 / 6.0
            fi = fi + sa * f * h1
            for n in range(2, 19):
                h1, h0 = e1 * h1 - e2 * h0, h1
                f = f / (n + 2)
                t = sa * f * h1 * (1.0 if n % 4 in (0, 1) else -1.0)
                fr, fi = (fr + t, fi) if n % 2 == 0 else (fr, fi + t)
        Fr, Fi = Fr.index_put((b, i), fr), Fi.index_put((b, i), fi)
    return Fr, Fi


def _amplitudes(g, ampl, vk7, prop, verts, nv, cosfov=None):
    """Sum over the given beams of their amplitude on every bin, without the bins' own phase: (4, nbins)
    complex, entries (1,1) (2,1) (1,2) (2,2)."""
    k = g.k
    w = (torch.arange(verts.shape[1], device=g.dev)[None] < nv[:, None]).to(verts.dtype)
    c = (verts * w[..., None]).sum(1) / nv[:, None]
    u = verts - c[:, None]
    n = torch.linalg.cross(u[:, 0], u[:, 1], dim=-1)
    ez = -n / torch.linalg.norm(n, dim=-1, keepdim=True)
    ey = torch.linalg.cross(ez, prop, dim=-1)
    ey = ey / torch.linalg.norm(ey, dim=-1, keepdim=True)
    ex = torch.linalg.cross(ey, ez, dim=-1)
    par = torch.linalg.cross(vk7, prop, dim=-1)
    anti = _dot(par, ez) / torch.linalg.norm(par, dim=-1) > ANTI
    C = torch.where(anti[:, None], -ampl, ampl)
    X, Y = (u * ex[:, None]).sum(-1), (u * ey[:, None]).sum(-1)
    amax = torch.linalg.norm(u, dim=-1).amax(1).detach()
    Kz = _dot(prop, ez)[:, None]
    d = [g.x[i] - c[:, i:i + 1] for i in range(3)]
    rho = torch.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
    kh = [q / rho for q in d]
    del d
    axis = lambda e: kh[0] * e[:, 0:1] + kh[1] * e[:, 1:2] + kh[2] * e[:, 2:3]
    k1, k2, k3 = axis(ex), axis(ey), axis(ez)
    qx, qy = k * (_dot(prop, ex)[:, None] - k1), k * (_dot(prop, ey)[:, None] - k2)
    Fr, Fi = _form_factor(qx, qy, X, Y, nv, amax)
    del qx, qy
    rc = c @ g.x
    ph = k * ((_dot(c, c)[:, None] - 2 * rc) / (rho + g.rad))     # k (|x - c| - |x|)
    Ec, Es = torch.cos(ph), torch.sin(ph)
    sr, si = -(Ec * Fi + Es * Fr) / LAM, (Ec * Fr - Es * Fi) / LAM
    del Fr, Fi, Ec, Es, ph, rc, rho
    if cosfov is not None:
        seen = ~(axis(prop) < cosfov[:, None])
        sr, si = sr * seen, si * seen
    k2c = torch.where(k2.abs() > K2CLAMP, torch.sign(k2) * K2CLAMP, k2)
    sq, s13 = torch.sqrt(1 - k2c * k2c), torch.sqrt(1 - k2 * k2)
    fwd = kh[2].abs() >= FWD_DOT
    hx = torch.where(fwd, g.xt[1] - c[:, 1:2], kh[1])
    hy = torch.where(fwd, -(g.xt[0] - c[:, 0:1]), -kh[0])
    nh = torch.sqrt(hx * hx + hy * hy)
    hx, hy = hx / nh, hy / nh
    e0, e1, e2 = ey[:, 0:1], ey[:, 1:2], ey[:, 2:3]
    p = (hx * (e0 - k2c * kh[0]) + hy * (e1 - k2c * kh[1])) / sq
    qh = (hx * (kh[1] * e2 - kh[2] * e1) + hy * (kh[2] * e0 - kh[0] * e2)) / s13
    da, db = -0.5 * (Kz * sq + k3 / sq), -0.5 * k1 * k2c / sq
    gg, hh = p * da + qh * db, p * db - qh * da
    fg, fh = torch.complex(sr * gg, si * gg), torch.complex(sr * hh, si * hh)
    A = torch.view_as_complex(C.reshape(-1, 4, 2).contiguous())       # (1,1) (2,1) (1,2) (2,2)
    JA = torch.stack([A[:, 1], -A[:, 0], A[:, 3], -A[:, 2]], 1)
    Xs = A.T @ fg + JA.T @ fh
    T = lambda a: torch.complex(a, torch.zeros_like(a))
    cp, sp = T(g.cphi), T(g.sphi)                                     # times [[-s, -c], [c, -s]]
    return torch.stack([-sp * Xs[0] + cp * Xs[2], -sp * Xs[1] + cp * Xs[3],
                        -cp * Xs[0] - sp * Xs[2], -cp * Xs[1] - sp * Xs[3]])


def _beams_of(b: BeamSet, g, fast, fov):
    verts, nv = _padded(b, g.dev)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(g.dev)
    cosfov = torch.cos(t(b.fov) if fov is None else torch.full((b.n,), fov, dtype=torch.float64, device=g.dev))
    return [t(b.ampl), t(b.vk7), t(b.prop), verts, nv, cosfov if fast else None]


def _sum(g, beams, i0, i1):
    X = torch.zeros((4, g.n), dtype=torch.complex128, device=g.dev)
    step = max(1, int(2.5e7 // g.n))
    for j in range(i0, i1, step):
        X += _amplitudes(g, *[None if a is None else a[j:min(i1, j + step)] for a in beams])
    return X * g.phase


def _mueller(X):
    """(16, nbins) of the amplitudes (1,1) (2,1) (1,2) (2,2)."""
    a, b, c, d = X[0], X[2], X[1], X[3]           # J = [[a, b], [c, d]]
    U = torch.tensor([[1, 0, 0, 1], [1, 0, 0, -1], [0, 1, 1, 0], [0, 1j, -1j, 0]], dtype=X.dtype, device=X.device)
    cj = lambda z: z.conj()
    K = torch.stack([a * cj(a), a * cj(b), b * cj(a), b * cj(b), a * cj(c), a * cj(d), b * cj(c), b * cj(d),
                     c * cj(a), c * cj(b), d * cj(a), d * cj(b), c * cj(c), c * cj(d), d * cj(c), d * cj(d)])
    return torch.einsum("ij,jkn,kl->iln", U, K.reshape(4, 4, -1), torch.linalg.inv(U)).real.reshape(16, -1)


def _weights(x):
    """Weights of the three-point panels on the nodes x; an even count ends with the last parabola's
    integral over the final interval."""
    n, w = len(x), np.zeros(len(x))

    def add(i, lo, hi):
        for j in range(3):
            o = [x[i + q] for q in range(3) if q != j]
            den = (x[i + j] - o[0]) * (x[i + j] - o[1])
            f = lambda t: t * t * t / 3 - (o[0] + o[1]) * t * t / 2 + o[0] * o[1] * t
            w[i + j] += (f(hi) - f(lo)) / den

    for i in range(0, n - 2, 2):
        add(i, x[i], x[i + 2])
    if n % 2 == 0:
        add(n - 3, x[n - 2], x[n - 1])
    return w


def _pairs(X):
    """The Fortran layout (phi fastest, entries (1,1) (2,1) (1,2) (2,2)) as doubles."""
    return torch.view_as_real(X.contiguous()).reshape(-1)


def _integrals(M, th, ph, k):
    wt, wp = _weights(th), _weights(ph)
    w = torch.from_numpy(((wt * np.sin(th) / k ** 2)[:, None] * wp).ravel()).to(M.device)
    c = torch.from_numpy(np.repeat(np.cos(th), len(ph))).to(M.device)
    return float((w * M[0]).sum()), float((w * c * M[0]).sum())


def _one_d(M, ph):
    return M.reshape(16, -1, len(ph)) @ torch.from_numpy(_weights(ph)).to(M.device)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("vis_batch", "vis_call"):
        return None      # flags, ids, and differences of input heights: equal, not near
    th, ph = _angles(case)
    g = _Bins(th, ph)
    if kind == "retrieval":
        return _exact_retrieval(case, seed, g)
    B, E, boff, eoff = _trees(case, seed)
    fast = case.get("fast_diff", False)
    b = _beams_of(B, g, fast, None)
    if kind == "diffraction":
        i = seed % B.n
        X = _sum(g, b, i, i + 1)
        return X.reshape(2, 2, g.nth, g.nph).transpose(0, 1).cpu().numpy()
    e = _beams_of(E, g, fast, EXT_FOV)
    if kind == "batch":
        M, I = 0.0, []
        for o in range(case["norient"]):
            xb, xe = _sum(g, b, boff[o], boff[o + 1]) * g.k, _sum(g, e, eoff[o], eoff[o + 1]) * g.k
            m = _mueller(xb + xe)
            M = M + m
            I += [v for x in (m, _mueller(xb), _mueller(xe)) for v in _integrals(x, th, ph, g.k)]
        return {"mueller": M.reshape(-1), "mueller_1d": _one_d(M, ph).reshape(-1), "integrals": np.array(I)}
    xb, xe = _sum(g, b, 0, B.n), _sum(g, e, 0, E.n)
    if kind == "diff_main":
        return {"beam": _pairs(xb), "ext": _pairs(xe)}
    xb, xe = xb * g.k, xe * g.k
    f = [0.0, 0.0]
    if case["scaling"]:
        f = [math.sqrt(_integrals(_mueller(x), th, ph, g.k)[0] / en) for x, en in zip((xb, xe), _energies(seed))]
        xb, xe = xb / f[0], xe / f[1]
    ms = [_mueller(x) for x in (xb + xe, xb, xe)]
    I = [_integrals(m, th, ph, g.k) for m in ms]
    back = int(np.argmin(np.abs(th - 2 * PI_R4)))
    par = [v[0] for v in I] + [v[1] / v[0] for v in I] + [float(ms[0][0, g.nph * back]) * 4 * PI_R4 / g.k ** 2] + f
    return {"beam": _pairs(xb), "ext": _pairs(xe), "mueller": torch.cat([m.reshape(-1) for m in ms]),
            "mueller_1d": torch.cat([_one_d(m, ph).reshape(-1) for m in ms]), "params": np.array(par)}


def _exact_retrieval(case, seed, g):
    dev = g.dev
    t, verts, ampl = _retrieval(case, seed, dev)
    ampl = dict(zip(("beams", "ext"), ampl))
    faces, rots = torch.as_tensor(t["faces"], device=dev), torch.as_tensor(t["rots"], dtype=torch.float64, device=dev)
    off = {"beams": t["beam_off"].cpu().numpy(), "ext": t["ext_off"].cpu().numpy()}
    step = max(1, int(4e6 // g.n))

    def parts(o):
        for k in ("beams", "ext"):
            for j in range(off[k][o], off[k][o + 1], step):
                q = slice(j, min(off[k][o + 1], j + step))
                vt = torch.einsum("ij,bvj->bvi", rots[o], verts[faces[t[k]["fi"][q] - 1]])
                nv = torch.full((vt.shape[0],), 3.0, dtype=torch.float64, device=dev)
                yield _amplitudes(g, ampl[k][q], t[k]["vk7"][q], t[k]["prop"][q], vt, nv) * (g.phase * g.k)

    X = torch.zeros((case["norient"], 4, g.n), dtype=torch.complex128, device=dev)
    with torch.no_grad():
        for o in range(case["norient"]):
            for a in parts(o):
                X[o] += a
    Xr = torch.view_as_real(X).permute(0, 1, 3, 2).reshape(case["norient"], 8, g.n).contiguous().requires_grad_(True)
    a = Xr * Xr
    i1, i2, i3, i4 = a[:, 0] + a[:, 1], a[:, 2] + a[:, 3], a[:, 4] + a[:, 5], a[:, 6] + a[:, 7]
    m11, m12 = (0.5 * (i1 + i3 + i2 + i4)).mean(0), (0.5 * (i1 - i3 + i2 - i4)).mean(0)
    t11, tp, w = _target(case, seed, dev)
    loss = (w * (((m11 - t11) / t11) ** 2 + (-m12 / m11 - tp) ** 2)).sum()
    loss.backward()
    G = Xr.grad
    for o in range(case["norient"]):
        for p in parts(o):
            r = torch.view_as_real(p).permute(0, 2, 1).reshape(8, g.n)
            (r * G[o]).sum().backward()
    return {"loss": loss.detach(), "X": Xr.detach(), "grad_vertices": verts.grad, "grad_beam": ampl["beams"].grad,
            "grad_ext": ampl["ext"].grad}
