"""What a user of matvis_amd has it compute, as cases that can be timed.

Five kinds of work, each through the package's public entry points:

* ``vis``: one ``simulate_vis`` call, host arrays in, host visibilities out
  (everything a script pays for: chunking, beam tables, uploads, the time
  loop, delivery);
* ``time``: one time sample of a set-up ``VisibilityEngine`` (rotation and
  cull, then beam, Z, HERK and expansion per frequency), the result left in
  device memory: the steady state of a long simulation;
* ``chain``: one time through the plugin classes (``CoordinateRotation``,
  ``GPUBeamInterpolator``, ``TauCalculator``, ``ZMatrixCalc``, a ``MatProd``),
  as a program that customises one of them drives them;
* ``batch``: many instances of different sizes as grouped HERKs in a captured
  graph, expanded to visibilities: a serving step;
* ``matprod``: the source sum alone, one ``MatProd`` fed with Z by chunk.

The split (mixed precision) forms deliver complex64, which holds all the
accuracy they have; the plain forms deliver what their precision gives.
"""

from __future__ import annotations

import math
from functools import lru_cache

import numpy as np
import torch

from matvis_amd import astro, simulate_vis, synth
from matvis_amd._lib import FORM_SPLIT_BF16, call
from matvis_amd.beams import GaussianBeam
from matvis_amd.core.coords import CoordinateRotation
from matvis_amd.core.getz import ZMatrixCalc
from matvis_amd.core.tau import TauCalculator
from matvis_amd.gpu import matprod as matprods
from matvis_amd.gpu.beams import GPUBeamInterpolator
from matvis_amd.gpu.gpu import build_engine
from matvis_amd.gpu.herk import expand, split_terms_alloc
from matvis_amd.gpu.herk_group import GroupedBatch, tile_for

C_LIGHT = 299792458.0
LAT = math.radians(synth.HERA_LAT_DEG)
#: share of the sky model above the horizon (sin(dec) uniform on [-1, 0.5])
UP = 0.6

#: matprod method -> relative cost of its source sum
METHODS = {"GPUMatMul": 4.0, "GPUMatMulSplitBF16": 1.0,
           "GPUMatMulSplitF16": 1.0}


def _case(name, kind, **kw):
    d = dict(kind=kind, nant=32, nsrc=1000, nfreq=1, ntimes=1, polarized=True,
             precision=2, method="GPUMatMul", terms=0, beam="grid", order=3,
             nbeam=1, coords="CoordinateRotationMatrix", chunks=1,
             pairs="all", ninst=0)
    d.update(kw)
    if name:
        d["name"] = name
    return d


def listed():
    return [
        # a script's first try, or a unit test: everything is latency
        _case("vis_tiny", "vis", nant=6, nsrc=120, polarized=False,
              precision=1, beam="gauss", order=1),
        # an ordinary call: a small hexagon, the ERFA rotation, double precision
        _case("vis_pol_erfa_f64", "vis", nant=37, nsrc=2500, nfreq=8, ntimes=4,
              coords="CoordinateRotationERFA"),
        # a larger call with each baseline once, in mixed precision
        _case("vis_pairs_f16", "vis", nant=128, nsrc=30011, nfreq=8, ntimes=4,
              precision=1, method="GPUMatMulSplitF16", pairs="upper"),
        # many channels of a small array, the defaults (single precision,
        # bilinear beam, one feed)
        _case("time_small_c64", "time", nant=32, nsrc=3000, nfreq=32,
              polarized=False, precision=1, order=1),
        # an odd-sized array whose antennas have four different beams
        _case("time_odd_f64", "time", nant=61, nsrc=20011, nfreq=6, nbeam=4),
        # a mid-sized array, one feed, mixed precision
        _case("time_mid_bf16", "time", nant=128, nsrc=50000, nfreq=16,
              polarized=False, precision=1, method="GPUMatMulSplitBF16"),
        # the full array and sky over the band, mixed precision
        _case("time_full_bf16", "time", nant=350, nsrc=100000, nfreq=20,
              precision=1, method="GPUMatMulSplitBF16"),
        # the full array in single precision (the default)
        _case("time_full_c64", "time", nant=350, nsrc=100000, nfreq=4,
              precision=1),
        # the full array in double precision
        _case("time_full_f64", "time", nant=350, nsrc=50000, nfreq=3),
        # a diffuse sky in chunks, four beams, three bfloat16 terms
        _case("time_diffuse_bf16x3", "time", nant=350, nsrc=196608, nfreq=2,
              precision=1, method="GPUMatMulSplitBF16", terms=3, nbeam=4,
              chunks=12),
        # the plugin classes one by one, two source chunks
        _case("chain_f64", "chain", nant=50, nsrc=6007, chunks=2),
        # a serving step: instances of three array sizes, ragged columns
        _case("batch_bf16", "batch", nant=350, nsrc=20000, ninst=24,
              precision=1, method="GPUMatMulSplitBF16"),
    ]


def _cost(c):
    """Relative work of a case (its source sums), for draw()."""
    m = c["nant"] * (2 if c["polarized"] else 1)
    k = c["nsrc"] * (2 if c["polarized"] else 1)
    w = METHODS[c["method"]] * (2.0 if c["terms"] == 3 else 1.0)
    if c["kind"] == "batch":
        return 0.25 * c["ninst"] * m * m * k * w
    return c["nfreq"] * c["ntimes"] * w * m * m * k


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vis", "time", "time", "time", "chain", "batch",
                       "matprod"])
    pol = rng.random() < 0.5
    method = rng.choice(list(METHODS))
    c = _case(None, kind, polarized=pol, method=method,
              nant=_log(rng, 6, 400), nsrc=_log(rng, 150, 120000),
              beam=rng.choice(["gauss", "grid"]), order=rng.choice([1, 3]))
    c["precision"] = 1 if method != "GPUMatMul" else rng.choice([1, 2])
    if method == "GPUMatMulSplitBF16" and rng.random() < 0.3:
        c["terms"] = 3
    top = _cost(next(x for x in listed() if x["name"] == "time_full_bf16"))
    if kind == "batch":
        c.update(ninst=rng.randint(2, 32), nant=rng.choice([64, 128, 350]),
                 nsrc=_log(rng, 3000, 40000), method="GPUMatMulSplitBF16",
                 precision=1, terms=0, polarized=True, nfreq=1)
        while _cost(c) > top:
            c["ninst"] = max(2, c["ninst"] // 2)
            c["nsrc"] = c["nsrc"] * 2 // 3
        return c
    if kind == "chain":
        # the chain keeps the phase, the beam and Z as arrays of their own
        c.update(nant=_log(rng, 6, 130), nsrc=_log(rng, 150, 20000),
                 method="GPUMatMul", precision=2, terms=0)
    elif kind == "matprod":
        c.update(nsrc=_log(rng, 50, 40000), nbeam=1)
    else:
        c.update(nfreq=_log(rng, 1, 32),
                 nbeam=1 if rng.random() < 0.7 else 4,
                 pairs=rng.choice(["all", "upper"]))
    if kind == "vis":
        c["ntimes"] = rng.randint(1, 5)
        c["coords"] = rng.choice(["CoordinateRotationMatrix",
                                  "CoordinateRotationERFA"])
    if c["nsrc"] > 5000:
        c["chunks"] = rng.choice([1, 1, 2, 5])
    while _cost(c) > 0.8 * top:
        if c["nfreq"] > 1:
            c["nfreq"] //= 2
        else:
            c["nsrc"] = c["nsrc"] * 2 // 3
    return c


# ------------------------------------------------------------------ inputs

@lru_cache(maxsize=8)
def _grid_beam(seed):
    """A smooth complex64 E-field beam on a 1 degree grid (a telescope keeps
    its beams from run to run)."""
    return synth.harmonic_efield_beam(seed=seed)


@lru_cache(maxsize=16)
def _perturbed_beam(seed, k):
    return synth.harmonic_efield_beam(seed=seed, perturb=0.05, perturb_seed=k)


def _beams(case):
    n = case["nbeam"]
    if case["beam"] == "gauss":
        return [GaussianBeam(sigma=math.radians(s))
                for s in (10.0, 14.0, 7.0, 20.0)[:n]]
    if n == 1:
        return [_grid_beam(4)]
    return [_perturbed_beam(4, k) for k in range(n)]


def _contexts(rng, ntimes):
    """Per-time astrometry contexts of an observer at the array's latitude
    (Sun direction and distance, barycentric velocity, precession-nutation,
    local Earth rotation angle, polar motion)."""
    e = rng.normal(size=3)
    v = rng.normal(size=3)
    v *= 9.9e-5 / np.linalg.norm(v)
    a, b, g = rng.uniform(-2e-3, 2e-3, size=3)
    ca, sa, cb, sb = math.cos(a), math.sin(a), math.cos(b), math.sin(b)
    cg, sg = math.cos(g), math.sin(g)
    bpn = (np.array([[ca, -sa, 0], [sa, ca, 0], [0, 0, 1.0]])
           @ np.array([[cb, 0, sb], [0, 1.0, 0], [-sb, 0, cb]])
           @ np.array([[1.0, 0, 0], [0, cg, -sg], [0, sg, cg]]))
    era = rng.uniform(0, 2 * math.pi)
    return [dict(eh=e / np.linalg.norm(e), em=1.0 + 0.016 * math.sin(era),
                 v=v, bm1=math.sqrt(1.0 - float(v @ v)), bpn=bpn,
                 eral=era + 0.00873 * t, xpl=5e-7, ypl=-8e-7,
                 sphi=math.sin(LAT), cphi=math.cos(LAT))
            for t in range(ntimes)]


def _inputs(case, seed):
    """The arrays a user's program holds, from the seed alone."""
    rng = np.random.default_rng(seed)
    nant, nsrc, nfreq = case["nant"], case["nsrc"], case["nfreq"]
    antpos = synth.hex_array(nant, 14.6, 0.02, seed=int(rng.integers(1 << 30)))
    ra, dec = synth.random_sky(nsrc, int(rng.integers(1 << 30)))
    flux0 = synth.lognormal_fluxes(nsrc, int(rng.integers(1 << 30)))
    freqs = np.linspace(110e6, 190e6, nfreq)
    index = rng.uniform(-1.2, -0.4, size=nsrc)
    fluxes = flux0[:, None] * np.exp(index[:, None]
                                     * np.log(freqs[None] / 150e6))
    times = synth.times_spaced(case["ntimes"], 2.0,
                               synth.START_JD + float(rng.uniform(0, 1)))
    loc = synth.hera_location()
    if case["coords"] == "CoordinateRotationERFA":
        params = {"astrom": _contexts(rng, case["ntimes"])}
    else:
        params = {"rotations": astro.rotation_matrices(times, loc)}
    beam_idx = (None if case["nbeam"] == 1
                else (np.arange(nant) % case["nbeam"]).astype(np.int32))
    pairs = (None if case["pairs"] == "all"
             else [(i, j) for i in range(nant) for j in range(i, nant)])
    return dict(antpos=antpos, ra=ra, dec=dec, fluxes=fluxes, freqs=freqs,
                times=times, loc=loc, params=params, beam_idx=beam_idx,
                pairs=pairs, beams=_beams(case))


def _options(case, w):
    """Keywords that simulate_vis and build_engine share."""
    kw = dict(polarized=case["polarized"], precision=case["precision"],
              beam_spline_opts={"order": case["order"]},
              beam_idx=w["beam_idx"], antpairs=w["pairs"],
              coord_method=case["coords"], coord_method_params=w["params"],
              matprod_method=case["method"], min_chunks=case["chunks"])
    if case["terms"]:
        kw["split_terms"] = case["terms"]
    return kw


def _instances(case):
    """(nant, nfeed, columns above the horizon) of a batch's instances."""
    rng = np.random.default_rng(case["ninst"])
    out = []
    for _ in range(case["ninst"]):
        nant = int(rng.choice([case["nant"], max(32, case["nant"] // 3), 64]))
        nup = int(math.exp(rng.uniform(math.log(case["nsrc"] / 10),
                                       math.log(case["nsrc"]))))
        out.append((nant, int(rng.integers(1, 3)), nup))
    return out


def _zmatrix(gen, m, ncols, dtype, device="cuda"):
    """Z as the path forms it: log-normal amplitudes, phases at random."""
    re = torch.float64 if dtype == torch.complex128 else torch.float32
    amp = torch.exp(0.5 * torch.randn((1, ncols), dtype=re, device=device,
                                      generator=gen))
    amp = amp * torch.rand((m, ncols), dtype=re, device=device, generator=gen)
    ph = 2 * math.pi * torch.rand((m, ncols), dtype=re, device=device,
                                  generator=gen)
    return torch.polar(amp, ph)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _batch_z(case, seed):
    gen = _gen(seed)
    return [(nant, nf, nup, _zmatrix(gen, nant * nf, nf * nup,
                                     torch.complex64))
            for nant, nf, nup in _instances(case)]


def _matprod_z(case, seed):
    gen = _gen(seed)
    nf = 2 if case["polarized"] else 1
    dt = torch.complex128 if case["precision"] == 2 else torch.complex64
    base, extra = divmod(case["nsrc"], case["chunks"])
    return [_zmatrix(gen, nf * case["nant"],
                     nf * max(1, base + (c < extra)), dt)
            for c in range(case["chunks"])]


def _make_matprod(case, pairs=None):
    nf = 2 if case["polarized"] else 1
    kw = {"split_terms": case["terms"]} if case["terms"] else {}
    mp = getattr(matprods, case["method"])(
        case["chunks"], nf, case["nant"], pairs, precision=case["precision"],
        **kw)
    mp.setup()
    out = np.zeros((mp.npairs, nf, nf), dtype=mp.ctype)
    return mp, out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        probs, shape = [], []
        for nant, nf, nup, z in _batch_z(case, seed):
            m, seg = nant * nf, -(-nup // 16) * 16
            terms = split_terms_alloc(2, m, nf * seg)
            call("mv_split_z", z.data_ptr(), 0, m, nf, nup, nf * nup, nup,
                 FORM_SPLIT_BF16, 2, 1.0, terms[0].data_ptr(),
                 terms[1].data_ptr(), None, m, seg,
                 torch.cuda.current_stream().cuda_stream)
            torch.cuda.current_stream().synchronize()
            ldv = -(-m // 128) * 128
            probs.append(dict(terms=terms, m=m, ldz=m, nseg=nf,
                              seg_stride=seg, seg_len=nup, ldv=ldv,
                              vacc=torch.zeros((ldv, ldv), device="cuda",
                                               dtype=torch.complex128),
                              scale=1.0, accumulate=False))
            shape.append((nant, nf))
        tiles = [tile_for(FORM_SPLIT_BF16, p["m"]) for p in probs]
        batch = GroupedBatch(FORM_SPLIT_BF16, 2, 3, probs, tiles)
        batch.capture()
        outs = [torch.zeros((a * a, f, f), dtype=torch.complex64,
                            device="cuda") for a, f in shape]
        return dict(kind=kind, batch=batch, probs=probs, shape=shape,
                    outs=outs)
    if kind == "matprod":
        mp, out = _make_matprod(case)
        return dict(kind=kind, z=_matprod_z(case, seed), mp=mp, out=out)
    w = _inputs(case, seed)
    if kind == "vis":
        kw = _options(case, w)
        return dict(kind=kind, kw=dict(
            ants=dict(enumerate(w["antpos"])), fluxes=w["fluxes"], ra=w["ra"],
            dec=w["dec"], freqs=w["freqs"], times=w["times"],
            beams=w["beams"], telescope_loc=w["loc"], use_gpu=True, **kw))
    sky = astro.SkyCoord(w["ra"], w["dec"])
    if kind == "time":
        engine, _ = build_engine(
            antpos=w["antpos"], freqs=w["freqs"], times=w["times"],
            skycoords=sky, telescope_loc=w["loc"], fluxes=w["fluxes"],
            beam_list=w["beams"], **_options(case, w))
        return dict(kind=kind, engine=engine, out=engine.new_output())
    # chain: one set-up object of each plugin
    chunk = -(-case["nsrc"] // case["chunks"])
    nf = 2 if case["polarized"] else 1
    prec = case["precision"]
    co = CoordinateRotation._methods[case["coords"]](
        flux=np.sqrt(0.5 * w["fluxes"][:, 0]), times=w["times"],
        telescope_loc=w["loc"], skycoords=sky, chunk_size=chunk,
        precision=prec, source_buffer=1.0, **w["params"])
    co.setup()
    beam = GPUBeamInterpolator(w["beams"], w["beam_idx"], case["polarized"],
                               case["nant"], float(w["freqs"][0]),
                               co.nsrc_alloc,
                               spline_opts={"order": case["order"]},
                               precision=prec)
    beam.setup()
    tau = TauCalculator(w["antpos"], float(w["freqs"][0]), co.nsrc_alloc,
                        precision=prec)
    tau.setup()
    zc = ZMatrixCalc(case["nant"], nf, nf, co.nsrc_alloc, co.ctype)
    zc.setup()
    mp, out = _make_matprod(case, w["pairs"])
    return dict(kind=kind, co=co, beam=beam, tau=tau, z=zc, mp=mp, out=out,
                chunks=case["chunks"])


# --------------------------------------------------------------------- run

def run(s):
    kind = s["kind"]
    if kind == "vis":
        return simulate_vis(**s["kw"])
    if kind == "time":
        return s["engine"].compute_time(0, s["out"])
    if kind == "matprod":
        for c, z in enumerate(s["z"]):
            s["mp"](z, c)
        return s["mp"].sum_chunks(s["out"])
    if kind == "chain":
        s["co"].rotate(0)
        for c in range(s["chunks"]):
            crd, flux, _ = s["co"].select_chunk(c, 0)
            a = s["beam"](crd[0], crd[1], check=False)
            z = s["z"](flux, a, s["tau"](crd), s["beam"].beam_idx)
            s["mp"](z, c)
        return s["mp"].sum_chunks(s["out"])
    s["batch"].replay()
    for p, (nant, nf), out in zip(s["probs"], s["shape"], s["outs"]):
        expand(p["vacc"], p["ldv"], 128, nant, nf, None, nant * nant, out)
    return s["outs"]


# -------------------------------------------------------------------- work

def work(case):
    kind = case["kind"]
    csz = 16 if case["precision"] == 2 else 8

    def herk(m, k):
        return 8.0 * k * m * (m + 1) / 2

    if kind == "batch":
        inst = _instances(case)
        return dict(bytes=sum(a * f * f * n * 8 + a * a * f * f * csz
                              for a, f, n in inst),
                    flops=sum(herk(a * f, f * n) for a, f, n in inst))
    nf = 2 if case["polarized"] else 1
    m = nf * case["nant"]
    npairs = (case["nant"] ** 2 if case["pairs"] == "all"
              else case["nant"] * (case["nant"] + 1) // 2)
    if kind == "matprod":
        k = nf * case["nsrc"]
        return dict(bytes=m * k * csz + npairs * nf * nf * csz,
                    flops=herk(m, k))
    grid = case["nbeam"] * nf * nf * 360 * 91 * 8 if case["beam"] == "grid" \
        else 0
    passes = case["nfreq"] * case["ntimes"]
    return dict(bytes=case["nsrc"] * (16 + 8 * case["nfreq"]) + grid
                + passes * npairs * nf * nf * csz,
                flops=passes * herk(m, nf * UP * case["nsrc"]))


# ------------------------------------------------------------------- exact

def _enu_exact(case, w):
    """Topocentric unit vectors (3, nsrc) of each time, FP64 on the GPU."""
    ra, dec = (torch.from_numpy(w[k]).cuda() for k in ("ra", "dec"))
    p = torch.stack([torch.cos(ra) * torch.cos(dec),
                     torch.cos(dec) * torch.sin(ra), torch.sin(dec)])
    out = []
    for t in range(case["ntimes"]):
        q = p
        if case["coords"] == "CoordinateRotationERFA":
            c = w["params"]["astrom"][t]
            srs = 1.97412574336e-8  # Schwarzschild radius of the Sun, au
            e = torch.tensor(c["eh"], device="cuda")[:, None]
            v = torch.tensor(c["v"], device="cuda")[:, None]
            den = (p * (p + e)).sum(0).clamp(min=1e-6)
            ex = e.expand_as(p)
            q = p + srs / c["em"] / den * torch.cross(
                p, torch.cross(ex, p, dim=0), dim=0)
            pdv = (q * v).sum(0)
            w2 = srs / c["em"]
            q = (c["bm1"] * q + (1 + pdv / (1 + c["bm1"])) * v
                 + w2 * (v - pdv * q * c["bm1"]))
            q = q / q.norm(dim=0)
            q = (torch.tensor(c["bpn"], device="cuda")[:, :, None]
                 * q[None]).sum(1)
            ce, se = math.cos(c["eral"]), math.sin(c["eral"])
            sx, cx = math.sin(c["xpl"]), math.cos(c["xpl"])
            sy, cy = math.sin(c["ypl"]), math.cos(c["ypl"])
            rot = (np.array([[0, 1.0, 0], [-c["sphi"], 0, c["cphi"]],
                             [c["cphi"], 0, c["sphi"]]])
                   @ np.array([[cx, 0, sx], [sx * sy, cy, -cx * sy],
                               [-sx * cy, sy, cx * cy]])
                   @ np.array([[ce, se, 0], [-se, ce, 0], [0, 0, 1.0]]))
        else:
            rot = w["params"]["rotations"][t]
        out.append(torch.stack([rot[i, 0] * q[0] + rot[i, 1] * q[1]
                                + rot[i, 2] * q[2] for i in range(3)]))
    return out


def _spline_matrix(n):
    """Cubic B-spline samples of its coefficients, mirrored ends."""
    a = (torch.eye(n, dtype=torch.float64) * 4
         + torch.diag(torch.ones(n - 1, dtype=torch.float64), 1)
         + torch.diag(torch.ones(n - 1, dtype=torch.float64), -1))
    a[0, 1] = a[n - 1, n - 2] = 2.0
    return (a / 6.0).cuda()


def _weights(x, order):
    f = torch.floor(x)
    t = x - f
    if order == 1:
        return f.long(), [1 - t, t]
    u = 1 - t
    return f.long() - 1, [u ** 3 / 6, (3 * t ** 3 - 6 * t ** 2 + 4) / 6,
                          (3 * u ** 3 - 6 * u ** 2 + 4) / 6, t ** 3 / 6]


def _mirror(i, n):
    i = i.abs() % (2 * (n - 1))
    return torch.where(i >= n, 2 * (n - 1) - i, i)


def _beam_planes_exact(case, beams):
    """Per beam (planes (nfeed, nax, nza, naz) complex128 or real, azmin)."""
    out = []
    for b in beams:
        d = torch.from_numpy(b.data_array[:, :, 0]).cuda().to(
            torch.complex128)
        if case["polarized"]:
            g = d.transpose(0, 1)  # (nfeed, nax, nza, naz)
        else:
            g = (d[:, 0].abs() ** 2).sum(0)[None, None].to(torch.complex128)
        g = torch.cat([g[..., -3:], g, g[..., :3]], -1)
        if case["order"] == 3:
            sz = _spline_matrix(g.shape[-2])
            sa = _spline_matrix(g.shape[-1])
            for k in range(g.shape[0]):
                for j in range(g.shape[1]):
                    parts = []
                    for part in (g[k, j].real, g[k, j].imag):
                        x = torch.linalg.solve(sz, part.contiguous())
                        x = torch.linalg.solve(sa, x.T.contiguous())
                        parts.append(x.T)
                    g[k, j] = torch.complex(parts[0], parts[1])
        daz = float(b.axis1_array[1] - b.axis1_array[0])
        dza = float(b.axis2_array[1] - b.axis2_array[0])
        out.append((g, daz, dza, float(b.axis1_array[0]) - 3 * daz))
    return out


def _beam_exact(case, beams, planes, crd):
    """(nbeam, nfeed, nax, nsrc) response at topocentric vectors crd."""
    e, n = crd[0], crd[1]
    l2 = e * e + n * n
    zeta = torch.sqrt((1 - l2).clamp(min=0))
    za = math.pi / 2 - torch.asin(zeta)
    az = torch.remainder(math.pi / 2 - torch.atan2(e, n), 2 * math.pi)
    nf = 2 if case["polarized"] else 1
    resp = []
    if case["beam"] == "gauss":
        for b in beams:
            a = torch.exp(-za ** 2 / (2 * b.sigma ** 2))
            a = a / math.sqrt(2.0) if case["polarized"] else a
            resp.append(a.to(torch.complex128).expand(nf, nf, -1))
        return torch.stack(resp)
    for g, daz, dza, azmin in planes:
        nza, naz = g.shape[-2:]
        x, y = za / dza, (az - azmin) / daz
        ok = (x >= 0) & (x <= nza - 1) & (y >= 0) & (y <= naz - 1)
        x0, wx = _weights(x, case["order"])
        y0, wy = _weights(y, case["order"])
        v = 0
        for i, wi in enumerate(wx):
            for j, wj in enumerate(wy):
                v = v + (wi * wj) * g[..., _mirror(x0 + i, nza),
                                      _mirror(y0 + j, naz)]
        v = torch.where(ok, v, torch.zeros_like(v))
        resp.append(v if case["polarized"] else torch.sqrt(v))
    return torch.stack(resp)


def _expand_exact(z, nant, nf, pairs):
    v = torch.mm(z.conj().resolve_conj(), z.T.contiguous())
    v = v.reshape(nant, nf, nant, nf).permute(0, 2, 3, 1)
    if pairs is None:
        return v.reshape(nant * nant, nf, nf)
    idx = torch.tensor(pairs, device="cuda")
    return v[idx[:, 0], idx[:, 1]]


def exact(case, seed):
    kind, nant = case["kind"], case["nant"]
    nf = 2 if case["polarized"] else 1
    if kind == "batch":
        return [_expand_exact(z.to(torch.complex128), a, f, None)
                for a, f, _, z in _batch_z(case, seed)]
    if kind == "matprod":
        return sum(_expand_exact(z.to(torch.complex128), nant, nf, None)
                   for z in _matprod_z(case, seed)).cpu().numpy()
    w = _inputs(case, seed)
    beams = w["beams"]
    planes = None if case["beam"] == "gauss" else _beam_planes_exact(case,
                                                                     beams)
    ant = torch.from_numpy(w["antpos"]).cuda()
    flux = torch.from_numpy(w["fluxes"]).cuda()
    bi = (torch.zeros(nant, dtype=torch.long) if w["beam_idx"] is None
          else torch.from_numpy(w["beam_idx"].astype(np.int64))).cuda()
    vis = []
    for enu in _enu_exact(case, w):
        up = enu[2] > 0
        crd = enu[:, up]
        resp = _beam_exact(case, beams, planes, crd)
        delay = (ant[:, 0:1] * crd[0] + ant[:, 1:2] * crd[1]
                 + ant[:, 2:3] * crd[2]) / C_LIGHT
        per = []
        for f, nu in enumerate(w["freqs"]):
            turns = delay * float(nu)
            ph = 2 * math.pi * (turns - torch.round(turns))
            e = torch.polar(torch.sqrt(0.5 * flux[up, f]).expand(nant, -1)
                            .contiguous(), ph)
            z = (resp[bi] * e[:, None, None, :]).reshape(nant * nf, -1)
            per.append(_expand_exact(z, nant, nf, w["pairs"]))
        vis.append(torch.stack(per))
    v = torch.stack(vis, 1)  # (nfreq, ntimes, npairs, nfeed, nfeed)
    if kind == "time":
        return v[:, 0]
    if kind == "chain":
        return v[0, 0].cpu().numpy()
    return (v if case["polarized"] else v[..., 0, 0]).cpu().numpy()
