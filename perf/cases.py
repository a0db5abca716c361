"""Performance cases: what users of the package have it compute, through its
public entry points.

A case is a dict of plain values.  prepare() makes what a program holds
before the call (structures, histograms, q meshes, output buffers, the one
Context it keeps), run() is one pass through the entry points, work() the
bytes and operations of a pass, and exact() the same results from torch or
numpy in FP64.  listed() holds the named cases, draw() others of the same
ranges.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "softx-d-16-00083_amd"))

import xansons_hip as xh  # noqa: E402
from xansons_hip import calculators as calc  # noqa: E402
from xansons_hip import structures as st  # noqa: E402
from xansons_hip.atoms import Atoms, Block  # noqa: E402

EPS = 1e-8                       # the calculators' sin(x) / (x + 1e-8)
SL = (3.63, 9.577, 7.63, 6.646)  # neutron scattering lengths, by element
_CTX = []


def _ctx():
    """The program's context: made once and kept, as its callers do."""
    if not _CTX:
        _CTX.append(xh.Context(0))
    return _CTX[0]


# ---------------------------------------------------------------- structures
def _rocksalt(ncell, vacancy, sigma, seed):
    return st.rocksalt_cube(ncell=ncell, vacancy=vacancy, sigma=sigma, seed_vac=2 * seed + 1,
                            seed_jit=2 * seed + 2)


def _structure(case, seed):
    """The atoms of a case: a rock-salt cube (with vacancies and displacements,
    or perfect), a nanoparticle, or a disordered solid."""
    kind = case["structure"]
    if kind == "rocksalt":
        # a few atoms at least are missing, so that seeds differ where nothing
        # is displaced
        vacancy = max(case["vacancy"], 10.0 / (8 * case["ncell"] ** 3))
        return _rocksalt(case["ncell"], vacancy, case["sigma"], seed)
    if kind == "disordered":
        n = case["natoms"]
        return st.disordered_cubic(n=math.ceil(n ** (1 / 3)), natoms=n, seed_jit=2 * seed + 1,
                                   seed_species=2 * seed + 2)
    rng = np.random.Generator(np.random.PCG64(seed))
    return st.particle(case["natoms"], case["n_el"], kind, case["a"], case["sigma"], rng)


def _diagonal(case):
    """The bounding-box diagonal that a case's structures stay below, whatever
    their displacements."""
    if case["structure"] == "rocksalt":
        m = case["ncell"]
        return 5.64 * math.sqrt(m * m + 2 * (m - 0.5) ** 2) + 20 * case["sigma"]
    per_cell = 2 if case["structure"] == "bcc" else 4
    v = case["natoms"] * case["a"] ** 3 / per_cell
    side = v ** (1 / 3) if case["structure"] == "cube" else 2 * (0.75 * v / math.pi) ** (1 / 3)
    return math.sqrt(3.0) * side + 20 * case["sigma"]


def _nhist(case):
    return int(_diagonal(case) / case["bin"]) + 1


def _ensemble(case, seed):
    """Uneven particles: their sizes, shapes and element numbers belong to the
    case, the species and displacements to the seed."""
    sizes = np.random.Generator(np.random.PCG64(case["count"]))
    rng = np.random.Generator(np.random.PCG64(seed))
    parts = []
    for _ in range(case["count"]):
        c = {"structure": ("fcc", "bcc", "cube", "core-shell")[int(sizes.integers(0, 4))],
             "natoms": int(np.exp(sizes.uniform(np.log(case["nmin"]), np.log(case["nmax"])))),
             "n_el": int(sizes.integers(1, 5)), "a": float(sizes.uniform(2.8, 4.2)),
             "sigma": 0.05, "bin": case["bin"]}
        parts.append((c, st.particle(c["natoms"], c["n_el"], c["structure"], c["a"], 0.05, rng)))
    return parts


def _natoms(case):
    """About the atoms of a case (exact for a disordered solid)."""
    return 8 * case["ncell"] ** 3 if case["structure"] == "rocksalt" else case["natoms"]


def _n_el(case):
    return {"rocksalt": 2, "disordered": 3}.get(case["structure"]) or case["n_el"]


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _empty(n, dtype=torch.float64):
    return torch.zeros(int(n), dtype=dtype, device="cuda")


def _blocks_of(counts):
    o, out = 0, []
    for c in counts:
        out.append(slice(o, o + int(c)))
        o += int(c)
    return out


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest whole call: host atoms of a 2 nm particle to I(q) and
        # rPDF, where launches, copies and waits count
        {"name": "whole_sphere_2k", "kind": "whole", "structure": "fcc", "natoms": 2000, "n_el": 1,
         "a": 4.078, "sigma": 0.05, "bin": 0.01, "nq": 1024, "qmin": 0.5, "qmax": 10.0},
        # the benchmark's histogram: a 980,000-atom crystal with displacements
        {"name": "hist_cube_980k", "kind": "hist", "structure": "rocksalt", "ncell": 50,
         "vacancy": 0.02, "sigma": 0.08, "bin": 0.005, "f64": True},
        # atoms given without displacement parameters: a perfect lattice
        {"name": "hist_lattice_110k", "kind": "hist", "structure": "rocksalt", "ncell": 24,
         "vacancy": 0.0, "sigma": 0.0, "bin": 0.005, "f64": True},
        # single-precision binning of a core-shell particle of three elements
        {"name": "hist_f32_core_shell_150k", "kind": "hist", "structure": "core-shell",
         "natoms": 150000, "n_el": 3, "a": 3.9, "sigma": 0.05, "bin": 0.01, "f64": False},
        # I(q) and rPDF from the large crystal's histogram
        {"name": "iq_rpdf_97k_bins", "kind": "iq", "ncell": 50, "bin": 0.005, "nhist": 97251,
         "ntypes": 3, "nq": 4096, "qmin": 0.2, "qmax": 25.0},
        # I(q) of many particles on one bin grid, on the matrix cores
        {"name": "iq_many_768", "kind": "iq_many", "count": 256, "nhist": 16384, "bin": 0.004,
         "nq": 8192, "qmin": 0.2, "qmax": 25.0, "nmax": 8000},
        # the manual's direct Debye example: an 8,000-atom NaCl cube
        {"name": "debye_nacl_8000", "kind": "debye", "structure": "rocksalt", "ncell": 10,
         "vacancy": 0.0, "sigma": 0.05, "nq": 1024, "qmin": 0.5, "qmax": 7.0},
        # partial Debye intensities of three structural blocks, host arrays
        {"name": "debye_partial_5k", "kind": "partial", "structure": "fcc", "natoms": 5000,
         "n_el": 2, "a": 4.078, "sigma": 0.05, "nblocks": 3, "nq": 700, "qmin": 0.3, "qmax": 14.0},
        # 2D pattern on a Cartesian q plane, a few orientations
        {"name": "plane_512_50k", "kind": "plane", "structure": "disordered", "natoms": 50000,
         "nu": 512, "nv": 512, "nrot": 8, "qmax": 8.0},
        # 2D pattern on the polar (q, phi) mesh of the 2D scenario
        {"name": "polar_256x360_20k", "kind": "polar", "structure": "core-shell", "natoms": 20000,
         "n_el": 2, "a": 3.9, "sigma": 0.05, "nq": 256, "nfi": 360, "nrot": 4, "qmax": 6.0},
        # a new ensemble of uneven particles: plan, histograms, I(q) and rPDF
        {"name": "ensemble_48", "kind": "ensemble", "count": 48, "nmin": 500, "nmax": 20000,
         "bin": 0.01, "nq": 2048, "qmin": 0.2, "qmax": 25.0},
        # the ensemble builder: symmetry images merged, vacancies, displacements, a cut-off
        {"name": "build_sphere_900k", "kind": "build", "ncell": 60, "occ": 0.98, "sigma": 0.08},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _particle(rng, lo, hi, max_el=4):
    return {"structure": rng.choice(["fcc", "bcc", "cube", "core-shell"]),
            "natoms": _log(rng, lo, hi), "n_el": rng.randint(1, max_el),
            "a": round(rng.uniform(2.8, 4.2), 3), "sigma": rng.choice([0.02, 0.05, 0.08])}


def draw(rng: random.Random):
    kind = rng.choice(["whole", "hist", "hist", "hist_f32", "iq", "iq_many", "debye", "debye",
                       "partial", "plane", "polar", "ensemble", "build"])
    q = {"qmin": round(rng.uniform(0.1, 0.6), 3), "qmax": round(rng.uniform(5.0, 25.0), 2)}
    if kind == "whole":
        return {"kind": "whole", **_particle(rng, 300, 20000), "bin": rng.choice([0.005, 0.01, 0.02]),
                "nq": _log(rng, 100, 2048), **q}
    if kind in ("hist", "hist_f32"):
        c = {"kind": "hist", "bin": round(rng.uniform(0.003, 0.02), 4), "f64": kind == "hist"}
        if rng.random() < 0.5:
            sigma = rng.choice([0.0, 0.03, 0.08])
            return {**c, "structure": "rocksalt", "ncell": _log(rng, 5, 44),
                    "vacancy": rng.choice([0.0, 0.02]), "sigma": sigma}
        return {**c, **_particle(rng, 1000, 400000)}
    if kind == "iq":
        n = _log(rng, 3000, 97251)
        return {"kind": "iq", "ncell": 50, "bin": round(0.005 * 97251 / n, 6), "nhist": n,
                "ntypes": rng.choice([1, 3, 6, 10]), "nq": _log(rng, 200, 4096), **q}
    if kind == "iq_many":
        return {"kind": "iq_many", "count": _log(rng, 48, 256), "nhist": 16384, "bin": 0.004,
                "nq": _log(rng, 1000, 8192), "nmax": _log(rng, 2000, 8000), **q}
    if kind == "debye":
        s = {"structure": "rocksalt", "ncell": _log(rng, 4, 13), "vacancy": 0.02, "sigma": 0.05} \
            if rng.random() < 0.5 else _particle(rng, 300, 16000)
        return {"kind": "debye", **s, "nq": _log(rng, 100, 2048), **q}
    if kind == "partial":
        return {"kind": "partial", **_particle(rng, 300, 10000, 3), "nblocks": rng.randint(2, 5),
                "nq": _log(rng, 100, 1024), **q}
    if kind == "plane":
        return {"kind": "plane", "structure": "disordered", "natoms": _log(rng, 2000, 50000),
                "nu": rng.randint(100, 512), "nv": rng.randint(100, 512), "nrot": rng.randint(1, 8),
                "qmax": round(rng.uniform(4.0, 10.0), 2)}
    if kind == "polar":
        return {"kind": "polar", **_particle(rng, 2000, 20000, 3), "nq": _log(rng, 64, 256),
                "nfi": rng.randint(60, 360), "nrot": rng.randint(1, 4),
                "qmax": round(rng.uniform(4.0, 10.0), 2)}
    if kind == "ensemble":
        return {"kind": "ensemble", "count": _log(rng, 8, 64), "nmin": 500,
                "nmax": _log(rng, 4000, 20000), "bin": 0.01, "nq": _log(rng, 500, 2048), **q}
    return {"kind": "build", "ncell": rng.randint(12, 60), "occ": round(rng.uniform(0.9, 1.0), 3),
            "sigma": rng.choice([0.0, 0.05, 0.08])}


# ---------------------------------------------------------------- prepare
def _q(case):
    return st.q_mesh(case["qmin"], case["qmax"], case["nq"])


def _model_hist(case, seed):
    """Histograms of the pair types of a displaced rock-salt cube: the distances
    of randomly drawn pairs of its atoms, scaled to all pairs.  Types beyond the
    three of two elements repeat them with other draws."""
    nh, bin_ = case["nhist"], case["bin"]
    ens = _rocksalt(case["ncell"], 0.02, 0.08, seed)
    x = _dev(ens.xyz64())
    s = _blocks_of(ens.el_count)
    g = torch.Generator(device="cuda").manual_seed(seed)
    draws = 4_000_000
    out = torch.zeros((case["ntypes"], nh), dtype=torch.int64, device="cuda")
    for p in range(case["ntypes"]):
        a, b = ((0, 0), (0, 1), (1, 1))[p % 3]
        na, nb = ens.el_count[a], ens.el_count[b]
        i = torch.randint(0, na, (draws,), generator=g, device="cuda")
        j = torch.randint(0, nb, (draws,), generator=g, device="cuda")
        r = (x[:, s[a]][:, i] - x[:, s[b]][:, j]).square().sum(0).sqrt()
        k = (r / bin_).long()
        h = torch.bincount(k[(k < nh) & (r > 0.5)], minlength=nh)
        out[p] = h * (na * nb // (2 if a == b else 1) // draws)
    return out, ens


def _pair_hists(x, counts, bin_, nh):
    """Counts of every pair type of one structure in FP64 (device tensor x, a
    (3, N) element-major SoA)."""
    s = _blocks_of(counts)
    out = []
    for a in range(len(counts)):
        for b in range(a, len(counts)):
            h = torch.zeros(nh, dtype=torch.int64, device=x.device)
            xa, xb = x[:, s[a]], x[:, s[b]]
            step = max(1, 16_000_000 // max(1, xb.shape[1]))
            for i in range(0, xa.shape[1], step):
                d = [xa[c, i:i + step, None] - xb[c][None, :] for c in range(3)]
                k = (((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]).sqrt() / bin_).long()
                if a == b:
                    m = torch.arange(xb.shape[1], device=x.device)[None, :] > \
                        torch.arange(i, i + k.shape[0], device=x.device)[:, None]
                    k = k[m]
                k = k.reshape(-1)
                h += torch.bincount(k[k < nh], minlength=nh)
            out.append(h)
    return torch.stack(out)


def prepare(case, seed):
    ctx = _ctx()
    kind = case["kind"]
    s = {"case": case, "ctx": ctx}
    if kind in ("whole", "hist", "debye", "partial", "plane", "polar"):
        ens = _structure(case, seed)
        s["ec"] = list(ens.el_count)
        s["n"] = ens.n
        P = ens.n_el * (ens.n_el + 1) // 2
    if kind == "whole":
        s["xyz"] = ens.xyz64()
        s["q"] = _q(case)
        s["sl"] = np.array(SL[:ens.n_el])
        s["rho0"] = ens.n / (4.0 / 3.0 * math.pi * (0.5 * np.ptp(s["xyz"], axis=1).max()) ** 3)
    elif kind == "hist":
        s["nhist"] = _nhist(case)
        s["xyz"] = _dev(ens.xyz64() if case["f64"] else ens.xyz)
        s["hist"], s["ovf"] = _empty(P * s["nhist"], torch.int64), _empty(1, torch.int64)
    elif kind == "iq":
        s["hist"], ens = _model_hist(case, seed)
        n_el = {1: 1, 3: 2, 6: 3, 10: 4}[case["ntypes"]]
        s["ec"] = [ens.n // n_el] * n_el
        s["sl"] = np.array(SL[:n_el])
        s["q"] = _dev(_q(case))
        s["S"] = _empty(case["ntypes"] * case["nq"])
        s["pdf"] = _empty((1 + case["ntypes"]) * case["nhist"])
        s["rho0"] = ens.n / (case["ncell"] * 5.64) ** 3
    elif kind == "iq_many":
        parts = st.c4_particles(case["count"], seed=seed, nmax=case["nmax"])
        s["hist"] = torch.cat([_pair_hists(_dev(p.xyz64()), p.el_count, case["bin"], case["nhist"])
                               for p in parts]).contiguous()
        s["q"] = _dev(_q(case))
        s["S"] = _empty(s["hist"].shape[0] * case["nq"])
    elif kind == "debye":
        s["xyz"], s["q"] = _dev(ens.xyz64()), _dev(_q(case))
        s["S"] = _empty(P * case["nq"])
    elif kind == "partial":
        s["xyz"], s["q"] = ens.xyz64(), _q(case)
        rng = np.random.Generator(np.random.PCG64(seed + 1))
        nb = case["nblocks"]
        s["blk"] = np.concatenate([rng.multinomial(c, [1.0 / nb] * nb) for c in ens.el_count])
    elif kind == "plane":
        nu, nv = case["nu"], case["nv"]
        hu, hv = 2 * case["qmax"] / (nu - 1), 2 * case["qmax"] / (nv - 1)
        s["q0"] = np.array([-case["qmax"], -case["qmax"], 0.0])
        s["du"], s["dv"] = np.array([hu, 0.0, 0.0]), np.array([0.0, hv, 0.0])
        qx, qy = s["q0"][0] + hu * np.arange(nu), s["q0"][1] + hv * np.arange(nv)
        mag = np.hypot(qx[None, :], qy[:, None]).ravel()
        s["ff"] = _dev(st.gaussian_ff(mag, st.gaussian_ff_coeffs(3, seed=seed)))
        s["rot"] = _dev(st.uniform_rotations(case["nrot"], seed=seed).reshape(-1, 9))
        s["xyz"], s["I"] = _dev(ens.xyz64()), _empty(nu * nv)
    elif kind == "polar":
        q = st.q_mesh(0.1, case["qmax"], case["nq"])
        fi = np.arange(case["nfi"]) * (2 * math.pi / case["nfi"])
        sn = q * (calc.default_wavelength(2 * case["qmax"]) * 0.25 / math.pi)
        cs = 1.0 - sn * sn
        qv = np.empty((q.size, fi.size, 3))
        qv[:, :, 0] = (cs * q)[:, None] * np.cos(fi)
        qv[:, :, 1] = (cs * q)[:, None] * np.sin(fi)
        qv[:, :, 2] = (-sn * q)[:, None]
        ff = st.gaussian_ff(q, st.gaussian_ff_coeffs(ens.n_el, seed=seed))
        s["qvec"] = _dev(qv.reshape(-1, 3))
        s["ff"] = _dev(np.repeat(ff[:, :, None], fi.size, axis=2).reshape(ens.n_el, -1))
        s["rot"] = _dev(st.uniform_rotations(case["nrot"], seed=seed).reshape(-1, 9))
        s["xyz"], s["I"] = _dev(ens.xyz64()), _empty(q.size * fi.size)
    elif kind == "ensemble":
        shapes, parts = zip(*_ensemble(case, seed))
        s["xyz"] = [_dev(p.xyz64()) for p in parts]
        s["ecs"] = [list(p.el_count) for p in parts]
        s["nhist"] = [_nhist(c) for c in shapes]
        s["sl"] = np.concatenate([np.array(SL[:p.n_el]) for p in parts])
        s["rho0"] = np.array([0.01 * (5 + k % 5) for k in range(case["count"])])
        nt = [len(e) * (len(e) + 1) // 2 for e in s["ecs"]]
        s["q"] = _dev(_q(case))
        s["hist"] = _empty(sum(t * h for t, h in zip(nt, s["nhist"])), torch.int64)
        s["pdf"] = _empty(sum((1 + t) * h for t, h in zip(nt, s["nhist"])))
        s["S"] = _empty(sum(nt) * case["nq"])
    elif kind == "build":
        a, nc = 5.64, case["ncell"]
        half = nc // 2
        eye = np.eye(3)
        sh = [(0.0, 0.0, 0.0), (0.5, 0.5, 0.0), (0.5, 0.0, 0.5), (0.0, 0.5, 0.5), (0.0, 0.0, 0.0)]
        s["blocks"] = [Block(
            r_atom=np.array([[-half, -half, -half], [-half + 0.5, -half, -half]]) * a, el=[0, 1],
            occ=np.full(2, case["occ"]), dev=np.full(2, case["sigma"]),
            p_symm=np.array([eye, eye, eye, eye, -eye]), r_symm=np.array(sh) * a, cell=eye * a,
            ncell=(nc,) * 3, rcut=half * a)]
        s["seed"] = seed
        # room for every site inside the cut-off
        sites = int(8 * 4 / 3 * math.pi * (half + 1) ** 3)
        s["xyz"] = _empty(3 * sites)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- run
def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "whole":
        I, pdf, ovf = calc.calc_pdf_and_debye(ctx, s["xyz"], s["ec"], s["q"], case["bin"],
                                              pdf_type=2, rho0=s["rho0"], sl=s["sl"],
                                              nhist=_nhist(case))
        return {"I": I, "pdf": pdf, "overflow": np.array([ovf])}
    if kind == "hist":
        ctx.hist_dev(s["xyz"].data_ptr(), s["n"], s["ec"], case["bin"], s["nhist"],
                     s["hist"].data_ptr(), s["ovf"].data_ptr(), f64=case["f64"])
        return {"hist": s["hist"], "overflow": s["ovf"]}
    if kind == "iq":
        ctx.hist_pairsum_dev(s["hist"].data_ptr(), case["ntypes"], case["nhist"], case["bin"],
                             s["q"].data_ptr(), case["nq"], s["S"].data_ptr())
        ctx.pdf_dev(s["hist"].data_ptr(), s["ec"], case["nhist"], case["bin"], "rPDF", s["rho0"],
                    s["sl"], s["pdf"].data_ptr())
        return {"S": s["S"], "pdf": s["pdf"]}
    if kind == "iq_many":
        ctx.hist_pairsum_dev(s["hist"].data_ptr(), s["hist"].shape[0], case["nhist"], case["bin"],
                             s["q"].data_ptr(), case["nq"], s["S"].data_ptr(), mfma=True)
        return {"S": s["S"]}
    if kind == "debye":
        ctx.debye_pairsum_dev(s["xyz"].data_ptr(), s["n"], s["ec"], s["q"].data_ptr(), case["nq"],
                              s["S"].data_ptr())
        return {"S": s["S"]}
    if kind == "partial":
        return {"S": ctx.partial_debye_pairsum(s["xyz"], s["ec"], s["blk"], case["nblocks"], s["q"])}
    if kind == "plane":
        ctx.amp2d_grid_dev(s["xyz"].data_ptr(), s["n"], s["ec"], s["q0"], s["du"], s["dv"],
                           case["nu"], case["nv"], s["rot"].data_ptr(), case["nrot"],
                           s["ff"].data_ptr(), s["I"].data_ptr())
        return {"I": s["I"]}
    if kind == "polar":
        ctx.amp2d_dev(s["xyz"].data_ptr(), s["n"], s["ec"], s["qvec"].data_ptr(),
                      s["qvec"].shape[0], s["rot"].data_ptr(), case["nrot"], s["ff"].data_ptr(),
                      s["I"].data_ptr())
        return {"I": s["I"]}
    if kind == "ensemble":
        b = xh.Batch(ctx, [(x.data_ptr(), ec) for x, ec in zip(s["xyz"], s["ecs"])], case["bin"],
                     nhist=s["nhist"], f64=True, device=True)
        b.run_dev(s["hist"].data_ptr(), s["q"].data_ptr(), case["nq"], s["S"].data_ptr(), "rPDF",
                  s["rho0"], s["sl"], s["pdf"].data_ptr())
        b.close()
        return {"hist": s["hist"], "S": s["S"], "pdf": s["pdf"]}
    a = Atoms(ctx, s["blocks"], 2, seed=s["seed"])
    a.copy_dev(s["xyz"].data_ptr())
    counts = a.el_count.astype(np.int64)
    a.close()
    return {"xyz": s["xyz"], "el_count": counts}


# ---------------------------------------------------------------- work
def _pairs(n):
    return n * (n - 1) / 2


def work(case):
    """Operations in FP units: 11 a pair for a histogram (three subtractions and
    products, two additions, root, division, conversion), a multiply-add a term
    for the sine sums, two of them a term for 2D amplitudes on a grid."""
    kind = case["kind"]
    if kind in ("whole", "hist", "debye", "partial", "plane", "polar"):
        n, e = _natoms(case), _n_el(case)
        P = e * (e + 1) // 2
    if kind in ("whole", "hist"):
        nh = _nhist(case)
        xyz = 3 * n * (8 if kind == "whole" or case["f64"] else 4)
        if kind == "hist":
            return {"bytes": xyz + 8 * P * nh, "flops": 11 * _pairs(n)}
        return {"bytes": xyz + 8 * (1 + P) * nh + 16 * case["nq"],
                "flops": 11 * _pairs(n) + 2 * P * nh * case["nq"]}
    if kind == "iq":
        t, nh, nq = case["ntypes"], case["nhist"], case["nq"]
        return {"bytes": 8 * t * nh + 8 * (1 + t) * nh + 8 * (1 + t) * nq, "flops": 2 * t * nh * nq}
    if kind == "iq_many":
        t, nh, nq = 3 * case["count"], case["nhist"], case["nq"]
        return {"bytes": 8 * t * nh + 8 * nq * (1 + t), "flops": 2 * t * nh * nq}
    if kind in ("debye", "partial"):
        parts = case["nblocks"] * (case["nblocks"] + 1) // 2 if kind == "partial" else 1
        return {"bytes": 24 * n + 8 * case["nq"] * (1 + P * parts),
                "flops": 2 * _pairs(n) * case["nq"]}
    if kind == "plane":
        k = case["nu"] * case["nv"]
        return {"bytes": 24 * n + 8 * k * (e + 1), "flops": 4 * n * k * case["nrot"]}
    if kind == "polar":
        k = case["nq"] * case["nfi"]
        return {"bytes": 24 * n + 8 * k * (e + 4), "flops": 10 * n * k * case["nrot"]}
    if kind == "ensemble":
        lo, hi, c = case["nmin"], case["nmax"], case["count"]
        n1 = (hi - lo) / math.log(hi / lo)
        n2 = (hi * hi - lo * lo) / 2 / math.log(hi / lo)
        bins = 5 * (n1 / 0.06) ** (1 / 3) * 1.7 / case["bin"]
        return {"bytes": c * (24 * n1 + 16 * bins + 40 * case["nq"]),
                "flops": c * (5.5 * n2 + 2 * bins * case["nq"])}
    sites = 8 * case["ncell"] ** 3 * math.pi / 6 * case["occ"]
    return {"bytes": 48 * sites, "flops": 30 * sites}


# ---------------------------------------------------------------- exact
def _sinc_sums(h, bin_, q):
    """S[p, iq] = sum_k h[p, k] sin(q r_k) / (q r_k + 1e-8), r_k = (k + 1/2) bin."""
    r = (torch.arange(h.shape[1], dtype=torch.float64, device=h.device) + 0.5) * bin_
    hd = h.double()
    out = torch.empty((h.shape[0], q.numel()), dtype=torch.float64, device=h.device)
    step = max(1, 64_000_000 // h.shape[1])
    for i in range(0, q.numel(), step):
        x = r[:, None] * q[None, i:i + step]
        out[:, i:i + step] = hd @ (torch.sin(x) / (x + EPS))
    return out


def _debye_sums(x, groups, pairs, q):
    """Rows of sum sin(q r)/(q r + 1e-8) over the pairs of each (group, group)."""
    out = torch.zeros((len(pairs), q.numel()), dtype=torch.float64, device=x.device)
    for row, (a, b) in enumerate(pairs):
        xa, xb = x[:, groups[a]], x[:, groups[b]]
        if not xa.shape[1] or not xb.shape[1]:
            continue
        r = ((xa[:, :, None] - xb[:, None, :]) ** 2).sum(0).sqrt()
        r = r[torch.triu(torch.ones_like(r, dtype=torch.bool), 1)] if a == b else r.reshape(-1)
        step = 1 << 15
        for i in range(0, r.numel(), step):
            t = r[i:i + step, None] * q[None, :]
            out[row] += (torch.sin(t) / (t + EPS)).sum(0)
    return out


def _rpdf(h, counts, bin_, rho0, sl, cpu_radius=True):
    """Total and partial rPDF of one structure; the radius of the CPU path runs
    on over the pair types, that of the GPU kernels starts anew for each."""
    n = float(sum(counts))
    P, nh = h.shape
    k = np.arange(nh) + 0.5
    f2 = sum(c * v for c, v in zip(counts, sl)) ** 2 / n ** 2
    out = np.zeros((1 + P, nh))
    p = 0
    for a in range(len(counts)):
        for b in range(a, len(counts)):
            r = (k + (p * nh if cpu_radius else 0)) * bin_
            sub = 4 * math.pi * rho0 * counts[a] * counts[b] / n ** 2 * (1 if a == b else 2)
            out[1 + p] = 2 * h[p] / (bin_ * n) / r - sub * r
            out[0] += out[1 + p] * sl[a] * sl[b] / f2
            p += 1
    return out


def _intensity(S, counts, sl):
    I, p = np.zeros(S.shape[1]), 0
    for a in range(len(counts)):
        for b in range(a, len(counts)):
            I += 2 * S[p] * sl[a] * sl[b]
            p += 1
    return (I + sum(c * v * v for c, v in zip(counts, sl))) / sum(counts)


def _amplitudes(xyz, counts, qvec, rot, ff):
    out = torch.zeros(qvec.shape[0], dtype=torch.float64, device=xyz.device)
    groups = _blocks_of(counts)
    for R in rot.reshape(-1, 3, 3):
        qr = qvec @ R                                   # R^T q
        re, im = torch.zeros_like(out), torch.zeros_like(out)
        for e, g in enumerate(groups):
            x = xyz[:, g]
            step = max(1, 32_000_000 // max(1, x.shape[1]))
            for i in range(0, qr.shape[0], step):
                ph = qr[i:i + step] @ x
                re[i:i + step] += ff[e, i:i + step] * torch.cos(ph).sum(1)
                im[i:i + step] += ff[e, i:i + step] * torch.sin(ph).sum(1)
        out += re * re + im * im
    return out


def _plane(s, case):
    """The amplitudes of a plane as products of the factors of its two axes."""
    nu, nv = case["nu"], case["nv"]
    xyz, groups = s["xyz"], _blocks_of(s["ec"])
    iu = torch.arange(nu, dtype=torch.float64, device="cuda")
    iv = torch.arange(nv, dtype=torch.float64, device="cuda")
    q0, du, dv = (_dev(s[k]) for k in ("q0", "du", "dv"))
    ff = s["ff"].reshape(-1, nv, nu)
    out = torch.zeros((nv, nu), dtype=torch.float64, device="cuda")
    for R in s["rot"].reshape(-1, 3, 3):
        A = torch.zeros((nv, nu), dtype=torch.complex128, device="cuda")
        for e, g in enumerate(groups):
            y = R @ xyz[:, g]                            # (R^T q) . x = q . (R x)
            U = torch.polar(torch.ones((), dtype=torch.float64, device="cuda"),
                            (du @ y)[:, None] * iu[None, :] + (q0 @ y)[:, None])
            V = torch.polar(torch.ones((), dtype=torch.float64, device="cuda"),
                            iv[:, None] * (dv @ y)[None, :])
            A += ff[e] * (V @ U)
        out += A.real ** 2 + A.imag ** 2
    return out.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("hist", "build"):
        # whole numbers; and positions whose random draws are the builder's own
        return None
    s = prepare(case, seed)
    if kind == "whole":
        h = _pair_hists(_dev(s["xyz"]), s["ec"], case["bin"], _nhist(case))
        S = _sinc_sums(h, case["bin"], _dev(s["q"])).cpu().numpy()
        return {"I": _intensity(S, s["ec"], s["sl"]),
                "pdf": _rpdf(h.cpu().numpy(), s["ec"], case["bin"], s["rho0"], s["sl"]),
                "overflow": None}
    if kind in ("iq", "iq_many"):
        S = _sinc_sums(s["hist"], case["bin"], s["q"]).reshape(-1)
        if kind == "iq_many":
            return {"S": S}
        pdf = _rpdf(s["hist"].cpu().numpy(), s["ec"], case["bin"], s["rho0"], s["sl"],
                    cpu_radius=False)
        return {"S": S, "pdf": pdf.reshape(-1)}
    if kind == "debye":
        g = _blocks_of(s["ec"])
        pairs = [(a, b) for a in range(len(g)) for b in range(a, len(g))]
        return {"S": _debye_sums(s["xyz"], g, pairs, s["q"]).reshape(-1)}
    if kind == "partial":
        nb = case["nblocks"]
        g = _blocks_of(s["blk"])
        x, q = _dev(s["xyz"]), _dev(s["q"])
        out = []
        for a in range(len(s["ec"])):
            for b in range(a, len(s["ec"])):
                for i in range(nb):
                    for j in range(i, nb):
                        S = _debye_sums(x, g, [(a * nb + i, b * nb + j)], q)[0]
                        if a != b and i != j:
                            S = S + _debye_sums(x, g, [(a * nb + j, b * nb + i)], q)[0]
                        out.append(S)
        P = len(s["ec"]) * (len(s["ec"]) + 1) // 2
        return {"S": torch.stack(out).reshape(P, nb * (nb + 1) // 2, q.numel())}
    if kind == "plane":
        return {"I": _plane(s, case)}
    if kind == "polar":
        return {"I": _amplitudes(s["xyz"], s["ec"], s["qvec"], s["rot"], s["ff"])}
    S, pdf, sl = [], [], list(s["sl"])
    for k, (x, ec) in enumerate(zip(s["xyz"], s["ecs"])):
        h = _pair_hists(x, ec, case["bin"], s["nhist"][k])
        S.append(_sinc_sums(h, case["bin"], s["q"]).reshape(-1))
        pdf.append(_rpdf(h.cpu().numpy(), ec, case["bin"], s["rho0"][k], sl[:len(ec)]).reshape(-1))
        sl = sl[len(ec):]
    return {"hist": None, "S": torch.cat(S), "pdf": np.concatenate(pdf)}

