"""Timed cases of the LAPW setup: what an exciting run asks of this library.

One pass of the SCF k loop is match + hamiltonandoverlapsetup per k-point
(seceqn.f90:57, seceqnfv.f90:76-77); every SCF iteration first remakes the
muffin-tin and interstitial tables (scf_cycle.f90:210-222); the eigensolve
that follows applies the reduced matrix to a block of vectors over and over.
The cells are the library's setup workloads (2, 8, 16, 64 atoms); drawn cells
are grids of 1 to 32 atoms with other cutoffs and angular momenta, so G+k
counts and matrix orders come out ragged.

    listed()              the cases
    draw(rng)             one more of the same ranges
    prepare(case, seed)   inputs, context and buffers on the GPU
    run(state)            one pass through the public entry points
    work(case)            bytes and flops the pass cannot do without
    exact(case, seed)     its outputs in plain NumPy / torch FP64
"""
import dataclasses
import functools
import math

import numpy as np
import torch

from exciting_amd import lapw, synth

# cells by name: the library's setup workloads
CONFIG = {"fcc2": 0, "sc8": 1, "ortho16": 2, "sc32": 4, "sc64": 3}
ALPHA = 1.0 / 137.03599911
Y00 = 0.28209479177387814
LMAXVR = 8


def _case(name, path, cell, **more):
    c = {"name": name, "path": path, "cell": cell, "nk": 1, "split": 0, "rel": "none",
         "n1": 0, "n2": 0, "n3": 0, "lmax": 0, "rgkmax": 0.0, "order": 0, "cols": 0}
    c.update(more)
    return c


def listed():
    return [
        # primitive cell, one k-point of the SCF loop: launches and latency
        _case("fcc2_setup", "setup", "fcc2"),
        # conventional cell, scalar relativity iora*: the reference's call
        # sequence newsystem (zeroed) + accumulating setup
        _case("sc8_iora_setup", "setup", "sc8", rel="iora"),
        # the Fortran drop-in: host arrays in and out, one k-point
        _case("sc8_host_dropin", "host", "sc8"),
        # all k-points of a cell in one grouped call
        _case("sc8_batch8", "batch", "sc8", nk=8),
        # the same in split precision, the serving mix's modulus count
        _case("sc8_batch8_split9", "batch", "sc8", nk=8, split=9),
        # hybrids (calc_vnlmat): match + the overlap alone
        _case("ortho16_overlap", "overlap", "ortho16"),
        # medium cell, grouped k-points
        _case("ortho16_batch8", "batch", "ortho16", nk=8),
        # supercell, one k-point: the headline setup
        _case("sc64_setup", "setup", "sc64"),
        # the same in split precision as the precision tuner picks it
        _case("sc64_setup_split7", "setup", "sc64", split=7),
        # per SCF iteration: muffin-tin tables of the supercell
        _case("sc64_hmlint", "hmlint", "sc64"),
        # per SCF iteration: step function and potential components
        _case("sc64_interstitial", "interstitial", "sc64"),
        # eigensolve: one Chebyshev step, 56 vectors (40 states) at the
        # supercell's matrix order
        _case("sc64_filter", "filter", "none", order=10364, cols=56),
    ]


def draw(rng):
    path = rng.choice(["setup", "setup", "batch", "batch", "overlap", "host", "hmlint",
                       "interstitial", "filter"])
    if path == "filter":
        order = int(math.exp(rng.uniform(math.log(600), math.log(10364))))
        return _case("", path, "none", order=order, cols=rng.randint(17, 80))
    lmax = rng.randint(6, 10)
    rgkmax = round(rng.uniform(6.0, 8.5), 3)
    # atoms over 1..32 (grids n1 x n2 x n3), about evenly over the logarithm
    grids = [(1, 1, 1), (1, 1, 2), (1, 1, 3), (1, 2, 2), (1, 2, 3), (2, 2, 2), (2, 2, 3),
             (1, 3, 4), (2, 3, 3), (2, 3, 4), (3, 3, 3), (2, 4, 4)]
    n1, n2, n3 = rng.choice(grids)
    atoms = n1 * n2 * n3
    nk, split, rel = 1, 0, "none"
    if path == "batch":
        nk = rng.randint(2, 8) if atoms <= 12 else rng.randint(2, 3)
    if path in ("setup", "batch"):
        split = rng.choice([0, 0, 7, 8, 9])
    if path in ("setup", "overlap", "host") and split == 0:
        rel = rng.choice(["none", "none", "zora", "iora"])
    if path == "host" and atoms > 12:
        n1, n2, n3 = 1, 3, 4
    return _case("", path, "grid", nk=nk, split=split, rel=rel, n1=n1, n2=n2, n3=n3,
                 lmax=lmax, rgkmax=rgkmax)


# ---- cells -----------------------------------------------------------------
def _spec(case, seed):
    """The case's cell: geometry and k-points belong to the case, the tables
    follow the seed."""
    if case["cell"] != "grid":
        return dataclasses.replace(_config(CONFIG[case["cell"]]), seed=seed)
    n = (case["n1"], case["n2"], case["n3"])
    rng = np.random.default_rng([*n, case["lmax"], int(1000 * case["rgkmax"]), case["nk"]])
    avec = 5.13 * np.diag(np.array(n, float)) + rng.uniform(-0.05, 0.05, (3, 3))
    pts = [[], []]
    for s in np.ndindex(*n):
        pts[sum(s) % 2].append((np.array(s, float) + rng.normal(0.0, 0.01, 3)) / np.array(n))
    pts = [np.array(p) for p in pts if p]
    los = [[0, 1, 2, 3], [0, 1, 2]]
    return synth.CellSpec(
        name="grid", avec=avec, positions=pts, rmt=[2.0] * len(pts), lmaxapw=case["lmax"],
        lmaxmat=case["lmax"], apword=2, lo_l=los[:len(pts)], rgkmax=case["rgkmax"],
        gmaxvr=12.0, kpoints=rng.uniform(-0.5, 0.5, (max(case["nk"], 1), 3)), seed=seed)


@functools.lru_cache(maxsize=None)
def _config(index):
    return synth.config(index)


@functools.lru_cache(maxsize=2)
def _build(key, seed):
    case = dict(key)
    spec = _spec(case, seed)
    step = max(1, len(spec.kpoints) // case["nk"])
    s = synth.build(spec, kpoints=[i * step for i in range(case["nk"])])
    if case["rel"] != "none":
        synth.add_relativity(s, seed=seed, iora=case["rel"] == "iora")
    if case["path"] == "hmlint":
        synth.add_mt_potential(s, LMAXVR, seed=seed)
    return s


def _system(case, seed):
    return _build(tuple(sorted((k, v) for k, v in case.items() if k != "name")), seed)


def _veffir(s, seed):
    return -0.3 + 0.2 * np.random.default_rng(seed).uniform(-1.0, 1.0, s.ngrtot)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a).ravel(order="F"))).cuda()


# ---- prepare / run ---------------------------------------------------------
def prepare(case, seed):
    path = case["path"]
    if path == "filter":
        return _prepare_filter(case, seed)
    s = _system(case, seed)
    st = {"case": case, "s": s, "ctx": lapw.Context(0).load(s)}
    z = lambda n, dt=torch.complex128: torch.zeros(n, dtype=dt, device="cuda")
    if path in ("setup", "overlap"):
        st["d"] = lapw.DeviceKPoint(s, 0)
        st["sys"] = lapw.newsystem(st["d"].rank, device="cuda")
        if path == "overlap":
            st["sys"].hamilton = None
    elif path == "batch":
        st["d"] = [lapw.DeviceKPoint(s, i) for i in range(case["nk"])]
        st["h"] = [z((d.rank, d.rank)) for d in st["d"]]
        st["o"] = [z((d.rank, d.rank)) for d in st["d"]]
        st["kp"] = [lapw.kpoint_struct(d, h, o) for d, h, o in zip(st["d"], st["h"], st["o"])]
    elif path == "host":
        st["a"] = np.zeros((s.ngkmax, s.apwordmax, (s.lmaxapw + 1) ** 2, s.natmtot),
                           dtype=np.complex128, order="F")
        st["sys"] = lapw.newsystem(s.nmat(0))
    elif path == "hmlint":
        st["v"], st["lofr"] = _dev(s.veffmt), _dev(s.lofr)
        na, m, mlo = s.natmtot, s.maxaa, max(s.maxnlo, 1)
        st["t"] = [z(m * m * na), z(mlo * m * na), z(mlo * mlo * na)]
    elif path == "interstitial":
        st["v"] = _dev(_veffir(s, seed))
        st["cg"], st["cr"] = z(s.ngrtot), z(s.ngrtot, torch.float64)
        st["ve"], st["me"] = z(s.ngvec), z(s.ngvec)
    return st


def run(st):
    path = st["case"]["path"]
    if path == "filter":
        return lapw.zgemm_cn(st["c"], st["x"], alpha=0.7, beta=-0.9, y0=st["x"], gamma=-0.4,
                             z=st["z"], hermitian=True)
    ctx, s, split = st["ctx"], st["s"], st["case"]["split"]
    flags = lapw.SPLIT(split) if split else 0
    if path == "setup":
        d, y = st["d"], st["sys"]
        if s.h1on:   # as the reference: zeroed by newsystem, then added to
            y.hamilton.za.zero_()
            y.overlap.za.zero_()
            flags |= lapw.ACCUMULATE
        ctx.match(d.ngk, d.gpc, d.tpgpc, d.sfacgp, d.apwalm)
        ctx.hamiltonandoverlapsetup(y, d.ngk, d.apwalm, d.igpig, d.vgpc, flags=flags)
        return d.apwalm, y.hamilton.za, y.overlap.za
    if path == "overlap":
        d, y = st["d"], st["sys"]
        ctx.match(d.ngk, d.gpc, d.tpgpc, d.sfacgp, d.apwalm)
        ctx.overlapsetup(y, d.ngk, d.apwalm, d.igpig, d.vgpc, flags=0)
        return d.apwalm, y.overlap.za
    if path == "batch":
        ctx.setup_batch(st["kp"], flags=flags | lapw.MATCH)
        return [(d.apwalm, h, o) for d, h, o in zip(st["d"], st["h"], st["o"])]
    if path == "host":
        k, y = s.kpts[0], st["sys"]
        y.hamilton.za.fill(0.0)
        y.overlap.za.fill(0.0)
        ctx.match(k.ngk, k.gpc, k.tpgpc, k.sfacgp, st["a"])
        ctx.hamiltonandoverlapsetup(y, k.ngk, st["a"], k.igpig, k.vgpc)
        return st["a"], y.hamilton.za, y.overlap.za
    if path == "hmlint":
        return ctx.hmlint(s.lmaxvr, st["v"], st["lofr"], True, *st["t"])
    ctx.gencfun(s.bvec, s.atposc, cfunig=st["cg"], cfunir=st["cr"])
    ctx.genveffig_device(st["v"], st["cr"], veffig=st["ve"], meffig=st["me"])
    return st["cg"], st["cr"], st["ve"], st["me"]


def _prepare_filter(case, seed):
    n, m = case["order"], case["cols"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *sh: torch.randn(*sh, dtype=torch.complex128, device="cuda", generator=g)
    c = rnd(n, n)
    c = 0.5 * (c + c.conj().t().contiguous())
    return {"case": case, "c": c, "x": rnd(n, m) / math.sqrt(n), "z": rnd(n, m) / math.sqrt(n)}


# ---- work ------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _sizes(key):
    s = _build(key, 1)
    return [k.ngk for k in s.kpts], s.nlotot, s.natmtot, s.maxaa, s.maxnlo, s.ngkmax, s.ngrtot, \
        s.ngvec, s.nrmtmax, s.nlomax


def work(case):
    if case["path"] == "filter":
        n, m = case["order"], case["cols"]
        return {"bytes": 16.0 * n * (n + 3 * m), "flops": 8.0 * n * n * m}
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    ngs, nlotot, na, M, nlo, ngkmax, ngrtot, ngvec, nr, nlomax = _sizes(key)
    if case["path"] == "interstitial":
        fft = 5.0 * ngrtot * math.log2(ngrtot)
        return {"bytes": 12.0 * ngrtot + 8.0 * ngrtot + 24.0 * ngrtot + 2 * 16.0 * ngvec,
                "flops": 3 * fft + ngrtot * na * 10.0}
    if case["path"] == "hmlint":
        nf = (_spec(case, 1).lmaxmat + 1) * 2 + nlomax
        lmm = (LMAXVR + 1) ** 2
        out = 16.0 * na * (M * M + nlo * M + nlo * nlo)
        return {"bytes": out + 8.0 * na * nr * (lmm + 4.0 * nf),
                "flops": na * (nf * (nf + 1) / 2) * nr * 2.0 * lmm}
    tables = 16.0 * na * (M * M + nlo * M)
    b = f = 0.0
    for g in ngs:
        n = g + nlotot
        one = case["path"] == "overlap"
        b += 16.0 * g * M * na + (1 if one else 2) * 16.0 * n * n + 16.0 * g * na
        f += na * ((4.0 if one else 8.0) * g * (g + 1) * M + (0.0 if one else 8.0 * M * M * g)
                   + 8.0 * nlo * M * g)
    return {"bytes": b + (0.0 if case["path"] == "overlap" else tables), "flops": f}


# ---- exact -----------------------------------------------------------------
def exact(case, seed):
    path = case["path"]
    if path == "filter":
        st = _prepare_filter(case, seed)
        return 0.7 * (st["c"] @ st["x"]) - 0.9 * st["x"] - 0.4 * st["z"]
    s = _system(case, seed)
    if path == "interstitial":
        return _exact_interstitial(s, _veffir(s, seed))
    if path == "hmlint":
        return _exact_hmlint(s)
    got = [_exact_k(s, ik, path == "overlap") for ik in range(case["nk"])]
    if path == "batch":
        return got
    if path == "host":   # Fortran arrays
        a, h, o = (t.cpu().numpy() for t in got[0])
        a = a.reshape((s.ngkmax, s.apwordmax, (s.lmaxapw + 1) ** 2, s.natmtot), order="F")
        return a, h.T, o.T
    return got[0]


def _jl(lmax, x):
    """j_l(x) and j_l'(x), l = 0..lmax, by downward recurrence normalised with
    sum (2l+1) j_l^2 = 1 (sign from j_0 or j_1)."""
    top = lmax + 40
    j = np.zeros((top + 2, x.size))
    j[top] = 1e-250
    for l in range(top, 0, -1):
        j[l - 1] = (2 * l + 1) / x * j[l] - j[l + 1]
        big = np.abs(j[l - 1]) > 1e200
        if big.any():
            j[:, big] *= 1e-200
    w = (2 * np.arange(top + 2) + 1.0)[:, None]
    scale = np.abs(j).max(axis=0)
    j /= scale
    j /= np.sqrt((w * j * j).sum(axis=0))
    j0, j1 = np.sin(x) / x, np.sin(x) / x ** 2 - np.cos(x) / x
    use0 = np.abs(j0) > np.abs(j1)
    j *= np.sign(np.where(use0, j0 * j[0], j1 * j[1]))
    d = np.zeros((lmax + 1, x.size))
    d[0] = -j[1]
    for l in range(1, lmax + 1):
        d[l] = j[l - 1] - (l + 1) / x * j[l]
    return j[:lmax + 1], d


def _ylm(lmax, theta, phi):
    """Spherical harmonics Y_lm with the Condon-Shortley phase, [lm, point]."""
    ct, sn = np.cos(theta), np.sin(theta)
    y = np.zeros(((lmax + 1) ** 2, theta.size), complex)
    pmm = np.full(theta.size, Y00)
    for m in range(lmax + 1):
        if m:
            pmm = -math.sqrt((2 * m + 1.0) / (2 * m)) * sn * pmm
        p0, p1 = np.zeros_like(pmm), pmm
        for l in range(m, lmax + 1):
            if l > m:
                a = math.sqrt((4.0 * l * l - 1.0) / (l * l - m * m))
                b = math.sqrt(((l - 1.0) ** 2 - m * m) / (4.0 * (l - 1.0) ** 2 - 1.0))
                p0, p1 = p1, a * (ct * p1 - b * p0)
            e = np.exp(1j * m * phi)
            y[l * (l + 1) + m] = p1 * e
            y[l * (l + 1) - m] = (-1) ** m * p1 * np.conj(e)
    return y


def _boundary(s, ias, sp, l):
    """Value and slope at the sphere of each radial function: d[i, j] =
    d^i u_j / dr^i, from the cubic through the last four radial points."""
    n = int(s.nrmt[sp])
    r = s.spr[n - 4:n, sp].astype(np.longdouble) - np.longdouble(s.rmt[sp])
    d = np.zeros((2, s.apwordmax))
    for j in range(s.apwordmax):
        f = s.apwfr[n - 4:n, 0, j, l, ias].astype(np.longdouble)
        for a in range(4):
            o = [r[b] for b in range(4) if b != a]
            den = (r[a] - o[0]) * (r[a] - o[1]) * (r[a] - o[2])
            d[0, j] += float(-o[0] * o[1] * o[2] / den * f[a])
            d[1, j] += float((o[0] * o[1] + o[0] * o[2] + o[1] * o[2]) / den * f[a])
    return d


def _exact_k(s, ik, only_o):
    """match and the setup of one k-point from the definitions, on the GPU in
    FP64: apwalm and (H,) O, flattened / row-major as the entry points lay
    them out (row-major storage of the transposes)."""
    k = s.kpts[ik]
    ng, L, p = k.ngk, s.lmaxapw, s.apwordmax
    n, lmm = ng + s.nlotot, (L + 1) ** 2
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    q = k.gpc[:ng]
    yc = np.conj(_ylm(L, k.tpgpc[0, :ng], k.tpgpc[1, :ng]))
    ylm = t(yc)
    sf = t(k.sfacgp[:ng, :].T)
    species = np.repeat(np.arange(s.nspecies), s.natoms)
    apw = torch.zeros((s.natmtot, lmm, p, s.ngkmax), dtype=torch.complex128, device=dev)
    H = None if only_o else torch.zeros((n, n), dtype=torch.complex128, device=dev)
    O = torch.zeros((n, n), dtype=torch.complex128, device=dev)
    lob = ng
    for ias in range(s.natmtot):
        sp = int(species[ias])
        jl, dj = _jl(L, q * s.rmt[sp])
        rad = np.zeros((lmm, p, ng), complex)
        for l in range(L + 1):
            b = np.stack([jl[l], q * dj[l]])
            a = np.linalg.solve(_boundary(s, ias, sp, l), b)
            rad[l * l:(l + 1) ** 2] = 4 * math.pi * 1j ** l / math.sqrt(s.omega) * a
        A = t(rad) * ylm[:, None, :] * sf[ias][None, None, :]
        apw[ias, :, :, :ng] = A
        f = A.reshape(lmm * p, ng)          # rows (l, m, io), io fastest
        fh = f.conj().t().contiguous()
        if H is not None:
            H[:ng, :ng] += fh @ (t(s.aa[:, :, ias]) @ f)
        W = f
        if s.h1aa is not None:
            h1 = np.stack([s.h1aa[:, :, l, ias].T for l in range(L + 1) for _ in range(2 * l + 1)])
            W = (A + torch.matmul(t(h1.astype(complex)), A)).reshape(lmm * p, ng)
        O[:ng, :ng] += fh @ W
        los = int(s.losize[sp])
        if not los:
            continue
        if H is not None:
            H[lob:lob + los, :ng] = t(s.loa[:los, :, ias]) @ f
            H[:ng, lob:lob + los] = H[lob:lob + los, :ng].conj().t()
            H[lob:lob + los, lob:lob + los] = t(s.lolo[:los, :los, ias])
        off = [0]
        for l in s.lorbl[:s.nlorb[sp], sp]:
            off.append(off[-1] + 2 * int(l) + 1)
        for i in range(int(s.nlorb[sp])):
            l = int(s.lorbl[i, sp])
            w = s.oalo[:, i, ias] + (0.0 if s.h1loa is None else s.h1loa[:, i, ias])
            v = (A[l * l:(l + 1) ** 2] * t(w)[None, :, None]).sum(dim=1)
            O[:ng, lob + off[i]:lob + off[i + 1]] = v.conj().t()
            for j in range(int(s.nlorb[sp])):
                if s.lorbl[j, sp] == l:
                    w = s.ololo[i, j, ias] + (0.0 if s.h1lolo is None else s.h1lolo[i, j, ias])
                    for m in range(2 * l + 1):
                        O[lob + off[i] + m, lob + off[j] + m] = w
        lob += los
    # interstitial: G_i - G_j looked up in the box
    gv = t(s.ivg[:, k.igpig[:ng] - 1].astype(np.int64))
    lo, hi = s.intgv[:, 0], s.intgv[:, 1]
    box = t(s.ivgig.ravel(order="F").astype(np.int64))
    tab = lambda x: torch.cat([t(np.zeros(1, complex)), t(np.asarray(x)[:s.ngvec])])
    cf, ve = tab(s.cfunig), tab(s.veffig)
    me = cf if s.valence_rel_none else tab(s.meffig)
    m2 = tab(s.m2effig) * (0.5 * ALPHA ** 2) if s.h1on else None
    g = t(k.vgpc[:, :ng])
    for i0 in range(0, ng, 512):
        i1 = min(ng, i0 + 512)
        idx = torch.zeros((i1 - i0, ng), dtype=torch.int64, device=dev)
        ok = torch.ones((i1 - i0, ng), dtype=torch.bool, device=dev)
        mul = 1
        for d in range(3):
            e = gv[d, i0:i1, None] - gv[d][None, :]
            ok &= (e >= int(lo[d])) & (e <= int(hi[d]))
            idx += (e - int(lo[d])) * mul
            mul *= int(hi[d] - lo[d] + 1)
        ig = torch.where(ok, box[torch.where(ok, idx, 0)], 0)
        ig = torch.where(ig <= s.ngvec, ig, 0)
        t1 = 0.5 * (g[:, i0:i1].t().contiguous() @ g)
        if H is not None:
            H[i0:i1, :ng] += ve[ig] + t1 * me[ig]
        O[i0:i1, :ng] += cf[ig] if m2 is None else cf[ig] + t1 * m2[ig]
    out = [apw.reshape(-1)]
    for x in (H, O):
        if x is not None:   # upper triangle, mirrored; storage of the transpose
            u = torch.triu(x, 1)
            out.append((torch.triu(x) + u.conj().t()).t().contiguous())
    return tuple(out)


def _exact_interstitial(s, veffir):
    v = s.bvec @ s.ivg.astype(float)
    gc = np.sqrt((v * v).sum(axis=0))
    fin = gc > 1e-6
    cf = np.where(fin, 0.0, 1.0).astype(complex)
    species = np.repeat(np.arange(s.nspecies), s.natoms)
    for sp in range(s.nspecies):
        R = s.rmt[sp]
        x = gc * R
        ff = np.full(gc.size, 4 * math.pi / s.omega * R ** 3 / 3.0)
        ff[fin] = 4 * math.pi / s.omega * (np.sin(x) - x * np.cos(x))[fin] / gc[fin] ** 3
        at = s.atposc[species == sp]
        for a in at:
            cf -= ff * np.exp(-1j * (v.T @ a))
    n = [int(x) for x in s.ngrid]
    j = [np.where(s.ivg[d] >= 0, s.ivg[d], n[d] + s.ivg[d]) for d in range(3)]
    grid = np.zeros(n, complex)
    grid[j[0], j[1], j[2]] = cf
    cr = np.fft.ifftn(grid).real * s.ngrtot
    vir = veffir.reshape(n, order="F")

    def comp(x):
        return np.fft.fftn(x)[j[0], j[1], j[2]][:s.ngvec] / s.ngrtot
    mass = cr / (1.0 - vir * (0.5 * ALPHA ** 2))
    return cf, cr.ravel(order="F"), comp(vir * cr), comp(mass)


def _spline_weights(x):
    """w with w . f = the integral of f by the reference's cubic spline rule
    (spline.f90, fderiv.f90 with m = -1), applied to all unit vectors."""
    n = x.size
    f = np.eye(n)
    h = np.diff(x)
    iw = 1.0 / h
    s = iw[:, None] * np.diff(f, axis=0)                # slopes
    c1, c2 = np.zeros(n), np.zeros((n, n))
    c1[0] = 1.0
    c2[0] = (s[1] - s[0]) / (x[2] - x[0])
    t1 = h[0] * iw[1]
    t2 = t1
    t3 = 0.5 / (t1 + 1.0)
    t4 = 3.0 * (s[1] - s[0]) * iw[1] - t2 * c2[0]
    c1[1], c2[1] = t3, t4
    for i in range(2, n - 1):
        t1 = h[i - 1] * iw[i]
        t2 = t1 * t3
        t3 = 1.0 / (2.0 * t1 + 2.0 - t2)
        t4 = 3.0 * (s[i] - s[i - 1]) * iw[i] - t2 * t4
        c1[i], c2[i] = t3, t4
    c1[n - 1] = 1.0
    c2[n - 1] = (s[n - 2] - s[n - 3]) / (x[n - 1] - x[n - 3])
    back = c2[n - 1]
    for i in range(n - 2, 0, -1):
        back = c2[i] - back * c1[i + 1]
        c2[i] = back
    b = c1[:, None] * c2
    c = np.diff(b, axis=0) / 3.0 * iw[:, None]
    a = s - (b[:-1] + c * h[:, None]) * h[:, None]
    hh = h[:, None]
    return ((((0.25 * c * hh + b[:-1] / 3.0) * hh + 0.5 * a) * hh + f[:-1]) * hh).sum(axis=0)


@functools.lru_cache(maxsize=4)
def _gaunt(l1max, l2max):
    """integral of conj(Y_lm1) R_lm2 Y_lm3, R the real harmonics, by
    Gauss-Legendre x uniform quadrature: [lm1, lm2, lm3]."""
    top = 2 * l1max + l2max
    c, w = np.polynomial.legendre.leggauss(top // 2 + 1)
    nphi = top + 1
    th = np.repeat(np.arccos(c), nphi)
    ph = np.tile(2 * math.pi / nphi * np.arange(nphi), c.size)
    wt = np.repeat(w * 2 * math.pi / nphi, nphi)
    y = _ylm(l1max, th, ph)
    y2 = _ylm(l2max, th, ph)
    r = np.zeros(y2.shape)
    for l in range(l2max + 1):
        for m in range(-l, l + 1):
            v = y2[l * (l + 1) + m]
            r[l * (l + 1) + m] = v.real if m == 0 else math.sqrt(2.0) * (
                v.real if m > 0 else v.imag)
    left = (np.conj(y) * wt)[:, None, :] * r[None]
    g = left.reshape(-1, wt.size) @ y.T
    return g.reshape(y.shape[0], y2.shape[0], y.shape[0])


def _exact_hmlint(s):
    """mt_kin + mt_pot without relativity: kinetic and potential radial
    integrals contracted with the Gaunt coefficients."""
    L, p, na = s.lmaxmat, s.apwordmax, s.natmtot
    nfa = (L + 1) * p
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.from_numpy(_gaunt(L, s.lmaxvr)).to(dev)
    species = np.repeat(np.arange(s.nspecies), s.natoms)
    mlo = max(s.maxnlo, 1)
    aa = np.zeros((s.maxaa, s.maxaa, na), complex, order="F")
    loa = np.zeros((mlo, s.maxaa, na), complex, order="F")
    lolo = np.zeros((mlo, mlo, na), complex, order="F")
    for ias in range(na):
        sp = int(species[ias])
        n, nl = int(s.nrmt[sp]), int(s.nlorb[sp])
        x = s.spr[:n, sp]
        w = _spline_weights(x)
        u = s.apwfr[:n, :, :, :L + 1, ias].transpose(0, 1, 3, 2).reshape(n, 2, nfa)
        u = np.concatenate([u, s.lofr[:n, :, :nl, ias]], axis=2)
        fl = [l for l in range(L + 1) for _ in range(p)] + [int(l) for l in s.lorbl[:nl, sp]]
        fl = np.array(fl)
        val, der = u[:, 0, :], u[:, 1, :]
        same = (fl[:, None] == fl[None, :]) * 0.5
        kin = (der * (w * x * x)[:, None]).T @ der \
            + (fl * (fl + 1.0))[:, None] * ((val * w[:, None]).T @ val)
        kin = kin * same
        vw = s.veffmt[:, :n, ias] * (w * x * x)[None, :]          # [lm2, r]
        pair = (val[:, :, None] * val[:, None, :]).reshape(n, -1)
        pot = (vw @ pair).reshape(-1, fl.size, fl.size)           # [lm2, f1, f2]
        rows = [(l * l + mi, l * p + io) for l in range(L + 1) for mi in range(2 * l + 1)
                for io in range(p)]
        lor = [(int(l) * int(l) + mi, nfa + i) for i, l in enumerate(s.lorbl[:nl, sp])
               for mi in range(2 * int(l) + 1)]
        full = rows + lor
        lm = torch.tensor([r[0] for r in full], device=dev)
        f = torch.tensor([r[1] for r in full], device=dev)
        pt = torch.from_numpy(pot).to(dev)
        tab = torch.zeros((len(full), len(full)), dtype=torch.complex128, device=dev)
        for c in range(pt.shape[0]):
            tab += g[:, c][lm[:, None], lm[None, :]] * pt[c][f[:, None], f[None, :]]
        kt = torch.from_numpy(kin).to(dev)[f[:, None], f[None, :]]
        tab += torch.where(lm[:, None] == lm[None, :], kt, torch.zeros_like(kt))
        tab = tab.cpu().numpy()
        na_, nl_ = len(rows), len(lor)
        aa[:na_, :na_, ias] = tab[:na_, :na_]
        loa[:nl_, :na_, ias] = tab[na_:, :na_]
        lolo[:nl_, :nl_, ias] = tab[na_:, na_:]
    return tuple(a.ravel(order="F") for a in (aa, loa, lolo))
