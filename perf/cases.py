"""The work that users of this package have it do, as cases that can be timed.

A case names a molecular system of the package's own workloads ((H2O)n on a jittered lattice, all-anti CkH2k+2,
benzene in water), a basis set, a functional and the entry point that a program calls:

  build       FuncPotential on resident tiles: P -> V_xc and E_xc, through device or host matrices
  serve       the same through xc.Server: host P in, host V_xc out, the captured build replayed
  packed      fock_build_packed over several small systems
  open_shell  the unrestricted build of a radical cation (host matrices)
  gradient    getGeomGradients of a restricted density
  embedding   one freeze-and-thaw sweep: every subsystem's density updated and its non-additive XC and
              kinetic potentials built on the cached densities
  coulomb     the density-fitted Coulomb matrix of an SCF iteration
  first_build a geometry seen for the first time: molecular grid, controller, one build

Densities are idempotent-like sums over perturbed free-atom orbitals (positive everywhere, with the
off-diagonal tails that a molecule's density has); the seed picks the geometry's jitter and the perturbation.
"""
import ctypes
import functools
import math

import torch  # before the package: its HIP runtime has to see the device first

import numpy as np

from serenity_amd import scf, workloads, xc

THRESHOLD = 1e-9        # radial threshold of the controllers (the default)
DEVICE = "cuda:0"


# ---- the cases ---------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one water, host matrices in and out, as a program's first test or a tiny subsystem
        dict(name="water1-svp-lda-host", kind="build", system="water", size=1, basis="DEF2-SVP", functional="LDA",
             precision="FP64", api="host"),
        # the SCF iteration of a small cluster (the package's first benchmark configuration)
        dict(name="water8-svp-lda-fp64", kind="build", system="water", size=8, basis="DEF2-SVP", functional="LDA",
             precision="FP64", api="device"),
        # a long chain molecule with a GGA: many blocks of moderate width (the second configuration)
        dict(name="alkane20-svp-pbe-fp64", kind="build", system="alkane", size=20, basis="DEF2-SVP",
             functional="PBE", precision="FP64", api="device"),
        # the large dense cluster in the mixed form that its SCF iterates with (the third configuration)
        dict(name="water64-tzvp-pbe-mixed", kind="build", system="water", size=64, basis="DEF2-TZVP",
             functional="PBE", precision="MIXED", api="device"),
        # the FP64 builds that finish every SCF, on a triple-zeta cluster
        dict(name="water32-tzvp-pbe-fp64", kind="build", system="water", size=32, basis="DEF2-TZVP",
             functional="PBE", precision="FP64", api="device"),
        # one request of the serving mix on FP32 tiles
        dict(name="serve-alkane11-tzvp-pbe", kind="serve", system="alkane", size=11, basis="DEF2-TZVP",
             functional="PBE", precision="FP32"),
        # waiting small requests of the serving mix as one pack
        dict(name="packed16-svp-pbe-fp32", kind="packed", size=8, basis="DEF2-SVP", functional="PBE",
             precision="FP32"),
        # an open shell: five waters less one electron
        dict(name="open-shell-water5-tzvp-pbe", kind="open_shell", system="water", size=5, basis="DEF2-TZVP",
             functional="PBE"),
        # a geometry step's XC gradient
        dict(name="gradient-alkane8-tzvp-pbe", kind="gradient", system="alkane", size=8, basis="DEF2-TZVP",
             functional="PBE"),
        # embedding: benzene and 12 waters, every subsystem visited once
        dict(name="embedding-water12-svp-pbe-tf", kind="embedding", size=12, basis="DEF2-SVP", functional="PBE"),
        # the Coulomb matrix of each iteration of the triple-zeta SCF
        dict(name="coulomb-water32-tzvp", kind="coulomb", system="water", size=32, basis="DEF2-TZVP"),
        # a system that arrives for the first time (a cold serving request, a geometry step)
        dict(name="first-build-water12-svp-pbe", kind="first_build", system="water", size=12, basis="DEF2-SVP",
             functional="PBE", precision="FP32"),
    ]


def _log_size(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49)))))))


def draw(rng):
    """One more case: waters up to 48 and chains up to 30 carbons as in the serving mix, both basis sets, LDA and
    PBE, every precision and entry point; the costly entry points over the part of the range that they serve."""
    kind = rng.choice(["build", "build", "build", "build", "serve", "packed", "open_shell", "gradient", "embedding",
                       "coulomb", "coulomb", "first_build"])
    system = rng.choice(["water", "alkane"])
    basis = rng.choice(["DEF2-SVP", "DEF2-TZVP"])
    functional = rng.choice(["LDA", "PBE", "PBE"])
    wide = dict(water=48, alkane=30)[system]
    if kind == "build":
        return dict(kind=kind, system=system, size=_log_size(rng, 1, wide), basis=basis, functional=functional,
                    precision=rng.choice(["FP64", "FP64", "FP32", "MIXED"]), api=rng.choice(["device", "device", "host"]))
    if kind == "serve":
        return dict(kind=kind, system=system, size=_log_size(rng, 1, wide), basis=basis, functional=functional,
                    precision="FP32")
    if kind == "packed":
        return dict(kind=kind, size=rng.randint(2, 8), basis=basis, functional=functional,
                    precision=rng.choice(["FP32", "FP64"]))
    if kind == "open_shell":
        return dict(kind=kind, system=system, size=_log_size(rng, 1, 12), basis=basis, functional=functional)
    if kind == "gradient":
        return dict(kind=kind, system=system, size=_log_size(rng, 1, 12), basis=basis, functional=functional)
    if kind == "embedding":
        return dict(kind=kind, size=rng.randint(2, 24), basis="DEF2-SVP", functional=functional)
    if kind == "coulomb":
        return dict(kind=kind, system=system, size=_log_size(rng, 1, dict(water=28, alkane=16)[system]), basis=basis)
    return dict(kind=kind, system=system, size=_log_size(rng, 1, 24), basis=basis, functional=functional,
                precision="FP32")


# ---- inputs -------------------------------------------------------------------------------------
def _geometry(system, size, seed):
    if system == "water":
        Z, X = workloads.water_cluster(4, 4, 4 if size > 48 else 3, seed=seed)
        return Z[:3 * size], X[:3 * size]
    return workloads.alkane(size, seed=seed)


@functools.lru_cache(maxsize=None)
def _element_factor(basis_name, z):
    """B with B B^T = the free-atom density matrix of the element in this basis."""
    e, U = np.linalg.eigh(scf.atomic_density_guess(basis_name, [z]))
    keep = e > 1e-3
    return U[:, keep] * np.sqrt(e[keep])


def _orbitals(basis_name, Z, X, seed):
    """(n x m) orbitals times sqrt(occupation): free-atom ones, perturbed with an amplitude that decays with the
    distance, so that P = B B^T is positive and dense as a molecule's is."""
    blocks = [_element_factor(basis_name, int(z)) for z in Z]
    n, m = sum(b.shape[0] for b in blocks), sum(b.shape[1] for b in blocks)
    B = np.zeros((n, m))
    atom = np.repeat(np.arange(len(Z)), [b.shape[0] for b in blocks])
    i = j = 0
    for b in blocks:
        B[i:i + b.shape[0], j:j + b.shape[1]] = b
        i, j = i + b.shape[0], j + b.shape[1]
    d = np.linalg.norm(X[:, None, :] - X[None, :, :], axis=2)
    R = torch.from_numpy(np.random.default_rng(seed).standard_normal((n, n), dtype=np.float32)).double()
    damp = torch.from_numpy(0.05 * np.exp(-d / 3.0))[atom][:, atom]
    B = torch.from_numpy(B)
    return B + (R * damp) @ B


def _density(basis_name, Z, X, seed):
    B = _orbitals(basis_name, Z, X, seed)
    return B @ B.T


@functools.lru_cache(maxsize=None)
def _context():
    return xc.Context(0)


def _resident(P):
    """A symmetric matrix on the device, and room for one of the same shape."""
    P = P.to(DEVICE).contiguous()
    return P, torch.zeros_like(P)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _controller(Z, X, basis, precision, derivative=1, grid=None):
    ctx = _context()
    grid = grid or xc.molecular_grid(Z, X, ctx=ctx)
    keep = {"FP64": False, "FP32": "only", "MIXED": True}[precision]
    return xc.BasisFunctionOnGridController(ctx, basis, grid, 128, THRESHOLD, derivative, keep_fp32=keep)


def _pack_members(case, seed):
    return [(s, k, _geometry(s, k, seed + k)) for s in ("water", "alkane") for k in range(1, case["size"] + 1)]


def _embedded(case, seed):
    """Geometries of benzene and the waters, and the whole system's."""
    Z, X, sub = workloads.benzene_water(case["size"], seed=seed)
    return [(Z[sub == i], X[sub == i]) for i in range(int(sub.max()) + 1)], Z, X


def prepare(case, seed):
    kind, name = case["kind"], case["basis"]
    s = dict(kind=kind)
    if kind == "packed":
        s["potentials"], s["P"], s["F"] = [], [], []
        for system, k, (Z, X) in _pack_members(case, seed):
            b = xc.BasisController.from_file(name, Z, X)
            s["potentials"].append(xc.FuncPotential(_controller(Z, X, b, case["precision"]), case["functional"],
                                                    case["precision"]))
            P, F = _resident(_density(name, Z, X, seed + k))
            s["P"].append(P)
            s["F"].append(F)
    elif kind == "embedding":
        parts, Z, X = _embedded(case, seed)
        grid = xc.molecular_grid(Z, X, ctx=_context())
        ctl, s["P"], s["F"] = [], [], []
        for i, (z, x) in enumerate(parts):
            b = xc.BasisController.from_file(name, z, x)
            ctl.append(_controller(z, x, b, "FP64", grid=grid))
            P, F = _resident(_density(name, z, x, seed + i))
            s["P"].append(P)
            s["F"].append([F, torch.zeros_like(F)])
        s["controllers"] = ctl
        s["potentials"] = [[xc.NAddFuncPotential(c, ctl[:i] + ctl[i + 1:], f, "FP64")
                            for f in (case["functional"], "TF")] for i, c in enumerate(ctl)]
        torch.cuda.synchronize()
        for c, P in zip(ctl, s["P"]):
            c.update_density(_ptr(P))
    else:
        Z, X = _geometry(case["system"], case["size"], seed)
        b = xc.BasisController.from_file(name, Z, X)
        P = _density(name, Z, X, seed)
        if kind == "coulomb":
            aux = xc.BasisController.from_file("RI_J_WEIGEND", Z, X)
            s["engine"] = xc.DensityFittedCoulomb(_context(), b, aux)
            s["P"] = np.asfortranarray(P.numpy())
        elif kind == "first_build":
            s.update(Z=Z, X=X, basis=b, functional=case["functional"], precision=case["precision"])
            s["P"], s["F"] = _resident(P)
        elif kind == "gradient":
            gga = case["functional"] in xc.GGA
            s["potential"] = xc.FuncPotential(_controller(Z, X, b, "FP64", 2 if gga else 1), case["functional"])
            s["P"], s["natoms"] = np.asfortranarray(P.numpy()), len(Z)
        elif kind == "open_shell":
            B = _orbitals(name, Z, X, seed)
            s["potential"] = xc.FuncPotential(_controller(Z, X, b, "FP64"), case["functional"])
            s["P"] = [np.asfortranarray((0.5 * C @ C.T).numpy()) for C in (B, B[:, 1:])]
        else:
            ctl = _controller(Z, X, b, case["precision"])
            if kind == "serve":
                s.update(server=xc.Server(_context(), nslots=1), controller=ctl, functional=case["functional"],
                         precision=case["precision"], P=np.asfortranarray(P.numpy()))
            else:
                s["potential"] = xc.FuncPotential(ctl, case["functional"], case["precision"])
                s["host"] = case["api"] == "host"
                if s["host"]:
                    s["P"] = np.asfortranarray(P.numpy())
                else:
                    s["P"], s["F"] = _resident(P)
    torch.cuda.synchronize()
    return s


# ---- one pass -----------------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "build":
        if s["host"]:
            F = s["potential"].getMatrix(s["P"])
            return dict(F=F, E=s["potential"].getEnergy())
        return dict(E=s["potential"].build_device(_ptr(s["P"]), _ptr(s["F"])), F=s["F"])
    if kind == "serve":
        F, E = s["server"].wait(s["server"].submit(s["controller"], s["functional"], s["precision"], s["P"]))
        return dict(F=F, E=E)
    if kind == "packed":
        E = xc.fock_build_packed(s["potentials"], [_ptr(P) for P in s["P"]], [_ptr(F) for F in s["F"]])
        return dict(E=np.array(E), F=s["F"])
    if kind == "open_shell":
        Fa, Fb = s["potential"].getMatrixUnrestricted(*s["P"])
        return dict(Fa=Fa, Fb=Fb, E=s["potential"].getEnergy())
    if kind == "gradient":
        return dict(G=s["potential"].getGeomGradients(s["P"], natoms=s["natoms"]), E=s["potential"].getEnergy())
    if kind == "embedding":
        E = []
        for ctl, P, F, pots in zip(s["controllers"], s["P"], s["F"], s["potentials"]):
            ctl.update_density(_ptr(P))
            E += [pot.build_cached(_ptr(f)) for pot, f in zip(pots, F)]
        return dict(E=np.array(E), F=s["F"])
    if kind == "coulomb":
        return dict(J=s["engine"].coulomb(s["P"]))
    pot = xc.FuncPotential(_controller(s["Z"], s["X"], s["basis"], s["precision"]), s["functional"], s["precision"])
    return dict(E=pot.build_device(_ptr(s["P"]), _ptr(s["F"])), F=s["F"])


# ---- the work that a pass cannot do without -----------------------------------------------------
@functools.lru_cache(maxsize=None)
def _extent(system, size, basis_name, part=None):
    """(grid points, AOs, mean of n_p^2): n_p = AOs above the threshold at a point, over a sample of a coarse grid."""
    if system == "benzene_water":
        parts, Z, X = _embedded(dict(size=size), 1)
        z, x = parts[part]
    else:
        z, x = Z, X = _geometry(system, size, 1)
    b = xc.BasisController.from_file(basis_name, z, x)
    g = xc.molecular_grid(Z, X, accuracy=1)
    pts = g.points[np.random.default_rng(1).permutation(len(g.points))[:400]]
    first = np.concatenate([[0], np.cumsum(b.nprim)])
    r2 = ((pts[:, None, :] - b.center[None]) ** 2).sum(2)
    seen = np.zeros(len(pts))
    for i in range(b.nshell):
        c, a = b.coef[first[i]:first[i + 1]], b.alpha[first[i]:first[i + 1]]
        seen += b.nfunc[i] * (np.abs((c * np.exp(-np.outer(r2[:, i], a))).sum(1)) > THRESHOLD)
    return 3930 * len(Z), b.nao, float((seen ** 2).mean()), float(seen.mean())


def _build_work(extent, functional, precision, spins=1, tables=True):
    """Both contractions, and the resident tiles (values, and gradients for a GGA) and matrices read once."""
    N, n, nb2, nb = extent
    size = 8 if precision == "FP64" else 4
    comps = 4 if functional in xc.GGA else 1
    return dict(flops=4.0 * N * nb2 * spins, bytes=(N * nb * comps * size if tables else 0) + spins * 16.0 * n * n + 16.0 * N)


def _add(works):
    return {k: float(sum(w[k] for w in works)) for k in ("bytes", "flops")}


def work(case):
    kind, name = case["kind"], case["basis"]
    if kind == "packed":
        return _add([_build_work(_extent(s, k, name), case["functional"], case["precision"])
                     for s, k, _ in _pack_members(case, 1)])
    if kind == "embedding":
        works = []
        for i in range(case["size"] + 1):
            e = _extent("benzene_water", case["size"], name, i)
            w = _build_work(e, case["functional"], "FP64")  # a density and a potential with the GGA
            t = _build_work(e, "TF", "FP64")                # a potential with the kinetic functional
            works += [w, dict(flops=t["flops"] / 2, bytes=t["bytes"] / 2)]
        return _add(works)
    extent = _extent(case["system"], case["size"], name)
    if kind == "coulomb":
        return _coulomb_work(case)
    if kind == "open_shell":
        return _build_work(extent, case["functional"], "FP64", spins=2)
    if kind == "gradient":
        w = _build_work(extent, case["functional"], "FP64")
        N, n, nb2, nb = extent
        return dict(flops=1.5 * w["flops"], bytes=w["bytes"] + (N * nb * 6 * 8 if case["functional"] in xc.GGA else 0))
    w = _build_work(extent, case["functional"], case.get("precision", "FP32"))
    if kind == "first_build":  # the tiles are written before they are read
        w["bytes"] *= 2
    return w


@functools.lru_cache(maxsize=None)
def _pairs(system, size, basis_name):
    """Significant primitive pairs of the orbital basis by l_A + l_B."""
    Z, X = _geometry(system, size, 1)
    b = xc.BasisController.from_file(basis_name, Z, X)
    l, a = np.repeat(b.l, b.nprim), b.alpha
    x, c = np.repeat(b.center, b.nprim, axis=0), np.abs(b.coef)
    shell = np.repeat(np.arange(b.nshell), b.nprim)
    count = np.zeros(8)
    for i in range(len(l)):
        p = a[i] + a
        K = c[i] * c * np.exp(-a[i] * a / p * ((x[i] - x) ** 2).sum(1)) * (math.pi / p) ** 1.5
        count += np.bincount((l[i] + l)[(K >= 1e-14) & (shell <= shell[i])], minlength=8)
    return count


def _coulomb_work(case):
    """Per primitive pair and auxiliary primitive, in both directions: Boys values, the R recursion and the contraction."""
    Z, X = _geometry(case["system"], case["size"], 1)
    aux = xc.BasisController.from_file("RI_J_WEIGEND", Z, X)
    h = lambda L: (L + 1) * (L + 2) * (L + 3) // 6  # noqa: E731
    naux, flops = np.bincount(aux.l, weights=aux.nprim, minlength=5), 0.0
    for L, q in enumerate(_pairs(case["system"], case["size"], case["basis"])):
        for l, k in enumerate(naux):
            flops += 2 * q * k * (30 + 3 * sum(h(i) for i in range(L + l + 1)) + 2 * h(L) * h(l))
    n = 43 * len(Z) // 3 if case["basis"] == "DEF2-TZVP" else 8 * len(Z)
    return dict(flops=flops + 2.0 * aux.nao ** 2, bytes=16.0 * n * n + 8.0 * aux.nao ** 2)


# ---- the same in plain 64-bit torch ---------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _harmonics(l):
    """Real solid harmonics (Racah normalisation, m = -l..l) as [(m index, coefficient, a, b, c)] over x^a y^b z^c
    (Helgaker, Jorgensen, Olsen, Molecular Electronic-Structure Theory, eq. 6.4.47)."""
    out = []
    for m in range(-l, l + 1):
        k, two_vm = abs(m), 1 if m < 0 else 0
        norm = math.sqrt((2 if m else 1) * math.factorial(l + k) * math.factorial(l - k)) / (2 ** k * math.factorial(l))
        terms = {}
        for t in range((l - k) // 2 + 1):
            for u in range(t + 1):
                for v2 in range(two_vm, k + 1, 2):  # v2 = 2 v
                    s = (-1) ** (t + (v2 - two_vm) // 2)
                    f = s * 0.25 ** t * math.comb(l, t) * math.comb(l - t, k + t) * math.comb(t, u) * math.comb(k, v2)
                    e = (2 * t + k - 2 * u - v2, 2 * u + v2, l - 2 * t - k)
                    terms[e] = terms.get(e, 0.0) + norm * f
        out += [(m + l, f, *e) for e, f in terms.items() if f]
    return out


def _aos(b, pts, centers=None):
    """AO values and gradients (4, points, AOs) by the shells' formulas, no screening."""
    centers = torch.from_numpy(b.center) if centers is None else centers
    cols, q = [], 0
    for i in range(b.nshell):
        l, k = int(b.l[i]), int(b.nprim[i])
        a, c = torch.from_numpy(b.alpha[q:q + k]), torch.from_numpy(b.coef[q:q + k])
        q += k
        d = pts - centers[i]
        e = c * torch.exp(-(d * d).sum(1, keepdim=True) * a)
        R, dR = e.sum(1), (-2.0 * a * e).sum(1)
        pw = [torch.ones_like(d)]
        for _ in range(l):
            pw.append(pw[-1] * d)
        Y = [[torch.zeros(len(pts), dtype=torch.float64) for _ in range(4)] for _ in range(2 * l + 1)]
        for m, f, *abc in _harmonics(l):
            mono = [pw[abc[x]][:, x] for x in range(3)]
            Y[m][0] = Y[m][0] + f * mono[0] * mono[1] * mono[2]
            for x in range(3):
                if abc[x]:
                    der = list(mono)
                    der[x] = abc[x] * pw[abc[x] - 1][:, x]
                    Y[m][1 + x] = Y[m][1 + x] + f * der[0] * der[1] * der[2]
        for y in Y:
            cols.append(torch.stack([R * y[0]] + [R * y[1 + x] + dR * d[:, x] * y[0] for x in range(3)]))
    return torch.stack(cols, 2)


def _vwn(rs, A, b, c, x0):
    Q, X0 = math.sqrt(4 * c - b * b), x0 * x0 + b * x0 + c
    x = rs.sqrt()
    X, at = x * x + b * x + c, torch.atan(Q / (2 * x + b))
    return A * (torch.log(x * x / X) + 2 * b / Q * at
                - b * x0 / X0 * (torch.log((x - x0) ** 2 / X) + 2 * (b + 2 * x0) / Q * at))


def _pw(rs, A, a1, b1, b2, b3, b4):
    s = rs.sqrt()
    return -2 * A * (1 + a1 * rs) * torch.log1p(1 / (2 * A * (b1 * s + b2 * rs + b3 * rs * s + b4 * rs * rs)))


def _exchange(functional, rho, sigma):
    """Of a closed shell with this total density."""
    if functional == "TF":
        return 0.3 * (3 * math.pi ** 2) ** (2 / 3) * rho ** (5 / 3)
    e = -0.75 * (3 / math.pi) ** (1 / 3) * rho ** (4 / 3)
    if functional == "PBE":
        s2 = sigma / (4 * (3 * math.pi ** 2) ** (2 / 3) * rho ** (8 / 3))
        e = e * (1.804 - 0.804 / (1 + 0.066725 * math.pi ** 2 / 3 / 0.804 * s2))
    return e


def _energy_density(functional, ra, rb, saa, sab, sbb):
    """Per volume, of two spin densities and their gradient products."""
    e = 0.5 * (_exchange(functional, 2 * ra, 4 * saa) + _exchange(functional, 2 * rb, 4 * sbb))
    if functional == "TF":
        return e
    rho, sigma = ra + rb, saa + 2 * sab + sbb
    rs, zeta = (3 / (4 * math.pi) / rho) ** (1 / 3), (ra - rb) / rho
    f = ((1 + zeta) ** (4 / 3) + (1 - zeta) ** (4 / 3) - 2) / (2 ** (4 / 3) - 2)
    fpp0 = 8 / (9 * (2 ** (4 / 3) - 2))
    if functional == "LDA":
        P = _vwn(rs, 0.0310907, 3.72744, 12.9352, -0.10498)
        F = _vwn(rs, 0.01554535, 7.06042, 18.0578, -0.32500)
        S = _vwn(rs, -1 / (6 * math.pi ** 2), 1.13107, 13.0045, -0.0047584)
        return e + rho * (P + S * f * (1 - zeta ** 4) / fpp0 + (F - P) * f * zeta ** 4)
    P = _pw(rs, 0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294)
    F = _pw(rs, 0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517)
    S = _pw(rs, 0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671)
    eps = P - S * f * (1 - zeta ** 4) / fpp0 + (F - P) * f * zeta ** 4
    phi = 0.5 * ((1 + zeta) ** (2 / 3) + (1 - zeta) ** (2 / 3))
    t2 = math.pi / (16 * (3 * math.pi ** 2) ** (1 / 3)) * sigma / (phi ** 2 * rho ** (7 / 3))
    gamma, beta = (1 - math.log(2)) / math.pi ** 2, 0.06672455060314922
    At2 = beta / gamma / torch.expm1(-eps / (gamma * phi ** 3)) * t2
    return e + rho * (eps + gamma * phi ** 3 * torch.log1p(beta / gamma * t2 * (1 + At2) / (1 + At2 * (1 + At2))))


def _dot(x, y):
    return (x[1:] * y[1:]).sum(0)


def _evaluate(functional, spins, w):
    """Energy of the spin densities (two of (4, points): density and gradient) and the weighted derivatives."""
    d = [s.detach().clone().requires_grad_(True) for s in spins]
    on = ((d[0][0] + d[1][0]) > 1e-14) & (d[0][0] > 1e-15) & (d[1][0] > 1e-15)
    a, b = d[0][:, on], d[1][:, on]
    E = (w[on] * _energy_density(functional, a[0], b[0], _dot(a, a), _dot(a, b), _dot(b, b))).sum()
    E.backward()
    return float(E.detach()), [x.grad for x in d]


def _on_grid(phi, P):
    """(4, points): density and gradient of P."""
    T = phi[0] @ P
    return torch.stack([(T * phi[0]).sum(1)] + [2 * (T * phi[1 + x]).sum(1) for x in range(3)])


def _assemble(phi, v):
    G = 0.5 * v[0][:, None] * phi[0] + sum(v[1 + x][:, None] * phi[1 + x] for x in range(3))
    M = phi[0].T @ G
    return M + M.T


def _chunks(grid, size=32768):
    pts, w = torch.from_numpy(grid.points), torch.from_numpy(grid.weights)
    return [(pts[i:i + size], w[i:i + size]) for i in range(0, len(w), size)]


def _exact_build(name, functional, Z, X, Ps, grid=None):
    """Energy and potential matrices of the spin densities Ps (their halves for a closed shell)."""
    b = xc.BasisController.from_file(name, Z, X)
    grid = grid or xc.molecular_grid(Z, X, ctx=_context())
    E, F = 0.0, [torch.zeros_like(P) for P in Ps]
    for pts, w in _chunks(grid):
        phi = _aos(b, pts)
        spins = [_on_grid(phi, P) for P in Ps]
        e, v = _evaluate(functional, spins * (2 // len(Ps)), w)
        E += e
        for f, x in zip(F, v):
            f += _assemble(phi, x)
    return E, F


def _exact_embedding(case, seed):
    """Each sweep step's non-additive energies and potentials."""
    parts, Z, X = _embedded(case, seed)
    grid = xc.molecular_grid(Z, X, ctx=_context())
    bases = [xc.BasisController.from_file(case["basis"], z, x) for z, x in parts]
    Ps = [0.5 * _density(case["basis"], z, x, seed + i) for i, (z, x) in enumerate(parts)]
    names = (case["functional"], "TF")
    E, F = np.zeros((len(parts), 2)), [[torch.zeros_like(P) for _ in names] for P in Ps]
    for pts, w in _chunks(grid):
        phis = [_aos(b, pts) for b in bases]
        spins = [_on_grid(phi, P) for phi, P in zip(phis, Ps)]
        for k, f in enumerate(names):
            e_sup, v_sup = _evaluate(f, [sum(spins)] * 2, w)
            alone = [_evaluate(f, [s] * 2, w) for s in spins]
            for i, (e, v) in enumerate(alone):
                E[i, k] += e_sup - sum(a[0] for a in alone)
                F[i][k] += _assemble(phis[i], v_sup[0] - v[0])
    return dict(E=E.reshape(-1), F=F)


def _exact_gradient(case, seed):
    """dE_xc / d(nuclei) at a fixed grid and density matrix, through the derivative of the AOs."""
    Z, X = _geometry(case["system"], case["size"], seed)
    b = xc.BasisController.from_file(case["basis"], Z, X)
    P = 0.5 * _density(case["basis"], Z, X, seed)
    xyz, E = torch.from_numpy(X).clone().requires_grad_(True), 0.0
    for pts, w in _chunks(xc.molecular_grid(Z, X, ctx=_context()), 8192):
        phi = _aos(b, pts, xyz[torch.from_numpy(b.atom).long()])
        s = _on_grid(phi, P)
        on = s.detach()[0] > 5e-15
        s, w = s[:, on], w[on]
        e = (w * _energy_density(case["functional"], s[0], s[0], *[_dot(s, s)] * 3)).sum()
        e.backward()
        E += float(e.detach())
    return dict(G=xyz.grad.numpy(), E=E)


def _hermite_index(L):
    return [(t, u, s - t - u) for s in range(L + 1) for t in range(s, -1, -1) for u in range(s - t, -1, -1)]


def _hermite_coulomb(L, alpha, d):
    """R_tuv(alpha, d) for t + u + v <= L, in the order of _hermite_index; alpha (...), d (..., 3)."""
    T = alpha * (d * d).sum(-1)
    # Boys functions: confluent series at the highest order below T = 35, downward recursion; erf form above
    e, small = torch.exp(-T), torch.where(T < 35.0, T, torch.zeros_like(T))
    term = torch.full_like(T, 1.0 / (2 * L + 1))
    top = term.clone()
    for k in range(1, 160):
        term = term * 2 * small / (2 * L + 2 * k + 1)
        top = top + term
    F = [None] * L + [torch.exp(-small) * top]
    for j in range(L, 0, -1):
        F[j - 1] = (2 * small * F[j] + torch.exp(-small)) / (2 * j - 1)
    big = torch.where(T < 35.0, torch.full_like(T, 35.0), T)
    up = [0.5 * torch.sqrt(math.pi / big) * torch.erf(big.sqrt())]
    for j in range(L):
        up.append(((2 * j + 1) * up[j] - e) / (2 * big))
    F = [torch.where(T < 35.0, f, g) for f, g in zip(F, up)]
    level = {}
    for n in range(L, -1, -1):
        new = {(0, 0, 0): (-2 * alpha) ** n * F[n]}
        for tuv in _hermite_index(L - n)[1:]:
            x = next(i for i in range(3) if tuv[i])
            one = tuple(c - (i == x) for i, c in enumerate(tuv))
            r = d[..., x] * level[one]
            if tuv[x] > 1:
                r = r + (tuv[x] - 1) * level[tuple(c - 2 * (i == x) for i, c in enumerate(tuv))]
            new[tuv] = r
        level = new
    return [level[tuv] for tuv in _hermite_index(L)]


def _hermite_pair(la, lb, p, PA, PB):
    """Hermite coefficients (pairs, functions of A, functions of B, tuv) of spherical function products."""
    E = [[[None] * (lb + 1) for _ in range(la + 1)] for _ in range(3)]
    for x in range(3):
        zero = torch.zeros_like(p)
        E[x][0][0] = [torch.ones_like(p)]
        for i in range(la + 1):
            for j in range(lb + 1):
                if i + j == 0:
                    continue
                old, X = (E[x][i - 1][j], PA[:, x]) if i else (E[x][i][j - 1], PB[:, x])
                get = lambda t: old[t] if 0 <= t < len(old) else zero  # noqa: E731,B023
                E[x][i][j] = [get(t - 1) / (2 * p) + X * get(t) + (t + 1) * get(t + 1) for t in range(i + j + 1)]
    tuvs = _hermite_index(la + lb)
    out = torch.zeros(len(p), 2 * la + 1, 2 * lb + 1, len(tuvs), dtype=torch.float64)
    for ma, fa, *a in _harmonics(la):
        for mb, fb, *c in _harmonics(lb):
            for k, tuv in enumerate(tuvs):
                if all(tuv[x] <= a[x] + c[x] for x in range(3)):
                    out[:, ma, mb, k] += fa * fb * E[0][a[0]][c[0]][tuv[0]] * E[1][a[1]][c[1]][tuv[1]] * E[2][a[2]][c[2]][tuv[2]]
    return out


def _hermite_shells(b, pairs):
    """Groups of one angular momentum: (L, exponent, centre, coefficients (k, functions, tuv), AO indices (k, functions))
    of the basis' own primitives, or of its significant primitive pairs (both orders of two shells as one)."""
    shell = torch.from_numpy(np.repeat(np.arange(b.nshell), b.nprim))
    a, c = torch.from_numpy(b.alpha), torch.from_numpy(b.coef)
    x, l = torch.from_numpy(b.center)[shell], torch.from_numpy(b.l)[shell]
    first = torch.from_numpy(b.first).long()[shell]
    for la in range(int(l.max()) + 1):
        for lb in range(int(l.max()) + 1) if pairs else [0]:
            i = torch.nonzero(l == la)[:, 0]
            if pairs:
                j = torch.nonzero(l == lb)[:, 0]
                i, j = (v.reshape(-1) for v in torch.meshgrid(i, j, indexing="ij"))
                i, j = i[shell[j] <= shell[i]], j[shell[j] <= shell[i]]
                p = a[i] + a[j]
                K = c[i] * c[j] * torch.exp(-a[i] * a[j] / p * ((x[i] - x[j]) ** 2).sum(1))
                keep = K.abs() * (math.pi / p) ** 1.5 >= 1e-14
                i, j, p, K = i[keep], j[keep], p[keep], K[keep]
                if not len(i):
                    continue
                C = (a[i, None] * x[i] + a[j, None] * x[j]) / p[:, None]
                E = K[:, None, None, None] * _hermite_pair(la, lb, p, C - x[i], C - x[j])
                yield la + lb, p, C, E, (first[i][:, None] + torch.arange(2 * la + 1), first[j][:, None] + torch.arange(2 * lb + 1))
            elif len(i):
                zero = torch.zeros(len(i), 3, dtype=torch.float64)
                E = c[i, None, None] * _hermite_pair(la, 0, a[i], zero, zero)[:, :, 0]
                yield la, a[i], x[i], E, first[i][:, None] + torch.arange(2 * la + 1)


def _interactions(bra, ket):
    """(bra tuv | ket tuv) of two groups: chunks (slice of the bra, tensor (bra, ket, bra tuv, ket tuv))."""
    L, p, C = bra[:3]
    l, a, A = ket[:3]
    T, t, all_ = _hermite_index(L), _hermite_index(l), {k: i for i, k in enumerate(_hermite_index(L + l))}
    step = max(1, 400000 // len(a) // len(all_) + 1)
    for i in range(0, len(p), step):
        q = p[i:i + step, None]
        R = _hermite_coulomb(L + l, q * a / (q + a), C[i:i + step, None] - A[None])
        pref = 2 * math.pi ** 2.5 / (q * a * (q + a).sqrt())
        yield slice(i, i + step), torch.stack([torch.stack([(-1) ** sum(k) * pref * R[all_[tuple(x + y for x, y in zip(K, k))]]
                                                            for k in t], -1) for K in T], -2)


def _exact_coulomb(case, seed):
    Z, X = _geometry(case["system"], case["size"], seed)
    b = xc.BasisController.from_file(case["basis"], Z, X)
    aux = xc.BasisController.from_file("RI_J_WEIGEND", Z, X)
    P = _density(case["basis"], Z, X, seed)
    fit, pairs = list(_hermite_shells(aux, False)), list(_hermite_shells(b, True))
    M, rhs, J = (torch.zeros(s, dtype=torch.float64) for s in ((aux.nao, aux.nao), (aux.nao,), (b.nao, b.nao)))
    for g in fit:
        for h in fit:
            for at, I in _interactions(g, h):
                block = torch.einsum("kat,ljs,klts->kalj", g[3][at], h[3], I)
                M.index_put_((g[4][at][:, :, None, None].expand(block.shape), h[4][None, None].expand(block.shape)),
                             block, accumulate=True)
    sym = [torch.where(g[4][0][:, 0] == g[4][1][:, 0], 1.0, 2.0).double() for g in pairs]
    D = [s[:, None] * torch.einsum("kab,kabt->kt", P[g[4][0][:, :, None], g[4][1][:, None, :]], g[3]) for g, s in zip(pairs, sym)]
    for g, d in zip(pairs, D):
        for h in fit:
            for at, I in _interactions(g, h):
                rhs.index_put_((h[4],), torch.einsum("kt,klts,ljs->lj", d[at], I, h[3]), accumulate=True)
    x = torch.cholesky_solve(rhs[:, None], torch.linalg.cholesky(M))[:, 0]
    for g, s in zip(pairs, sym):
        V = torch.zeros(len(g[1]), len(_hermite_index(g[0])), dtype=torch.float64)
        for h in fit:
            c = torch.einsum("lj,ljs->ls", x[h[4]], h[3])
            for at, I in _interactions(g, h):
                V[at] += torch.einsum("klts,ls->kt", I, c)
        block = 0.5 * s[:, None, None] * torch.einsum("kt,kabt->kab", V, g[3])
        at = (g[4][0][:, :, None].expand(block.shape), g[4][1][:, None, :].expand(block.shape))
        J.index_put_(at, block, accumulate=True)
        J.index_put_(at[::-1], block, accumulate=True)
    return dict(J=J)


def exact(case, seed):
    """What run() returns for these inputs, in plain 64-bit torch on the host; None where that takes long."""
    kind, name = case["kind"], case["basis"]
    torch.set_num_threads(min(16, torch.get_num_threads()))
    if kind == "coulomb":
        return _exact_coulomb(case, seed) if work(case)["flops"] < 3e8 else None
    if kind == "embedding":
        return _exact_embedding(case, seed) if case["size"] <= 12 else None
    if kind == "packed":
        if case["size"] > 4:
            return None
        E, F = [], []
        for _, k, (Z, X) in _pack_members(case, seed):
            e, f = _exact_build(name, case["functional"], Z, X, [0.5 * _density(name, Z, X, seed + k)])
            E.append(e)
            F += f
        return dict(E=np.array(E), F=F)
    N, n = _extent(case["system"], case["size"], name)[:2]
    if 4.0 * N * n * n > 3e11 or kind == "gradient" and N * n > 4e7:
        return None
    if kind == "gradient":
        return _exact_gradient(case, seed)
    Z, X = _geometry(case["system"], case["size"], seed)
    if kind == "open_shell":
        B = _orbitals(name, Z, X, seed)
        E, F = _exact_build(name, case["functional"], Z, X, [0.5 * C @ C.T for C in (B, B[:, 1:])])
        return dict(E=E, Fa=F[0], Fb=F[1])
    E, F = _exact_build(name, case["functional"], Z, X, [0.5 * _density(name, Z, X, seed)])
    return dict(E=E, F=F[0])
