"""The work a program has this framework do, as timed cases: quadratures (restricted, unrestricted, batched), XC gradients,
the set-up of a new geometry, and the integrals and Coulomb term of the SCF wrapper, on water clusters of 1 to 128
molecules (the systems of the repository's benchmark and tests, at liquid density), in both precisions.

listed() and draw(rng) give cases; prepare(case, seed) what a program holds before the call; run(state) one pass through
the public entry points; work(case) the bytes and operations of a pass; exact(case, seed) the same outputs from plain torch
in 64 bits, written from the mathematics (grid, basis functions, functionals, Gaussian integrals, automatic derivatives).
"""

import itertools
import json
import math
import os

import numpy as np
import torch

from pdynamo3_amd import basis, densities, integrator, molecules, scf
from pdynamo3_amd.definitions import functional_ids

_DATA = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pdynamo3_amd", "data")
ORBITAL, FIT = "6-31g_st", "dgauss-a1-dftjfit"
VOLUME = 45.6                                      # cubic Angstrom per water of the benchmark's clusters


def _case(kind, waters, **options):
    case = {"kind": kind, "waters": waters, "spherical": False, "functional": "blyp", "precision": "fp64", "accuracy": 2}
    case.update(options)
    return case


def listed():
    def named(name, *a, **k):
        return dict(_case(*a, **k), name=name)
    return [
        # One SCF iteration's quadrature of the smallest molecule with the drop-in's defaults: launches and latency.
        named("fock_1_fp64", "fock", 1, spherical=True, functional="pbe"),
        # An ordinary SCF iteration in the fast precision (the benchmark's PBE system).
        named("fock_16_mixed", "fock", 16, functional="pbe", precision="mixed"),
        # The headline system in both precisions.
        named("fock_64_fp64", "fock", 64),
        named("fock_64_mixed", "fock", 64, precision="mixed"),
        # The benchmark's largest system.
        named("fock_128_mixed", "fock", 128, functional="pbe", precision="mixed"),
        # An open-shell molecule (a cation radical), alpha and beta Fock matrices, reference default functions.
        named("uks_9_fp64", "uks", 9, spherical=True, functional="b3lyp"),
        # The request loop: the quadratures of several molecules in one call.
        named("batch_8_mixed", "batch", 10, jobs=8, functional="pbe", precision="mixed"),
        # Forces at the end of an SCF: a geometry step of a large cluster, and a small open-shell one.
        named("gradients_64", "gradients", 64, functional="blyp"),
        named("gradients_uks_5", "gradients_uks", 5, spherical=True, functional="pbe"),
        # A new geometry: grid, basis values and the first quadrature, as every step of an optimisation needs them.
        named("geometry_24_mixed", "geometry", 24, functional="pbe", precision="mixed"),
        # The SCF's integrals at a new geometry: one-electron matrices, electron-fit integrals, fit matrix, first J.
        named("integrals_16", "integrals", 16),
        # The Coulomb term of one SCF iteration on resident integrals.
        named("coulomb_48", "coulomb", 48),
    ]


def draw(rng):
    kind = rng.choice(["fock", "fock", "fock", "uks", "batch", "gradients", "gradients_uks", "geometry", "integrals", "coulomb"])
    most = {"fock": 96, "uks": 40, "batch": 12, "gradients": 32, "gradients_uks": 16, "geometry": 48, "integrals": 14,
            "coulomb": 40}[kind]
    waters = int(round(math.exp(rng.uniform(0.0, math.log(most)))))
    case = _case(kind, waters, spherical=rng.random() < 0.5, functional=rng.choice(["blyp", "pbe", "b3lyp", "lda"]),
                 precision=rng.choice(["fp64", "mixed"]), accuracy=rng.choice([1, 2, 2, 3]) if waters <= 24 else 2)
    if kind == "batch":
        case["jobs"] = rng.randint(2, 12)
    return case


# ---------------------------------------------------------------------------------------------------------------------
# Inputs, from the seed.
# ---------------------------------------------------------------------------------------------------------------------
def _cluster(waters, seed):
    """Atomic numbers, coordinates (bohr), rotations and centres of a random cluster at liquid density."""
    Z, xyz, rotations, centres = molecules.water_cluster(waters, (VOLUME * waters) ** (1.0 / 3.0), seed)
    return Z, molecules.to_bohr(xyz), rotations, centres


def _orbitals(rotations, centres, spherical, rng):
    """Occupied orbitals of a cluster, functions x orbitals: the rotated monomer orbitals with random couplings within a
    water and, falling off with distance, between waters."""
    P1, _ = densities.load_monomer_density(ORBITAL, spherical)
    e, U = np.linalg.eigh(P1)
    occupied = U[:, -5:] * np.sqrt(e[-5:])
    b = basis.load_basis(ORBITAL)
    m, k = P1.shape[0], len(rotations)
    C = np.zeros((m * k, 5 * k))
    for w, R in enumerate(rotations):
        C[w * m:(w + 1) * m, 5 * w:5 * (w + 1)] = densities.monomer_rotation(np.asarray(R), b, spherical).T @ occupied
    d = np.linalg.norm(centres[:, None, :] - centres[None, :, :], axis=2)
    size = np.where(d > 0.0, 0.05 * np.exp(-(d - 2.6) / 1.2), 0.02)
    return C + rng.normal(size=C.shape) * np.repeat(np.repeat(size, m, axis=0), 5, axis=1)


def _packed(C):
    P = C @ C.T
    return np.ascontiguousarray(P[np.tril_indices(P.shape[0])])


def _molecules(case, seed):
    """Per molecule of the case: (Z, xyz, element specification, packed densities: one, or alpha and beta)."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "batch":
        sizes = [max(1, int(case["waters"] * f)) for f in np.linspace(0.5, 1.5, case["jobs"])]
    else:
        sizes = [case["waters"]]
    out = []
    for waters in sizes:
        Z, xyz, rotations, centres = _cluster(waters, int(rng.integers(1 << 30)))
        spec = basis.element_spec(basis.load_basis(ORBITAL), Z)
        if "uks" in case["kind"]:
            a = _orbitals(rotations, centres, case["spherical"], rng)
            b = _orbitals(rotations, centres, case["spherical"], rng)
            P = [_packed(a * math.sqrt(0.5)), _packed(np.delete(b, 0, axis=1) * math.sqrt(0.5))]
        else:
            P = [_packed(_orbitals(rotations, centres, case["spherical"], rng))]
        out.append((Z, xyz, spec, P))
    return out


def _fit_coefficients(case, seed, n):
    return np.random.default_rng(seed + 1).normal(size=n) * 0.1


def prepare(case, seed):
    kind, state = case["kind"], {"case": case}
    mols = _molecules(case, seed)
    state["ids"] = list(functional_ids(case["functional"]))
    if kind in ("integrals", "coulomb"):
        Z, xyz, spec, (P,) = mols[0]
        fit_basis = basis.load_basis(FIT)
        fit = basis.element_spec(fit_basis, Z)
        state.update(Z=Z, xyz=xyz, spec=spec, fit=fit, P=P, F=np.zeros_like(P))
        state["c"] = _fit_coefficients(case, seed, basis.number_of_functions(fit_basis, Z, True))
        if kind == "coulomb":
            state["integrals"] = scf.GPUIntegrals(Z, xyz, spec, case["spherical"], fit)
        return state
    state["jobs"] = []
    for Z, xyz, spec, P in mols:
        grid = None
        if kind != "geometry":
            grid = integrator.QuadratureGrid(Z, xyz, case["accuracy"])
            grid.set_basis(spec, case["spherical"], case["precision"])
        state["jobs"].append({"Z": Z, "xyz": xyz, "spec": spec, "P": P, "V": [np.zeros_like(p) for p in P], "grid": grid})
    if kind == "batch":
        state["batch"] = integrator.QuadratureBatch(len(mols))
    return state


# ---------------------------------------------------------------------------------------------------------------------
# One pass.
# ---------------------------------------------------------------------------------------------------------------------
def run(state):
    case, kind, ids = state["case"], state["case"]["kind"], state["ids"]
    if kind == "coulomb":
        state["F"].fill(0.0)
        b = state["integrals"].fit_b(state["P"])
        state["integrals"].fit_fock(state["c"], state["F"])
        return {"b": b, "fock": state["F"]}
    if kind == "integrals":
        ints = scf.GPUIntegrals(state["Z"], state["xyz"], state["spec"], case["spherical"], state["fit"])
        S, T, V = ints.one_electron()
        M = ints.fit_matrix()
        state["F"].fill(0.0)
        b = ints.fit_b(state["P"])
        ints.fit_fock(state["c"], state["F"])
        ints.close()
        return {"overlap": S, "kinetic": T, "nuclear": V, "fit": M, "b": b, "fock": state["F"]}
    jobs = state["jobs"]
    if kind == "batch":
        for j in jobs:
            j["V"][0].fill(0.0)
        results, _ = state["batch"].integrate([(j["grid"], ids, j["P"][0], j["V"][0]) for j in jobs])
        return {"jobs": [{"en": np.array(r), "fock": j["V"][0]} for r, j in zip(results, jobs)]}
    j = jobs[0]
    if kind == "gradients":
        return {"gradients": j["grid"].gradients(ids, j["P"][0])}
    if kind == "gradients_uks":
        return {"gradients": j["grid"].gradients_uks(ids, j["P"][0], j["P"][1])}
    for V in j["V"]:
        V.fill(0.0)
    if kind == "uks":
        e, n, _ = j["grid"].integrate_uks(ids, j["P"][0], j["P"][1], j["V"][0], j["V"][1])
        return {"en": np.array([e, n]), "fock": j["V"][0], "fock_beta": j["V"][1]}
    if kind == "geometry":
        grid = integrator.QuadratureGrid(j["Z"], j["xyz"], case["accuracy"])
        grid.set_basis(j["spec"], case["spherical"], case["precision"])
        e, n, _ = grid.integrate(ids, j["P"][0], j["V"][0])
        counts = np.array([grid.number_of_points, grid.number_of_blocks, grid.number_of_functions])
        grid.close()
        return {"en": np.array([e, n]), "fock": j["V"][0], "counts": counts}
    e, n, _ = j["grid"].integrate(ids, j["P"][0], j["V"][0])
    return {"en": np.array([e, n]), "fock": j["V"][0]}


# ---------------------------------------------------------------------------------------------------------------------
# Work of a pass.
# ---------------------------------------------------------------------------------------------------------------------
# Grid points per water by accuracy, and the mean and the mean square of the kept functions per point, on clusters of
# these sizes (Cartesian functions; spherical ones are 18/19 of them).
_POINTS = {0: 7700.0, 1: 28000.0, 2: 39000.0, 3: 77000.0, 4: 270000.0}
_WATERS = [1, 2, 4, 8, 16, 32, 64, 128]
_KEPT = [16.0, 26.4, 47.3, 67.1, 73.5, 95.2, 110.8, 125.7]
_KEPT_RMS = [17.1, 27.8, 50.0, 72.8, 85.3, 114.0, 133.8, 153.9]


def _quadrature_work(case, waters, spins=1):
    ratio = 18.0 / 19.0 if case["spherical"] else 1.0
    points = _POINTS[case["accuracy"]] * waters
    x = math.log(waters)
    kept = ratio * float(np.interp(x, np.log(_WATERS), _KEPT))
    square = (ratio * float(np.interp(x, np.log(_WATERS), _KEPT_RMS))) ** 2
    n = (18 if case["spherical"] else 19) * waters
    return points, kept, square, n, spins


def work(case):
    kind, waters = case["kind"], case["waters"]
    if kind in ("integrals", "coulomb"):
        n, fit = (18 if case["spherical"] else 19) * waters, 39 * waters
        # Function pairs within reach of each other (about eight waters around each), times the fit functions.
        rows = min(n * n / 2.0, n * 19.0 * 8.0)
        if kind == "coulomb":   # every integral read once, used in both contractions
            return {"bytes": 8.0 * rows * fit, "flops": 4.0 * rows * fit}
        return {"bytes": 8.0 * rows * fit + 8.0 * (4.0 * n * n / 2 + fit * fit / 2), "flops": 200.0 * rows * fit}
    if kind == "batch":
        parts = [work(dict(case, kind="fock", waters=max(1, int(waters * f)))) for f in np.linspace(0.5, 1.5, case["jobs"])]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    spins = 2 if "uks" in kind else 1
    points, kept, square, n, spins = _quadrature_work(case, waters, spins)
    # Stored values and gradients read once; X = P Phi and the lower triangle of V, 2 kept^2 operations per point each.
    bytes_, flops = points * kept * (32.0 if case["precision"] == "fp64" else 17.0), spins * 4.0 * square * points
    if kind == "geometry":      # points made, values evaluated, stored and read
        bytes_, flops = 2.0 * bytes_ + 32.0 * points, flops + 60.0 * kept * points
    elif kind.startswith("gradients"):   # values and derivatives evaluated, both products, cell functions of near atoms
        bytes_, flops = 32.0 * points + 24.0 * 3 * waters, flops + (200.0 * kept + 40.0 * 3 * waters) * points
    return {"bytes": bytes_ + 16.0 * spins * n * (n + 1) / 2, "flops": flops}


# ---------------------------------------------------------------------------------------------------------------------
# The same outputs in 64 bits.
# ---------------------------------------------------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _tensor(x):
    return torch.as_tensor(np.asarray(x, dtype=np.float64), device=_device())


def exact(case, seed):
    kind, waters = case["kind"], case["waters"]
    most = {"fock": 64, "uks": 64, "batch": 12, "gradients": 16, "gradients_uks": 16, "geometry": 64, "integrals": 16,
            "coulomb": 16}[kind]
    if waters > most or (case["accuracy"] > 2 and waters > 20):
        return None
    mols = _molecules(case, seed)
    if kind in ("integrals", "coulomb"):
        Z, xyz, _, (P,) = mols[0]
        fit = basis.number_of_functions(basis.load_basis(FIT), Z, True)
        out = _exact_integrals(Z, xyz, case["spherical"], P, _fit_coefficients(case, seed, fit), kind == "integrals")
        return out
    results = []
    for Z, xyz, _, P in mols:
        e, n, derivatives = _exact_xc(case, Z, xyz, P, kind.startswith("gradients"))
        if kind.startswith("gradients"):
            return {"gradients": derivatives}
        results.append({"en": np.array([e, n]), "fock": derivatives[0]})
        if kind == "uks":
            results[-1]["fock_beta"] = derivatives[1]
    if kind == "batch":
        return {"jobs": results}
    if kind == "geometry":
        results[0]["counts"] = None
    return results[0]


# Basis functions ---------------------------------------------------------------------------------------------------
def _cartesians(l):
    return [(l - y - z, y, z) for z in range(l + 1) for y in range(l - z + 1)]


def _odd(n):
    return math.prod(range(1, n + 1, 2))


def _functions(l, spherical):
    """Functions x monomials of one shell: normalised Cartesians, or real solid harmonics (m = 0, 1c, 1s, 2c, 2s)."""
    pw = _cartesians(l)
    if not spherical or l == 0:
        return np.diag([math.sqrt(_odd(2 * l - 1) / math.prod(_odd(2 * k - 1) for k in p)) for p in pw])
    terms = {1: [{(0, 0, 1): 1.0}, {(1, 0, 0): 1.0}, {(0, 1, 0): 1.0}],
             2: [{(0, 0, 2): 1.0, (2, 0, 0): -0.5, (0, 2, 0): -0.5}, {(1, 0, 1): math.sqrt(3.0)}, {(0, 1, 1): math.sqrt(3.0)},
                 {(2, 0, 0): math.sqrt(0.75), (0, 2, 0): -math.sqrt(0.75)}, {(1, 1, 0): math.sqrt(3.0)}]}[l]
    return np.array([[t.get(p, 0.0) for p in pw] for t in terms])


def _shells(label, Z, spherical):
    """(atom, l, exponents, coefficients with the primitives' norms, first function) of every shell of one l."""
    with open(os.path.join(_DATA, "basis_{:s}.json".format(label))) as f:
        elements = json.load(f)["elements"]
    out, first = [], 0
    for a, z in enumerate(Z):
        for sh in elements[str(int(z))]["shells"]:
            ex = np.array(sh["exponents"])
            for k, l in enumerate(range(sh["lLow"], sh["lHigh"] + 1)):
                norm = (np.pi / (2.0 * ex)) ** 1.5 * _odd(2 * l - 1) / (4.0 * ex) ** l
                out.append((a, l, ex, np.array(sh["coefficients"])[:, k] / np.sqrt(norm), first))
                first += 2 * l + 1 if spherical else len(_cartesians(l))
    return out, first


def _values(points, xyz, groups, n):
    """Phi and its three derivatives at the points, points x functions each; groups: shells alike but for their atoms."""
    out = [points.new_zeros(points.shape[0], n) for _ in range(4)]
    for atoms, l, ex, co, T, columns in groups:
        d = points[:, None, :] - xyz[atoms][None]
        r2 = (d * d).sum(-1)
        R = R1 = 0.0
        for a, c in zip(ex, co):
            g = c * torch.exp(-a * r2)
            R, R1 = R + g, R1 - 2.0 * a * g
        powers = [[torch.ones_like(r2)] + [d[..., k] ** i for i in range(1, l + 1)] for k in range(3)]
        cart = [[], [], [], []]
        for p in _cartesians(l):
            m = [powers[k][p[k]] for k in range(3)]
            full = m[0] * m[1] * m[2]
            cart[0].append(full * R)
            for k in range(3):
                lower = 0.0
                if p[k] > 0:
                    others = [m[q] for q in range(3) if q != k]
                    lower = p[k] * powers[k][p[k] - 1] * others[0] * others[1] * R
                cart[1 + k].append(lower + full * d[..., k] * R1)
        for k in range(4):
            f = torch.stack(cart[k], -1) @ T.T
            out[k] = out[k].index_copy(1, columns, f.reshape(f.shape[0], -1))
    return out


def _groups(label, Z, spherical):
    shells, n = _shells(label, Z, spherical)
    same = {}
    for a, l, ex, co, first in shells:
        same.setdefault((l, tuple(ex), tuple(co)), []).append((a, first))
    groups = []
    for (l, ex, co), members in same.items():
        T = _functions(l, spherical)
        columns = [first + k for _, first in members for k in range(T.shape[0])]
        groups.append((torch.tensor([a for a, _ in members], device=_device()), l, ex, co, _tensor(T),
                       torch.tensor(columns, device=_device())))
    return groups, n


# Grid --------------------------------------------------------------------------------------------------------------
def _sphere(size):
    """Points and weights of the octahedral rule with the given number of points, from its orbits."""
    with open(os.path.join(_DATA, "lebedev.json")) as f:
        orbits = json.load(f)[str(size)]
    out = []
    for kind, a, b, w in orbits:
        v = {1: (1.0, 0.0, 0.0), 2: (math.sqrt(0.5), math.sqrt(0.5), 0.0), 3: (math.sqrt(1.0 / 3.0),) * 3,
             4: (a, a, math.sqrt(max(0.0, 1.0 - 2.0 * a * a))), 5: (a, math.sqrt(max(0.0, 1.0 - a * a)), 0.0),
             6: (a, b, math.sqrt(max(0.0, 1.0 - a * a - b * b)))}[int(kind)]
        images = {tuple(s * x + 0.0 for s, x in zip(signs, p)) for p in itertools.permutations(v)
                  for signs in itertools.product((1.0, -1.0), repeat=3)}
        out += [p + (w,) for p in sorted(images)]
    assert len(out) == size
    return np.array(out)


_SIZES = [6, 14, 26, 38, 50, 74, 86, 110, 146, 170, 194, 230, 266, 302, 350, 434, 590, 770, 974, 1202, 1454]
_BRAGG = {1: 0.35, 8: 0.60}
_LEVELS = {0: (21, 194, 20.0), 1: (35, 434, 25.0), 2: (49, 434, 30.0), 3: (70, 590, 35.0), 4: (100, 1454, 35.0)}


def _atom_grid(z, accuracy):
    """Points relative to a nucleus (H or O) and their weights without the cell function."""
    shells, largest, far = _LEVELS[accuracy]
    scale = 1.0e-10 / 5.291772083e-11 * _BRAGG[z]
    rules, points, weights = {}, [], []
    for i in range(1, shells + 1):
        x = i / (1.0 + shells)
        r = scale * (x / (1.0 - x)) ** 2
        if r > far:
            break
        size = largest
        if r <= 0.2 * scale:
            wanted = math.ceil(largest * r / (0.2 * scale))
            size = 38 if wanted < 38 else next(s for s in _SIZES if s >= wanted)
        u = rules.setdefault(size, _sphere(size) if size not in rules else None)
        points.append(r * u[:, :3])
        weights.append(u[:, 3] * 4.0 * math.pi * 2.0 * scale ** 3 * x ** 5 / (1.0 - x) ** 7 / (1.0 + shells))
    return np.concatenate(points), np.concatenate(weights)


def _cells(points, own, xyz, Z):
    """The own atom's share of each point (Becke's cells with Bragg size adjustment)."""
    r = torch.linalg.vector_norm(points[:, None, :] - xyz[None], dim=-1)
    eye = torch.eye(len(Z), dtype=torch.bool, device=xyz.device)
    d = xyz[:, None, :] - xyz[None]
    R = torch.sqrt((d * d).sum(-1) + eye)
    chi = _tensor([_BRAGG[int(z)] for z in Z])
    u = (chi[:, None] - chi[None]) / (chi[:, None] + chi[None])
    a = torch.clamp(u / (u * u - 1.0), -0.5, 0.5)
    mu = (r[:, :, None] - r[:, None, :]) / R
    nu = mu + a * (1.0 - mu * mu)
    # The smooth step is 1/2 less a multiple of the integral of (1 - x^2)^10 from 0 to nu.
    c = [(-1.0) ** t * math.comb(10, t) / (2 * t + 1) for t in range(11)]
    nu2, poly = nu * nu, c[10]
    for t in range(9, -1, -1):
        poly = poly * nu2 + c[t]
    s = torch.where(eye, 1.0, 0.5 - 0.5 / sum(c) * poly * nu)
    cell = torch.prod(s, dim=2)
    return cell.gather(1, own[:, None])[:, 0] / cell.sum(1)


# Functionals: energy per volume of (rho_a, rho_b, |grad rho_a|^2, grad a . grad b, |grad rho_b|^2) -------------------
def _f_zeta(z):
    return ((1.0 + z) ** (4.0 / 3.0) + (1.0 - z) ** (4.0 / 3.0) - 2.0) / (2.0 ** (4.0 / 3.0) - 2.0)


def _slater(a, b, *_):
    return -1.5 * (0.75 / math.pi) ** (1.0 / 3.0) * (a ** (4.0 / 3.0) + b ** (4.0 / 3.0))


def _b88(a, b, saa, sab, sbb):
    e = _slater(a, b)
    for r, s in ((a, saa), (b, sbb)):
        r43 = r ** (4.0 / 3.0)
        x = torch.sqrt(s + 1.0e-60) / r43
        e = e - 0.0042 * r43 * x * x / (1.0 + 6.0 * 0.0042 * x * torch.asinh(x))
    return e


def _pbe_x(a, b, saa, sab, sbb):
    kappa, mu, e = 0.804, 0.2195149727645171, 0.0
    for r, s in ((a, saa), (b, sbb)):
        s2 = 4.0 * s / (4.0 * (3.0 * math.pi ** 2) ** (2.0 / 3.0) * (2.0 * r) ** (8.0 / 3.0))
        unif = -0.75 * (3.0 / math.pi) ** (1.0 / 3.0) * (2.0 * r) ** (4.0 / 3.0)
        e = e + 0.5 * unif * (1.0 + kappa - kappa / (1.0 + mu * s2 / kappa))
    return e


def _pbe_c(a, b, saa, sab, sbb):
    rho = a + b
    z = (a - b) / rho
    rs = (3.0 / (4.0 * math.pi * rho)) ** (1.0 / 3.0)

    def fit(A, al, b1, b2, b3, b4):
        q = 2.0 * A * (b1 * rs ** 0.5 + b2 * rs + b3 * rs ** 1.5 + b4 * rs * rs)
        return -2.0 * A * (1.0 + al * rs) * torch.log1p(1.0 / q)
    e0 = fit(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294)
    e1 = fit(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517)
    stiff = -fit(0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671)
    f2, f, z4 = 1.709920934161365617563962776245, _f_zeta(z), z ** 4
    ec = e0 + stiff * f * (1.0 - z4) / f2 + (e1 - e0) * f * z4
    beta, gamma = 0.06672455060314922, (1.0 - math.log(2.0)) / math.pi ** 2
    phi = 0.5 * ((1.0 + z) ** (2.0 / 3.0) + (1.0 - z) ** (2.0 / 3.0))
    t2 = (saa + 2.0 * sab + sbb) / (16.0 * 2.0 ** (2.0 / 3.0) * phi ** 2 * rs * rho ** (8.0 / 3.0))
    A = beta / gamma / torch.expm1(-ec / (gamma * phi ** 3))
    return rho * (ec + gamma * phi ** 3 * torch.log1p(beta / gamma * t2 * (1.0 + A * t2) / (1.0 + A * t2 + (A * t2) ** 2)))


def _lyp(a, b, saa, sab, sbb):
    A, B, C, D = 0.04918, 0.132, 0.2533, 0.349
    rho, s = a + b, saa + 2.0 * sab + sbb
    r3 = rho ** (-1.0 / 3.0)
    omega = torch.exp(-C * r3) / (1.0 + D * r3) * rho ** (-11.0 / 3.0)
    delta = C * r3 + D * r3 / (1.0 + D * r3)
    cf = 0.3 * (3.0 * math.pi ** 2) ** (2.0 / 3.0)
    inner = (2.0 ** (11.0 / 3.0) * cf * (a ** (8.0 / 3.0) + b ** (8.0 / 3.0)) + (47.0 - 7.0 * delta) / 18.0 * s
             - (2.5 - delta / 18.0) * (saa + sbb) - (delta - 11.0) / 9.0 * (a / rho * saa + b / rho * sbb))
    tail = -2.0 / 3.0 * rho ** 2 * s + (2.0 / 3.0 * rho ** 2 - a * a) * sbb + (2.0 / 3.0 * rho ** 2 - b * b) * saa
    return -4.0 * A / (1.0 + D * r3) * a * b / rho - A * B * omega * (a * b * inner + tail)


def _vwn(a, b, rpa):
    rho = a + b
    z, x = (a - b) / rho, (3.0 / (4.0 * math.pi * rho)) ** (1.0 / 6.0)

    def fit(A, b, c, x0):
        Q, X, X0 = math.sqrt(4.0 * c - b * b), x * x + b * x + c, x0 * x0 + b * x0 + c
        at = torch.atan(Q / (2.0 * x + b))
        return A * (torch.log(x * x / X) + 2.0 * b / Q * at
                    - b * x0 / X0 * (torch.log((x - x0) ** 2 / X) + 2.0 * (2.0 * x0 + b) / Q * at))
    if rpa:   # the fits to the RPA energies, interpolated between the two limits (as B3LYP takes them)
        e0, e1 = fit(0.0310907, 13.0720, 42.7198, -0.409286), fit(0.01554535, 20.1231, 101.578, -0.743294)
        return rho * (e0 + (e1 - e0) * _f_zeta(z))
    e0, e1 = fit(0.0310907, 3.72744, 12.9352, -0.10498), fit(0.01554535, 7.06042, 18.0578, -0.32500)
    stiff = fit(-1.0 / (6.0 * math.pi ** 2), 1.13107, 13.0045, -0.0047584)
    f, z4 = _f_zeta(z), z ** 4
    return rho * (e0 + stiff * f * (1.0 - z4) * 9.0 * (2.0 ** (1.0 / 3.0) - 1.0) / 4.0 + (e1 - e0) * f * z4)


_FUNCTIONALS = {
    "lda": lambda *v: _slater(*v) + _vwn(v[0], v[1], False),
    "blyp": lambda *v: _b88(*v) + _lyp(*v),
    "pbe": lambda *v: _pbe_x(*v) + _pbe_c(*v),
    "b3lyp": lambda *v: 0.08 * _slater(*v) + 0.72 * _b88(*v) + 0.19 * _vwn(v[0], v[1], True) + 0.81 * _lyp(*v)}


def _exact_xc(case, Z, xyz, P, gradients):
    """E_xc, electrons, and the derivatives of E_xc: with respect to each packed density (the Fock matrices), or to the
    nuclei, the grid moving with them (gradients)."""
    groups, n = _groups(ORBITAL, Z, case["spherical"])
    spins, rows, cols = [], *np.tril_indices(n)
    for p in P:
        D = np.zeros((n, n))
        D[rows, cols] = D[cols, rows] = p
        spins.append(_tensor(D).requires_grad_(not gradients))
    centres = _tensor(xyz).requires_grad_(gradients)
    atoms = {int(z): _atom_grid(int(z), case["accuracy"]) for z in set(Z)}
    step = max(256, min(1 << 15, int(4.0e8 / (len(Z) ** 2 + 8.0 * n)) // (4 if gradients else 1)))
    energy = electrons = 0.0
    owns = np.concatenate([np.full(len(atoms[int(z)][1]), a) for a, z in enumerate(Z)])
    relative = np.concatenate([atoms[int(z)][0] for z in Z])
    bare = np.concatenate([atoms[int(z)][1] for z in Z])
    for k in range(0, len(owns), step):
        own = torch.tensor(owns[k:k + step], device=_device())
        points = _tensor(relative[k:k + step]) + centres[own]
        w = _tensor(bare[k:k + step]) * _cells(points, own, centres, Z)
        phi = _values(points, centres, groups, n)
        rho, grad = [], []
        for D in spins:
            X = phi[0] @ D
            rho.append((phi[0] * X).sum(1))
            grad.append([2.0 * (phi[1 + c] * X).sum(1) for c in range(3)])
        if len(spins) == 1:
            rho, grad = [0.5 * rho[0]] * 2, [[0.5 * g for g in grad[0]]] * 2
        keep = (rho[0] + rho[1] > 5.0e-13) & (rho[0] > 1.0e-13) & (rho[1] > 1.0e-13)
        dot = [sum(g * h for g, h in zip(grad[i], grad[j]))[keep] for i, j in ((0, 0), (0, 1), (1, 1))]
        part = (w[keep] * _FUNCTIONALS[case["functional"]](rho[0][keep], rho[1][keep], *dot)).sum()
        part.backward()
        energy += float(part.detach())
        electrons += float((w * (rho[0] + rho[1])).sum().detach())
    if gradients:
        return energy, electrons, centres.grad.cpu().numpy()
    V = [(0.5 * (D.grad + D.grad.T)).cpu().numpy()[rows, cols] for D in spins]
    return energy, electrons, V


# Gaussian integrals (Hermite expansions; Helgaker, Jorgensen, Olsen, Molecular Electronic-Structure Theory, ch. 9) ----
def _hermites(L):
    return [(t, u, v) for t in range(L + 1) for u in range(L + 1 - t) for v in range(L + 1 - t - u)]


def _expansion(la, lb, p, pa, pb, first):
    """E[i][j][t] in one dimension of x_A^i x_B^j exp(...), from E[0][0][0] = first."""
    E = [[None] * (lb + 1) for _ in range(la + 1)]
    E[0][0] = [first]

    def up(e, x):
        g = lambda t: e[t] if 0 <= t < len(e) else 0.0   # noqa: E731
        return [g(t - 1) / (2.0 * p) + x * g(t) + (t + 1) * g(t + 1) for t in range(len(e) + 1)]
    for i in range(la + 1):
        if i:
            E[i][0] = up(E[i - 1][0], pa)
        for j in range(1, lb + 1):
            E[i][j] = up(E[i][j - 1], pb)
    return E


def _boys(L, T):
    """F_0 .. F_L."""
    small = T < 0.05
    out = []
    for n in range(L + 1):
        series = sum((-T) ** k / (math.factorial(k) * (2 * n + 2 * k + 1)) for k in range(9))
        safe = torch.where(small, torch.ones_like(T), T)
        a = torch.full_like(T, n + 0.5)
        out.append(torch.where(small, series, torch.special.gammainc(a, safe) * math.gamma(n + 0.5) / (2.0 * safe ** (n + 0.5))))
    return out


def _coulomb(L, alpha, d):
    """{(t, u, v): R_tuv} for t + u + v <= L."""
    F = _boys(L, alpha * (d * d).sum(-1))
    level = {}
    for n in range(L, -1, -1):
        new = {(0, 0, 0): (-2.0 * alpha) ** n * F[n]}
        for s in range(1, L - n + 1):
            for h in _hermites(s):
                if sum(h) != s:
                    continue
                k = next(i for i in range(3) if h[i])
                one = tuple(h[i] - (i == k) for i in range(3))
                new[h] = d[..., k] * level[one]
                if one[k]:
                    two = tuple(one[i] - (i == k) for i in range(3))
                    new[h] = new[h] + one[k] * level[two]
        level = new
    return level


def _pairs(left, right, xyz, diagonal):
    """Primitive pairs of the shell pairs (A, B) of two lists, A not before B: shells, exponents, product, indices."""
    shells = [(i, j) for i in left for j in right if not diagonal or i[4] >= j[4]]
    which, a, b, c, A, B = [], [], [], [], [], []
    for k, (s, t) in enumerate(shells):
        for ea, ca in zip(s[2], s[3]):
            for eb, cb in zip(t[2], t[3]):
                which.append(k), a.append(ea), b.append(eb), c.append(ca * cb), A.append(xyz[s[0]]), B.append(xyz[t[0]])
    a, b, A, B = _tensor(a), _tensor(b), _tensor(A).reshape(-1, 3), _tensor(B).reshape(-1, 3)
    return shells, torch.tensor(which, device=_device()), a, b, _tensor(c), A, B


def _pair_table(la, lb, E, H):
    """Pair coefficients [primitive pairs, Cartesian pairs, Hermites]."""
    out = []
    for x in _cartesians(la):
        for y in _cartesians(lb):
            for h in H:
                f = 1.0
                for k in range(3):
                    e = E[k][x[k]][y[k]]
                    f = f * e[h[k]] if h[k] < len(e) else None
                    if f is None:
                        break
                out.append(torch.zeros_like(E[0][0][0][0]) if f is None else f)
    return torch.stack(out, -1).reshape(-1, len(_cartesians(la)) * len(_cartesians(lb)), len(H))


def _single_table(l, g, H):
    """One shell's coefficients [shells, Cartesians, Hermites], with the sign of the second charge distribution."""
    zero, one = torch.zeros_like(g), torch.ones_like(g)
    e = _expansion(l, 0, g, zero, zero, one)
    out = []
    for x in _cartesians(l):
        for h in H:
            f = one * (-1.0) ** sum(h)
            for k in range(3):
                f = f * (e[x[k]][0][h[k]] if h[k] <= x[k] else zero)
            out.append(f)
    return torch.stack(out, -1).reshape(-1, len(_cartesians(l)), len(H))


def _exact_integrals(Z, xyz, spherical, P, coefficients, everything):
    shells, n = _shells(ORBITAL, Z, spherical)
    fits, nf = _shells(FIT, Z, True)
    D, out = np.zeros((n, n)), {}
    rows, cols = np.tril_indices(n)
    D[rows, cols] = D[cols, rows] = P
    D, C = _tensor(D), _tensor(coefficients)
    S, T, V, J = (torch.zeros(n, n, dtype=torch.float64, device=_device()) for _ in range(4))
    b = torch.zeros(nf, dtype=torch.float64, device=_device())
    transform = lambda l, s: _tensor(_functions(l, s))   # noqa: E731
    by_l = lambda s: {l: [x for x in s if x[1] == l] for l in sorted({x[1] for x in s})}   # noqa: E731
    orbital, fitting = by_l(shells), by_l(fits)
    centres, charges = _tensor(xyz), _tensor(np.asarray(Z, dtype=float))
    width = 4.0 / (1.0e-4 ** 2 * math.pi)
    for la, left in orbital.items():
        for lb, right in orbital.items():
            sets, which, a, bb, cc, A, B = _pairs(left, right, xyz, True)
            if not sets:
                continue
            Ta, Tb = transform(la, spherical), transform(lb, spherical)
            p = a + bb
            centre = (a[:, None] * A + bb[:, None] * B) / p[:, None]
            H = _hermites(la + lb)
            E = [_expansion(la, lb + 2, p, (centre - A)[:, k], (centre - B)[:, k],
                            torch.exp(-a * bb / p * (A - B)[:, k] ** 2)) for k in range(3)]
            table = _pair_table(la, lb, E, H)
            ia = torch.tensor([[s[4] + k for k in range(Ta.shape[0])] for s, _ in sets], device=_device())
            ib = torch.tensor([[t[4] + k for k in range(Tb.shape[0])] for _, t in sets], device=_device())

            def finish(block):
                """Contracted functions [shell pairs, A, B] of primitive Cartesian blocks [primitive pairs, A B]."""
                m = block.new_zeros(len(sets), block.shape[1]).index_add(0, which, cc[:, None] * block)
                return Ta @ m.reshape(len(sets), Ta.shape[1], Tb.shape[1]) @ Tb.T

            def put(M, block):
                M[ia[:, :, None], ib[:, None, :]] = block
            if everything:
                root, overlap, kinetic = torch.sqrt(math.pi / p), [], []
                for x in _cartesians(la):
                    for y in _cartesians(lb):
                        s = [E[k][x[k]][y[k]][0] * root for k in range(3)]
                        t = []
                        for k in range(3):
                            j = y[k]
                            low = 0.5 * j * (j - 1) * E[k][x[k]][j - 2][0] * root if j > 1 else 0.0
                            t.append(-2.0 * bb * bb * E[k][x[k]][j + 2][0] * root + bb * (2 * j + 1) * s[k] - low)
                        overlap.append(s[0] * s[1] * s[2])
                        kinetic.append(t[0] * s[1] * s[2] + s[0] * t[1] * s[2] + s[0] * s[1] * t[2])
                put(S, finish(torch.stack(overlap, 1)))
                put(T, finish(torch.stack(kinetic, 1)))
                total = torch.zeros_like(table[:, :, 0])
                for k in range(len(Z)):
                    R = _coulomb(la + lb, p * width / (p + width), centre - centres[k])
                    R = torch.stack([R[h] for h in H], -1)
                    factor = -charges[k] * 2.0 * math.pi / p * torch.sqrt(width / (p + width))
                    total = total + factor[:, None] * (table * R[:, None, :]).sum(-1)
                put(V, finish(total))
            weight = torch.where(ia[:, :, None] == ib[:, None, :], 1.0, 2.0)
            inside = (ia[:, :, None] >= ib[:, None, :]) * 1.0
            density = D[ia[:, :, None], ib[:, None, :]] * weight * inside
            # Back to primitive Cartesian weights, so that each chunk of pairs adds its part of b.
            carts = (Ta.T @ density @ Tb).reshape(len(sets), -1)[which] * cc[:, None]
            for lc, third in fitting.items():
                Tc, Hc = transform(lc, True), _hermites(lc)
                g = _tensor([s[2][0] for s in third])
                norm = _tensor([s[3][0] for s in third])
                where = _tensor(np.array([xyz[s[0]] for s in third]))
                single = _single_table(lc, g, Hc) * norm[:, None, None]
                ic = torch.tensor([[s[4] + k for k in range(Tc.shape[0])] for s in third], device=_device())
                cart_c = C[ic] @ Tc
                chunk = max(1, int(2.0e8 / (len(third) * len(H) * len(Hc) * 4)))
                fock = []
                for k in range(0, len(p), chunk):
                    q = p[k:k + chunk, None]
                    alpha = q * g / (q + g)
                    R = _coulomb(la + lb + lc, alpha, centre[k:k + chunk, None, :] - where)
                    scale = 2.0 * math.pi ** 2.5 / (q * g * torch.sqrt(q + g))
                    one = table[k:k + chunk]
                    folded = (carts[k:k + chunk, :, None] * one).sum(1)
                    charge = torch.einsum("mch,mc->mh", single, cart_c)
                    left_sum = torch.zeros(single.shape[0], len(Hc), dtype=torch.float64, device=_device())
                    right_sum = torch.zeros(q.shape[0], len(H), dtype=torch.float64, device=_device())
                    for i, h in enumerate(H):
                        for j, hc in enumerate(Hc):
                            r = scale * R[tuple(x + y for x, y in zip(h, hc))]
                            left_sum[:, j] += folded[:, i] @ r
                            right_sum[:, i] += r @ charge[:, j]
                    b.index_add_(0, ic.reshape(-1), ((left_sum[:, None, :] * single).sum(-1) @ Tc.T).reshape(-1))
                    fock.append((one * right_sum[:, None, :]).sum(-1))
                J[ia[:, :, None], ib[:, None, :]] += finish(torch.cat(fock))
    packed = lambda M: torch.where(M != 0.0, M, M.T).cpu().numpy()[rows, cols]   # noqa: E731
    out = {"b": b.cpu().numpy(), "fock": packed(J)}
    if everything:
        out.update(overlap=packed(S), kinetic=packed(T), nuclear=packed(V), fit=_exact_fit(fitting, nf, xyz))
    return out


def _exact_fit(fitting, nf, xyz):
    """The Coulomb matrix of the fit functions, and their integrals in its last row (packed)."""
    M = torch.zeros(nf + 1, nf + 1, dtype=torch.float64, device=_device())
    for lc, left in fitting.items():
        Tc, Hc = _tensor(_functions(lc, True)), _hermites(lc)
        g, norm = _tensor([s[2][0] for s in left]), _tensor([s[3][0] for s in left])
        one = _single_table(lc, g, Hc) * norm[:, None, None] * _tensor([(-1.0) ** sum(h) for h in Hc])
        ic = torch.tensor([[s[4] + k for k in range(Tc.shape[0])] for s in left], device=_device())
        M[nf, ic.reshape(-1)] = ((one[:, :, Hc.index((0, 0, 0))] * ((math.pi / g) ** 1.5)[:, None]) @ Tc.T).reshape(-1)
        for ld, right in fitting.items():
            Td, Hd = _tensor(_functions(ld, True)), _hermites(ld)
            h, other = _tensor([s[2][0] for s in right]), _tensor([s[3][0] for s in right])
            two = _single_table(ld, h, Hd) * other[:, None, None]
            jd = torch.tensor([[s[4] + k for k in range(Td.shape[0])] for s in right], device=_device())
            q = g[:, None]
            d = _tensor(np.array([xyz[s[0]] for s in left]))[:, None, :] - _tensor(np.array([xyz[s[0]] for s in right]))
            R = _coulomb(lc + ld, q * h / (q + h), d)
            scale = 2.0 * math.pi ** 2.5 / (q * h * torch.sqrt(q + h))
            block = 0.0
            for i, hc in enumerate(Hc):
                for j, hd in enumerate(Hd):
                    r = scale * R[tuple(x + y for x, y in zip(hc, hd))]
                    block = block + r[:, :, None, None] * one[:, None, :, None, i] * two[None, :, None, :, j]
            block = torch.einsum("xc,mncd,yd->mnxy", Tc, block, Td)
            M[ic[:, None, :, None], jd[None, :, None, :]] = block
    return M.cpu().numpy()[np.tril_indices(nf + 1)]
