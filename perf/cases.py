"""Performance cases of the RI-J/K framework: what its users have it do, over the
range of systems they do it for.

A program around this library holds a molecule's fitted B tensor in a
JKContext and calls builds in a loop (every RHF or CASSCF iteration, every
orbital step of a direct minimisation), forms a new B at every geometry, and
builds batches of molecules. Systems are real ones in cc-pVDZ with
cc-pVDZ-JKFIT: water clusters (compact) and all-trans alkanes (extended), the
geometries of `nopt_amd.geometry`. FP64 is the mode that converges an SCF, int8
the mixed mode of its earlier iterations and of everything that needs 1e-7.

A case: kind (what is called), system, n and shape (the molecule), prec, and
for some kinds one more number. prepare() makes core-guess orbitals rotated by a random
occupied-virtual mixing of size 1e-2 (seeded), their densities, and a context
with B formed, all of which such a program has in hand before its call.
"""
import functools

import numpy as np
import torch

from nopt_amd import geometry
from nopt_amd.autograd import rhf_energy
from nopt_amd.jk import JKContext, RaggedPlan
from nopt_amd.molecule import Molecule

KINDS = ("device", "host", "pair", "gradient", "ragged", "geometry", "active")


def listed():
    return [
        # one SCF iteration of the smallest molecule (24 functions, 5 orbitals):
        # launches and latency
        dict(name="water_fp64", kind="device", system="water", n=1, prec="fp64"),
        # the same in the mixed mode for a few molecules (72 functions)
        dict(name="water3_int8", kind="device", system="water", n=3, prec="int8"),
        # the headline system C20H42 (490 functions, 2366 auxiliary functions,
        # 81 orbitals), the converging mode and the mixed mode
        dict(name="c20_fp64", kind="device", system="alkane", n=20, prec="fp64"),
        dict(name="c20_int8", kind="device", system="alkane", n=20, prec="int8"),
        # the drop-in call on host arrays, as an SCF code linked against the
        # library makes it (250 functions)
        dict(name="c10_host_fp64", kind="host", system="alkane", n=10, prec="fp64"),
        # the two densities of a CASSCF step, inactive and total, in one call
        dict(name="cas_pair_fp64", kind="pair", system="water", n=8, prec="fp64"),
        dict(name="cas_pair_int8", kind="pair", system="water", n=13, prec="int8"),
        # forward and backward of E_RHF(C): a step of a torch optimiser over
        # orbital rotations
        dict(name="c12_gradient_fp64", kind="gradient", system="alkane", n=12, prec="fp64"),
        # a ragged batch of clusters of 1..16 molecules, two densities each, as
        # one plan
        dict(name="ragged_int8", kind="ragged", system="water", n=16, prec="int8", count=12),
        # a new geometry: B from the integrals and the metric on the host, then
        # the first build of its SCF
        dict(name="c10_geometry", kind="geometry", system="alkane", n=10, prec="int8"),
        # the active-space integrals of a CASSCF step (10 active orbitals)
        dict(name="water10_active", kind="active", system="water", n=10, prec="fp64", active=10),
        # a large cluster with B as the packed triangle alone (768 functions,
        # 160 orbitals): what a system whose full rows do not fit runs
        dict(name="water32_compact_int8", kind="device", system="water", n=32, prec="int8", compact=True),
    ]


def draw(rng):
    kind = rng.choices(KINDS, weights=(4, 2, 2, 2, 1, 1, 1))[0]
    system = rng.choice(("water", "alkane")) if kind in ("device", "host", "gradient", "geometry") else "water"
    top = {"device": 20, "host": 14, "pair": 14, "gradient": 14, "ragged": 12, "geometry": 8, "active": 14}[kind]
    # sizes spread over the logarithm; a cluster of n waters is about as large
    # as an alkane of n carbons
    n = min(top, max(1, int(round(np.exp(rng.uniform(0.0, np.log(top + 0.49)))))))
    case = dict(kind=kind, system=system, n=n, prec=rng.choice(("fp64", "int8")))
    case["shape"] = rng.randint(1, 9999) if system == "water" else round(rng.uniform(1.46, 1.62), 4)
    if kind == "device" and case["prec"] == "int8":
        case["compact"] = rng.random() < 0.3
    if kind == "ragged":
        case.update(n=max(3, n), prec="int8", count=rng.randint(3, 10))
    if kind == "pair":
        case["n"] = max(2, n)  # ten active orbitals beside the core
    if kind == "active":
        case.update(n=max(2, n), prec="fp64", active=rng.randint(2, 24))
    return case


# ------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=16)
def molecule(system, n, shape):
    """Host arrays of one molecule (shape: an alkane's C-C distance, a
    cluster's placement seed), the same for every pass over it: packed
    (P|mn), the metric, the core Hamiltonian and its orbitals (rows)."""
    sym, xyz = geometry.alkane(n, r_cc=shape) if system == "alkane" else geometry.water_cluster(n, seed=shape)
    m = Molecule.from_angstrom(sym, xyz, basis="cc-pvdz", aux="cc-pvdz-jkfit")
    S, T, V = m.one_electron()
    s, U = np.linalg.eigh(S)
    X = U @ np.diag(s ** -0.5) @ U.T
    C = X @ np.linalg.eigh(X.T @ (T + V) @ X)[1]
    return dict(nbf=m.nbf, naux=m.naux, nocc=m.nocc, eri3=m.eri3_packed(), metric=m.metric(), H=T + V,
                C=np.ascontiguousarray(C.T))


def rotated(m, seed):
    """All orbitals as rows, occupied and virtual ones mixed at random, and
    orthonormal again within the occupied set."""
    rng = np.random.default_rng([20, seed])
    C, o = m["C"], m["nocc"]
    kappa = 1e-2 * rng.standard_normal((o, m["nbf"] - o))
    w, U = np.linalg.eigh(np.eye(o) + kappa @ kappa.T)
    occ = (U * w ** -0.5) @ U.T @ (C[:o] + kappa @ C[o:])
    return np.vstack([occ, C[o:]])


def pair_factors(m, seed):
    """The orbital factors of a CASSCF step: the inactive orbitals, and
    [sqrt(2) C_core; NO sqrt(n/2)] with 10 active orbitals and a random
    positive 1-RDM of trace 10."""
    C, ncore = rotated(m, seed), m["nocc"] - 5
    rng = np.random.default_rng([21, seed])
    A = rng.standard_normal((10, 10))
    occ, W = np.linalg.eigh(A @ A.T * (10.0 / np.trace(A @ A.T)))
    NO = W.T @ C[ncore:ncore + 10]
    return C[:ncore], np.vstack([np.sqrt(2.0) * C[:ncore], NO * np.sqrt(0.5 * np.clip(occ, 0.0, None))[:, None]])


def systems(case):
    """(system, n, shape) of every molecule of a case."""
    shape = case.get("shape", 1.54 if case["system"] == "alkane" else 1)
    if case["kind"] != "ragged":
        return [(case["system"], case["n"], shape)]
    sizes = geometry.batch_sizes(case["count"], case["n"], seed=0)
    sizes = [max(2, v) for v in sizes[:-1]] + [case["n"]]  # ten active orbitals beside the core
    return [(case["system"], v, shape + k) for k, v in enumerate(sizes)]


def gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def context(case, m):
    form = "int8" if case.get("compact") or case["kind"] == "ragged" else "both"
    ctx = JKContext(m["nbf"], m["naux"], keep=form, compact=bool(case.get("compact")))
    ctx.set_B(m["eri3"], m["metric"])
    return ctx


def device_items(factors, n):
    """(D, C, J, K) tensors of each factor and the items of a batched build."""
    tensors, items = [], []
    for f in factors:
        C = gpu(f)
        D = C.T @ C
        J, K = torch.empty(n, n, dtype=torch.float64, device="cuda"), torch.empty(n, n, dtype=torch.float64, device="cuda")
        tensors.append((D, C, J, K))
        items.append((D.data_ptr(), C.data_ptr(), len(f), J.data_ptr(), K.data_ptr()))
    return tensors, items


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, prec=case["prec"])
    mols = [molecule(*key) for key in systems(case)]
    m = mols[0]
    occ = None if kind in ("pair", "ragged") else np.ascontiguousarray(rotated(m, seed)[:m["nocc"]])
    if kind == "geometry":
        s.update(ctx=JKContext(m["nbf"], m["naux"]), m=m, C=occ, D=occ.T @ occ)
        return s
    if kind == "ragged":
        s["ctx"] = [context(case, x) for x in mols]
        made = [device_items(pair_factors(x, seed + 1000 * k), x["nbf"]) for k, x in enumerate(mols)]
        torch.cuda.synchronize()
        s["tensors"] = [t for ts, _ in made for t in ts]
        s["plan"] = RaggedPlan([(c, items) for c, (_, items) in zip(s["ctx"], made)])
        return s
    s["ctx"] = context(case, m)
    if kind == "host":
        s.update(C=occ, D=occ.T @ occ)
    elif kind == "active":
        o, a = m["nocc"], min(case["active"], m["nbf"])
        lo = max(0, o - a // 2)
        s["C"] = np.ascontiguousarray(rotated(m, seed)[lo:lo + a])
    elif kind == "gradient":
        s.update(C=gpu(occ).requires_grad_(True), H=gpu(m["H"]))
    else:
        s["tensors"], s["items"] = device_items(pair_factors(m, seed) if kind == "pair" else [occ], m["nbf"])
        torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- passes
def run(s):
    kind, ctx, prec = s["kind"], s["ctx"], s["prec"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "device":
        D, C, n, J, K = s["items"][0]
        ctx.build_device(D, C, n, J, K, prec=prec, stream=stream)
        return s["tensors"][0][2:]
    if kind == "pair":
        ctx.build_batch_device(s["items"], prec=prec, stream=stream)
        return [t[2:] for t in s["tensors"]]
    if kind == "ragged":
        s["plan"].launch(stream)
        return [t[2:] for t in s["tensors"]]
    if kind == "host":
        return ctx.build(s["D"], s["C"], prec=prec)
    if kind == "geometry":
        ctx.set_B(s["m"]["eri3"], s["m"]["metric"])
        return ctx.build(s["D"], s["C"], prec=prec)
    if kind == "active":
        return ctx.active_ints(s["C"])
    s["C"].grad = None
    E = rhf_energy(s["C"], s["H"], ctx, prec=prec)
    E.backward()
    return E.detach(), s["C"].grad


@functools.lru_cache(maxsize=None)
def dims(system, n):
    """(functions, auxiliary functions, occupied orbitals): 24 and 116 of a
    water molecule; 14 and 70 of a carbon, 5 and 23 of a hydrogen atom."""
    if system == "water":
        return 24 * n, 116 * n, 5 * n
    return 14 * n + 5 * (2 * n + 2), 70 * n + 23 * (2 * n + 2), 4 * n + 1


def work(case):
    """Every value of B's triangle read once (8 bytes, 5 in the integer form),
    the densities and factors read, J and K written; the half-transform, one
    triangle of K, and the Coulomb pair."""
    total = dict(bytes=0.0, flops=0.0)
    for system, n, _ in systems(case):
        nbf, naux, nocc = dims(system, n)
        pairs = nbf * (nbf + 1) // 2
        per = 5 if case["prec"] == "int8" else 8
        if case["kind"] == "active":
            a = min(case["active"], nbf)
            total["bytes"] += 8.0 * naux * pairs + 8.0 * (2 * a * nbf + a ** 4)
            total["flops"] += 2.0 * naux * (nbf * nbf * a + nbf * a * a + a ** 4 / 4)
            continue
        facs = [nocc - 5, nocc + 5] if case["kind"] in ("pair", "ragged") else [nocc]
        total["bytes"] += per * naux * pairs + sum(8.0 * (3 * nbf * nbf + f * nbf) for f in facs)
        total["flops"] += sum(2.0 * naux * nbf * nbf * f + naux * f * nbf * (nbf + 1.0) + 8.0 * naux * pairs for f in facs)
        if case["kind"] == "gradient":
            total["bytes"] += 8.0 * (nbf * nbf + nocc * nbf)
            total["flops"] += 4.0 * nbf * nbf * nocc
        if case["kind"] == "geometry":  # the integrals and the metric come in, B goes out
            total["bytes"] += 16.0 * naux * pairs + 8.0 * naux * naux
            total["flops"] += naux ** 3 / 3.0 + 1.0 * naux * naux * pairs
    return total


# ---------------------------------------------------------------------- exact
def fitted(m):
    """B[Q][m][n] = L^-1 (P|mn) of V = L L^T, full rows, FP64."""
    n = m["nbf"]
    L = torch.linalg.cholesky(gpu(m["metric"]))
    packed = gpu(m["eri3"])
    for part in packed.split(2048, dim=1):  # the solver's workspace grows with the columns
        part.copy_(torch.linalg.solve_triangular(L, part.contiguous(), upper=False))
    r, c = np.tril_indices(n)
    where = np.empty((n, n), dtype=np.int64)
    where[r, c] = where[c, r] = np.arange(len(r))
    return packed[:, gpu(where.reshape(-1))]  # naux x n*n


def jk(B, C):
    """J and K of the factor C (orbitals as rows) over the fitted B."""
    n, naux = C.shape[1], B.shape[0]
    D = C.T @ C
    J = (B.T @ (B @ D.reshape(-1))).reshape(n, n)
    X = (B.reshape(naux * n, n) @ C.T.contiguous()).reshape(naux, n, -1).permute(1, 0, 2).reshape(n, -1)
    return J, X @ X.T


def exact(case, seed):
    kind = case["kind"]
    mols = [molecule(*key) for key in systems(case)]
    if kind == "ragged":
        out = []
        for k, m in enumerate(mols):
            B = fitted(m)
            out += [jk(B, gpu(f)) for f in pair_factors(m, seed + 1000 * k)]
        return out
    m = mols[0]
    B = fitted(m)
    if kind == "pair":
        return [jk(B, gpu(f)) for f in pair_factors(m, seed)]
    if kind == "active":
        o, a, n = m["nocc"], min(case["active"], m["nbf"]), m["nbf"]
        lo = max(0, o - a // 2)
        C = gpu(rotated(m, seed)[lo:lo + a])
        half = (B.reshape(-1, n) @ C.T.contiguous()).reshape(-1, n, a)  # Q, m, a2
        R = torch.matmul(C, half).transpose(1, 2).reshape(-1, a * a)  # Q, a2, a1
        return (R.T @ R).reshape(a, a, a, a).cpu().numpy()
    C = gpu(rotated(m, seed)[:m["nocc"]])
    J, K = jk(B, C)
    if kind == "gradient":
        H = gpu(m["H"])
        F = H + 2.0 * J - K
        return ((C.T @ C) * (H + F)).sum(), 4.0 * C @ F
    return J, K
