"""Workloads that stand for the framework's use: searches and searches with gradients.

Every case is one public call (or one step of the persistent or Verlet
objects) on device tensors, in the sizes of the repository's benchmark
configurations and around them.  The order of a list's pairs is unspecified
for periodic structures, so those cases return what a program makes of the
list through the call's own autograd: the gradients of a pair energy with
respect to positions (forces) and cell (virial), to which every pair's i, j,
S and D contributes.  Lists of molecules come by source and target and are
returned whole.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

from tonari_amd import neighbor_list
from tonari_amd.persistent import NeighborListPlan
from tonari_amd.pyg import neighbor_graph
from tonari_amd.verlet import VerletList

DTYPES = {"f32": torch.float32, "f64": torch.float64}
REST = 1.5  # rest length of the harmonic pair energy 0.5 (d - REST)^2
SKIN = 1.0  # Verlet skin


def listed():
    return [
        # one small molecule: an interactive call or a geometry optimisation's step, all latency
        {"name": "molecule", "kind": "molecules", "dtype": "f32", "structures": 1, "lo": 24, "hi": 24,
         "cutoff": 5.0, "quantities": "ijD", "half": False, "sorted": False, "batched": False},
        # one small crystal with forces and virial: a relaxation's step, all latency
        {"name": "crystal", "kind": "crystals", "dtype": "f32", "structures": 1, "lo": 16, "hi": 16,
         "cutoff": 6.0, "quantities": "ijSD", "algorithm": "auto", "api": "list", "packing": "solid",
         "batched": False},
        # the 512-atom float64 box of the benchmark's first configuration, by explicit brute force
        {"name": "box_brute", "kind": "box", "dtype": "f64", "atoms": 512, "density": 0.064,
         "cutoff": 5.0, "quantities": "ijSdD", "algorithm": "brute_force", "half": False},
        # a training batch of crystals under 'auto' (brute-force and cell-list structures mixed),
        # through the graph adapter, with forces and stress
        {"name": "crystals_graph", "kind": "crystals", "dtype": "f32", "structures": 32, "lo": 2,
         "hi": 200, "cutoff": 5.0, "quantities": "Dd", "algorithm": "auto", "api": "graph",
         "packing": "solid", "batched": True},
        # the benchmark's batch of 256 small triclinic crystals (many images), brute force
        {"name": "crystals", "kind": "crystals", "dtype": "f32", "structures": 256, "lo": 2, "hi": 64,
         "cutoff": 6.0, "quantities": "PSD", "algorithm": "brute_force", "api": "list",
         "packing": "loose", "batched": True},
        # the same kind of batch as one molecular-dynamics step on a Verlet list
        {"name": "crystals_verlet", "kind": "crystals", "dtype": "f32", "structures": 128, "lo": 2,
         "hi": 64, "cutoff": 6.0, "quantities": "PSD", "algorithm": "auto", "api": "verlet",
         "packing": "loose", "batched": True},
        # the benchmark's batch of 1,024 molecules: half list, sorted, forward only
        {"name": "molecules", "kind": "molecules", "dtype": "f32", "structures": 1024, "lo": 20,
         "hi": 120, "cutoff": 5.0, "quantities": "ijd", "half": True, "sorted": True, "batched": True},
        # a dynamics step of 128 molecules on the persistent plan (no allocation, no count wait)
        {"name": "molecules_plan", "kind": "plan", "dtype": "f32", "structures": 128, "lo": 20,
         "hi": 120, "cutoff": 5.0, "quantities": "ijD"},
        # clusters of 500 to 2,000 atoms in float64: the largest molecules searched without a grid
        {"name": "clusters", "kind": "clusters", "dtype": "f64", "structures": 48, "lo": 500,
         "hi": 2000, "cutoff": 6.0, "quantities": "ijSd", "sorted": True},
        # a liquid-sized float64 half list through the cell list: energies in d, forces
        {"name": "box_half", "kind": "box", "dtype": "f64", "atoms": 20000, "density": 0.1,
         "cutoff": 6.0, "quantities": "ijSd", "algorithm": "auto", "half": True},
        # the benchmark's flagship: 100,000 atoms, float32, cell list, 'PD', here with its forces
        {"name": "box", "kind": "box", "dtype": "f32", "atoms": 100000, "density": 0.1,
         "cutoff": 6.0, "quantities": "PD", "algorithm": "cell_list", "half": False},
        # mixed slabs of the benchmark's last configuration: float64, skewed cells, vacuum, self
        # pairs, sorted; the largest outputs
        {"name": "slabs", "kind": "slabs", "dtype": "f64", "structures": 16, "lo": 2000, "hi": 20000,
         "cutoff": 8.0, "quantities": "ijSdD"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["molecules", "crystals", "crystals", "box", "box", "slabs", "clusters", "plan"])
    dtype = rng.choice(["f32", "f32", "f64"])
    cutoff = round(rng.uniform(4.0, 6.5), 2)
    if kind in ("molecules", "plan"):
        lo = rng.randint(5, 60)
        case = {"kind": kind, "dtype": dtype, "structures": _log_int(rng, 1, 1024), "lo": lo,
                "hi": rng.randint(lo, 130), "cutoff": cutoff,
                "quantities": rng.choice(["ijd", "ijD", "ijSD", "PSd"])}
        if kind == "molecules":
            case.update(half=rng.random() < 0.5, sorted=rng.random() < 0.5, batched=True)
        return case
    if kind == "clusters":
        lo = _log_int(rng, 130, 1200)
        return {"kind": kind, "dtype": dtype, "structures": _log_int(rng, 1, 48), "lo": lo,
                "hi": rng.randint(lo, 2000), "cutoff": cutoff, "quantities": rng.choice(["ijSd", "ijD"]),
                "sorted": rng.random() < 0.5}
    if kind == "crystals":
        lo = rng.randint(1, 20)
        packing = rng.choice(["solid", "loose"])
        return {"kind": kind, "dtype": dtype, "structures": _log_int(rng, 1, 256), "lo": lo,
                "hi": rng.randint(lo + 1, 200 if packing == "solid" else 64), "cutoff": cutoff,
                "quantities": rng.choice(["PSD", "ijSD", "Dd", "ijSd"]),
                "algorithm": rng.choice(["auto", "auto", "brute_force"]) if packing == "loose" else "auto",
                "api": rng.choice(["list", "list", "graph", "verlet"]), "packing": packing,
                "batched": True}
    if kind == "box":
        return {"kind": kind, "dtype": dtype, "atoms": _log_int(rng, 600, 100000),
                "density": round(rng.uniform(0.05, 0.11), 3), "cutoff": round(rng.uniform(4.0, 6.0), 2),
                "quantities": rng.choice(["PD", "ijD", "ijSd", "ijSdD"]),
                "algorithm": rng.choice(["auto", "cell_list"]), "half": rng.random() < 0.4}
    lo = _log_int(rng, 300, 4000)
    return {"kind": kind, "dtype": dtype, "structures": rng.randint(1, 12), "lo": lo,
            "hi": lo * rng.randint(1, 4), "cutoff": round(rng.uniform(5.0, 8.0), 2),
            "quantities": rng.choice(["ijSdD", "ijSd"])}


# ------------------------------------------------------------------ inputs


def _sizes(case):
    """Atoms of each structure, fixed by the case so that its outputs keep one shape; the seed gives their order."""
    rng = np.random.Generator(np.random.PCG64(case["structures"]))
    n, lo, hi = case["structures"], case["lo"], case["hi"]
    if case["kind"] in ("slabs", "clusters"):
        # one size of each of n equal shares of the logarithm
        u = (np.arange(n) + rng.uniform(0.0, 1.0, n)) / n
        return np.rint(np.exp(np.log(lo) + u * (np.log(hi) - np.log(lo)))).astype(np.int64)
    return rng.integers(lo, hi + 1, n)


def _gaussian_molecules(sizes, rng, sigma=3.0, dmin=1.0):
    """Gaussian clouds whose atoms keep a least distance: an atom too near to an earlier one is drawn again."""
    n, width = len(sizes), int(max(sizes))
    gen = torch.Generator(device="cuda").manual_seed(int(rng.integers(1 << 62)))
    x = torch.randn(n, width, 3, generator=gen, device="cuda", dtype=torch.float64) * sigma
    live = torch.arange(width, device="cuda")[None, :] < torch.as_tensor(sizes, device="cuda")[:, None]
    earlier = torch.ones(width, width, dtype=torch.bool, device="cuda").tril(-1)
    for _ in range(1000):
        step = max(1, 20_000_000 // (width * width))
        near = torch.cat([((torch.cdist(p, p) < dmin) & earlier).any(2) for p in x.split(step)]) & live
        if not bool(near.any()):
            break
        new = torch.randn(n, width, 3, generator=gen, device="cuda", dtype=torch.float64) * sigma
        x = torch.where(near[..., None], new, x)
    return x[live].cpu().numpy()


def _isolated(case):
    """(positions of each structure, each atom's move to a later step): fixed by the case, since their
    lists are returned whole and the number of pairs must not change."""
    rng = np.random.Generator(np.random.PCG64(case["structures"] + 1))
    sizes = _sizes(case)
    if case["kind"] == "clusters":
        pos = [_ball(int(n), rng) for n in sizes]
    else:
        pos = np.split(_gaussian_molecules(sizes, rng), np.cumsum(sizes)[:-1])
    return pos, [rng.uniform(-0.1, 0.1, p.shape) for p in pos]


def _ball(n, rng, spacing=2.2, jitter=0.25):
    """The n sites of a cubic lattice nearest to its middle, each moved a little."""
    m = int(math.ceil((n * 3 / (4 * math.pi)) ** (1 / 3))) + 1
    g = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = g[np.argsort((g * g).sum(1), kind="stable")[:n]]
    return g * spacing + rng.normal(0.0, jitter, (n, 3))


def _cell(lengths, angles):
    (a, b, c), (al, be, ga) = lengths, np.radians(angles)
    cx, cy = math.cos(be), (math.cos(al) - math.cos(be) * math.cos(ga)) / math.sin(ga)
    return np.array([[a, 0, 0], [b * math.cos(ga), b * math.sin(ga), 0],
                     [c * cx, c * cy, c * math.sqrt(1 - cx * cx - cy * cy)]])


def _angles(rng, lo, hi):
    while True:
        al, be, ga = angles = rng.uniform(lo, hi, 3)
        x, y, z = np.cos(np.radians(angles))
        if 1 - x * x - y * y - z * z + 2 * x * y * z > 1e-3:
            return angles


def _structures(case, rng):
    """(positions in float64, their move to a later step, cells, pbc, sizes) of a case."""
    kind = case["kind"]
    if kind == "box":
        n = case["atoms"]
        edge = (n / case["density"]) ** (1 / 3)
        return (rng.uniform(0.0, edge, (n, 3)), np.zeros((n, 3)), np.eye(3)[None] * edge,
                np.ones((1, 3), bool), np.array([n]))
    if kind in ("molecules", "plan", "clusters"):
        # the seed gives the order of the structures and of the atoms in each, and mirrors the axes
        pos, moves = [], []
        base, step = _isolated(case)
        for b in rng.permutation(len(base)):
            order, mirror = rng.permutation(len(base[b])), rng.choice([-1.0, 1.0], 3)
            pos.append(base[b][order] * mirror)
            moves.append(step[b][order] * mirror)
        sizes = np.array([len(p) for p in pos])
        return (np.concatenate(pos), np.concatenate(moves), np.zeros((len(sizes), 3, 3)),
                np.zeros((len(sizes), 3), bool), sizes)
    sizes = rng.permutation(_sizes(case))
    pos, cells = [], []
    for n in sizes:
        f = rng.uniform(0.0, 1.0, (n, 3))
        if kind == "slabs":
            a, b, slab = rng.uniform(30.0, 60.0, 3)
            cell = _cell((a, b, slab + 20.0), _angles(rng, 70.0, 110.0))
            f[:, 2] *= slab / (slab + 20.0)
        elif case["packing"] == "solid":
            # about 16 cubic angstroms per atom
            cell = _cell(rng.uniform(0.7, 1.4, 3), _angles(rng, 75.0, 105.0))
            cell *= (16.0 * n / abs(np.linalg.det(cell))) ** (1 / 3)
        else:
            cell = _cell(rng.uniform(3.0, 12.0, 3), _angles(rng, 60.0, 120.0))
        pos.append(f @ cell)
        cells.append(cell)
    pbc = np.tile([True, True, kind != "slabs"], (len(sizes), 1))
    moves = rng.uniform(-0.1, 0.1, (int(sizes.sum()), 3))
    return np.concatenate(pos), moves, np.stack(cells), pbc, sizes


def _inputs(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    pos, moves, cells, pbc, sizes = _structures(case, rng)
    dtype = DTYPES[case["dtype"]]
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    t = {"pos": torch.as_tensor(pos).to("cuda", dtype).contiguous(),
         "cell": torch.as_tensor(cells).to("cuda", dtype).contiguous(),
         "pbc": torch.as_tensor(pbc).to("cuda"), "ptr": torch.as_tensor(ptr).to("cuda")}
    if _api(case) in ("verlet", "plan"):
        # the positions of a later step, moved by far less than half the skin
        t["next"] = torch.as_tensor(pos + moves).to("cuda", dtype).contiguous()
    return t


def _api(case):
    return "plan" if case["kind"] == "plan" else case.get("api", "list")


def _with_gradients(case):
    return case["kind"] in ("crystals", "box", "slabs")


def prepare(case, seed):
    t = _inputs(case, seed)
    pos, cell, pbc, ptr = t["pos"], t["cell"], t["pbc"], t["ptr"]
    state = {"case": case, "pos": pos, "cell": cell, "pbc": pbc, "ptr": ptr}
    if _api(case) == "verlet":
        state["list"] = VerletList(case["quantities"], case["cutoff"], SKIN,
                                   algorithm=case["algorithm"], mode="filter")
        state["list"](pos, cell, pbc, ptr)
        state["pos"] = t["next"]
    elif _api(case) == "plan":
        pairs, = neighbor_list("P", pos, cell, pbc, case["cutoff"], ptr)
        state["plan"] = NeighborListPlan(case["quantities"], pos, cell, pbc, case["cutoff"], ptr,
                                         capacity=int(1.25 * pairs.shape[0]) + 1024)
        state["next"] = t["next"]
    if not case.get("batched", True):
        state.update(cell=cell[0].contiguous(), pbc=pbc[0].contiguous(), ptr=None)
    if _with_gradients(case):
        state["pos"].requires_grad_(True)
        state["cell"].requires_grad_(True)
    return state


# -------------------------------------------------------------------- runs


def _forces(case, by, pos, cell):
    """Gradients of 0.5 sum (d - REST)^2 where the call gives d, else of 0.5 sum |D|^2."""
    if by.get("d") is not None:
        d = by["d"]
        return torch.autograd.grad(d, (pos, cell), d.detach() - REST)
    D = by["D"]
    return torch.autograd.grad(D, (pos, cell), D.detach())


def run(state):
    case = state["case"]
    pos, cell, pbc, ptr, q = state["pos"], state["cell"], state["pbc"], state["ptr"], case["quantities"]
    if _api(case) == "plan":
        plan = state["plan"]
        plan.positions.copy_(state["next"])
        plan.run()
        n = plan.check()
        return [x[:n] for x in plan.outputs]
    if _api(case) == "verlet":
        out = state["list"](pos, cell, pbc, ptr)
    elif _api(case) == "graph":
        g = neighbor_graph(pos, cell, pbc, case["cutoff"], ptr, vectors="D" in q, lengths="d" in q,
                           shifts="S" in q, algorithm=case["algorithm"])
        by = {"D": g.edge_vectors, "d": g.edge_lengths}
        return {"pairs": g.edge_index.shape[1], "grads": _forces(case, by, pos, cell)}
    else:
        out = neighbor_list(q, pos, cell, pbc, case["cutoff"], ptr,
                            algorithm=case.get("algorithm", "auto"),
                            sorted=case.get("sorted", False) or case["kind"] == "slabs",
                            half_list=case.get("half", False),
                            include_self=case["kind"] == "slabs")
    if not _with_gradients(case):
        return list(out)
    by = dict(zip(q, out))
    return {"pairs": out[0].shape[0], "grads": _forces(case, by, pos, cell)}


# ------------------------------------------------------- work and tolerance


def _expected(case):
    """(atoms, pairs) of a case, about: the mean over inputs."""
    rng = np.random.Generator(np.random.PCG64(0))
    kind, rc = case["kind"], case["cutoff"]
    sphere = 4 / 3 * math.pi * rc**3
    half = 0.5 if case.get("half") else 1.0
    if kind == "box":
        return case["atoms"], half * case["atoms"] * case["density"] * sphere
    n = _sizes(case).astype(np.float64)
    rounds = max(1, 2000 // case["structures"])
    pairs = 0.0
    for _ in range(rounds):
        if kind in ("molecules", "plan"):
            x = rc / (3.0 * math.sqrt(2.0))  # distances of two atoms of a Gaussian cloud
            share = math.erf(x / math.sqrt(2)) - math.sqrt(2 / math.pi) * x * math.exp(-x * x / 2)
            pairs += half * share * (n * (n - 1)).sum() / rounds
        elif kind == "clusters":
            r = 2.2 * (3 * n / (4 * math.pi)) ** (1 / 3)  # radius of the ball
            u = np.minimum(rc / (2 * r), 1.0)
            pairs += (n * n * (8 * u**3 - 9 * u**4 + 2 * u**6)).sum() / rounds
        elif kind == "slabs":
            a, b, c = rng.uniform(30.0, 60.0, (3, len(n)))
            v = a * b * c * 0.93  # mean volume factor of the angles
            pairs += (n * (1 + n / v * sphere * (1 - 3 * rc / (8 * c)))).sum() / rounds
        elif case["packing"] == "solid":
            pairs += (n * sphere / 16.0).sum() / rounds
        else:
            v = np.prod(rng.uniform(3.0, 12.0, (3, len(n))), 0) * 0.82
            pairs += (n * n / v * sphere).sum() / rounds
    return n.sum(), pairs


def work(case):
    atoms, pairs = _expected(case)
    s = 4 if case["dtype"] == "f32" else 8
    width = {"i": 8, "j": 8, "P": 16, "S": 12, "d": s, "D": 3 * s}
    row = sum(width[c] for c in case["quantities"]) + (16 if _api(case) == "graph" else 0)
    nbytes = atoms * 3 * s + pairs * row
    flops = 8.0 * pairs
    if _with_gradients(case):
        # the gradient reads every pair's i, j, S and upstream gradient (and D and d for that
        # of d) and writes the forces
        nbytes += pairs * (28 + (5 * s if "d" in case["quantities"] else 3 * s)) + atoms * 3 * s
        flops += 24.0 * pairs
    if _api(case) == "verlet":
        nbytes += 8.0 * pairs * ((case["cutoff"] + SKIN) / case["cutoff"]) ** 3
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # measured: repeats of one case (float atomics in another order) differ by up to 2.8e-7 in
    # float32 and 8e-16 in float64, and are up to 5e-7 and 1.3e-15 from float64 and exact sums
    # of the same pairs; single entries by 1.4e-6 and 3e-15 of the root mean square
    eps = 2.0**-23 if case["dtype"] == "f32" else 2.0**-52
    if _with_gradients(case):
        return {"rel": 20 * eps, "max": 100 * eps}
    return {"rel": 2 * eps, "max": 8 * eps}


# ------------------------------------------------------------------- exact


def _gradients64(case, t, pos64, cell64):
    """Gradients in float64 of every pair that the public predicate keeps in the working precision:
    D = ((p_j - p_i) + S0 c0) + S1 c1) + S2 c2, |D|^2 < cutoff^2, rounded after every operation.
    Each structure's images are laid out, sorted along x, and compared with chunks of sources."""
    rc, dtype = case["cutoff"], t["pos"].dtype
    cut2 = torch.tensor(rc * rc, dtype=torch.float64).to(dtype).item()
    by_d = "d" in case["quantities"]
    half, own = case.get("half", False), case["kind"] == "slabs"
    gp, gc = torch.zeros_like(pos64), torch.zeros_like(cell64)
    pairs = 0
    ptr, cells, pbc = t["ptr"].tolist(), cell64.cpu().numpy(), t["pbc"].cpu().numpy()
    start = t.get("next", t["pos"])
    for b in range(len(ptr) - 1):
        lo, hi = ptr[b], ptr[b + 1]
        if hi == lo:
            continue
        p, p64 = start[lo:hi], pos64[lo:hi]
        c, c64 = t["cell"][b], cell64[b]
        reach = np.where(pbc[b], np.floor(1.2 + (rc + 0.1) * np.linalg.norm(np.linalg.inv(cells[b]), axis=0)), 0)
        axes = [torch.arange(-int(r), int(r) + 1, device="cuda") for r in reach]
        shifts = torch.cartesian_prod(*axes)
        low, high = p64.min(0).values - rc - 0.01, p64.max(0).values + rc + 0.01
        found = []
        for S in shifts.split(max(1, 20_000_000 // (hi - lo))):
            x = p64[None] + (S.double() @ c64)[:, None]
            s, j = torch.nonzero(((x > low) & (x < high)).all(2), as_tuple=True)
            found.append((x[s, j, 0], S[s], j))
        x = torch.cat([f[0] for f in found])
        order = torch.argsort(x)
        x, S, j = x[order], torch.cat([f[1] for f in found])[order], torch.cat([f[2] for f in found])[order]
        Sd = S.to(dtype)
        by_x = torch.argsort(p64[:, 0])
        xs = p64[by_x, 0]
        chunk = max(16, min(1024, 8_000_000 // max(1, len(x))))
        for k in range(0, hi - lo, chunk):
            src = by_x[k:k + chunk]
            edge = torch.stack([xs[k] - rc - 0.01, xs[min(k + chunk, hi - lo) - 1] + rc + 0.01])
            u, v = torch.searchsorted(x, edge).tolist()
            jj, SS, SSd = j[u:v], S[u:v], Sd[u:v]
            d2 = None
            for a in range(3):
                D = p[jj, a][None] - p[src, a][:, None]
                for r in range(3):
                    D = D + (SSd[:, r] * c[r, a])[None]
                d2 = D * D if d2 is None else d2 + D * D
            keep = d2 < cut2
            zero = (SS == 0).all(1)[None]
            same = src[:, None] == jj[None]
            if half:
                neg = (SS[:, 0] < 0) | ((SS[:, 0] == 0) & ((SS[:, 1] < 0) | ((SS[:, 1] == 0) & (SS[:, 2] < 0))))
                keep &= (src[:, None] < jj[None]) | (same & neg[None])
            if not own:
                keep &= ~(same & zero)
            m, n = torch.nonzero(keep, as_tuple=True)
            i, jn, Sn = src[m], jj[n], SS[n].double()
            D = p64[jn] - p64[i] + Sn @ c64
            g = D
            if by_d:
                d = torch.linalg.vector_norm(D, dim=1)
                g = torch.where(d > 0, (d - REST) / d, torch.zeros_like(d))[:, None] * D
            gp[lo:hi].index_add_(0, jn, g)
            gp[lo:hi].index_add_(0, i, -g)
            gc[b] += Sn.T @ g
            pairs += len(i)
    return gp, gc, pairs


def exact(case, seed):
    t = _inputs(case, seed)
    start = t.get("next", t["pos"])
    pos64, cell64 = start.double(), t["cell"].double()
    if _with_gradients(case):
        gp, gc, pairs = _gradients64(case, t, pos64, cell64)
        return {"pairs": pairs, "grads": (gp, gc if case.get("batched", True) else gc[0])}
    # molecules: by source, then target; d2 = (dx dx + dy dy) + dz dz in the working precision decides
    cut2 = torch.tensor(case["cutoff"] ** 2, dtype=torch.float64).to(start.dtype).item()
    ptr = t["ptr"].tolist()
    rows = {c: [] for c in case["quantities"]}
    for lo, hi in zip(ptr[:-1], ptr[1:]):
        p = start[lo:hi]
        D = p[None] - p[:, None]
        keep = (D[..., 0] * D[..., 0] + D[..., 1] * D[..., 1]) + D[..., 2] * D[..., 2] < cut2
        keep &= ~torch.eye(hi - lo, dtype=torch.bool, device="cuda")
        if case.get("half"):
            keep = keep.triu(1)
        i, j = torch.nonzero(keep, as_tuple=True)
        D64 = pos64[lo + j] - pos64[lo + i]
        made = {"i": lo + i, "j": lo + j, "P": torch.stack([lo + i, lo + j], 1),
                "S": torch.zeros(len(i), 3, dtype=torch.int32, device="cuda"), "D": D64,
                "d": torch.linalg.vector_norm(D64, dim=1)}
        for c in rows:
            rows[c].append(made[c])
    return [torch.cat(rows[c]) for c in case["quantities"]]
