"""Performance cases: the calls that a docking program makes, over the sizes
it makes them at.

Kinds (one pass is one or more public calls with host arrays in and out):
  search      one ligand against a resident protein: conformers x rotations
  batch       several uneven ligands in one Batch
  serve       concurrent requests on two resident proteins through a Server
  rescore     FP64 grid score of retained poses, with the gradient
  refine      rigid-body descent of retained poses
  conformers  random-torsion conformers of a chain ligand
  build       potential grids and spectra from the protein's atoms

Proteins, ligands and poses are synthetic: uniform protein atoms with capped
soft-core Lennard-Jones and Coulomb grids, self-avoiding chain ligands with
perturbed torsions, uniform rotations.  Everything is made from the seed with
numpy and torch.
"""
import math

import numpy as np
import torch

import cdocker_amd as cdk

PROBES = np.array([1.2, 1.5, 1.7, 1.8, 1.9, 2.0, 2.1, 2.2], np.float32)
# grid edge: (protein atoms, box in A, spacing in A)
PROTEINS = {32: (900, 16.0, 0.5), 48: (2000, 24.0, 0.5), 64: (3000, 32.0, 0.5), 96: (8000, 48.0, 0.5),
            128: (8000, 48.0, 0.375)}
LJ_CUT, EL_CUT, LJ_CAP, EL_CAP = 8.0, 12.0, 3.0, 20.0


def listed():
    return [
        # ordinary screening call: a drug-sized ligand, a few conformers x 2000 rotations
        {"name": "search64", "kind": "search", "n": 64, "natom": 40, "nconf": 5, "nquat": 2000, "shared": False},
        # one batch of 50 rotations of one conformer: the smallest call a driver makes
        {"name": "search64_one_batch", "kind": "search", "n": 64, "natom": 24, "nconf": 1, "nquat": 50,
         "shared": False},
        # larger ligand, odd counts, one rotation set shared by the conformers
        {"name": "search64_ragged", "kind": "search", "n": 64, "natom": 57, "nconf": 7, "nquat": 333, "shared": True},
        # the small grid: 24-atom ligand, 500 rotations
        {"name": "search48", "kind": "search", "n": 48, "natom": 24, "nconf": 1, "nquat": 500, "shared": False},
        # large binding sites
        {"name": "search96", "kind": "search", "n": 96, "natom": 40, "nconf": 2, "nquat": 1000, "shared": False},
        {"name": "search128", "kind": "search", "n": 128, "natom": 50, "nconf": 1, "nquat": 1000, "shared": False},
        # virtual screening: uneven ligands sharing launches
        {"name": "batch64", "kind": "batch", "n": 64, "nlig": 16, "nquat": 100},
        # a server holding a 64^3 and a 96^3 protein, requests of both in flight
        {"name": "serve", "kind": "serve", "nreq": 6, "nquat": 250},
        # the poses a search retained, rescored and refined
        {"name": "rescore", "kind": "rescore", "n": 64, "natom": 40, "npose": 1000},
        {"name": "refine", "kind": "refine", "n": 64, "natom": 40, "npose": 1000, "steps": 50},
        # conformer generation ahead of a search: the first 200 that pass
        {"name": "conformers", "kind": "conformers", "natom": 40, "ntrial": 20000, "keep": 200},
        # a new protein: grids and spectra from its atoms
        {"name": "build64", "kind": "build", "n": 64, "natom": 3000},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search"] * 6 + ["batch", "serve", "rescore", "refine", "conformers", "build"])
    if kind == "search":
        n = rng.choice([32, 48, 64, 64, 96, 128])
        natom = rng.randint(8, 40) if n == 32 else rng.randint(12, 80)
        most = {32: 16000, 48: 12000, 64: 9000, 96: 1900, 128: 950}[n] * 40 // max(natom, 40)
        nconf = rng.randint(1, 12)
        return {"kind": kind, "n": n, "natom": natom, "nconf": nconf,
                "nquat": max(20, _logint(rng, 30, most) // nconf), "shared": rng.random() < 0.25}
    if kind == "batch":
        return {"kind": kind, "n": rng.choice([48, 64]), "nlig": rng.randint(2, 16), "nquat": _logint(rng, 20, 100)}
    if kind == "serve":
        return {"kind": kind, "nreq": rng.randint(2, 6), "nquat": _logint(rng, 50, 250)}
    if kind in ("rescore", "refine"):
        c = {"kind": kind, "n": rng.choice([48, 64, 96]), "natom": rng.randint(12, 80), "npose": _logint(rng, 10, 1500)}
        if kind == "refine":
            c["steps"] = rng.randint(20, 100)
        return c
    if kind == "conformers":
        c = {"kind": kind, "natom": rng.randint(12, 48), "ntrial": _logint(rng, 2000, 16000)}
        return dict(c, keep=c["ntrial"] // 100)
    return {"kind": kind, "n": rng.choice([32, 48, 64]), "natom": _logint(rng, 500, 3000)}


# ---- inputs ----------------------------------------------------------------
def _protein_atoms(rs, natom, box):
    return dict(xyz=rs.uniform(0.0, box, (natom, 3)), charge=0.3 * rs.standard_normal(natom),
                epsilon=rs.uniform(0.05, 0.25, natom), radius=rs.choice(PROBES, natom).astype(np.float64))


def _grid_axis(box, n, h):
    return np.float64(np.float32(box / 2) - np.float32((n - 1) * h) / np.float32(2)) + np.arange(n) * h


def _potential_grids(p, n, h, box):
    """[9][n][n][n] float64: the probes' Lennard-Jones grids, then Coulomb."""
    dev = "cuda"
    t = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=dev)  # noqa: E731
    ax = t(_grid_axis(box, n, h))
    xyz, q = t(p["xyz"]), t(p["charge"])
    R6 = (t(p["radius"])[:, None] + t(PROBES.astype(np.float64))[None]) ** 6
    se = torch.sqrt(t(p["epsilon"]))[:, None]
    w12, w6 = se * R6 * R6, -2.0 * se * R6
    out = torch.empty((9, n * n * n), dtype=torch.float64, device=dev)
    # one (i, j) column block of grid points at a time
    pts = torch.stack(torch.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
    step = max(1, (1 << 27) // max(len(q), 1))
    for a in range(0, len(pts), step):
        x = pts[a:a + step]
        d2 = (x[:, 0:1] - xyz[None, :, 0]) ** 2
        d2 += (x[:, 1:2] - xyz[None, :, 1]) ** 2
        d2 += (x[:, 2:3] - xyz[None, :, 2]) ** 2
        inv = 1.0 / torch.clamp_min(d2, 1e-4)
        inv[d2 > EL_CUT * EL_CUT] = 0.0
        el = (inv @ q) * (332.0636 / 4.0)
        out[8, a:a + step] = torch.clamp(el, -EL_CAP, EL_CAP)
        inv[d2 > LJ_CUT * LJ_CUT] = 0.0
        inv = inv * inv * inv
        lj = inv @ w6
        inv *= inv
        lj += inv @ w12
        out[:8, a:a + step] = torch.clamp_max(lj, LJ_CAP).T
    return out.reshape(9, n, n, n)


def _frame(n):
    natom, box, h = PROTEINS[n]
    mid = np.full(3, box / 2, np.float32)
    length = np.full(3, (n - 1) * h, np.float32)
    return natom, box, h, mid, length


def _grid_values(n, seed):
    natom, box, h, _, _ = _frame(n)
    p = _protein_atoms(np.random.default_rng([seed, 1, n]), natom, box)
    return _potential_grids(p, n, h, box).float().cpu().numpy()


def _chain(rs, natom):
    """Self-avoiding chain, 1.5 A bonds, 1.2 A between non-bonded atoms."""
    x = np.zeros((natom, 3))
    for i in range(1, natom):
        for _ in range(10000):
            v = rs.standard_normal(3)
            c = x[i - 1] + 1.5 * v / np.linalg.norm(v)
            if i < 2 or ((x[:i - 1] - c) ** 2).sum(1).min() >= 1.44:
                break
        x[i] = c
    return x - x.mean(0)


def _conformers(rs, x, nconf):
    """Conformer 0 is the chain; the others twist every bond by N(0, 0.6)."""
    out = np.repeat(x[None], nconf, 0)
    for b in range(1, len(x) - 2):
        u = out[:, b + 1] - out[:, b]
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        t = 0.6 * rs.standard_normal(nconf)
        t[0] = 0.0
        v = out[:, b + 2:] - out[:, b + 1:b + 2]
        c, s, uu = np.cos(t)[:, None, None], np.sin(t)[:, None, None], u[:, None, :]
        out[:, b + 2:] = (out[:, b + 1:b + 2] + v * c + np.cross(np.broadcast_to(uu, v.shape), v) * s
                          + uu * (v * uu).sum(-1, keepdims=True) * (1 - c))
    return (out - out.mean(1, keepdims=True)).astype(np.float32)


def _ligand(rs, natom, nconf):
    q = 0.25 * rs.standard_normal(natom)
    return dict(charge=(q - q.mean()).astype(np.float32), epsilon=rs.uniform(0.05, 0.20, natom).astype(np.float32),
                radius=rs.choice(PROBES, natom).astype(np.float32), conformers=_conformers(rs, _chain(rs, natom), nconf))


def _quats(rs, *shape):
    q = rs.standard_normal(shape + (4,))
    return (q / np.linalg.norm(q, axis=-1, keepdims=True)).astype(np.float32)


def _jobs(case, seed):
    """The searches of a case: ligand, conformers, rotations, grid edge."""
    rs = np.random.default_rng([seed, 2])
    size = np.random.default_rng(sum(v for v in case.values() if isinstance(v, int)))  # sizes from the case alone
    if case["kind"] == "search":
        lig = _ligand(rs, case["natom"], case["nconf"])
        q = _quats(rs, case["nquat"]) if case["shared"] else _quats(rs, case["nconf"], case["nquat"])
        return [dict(lig, quats=q, n=case["n"])]
    jobs = []
    for i in range(case["nlig"] if case["kind"] == "batch" else case["nreq"]):
        if case["kind"] == "batch":
            n, natom, nconf = case["n"], int(size.integers(15, 61)), int(size.integers(1, 7))
        else:
            n, natom, nconf = (64, 96)[i % 2], int(size.integers(15, 81)), int(size.integers(1, 5))
        jobs.append(dict(_ligand(rs, natom, nconf), quats=_quats(rs, nconf, case["nquat"]), n=n))
    return jobs


def _poses(case, seed):
    """(ligand, poses [npose][natom][3]): rigid placements in the grid box."""
    rs = np.random.default_rng([seed, 3])
    lig = _ligand(rs, case["natom"], 1)
    x = lig["conformers"][0].astype(np.float64)
    q = _quats(rs, case["npose"]).astype(np.float64)
    w, v = q[:, None, :1], np.broadcast_to(q[:, None, 1:], (len(q),) + x.shape)
    r = np.broadcast_to(x, v.shape)
    c = np.cross(v, r) + w * r
    r = r + 2.0 * np.cross(v, c)
    _, box, h, _, _ = _frame(case["n"])
    ax = _grid_axis(box, case["n"], h)
    lo, hi = ax[0] - r.min(1), ax[-1] - r.max(1)
    return lig, r + (lo + rs.uniform(0.05, 0.95, lo.shape) * (hi - lo))[:, None, :]


def _chain_rotors(natom):
    b = np.arange(1, max(natom - 2, 1))
    rot = np.stack([b - 1, b, b + 1, b + 2], 1).astype(np.int32)
    moving = (np.arange(natom)[None] >= rot[:, 3:4]).astype(np.uint8)
    sep = np.abs(np.arange(natom)[:, None] - np.arange(natom)[None])
    return rot, moving, (sep <= 3).astype(np.uint8)


_CTX = None


def _context():
    """The program's one device context."""
    global _CTX
    if _CTX is None:
        _CTX = cdk.Context(0)
    return _CTX


def _protein(n, seed):
    _, _, h, mid, length = _frame(n)
    return cdk.Protein(_context(), _grid_values(n, seed), PROBES, h, mid, length)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "ctx": _context()}
    if kind in ("search", "batch"):
        s["protein"] = _protein(case["n"], seed)
        s["jobs"] = [(cdk.Ligand(s["protein"], j["charge"], j["epsilon"], j["radius"]), j["conformers"], j["quats"])
                     for j in _jobs(case, seed)]
    elif kind == "serve":
        s["proteins"] = [_protein(64, seed), _protein(96, seed)]
        s["server"] = cdk.Server(s["ctx"], s["proteins"], 32 << 30, 4096)
        s["jobs"] = [((64, 96).index(j["n"]), j) for j in _jobs(case, seed)]
    elif kind in ("rescore", "refine"):
        s["protein"] = _protein(case["n"], seed)
        lig, s["poses"] = _poses(case, seed)
        s["ligand"] = cdk.Ligand(s["protein"], lig["charge"], lig["epsilon"], lig["radius"])
        s["steps"] = case.get("steps", 0)
    elif kind == "conformers":
        s["coords"] = _chain(np.random.default_rng([seed, 4]), case["natom"])
        s["rotors"], s["moving"], s["exclude"] = _chain_rotors(case["natom"])
        s["ntrial"], s["keep"], s["seed"] = case["ntrial"], case["keep"], seed
    else:
        _, box, h, mid, length = _frame(case["n"])
        s["atoms"] = _protein_atoms(np.random.default_rng([seed, 5]), case["natom"], box)
        s["frame"] = (case["n"], h, mid, length)
    return s


def _found(e, idx, mc):
    return {"energy": e, "index": idx, "mincoor": mc}


def run(s):
    kind = s["kind"]
    if kind == "search":
        (lig, conf, quats), = s["jobs"]
        return _found(*cdk.search(s["ctx"], s["protein"], lig, conf, quats))
    if kind == "batch":
        b = cdk.Batch(s["ctx"], s["protein"])
        ids = [b.add(*job) for job in s["jobs"]]
        b.run()
        out = [_found(*b.results(i)) for i in ids]
        b.close()
        return out
    if kind == "serve":
        srv = s["server"]
        ids = [srv.submit(p, j["charge"], j["epsilon"], j["radius"], j["conformers"], j["quats"])
               for p, j in s["jobs"]]
        return [_found(*srv.result(i)[:3]) for i in ids]
    if kind == "rescore":
        e, g, inside = cdk.rescore_poses(s["protein"], s["ligand"], s["poses"], want_grad=True)
        return {"energy": e, "grad": g, "inside": inside}
    if kind == "refine":
        x, e = cdk.refine_poses(s["protein"], s["ligand"], s["poses"], steps=s["steps"])
        return {"poses": x, "energy": e}
    if kind == "conformers":
        x, t = cdk.generate_conformers(s["ctx"], s["coords"], s["rotors"], s["moving"], s["exclude"], s["ntrial"],
                                       s["seed"], max_keep=s["keep"])
        return {"conformers": x, "trial": t}
    a, (n, h, mid, length) = s["atoms"], s["frame"]
    p = cdk.Protein.build(s["ctx"], a["xyz"], a["charge"], a["epsilon"], a["radius"], PROBES, n, h, mid, length,
                          LJ_CUT, EL_CUT, LJ_CAP, EL_CAP)
    out = {"grids": p.grids(), "spectrum": p.spectrum(8)}
    p.close()
    return out


# ---- work ------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("search", "batch", "serve"):
        byt = flops = 0.0
        for j in _jobs(case, 1):
            n, natom = j["n"], j["conformers"].shape[1]
            poses = j["conformers"].shape[0] * j["quats"].shape[-2]
            c = len(np.unique(j["radius"])) + 1
            # per pose: a real 3-D transform per channel and one back, a
            # complex multiply-add per channel and half-spectrum point
            half = n * n * (n // 2 + 1)
            flops += poses * ((c + 1) * 2.5 * n ** 3 * 3 * math.log2(n) + 8.0 * c * half)
            # the channels' spectra once, coordinates, rotations, results
            byt += 8.0 * c * half + j["conformers"].nbytes + j["quats"].nbytes + poses * 28
        return {"bytes": byt, "flops": flops}
    if kind in ("rescore", "refine"):
        atoms = case["natom"] * case["npose"]
        evals = case.get("steps", 0) + 1
        # eight corners of two grids per atom: value and gradient
        return {"bytes": atoms * 48.0 + case["npose"] * 12.0, "flops": evals * atoms * 8 * 24.0}
    if kind == "conformers":
        na, nt = case["natom"], case["ntrial"]
        # Rodrigues rotation of the moved atoms per rotor, then the pair test
        return {"bytes": case["keep"] * na * 24.0 + na * 24.0, "flops": nt * (0.5 * na * na * 40.0 + 0.5 * na * na * 8.0)}
    n, natom = case["n"], case["natom"]
    g, (_, box, h) = float(n) ** 3, PROTEINS[n]
    near = natom * min(1.0, 4.0 / 3.0 * math.pi * LJ_CUT ** 3 / box ** 3)
    return {"bytes": natom * 48.0 + 9 * g * 4 + n * n * (n // 2 + 1) * 8.0,
            "flops": g * near * (12 + 8 * 8) + 9 * 2.5 * g * 3 * math.log2(n)}


# ---- 64-bit results --------------------------------------------------------
def _search64(job, grids):
    """Best energy per pose by FP64 transforms, and the rotated minima."""
    n, dev = job["n"], "cuda"
    h = PROTEINS[n][2]
    x = torch.as_tensor(job["conformers"].astype(np.float64), device=dev)
    nconf, natom = x.shape[:2]
    q = torch.as_tensor(job["quats"].astype(np.float64), device=dev)
    q = q.expand(nconf, *q.shape[-2:])
    nquat = q.shape[1]
    # q p conj(q): |q|^2 stays in, as the quaternion product has it
    w, v = q[..., None, :1], q[..., None, 1:]
    p = x[:, None]
    v, p = torch.broadcast_tensors(v, p)
    r = (w * w - (v * v).sum(-1, keepdim=True)) * p + 2 * (v * p).sum(-1, keepdim=True) * v \
        + 2 * w * torch.linalg.cross(v, p)
    r = r.reshape(nconf * nquat, natom, 3)
    mn = r.min(1).values
    win = n - ((r.max(1).values - mn) / h).floor().long() - 2
    u = (r - mn[:, None]) / h
    cell = u.floor()
    f, cell = u - cell, cell.long()
    ok = ((cell.max(1).values + 2 <= n) & (win > 0)).all(1)
    used = [c for c in range(8) if (job["radius"] == PROBES[c]).any()]
    wt = []
    for c in used:
        wt.append(np.where(job["radius"] == PROBES[c], np.sqrt(job["epsilon"].astype(np.float64)), 0.0))
    wt.append(job["charge"].astype(np.float64))
    wt = torch.as_tensor(np.stack(wt), device=dev)
    P = torch.fft.rfftn(grids[used + [8]].double(), dim=(1, 2, 3))
    at = torch.arange(n, device=dev)
    inf = torch.tensor(float("inf"), dtype=torch.float64, device=dev)
    best = torch.full((len(r),), float("inf"), dtype=torch.float64, device=dev)
    step = max(1, (1 << 23) // n ** 3)
    for a in range(0, len(r), step):
        b = min(step, len(r) - a)
        acc = 0
        c0 = cell[a:a + b].clamp(0, n - 2)
        base = torch.arange(b, device=dev)[:, None] * n ** 3
        for c in range(len(wt)):
            on = (wt[c] != 0).nonzero()[:, 0]
            L = torch.zeros(b * n ** 3, dtype=torch.float64, device=dev)
            for k in range(8):
                d = torch.tensor([k >> 2, k >> 1 & 1, k & 1], device=dev)
                fk = torch.where(d == 1, f[a:a + b, on], 1 - f[a:a + b, on]).prod(-1) * wt[c, on]
                ck = c0[:, on] + d
                L.index_add_(0, (base + (ck[..., 0] * n + ck[..., 1]) * n + ck[..., 2]).reshape(-1), fk.reshape(-1))
            acc = acc + torch.fft.rfftn(L.view(b, n, n, n), dim=(1, 2, 3)).conj() * P[c]
        e = torch.fft.irfftn(acc, s=(n, n, n), dim=(1, 2, 3))
        wa = win[a:a + b]
        out = (at[None, :, None, None] >= wa[:, 0, None, None, None]) \
            | (at[None, None, :, None] >= wa[:, 1, None, None, None]) \
            | (at[None, None, None, :] >= wa[:, 2, None, None, None])
        best[a:a + b] = torch.where(out, inf, e).reshape(b, -1).min(1).values
    best = torch.where(ok, best, inf)
    return _found(best.reshape(nconf, nquat).cpu().numpy(), None, mn.reshape(nconf, nquat, 3).cpu().numpy())


def _rescore64(case, seed):
    lig, r = _poses(case, seed)
    n = case["n"]
    _, box, h, _, _ = _frame(n)
    g = _grid_values(n, seed).astype(np.float64)
    u = (r - _grid_axis(box, n, h)[0]) / h
    i = np.floor(u)
    f, i = u - i, i.astype(int)
    on = ((i >= 0) & (i <= n - 2)).all(-1)
    i = np.clip(i, 0, n - 2)
    ch = np.argmin(np.abs(lig["radius"][:, None] - PROBES[None]), 1)
    wv, wq = np.sqrt(lig["epsilon"]).astype(np.float64), lig["charge"].astype(np.float64)
    e, grad = np.zeros(on.shape), np.zeros(r.shape)
    for k in range(8):
        d = np.array([k >> 2, k >> 1 & 1, k & 1])
        c = i + d
        v = wq * g[8, c[..., 0], c[..., 1], c[..., 2]] + wv * g[ch, c[..., 0], c[..., 1], c[..., 2]]
        t, s = np.where(d == 1, f, 1 - f), np.where(d == 1, 1.0, -1.0)
        e += v * t.prod(-1)
        for a in range(3):
            grad[..., a] += v * s[a] * t[..., (a + 1) % 3] * t[..., (a + 2) % 3] / h
    return {"energy": np.where(on, e, 0).sum(1), "grad": np.where(on[..., None], grad, 0.0), "inside": None}


def _uniform64(seed, trials, rotor):
    """splitmix64 finaliser of the (seed, trial, rotor) counter -> [0, 1)."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * (
            trials.astype(np.uint64) * np.uint64(0x100000001) + np.uint64(rotor + 1))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
    return (z >> np.uint64(11)).astype(np.float64) / 9007199254740992.0


def _conformers64(case, seed):
    x0 = _chain(np.random.default_rng([seed, 4]), case["natom"])
    rot, moving, exclude = _chain_rotors(case["natom"])
    nt = case["ntrial"]
    trials = np.arange(nt)
    x = np.repeat(x0[None], nt, 0)
    for r, (a, b, c, d) in enumerate(rot):
        b1, b2, b3 = x[:, b] - x[:, a], x[:, c] - x[:, b], x[:, d] - x[:, c]
        n1, n2 = np.cross(b1, b2), np.cross(b2, b3)
        u = b2 / np.linalg.norm(b2, axis=1, keepdims=True)
        phi = np.arctan2((np.cross(n1, n2) * u).sum(1), (n1 * n2).sum(1))
        ang = (-np.pi + 2 * np.pi * _uniform64(seed, trials, r) - phi)[:, None, None]
        on = moving[r].nonzero()[0]
        v, uu = x[:, on] - x[:, c:c + 1], u[:, None]
        x[:, on] = (x[:, c:c + 1] + v * np.cos(ang) + np.cross(np.broadcast_to(uu, v.shape), v) * np.sin(ang)
                    + uu * (v * uu).sum(-1, keepdims=True) * (1 - np.cos(ang)))
    ok = np.ones(nt, bool)
    for i in range(case["natom"]):
        j = (exclude[i, i + 1:] == 0).nonzero()[0] + i + 1
        if len(j):
            ok &= ((x[:, j] - x[:, i:i + 1]) ** 2).sum(-1).min(1) >= 1.2 * 1.2
    return {"conformers": x[ok][:case["keep"]], "trial": None}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("search", "batch", "serve"):
        jobs = _jobs(case, seed)
        grids = {n: torch.as_tensor(_grid_values(n, seed), device="cuda") for n in {j["n"] for j in jobs}}
        found = [_search64(j, grids[j["n"]]) for j in jobs]
        return found[0] if kind == "search" else found
    if kind == "rescore":
        return _rescore64(case, seed)
    if kind == "refine":
        return None  # a descent whose accepted steps turn on the last bits
    if kind == "conformers":
        return _conformers64(case, seed)
    _, box, h, _, _ = _frame(case["n"])
    p = _protein_atoms(np.random.default_rng([seed, 5]), case["natom"], box)
    g = _potential_grids(p, case["n"], h, box)
    return {"grids": g.cpu().numpy(), "spectrum": torch.fft.rfftn(g[8]).cpu().numpy()}
