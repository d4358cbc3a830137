"""The work a user of this package has it do, as timed cases.

Every case goes through a public entry point: the plain pass over a resident
deck (minibude_amd.model.Context), the pass over caller device buffers
(bude_mi355x_fasten_noalloc), the ragged batch (minibude_amd.batch), the
combined screen with either surrogate (minibude_amd.combined), the learned
prescreen's network (minibude_amd.screen) and the one-atom energies the
learned field trains on (minibude_amd.atomnet).  Decks have the benchmark
workloads' distributions (minibude_amd.deck).
"""
import math

import numpy as np
import torch

from minibude_amd import atomnet, capi, combined, screen
from minibude_amd import deck as D
from minibude_amd.batch import Batch, LigandSet
from minibude_amd.capi import BatchConfig
from minibude_amd.model import PPWIS, Context

NTYPES = 34
HALF_WIDTH = 20.0  # of the cube the synthetic proteins fill (deck.synth_protein)


def listed():
    return [
        # one work-group of poses: the smallest call of the driver (-n 64), where latency counts
        dict(name="plain_tiny", kind="plain", natpro=938, natlig=26, nposes=64, ppwi=1, wgsize=64),
        # a pose count that divides nothing, a few thousand poses
        dict(name="plain_odd", kind="plain", natpro=700, natlig=19, nposes=4097, ppwi=4, wgsize=64),
        # the driver's ordinary run: the shape of the small benchmark deck
        dict(name="plain_small_deck", kind="plain", natpro=938, natlig=26, nposes=65536, ppwi=1, wgsize=256),
        # the shape of the large benchmark deck: a ligand as large as the protein
        dict(name="plain_large_ligand", kind="plain", natpro=2672, natlig=2672, nposes=65536, ppwi=1, wgsize=64),
        # the single-GPU workload, bench.py's headline
        dict(name="plain_million", kind="plain", natpro=4096, natlig=64, nposes=1048576, ppwi=1, wgsize=256),
        # a serving loop that keeps its own device buffers and may not allocate
        dict(name="noalloc_4096", kind="noalloc", natpro=938, natlig=26, nposes=4096, ppwi=1, wgsize=64),
        # a quarter of the ragged screen: many ligands of 8-96 atoms, 4,096-65,536 poses each, one launch
        dict(name="batch_ragged", kind="batch", natpro=4096, nligands=64, least=4096, most=65536, ppwi=1, wgsize=64,
             waves=4),
        # one protein of a combined screen with the energy maps
        dict(name="combined_maps", kind="combined", surrogate="field", natpro=2046, nligands=64, nposes=65536,
             steps=3000),
        # one protein of a combined screen with the learned per-atom field, trained in the call
        dict(name="combined_learned", kind="combined", surrogate="mlp", natpro=2046, nligands=16, nposes=65536,
             steps=3000),
        # forward and backward of the prescreen's network at its training batch
        dict(name="mlp_gradients", kind="mlp_grad", rows=8192),
        # the prescreen's network over a pose set
        dict(name="mlp_predict", kind="mlp_predict", nposes=1048576),
        # exact labels of single atoms, as the learned field trains on
        dict(name="atom_labels", kind="atoms", natpro=4096, npoints=262144),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plain", "plain", "plain", "plain", "noalloc", "batch", "batch", "combined", "mlp", "atoms"])
    if kind in ("plain", "noalloc"):
        while True:
            c = dict(kind=kind, natpro=_log(rng, 64, 6000), natlig=_log(rng, 1, 128),
                     nposes=_log(rng, 64, 1 << 20 if kind == "plain" else 1 << 16), ppwi=rng.choice(PPWIS),
                     wgsize=rng.choice([64, 128, 256, 512, 1024]))
            # (a few poses at a large ppwi are one long wave: those stay short too)
            pairs = c["natpro"] * c["natlig"]
            if pairs * c["nposes"] <= 1e11 and pairs * c["ppwi"] <= 5e6:
                return c
    if kind == "batch":
        least = _log(rng, 64, 8192)
        return dict(kind=kind, natpro=_log(rng, 300, 4096), nligands=rng.randint(2, 48), least=least,
                    most=least * rng.randint(2, 5), ppwi=rng.choice([1, 2, 4]), wgsize=rng.choice([64, 256]),
                    waves=rng.choice([4, 8]))
    if kind == "combined":
        # (the learned field trains in the call whatever the size: fewer steps keep a drawn case short)
        surrogate = rng.choice(["field", "field", "mlp"])
        return dict(kind=kind, surrogate=surrogate, natpro=_log(rng, 900, 4000),
                    nligands=rng.randint(4, 16 if surrogate == "mlp" else 48), nposes=_log(rng, 16384, 65536),
                    steps=1000)
    if kind == "mlp":
        if rng.random() < 0.5:
            return dict(kind="mlp_grad", rows=32 * _log(rng, 1, 512))
        return dict(kind="mlp_predict", nposes=_log(rng, 1000, 1 << 20))
    return dict(kind="atoms", natpro=_log(rng, 300, 6000), npoints=_log(rng, 1000, 1 << 18))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _deck(case, seed):
    return D.synth_deck(case["natpro"], case["natlig"], case["nposes"], seed, NTYPES)


def _ragged(case, seed):
    """ragged_workload's set with the ligands' sizes drawn for the case and their contents for the seed."""
    rs = np.random.RandomState(case["nligands"] * 65537 + case["least"])
    ligands, poses = [], []
    for i in range(case["nligands"]):
        ligands.append(D.synth_ligand(seed * 1009 + i, int(rs.randint(8, 97)), NTYPES))
        poses.append(D.synth_poses(seed * 1009 + i, int(rs.randint(case["least"], case["most"] + 1))))
    return LigandSet(D.synth_protein(seed, case["natpro"], NTYPES), D.synth_forcefield(seed, NTYPES), ligands, poses)


def _mlp_weights(seed):
    """The prescreen's network as it starts training: He-scaled normal weights, small biases."""
    rs = np.random.RandomState(seed % (1 << 31))
    shapes = ((21, 256), (256, 256), (256, 256), (256, 1))
    W = [(rs.standard_normal(s) * math.sqrt(2.0 / s[0])).astype(np.float32) for s in shapes]
    b = [(0.05 * rs.standard_normal(s[1])).astype(np.float32) for s in shapes]
    return W, b


def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)).cuda()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "plain":
        return dict(case=case, ctx=Context(_deck(case, seed)))
    if kind == "noalloc":
        d = _deck(case, seed)
        return dict(case=case, protein=_device(d.protein), ligand=_device(d.ligand), ff=_device(d.forcefield),
                    poses=torch.from_numpy(d.poses).cuda(), energies=torch.empty(d.nposes, device="cuda"))
    if kind == "batch":
        return dict(case=case, batch=Batch(_ragged(case, seed)),
                    cfg=BatchConfig(case["ppwi"], case["wgsize"], case["waves"], 0, 1))
    if kind == "combined":
        w = combined.combined_workload(nproteins=1, nligands=case["nligands"], nposes=case["nposes"],
                                       seed=seed % 1000, natpro_range=(case["natpro"], case["natpro"]))
        cfg = combined.default_config(case["surrogate"], steps=case["steps"], seed=seed)
        return dict(case=case, protein=w.proteins[0],
                    screen=combined.Combined(w.forcefield, w.ligands, w.poses, cfg))
    if kind == "mlp_grad":
        W, b = _mlp_weights(seed)
        feat = screen.features(D.synth_poses(seed, case["rows"])).astype(np.float32)
        target = np.random.RandomState(seed % (1 << 31)).standard_normal(case["rows"]).astype(np.float32)
        return dict(case=case, feat=feat, target=target, W=W, b=b)
    if kind == "mlp_predict":
        W, b = _mlp_weights(seed)
        return dict(case=case, poses=D.synth_poses(seed, case["nposes"]), W=W, b=b)
    rs = np.random.RandomState(seed % (1 << 31))
    points = rs.uniform(-15.0, 15.0, (case["npoints"], 3)).astype(np.float32)
    types = rs.randint(0, NTYPES, case["npoints"]).astype(np.int32)
    return dict(case=case, protein=D.synth_protein(seed, case["natpro"], NTYPES), ff=D.synth_forcefield(seed, NTYPES),
                points=points, types=types)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "plain":
        return state["ctx"].fasten(case["ppwi"], case["wgsize"]).energies
    if kind == "noalloc":
        p, l, f, q, e = (state[k] for k in ("protein", "ligand", "ff", "poses", "energies"))
        n = case["nposes"]
        capi.check(capi.lib().bude_mi355x_fasten_noalloc(0, p.data_ptr(), case["natpro"], l.data_ptr(), case["natlig"],
                                                         f.data_ptr(), NTYPES, q.data_ptr(), n, n, case["ppwi"],
                                                         case["wgsize"], e.data_ptr(),
                                                         torch.cuda.current_stream().cuda_stream))
        return e
    if kind == "batch":
        state["batch"].run(state["cfg"])
        return [state["batch"].energies(i) for i in range(case["nligands"])]
    if kind == "combined":
        s = state["screen"]
        s.screen(state["protein"])
        # the exact energies of the selected poses, by pose, of every pair
        out = np.full((case["nligands"], case["nposes"]), np.nan, np.float32)
        for i in range(case["nligands"]):
            idx, e = s.selected(i)
            out[i, idx] = e
        return out
    if kind == "mlp_grad":
        pred, loss, gW, gb = screen.mlp_forward_backward(state["feat"], state["target"], state["W"], state["b"])
        return dict(pred=pred, loss=loss, gW=gW, gb=gb)
    if kind == "mlp_predict":
        return screen.mlp_predict(state["poses"], state["W"], state["b"])
    return atomnet.atom_energies(state["protein"], state["ff"], state["points"], state["types"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

PAIR_FLOPS = 20  # three differences, the distance (6), three hinges (9), the sums


def _pair_terms(p, l):
    """The 64-bit pair terms of a protein and a ligand forcefield row: (radij,
    charge weight, charge range, desolvation weight, desolvation range); a
    weight is 0 where the term is off."""
    radij = float(p["radius"]) + float(l["radius"])
    q = float(p["elsc"]) * float(l["elsc"])
    if 69 in (int(p["hbtype"]), int(l["hbtype"])):
        q = -abs(q)
    ff = int(p["hbtype"]) == 70 and int(l["hbtype"]) == 70
    ph, lh = float(p["hphb"]), float(l["hphb"])
    on = ph != 0.0 and (ph < 0.0 or lh < 0.0)
    reach = 5.5 if ph < 0.0 and lh < 0.0 else 1.0
    wd = (-ph if ph < 0.0 < lh else ph) + (-lh if lh < 0.0 < ph else lh)
    return radij, 45.0 * q, 4.0 if ff else 2.0, wd if on else 0.0, reach


def _reached():
    """The share of a protein's atoms within reach of a ligand atom well inside it (every term of a pair further
    off is zero), mean over the types."""
    ff = D.synth_forcefield(0, NTYPES)
    v = 0.0
    for p in ff:
        for l in ff:
            radij, _, cr, wd, dr = _pair_terms(p, l)
            v += 4.0 / 3.0 * math.pi * (radij + max(cr, dr if wd else 0.0)) ** 3
    return min(1.0, v / NTYPES ** 2 / (2.0 * HALF_WIDTH) ** 3)


def work(case):
    kind = case["kind"]
    if kind in ("plain", "noalloc"):
        return dict(bytes=28.0 * case["nposes"] + 16.0 * (case["natpro"] + case["natlig"] + NTYPES),
                    flops=PAIR_FLOPS * _reached() * case["nposes"] * case["natlig"] * case["natpro"])
    if kind == "batch":
        poses, atoms = case["nligands"] * (case["least"] + case["most"]) / 2.0, 52.0
        return dict(bytes=28.0 * poses + 16.0 * (case["natpro"] + atoms * case["nligands"]),
                    flops=PAIR_FLOPS * _reached() * poses * atoms * case["natpro"])
    if kind == "combined":
        # every pose read once and scored, its atoms looked up in the surrogate; 2 % of the poses and the sampled ones
        # exactly; the surrogate itself
        poses, atoms = float(case["nligands"]) * case["nposes"], 52.0
        learned = case["surrogate"] == "mlp"
        net = 2.0 * (42 * 32 + 32 * 32 + 32)
        exact = 0.02 * poses + (4096 if learned else 1024) * case["nligands"]
        flops = PAIR_FLOPS * _reached() * case["natpro"] * exact * atoms + poses * atoms * (net if learned else 40.0)
        if learned:
            flops += 3.0 * net * 32768 * case["steps"] + PAIR_FLOPS * _reached() * case["natpro"] * (1 << 22)
        else:
            flops += PAIR_FLOPS * _reached() * case["natpro"] * NTYPES * 62.0 ** 3
        return dict(bytes=24.0 * poses + 16.0 * (case["natpro"] + atoms * case["nligands"]) + 8.0 * 0.02 * poses,
                    flops=flops)
    if kind == "mlp_grad":
        params = 21 * 256 + 2 * 65536 + 256 + 769
        return dict(bytes=case["rows"] * (21 + 2) * 4.0 + 8.0 * params, flops=6.0 * params * case["rows"])
    if kind == "mlp_predict":
        params = 21 * 256 + 2 * 65536 + 256 + 769
        return dict(bytes=28.0 * case["nposes"] + 4.0 * params, flops=2.0 * params * case["nposes"])
    return dict(bytes=20.0 * case["npoints"] + 16.0 * case["natpro"],
                flops=PAIR_FLOPS * _reached() * case["npoints"] * case["natpro"])


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

MOST_PAIRS = 7e10  # beyond this the 64-bit pass takes too long


def _atom_energies64(protein, ff, points, ltype):
    """Energy (not yet halved) of one ligand atom of type `ltype` at each of points (n, 3), float64 on the GPU."""
    out = torch.zeros(len(points), dtype=torch.float64, device="cuda")
    p2 = (points * points).sum(1, keepdim=True)
    for t in np.unique(protein["type"]):
        a = protein[protein["type"] == t]
        xyz = torch.from_numpy(np.stack([a["x"], a["y"], a["z"]], 1).astype(np.float64)).cuda()
        radij, wq, cr, wd, dr = _pair_terms(ff[t], ff[ltype])
        d = torch.addmm(p2 + (xyz * xyz).sum(1), points, xyz.T, alpha=-2.0).clamp_(min=0.0).sqrt_()
        out += 76.0 * (1.0 - d / radij).clamp_(min=0.0).sum(1)
        if wq:
            out += wq * ((radij - d) / cr).add_(1.0).clamp_(0.0, 1.0).sum(1)
        if wd:
            out += wd * ((radij - d) / dr).add_(1.0).clamp_(0.0, 1.0).sum(1)
    return out


def _pose_energies64(protein, ligand, ff, poses):
    q = torch.from_numpy(poses).cuda().double()
    s, c = torch.sin(q[:3]), torch.cos(q[:3])
    R = torch.stack([
        torch.stack([c[1] * c[2], s[0] * s[1] * c[2] - c[0] * s[2], c[0] * s[1] * c[2] + s[0] * s[2]], -1),
        torch.stack([c[1] * s[2], s[0] * s[1] * s[2] + c[0] * c[2], c[0] * s[1] * s[2] - s[0] * c[2]], -1),
        torch.stack([-s[1], s[0] * c[1], c[0] * c[1]], -1)], -2)
    e = torch.zeros(q.shape[1], dtype=torch.float64, device="cuda")
    for a in ligand:
        x = torch.tensor([float(a["x"]), float(a["y"]), float(a["z"])], dtype=torch.float64, device="cuda")
        at = (R * x).sum(-1) + q[3:].T
        for i in range(0, len(at), 1 << 19):
            e[i:i + (1 << 19)] += _atom_energies64(protein, ff, at[i:i + (1 << 19)], int(a["type"]))
    return 0.5 * e


def _gelu(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


def _mlp64(x, W, b):
    x = torch.from_numpy(np.ascontiguousarray(x, np.float64)).cuda()
    W = [torch.from_numpy(w).cuda().double().requires_grad_() for w in W]
    b = [torch.from_numpy(v).cuda().double().requires_grad_() for v in b]
    for i in range(3):
        x = _gelu(x @ W[i] + b[i])
    return (x @ W[3] + b[3]).reshape(-1), W, b


def exact(case, seed):
    kind = case["kind"]
    if kind in ("plain", "noalloc"):
        if case["natpro"] * case["natlig"] * case["nposes"] > MOST_PAIRS:
            return None
        d = _deck(case, seed)
        return _pose_energies64(d.protein, d.ligand, d.forcefield, d.poses)
    if kind == "batch":
        w = _ragged(case, seed)
        if w.interactions > MOST_PAIRS:
            return None
        return [_pose_energies64(w.protein, l, w.forcefield, p) for l, p in zip(w.ligands, w.poses)]
    if kind == "combined":
        return None
    if kind in ("mlp_grad", "mlp_predict"):
        s = prepare(case, seed)
        if kind == "mlp_predict":
            with torch.no_grad():
                return torch.cat([_mlp64(screen.features(s["poses"][:, i:i + (1 << 17)]), s["W"], s["b"])[0]
                                  for i in range(0, case["nposes"], 1 << 17)])
        pred, W, b = _mlp64(s["feat"], s["W"], s["b"])
        loss = (pred - torch.from_numpy(s["target"]).cuda().double()).square().mean()
        loss.backward()
        return dict(pred=pred, loss=float(loss), gW=[w.grad for w in W], gb=[v.grad for v in b])
    s = prepare(case, seed)
    points = torch.from_numpy(s["points"]).cuda().double()
    types = torch.from_numpy(s["types"]).cuda()
    out = torch.zeros(len(points), dtype=torch.float64, device="cuda")
    for t in range(NTYPES):
        at = (types == t).nonzero().reshape(-1)
        if len(at):
            out[at] = 0.5 * _atom_energies64(s["protein"], s["ff"], points[at], t)
    return out
