"""The sorted-item pass and the direct pass (small decks) behind
Context.fasten and the no-allocation entry point against the tiled kernel
(Batch.run_separate: one tiled launch per ligand): the pairs the sorted pass
leaves out are exactly zero and the rest are summed in the same order, so
every energy is equal bit for bit."""
import ctypes
import time

import numpy as np
import pytest
import torch

from minibude_amd import atomnet, capi
from minibude_amd import deck as D
from minibude_amd.batch import Batch, LigandSet
from minibude_amd.capi import BatchConfig
from minibude_amd.model import Context

pytestmark = pytest.mark.gpu


def tiled(d: D.Deck, device: int) -> np.ndarray:
    with Batch(LigandSet(d.protein, d.forcefield, [d.ligand], [d.poses]), device) as b:
        b.clear()
        b.run_separate(1, 256)
        return b.energies(0)


def same(d: D.Deck, device: int, label: str) -> np.ndarray:
    with Context(d, device) as c:
        got = c.fasten(1, 256).energies
    want = tiled(d, device)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"{label}: {np.count_nonzero(got != want)} differ"
    return got


@pytest.mark.parametrize("natpro, natlig, nposes, ntypes", [
    (938, 26, 65536, 34),    # the small deck
    (4096, 64, 1025, 34),    # just past one block of 1,024 poses
    (2000, 12, 8193, 34),    # a block of one pose
    (4095, 9, 131073, 3),    # few types: long rows, whole units of 4 x 64 items and a remainder
    (63, 1, 2500000, 1),     # one atom, one type, fewer protein atoms than lanes
    (65, 1030, 65537, 34),   # more than one chunk of items
])
def test_sorted_equals_tiled(gpu_device, natpro, natlig, nposes, ntypes):
    same(D.synth_deck(natpro, natlig, nposes, seed=71, ntypes=ntypes), gpu_device, f"{natpro}x{natlig}x{nposes}")


@pytest.mark.parametrize("natpro, natlig, nposes, ntypes", [
    (5, 1, 1, 2),          # one pose, fewer groups than waves
    (938, 26, 65, 34),     # 16 waves per tile, a tile of one pose
    (300, 200, 4097, 34),  # two waves per tile
    (40, 300, 8191, 300),  # more groups than fit in LDS
    (40, 300, 4096, 34),   # one wave per tile, four tiles per work-group
])
def test_direct_equals_tiled(gpu_device, natpro, natlig, nposes, ntypes):
    same(D.synth_deck(natpro, natlig, nposes, seed=74, ntypes=ntypes), gpu_device, f"{natpro}x{natlig}x{nposes}")


def test_noalloc_in_several_passes(gpu_device):
    # the sums of 1,000 ligand atoms fit the fixed scratch for some 700 poses at a time
    d = D.synth_deck(400, 1000, 5001, seed=75)
    up = [torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)).cuda()
          for a in (d.protein, d.ligand, d.forcefield, d.poses)]
    e = torch.full((d.nposes,), float("nan"), device="cuda")
    torch.cuda.synchronize()
    p = [ctypes.c_void_p(t.data_ptr()) for t in up]
    capi.check(capi.lib().bude_mi355x_fasten_noalloc(gpu_device, p[0], d.natpro, p[1], d.natlig, p[2], d.ntypes, p[3],
                                                     d.nposes, d.nposes, 1, 64, ctypes.c_void_p(e.data_ptr()), None))
    assert np.array_equal(e.cpu().numpy().view(np.uint32), tiled(d, gpu_device).view(np.uint32))


def test_noalloc_over_many_poses(gpu_device):
    # more poses of a small protein than the fixed scratch holds sums for in
    # some 60 passes: scored by the tiled kernel, as fast as that (the passes
    # took 1.8 times as long), or left alone where the deck is rejected
    d = D.synth_deck(64, 64, 1 << 20, seed=76)
    with Batch(LigandSet(d.protein, d.forcefield, [d.ligand], [d.poses]), gpu_device) as b:
        ms = min(b.run_separate(4, 64, 1, 4)[1:])
        want = b.energies(0)
    up = [torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)).cuda()
          for a in (d.protein, d.ligand, d.forcefield, d.poses)]
    e = torch.full((d.nposes,), float("nan"), device="cuda")
    p = [ctypes.c_void_p(t.data_ptr()) for t in up]

    def call(ntypes):
        torch.cuda.synchronize()
        t = time.perf_counter()
        st = capi.lib().bude_mi355x_fasten_noalloc(gpu_device, p[0], d.natpro, p[1], d.natlig, p[2], ntypes, p[3],
                                                   d.nposes, d.nposes, 4, 64, ctypes.c_void_p(e.data_ptr()), None)
        return st, (time.perf_counter() - t) * 1e3

    assert call(int(d.protein["type"].max()))[0] == capi.BUDE_ERR_INVALID_ARGUMENT  # (one type too few)
    assert bool(torch.isnan(e).all())
    times = []
    for _ in range(6):
        st, t = call(d.ntypes)
        capi.check(st)
        times.append(t)
    assert np.array_equal(e.cpu().numpy().view(np.uint32), want.view(np.uint32))
    assert min(times) <= 1.45 * ms + 0.1


@pytest.mark.parametrize("natlig, nposes", [
    ([1], [1]),
    ([16, 17, 33], [64, 65, 1]),                # whole rounds of 16 atoms and remainders, masked tiles
    ([96, 8, 40], [700, 1300, 64]),
])
def test_few_tiles_equal_tiled(gpu_device, natlig, nposes):
    n = len(natlig)
    ls = LigandSet(D.synth_protein(76, 500, 34), D.synth_forcefield(76, 34),
                   [D.synth_ligand(77 + i, natlig[i], 34) for i in range(n)],
                   [D.synth_poses(87 + i, nposes[i]) for i in range(n)])
    with Batch(ls, gpu_device) as b:
        b.clear()
        b.run_separate(1, 64)
        want = [b.energies(i) for i in range(n)]
        for graph in (0, 1):
            b.clear()
            b.run(BatchConfig(2, 64, 4, 0, graph), warmup=0, iterations=2)
            for i in range(n):
                assert np.array_equal(b.energies(i).view(np.uint32), want[i].view(np.uint32)), (graph, i)


@pytest.mark.parametrize("natpro, npoints, ntypes", [
    (300, 1, 3),
    (938, 1000, 34),        # fewer points of a type than a wave's lanes
    (4096, 70001, 34),
    (1500, 300000, 1),      # one type, several items per lane, a remainder
])
def test_atom_energies_equal_tiled(gpu_device, natpro, npoints, ntypes):
    rng = np.random.default_rng(78)
    pro, ff = D.synth_protein(79, natpro, ntypes), D.synth_forcefield(79, ntypes)
    pts = rng.uniform(-25, 25, (npoints, 3)).astype(np.float32)
    types = rng.integers(0, ntypes, npoints).astype(np.int32)
    got = atomnet.atom_energies(pro, ff, pts, types, gpu_device)
    used = np.unique(types)
    ligs, poses = [], []
    for t in used:  # a one-atom ligand at its frame's origin, translated to the points
        lig = np.zeros(1, capi.ATOM_DTYPE)
        lig["type"] = t
        ligs.append(lig)
        p = np.zeros((6, int((types == t).sum())), np.float32)
        p[3:] = pts[types == t].T
        poses.append(p)
    with Batch(LigandSet(pro, ff, ligs, poses), gpu_device) as b:
        b.run_separate(1, 64)
        for i, t in enumerate(used):
            assert np.array_equal(got[types == t].view(np.uint32), b.energies(i).view(np.uint32)), t


def test_poses_out_of_reach_and_not_finite(gpu_device):
    d = D.synth_deck(938, 26, 65536, seed=72)
    d.poses[3, ::7] += 1000.0     # far from the protein
    d.poses[4, ::11] = np.nan
    d.poses[5, 5::13] = np.inf
    d.poses[3, 6::13] = -np.inf
    d.poses[0, 3::17] = np.nan    # no rotation
    e = same(d, gpu_device, "scattered")
    assert np.all(e[::11] == 0.0) and np.all(e[::7] == 0.0)
    d.poses[3:] = d.poses[3:, :1]  # every pose at one place
    d.poses[:3] = 0.1
    same(d, gpu_device, "one place")


@pytest.mark.parametrize("field, value", [("radius", -3.0), ("radius", 0.0), ("elsc", 1e30), ("hphb", -np.inf)])
def test_forcefields_without_a_reach(gpu_device, field, value):
    # a radius sum that is not positive or a weight that is not finite: no pair may be left out
    d = D.synth_deck(600, 20, 65536, seed=73)
    d.forcefield[field][3] = value
    same(d, gpu_device, f"{field}={value}")


@pytest.mark.parametrize("nlig, natlig, nposes, ntypes", [
    (40, 64, 64, 34),      # rows of few items: 9 bits of cells
    (60, 600, 8, 200),     # 6
    (30, 4096, 1, 1000),   # 3
    (20, 5000, 1, 5000),   # a row for every atom: one cell a type
])
def test_short_segments_equal_direct(gpu_device, nlig, natlig, nposes, ntypes):
    ff = D.synth_forcefield(90, ntypes)
    pro = D.synth_protein(90, 5000, min(ntypes, 12))
    ligs = [D.synth_ligand(100 + i, natlig, ntypes) for i in range(nlig)]
    if ntypes >= natlig:
        for l in ligs:
            l["type"] = np.arange(natlig)
    poses = [D.synth_poses(200 + i, nposes) for i in range(nlig)]
    want = []
    for l, q in zip(ligs, poses):  # (the direct pass: too few items each to sort)
        with Context(D.Deck(pro, l, ff, q), gpu_device) as c:
            want.append(c.fasten(1, 64).energies)
    with Batch(LigandSet(pro, ff, ligs, poses), gpu_device) as b:
        b.clear()
        b.run(BatchConfig(1, 64, 4, 0, 1), warmup=1, iterations=2)
        for i in range(nlig):
            assert np.array_equal(b.energies(i).view(np.uint32), want[i].view(np.uint32)), i


def test_scratch_of_short_segments_is_bounded(gpu_device):
    # 4.2 M items in 1,024 segments: 20 bytes an item, up to 16 of counts, 48 a
    # pose, and the batch itself (a row of 4,096 counts per type and segment
    # would be 490 MB alone)
    nlig, natlig, nposes = 1024, 64, 64
    ls = LigandSet(D.synth_protein(91, 300, 34), D.synth_forcefield(91, 34),
                   [D.synth_ligand(300 + i, natlig, 34) for i in range(nlig)],
                   [D.synth_poses(400 + i, nposes) for i in range(nlig)])
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    with Batch(ls, gpu_device):
        held = before - torch.cuda.mem_get_info()[0]
    assert held < nlig * natlig * nposes * 36 + nlig * natlig * 34 * 32 + nlig * nposes * 100 + (64 << 20)


@pytest.mark.parametrize("natpro, natlig, nposes", [(1, 64, 262145), (4, 64, 262144), (16, 8, 1048576),
                                                    (64, 64, 1048576), (64, 1, 1048577)])
def test_small_proteins_equal_tiled_and_are_no_slower(gpu_device, natpro, natlig, nposes):
    # sorting an item costs more than the few pairs of a small protein (the
    # sorted pass takes 2.5 to 20 times the tiled kernel's time in these but
    # the fourth); half again is far above what a repeated pass varies by
    d = D.synth_deck(natpro, natlig, nposes, seed=92)
    with Context(d, gpu_device) as c, Batch(LigandSet(d.protein, d.forcefield, [d.ligand], [d.poses]), gpu_device) as b:
        for ppwi in (1, 4):
            b.clear()
            t = min(b.run_separate(ppwi, 64, 1, 6)[1:])
            got = c.fasten(ppwi, 64, 1, 6)
            assert np.array_equal(got.energies.view(np.uint32), b.energies(0).view(np.uint32)), ppwi
            assert min(got.device_ms[1:]) <= 1.5 * t + 0.02, ppwi


def test_a_batch_against_a_small_protein_equals_tiled(gpu_device):
    # sorted with one pose per work-item, the persistent kernel with more
    n = 6
    ls = LigandSet(D.synth_protein(93, 60, 34), D.synth_forcefield(93, 34),
                   [D.synth_ligand(94 + i, 40 + i, 34) for i in range(n)],
                   [D.synth_poses(104 + i, 180000 + 11 * i) for i in range(n)])
    with Batch(ls, gpu_device) as b:
        b.run_separate(1, 64)
        want = [b.energies(i) for i in range(n)]
        for graph in (0, 1):
            for ppwi in (1, 2, 4, 8):
                b.clear()
                b.run(BatchConfig(ppwi, 64, 4, 0, graph), warmup=0, iterations=2)
                for i in range(n):
                    assert np.array_equal(b.energies(i).view(np.uint32), want[i].view(np.uint32)), (graph, ppwi, i)


@pytest.mark.parametrize("natpro, npoints", [(1000, 999), (1000, 1000), (300, 5199), (300, 5200)])
def test_atom_energies_either_side_of_sorting(gpu_device, natpro, npoints):
    rng = np.random.default_rng(95)
    pro, ff = D.synth_protein(96, natpro, 34), D.synth_forcefield(96, 34)
    pts = rng.uniform(-20, 20, (npoints + 500, 3)).astype(np.float32)
    types = rng.integers(0, 34, npoints + 500).astype(np.int32)
    got = atomnet.atom_energies(pro, ff, pts[:npoints], types[:npoints], gpu_device)
    more = atomnet.atom_energies(pro, ff, np.repeat(pts, 2, 0), np.repeat(types, 2), gpu_device)[::2]  # (sorted)
    few = np.concatenate([atomnet.atom_energies(pro, ff, pts[i:i + 50], types[i:i + 50], gpu_device)
                          for i in range(0, npoints, 50)])[:npoints]  # (grouped on the host)
    assert np.array_equal(got.view(np.uint32), more[:npoints].view(np.uint32))
    assert np.array_equal(got.view(np.uint32), few.view(np.uint32))
