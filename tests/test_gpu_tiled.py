"""The register-blocked kernels by themselves: the tiled kernel through
Batch.run_separate (a deck's own call may be scored by another form, whatever
its arguments) and the persistent kernel on sets that are neither sorted (a
pair without a reach) nor few tiles.  A register block only changes which lane
holds a pose, never the sums."""
import numpy as np
import pytest

import oracle_lib as O
from minibude_amd import combined as C
from minibude_amd import deck as D
from minibude_amd import screen as S
from minibude_amd.batch import Batch, LigandSet
from minibude_amd.capi import BatchConfig

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("ppwi", [4, 8, 16])
def test_blocks_over_a_full_device_equal_single_poses(gpu_device, ppwi):
    # four waves per SIMD and more, where blocks of eight become blocks of four
    n = 262144 * ppwi + 65
    ls = LigandSet(D.synth_protein(41, 12, 34), D.synth_forcefield(41, 34), [D.synth_ligand(42, 3, 34)],
                   [D.synth_poses(43, n)])
    with Batch(ls, gpu_device) as b:
        b.run_separate(1, 64)
        want = b.energies(0)
        for wgsize in (64, 512, 1024):
            b.clear()
            b.run_separate(ppwi, wgsize)
            assert np.array_equal(bits(b.energies(0)), bits(want)), wgsize


def unreachable(natpro, natlig, nposes, seed, ntypes=34):
    """Ligands of natlig[i] atoms with nposes[i] poses that have a pair without a reach."""
    ff = D.synth_forcefield(seed, ntypes)
    ff["radius"][3] = 0.0
    pro = D.synth_protein(seed, natpro, ntypes)
    pro["type"][0] = 3
    ligs = [D.synth_ligand(seed + 1 + i, n, ntypes) for i, n in enumerate(natlig)]
    for l in ligs:
        l["type"][0] = 3
    return LigandSet(pro, ff, ligs, [D.synth_poses(seed + 1 + i, n) for i, n in enumerate(nposes)])


def test_few_tiles_of_small_ligands(gpu_device):
    # a tile's 16 waves have nothing to share in a ligand of two atoms: the
    # persistent kernel takes them, in a quarter of the time that eight atoms
    # take (shared tiles took three quarters)
    times = []
    for natlig in (2, 8):
        ls = unreachable(4096, [natlig] * 64, [4096] * 64, 44)
        with Batch(ls, gpu_device) as b:
            b.run_separate(1, 64)
            want = [b.energies(i) for i in range(64)]
            for cfg in (BatchConfig(1, 64, 4, 0, 1), BatchConfig(4, 256, 8, 1, 0)):
                b.clear()
                t = min(b.run(cfg, 1, 4)[1:])
                assert all(np.array_equal(bits(b.energies(i)), bits(want[i])) for i in range(64)), (natlig, cfg.ppwi)
            times.append(t)
    assert times[0] < 0.5 * times[1]


def test_selections_of_many_rows_without_a_reach(gpu_device):
    # some 9,400 and 4,700 tiles of selected rows, through the index
    ls = unreachable(300, [5, 17], [400000, 200000], 46)
    cfg = C.default_config("field", keep_fraction=0.5, widen_max=0.5, gate_z=0.0, grid_spacing=1.5)
    with C.Combined(ls.forcefield, ls.ligands, ls.poses, cfg, gpu_device) as c:
        c.screen(ls.protein)
        c.exhaustive()
        for l in range(2):
            idx, e = c.selected(l)
            assert len(idx) >= len(c.exact(l)) // 2 and np.array_equal(bits(e), bits(c.exact(l)[idx])), l
    cfg = S.default_config(epochs=1, batch=1024, keep_fraction=0.75)
    with S.Screen(ls.protein, ls.ligands[0], ls.forcefield, cfg, gpu_device) as s:
        s.train(D.synth_poses(48, 16384))
        s.load(ls.poses[0])
        s.run()
        idx, e = s.selected()
        exact = s.exhaustive()[0]
        assert len(idx) >= 300000 and np.array_equal(bits(e), bits(exact[idx]))


def test_every_block_and_group_size(gpu_device):
    # groups of 0 to 23 atoms and some larger, so that every exit of the
    # pipelined pair loop is taken, by every register block and work-group
    # size, against the FP64 oracle (16 FP32 epsilons of the sum of the terms'
    # magnitudes, as for the deck's own call)
    ntypes = 34
    sizes = [t if t < 24 else 24 + 3 * (t - 24) for t in range(ntypes)]
    pro = D.synth_protein(51, sum(sizes), ntypes)
    pro["type"] = np.repeat(np.arange(ntypes, dtype=np.int32), sizes)
    d = D.Deck(pro[np.random.default_rng(6).permutation(len(pro))], D.synth_ligand(52, 12, ntypes),
               D.synth_forcefield(51, ntypes), D.synth_poses(53, 2000))
    e64, mag = O.fasten_f64_mag(d, 0, d.nposes)
    with Batch(LigandSet(d.protein, d.forcefield, [d.ligand], [d.poses]), gpu_device) as b:
        b.run_separate(1, 64)
        want = b.energies(0)
        ok = mag > 0
        assert np.all(want[~ok] == 0.0)
        assert np.max(np.abs(want.astype(np.float64) - e64)[ok] / mag[ok]) < 16.0 * 2.0 ** -24
        for ppwi in (1, 2, 4, 8, 16, 128):
            for wgsize in (64, 128, 256, 512, 1024):
                b.clear()
                b.run_separate(ppwi, wgsize)
                assert np.array_equal(bits(b.energies(0)), bits(want)), (ppwi, wgsize)


@pytest.mark.parametrize("cfg", [BatchConfig(1, 64, 4, 0, 0), BatchConfig(2, 256, 8, 1, 1), BatchConfig(4, 128, 2, 0, 1),
                                 BatchConfig(8, 512, 1, 1, 0)], ids=lambda c: f"p{c.ppwi}w{c.wgsize}")
def test_persistent_kernel_equals_tiled(gpu_device, cfg):
    ls = unreachable(120, [1, 7, 20, 33], [150001, 64, 90000, 60063], 54)  # 4,690 tiles of 64
    with Batch(ls, gpu_device) as b:
        b.run_separate(1, 64)
        want = [b.energies(i) for i in range(4)]
        b.clear()
        b.run(cfg, warmup=1, iterations=2)
        for i in range(4):
            assert np.array_equal(bits(b.energies(i)), bits(want[i])), i
