"""What the library does without the memory it would like:
BUDE_MI355X_MAX_ALLOC_MB makes every larger allocation fail as out of memory.
The sorted passes then give way to the kernels that need no scratch, whose
energies are the same bits."""
import numpy as np
import pytest

from minibude_amd import combined as C
from minibude_amd import deck as D
from minibude_amd import screen as S
from minibude_amd.model import Context

pytestmark = pytest.mark.gpu

LIMIT = "BUDE_MI355X_MAX_ALLOC_MB"


def same_bits(a, b):
    return len(a) == len(b) and np.array_equal(np.ascontiguousarray(a).view(np.uint32),
                                               np.ascontiguousarray(b).view(np.uint32))


@pytest.mark.parametrize("mixed", [False, True])
def test_a_pass_without_room_leaves_later_screens_as_they_are(gpu_device, monkeypatch, mixed):
    # 6.5 M items to score every pose (130 MB and more), 0.3 M to rescore a
    # selection: both worth sorting, the first without the memory for it
    # (mixed: some pairs' poses, behind a validation bound between the pairs')
    w = C.combined_workload(nproteins=2, nligands=6, nposes=20000, seed=51, natpro_range=(800, 1000),
                            natlig_range=(40, 70))
    cfg = C.default_config("field", keep_fraction=0.05, gate_z=0.0, grid_spacing=1.5)
    if mixed:
        with C.Combined(w.forcefield, w.ligands, w.poses, cfg, gpu_device) as c:
            c.screen(w.proteins[0])
            cfg.max_val_rmse = float(np.median([c.pair(l).val_rmse_calibrated for l in range(6)]))
    out = {}
    for mb in (None, "24"):
        with C.Combined(w.forcefield, w.ligands, w.poses, cfg, gpu_device) as c:
            if mb:
                monkeypatch.setenv(LIMIT, mb)
            got = []
            for p in w.proteins:
                r = c.screen(p)
                assert not mixed or p is not w.proteins[0] or 0 < r.fallback_pairs < 6
                got += [x for l in range(6) for x in c.selected(l)]
                c.exhaustive()
                got += [c.exact(l) for l in range(6)]
                c.screen(p)
                got += [x for l in range(6) for x in c.selected(l)]
            out[mb] = got
            monkeypatch.delenv(LIMIT, raising=False)
    assert all(same_bits(a, b) for a, b in zip(out[None], out["24"]))


@pytest.mark.parametrize("mb", ["16", "4"])  # no room to sort; none for the direct pass's sums (6.8 MB) either
def test_a_deck_without_room_for_scratch_is_scored(gpu_device, monkeypatch, mb):
    d = D.synth_deck(938, 26, 65536, seed=52)
    with Context(d, gpu_device) as c:
        want = c.fasten(1, 64).energies
    monkeypatch.setenv(LIMIT, mb)
    with Context(d, gpu_device) as c:
        assert same_bits(c.fasten(1, 64).energies, want)


def test_a_prescreen_without_room_for_scratch_is_scored(gpu_device, monkeypatch):
    w = S.screen_workload(ntrain=16384, nscreen=60000, natlig=20, natpro=900)
    cfg = S.default_config(epochs=1, batch=1024, keep_fraction=0.1)
    out = {}
    for mb in (None, "8"):
        with S.Screen(w.protein, w.ligand, w.forcefield, cfg, gpu_device) as s:
            if mb:
                monkeypatch.setenv(LIMIT, mb)
            got = []
            s.train(w.train_poses)
            for poses in (w.screen_poses[:, :50000], w.screen_poses):
                s.load(np.ascontiguousarray(poses))
                s.run()
                got += [*s.selected(), s.exhaustive()[0]]
            out[mb] = got
    assert all(same_bits(a, b) for a, b in zip(out[None], out["8"]))
