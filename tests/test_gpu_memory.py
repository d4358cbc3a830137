"""What the library does without the memory it would like:
BUDE_MI355X_MAX_MEMORY_MB bounds what its objects hold.  The sorted passes give
way to the kernels that need no scratch, whose energies are the same bits, and
what an object can do without is never in the way of what it needs."""
import numpy as np
import pytest

from minibude_amd import capi
from minibude_amd import combined as C
from minibude_amd import deck as D
from minibude_amd import screen as S
from minibude_amd.model import Context

pytestmark = pytest.mark.gpu

LIMIT = "BUDE_MI355X_MAX_MEMORY_MB"


def same_bits(a, b):
    return len(a) == len(b) and np.array_equal(np.ascontiguousarray(a).view(np.uint32),
                                               np.ascontiguousarray(b).view(np.uint32))


class Bound:
    """Bounds the memory of the library's objects to some MB more than they hold."""

    def __init__(self, monkeypatch, device):
        self.patch, self.device = monkeypatch, device
        self.held = 0

    def here(self):
        tiny = D.synth_deck(8, 1, 8, seed=50)
        for step in (1024, 64, 4, 1):  # the least bound a deck of a few kilobytes is accepted under
            while True:
                self.patch.setenv(LIMIT, str(self.held))
                try:
                    Context(tiny, self.device).close()
                    break
                except capi.BudeError:
                    self.held += step
            if step > 1:
                self.held = max(0, self.held - step)
        return self

    def more(self, mb):
        self.patch.setenv(LIMIT, str(self.held + mb))

    def off(self):
        self.patch.delenv(LIMIT, raising=False)


@pytest.fixture
def bound(monkeypatch, gpu_device):
    return Bound(monkeypatch, gpu_device)


@pytest.mark.parametrize("mixed", [False, True])
def test_a_pass_without_room_leaves_later_screens_as_they_are(gpu_device, bound, mixed):
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
    out = []
    for bounded in (False, True):
        with C.Combined(w.forcefield, w.ligands, w.poses, cfg, gpu_device) as c:
            got = []
            for p in w.proteins:
                r = c.screen(p)
                assert not mixed or p is not w.proteins[0] or 0 < r.fallback_pairs < 6
                if bounded and p is w.proteins[0]:
                    bound.here().more(16)
                got += [x for l in range(6) for x in c.selected(l)]
                c.exhaustive()
                got += [c.exact(l) for l in range(6)]
                c.screen(p)
                got += [x for l in range(6) for x in c.selected(l)]
            out.append(got)
    assert all(same_bits(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("natpro, natlig, nposes, mb", [
    (938, 26, 65536, 16),   # no room to sort
    (938, 26, 65536, 4),    # nor for the direct pass's sums (6.8 MB)
    (30, 400, 32768, 16),   # not sorted: no room for the sums (52 MB)
])
def test_a_deck_without_room_for_scratch_is_scored(gpu_device, bound, natpro, natlig, nposes, mb):
    d = D.synth_deck(natpro, natlig, nposes, seed=52)
    with Context(d, gpu_device) as c:
        want = c.fasten(1, 64).energies
    bound.here().more(mb)
    with Context(d, gpu_device) as c:
        assert same_bits(c.fasten(1, 64).energies, want)


def test_a_prescreen_without_room_for_scratch_is_scored(gpu_device, bound):
    w = S.screen_workload(ntrain=16384, nscreen=60000, natlig=20, natpro=900)
    cfg = S.default_config(epochs=1, batch=1024, keep_fraction=0.1)
    out = []
    for bounded in (False, True):
        with S.Screen(w.protein, w.ligand, w.forcefield, cfg, gpu_device) as s:
            if bounded:
                bound.here().more(32)
            got = []
            s.train(w.train_poses)
            for poses in (w.screen_poses[:, :50000], w.screen_poses):
                s.load(np.ascontiguousarray(poses))
                s.run()
                got += [*s.selected(), s.exhaustive()[0]]
            out.append(got)
    assert all(same_bits(a, b) for a, b in zip(*out))


def test_scratch_is_not_in_the_way_of_a_decks_buffers(gpu_device, bound):
    # 56 MB of poses and energies, and some 150 MB of scratch: any bound that
    # holds the first is enough
    d = D.synth_deck(2000, 1, 2000000, seed=53)
    with Context(d, gpu_device) as c:
        want = c.fasten(1, 64).energies
    bound.here()
    for mb in range(57, 240, 5):
        bound.more(mb)
        with Context(d, gpu_device) as c:
            assert same_bits(c.fasten(1, 64).energies, want), mb


@pytest.mark.parametrize("surrogate", ["field", "mlp"])
def test_scratch_is_not_in_the_way_of_a_screen(gpu_device, bound, surrogate):
    # the rescoring of half of all poses takes 80 MB and more of scratch (and
    # the learned field's index 30 MB), the rest of the object and its screens
    # less than 48: a bound of that or more is enough
    w = C.combined_workload(nproteins=2, nligands=6, nposes=20000, seed=54, natpro_range=(800, 1000),
                            natlig_range=(40, 70))
    cfg = C.default_config(surrogate, keep_fraction=0.5, widen_max=0.5, gate_z=0.0, grid_spacing=1.5, steps=20,
                           train_points=1 << 18)

    def screens():
        with C.Combined(w.forcefield, w.ligands, w.poses, cfg, gpu_device) as c:
            got = []
            c.screen_batch(w.proteins, lambda i: got.extend(x for l in range(6) for x in c.selected(l)))
            c.set_keep(0.6)
            c.screen(w.proteins[0])
            got.extend(x for l in range(6) for x in c.selected(l))
            c.exhaustive()
            got.append(c.recall(0.01))
        return got

    want = screens()
    bound.here()
    for mb in range(48, 208, 10):
        bound.more(mb)
        assert all(same_bits(a, b) for a, b in zip(screens(), want)), mb
