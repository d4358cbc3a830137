"""What the library does without the memory it would like:
BUDE_MI355X_MAX_ALLOC_MB makes every larger allocation fail as out of memory.
The sorted passes then give way to the kernels that need no scratch, whose
energies are the same bits."""
import numpy as np
import pytest

from minibude_amd import combined as C

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
