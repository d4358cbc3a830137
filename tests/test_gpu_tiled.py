"""The register-blocked kernels by themselves: the tiled kernel through
Batch.run_separate (a deck's own call may be scored by another form, whatever
its arguments) and the persistent kernel on sets that are neither sorted (a
pair without a reach) nor few tiles.  A register block only changes which lane
holds a pose, never the sums."""
import numpy as np
import pytest

import oracle_lib as O
from minibude_amd import deck as D
from minibude_amd.batch import Batch, LigandSet
from minibude_amd.model import Context

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
