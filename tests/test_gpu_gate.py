"""The combined screen's validation statistics against numpy on the screen's
own samples: both are FP64 sums in another order, reported in FP32 (6e-8);
the error deviation is a difference of variances a few orders apart, which
costs some digits of 1e-16, so 1e-5 relative is far above both."""
import numpy as np
import pytest

from minibude_amd import combined as C
from minibude_amd import deck as D

pytestmark = pytest.mark.gpu


def numpy_stats(e, p, keep, top, clip_q):
    n = len(e)
    e, p = e.astype(np.float64), p.astype(np.float64)
    oe, op = np.argsort(e, kind="stable"), np.argsort(p, kind="stable")

    def q(f):
        x = f * (n - 1)
        i = int(x)
        return e[oe[i]] * (1 - (x - i)) + e[oe[i + 1]] * (x - i) if i + 1 < n else e[oe[n - 1]]

    nt = min(n, max(8, int(np.ceil(0.25 * n))))
    x, y = e[oe[:nt]], p[oe[:nt]]
    ve, vp, cv = x.var(), y.var(), ((x - x.mean()) * (y - y.mean())).mean()
    a = cv / ve if ve > 0 else 0.0
    sd = np.sqrt(max(0.0, vp - a * cv)) / a if a > 0 else np.inf
    kt = max(1, int(np.floor(0.05 * n + 0.5)))
    ks = min(n, max(kt, int(np.floor(0.10 * n + 0.5))))
    recall = np.isin(oe[:kt], op[:ks]).mean()
    clip = e[oe[min(n - 1, int(np.float64(np.float32(clip_q)) * n))]]
    t = np.minimum(e, clip)
    mu, sigma = np.float32(t.mean()), np.float32(np.sqrt(max(1e-12, (t * t).mean() - float(np.float32(t.mean())) ** 2)))
    y, x = (t - mu) / sigma, (np.minimum(p, clip) - mu) / sigma
    cxy = ((x - x.mean()) * (y - y.mean())).mean()
    cal = max(0.0, y.var() - cxy * cxy / x.var()) if x.var() > 0 and cxy > 0 else y.var()
    return (q(keep) - q(top)) / sd, recall, np.sqrt(((x - y) ** 2).mean()), np.sqrt(cal)


@pytest.mark.parametrize("labels", [48, 1000, 1024, 4096])  # a wave, not a power of two, one, the most
def test_pair_statistics(gpu_device, labels):
    ff = D.synth_forcefield(91, 34)
    ligs = [D.synth_ligand(92 + i, 9 + 11 * i, 34) for i in range(3)]
    poses = [D.synth_poses(95 + i, n) for i, n in enumerate((5000, 4097, 900))]  # (the last: fewer poses than labels)
    cfg = C.default_config("field", grid_spacing=1.0, gate_z=0.0, labels_per_pair=labels)
    with C.Combined(ff, ligs, poses, cfg, gpu_device) as c:
        c.screen(D.synth_protein(99, 700, 34))
        for l in range(3):
            idx, e = c.labels(l)
            r = c.pair(l)
            want = numpy_stats(e, c.scores(l)[idx], 0.02, 0.01, cfg.clip_quantile)
            got = (r.gate_z, r.sample_recall, r.val_rmse, r.val_rmse_calibrated)
            np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-7, err_msg=f"pair {l}")
