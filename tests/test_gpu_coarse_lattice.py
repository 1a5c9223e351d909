"""Coarse squared differences over the forms the translation lattice and the pixel layout can take, against the FP64
oracle: every number of positive shifts (0 .. 9; 8 keeps the zero shift beside the matrix columns, 9 takes two column
tiles), coarse sizes whose rows end inside a step of 8 pixels, partial orientation tiles, single and several classes.

Tolerance 2e-6 relative: the stored float32 value rounds by 6e-8, and the float32 sums (at most 9 matrix steps of 4 and
17 row pairs, magnitudes below the value itself) by a few ulp each.
"""
import numpy as np
import pytest

import relion_amd as ra
from problems import make_problem
from test_gpu_parity import rel, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shifts,box,px,order,diameter,extra", [
    (0, 32, 4.0, 1, 60.0, {}),
    (1, 32, 4.0, 1, 60.0, {}),
    (2, 36, 3.0, 1, 60.0, dict(nr_classes=2)),
    (3, 32, 4.0, 1, 80.0, dict(current_size=28)),
    (4, 40, 3.0, 1, 100.0, dict(local=True, sigma_ang=12.0)),
    (5, 32, 4.0, 1, 100.0, {}),
    (6, 48, 2.5, 1, 90.0, dict(scale_correction=True, perturb_meta=True)),
    (7, 32, 4.0, 1, 60.0, dict(separate_nomask=True)),
    (8, 40, 3.0, 1, 100.0, {}),
    (8, 36, 3.0, 2, 80.0, dict(local=True, sigma_ang=9.0, nr_classes=2)),
    (9, 40, 3.0, 1, 80.0, {}),
])
def test_coarse_diff2_lattices(shifts, box, px, order, diameter, extra):
    p = make_problem(box=box, px=px, order=order, offset_range_px=0.5 * shifts, offset_step_px=0.5,
                     diameter=diameter, n=3, snr=0.3, nr_blobs=20, seed=17 + shifts, **extra)
    es, rg, _, _, _ = run_gpu(p)
    ro, _, _, dbg = run_oracle(p, (0, 1, 2))
    _, _, nt = ra.sampling_counts(p.cfg)
    for ip in range(3):
        d2g = es.coarse(ip)[0]
        d2o = dbg[ip]["coarse_diff2"]
        ok = d2o >= 0
        assert d2g.size == d2o.size and d2g.size % nt == 0
        assert np.array_equal(d2g >= 0, ok)
        assert rel(d2g[ok], d2o[ok]).max() < 2e-6
    assert np.array_equal(rg["best_ihidden_over"], ro["best_ihidden_over"])


def test_coarse_diff2_of_a_perfect_match_stays_evaluated():
    """A noise-free particle at a grid pose: its diff2 is zero up to rounding and must not turn negative, which marks
    poses that were never evaluated."""
    p = make_problem(box=32, px=4.0, order=1, offset_range_px=2, offset_step_px=1, n=2, snr=1e9, nr_blobs=20, seed=5)
    p.sigma2_noise = np.full(17, 1e-4 * float(np.mean(p.fimg.astype(np.float64) ** 2)))
    es, _, _, _, _ = run_gpu(p)
    for ip in range(2):
        d2 = es.coarse(ip)[0]
        assert (d2 >= 0).all()
