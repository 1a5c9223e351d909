"""The coarse significance selection against its definition, evaluated in numpy on the same FP64 weights: the threshold
is the weight at which the descending cumulative sum first exceeds the fraction of the sum, capped by rank, and the mask,
the counts and the fine pass's poses follow from it. Exact except where a cumulative sum meets the target within the
rounding of a sum (1e-12 relative), which none of these inputs does.

The cases reach each state of the selection: all candidates in one list; more significant poses than the list holds
(4,096), found by one histogram or refined digit by digit, over several segments and down to weights that differ in their
last bits only; thousands of equal weights; the rank cap in all of them, below and above the list's length; several
segments per particle; weights spread over hundreds of binary orders by the priors.
"""
import numpy as np
import pytest

import relion_amd as ra
from problems import make_problem
from test_gpu_parity import run_gpu

pytestmark = pytest.mark.gpu


def _problem(kind):
    kw = dict(box=32, px=4.0, order=1, offset_range_px=3, offset_step_px=1, n=3, snr=0.3, nr_blobs=20, seed=21)
    if kind == "sharp":
        return make_problem(**kw)
    if kind == "sharp_capped":
        return make_problem(**dict(kw, snr=0.02, maxsig=3))
    if kind == "segments":  # 864 x 81 poses: several segments of 4,096
        return make_problem(**dict(kw, order=2, offset_range_px=5, n=2))
    caps = dict(broad_capped=5000, broad_capped_low=300, segments_broad_capped=9000, near_equal_capped=6000,
                equal_capped=5000)
    if kind.startswith("segments_broad"):
        kw.update(order=2, offset_range_px=5, n=2)
    p = make_problem(**dict(kw, snr=1e-3, maxsig=caps.get(kind, 0)))
    if "broad" in kind:  # a model noise far above the images, flat offset priors
        p.sigma2_noise = 100.0 * p.sigma2_noise
        p.cfg.sigma2_offset = 1e6
    if kind.startswith("near_equal"):  # flat priors, diff2 spread over some 1e-6: the weights share more than 20 bits
        p.sigma2_noise = 1e8 * p.sigma2_noise
        p.pdf_direction = np.full_like(p.pdf_direction, 1.0 / p.pdf_direction.size)
        p.cfg.sigma2_offset = 1e14
    if kind.startswith("equal"):  # no reference: every diff2 of a particle is the same and the weights are the priors
        p.volumes = [np.zeros_like(v) for v in p.volumes]
        p.pdf_direction = np.full_like(p.pdf_direction, 1.0 / p.pdf_direction.size)
        p.cfg.sigma2_offset = 1e6
    if kind == "far_prior":  # offset priors from exp(-600) up
        for i in range(3):
            p.meta[i].prior_offset_x = 40.0 * (i + 1)
        p.cfg.sigma2_offset = 200.0
    return p


@pytest.mark.parametrize("kind", ["sharp", "sharp_capped", "segments", "broad", "broad_capped", "broad_capped_low",
                                  "segments_broad", "segments_broad_capped", "near_equal", "near_equal_capped", "equal",
                                  "equal_capped", "far_prior"])
def test_selection_is_its_definition(kind):
    p = _problem(kind)
    es, res, _, _, _ = run_gpu(p)
    n = len(p.meta)
    biggest = 0
    for ip in range(n):
        d2, w, m, _ = es.coarse(ip)
        pos = np.sort(w[w > 0])[::-1]
        cum = np.cumsum(pos)
        total = w.sum()
        assert abs(total - res["coarse_sum_weight"][ip]) <= 1e-12 * total
        target = p.cfg.adaptive_fraction * res["coarse_sum_weight"][ip]
        k = int(np.argmax(cum > target)) if (cum > target).any() else len(pos) - 1
        if p.cfg.maximum_significants > 0:
            k = min(k, p.cfg.maximum_significants - 1)
        if kind != "equal":  # ranks among equal weights depend on the rounding of their sums
            assert res["nr_significant"][ip] == k + 1
        assert res["coarse_significant_weight"][ip] == pos[k]
        sig = (w >= pos[k]) & (w > 0)
        assert np.array_equal(m.astype(bool), sig)
        assert np.array_equal(np.unique(es.fine(ip)[0] >> 5), np.flatnonzero(sig))
        assert res["nr_fine_evaluated"][ip] == 32 * sig.sum()
        biggest = max(biggest, int(sig.sum()))
    assert (biggest > 4096) == (("broad" in kind or "equal" in kind) and kind != "broad_capped_low")
    if kind.startswith("near_equal"):
        assert 0 < pos[0] / pos[-1] - 1 < 2.0 ** -20 and np.unique(pos).size > 100
    # without the intermediates kept (weights and mask not stored): the same particles' results
    _, res2, _, _, _ = run_gpu(p, keep=False)
    for f in ("coarse_significant_weight", "nr_significant", "coarse_sum_weight", "coarse_min_diff2",
              "nr_fine_evaluated", "best_ihidden_over"):
        if f == "coarse_sum_weight":
            assert np.allclose(res[f], res2[f], rtol=1e-12, atol=0.0)
        else:
            assert np.array_equal(res[f], res2[f]), f


@pytest.mark.parametrize("order,range_px,snr", [(1, 1.0, 0.3), (1, 2.5, 0.3), (2, 3.0, 0.3), (1, 2.5, 0.003)])
def test_whole_fraction_keeps_every_positive_weight(order, range_px, snr):
    """adaptive_fraction 1: the descending sum never exceeds the whole sum, so every pose of positive weight (up to 700
    above the minimum) is significant, whatever the blocks saw first. One, three and many segments of 4,096 poses; few
    and more than 4,096 poses of positive weight; with the intermediates kept and without."""
    p = make_problem(box=32, px=4.0, order=order, offset_range_px=range_px, offset_step_px=1, n=3, snr=snr, nr_blobs=20,
                     seed=21, fraction=1.0)
    print(f"[whole] order {order} range {range_px} snr {snr}", flush=True)
    es, res, _, _, _ = run_gpu(p)
    for ip in range(3):
        _, w, m, _ = es.coarse(ip)
        pos = w[w > 0]
        assert res["nr_significant"][ip] == pos.size
        assert res["coarse_significant_weight"][ip] == pos.min()
        assert np.array_equal(m.astype(bool), w > 0)
        assert np.array_equal(np.unique(es.fine(ip)[0] >> 5), np.flatnonzero(w > 0))
    for _ in range(3):
        _, res2, _, _, _ = run_gpu(p, keep=False)
        for f in ("coarse_significant_weight", "nr_significant", "coarse_min_diff2", "nr_fine_evaluated",
                  "best_ihidden_over"):
            assert np.array_equal(res[f], res2[f]), f
