"""How a run's particles are cut into chunks: the arithmetic alone, on the CPU. The per-orientation state of a chunk is
addressed by 32-bit offsets, so a chunk's orientations stay below 2^31 whatever the memory budget allows, and its
coarse intermediates (5 bytes a pose, 4 an orientation) within 24 GB.
"""
import numpy as np
import pytest

import relion_amd as ra


def _config(order, classes, range_px=0.0, local=False):
    return ra.make_config(64, 2.0, order, offset_range=2.0 * range_px, offset_step=2.0, coarse_size=24, nr_classes=classes,
                          local_search=local, sigma_ang=5.0 if local else 0.0)


def _per_particle(cfg, n, off=None):
    nd, npsi, nt = ra.sampling_counts(cfg)
    o = np.full(n, nd * npsi if not cfg.local_search else max(1, nd * npsi // 8), np.int64)
    if off is not None:
        own = np.diff(np.asarray(off, np.int64))
        o = np.where(own > 0, own, o)
    return cfg.nr_classes * o, nt


@pytest.mark.parametrize("order,classes,n", [(4, 1, 20000), (3, 4, 40000), (4, 3, 9000), (5, 1, 3000), (2, 1, 50000)])
def test_offsets_of_single_translation_searches_fit_32_bits(order, classes, n):
    cfg = _config(order, classes)
    orients, nt = _per_particle(cfg, n)
    assert nt == 1
    starts = ra.chunk_plan(cfg, n)
    assert starts[0] == 0 and starts[-1] == n and (np.diff(starts) > 0).all()
    for a, b in zip(starts[:-1], starts[1:]):
        assert orients[a:b].sum() < 2 ** 31
        assert (orients[a:b] * 9).sum() <= 24.0e9
    # the budget alone would not have kept them there (order 2 with one class fits either way)
    fixed = np.diff(starts).max() * orients[0] > 0.9 * 2 ** 31
    assert fixed or np.diff(starts).max() == 16384


def test_lists_with_exhaustive_fallbacks():
    cfg = _config(4, 2)
    n, rng = 12000, np.random.default_rng(1)
    count = np.where(np.arange(n) % 7 == 0, 0, rng.integers(1, 240000, n) // 8)
    off = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)
    orients, _ = _per_particle(cfg, n, off)
    nd, npsi, _ = ra.sampling_counts(cfg)
    starts = ra.chunk_plan(cfg, n, off)
    assert starts[0] == 0 and starts[-1] == n
    for a, b in zip(starts[:-1], starts[1:]):
        assert orients[a:b].sum() + 2 * nd * npsi < 2 ** 31


@pytest.mark.parametrize("local", [False, True])
def test_many_translations_are_cut_by_memory_and_pool(local):
    cfg = _config(3, 1, range_px=6.0, local=local)
    n = 5000
    orients, nt = _per_particle(cfg, n)
    starts = ra.chunk_plan(cfg, n, pool=2000)
    sizes = np.diff(starts)
    assert sizes[0] <= 500 and sizes.max() <= 2000  # the first chunk: a quarter of the pool
    for a, b in zip(starts[:-1], starts[1:]):
        assert (orients[a:b] * (5 * nt + 4)).sum() <= 24.0e9
    # one particle beyond every bound still makes a chunk
    big = _config(5, 1000)
    assert np.array_equal(ra.chunk_plan(big, 2), [0, 1, 2])
