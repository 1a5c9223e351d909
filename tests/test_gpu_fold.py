"""The backprojector's read-back and clearing over volume sizes around the fold's tiles (16 x 16 columns, 32 planes a
block): padded sizes 19, 35, 63, 67 and 99. After initMdl every voxel is exactly zero, also after an E-step scattered
into it, and a second E-step gives the first one's sums up to the order of the atomic additions (float32: 1e-5 of the
norm)."""
import numpy as np
import pytest

from problems import make_problem
from test_gpu_parity import run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,cur", [(32, 8), (32, 16), (32, 30), (32, 32), (48, 48)])
def test_clear_scatter_and_fold(box, cur):
    p = make_problem(box=box, px=4.0, order=1, offset_range_px=2, offset_step_px=1, n=4, snr=0.5, nr_blobs=20, seed=3,
                     current_size=cur)
    es, _, _, (first,), (_, (bp,)) = run_gpu(p)
    _, _, (bpd, bpw), _ = run_oracle(p)
    re, im, w = first
    err = np.sqrt(((re - bpd[0, ..., 0]) ** 2 + (im - bpd[0, ..., 1]) ** 2).sum() / (bpd[0] ** 2).sum())
    assert err <= 1e-4
    assert np.linalg.norm(w - bpw[0]) <= 1e-4 * np.linalg.norm(bpw[0])
    bp.initMdl()
    for a in bp.getMdlData():
        assert not a.any()
    es.run(p.fimg, p.fctf, p.meta)
    for a, b in zip(bp.getMdlData(), first):
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)
    for a, b in zip(bp.getMdlData(), bp.getMdlDataNoAlloc()):
        assert np.array_equal(a, b)
