"""Packing of a prepared reference into the projector's bricks: only the bricks within the window's radius are written,
so a projector that held other data, one whose far bricks are known to be clear, and one packed whole from the same
values project the same reference. The E-step's FP32 and FP64 sums over poses are in a fixed order: results are equal
but for the posterior's floating-point atomics (1e-5)."""
import numpy as np
import pytest

import relion_amd as ra
from problems import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,current", [(32, 32), (32, 18), (40, 26), (48, 48)])
def test_windowed_pack_projects_the_same_reference(box, current):
    print(f"[pack] box {box} current {current}", flush=True)
    p = make_problem(box=box, px=4.0, order=1, offset_range_px=2, offset_step_px=1, n=4, snr=0.5, nr_blobs=20, seed=3,
                     current_size=current)
    vol = ra.synth_real_map(p.extra["spec"], 0, box)
    dims = ra.volume_dims(p.cfg.current_size)
    pr = ra.AccProjector(0)
    _, data = pr.computeFourierTransformMap(vol, current, 2.0, return_data=True)
    rng = np.random.default_rng(box)
    noise = rng.normal(size=data.shape + (2,))
    results = []
    for step in ("new", "clear", "dirty", "whole"):
        if step == "dirty":
            pr.initMdl(noise)
        if step == "whole":
            pr.initMdl(data)
        else:
            pr.computeFourierTransformMap(vol, current, 2.0)
        bp = ra.AccBackprojector(0)
        bp.setMdlDim(*dims, 2.0)
        bp.initMdl()
        es = ra.ExpectationStep(p.cfg, 0)
        es.set_model([pr], [bp], p.pdf_class, p.sigma2_noise, pdf_direction=p.pdf_direction)
        res, _ = es.run(p.fimg, p.fctf, p.meta)
        results.append(res)
        es.close()
        bp.clear()
    for res in results[1:]:
        assert np.array_equal(res["best_ihidden_over"], results[0]["best_ihidden_over"])
        assert np.allclose(res["dLL"], results[0]["dLL"], rtol=1e-5)
        assert np.allclose(res["pmax"], results[0]["pmax"], rtol=1e-5)
    pr.clear()
