"""Packing of a prepared reference into the projector's bricks: only the bricks within the window's radius are written,
the ones beyond are cleared when they may hold something else. The packed memory is compared with the plain volume it
stands for, bit for bit, also after other data filled the projector; and the E-step's results of projectors that got there
by different ways are equal but for the order of floating-point atomics (1e-5), the samples' bricks being within reach."""
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


def _corners(plain):
    """[z][y][x] base voxels of [2][2][2] corners (re, im) of a plain volume [Z][Y][X]."""
    v = np.stack([plain.real, plain.imag], -1).astype(np.float32)
    Z, Y, X = plain.shape
    out = np.empty((Z - 1, Y - 1, X - 1, 2, 2, 2, 2), np.float32)
    for dz in range(2):
        for dy in range(2):
            for dx in range(2):
                out[..., dz, dy, dx, :] = v[dz:Z - 1 + dz, dy:Y - 1 + dy, dx:X - 1 + dx]
    return out


def _bases(pr):
    p = pr.packed()
    nz, ny, nx = p.shape[:3]
    p = p.transpose(0, 3, 1, 4, 2, 5, 6, 7, 8, 9).reshape(4 * nz, 4 * ny, 4 * nx, 2, 2, 2, 2)
    X, Y, Z = pr.dims[:3]
    return p[:Z - 1, :Y - 1, :X - 1]


@pytest.mark.parametrize("box,current,pad", [(32, 32, 2.0), (32, 18, 2.0), (40, 26, 2.0), (48, 48, 2.0), (36, 30, 1.5),
                                             (60, 60, 1.0)])
def test_packed_memory_is_the_plain_volume(box, current, pad):
    print(f"[pack] box {box} current {current} pad {pad}", flush=True)
    rng = np.random.default_rng(box)
    pr = ra.AccProjector(0)
    dims = ra.volume_dims(current, pad)
    pr.setMdlDim(*dims, pad)
    for step in ("new", "again", "noise", "window", "window again"):
        if step == "noise":
            shape = (dims[2], dims[1], dims[0])
            data = rng.normal(size=shape) + 1j * rng.normal(size=shape)
            pr.initMdl(data)
        else:
            vol = rng.normal(size=(box,) * 3).astype(np.float32)
            _, data = pr.computeFourierTransformMap(vol, current, pad, return_data=True)
            far = np.add.outer(np.add.outer(np.arange(-(dims[2] // 2), dims[2] // 2 + 1) ** 2,
                                            np.arange(-(dims[1] // 2), dims[1] // 2 + 1) ** 2), np.arange(dims[0]) ** 2)
            assert not data[far > (dims[0] - 2) ** 2].any()  # the window: radius xdim - 2
        assert np.array_equal(_bases(pr), _corners(data)), step
    pr.clear()
