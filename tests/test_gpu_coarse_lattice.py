"""Coarse squared differences over the forms the translation lattice and the pixel layout can take, against the FP64
oracle: every number of positive shifts (0 .. 9; 8 keeps the zero shift beside the matrix columns, 9 takes two column
tiles), coarse sizes whose rows end inside a step of 8 pixels, partial orientation tiles, single and several classes.

Tolerance 2e-6 relative: the stored float32 value rounds by 6e-8, and the float32 sums (at most 9 matrix steps of 4 and
17 row pairs, magnitudes below the value itself) by a few ulp each.
"""
import copy

import numpy as np
import pytest

import oracle
import relion_amd as ra
from problems import make_problem
from test_gpu_parity import rel, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp64", [False, True])
def test_matrix_instruction_lane_layout(fp64):
    rng = np.random.default_rng(0)
    for _ in range(4):
        A = rng.integers(-8, 9, size=(16, 4)).astype(np.float64)
        B = rng.integers(-8, 9, size=(4, 16)).astype(np.float64)
        assert np.array_equal(ra.selftest_mfma_lattice(A, B, fp64), A @ B)


@pytest.mark.parametrize("precision", [ra.RLN_PREC_PLAIN_FP32, ra.RLN_PREC_SPLIT_BF16])
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
def test_coarse_diff2_lattices(shifts, box, px, order, diameter, extra, precision):
    p = make_problem(box=box, px=px, order=order, offset_range_px=0.5 * shifts, offset_step_px=0.5,
                     diameter=diameter, n=3, snr=0.3, nr_blobs=20, seed=17 + shifts, **extra)
    p.cfg.precision = precision
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


def _particles_at_grid_poses(shifts, ratio, n=2):
    """Projections of the reference at coarse poses, with noise of 1 / ratio of their mean power and that noise as the
    model's: the differences of the true poses hold only the noise."""
    p = make_problem(box=32, px=4.0, order=1, offset_range_px=0.5 * shifts, offset_step_px=0.5, n=n, snr=1.0, nr_blobs=20,
                     seed=5)
    rot, tilt, psi, tx, ty = ra.sampling_grid(p.cfg)
    rng = np.random.default_rng(11 + shifts)
    img = np.zeros(p.fimg.shape[:3], complex)
    poses = []
    for i in range(n):
        d, j, t = rng.integers(rot.size), rng.integers(psi.size), rng.integers(tx.size)
        ref = oracle.project(p.volumes[0], 16, 2.0, oracle.euler(rot[d], tilt[d], psi[j]), 32)
        ref = oracle.shift_image(ref, 32, -tx[t] / 4.0, -ty[t] / 4.0)
        img[i] = ref * p.fctf[i]
        poses.append((d * psi.size + j) * tx.size + t)
    var = float(np.mean(np.abs(img) ** 2)) / ratio
    img += np.sqrt(var / 2) * (rng.normal(size=img.shape) + 1j * rng.normal(size=img.shape))
    p.fimg = np.stack([img.real, img.imag], -1).astype(np.float32)
    p.sigma2_noise = np.full(17, var)
    return p, poses


def _projection_power(p):
    """Power sum |c P|^2 of every coarse pose: the diff2 of particles that are zero."""
    q = copy.copy(p)
    q.fimg = np.zeros_like(p.fimg)
    _, _, _, dbg = run_oracle(q, (0, 1))
    return [dbg[i]["coarse_diff2"] for i in range(2)]


@pytest.mark.parametrize("shifts", [0, 3, 6, 8, 9])
@pytest.mark.parametrize("ratio", [10.0, 1e3, 1e5, 1e7])
def test_plain_diff2_of_strong_signals(ratio, shifts):
    """The plain setting's error follows the squared differences, not the signal's power: projections perturbed by e of
    their norm |cP| change D = sum |cP - y|^2 by at most 2 sqrt(D) e |cP| + (e |cP|)^2, and the float32 factors and result
    round D by a few 6e-8. e = 1e-6: the float32 reference values, sample coordinates (2e-6 of a voxel at the radius of 32
    voxels) and interpolation are off by a few 6e-8 of the values, at random over the pixels. Float32 sums of the expanded
    squares (the split setting) are off by some 1e-7 |cP|^2 and leave this bound where the power is 1,000 times D. No pose
    turns negative, which marks poses that were never evaluated."""
    p, poses = _particles_at_grid_poses(shifts, ratio)
    print(f"[strong] ratio {ratio} shifts {shifts}", flush=True)
    es, rg, _, _, _ = run_gpu(p)
    ro, _, _, dbg = run_oracle(p, (0, 1))
    power = _projection_power(p)
    for ip in range(2):
        d2, o, a = es.coarse(ip)[0].astype(np.float64), dbg[ip]["coarse_diff2"], power[ip]
        assert (d2 >= 0).all()
        bound = 2e-6 * np.sqrt(o * a) + 1e-12 * a + 5e-7 * o
        err = np.abs(d2 - o)
        print(f"[strong] worst {(err / bound).max():.3f} of the bound, at the pose {err[poses[ip]]:.2g}; float32 sums about "
              f"{1e-7 * a[poses[ip]]:.2g}; diff2 {o[poses[ip]]:.3g} (power {a[poses[ip]]:.3g})", flush=True)
        assert (err <= bound).all()
        assert np.argmin(d2) == np.argmin(o) == poses[ip]
    assert np.array_equal(rg["best_ihidden_over"], ro["best_ihidden_over"])


def test_x_phases_beyond_64_kilobytes_of_shared_memory():
    """Coarse size 656: the FP64 x phases and the staged rows take 67 KB. The two settings agree to the float32 sums' error:
    each lane adds 27,000 positive terms to the norm, which rounds at random to sqrt(27,000) 6e-8 = 1e-5 of it, and diff2
    is the norm and more for images unlike the reference."""
    box = 656
    rng = np.random.default_rng(3)
    cfg = ra.make_config(box, 1.0, 0, offset_range=1.0, offset_step=1.0, coarse_size=box, padding_factor=1.0)
    dims = ra.volume_dims(box, 1.0)
    pr, bp = ra.AccProjector(0), ra.AccBackprojector(0)
    pr.computeFourierTransformMap(rng.standard_normal((box,) * 3, np.float32), box, 1.0)
    bp.setMdlDim(*dims, 1.0)
    img = rng.standard_normal((1, box, box // 2 + 1, 2), np.float32) * np.float32(1e-3)
    ctf = np.ones((1, box, box // 2 + 1), np.float32)
    meta = (ra.ParticleMeta * 1)()
    meta[0].scale = 1.0
    out = []
    for precision in (ra.RLN_PREC_PLAIN_FP32, ra.RLN_PREC_SPLIT_BF16):
        cfg.precision = precision
        bp.initMdl()
        es = ra.ExpectationStep(cfg, 0)
        es.keep_intermediates(True)
        es.set_model([pr], [bp], np.ones(1), np.full(box // 2 + 1, 1e-6), pdf_direction=np.full((1, 12), 1 / 12))
        print(f"[lds] precision {precision}", flush=True)
        es.run(img, ctf, meta)
        out.append(es.coarse(0)[0])
        es.close()
    pr.clear()
    bp.clear()
    assert np.isfinite(out[0]).all() and (out[0] > 0).all()
    assert rel(out[1], out[0]).max() < 1e-5
