"""Measured cases of the E-step framework: inputs, one pass through the public entry points, the work a pass cannot do
without, and the results in 64 bits by plain torch.

Six families, each one path that a program using this package takes:

- ``estep``: one expectation step over a set of particles and the map it ends in, as a refinement iteration does it:
  the backprojectors are cleared, ``ExpectationStep.run`` searches every particle's poses, and
  ``AccBackprojector.reconstruct`` (relion_refine's default, without gridding iterations) turns the sums into the
  classes' maps. With ``renew`` the iteration starts from the real-space map: reference preparation and ``set_model``
  are part of the pass.
- ``imgprep``: particle images prepared for the E-step (mask, transforms, spectra, CTF), device to device as a
  pipeline does it, or host to host.
- ``refprep``: a real-space map prepared into the projector (its power spectrum, and for small boxes the padded
  transform, come back).
- ``recon``: a map reconstructed from accumulated sums with the gridding iterations and the MAP term.
- ``train``: one epoch of the pose proposal's training, ending with its parameters.
- ``predict``: the pose proposal's top bins for a set of particles.

Particles are noisy projections of maps of Gaussian blobs under a CTF, as in the tests and the benchmark.
"""
import math

import numpy as np
import torch

import relion_amd as ra
from relion_amd.proposal import PoseProposal

PAD = 2.0
LIST_BINS = 16          # orientation lists: bins per particle, as the proposal's top 16
PREDICT_TOPK = 16
TRAIN_LR = 3e-5
GRID_ITERATIONS = 10    # relion's default of max_iter_preweight
TAU2_FUDGE = 4.0


# ------------------------------------------------------------------------------------------------
# cases
# ------------------------------------------------------------------------------------------------
def _estep(name=None, family="estep", box=64, cur=0, px=2.0, order=2, classes=1, n=8, search="global", split=False,
           range_px=5.0, step_px=1.0, diameter=100.0, snr=0.1, blobs=40, scale=False, nomask=False, renew=False):
    c = dict(family=family, box=box, cur=cur or box, px=px, order=order, classes=classes, n=n, search=search,
             split=split, range_px=range_px, step_px=step_px, diameter=diameter, snr=snr, blobs=blobs, scale=scale,
             nomask=nomask, renew=renew)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a handful of particles at a small box: what an interactive check or a test asks for; launches and latency
        _estep("estep_box64_8_particles", n=8),
        # the first iteration of a 3-D refinement at relion_refine's defaults (7.5 degrees, 5 px range, 2 px step), the
        # reference low-passed to a small current size: reference preparation, model, E-step and reconstruction
        _estep("first_iteration_box128", box=128, cur=58, px=2.0, order=2, n=1000, range_px=5.0, step_px=2.0,
               diameter=180.0, snr=0.05, blobs=60, renew=True),
        # an exhaustive search in the default precision at a fine angular step
        _estep("estep_global_box128_plain", box=128, px=2.0, order=3, n=101, range_px=6.0, step_px=1.0, diameter=180.0,
               snr=0.05, blobs=60),
        # 3-D classification: four classes, exhaustive, split precision (the benchmark's classification leg)
        _estep("classification_box128_k4_split", box=128, px=2.0, order=3, classes=4, n=151, range_px=6.0, step_px=1.0,
               diameter=180.0, snr=0.05, blobs=60, split=True),
        # the local searches of late refinement in the default precision: current size below the box, group scale
        # corrections, separate unmasked images
        _estep("estep_local_box192_plain", box=192, cur=160, px=1.3, order=3, n=1501, search="local", range_px=5.0,
               step_px=0.75, diameter=180.0, snr=0.05, blobs=100, scale=True, nomask=True),
        # proposal-seeded search at the benchmark's headline geometry: short orientation lists, few exhaustive fallbacks
        _estep("estep_lists_box256_split", box=256, px=1.0, order=3, n=2048, search="lists", range_px=4.0, step_px=0.5,
               diameter=200.0, snr=0.03, blobs=150, split=True),
        # image preparation of a large set, noise background (relion's default), device to device
        dict(name="imgprep_box256_noise", family="imgprep", box=256, cur=256, px=1.0, n=2048, diameter=200.0,
             noise=True, device=True),
        # a small set of an uneven box on host arrays, zero background, window below the box
        dict(name="imgprep_box90_host", family="imgprep", box=90, cur=60, px=2.7, n=37, diameter=180.0, noise=False,
             device=False),
        # reference preparation at the benchmark's size
        dict(name="refprep_box256", family="refprep", box=256, cur=256, px=1.0, blobs=150, data=False),
        # reconstruction with the gridding iterations and the MAP term
        _estep("recon_gridding_box128", family="recon", box=128, cur=100, px=2.0, order=2, n=200, range_px=5.0,
               step_px=2.0, diameter=180.0, snr=0.1, blobs=60),
        # the proposal's training: 16 batches of 256 and the parameters read back
        dict(name="proposal_train_16_batches", family="train", box=64, px=4.0, n=4096, batch=256),
        # the proposal's inference at the benchmark's box
        dict(name="proposal_predict_box256", family="predict", box=256, px=1.0, n=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even(v):
    return 2 * int(round(v / 2))


def _estep_cost(c):
    """Coarse contraction plus fine sampling, in multiply-adds."""
    nd, npsi, nt, sc, poses = _search_size(c)
    return c["n"] * (poses * sc * (sc / 2 + 1) * 2 + 400.0 * c["cur"] * (c["cur"] / 2 + 1))


def _draw_estep(rng):
    limit = _estep_cost(listed()[3])
    while True:
        box = _even(_log_int(rng, 48, 256))
        px = rng.choice([1.0, 1.3, 2.0, 2.7, 4.0])
        search = rng.choice(["global", "global", "local", "lists"])
        classes = rng.choice([1, 1, 1, 2, 3, 4]) if box <= 128 else 1
        order = rng.choice([1, 2, 2, 3]) if search == "global" else rng.choice([2, 3])
        step = rng.choice([0.5, 0.75, 1.0, 1.5, 2.0])
        reach = step * rng.uniform(2.0, 7.0)
        cur = box if rng.random() < 0.5 else max(32, _even(box * rng.uniform(0.45, 1.0)))
        c = _estep(box=box, cur=cur, px=px, order=order, classes=classes, n=_log_int(rng, 1, 3000), search=search,
                   split=rng.random() < 0.4, range_px=round(reach, 2), step_px=step,
                   diameter=round(box * px * rng.uniform(0.6, 0.85), 1), snr=round(rng.uniform(0.04, 0.15), 3),
                   blobs=rng.randint(40, 150), scale=rng.random() < 0.3, nomask=rng.random() < 0.4,
                   renew=rng.random() < 0.3)
        if c["snr"] * c["cur"] < 5.0:
            c["snr"] = round(5.0 / c["cur"], 3)
        if _estep_cost(c) <= limit:
            return c


def draw(rng):
    kind = rng.choice(["estep"] * 7 + ["imgprep"] * 2 + ["refprep", "recon", "train", "predict"])
    if kind == "estep":
        return _draw_estep(rng)
    if kind == "imgprep":
        box = _even(_log_int(rng, 48, 360))
        n = min(_log_int(rng, 1, 2048), int(2048 * 256 * 256 / (box * box)))
        device = rng.random() < 0.6
        if not device:
            n = min(n, 200)
        px = rng.choice([1.0, 1.3, 2.7])
        return dict(family="imgprep", box=box, cur=box if rng.random() < 0.5 else max(24, _even(box * rng.uniform(0.4, 1))),
                    px=px, n=n, diameter=round(box * px * rng.uniform(0.6, 0.9), 1), noise=rng.random() < 0.5,
                    device=device)
    if kind == "refprep":
        box = _even(_log_int(rng, 40, 256))
        return dict(family="refprep", box=box, cur=box if rng.random() < 0.5 else max(24, _even(box * rng.uniform(0.4, 1))),
                    px=rng.choice([1.0, 2.0]), blobs=rng.randint(40, 150), data=box <= 72)
    if kind == "recon":
        box = _even(_log_int(rng, 40, 128))
        return _estep(family="recon", box=box, cur=max(24, _even(box * rng.uniform(0.4, 1.0))), px=rng.choice([2.0, 2.7]),
                      order=2, n=_log_int(rng, 20, 200), range_px=4.0, step_px=2.0, diameter=1.4 * box,
                      snr=round(rng.uniform(0.1, 0.2), 3), blobs=60)
    if kind == "train":
        batch = rng.choice([64, 128, 256, 200])
        return dict(family="train", box=64, px=4.0, n=batch * rng.randint(2, 16) + rng.randint(0, 63), batch=batch)
    return dict(family="predict", box=_even(_log_int(rng, 64, 256)), px=rng.choice([1.0, 2.0]), n=_log_int(rng, 1, 4096))


# ------------------------------------------------------------------------------------------------
# sampling, as HEALPix (Gorski et al. 2005) and relion define it
# ------------------------------------------------------------------------------------------------
def _healpix(order):
    """(rot, tilt) in degrees of every NEST pixel."""
    nside = 1 << order
    p = np.arange(12 * nside * nside, dtype=np.int64)
    face, within = p >> (2 * order), p & (nside * nside - 1)
    ix = np.zeros_like(p)
    iy = np.zeros_like(p)
    for b in range(order):
        ix |= ((within >> (2 * b)) & 1) << b
        iy |= ((within >> (2 * b + 1)) & 1) << b
    ring = (2 + face // 4) * nside - ix - iy - 1
    north, south = ring < nside, ring > 3 * nside
    nr = np.where(north, ring, np.where(south, 4 * nside - ring, nside))
    z = np.where(north, 1.0 - nr ** 2 / (3.0 * nside ** 2),
                 np.where(south, nr ** 2 / (3.0 * nside ** 2) - 1.0, (2 * nside - ring) * 2.0 / (3.0 * nside)))
    shift = np.where(north | south, 0, (ring - nside) & 1)
    first = np.array([1, 3, 5, 7, 0, 2, 4, 6, 1, 3, 5, 7])[face]
    j = (first * nr + ix - iy + 1 + shift) // 2
    j = np.where(j > 4 * nside, j - 4 * nside, np.where(j < 1, j + 4 * nside, j))
    rot = np.degrees((j - 0.5 * (shift + 1)) * (0.5 * np.pi) / nr)
    rot = np.where(rot > 180.0, rot - 360.0, rot)
    return rot, np.degrees(np.arccos(z))


def _rotations(rot, tilt, psi):
    """Rz(psi) Ry(tilt) Rz(rot) of angles in degrees, [..., 3, 3]."""
    a, b, g = (np.radians(np.asarray(v, np.float64)) for v in (rot, tilt, psi))
    a, b, g = np.broadcast_arrays(a, b, g)
    one, nul = np.ones_like(a), np.zeros_like(a)

    def mat(*v):
        return np.stack(v, -1).reshape(a.shape + (3, 3))

    def rz(t):
        return mat(np.cos(t), np.sin(t), nul, -np.sin(t), np.cos(t), nul, nul, nul, one)

    ry = mat(np.cos(b), nul, -np.sin(b), nul, one, nul, np.sin(b), nul, np.cos(b))
    return rz(g) @ ry @ rz(a)


def _translations(c):
    """Coarse translations in Angstrom [NT][2]: the lattice points of a disc, x slow."""
    step, reach = c["step_px"] * c["px"], c["range_px"] * c["px"]
    m = math.ceil(reach / step)
    return np.array([(i * step, j * step) for i in range(-m, m + 1) for j in range(-m, m + 1)
                     if (i * step) ** 2 + (j * step) ** 2 < reach * reach + 0.001])


def _n_psi(order):
    return 6 << order


def _sigma_ang(c):
    return 30.0 / (1 << c["order"]) * 2.0  # two coarse steps of half width 360 / (6 2^order) / 2


def _coarse_size(c):
    step = 360.0 / _n_psi(c["order"])
    res = step / 360.0 * math.pi * c["diameter"] / 1.2
    return min(2 * math.ceil(c["px"] * c["box"] / res), c["cur"])


def _search_size(c):
    """(directions, psi angles, translations, coarse size, coarse poses of a particle on average)."""
    nd, npsi, nt, sc = 12 << (2 * c["order"]), _n_psi(c["order"]), len(_translations(c)), _coarse_size(c)
    o = nd * npsi
    if c["search"] == "local":
        s = 3.0 * _sigma_ang(c)
        o *= 0.5 * (1.0 - math.cos(math.radians(min(180.0, s)))) * min(1.0, s / 180.0)
    elif c["search"] == "lists":
        o = min(o, 12 * LIST_BINS) + o * (c["n"] // 1000) / c["n"]
    return nd, npsi, nt, sc, c["classes"] * o * nt


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
def _blobs(c, seed, k):
    """Blob set of class k: centres (pixels from the centre), sigma (pixels), amplitude; classes share 30%."""
    out = []
    n = c["blobs"]
    shared = int(0.3 * n) if c.get("classes", 1) > 1 else 0
    for which, m in ((99, shared), (k, n - shared)):
        g = np.random.default_rng([seed, 1, which])
        d = g.normal(size=(m, 3))
        d *= (0.375 * c["box"] * g.random((m, 1)) ** (1.0 / 3.0)) / np.linalg.norm(d, axis=1, keepdims=True)
        out.append(np.concatenate([d, g.uniform(1.5, 3.0, (m, 1)), g.uniform(0.5, 1.0, (m, 1))], 1))
    return np.concatenate(out)


def _real_map(c, seed, k, dev):
    """The class's map [box]^3 (z, y, x), origin at box / 2, float32 on the device."""
    b = torch.tensor(_blobs(c, seed, k), device=dev)
    x = torch.arange(c["box"], device=dev, dtype=torch.float64) - c["box"] // 2
    g = [torch.exp(-(x[None, :] - b[:, i:i + 1]) ** 2 / (2 * b[:, 3:4] ** 2)) for i in range(3)]
    zy = (g[2] * b[:, 4:5])[:, :, None] * g[1][:, None, :]
    return (zy.reshape(len(b), -1).T.contiguous() @ g[0]).reshape((c["box"],) * 3).float().contiguous()


def _freq(s, dev, dtype=torch.float64):
    y = torch.arange(s, device=dev, dtype=dtype)
    return torch.where(y > s // 2, y - s, y), torch.arange(s // 2 + 1, device=dev, dtype=dtype)


def _ctf_images(c, defocus, s, dev):
    """CTF images float64 [n][s][s/2+1] of (defocus U, defocus V, azimuth in degrees), 300 kV, Cs 2.7 mm, Q0 0.1."""
    y, x = _freq(s, dev)
    d = torch.as_tensor(defocus, device=dev, dtype=torch.float64)
    a = torch.deg2rad(d[:, 2])
    axx = -(d[:, 0] * a.cos() ** 2 + d[:, 1] * a.sin() ** 2)
    axy = -(d[:, 0] - d[:, 1]) * a.sin() * a.cos()
    ayy = -(d[:, 0] * a.sin() ** 2 + d[:, 1] * a.cos() ** 2)
    f = 1.0 / (c["box"] * c["px"])
    X, Y = x[None, None, :] * f, y[None, :, None] * f
    u2 = X * X + Y * Y
    lam = 12.2643247 / math.sqrt(300e3 * (1.0 + 300e3 * 0.978466e-6))
    q = (axx[:, None, None] * X * X + 2.0 * axy[:, None, None] * X * Y + ayy[:, None, None] * Y * Y)
    gamma = math.pi * lam * q + math.pi / 2 * 2.7e7 * lam ** 3 * u2 * u2 - math.atan(0.1 / math.sqrt(1 - 0.01))
    return -torch.sin(gamma)


def _particles(c, seed, dev):
    """n particles at current size on the device: images complex64, CTFs float32, the mean noise variance of a Fourier
    component and what was drawn for them."""
    n, s, N, K = c["n"], c["cur"], float(c["box"]), c.get("classes", 1)
    g = np.random.default_rng([seed, 2])
    kc = g.integers(0, K, n)
    rot, psi = g.uniform(-180.0, 180.0, n), g.uniform(0.0, 360.0, n)
    tilt = np.degrees(np.arccos(g.uniform(-1.0, 1.0, n)))
    reach = min(3.0, 0.6 * c.get("range_px", 5.0))
    shift = g.uniform(-reach, reach, (n, 2))
    defU = g.uniform(8000.0, 25000.0, n)
    defocus = np.stack([defU, defU - g.uniform(0.0, 300.0, n), g.uniform(0.0, 180.0, n)], 1)
    scale = g.uniform(0.8, 1.2, n) if c.get("scale") else np.ones(n)
    A = _rotations(rot, tilt, psi)
    y, x = _freq(s, dev, torch.float32)
    r2 = y[:, None] ** 2 + x[None, :] ** 2
    inside = (r2 <= (s // 2) ** 2)
    img = torch.empty((n, s, s // 2 + 1), dtype=torch.complex64, device=dev)
    ctf = torch.empty((n, s, s // 2 + 1), dtype=torch.float32, device=dev)
    tg = torch.Generator(device=dev)
    tg.manual_seed(seed * 7 + 3)
    blobs = [_blobs(c, seed, k) for k in range(K)]
    var = 0.0
    step = max(1, int(2.0e8 / (blobs[0].shape[0] * s * 12)))
    for i0 in range(0, n, step):
        i1 = min(n, i0 + step)
        b = torch.tensor(np.stack([blobs[k] for k in kc[i0:i1]]), device=dev)
        uv = b[:, :, :3] @ torch.tensor(A[i0:i1, :2].transpose(0, 2, 1).copy(), device=dev)  # [m][blob][2]
        uv = (uv - torch.tensor(shift[i0:i1], device=dev)[:, None, :])
        sg, amp = b[:, :, 3], b[:, :, 4] * (2 * math.pi * b[:, :, 3] ** 2) ** 1.5 / (N * N)

        def axis(k, u, w):
            ph = k.double() * u[..., None] / N
            ph = (-2 * math.pi * (ph - torch.round(ph))).float()
            env = torch.exp(-2 * math.pi ** 2 * (sg ** 2)[..., None] * (k.double() / N) ** 2) * w[..., None]
            return torch.polar(env.float(), ph)

        ex, ey = axis(x, uv[..., 0], amp), axis(y, uv[..., 1], torch.ones_like(amp))
        m = torch.matmul(ey.transpose(1, 2).contiguous(), ex)
        cv = _ctf_images(c, defocus[i0:i1], s, dev).float()
        m = m * cv * torch.tensor(scale[i0:i1], device=dev, dtype=torch.float32)[:, None, None]
        p = (m.abs() ** 2 * inside).sum((1, 2)) / inside.sum()
        v = p / (2.0 * c.get("snr", 0.05))
        var += float(v.double().sum())
        noise = torch.randn((i1 - i0, s, s // 2 + 1, 2), generator=tg, device=dev)
        img[i0:i1] = m + torch.view_as_complex(noise) * v.sqrt()[:, None, None]
        ctf[i0:i1] = cv
    ps = g.normal(0.0, 2.0, (n, 3))
    prior = np.stack([rot + ps[:, 0], np.clip(tilt + ps[:, 1], 0.0, 180.0), np.mod(psi + ps[:, 2], 360.0)], 1)
    drawn = dict(rot=rot, tilt=tilt, psi=psi, shift=shift, kc=kc, prior=prior, scale=scale, g=g)
    return img, ctf, var / n, drawn


def _lists(c, d, seed):
    """Orientation lists as the proposal's top bins make them: the bin of the true pose and 15 others, each four
    directions by three psi angles; every thousandth particle keeps the exhaustive grid (an empty list)."""
    g = np.random.default_rng([seed, 4])
    prot, ptilt = _healpix(c["order"] - 1)
    npsi, nd, n = _n_psi(c["order"]), 12 << (2 * c["order"]), c["n"]

    def unit(r, t):
        r, t = np.radians(r), np.radians(t)
        return np.stack([np.sin(t) * np.cos(r), np.sin(t) * np.sin(r), np.cos(t)], -1)

    bins_d = g.integers(0, nd // 4, (n, LIST_BINS))
    bins_p = g.integers(0, npsi // 2, (n, LIST_BINS))
    bins_d[:, 0] = np.argmax(unit(d["rot"], d["tilt"]) @ unit(prot, ptilt).T, 1)
    bins_p[:, 0] = np.round(d["psi"] / (720.0 / npsi)).astype(np.int64) % (npsi // 2)
    dirs = 4 * bins_d[:, :, None, None] + np.arange(4)[None, None, :, None]
    psis = (2 * bins_p[:, :, None, None] + np.arange(-1, 2)[None, None, None, :]) % npsi
    full = (dirs * npsi + psis).reshape(n, -1)
    sets = [np.unique(row).astype(np.int32) for row in full]
    for i in range(n // 1000):
        sets[(1000 * i + 500) % n] = np.zeros(0, np.int32)
    return sets


def _estep_problem(c, seed, dev):
    """Everything an E-step needs as plain data: maps, images, model spectra, per-particle metadata, lists."""
    p = dict(case=c)
    p["maps"] = [_real_map(c, seed, k, dev) for k in range(c["classes"])]
    p["fimg"], p["fctf"], var, d = _particles(c, seed, dev)
    ns = c["box"] // 2 + 1
    p["sigma2"] = var * (1.0 + 0.2 * np.cos(np.arange(ns) / 3.0))
    g = np.random.default_rng([seed, 3])
    nd = 12 << (2 * c["order"])
    p["pdf_class"] = np.full(c["classes"], 1.0 / c["classes"])
    p["pdf_direction"] = (1.0 + 0.1 * g.random((c["classes"], nd))) / nd / c["classes"]
    p["dvp"] = np.where(np.arange(ns) < 0.7 * ns, 10.0, 1.0)[None, :].repeat(c["classes"], 0) if c["scale"] else None
    p["nomask"] = (p["fimg"] * 1.05).contiguous() if c["nomask"] else None
    meta = (ra.ParticleMeta * c["n"])()
    old, pri = np.zeros((c["n"], 2)), np.zeros((c["n"], 2))
    if c["scale"]:
        old, pri = g.integers(-1, 2, (c["n"], 2)).astype(float), g.uniform(-1.0, 1.0, (c["n"], 2))
    xi2 = g.uniform(0.0, 50.0, c["n"]) if c["cur"] < c["box"] else np.zeros(c["n"])
    for i in range(c["n"]):
        m = meta[i]
        m.old_offset_x, m.old_offset_y = old[i]
        m.prior_offset_x, m.prior_offset_y = pri[i]
        m.prior_rot, m.prior_tilt, m.prior_psi = d["prior"][i]
        m.scale, m.highres_Xi2 = d["scale"][i], xi2[i]
    p.update(meta=meta, old=old, pri=pri, xi2=xi2, scale=d["scale"], prior=d["prior"])
    p["sets"] = _lists(c, d, seed) if c["search"] == "lists" else None
    return p


def _estep_config(c):
    sig = _sigma_ang(c) if c["search"] == "local" else 0.0
    return ra.make_config(c["box"], c["px"], c["order"], offset_range=c["range_px"] * c["px"],
                          offset_step=c["step_px"] * c["px"], coarse_size=_coarse_size(c), current_size=c["cur"],
                          nr_classes=c["classes"], padding_factor=PAD, local_search=c["search"] == "local",
                          sigma_ang=sig, do_scale_correction=c["scale"],
                          precision=ra.RLN_PREC_SPLIT_BF16 if c["split"] else ra.RLN_PREC_PLAIN_FP32)


def _set_model(st):
    p = st["p"]
    for k, pr in enumerate(st["pr"]):
        pr.computeFourierTransformMap(p["maps"][k].data_ptr(), p["case"]["cur"], PAD, ori_size=p["case"]["box"],
                                      on_device=True)
    st["es"].set_model(st["pr"], st["bp"], p["pdf_class"], p["sigma2"],
                       pdf_direction=None if p["case"]["search"] == "local" else p["pdf_direction"],
                       data_vs_prior=p["dvp"])


def _prepare_estep(c, seed, dev):
    p = _estep_problem(c, seed, dev)
    dims = ra.volume_dims(c["cur"], PAD)
    st = dict(family=c["family"], p=p, pr=[], bp=[])
    for _ in range(c["classes"]):
        pr, bp = ra.AccProjector(0), ra.AccBackprojector(0)
        pr.setMdlDim(*dims, PAD)
        bp.setMdlDim(*dims, PAD)
        bp.initMdl()
        st["pr"].append(pr)
        st["bp"].append(bp)
    st["es"] = ra.ExpectationStep(_estep_config(c), 0)
    torch.cuda.synchronize()
    _set_model(st)
    st["out"] = torch.zeros((c["classes"],) + (c["box"],) * 3, device=dev)
    if p["sets"] is not None:
        cnt = np.array([len(s) for s in p["sets"]])
        st["off"] = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
        st["og"] = np.concatenate(p["sets"]).astype(np.int32)
    return st


def _run_estep_only(st):
    p = st["p"]
    if p["sets"] is not None:
        st["es"].set_orientation_lists(st["off"], st["og"])
    return st["es"].run(p["fimg"].data_ptr(), p["fctf"].data_ptr(), p["meta"],
                        fimg_nomask=None if p["nomask"] is None else p["nomask"].data_ptr(), on_device=True)


#: per-particle results compared as numbers (the angles and offsets are the decoding of best_ihidden_over)
RESULTS = ("pmax", "nr_significant", "dLL", "sum_weight", "min_diff2", "wsum_norm_correction", "signal_product",
           "reference_power")


def _run_estep(st):
    c = st["p"]["case"]
    if c["renew"]:
        _set_model(st)
    for bp in st["bp"]:
        bp.initMdl()
    res, ws = _run_estep_only(st)
    for k, bp in enumerate(st["bp"]):
        bp.reconstruct(c["box"], do_map=False, skip_gridding=True, out_address=st["out"][k].data_ptr())
    out = {f: res[f] for f in RESULTS}
    out["best"] = res["best_ihidden_over"]
    out.update({"wsum_" + f: np.asarray(v) for f, v in ws.items()})
    out["map"] = st["out"]
    return out


def _tau2(p):
    ns = p["case"]["box"] // 2 + 1
    return 2.0 * p["sigma2"].mean() * np.exp(-np.arange(ns) / (0.2 * ns))


def _prepare_recon(c, seed, dev):
    st = _prepare_estep(c, seed, dev)
    _run_estep_only(st)
    st["tau2"] = _tau2(st["p"])
    return st


def _run_recon(st):
    c = st["p"]["case"]
    st["bp"][0].reconstruct(c["box"], max_iter_preweight=GRID_ITERATIONS, do_map=True, tau2=st["tau2"],
                            tau2_fudge=TAU2_FUDGE, normalise=float(c["n"]), skip_gridding=False,
                            out_address=st["out"][0].data_ptr())
    return {"map": st["out"]}


def _prep_inputs(c, seed, dev):
    """Real-space particles: noise with a blob of signal, and their metadata."""
    n, N = c["n"], c["box"]
    tg = torch.Generator(device=dev)
    tg.manual_seed(seed * 5 + 1)
    x = torch.arange(N, device=dev, dtype=torch.float32) - N // 2
    blob = torch.exp(-(x[:, None] ** 2 + x[None, :] ** 2) / (2 * (0.15 * N) ** 2))
    img = torch.randn((n, N, N), generator=tg, device=dev) + 0.3 * blob
    g = np.random.default_rng([seed, 5])
    defU = g.uniform(8000.0, 25000.0, n)
    m = dict(norm_correction=g.uniform(0.8, 1.2, n), old_offset_x=g.uniform(-4.0, 4.0, n),
             old_offset_y=g.uniform(-4.0, 4.0, n), defocus_u=defU, defocus_v=defU - g.uniform(0.0, 300.0, n),
             defocus_angle=g.uniform(0.0, 180.0, n), bfactor=np.zeros(n), kfactor=np.ones(n), phase_shift=np.zeros(n),
             part_id=np.arange(n))
    sigma2 = (1.0 + 0.3 * np.cos(np.arange(N // 2 + 1) / 5.0)) / (2.0 * N * N)
    return img, m, sigma2


def _prepare_imgprep(c, seed, dev):
    img, m, sigma2 = _prep_inputs(c, seed, dev)
    ip = ra.ImagePreparation(c["box"], c["cur"], c["px"], c["diameter"], zero_mask=not c["noise"], random_seed=seed,
                             avg_norm_correction=1.0)
    ip.set_sigma2_noise(sigma2)
    metas = ip.meta_array([{k: (int(v[i]) if k == "part_id" else float(v[i])) for k, v in m.items()}
                           for i in range(c["n"])])
    st = dict(family="imgprep", c=c, ip=ip, metas=metas)
    if c["device"]:
        s = c["cur"]
        st["img"] = img
        st["out"] = [torch.zeros((c["n"], s, s // 2 + 1), dtype=t, device=dev)
                     for t in (torch.complex64, torch.complex64, torch.float32)]
    else:
        st["img"] = img.cpu().numpy()
    return st


def _run_imgprep(st):
    if not st["c"]["device"]:
        return st["ip"].getFourierTransformsAndCtfs(st["img"], st["metas"])
    a, b, f = st["out"]
    hx, power, off = st["ip"].run_device(st["c"]["n"], st["img"].data_ptr(), st["metas"], a.data_ptr(), b.data_ptr(),
                                         f.data_ptr())
    return dict(fimg=a, fimg_nomask=b, fctf=f, highres_Xi2=hx, power=power, old_offset=off)


def _prepare_refprep(c, seed, dev):
    st = dict(family="refprep", c=c, map=_real_map(c, seed, 0, dev), pr=ra.AccProjector(0))
    st["pr"].setMdlDim(*ra.volume_dims(c["cur"], PAD), PAD)
    return st


def _run_refprep(st):
    c = st["c"]
    r = st["pr"].computeFourierTransformMap(st["map"].data_ptr(), c["cur"], PAD, ori_size=c["box"], on_device=True,
                                            return_data=c["data"])
    return dict(power=r[0], data=r[1]) if c["data"] else dict(power=r)


NET = dict(window=64, channels=64, healpix_order=2, n_psi_bins=24)  # the benchmark's network


def _net_params(seed, dev):
    """He-normal convolutions and the fully connected layer in the library's parameter order, float32."""
    tg = torch.Generator(device=dev)
    tg.manual_seed(seed * 11 + 5)
    parts, cin, C = [], 1, NET["channels"]
    for _ in range(6):
        kp = 16 if cin == 1 else 9 * cin
        w = torch.zeros((C, kp), device=dev)
        w[:, :9 * cin] = torch.randn((C, 9 * cin), generator=tg, device=dev) * math.sqrt(2.0 / (9 * cin))
        parts += [w.reshape(-1), torch.zeros(C, device=dev)]
        cin = C
    F, nb = C * (NET["window"] // 8) ** 2, (12 << (2 * NET["healpix_order"])) * NET["n_psi_bins"]
    parts += [(torch.randn((nb, F), generator=tg, device=dev) / math.sqrt(F)).reshape(-1), torch.zeros(nb, device=dev)]
    return torch.cat(parts).cpu().numpy()


def _net_particles(c, seed, dev):
    cc = dict(c, cur=c["box"], blobs=60, snr=0.1)
    img, ctf, _, d = _particles(cc, seed, dev)
    return img, ctf, np.stack([d["rot"], d["tilt"], d["psi"]], 1)


def _prepare_net(c, seed, dev):
    img, ctf, poses = _net_particles(c, seed, dev)
    pp = PoseProposal(seed=seed, **NET)
    pp.set_params(_net_params(seed, dev))
    if c["family"] == "train":
        torch.cuda.synchronize()
        pp.add_images(img.data_ptr(), ctf.data_ptr(), c["box"], poses, on_device=True)
    return dict(family=c["family"], c=c, pp=pp, img=img, ctf=ctf)


def _run_train(st):
    loss = st["pp"].train(epochs=1, batch=st["c"]["batch"], lr=TRAIN_LR)
    return dict(loss=loss, params=st["pp"].get_params())


def _run_predict(st):
    c = st["c"]
    bins, probs = st["pp"].predict(st["img"].data_ptr(), st["ctf"].data_ptr(), c["n"], c["box"], topk=PREDICT_TOPK,
                                   on_device=True)
    return dict(bins=bins, probs=probs)


_PREPARE = dict(estep=_prepare_estep, imgprep=_prepare_imgprep, refprep=_prepare_refprep, recon=_prepare_recon,
                train=_prepare_net, predict=_prepare_net)
_RUN = dict(estep=_run_estep, imgprep=_run_imgprep, refprep=_run_refprep, recon=_run_recon, train=_run_train,
            predict=_run_predict)


def prepare(case, seed):
    return _PREPARE[case["family"]](case, seed, torch.device("cuda:0"))


def run(state):
    return _RUN[state["family"]](state)


# ------------------------------------------------------------------------------------------------
# work and tolerance
# ------------------------------------------------------------------------------------------------
def _net_flops():
    """Multiply-adds times two of one image through the network, forward."""
    C, W = NET["channels"], NET["window"]
    conv = 2.0 * C * 9 * (W * W + C * sum((W >> k) ** 2 for k in (1, 1, 2, 2, 3)))
    return conv + 2.0 * C * (W // 8) ** 2 * (12 << (2 * NET["healpix_order"])) * NET["n_psi_bins"]


def work(case):
    c, f = case, case["family"]
    if f in ("estep", "recon"):
        s, N = c["cur"], c["box"]
        S = 2 * (s + 1) + 1
        half = S * S * (S // 2 + 1)
        if f == "recon":
            # the sums read, the map written; each gridding iteration is a transform there and one back
            fft = 2.5 * S ** 3 * math.log2(S ** 3)
            return dict(bytes=12.0 * half + 4.0 * N ** 3, flops=(2 * GRID_ITERATIONS) * fft)
        nd, npsi, nt, sc, poses = _search_size(c)
        pix = s * (s // 2 + 1)
        # images and CTF read, the reference sampled, the sums and maps written; the coarse cross term, and at least
        # one coarse pose's 8 orientations and 4 shifts at the current size
        return dict(bytes=c["n"] * pix * (20.0 if c["nomask"] else 12.0) + c["classes"] * (20.0 * half + 4.0 * N ** 3),
                    flops=c["n"] * (4.0 * poses * sc * (sc // 2 + 1) + 8.0 * pix * 60.0))
    if f == "imgprep":
        N, s = c["box"], c["cur"]
        fft = 2.5 * N * N * math.log2(N * N)
        return dict(bytes=c["n"] * (4.0 * N * N + 20.0 * s * (s // 2 + 1)), flops=c["n"] * fft * (3 if c["noise"] else 2))
    if f == "refprep":
        N, S, P = c["box"], 2 * (c["cur"] + 1) + 1, 2 * c["box"]
        return dict(bytes=4.0 * N ** 3 + 8.0 * S * S * (S // 2 + 1), flops=2.5 * P ** 3 * math.log2(P ** 3))
    nb = (12 << (2 * NET["healpix_order"])) * NET["n_psi_bins"]
    params = nb * (NET["channels"] * (NET["window"] // 8) ** 2 + 1) + 5 * NET["channels"] * 9 * NET["channels"]
    if f == "train":
        steps = c["n"] // c["batch"]
        # each step reads and writes the weights and both moments; every image once forward, twice backward
        return dict(bytes=steps * params * 24.0 + c["n"] * 2.0 * NET["window"] ** 2,
                    flops=3.0 * _net_flops() * steps * c["batch"])
    w = NET["window"]
    return dict(bytes=c["n"] * 12.0 * w * (w // 2 + 1) + 2.0 * params, flops=c["n"] * _net_flops())


def tolerance(case):
    f = case["family"]
    if f == "estep":
        # against 64 bits the results are within 5e-5 in the default precision and 1e-4 in split precision, unless the
        # rounding of a coarse squared difference moves a pose across the significance threshold: one particle of 4096
        # did in split precision, which moved the map by 0.0099 and that particle's weights by their own size
        return {"rel": 0.02, "max": 0.9, "differ": 0.01}
    if f == "imgprep":
        return {"rel": 1e-6, "max": 5e-5}  # float32 transforms: 2e-7 from 64 bits
    if f == "refprep":
        return {"rel": 1e-6, "max": 5e-5}  # float32 transform: 3e-8 in the spectrum
    if f == "recon":
        return {"rel": 1e-5, "max": 1e-3}  # float32 sums: 2e-6 from 64 bits
    if f == "train":
        return {"rel": 1e-3, "max": 0.1}  # bf16 products; another order of the sums moves the parameters by 5e-5
    return {"rel": 1e-2, "max": 0.2, "differ": 0.01}  # bf16 products: 5e-3 from 64 bits


# ------------------------------------------------------------------------------------------------
# the same results in 64 bits
# ------------------------------------------------------------------------------------------------
def _round(v):
    return int(math.floor(v + 0.5))


def _exact_reference(vol, cur):
    """Projector volume complex128 [S][S][S/2+1] (z, y from -(S/2), x from 0) and power spectrum of a map."""
    dev, N = vol.device, vol.shape[0]
    P = 2 * N
    q = torch.arange(N, device=dev, dtype=torch.float64) - N // 2
    r = torch.sqrt(q[:, None, None] ** 2 + q[None, :, None] ** 2 + q[None, None, :] ** 2)
    v = vol.double() / torch.sinc(r / P) ** 2
    pad = torch.zeros((P, P, P), device=dev, dtype=torch.float64)
    o = P // 2 - N // 2
    pad[o:o + N, o:o + N, o:o + N] = v
    F = torch.fft.rfftn(pad)
    del pad
    rr = _round(PAD * (min(cur, N) // 2))
    S = 2 * (rr + 1) + 1
    h = S // 2
    k = torch.arange(-h, h + 1, device=dev)
    x = torch.arange(h + 1, device=dev)
    ok = (k > -P // 2) & (k <= P // 2)
    kk = torch.where(k < 0, k + P, k).clamp(0, P - 1)
    xx = x.clamp(max=P // 2)
    D = F[kk][:, kk][:, :, xx]
    del F
    r2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + x[None, None, :] ** 2
    keep = (r2 <= rr * rr) & ok[:, None, None] & ok[None, :, None] & (x <= P // 2)[None, None, :]
    sign = 1.0 - 2.0 * ((kk[:, None, None] + kk[None, :, None] + xx[None, None, :]) & 1)
    D = torch.where(keep, D * sign * (PAD ** 3 * N / float(P) ** 3), torch.zeros_like(D))
    shell = torch.floor(torch.sqrt(r2.double()) / PAD + 0.5).long()
    use = keep & (shell < N // 2 + 1)
    ps = torch.bincount(shell[use], weights=(D[use].abs() ** 2 / 2), minlength=N // 2 + 1)
    cnt = torch.bincount(shell[use], minlength=N // 2 + 1)
    return D, torch.where(cnt > 0, ps / cnt.clamp(min=1), torch.zeros_like(ps))


def _corners(pts, S):
    """(Hermitian flip, flat base index, inside, eight corner weights) of points [m][3] (x, y, z)."""
    h = S // 2
    neg = pts[:, 0] < 0
    p = torch.where(neg[:, None], -pts, pts)
    b = torch.floor(p)
    f = p - b
    i = b.long()
    i[:, 1:] += h
    inside = (i[:, 0] + 1 < h + 1) & (i[:, 1:] >= 0).all(1) & (i[:, 1:] + 1 < S).all(1)
    i = torch.where(inside[:, None], i, torch.zeros_like(i))
    base = (i[:, 2] * S + i[:, 1]) * (h + 1) + i[:, 0]
    w = [1 - f, f]
    ws = torch.stack([w[(c >> 2) & 1][:, 2] * w[(c >> 1) & 1][:, 1] * w[c & 1][:, 0] for c in range(8)], 1)
    off = torch.tensor([((c >> 2) & 1) * S * (h + 1) + ((c >> 1) & 1) * (h + 1) + (c & 1) for c in range(8)],
                       device=pts.device)
    return neg, base, inside, ws, off


def _project(V, frames, yx):
    """Trilinear samples complex128 [frames][pixels] of V at frames [m][2][3] (rows e0, e1) times pixels (y, x)."""
    S = V.shape[0]
    pts = (yx[None, :, 1:2] * frames[:, None, 0] + yx[None, :, 0:1] * frames[:, None, 1]).reshape(-1, 3)
    neg, base, inside, ws, off = _corners(pts, S)
    flat = V.reshape(-1)
    v = sum(flat[base + off[c]] * ws[:, c] for c in range(8)) * inside
    return torch.where(neg, v.conj(), v).reshape(len(frames), len(yx))


def _pixels(s, N, dev):
    """(frequency y, x) [P][2] and resolution shell (-1: none) of an image of size s."""
    y, x = _freq(s, dev)
    yx = torch.stack([y[:, None].expand(s, s // 2 + 1), x[None, :].expand(s, s // 2 + 1)], -1).reshape(-1, 2)
    ires = torch.floor(yx.pow(2).sum(1).sqrt() + 0.5).long()
    none = (ires >= s // 2 + 1) | ((yx[:, 1] == 0) & (yx[:, 0] < 0))
    return yx, torch.where(none, torch.full_like(ires, -1), ires)


def _threshold(w, total, fraction=0.999):
    """Weight at which the descending cumulative sum first exceeds fraction * total, and its rank."""
    d = torch.sort(w[w > 0], descending=True).values
    cum = torch.cumsum(d, 0)
    hit = torch.nonzero(cum > fraction * total)
    k = int(hit[0]) if len(hit) else len(d) - 1
    return d[k], k + 1


class _ExactEstep:
    """The expectation step particle by particle in complex128."""

    def __init__(self, p, dev):
        c = self.c = p["case"]
        self.p, self.dev = p, dev
        self.N, self.s, self.sc, self.K = c["box"], c["cur"], _coarse_size(c), c["classes"]
        self.vols = [_exact_reference(m, c["cur"])[0] for m in p["maps"]]
        self.S = self.vols[0].shape[0]
        self.rot, self.tilt = _healpix(c["order"])
        self.npsi = _n_psi(c["order"])
        self.psi = np.arange(self.npsi) * 360.0 / self.npsi
        t = _translations(c) / c["px"]  # pixels
        self.tA = t * c["px"]
        h = c["step_px"] / 4.0
        self.over = np.stack([t + d for d in ((-h, -h), (-h, h), (h, -h), (h, h))], 1)  # [NT][4][2]
        s2 = torch.tensor(p["sigma2"], device=dev)

        def minv(ires):
            return torch.where(ires > 0, 1.0 / s2[ires.clamp(min=0)], torch.zeros(1, device=dev, dtype=torch.float64))

        rmax = self.s // 2
        yx, ires = _pixels(self.sc, self.N, dev)
        r2 = yx.pow(2).sum(1)
        self.c_keep = torch.nonzero(minv(ires) > 0).flatten()
        self.c_yx, self.c_minv = yx[self.c_keep], minv(ires)[self.c_keep]
        self.c_proj = r2[self.c_keep] <= min(self.sc // 2, rmax) ** 2
        self.f_yx, self.f_ires = _pixels(self.s, self.N, dev)
        self.f_minv = minv(self.f_ires)
        self.f_r2 = self.f_yx.pow(2).sum(1)
        self.f_proj = self.f_r2 <= rmax * rmax
        row = torch.arange(self.s, device=dev)[:, None].expand(self.s, self.s // 2 + 1).reshape(-1)
        self.f_bp = (self.f_r2 <= rmax * rmax) & ~((row >= self.s // 2 + 1) & (self.f_yx[:, 1] == 0))
        self.minv_w = self.f_minv.clone()
        self.minv_w[0] = 1.0 / s2[0]
        self.logs2 = float(torch.log(2 * math.pi * s2[self.f_ires[self.f_ires > 0]]).sum())
        # window of the coarse pixels in the fine image
        y = self.c_yx[:, 0].long()
        self.c_src = torch.where(y < 0, y + self.s, y) * (self.s // 2 + 1) + self.c_yx[:, 1].long()
        self.finer = _healpix(c["order"] + 1)
        d, q = np.meshgrid(np.arange(len(self.rot)), np.arange(self.npsi), indexing="ij")
        fr = PAD * _rotations(self.rot[d.ravel()], self.tilt[d.ravel()], self.psi[q.ravel()])[:, :2]
        self.coarse = []
        for k in range(self.K):
            out = torch.empty((len(fr), len(self.c_yx)), dtype=torch.complex128, device=dev)
            for i in range(0, len(fr), 2048):
                out[i:i + 2048] = _project(self.vols[k], torch.tensor(fr[i:i + 2048], device=dev), self.c_yx)
            self.coarse.append(out * self.c_proj)
        self.pd_mean = float(np.repeat(p["pdf_direction"], self.npsi, 1).mean())
        self.ph_c = self._phase(t, self.c_yx)
        n = self.S * self.S * (self.S // 2 + 1)
        self.bp = [(torch.zeros(n, dtype=torch.complex128, device=dev), torch.zeros(n, dtype=torch.float64, device=dev))
                   for _ in range(self.K)]
        self.res = {f: np.zeros(c["n"]) for f in RESULTS}
        self.ws = dict(sigma2_noise=torch.zeros(self.N // 2 + 1, dtype=torch.float64, device=dev),
                       pdf_class=np.zeros(self.K), pdf_direction=np.zeros((self.K, len(self.rot))), sigma2_offset=0.0,
                       sumw_group=0.0, signal_product=0.0, reference_power=0.0, LL=0.0, ave_Pmax=0.0)

    def _phase(self, shifts, yx):
        t = torch.tensor(np.asarray(shifts), device=self.dev)
        a = -2 * math.pi / self.N * (t[:, 0:1] * yx[None, :, 1] + t[:, 1:2] * yx[None, :, 0])
        return torch.polar(torch.ones_like(a), a)

    def _orientations(self, i):
        """Global orientation indices of particle i and their normalised priors, [K][n] in search order."""
        c, p = self.c, self.p
        if c["search"] == "local":
            sig = _sigma_ang(c)

            def unit(r, t):
                r, t = np.radians(r), np.radians(t)
                return np.stack([np.sin(t) * np.cos(r), np.sin(t) * np.sin(r), np.cos(t)], -1)

            pr, pt, pp = p["prior"][i]
            ang = np.degrees(np.arccos(np.clip(unit(self.rot, self.tilt) @ unit(pr, pt), -1.0, 1.0)))
            di = np.nonzero(ang < 3 * sig)[0]
            dp = np.exp(-0.5 * (ang[di] / sig) ** 2)
            if not len(di):
                di, dp = np.array([int(np.argmin(ang))]), np.ones(1)
            dpsi = np.abs(self.psi - pp)
            dpsi = np.where(dpsi > 180.0, np.abs(dpsi - 360.0), dpsi)
            pi = np.nonzero(dpsi < 3 * sig)[0]
            pw = np.exp(-0.5 * (dpsi[pi] / sig) ** 2)
            if not len(pi):
                pi, pw = np.array([int(np.argmin(dpsi))]), np.ones(1)
            og = (di[:, None] * self.npsi + pi[None, :]).ravel()
            w = (dp[:, None] * pw[None, :]).ravel()
            return og, np.repeat((w / w.mean())[None], self.K, 0)
        og = np.arange(len(self.rot) * self.npsi)
        if p["sets"] is not None and len(p["sets"][i]):
            og = p["sets"][i].astype(np.int64)
        return og, p["pdf_direction"][:, og // self.npsi] / self.pd_mean

    def particle(self, i):
        c, p, dev = self.c, self.p, self.dev
        og, po = self._orientations(i)
        X = p["fimg"][i].reshape(-1).to(torch.complex128)
        Xn = X if p["nomask"] is None else p["nomask"][i].reshape(-1).to(torch.complex128)
        C = p["fctf"][i].reshape(-1).double()
        sc = p["scale"][i] if c["scale"] else 1.0
        # coarse pass
        q = (0.5 * self.c_minv).sqrt()
        Y = q * X[self.c_src] * self.ph_c
        cc = q * C[self.c_src] * sc
        ogt = torch.tensor(og, device=dev)
        d2 = []
        for k in range(self.K):
            part = []
            for o0 in range(0, len(og), 8192):
                A = self.coarse[k][ogt[o0:o0 + 8192]] * cc
                part.append(A.abs().pow(2).sum(1)[:, None] - 2.0 * (A @ Y.conj().T.contiguous()).real)
            d2.append(torch.cat(part))
        d2 = torch.stack(d2)  # [K][o][t]
        s2o = (c["range_px"] * c["px"] / 3.0) ** 2
        off = (p["old"][i] + self.tA - p["pri"][i]) * c["px"]
        pt = np.exp(-(off ** 2).sum(1) / (2 * s2o))
        pt = torch.tensor(pt / pt.mean(), device=dev)
        prior = torch.tensor(po, device=dev)[:, :, None] * pt
        e = d2 - d2.min()
        w = torch.where(e > 700.0, torch.zeros_like(e), prior * torch.exp(-e))
        thr, nsig = _threshold(w.flatten(), float(w.sum()))
        self.res["nr_significant"][i] = nsig
        k_i, o_i, t_i = (v.cpu().numpy() for v in torch.nonzero((w >= thr) & (w > 0), as_tuple=True))
        del d2, e, w
        # fine pass: the orientations with a significant translation, eight finer ones each
        jobs, job_of = np.unique(np.stack([k_i, o_i], 1), axis=0, return_inverse=True)
        job_of = job_of.reshape(-1)
        ts, t_of = np.unique(t_i, return_inverse=True)
        q = (0.5 * self.f_minv).sqrt()
        over = self.over[ts].reshape(-1, 2)
        ph = self._phase(over, self.f_yx)
        half = 360.0 / self.npsi / 4.0
        refs, frames, cross, aa = [], [], [], []
        Yq = ((q * X) * ph).conj().T.contiguous()
        frot, ftilt = self.finer
        for k, o in jobs:
            d, ps = divmod(int(og[o]), self.npsi)
            r = np.array([(frot[4 * d + m], ftilt[4 * d + m], self.psi[ps] + h) for m in range(4) for h in (-half, half)])
            fr = torch.tensor(PAD * _rotations(r[:, 0], r[:, 1], r[:, 2])[:, :2], device=dev)
            R = _project(self.vols[k], fr, self.f_yx) * (self.f_proj * C * sc)
            refs.append(R)
            frames.append(fr)
            A = R * q
            aa.append(A.abs().pow(2).sum(1))
            cross.append((A @ Yq).real)
        base = p["xi2"][i] / 2.0 + float(((q * X).abs() ** 2).sum())
        d2f = torch.stack([a[:, None] - 2.0 * x for a, x in zip(aa, cross)]) + base  # [job][8][t * 4]
        d2f = d2f.reshape(len(jobs), 8, len(ts), 4)[job_of, :, t_of]  # [pair][8][4]
        pf = prior[k_i, o_i, t_i][:, None, None]
        mind = float(d2f.min())
        e = d2f - mind
        w = torch.where(e > 700.0, torch.zeros_like(e), pf * torch.exp(-e))
        tot = float(w.sum())
        thr, _ = _threshold(w.flatten(), tot)
        r = self.res
        r["pmax"][i], r["sum_weight"][i], r["min_diff2"][i] = float(w.max()) / tot, tot, mind
        r["dLL"][i] = math.log(tot) - mind - self.logs2
        # weighted sums
        sig = torch.nonzero(w >= thr).cpu().numpy()
        wn = (w / tot).cpu().numpy()
        px2 = c["px"] ** 2
        groups = {}
        for s, r8, u in sig:
            groups.setdefault((int(job_of[s]), int(r8)), []).append((int(t_of[s]), int(u), wn[s, r8, u]))
        scw = max(0.001, sc)
        xa_ok = torch.zeros_like(self.f_ires, dtype=torch.bool)
        if c["scale"]:
            xa_ok = (self.f_ires > -1) & torch.tensor(p["dvp"][0] > 3.0, device=dev)[self.f_ires.clamp(min=0)]
        shell = (self.f_ires > -1)
        xa = aa_ = nc = 0.0
        for (j, r8), tu in groups.items():
            k, o = jobs[j]
            wv = np.array([v[2] for v in tu])
            idx = [4 * v[0] + v[1] for v in tu]
            wt = torch.tensor(wv, device=dev)
            P = ph[idx]
            R = refs[j][r8] * (scw / sc)
            Yt = X * P
            wd = (wt[:, None] * (R - Yt).abs().pow(2)).sum(0) * shell
            self.ws["sigma2_noise"].index_add_(0, self.f_ires[shell], wd[shell])
            nc += float(wd.sum())
            if c["scale"]:
                xa += float(((wt[:, None] * (R * Yt.conj()).real).sum(0) * xa_ok).sum())
                aa_ += float((wv.sum() * R.abs().pow(2) * xa_ok).sum())
            ctf = C * scw
            num = (wt[:, None] * (Xn * P)).sum(0) * ctf * self.minv_w
            den = wv.sum() * ctf * ctf * self.minv_w
            use = torch.nonzero(self.f_bp & (den > 0)).flatten()
            fr = frames[j][r8]
            pts = self.f_yx[use, 1:2] * fr[0] + self.f_yx[use, 0:1] * fr[1]
            neg, b, inside, cw, off8 = _corners(pts, self.S)
            val = torch.where(neg, num[use].conj(), num[use])
            D, W = self.bp[k]
            for m in range(8):
                g = cw[:, m] * inside
                D.index_add_(0, b + off8[m], val * g)
                W.index_add_(0, b + off8[m], den[use] * g)
            dlt = p["pri"][i] - p["old"][i] - over[idx]
            self.ws["sigma2_offset"] += float((wv * px2 * (dlt ** 2).sum(1)).sum())
            self.ws["sumw_group"] += wv.sum()
            self.ws["pdf_class"][k] += wv.sum()
            self.ws["pdf_direction"][k, int(og[o]) // self.npsi] += wv.sum()
        if c["scale"]:
            xa, aa_ = xa / sc, aa_ / sc ** 2
        r["wsum_norm_correction"][i], r["signal_product"][i], r["reference_power"][i] = nc, xa, aa_
        self.ws["signal_product"] += xa
        self.ws["reference_power"] += aa_
        self.ws["LL"] += r["dLL"][i]
        self.ws["ave_Pmax"] += r["pmax"][i]


def _kaiser_table(dev, steps=10000, radius=3.8, alpha=15.0):
    """Transform of the order-0 Kaiser-Bessel blob (Lewitt 1990) at floor steps of 0.5 / steps, relative to 0."""
    w = torch.arange(steps, dtype=torch.float64) * (0.5 / steps)
    t = 2 * math.pi * radius * w
    s = (alpha * alpha - t * t).abs().sqrt().clamp(min=1e-12)
    sinc = (torch.sin(s) / s - torch.cos(s)) / (s * s)
    sinh = (torch.cosh(s) - torch.sinh(s) / s) / (s * s)
    near = torch.full_like(s, 1.0 / 3.0)
    f = torch.where(s < 1e-3, near, torch.where(t > alpha, sinc, sinh))
    return (f / f[0]).to(dev)


def _exact_map(D, W, S, c, gridding=False, tau2=None, normalise=1.0):
    """The map reconstructed from sums D (complex128), W (float64), flat [S][S][S/2+1] around the centre."""
    dev, N, h, rmax = D.device, c["box"], S // 2, c["cur"] // 2
    P = 2 * N
    k = torch.arange(-h, h + 1, device=dev)
    x = torch.arange(h + 1, device=dev)
    r2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + x[None, None, :] ** 2
    lim = _round(rmax * PAD) ** 2
    D = torch.where(r2 <= lim, D.reshape(S, S, h + 1), torch.zeros(1, dtype=torch.complex128, device=dev))
    W = torch.where(r2 <= lim, W.reshape(S, S, h + 1), torch.zeros(1, dtype=torch.float64, device=dev))
    r = r2.double().sqrt() / PAD
    if tau2 is not None:
        t = torch.tensor(tau2, device=dev)
        ires = torch.floor(r + 0.5).long()
        W = W + torch.where((r2 < lim) & (ires >= 3), 1.0 / (PAD ** 3 * TAU2_FUDGE * t[ires.clamp(max=len(t) - 1)]),
                            torch.zeros(1, dtype=torch.float64, device=dev))
    if gridding:
        D, W = D / normalise, W / normalise
        new = (r2 < lim).double()
        m = torch.arange(S, device=dev)
        m = torch.where(m < S // 2, m, m - S).double()
        rv = torch.sqrt(m[:, None, None] ** 2 + m[None, :, None] ** 2 + m[None, None, :] ** 2) / (N * PAD)
        table = _kaiser_table(dev)
        idx = (rv / (0.5 / len(table))).long()
        blob = torch.where(idx < len(table), table[idx.clamp(max=len(table) - 1)], torch.zeros_like(rv))
        for _ in range(GRID_ITERATIONS):
            f = torch.fft.ifftshift((new * W), dim=(0, 1)).to(torch.complex128)
            f = torch.fft.rfftn(torch.fft.irfftn(f, s=(S, S, S), norm="forward") * blob) / float(S) ** 3
            f = torch.fft.fftshift(f.abs(), dim=(0, 1))
            new = torch.where(r2 < lim, new / f.clamp(min=1e-6), new)
        D = D * new
    else:
        ires = torch.floor(r).long().clamp(max=rmax - 1)
        use = r2 < lim
        tot = torch.bincount(ires[use], weights=W[use], minlength=rmax)
        cnt = torch.bincount(ires[use], minlength=rmax)
        avg = torch.where(cnt > 0, tot / (1000.0 * cnt.clamp(min=1)), torch.zeros_like(tot))
        w = torch.maximum(W, avg[ires])
        D = torch.where(w != 0, D / torch.where(w != 0, w, torch.ones_like(w)), D)
    F = torch.zeros((P, P, P // 2 + 1), dtype=torch.complex128, device=dev)
    m = min(h, P // 2)
    kk = torch.arange(-m if P // 2 > m else -m + 1, m + 1, device=dev)
    xx = torch.arange(m + 1, device=dev)
    sub = D[kk + h][:, kk + h][:, :, xx]
    if P // 2 > h:
        rr = kk[:, None, None] ** 2 + kk[None, :, None] ** 2 + xx[None, None, :] ** 2
        sub = torch.where(rr <= h * h, sub, torch.zeros_like(sub))
    wrap = torch.where(kk < 0, kk + P, kk)
    sub = sub * (1.0 - 2.0 * ((wrap[:, None, None] + wrap[None, :, None] + xx) & 1))
    F[wrap[:, None, None], wrap[None, :, None], xx[None, None, :]] = sub
    v = torch.fft.irfftn(F, s=(P, P, P), norm="forward")
    del F
    o = P // 2 - N // 2
    v = v[o:o + N, o:o + N, o:o + N] / (PAD ** 3 * N)
    q = torch.arange(N, device=dev, dtype=torch.float64) - N // 2
    r = torch.sqrt(q[:, None, None] ** 2 + q[None, :, None] ** 2 + q[None, None, :] ** 2)
    rad, width = N / 2.0, 3.0
    edge = torch.where(r > rad + width, torch.ones_like(r), 0.5 + 0.5 * torch.cos(math.pi * (rad + width - r) / width))
    edge = torch.where(r >= rad, edge, torch.zeros_like(r))
    bg = (edge * v).sum() / edge.sum()
    v = (1 - edge) * v + edge * bg
    return v / torch.sinc(r / P) ** 2


def _exact_estep(c, seed, dev):
    e = _ExactEstep(_estep_problem(c, seed, dev), dev)
    for i in range(c["n"]):
        e.particle(i)
    return e


def _exact_imgprep(c, seed, dev):
    img, m, sigma2 = _prep_inputs(c, seed, dev)
    n, N, s = c["n"], c["box"], c["cur"]
    xh, xs = N // 2 + 1, s // 2 + 1
    dx, dy = (np.floor(m[k] + 0.5).astype(int) for k in ("old_offset_x", "old_offset_y"))
    q = torch.arange(N, device=dev, dtype=torch.float64) - N // 2
    r = torch.sqrt(q[:, None] ** 2 + q[None, :] ** 2)
    rad, width = c["diameter"] / (2.0 * c["px"]), 5.0
    edge = torch.where(r > rad + width, torch.ones_like(r), 0.5 + 0.5 * torch.cos(math.pi * (rad + width - r) / width))
    edge = torch.where(r >= rad, edge, torch.zeros_like(r))
    y, x = _freq(N, dev)
    ires = torch.floor(torch.sqrt(y[:, None] ** 2 + x[None, :] ** 2) + 0.5).long()
    ws, wx = _freq(s, dev)
    rows = torch.where(ws < 0, ws + N, ws).long()
    sign = 1.0 - 2.0 * ((torch.arange(s, device=dev)[:, None] + torch.arange(xs, device=dev)[None, :]) & 1)
    count = (ires > 0) & (ires < xh) & ~((x[None, :] == 0) & (y[:, None] < 0))
    out = dict(fimg=torch.empty((n, s, xs), dtype=torch.complex128, device=dev), highres_Xi2=np.zeros(n),
               power=np.zeros((n, xh)), old_offset=np.stack([dx, dy], 1).astype(float))
    out["fimg_nomask"] = torch.empty_like(out["fimg"])
    sg = torch.tensor(np.sqrt(sigma2), device=dev)
    for i in range(n):
        v = torch.zeros((N, N), dtype=torch.float64, device=dev)
        a, b = dy[i], dx[i]
        v[max(0, a):N + min(0, a), max(0, b):N + min(0, b)] = img[i].double()[max(0, -a):N + min(0, -a),
                                                                               max(0, -b):N + min(0, -b)]
        v = v / m["norm_correction"][i]
        if c["noise"]:
            add = _exact_noise(seed + i, N, sg, ires, dev)
        else:
            add = (edge * v).sum() / edge.sum()
        for key, w in (("fimg", (1 - edge) * v + edge * add), ("fimg_nomask", v)):
            F = torch.fft.rfft2(w) / (N * N)
            out[key][i] = F[rows][:, :xs] * sign
            if key == "fimg":
                pw = torch.where(count, F.abs() ** 2, torch.zeros_like(r[:, :xh]))
                out["power"][i] = torch.bincount(ires[count], weights=pw[count], minlength=xh)[:xh].cpu().numpy()
        out["highres_Xi2"][i] = out["power"][i][s // 2 + 1:].sum() if s < N else 0.0
    ctf = _ctf_images(c, np.stack([m["defocus_u"], m["defocus_v"], m["defocus_angle"]], 1), s, dev)
    tiny = torch.where(ctf >= 0, 1e-8, -1e-8).double()
    out["fctf"] = torch.where(ctf.abs() < 1e-8, tiny, ctf)
    for k in ("fimg", "fimg_nomask", "fctf"):
        if not c["device"]:
            out[k] = out[k].cpu().numpy()
    return out


def _exact_noise(seed, N, sg, ires, dev):
    """The documented counter-based noise image: splitmix64 uniforms, Box-Muller, Hermitian edge columns."""
    xh = N // 2 + 1

    def const(v):
        return v - (1 << 64) if v >= 1 << 63 else v

    def shr(z, k):
        return (z >> k) & ((1 << (64 - k)) - 1)

    def mix(z):
        z = z + const(0x9E3779B97F4A7C15)
        z = (z ^ shr(z, 30)) * const(0xBF58476D1CE4E5B9)
        z = (z ^ shr(z, 27)) * const(0x94D049BB133111EB)
        return z ^ shr(z, 31)

    i = torch.arange(N, device=dev)[:, None].expand(N, xh)
    j = torch.arange(xh, device=dev)[None, :].expand(N, xh)
    ip = torch.where(i < xh, i, i - N)
    edge = (j == 0) | (j == N // 2)
    flip = edge & (ip < 0)
    e = torch.where(flip, -ip, i) * xh + j
    h1 = mix(mix(torch.tensor(seed, device=dev)) + e)
    h2 = mix(h1)
    u1, u2 = ((shr(h, 11).double() + 0.5) * 2.0 ** -53 for h in (h1, h2))
    rr = torch.sqrt(-2.0 * torch.log(u1))
    s = torch.where(ires < xh, sg[ires.clamp(max=xh - 1)], torch.zeros(1, dtype=torch.float64, device=dev))
    re, im = s * rr * torch.cos(2 * math.pi * u2), s * rr * torch.sin(2 * math.pi * u2)
    im = torch.where(flip, -im, torch.where(edge & ((ip == 0) | (ip == N // 2)), torch.zeros_like(im), im))
    return torch.fft.irfft2(torch.complex(re, im), s=(N, N), norm="forward")


def _exact_predict(c, seed, dev):
    img, ctf, _ = _net_particles(c, seed, dev)
    w = torch.tensor(_net_params(seed, dev), device=dev).double()
    W, C, s = NET["window"], NET["channels"], c["box"]
    y = torch.arange(W, device=dev)
    rows = torch.where(y < W // 2, y, y - W + s)  # the window's rows are ky = -W / 2 .. W / 2 - 1
    probs = []
    for i0 in range(0, c["n"], 256):
        F = img[i0:i0 + 256][:, rows, :W // 2 + 1].to(torch.complex128)
        F = F * torch.where(ctf[i0:i0 + 256][:, rows, :W // 2 + 1] < 0, -1.0, 1.0).double()
        v = torch.fft.irfft2(F, s=(W, W), norm="forward")
        v = v - v.mean((1, 2), keepdim=True)
        v = v / v.pow(2).mean((1, 2), keepdim=True).sqrt()
        a, o, cin, H = v[:, None], 0, 1, W
        for l in range(6):
            st, kp = (1, 2)[l & 1], (16 if cin == 1 else 9 * cin)
            wl = w[o:o + C * kp].reshape(C, kp)[:, :9 * cin]
            o += C * kp
            b = w[o:o + C]
            o += C
            cols = torch.nn.functional.unfold(a, 3, padding=1, stride=st)  # [n][cin * 9][pixels]
            cols = cols.reshape(len(a), cin, 9, -1).transpose(1, 2).reshape(len(a), 9 * cin, -1).contiguous()
            H = (H - 1) // st + 1
            a = torch.relu(torch.matmul(wl, cols) + b[:, None]).reshape(len(a), C, H, H)
            cin = C
        f = a.permute(0, 2, 3, 1).reshape(len(a), -1)
        nb = (12 << (2 * NET["healpix_order"])) * NET["n_psi_bins"]
        z = f @ w[o:o + nb * f.shape[1]].reshape(nb, -1).T.contiguous() + w[o + nb * f.shape[1]:]
        probs.append(torch.topk(torch.softmax(z, 1), PREDICT_TOPK, 1).values)
    return dict(bins=None, probs=torch.cat(probs).cpu().numpy())


def exact(case, seed):
    dev = torch.device("cuda:0") if torch.cuda.is_available() else torch.device("cpu")
    f = case["family"]
    if f == "estep":
        if case["n"] > 2100:
            return None  # about 10 ms a particle
        e = _exact_estep(case, seed, dev)
        out = dict(e.res, best=None)
        out.update({"wsum_" + k: v.cpu().numpy() if torch.is_tensor(v) else np.asarray(v) for k, v in e.ws.items()})
        e.coarse = None
        out["map"] = torch.stack([_exact_map(D, W, e.S, case) for D, W in e.bp])
        return out
    if f == "recon":
        e = _exact_estep(case, seed, dev)
        tau2 = _tau2(e.p)
        return {"map": _exact_map(*e.bp[0], e.S, case, True, tau2, float(case["n"]))[None]}
    if f == "imgprep":
        return _exact_imgprep(case, seed, dev)
    if f == "refprep":
        D, ps = _exact_reference(_real_map(case, seed, 0, dev), case["cur"])
        return dict(power=ps.cpu().numpy(), data=D.cpu().numpy()) if case["data"] else dict(power=ps.cpu().numpy())
    if f == "predict":
        return _exact_predict(case, seed, dev)
    return None  # training: the batches' order is the library's own shuffle
