"""Performance cases of the pattern-offset library: what its users have it do.

Every case is one pass through a public entry point of the Python package (or, for
the deformation post-step on device-resident results, of the C ABI):

  offsets  GpuOffset.process_device: a batch of patterns in HBM, results in HBM
  host     GpuOffset.get_offset: patterns and results in host memory
  serve    Server: single-pattern requests to two resident plans, all waited for
  post     emida_fit_deformation: a batch of ROI results in HBM

Inputs are EBSD-like patterns made on the GPU from the seed, as they are after
background correction: weak broad bands and many sharp band edges, resampled under a
small strain and a drift of up to two pixels, with the counting noise of an average
over four frames.  Sharp features in every ROI and a drift off the half pixel keep a
ROI's whole-pixel peak from hanging on the last bits of a correlation value.

Results of a float pipeline are handed on as float32 (the least-squares fit runs in
double on float correlation values); those of a double pipeline as they are.
"""
import ctypes
import math

import numpy as np
import torch

import emida_amd
from emida_amd import _capi as C

POLICIES = {"fft": emida_amd.CROSS_POLICY_FFT, "brute": emida_amd.CROSS_POLICY_BRUTE,
            "mfma": emida_amd.CROSS_POLICY_BRUTE_MFMA}
NP = {"f32": np.float32, "f64": np.float64, "u16": np.uint16}
TORCH = {"f32": torch.float32, "f64": torch.float64}


def _offsets(name, policy, T, IN, w, h, kx, ky, sx, sy, fit, batch, cx=0, cy=0, kind="offsets"):
    """cx, cy: correlation window, 0 for the full 2s - 1."""
    c = dict(kind=kind, policy=policy, T=T, IN=IN, w=w, h=h, kx=kx, ky=ky, sx=sx, sy=sy, fit=fit, batch=batch,
             cx=cx, cy=cy)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one pattern from host memory to host offsets, as a live
        # acquisition or a single-pattern script does it
        _offsets("fft_f32_host_one", "fft", "f32", "u16", 873, 873, 20, 20, 64, 64, 5, 1, kind="host"),
        # the headline configuration: scan patterns in HBM, 400 ROIs of 64 x 64, float FFT
        _offsets("fft_f32_64px_b64", "fft", "f32", "u16", 873, 873, 20, 20, 64, 64, 5, 64),
        # larger ROIs: 100 of 128 x 128
        _offsets("fft_f32_128px_b64", "fft", "f32", "u16", 873, 873, 10, 10, 128, 128, 7, 64),
        # the headline ROIs in double precision
        _offsets("fft_f64_64px_b16", "fft", "f64", "u16", 873, 873, 20, 20, 64, 64, 5, 16),
        # radius 48 as in the reference's example ROI file, in double: the driver's batch of 8
        _offsets("fft_f64_96px_b8", "fft", "f64", "u16", 873, 873, 9, 9, 96, 96, 7, 8),
        # non-square ROIs of odd sides on a wide detector image, float pixels
        _offsets("fft_f32_wide_f32in", "fft", "f32", "f32", 1344, 1001, 7, 6, 161, 95, 5, 16),
        # brute force in double, small patterns: the reference's default policy and precision
        _offsets("brute_f64_32px_b16", "brute", "f64", "u16", 256, 256, 5, 5, 32, 32, 3, 16),
        # brute force in double, 100 ROIs of 128 x 128
        _offsets("brute_f64_128px_b16", "brute", "f64", "u16", 873, 873, 10, 10, 128, 128, 7, 16),
        # brute force in float over a search window smaller than the slice, odd sizes
        _offsets("brute_f32_window", "brute", "f32", "f32", 640, 480, 9, 7, 75, 61, 5, 12, 41, 33),
        # exact peaks through the matrix cores, 100 ROIs of 128 x 128 in double: the largest
        _offsets("mfma_f64_128px_b128", "mfma", "f64", "u16", 873, 873, 10, 10, 128, 128, 7, 128),
        # serving: 64 single-pattern requests to a float FFT plan (400 ROIs of 64 x 64) and
        # a matrix-core plan (400 ROIs of 32 x 32)
        dict(name="serve_two_plans", kind="serve", w=873, h=873, requests=64, k=20, s_fft=64, s_mfma=32, fit=5),
        # strain and rotation of a part of a scan from its ROI results
        dict(name="post_400rois", kind="post", w=873, h=873, rois=400, patterns=5000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("fft", "fft", "fft", "brute", "brute", "mfma", "mfma", "post", "host"))
    if kind == "post":
        rois = _log_int(rng, 20, 1200)
        return dict(kind="post", w=873, h=873, rois=rois, patterns=min(_log_int(rng, 100, 20000), 2000000 // rois))
    T = rng.choice(("f32", "f64"))
    IN = rng.choice(("u16", "u16", "u16", T))
    w = rng.randint(300, 1100)
    h = w if rng.random() < 0.5 else rng.randint(300, 1100)
    fit = rng.choice((3, 5, 7, 9))
    square = rng.random() < 0.6
    cx = cy = 0
    if kind in ("fft", "host"):
        sx = _log_int(rng, 18, 200)
        sy = sx if square else _log_int(rng, 18, 200)
        per = 4 * sx * sy * (4 if T == "f64" else 1)
        most = 1.5e8 if kind == "fft" else 8e6
    elif kind == "brute":
        sx = _log_int(rng, 16, 110)
        sy = sx if square else _log_int(rng, 16, 110)
        if rng.random() < 0.3:
            cx, cy = (2 * rng.randint(10, max(11, s - 2)) + 1 for s in (sx, sy))
            cx, cy = min(cx, 2 * sx - 1), min(cy, 2 * sy - 1)
        per = 2 * sx * sy * (cx or 2 * sx) * (cy or 2 * sy) / 4
        most = 3e10
    else:
        sx = 8 * _log_int(rng, 2, 16)
        sy = sx if square else _log_int(rng, 16, 128)
        per = 2 * (sx * sy) ** 2
        most = 2e12
    kx, ky = (max(1, min(rng.randint(2, 20), s // 24)) for s in (w, h))
    batch = max(1, min(_log_int(rng, 1, 64), int(most / (per * kx * ky))))
    while kx * ky * per > most and (kx > 1 or ky > 1):
        kx, ky = max(1, kx // 2), max(1, ky // 2)
    return _offsets("", "fft" if kind == "host" else kind, T, IN, w, h, kx, ky, sx, sy, fit, batch, cx, cy,
                    kind="host" if kind == "host" else "offsets")


# ------------------------------------------------------------------ inputs

def _generator(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + tag) & 0x7FFFFFFF)
    return g


def _clean(w, h, g):
    """Noise-free reference pattern, float32 (h, w)."""
    y, x = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float32) - (h - 1) / 2,
                          torch.arange(w, device="cuda", dtype=torch.float32) - (w - 1) / 2, indexing="ij")
    half = 0.5 * math.hypot(w, h)
    img = torch.zeros(h, w, device="cuda")
    for n, (s0, s1), (a0, a1) in ((30, (6.0, 20.0), (100.0, 400.0)), (400, (1.5, 2.5), (1000.0, 4000.0))):
        u = torch.rand(4, n, generator=g, device="cuda").cpu().numpy()
        for b in range(n):
            th, rho = math.pi * u[0, b], half * (2 * u[1, b] - 1)
            s, a = s0 + (s1 - s0) * u[2, b], a0 + (a1 - a0) * u[3, b]
            d = x * math.cos(th) + (y * math.sin(th) - rho)
            img += a * torch.exp(d * d * (-0.5 / (s * s)))
    f = 1.5 * max(w, h)
    return 8000.0 + img * torch.exp((x * x + y * y) * (-0.5 / (f * f)))


def _noisy(img, g):
    n = img + 0.5 * img.sqrt() * torch.randn(img.shape, generator=g, device="cuda")
    return n.round_().clamp_(0, 65535)


def _pixels(img, IN):
    # uint16 pixels are kept as the int16 of the same bits: torch has few uint16 operations
    return img.to(torch.int32).to(torch.int16) if IN == "u16" else img.to(TORCH[IN])


def _patterns(w, h, n, reach, IN, seed):
    """(reference, n deformed patterns) as (h, w) and (n, h, w) device tensors."""
    g = _generator(seed, 1)
    clean = _clean(w, h, g)
    ref = _pixels(_noisy(clean, g), IN)
    eps = torch.randn(n, 2, 2, generator=g, device="cuda") * 5e-5
    whole = torch.randint(-reach, reach + 1, (n, 2), generator=g, device="cuda")
    t = whole + (torch.rand(n, 2, generator=g, device="cuda") - 0.5) * 0.3
    back = torch.linalg.inv(torch.eye(2, device="cuda") + eps)  # source = back (x - t), about the centre
    out = []
    half = torch.tensor([(w - 1) / 2, (h - 1) / 2], device="cuda")
    for i in range(0, n, 16):
        b, s = back[i:i + 16], t[i:i + 16]
        theta = torch.empty(len(b), 2, 3, device="cuda")  # normalised coordinates: x / half
        theta[:, :, :2] = b * (half[None, :] / half[:, None])
        theta[:, :, 2] = -(b * s[:, None, :]).sum(-1) / half
        grid = torch.nn.functional.affine_grid(theta, (len(b), 1, h, w), align_corners=True)
        img = torch.nn.functional.grid_sample(clean.expand(len(b), 1, h, w), grid, mode="bicubic",
                                              padding_mode="border", align_corners=True)
        out.append(_pixels(_noisy(img[:, 0], g), IN))
    return ref, torch.cat(out)


def _begins(case):
    """Corners of a kx x ky grid of sx x sy ROIs, four pixels off the border, x fastest."""
    xs = np.linspace(4, case["w"] - case["sx"] - 4, case["kx"]).astype(int)
    ys = np.linspace(4, case["h"] - case["sy"] - 4, case["ky"]).astype(int)
    return [(int(x), int(y)) for y in ys for x in xs]


def _cross(case):
    return (case["cx"] or 2 * case["sx"] - 1, case["cy"] or 2 * case["sy"] - 1)


def _reach(case):
    return 2 if min(case["sx"], case["sy"]) >= 40 else 1


def _host(t):
    a = t.cpu().numpy()
    return a.view(np.uint16) if a.dtype == np.int16 else a


_STREAM = []


def _stream():
    """The stream the program runs its device passes on."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def _post_inputs(case, seed):
    """ROI middles, offsets under small homographies with fit noise, fit coefficients."""
    g = _generator(seed, 2)
    P, N = case["patterns"], case["rois"]
    rnd = lambda *s: torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)
    nrm = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.float64)
    size = torch.tensor([case["w"], case["h"]], device="cuda", dtype=torch.float64)
    mids = (40 + rnd(N, 2) * (size - 80)).round()
    z = 0.7 * case["w"]
    F = torch.eye(3, device="cuda", dtype=torch.float64) + nrm(P, 3, 3) * 2e-3
    r = torch.cat([mids - size / 2, torch.full((N, 1), z, device="cuda", dtype=torch.float64)], 1)
    q = (F[:, None] * r[None, :, None, :]).sum(-1)
    offs = q[..., :2] / q[..., 2:] * z - r[None, :, :2] + nrm(P, N, 2) * 0.02
    coefs = nrm(P, N, 6)
    coefs[..., 0] *= 100
    coefs[..., 3] = -0.2 - rnd(P, N)
    coefs[..., 5] = -0.2 - rnd(P, N)
    coefs[..., 4] *= 0.3  # a few percent of the ROIs have no maximum
    return mids, offs.contiguous(), coefs


def prepare(case, seed):
    if case["kind"] == "post":
        mids, offs, coefs = _post_inputs(case, seed)
        P = case["patterns"]
        new = lambda *s: torch.empty(*s, device="cuda", dtype=torch.float64)
        return dict(case=case, mids=mids, offs=offs, coefs=coefs, mask=torch.empty(P, device="cuda", dtype=torch.int32),
                    quality=new(P), H=new(P, 3, 3), F=new(P, 3, 3), epsilon=new(P, 3, 3), omega=new(P, 3, 3),
                    calib=C.Calib(case["w"] / 2, case["h"] / 2, 0.7 * case["w"]))
    if case["kind"] == "serve":
        ref, pics = _patterns(case["w"], case["h"], case["requests"], 2, "u16", seed)
        ref, pics = _host(ref), _host(pics)
        srv = emida_amd.Server(max_batch=16, streams=4, max_queued=256)
        plans = []
        for s, policy in ((case["s_fft"], "fft"), (case["s_mfma"], "mfma")):
            begins = _begins(dict(w=case["w"], h=case["h"], sx=s, sy=s, kx=case["k"], ky=case["k"]))
            plans.append(srv.add_plan(np.float32, ref, begins, (s, s), None, POLICIES[policy], case["fit"]))
        n = case["k"] ** 2
        return dict(case=case, srv=srv, plans=plans, pics=list(pics), ref=ref,
                    offs=np.empty((case["requests"], n, 2)), coefs=np.empty((case["requests"], n, 6)))
    ref, pics = _patterns(case["w"], case["h"], case["batch"], _reach(case), case["IN"], seed)
    plan = emida_amd.GpuOffset(NP[case["T"]], NP[case["IN"]], (case["w"], case["h"]), _begins(case),
                               (case["sx"], case["sy"]), _cross(case), case["batch"], POLICIES[case["policy"]],
                               case["fit"])
    plan.allocate_memory(_host(ref))
    if case["kind"] == "host":
        return dict(case=case, plan=plan, pics=_host(pics))
    n, wide = plan.total_slices, case["T"] == "f64"
    return dict(case=case, plan=plan, pics=pics, n=n,
                maxes=torch.zeros(n, 4 if wide else 2, device="cuda", dtype=torch.int32),
                neighbors=torch.empty(n, case["fit"], case["fit"], device="cuda", dtype=TORCH[case["T"]]),
                results=torch.empty(8 * n, device="cuda", dtype=torch.float64),
                results32=None if wide else torch.empty(8 * n, device="cuda", dtype=torch.float32))


# ------------------------------------------------------------------ one pass

def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    case = state["case"]
    if case["kind"] == "host":
        offs, coefs = state["plan"].get_offset(state["pics"])
        kind = NP[case["T"]]
        return {"offsets": offs.astype(kind, copy=False), "coefs": coefs.astype(kind, copy=False)}
    if case["kind"] == "serve":
        srv, offs, coefs = state["srv"], state["offs"], state["coefs"]
        ids = [srv.submit(state["plans"][i % 2], p, offs[i], coefs[i])[0] for i, p in enumerate(state["pics"])]
        for rid in ids:
            srv.wait(rid)
        return {"offsets": offs.astype(np.float32), "coefs": coefs.astype(np.float32)}
    stream = _stream()
    if case["kind"] == "post":
        s = state
        C.check(C.lib().emida_fit_deformation(_ptr(s["mids"]), 0, case["rois"], _ptr(s["offs"]), _ptr(s["coefs"]),
                                              case["patterns"], s["calib"], 1e-6, 10, _ptr(s["mask"]),
                                              _ptr(s["quality"]), _ptr(s["H"]), _ptr(s["F"]), _ptr(s["epsilon"]),
                                              _ptr(s["omega"]), ctypes.c_void_p(stream.cuda_stream)))
        return {k: s[k] for k in ("mask", "quality", "H", "F", "epsilon", "omega")}
    n, maxes, results = state["n"], state["maxes"], state["results"]
    state["plan"].process_device(state["pics"].data_ptr(), case["batch"], maxes.data_ptr(),
                                 state["neighbors"].data_ptr(), results.data_ptr(), results[2 * n:].data_ptr(),
                                 stream.cuda_stream)
    if case["T"] == "f32":
        with torch.cuda.stream(stream):
            results = state["results32"].copy_(results)
        peak, index = maxes[:, 0].view(torch.float32), maxes[:, 1]
    else:
        peak, index = maxes[:, :2].view(torch.float64)[:, 0], maxes[:, 2]
    return {"offsets": results[:2 * n].view(n, 2), "coefs": results[2 * n:].view(n, 6), "peak": peak,
            "index": index, "neighbors": state["neighbors"]}


# ------------------------------------------------------------------ what a pass needs

def _overlap(s, c):
    r = (c - 1) // 2
    return sum(max(0, s - abs(d)) for d in range(-r, c - r))


def _slice_flops(policy, sx, sy, cx, cy):
    if policy == "fft":  # two real 2s x 2s transforms and a product with half a spectrum
        a = 4.0 * sx * sy
        return 2 * 2.5 * a * math.log2(a) + 6 * (sx + 1) * 2 * sy
    return 2.0 * _overlap(sx, cx) * _overlap(sy, cy)


def work(case):
    if case["kind"] == "post":
        P, N = case["patterns"], case["rois"]
        return {"bytes": 16.0 * N + 64.0 * P * N + P * (4 + 8 + 4 * 72), "flops": P * (N * (45 * 4 + 20.0) + 20000)}
    if case["kind"] == "serve":
        R, n = case["requests"], case["k"] ** 2
        flops = [_slice_flops(p, s, s, 2 * s - 1, 2 * s - 1) for p, s in (("fft", case["s_fft"]), ("mfma", case["s_mfma"]))]
        return {"bytes": R * (2.0 * case["w"] * case["h"] + 64 * n), "flops": R * n * sum(flops) / 2}
    n = case["kx"] * case["ky"] * case["batch"]
    t, px = (8 if case["T"] == "f64" else 4), {"u16": 2, "f32": 4, "f64": 8}[case["IN"]]
    out = 64 if case["kind"] == "host" else 64 + 2 * t + t * case["fit"] ** 2
    return {"bytes": float(px * case["w"] * case["h"] * case["batch"] + out * n),
            "flops": n * _slice_flops(case["policy"], case["sx"], case["sy"], *_cross(case))}


# ------------------------------------------------------------------ in 64 bits, plain torch and numpy

def _windowed(pics, begins, sx, sy):
    """Mean-free Hann-windowed slices of (n, h, w) patterns: (n, rois, sy, sx), float64."""
    hann = lambda s: torch.from_numpy(0.5 * (1 - np.cos(2 * np.pi * np.arange(s) / (s - 1)))).cuda()
    cut = torch.stack([pics[:, y:y + sy, x:x + sx] for x, y in begins], 1).double()
    cut = cut - cut.mean((-2, -1), keepdim=True)
    return cut * hann(sx) * hann(sy)[:, None]


def _exact_offsets(ref, pics, begins, policy, sx, sy, cx, cy, fit):
    r, dev = (fit - 1) // 2, pics.device
    if pics.dtype == torch.int16:
        pics, ref = (t.to(torch.int32).bitwise_and(0xFFFF) for t in (pics, ref))
    if policy == "fft":
        cx, cy = 2 * sx - 1, 2 * sy - 1
    rx, ry = (cx - 1) // 2, (cy - 1) // 2
    spectrum = torch.fft.rfft2(_windowed(ref[None], begins, sx, sy), s=(2 * sy, 2 * sx)).conj()
    k = np.arange(fit * fit)
    x, y = k % fit, k // fit
    fitm = torch.from_numpy(np.linalg.pinv(np.stack([np.ones(fit * fit), x, y, x * x, x * y, y * y], 1))).to(dev)
    outs = []
    step = max(1, int(4e7 / (len(begins) * 4 * sx * sy)))
    for i in range(0, len(pics), step):
        c = torch.fft.irfft2(torch.fft.rfft2(_windowed(pics[i:i + step], begins, sx, sy), s=(2 * sy, 2 * sx)) * spectrum,
                             s=(2 * sy, 2 * sx))
        c = torch.roll(c, (ry, rx), (-2, -1))[..., :cy, :cx].reshape(-1, cy, cx)
        if policy == "fft":
            c = c * (4.0 * sx * sy)
        peak, at = c.flatten(1).max(1)
        py, px = at // cx, at % cx
        gy = (py[:, None] + torch.from_numpy(y - r).to(dev)).clamp(0, cy - 1)
        gx = (px[:, None] + torch.from_numpy(x - r).to(dev)).clamp(0, cx - 1)
        nb = c.flatten(1).gather(1, gy * cx + gx)
        co = (nb[:, None, :] * fitm[None]).sum(-1)
        _, b, cc, d, e, f = co.unbind(1)
        oy = (b * e - 2 * cc * d) / (4 * f * d - e * e)
        ox = (-e * oy - b) / (2 * d)
        off = torch.stack([-(px - rx - r + ox), -(py - ry - r + oy)], 1)
        index = ((py - ry) % (2 * sy)) * 2 * sx + (px - rx) % (2 * sx) if policy == "fft" else at
        outs.append((off, co, peak, index.to(torch.int32), nb.view(-1, fit, fit)))
    return [torch.cat(v) for v in zip(*outs)]


def _exact_post(case, seed):
    mids, offs, coefs = (t.cpu().numpy() for t in _post_inputs(case, seed))
    P, N = case["patterns"], case["rois"]
    cal = np.array([case["w"] / 2, case["h"] / 2])
    z = 0.7 * case["w"]
    det = coefs[..., 3] * coefs[..., 5] - (coefs[..., 4] / 2) ** 2
    use = det > 1e-6
    old, new = np.broadcast_to(mids - cal, (P, N, 2)), mids + offs - cal
    zero, one = np.zeros((P, N)), np.full((P, N), z)
    r = np.stack([old[..., 0], old[..., 1], one], -1)
    A = np.concatenate([np.concatenate([-r * z, np.stack([zero] * 3, -1), r * new[..., :1]], -1),
                        np.concatenate([np.stack([zero] * 3, -1), -r * z, r * new[..., 1:]], -1)], 1)
    A *= np.concatenate([use, use], 1)[..., None]
    # the right singular vector of the smallest singular value, from the R factor
    H = np.linalg.svd(np.linalg.qr(A, mode="r"))[2][:, -1].reshape(P, 3, 3)
    F = H / np.cbrt(np.linalg.det(H))[:, None, None]
    u, s, vt = np.linalg.svd(F)
    eps = np.einsum("pki,pk,pkj->pij", vt, np.log(s), vt)
    rot = u @ vt
    skew = (rot - rot.transpose(0, 2, 1)) / 2
    sin = np.sqrt((skew ** 2).sum((1, 2)) / 2)
    omega = skew * (np.arcsin(sin) / sin)[:, None, None]
    out = {"mask": (use.sum(1) > 10).astype(np.int32), "quality": np.median(det, 1), "H": H / H[:, 2:, 2:], "F": F,
           "epsilon": eps, "omega": omega}
    for k in ("H", "F", "epsilon", "omega"):
        out[k][out["mask"] == 0] = np.nan
    return out


def exact(case, seed):
    if case["kind"] == "post":
        return _exact_post(case, seed)
    names = ("offsets", "coefs", "peak", "index", "neighbors")
    if case["kind"] == "serve":
        ref, pics = _patterns(case["w"], case["h"], case["requests"], 2, "u16", seed)
        offs = torch.empty(case["requests"], case["k"] ** 2, 2, dtype=torch.float64)
        coefs = torch.empty(case["requests"], case["k"] ** 2, 6, dtype=torch.float64)
        for j, (s, policy) in enumerate(((case["s_fft"], "fft"), (case["s_mfma"], "mfma"))):
            begins = _begins(dict(w=case["w"], h=case["h"], sx=s, sy=s, kx=case["k"], ky=case["k"]))
            mine = pics[j::2]
            o, c = _exact_offsets(ref, mine, begins, policy, s, s, 2 * s - 1, 2 * s - 1, case["fit"])[:2]
            offs[j::2], coefs[j::2] = o.view(len(mine), -1, 2).cpu(), c.view(len(mine), -1, 6).cpu()
        return {"offsets": offs.numpy(), "coefs": coefs.numpy()}
    ref, pics = _patterns(case["w"], case["h"], case["batch"], _reach(case), case["IN"], seed)
    got = _exact_offsets(ref, pics, _begins(case), case["policy"], case["sx"], case["sy"], *_cross(case), case["fit"])
    return dict(zip(names[:2], (t.cpu().numpy() for t in got[:2]))) if case["kind"] == "host" else dict(zip(names, got))
