"""Performance cases: the work a user of this library has it do.

Each case goes through the public entry points (the ctypes binding of the C
ABI) on inputs resident where a program would have them, over the range the
library is used in: the smallest images (64 x 64, where launches and latency
count) to the largest (8192 x 8192), compiled line lengths and arbitrary ones,
square and not, single images, batches and a request server.

Kinds of case
  hio          the HIO loop on resident state (imresh_hio_iterations), the time
               of every reconstruction: constraint, FFT, modulus, inverse FFT.
               The state is a late one: g' near the object, the support known.
  host         one whole reconstruction of a host array (shrinkWrap itself)
  batch        many images of mixed sizes in one call
  serve        requests of arbitrary sizes through the server
  mask         the operators of a mask update: norm, blur, maximum, cut-off,
               HIO error
  simulate     the forward model of an object, and a photon-counting
               measurement of a pattern
  fft          a complex 2-D transform forth and back

The loop amplifies rounding while it is far from a solution (about twice an
iteration), so whole reconstructions here run a few iterations only, which is
where two evaluations can still be compared; the long loops start near one.
"""
import math
import random

import numpy as np
import torch

import imresh_amd as im

DEV = "cuda"
FLT_MIN = float(np.finfo(np.float32).tiny)
BETA = 0.9
BATCH_SIZES = (64, 96, 128, 200, 256, 384, 512, 768, 1024)
# compiled line lengths a drawn image may have; others are arbitrary
PLAN_SIZES = (64, 96, 128, 160, 192, 200, 256, 320, 384, 512, 640, 768, 1024, 1280, 1536, 2048, 2560,
              3072, 4096, 5120, 6144, 8192)


def listed():
    return [
        # the smallest image anybody reconstructs, through the host call of the reference
        {"name": "host_64x64", "kind": "host", "w": 64, "h": 64, "cycles": 2, "hio": 2},
        # one cycle's loop (the default 20 iterations) on a small image: latency of 40 launches
        {"name": "hio_256x256", "kind": "hio", "w": 256, "h": 256, "iters": 20},
        # an ordinary detector image, not square
        {"name": "hio_1024x768", "kind": "hio", "w": 1024, "h": 768, "iters": 20},
        # the benchmark's image, one cycle's loop
        {"name": "hio_2048x2048", "kind": "hio", "w": 2048, "h": 2048, "iters": 20},
        # the first size whose state exceeds the Infinity Cache
        {"name": "hio_4096x4096", "kind": "hio", "w": 4096, "h": 4096, "iters": 4},
        # the largest image
        {"name": "hio_8192x8192", "kind": "hio", "w": 8192, "h": 8192, "iters": 2},
        # an arbitrary crop: neither length has a compiled transform
        {"name": "hio_1373x1101", "kind": "hio", "w": 1373, "h": 1101, "iters": 10},
        # mixed sizes in one call (the sizes of the batched workload)
        {"name": "batch_24", "kind": "batch", "count": 24, "sizes_seed": 3, "cycles": 2, "hio": 2},
        # a burst of requests of arbitrary sizes
        {"name": "serve_12", "kind": "serve", "count": 12, "sizes_seed": 5, "lo": 128, "hi": 1024,
         "cycles": 2, "hio": 1},
        # a program that drives the operators itself
        {"name": "mask_1000x1200", "kind": "mask", "w": 1000, "h": 1200, "sigma": 3.0},
        # object -> pattern, and a pattern's measurement
        {"name": "simulate_2048x2048", "kind": "simulate", "w": 2048, "h": 2048, "photons": 1e9},
        # transforms of a ragged size
        {"name": "fft_1500x1200", "kind": "fft", "w": 1500, "h": 1200},
    ]


def _length(rng, lo, hi):
    """A line length: half compiled ones, half anything, log-uniform."""
    if rng.random() < 0.5:
        return rng.choice([n for n in PLAN_SIZES if lo <= n <= hi])
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hio", "hio", "hio", "hio", "fft", "simulate", "mask", "host", "batch", "serve"])
    if kind in ("hio", "fft", "simulate", "mask"):
        while True:
            w = _length(rng, 64, 4096)
            h = w if rng.random() < 0.3 else _length(rng, 64, 4096)
            if w * h <= 8 << 20 or (w in PLAN_SIZES and h in PLAN_SIZES):
                break
    if kind == "hio":
        # up to one cycle's loop, shorter on the large images
        return {"kind": kind, "w": w, "h": h, "iters": max(2, min(20, (16 << 20) // (w * h)))}
    if kind == "mask":
        return {"kind": kind, "w": w, "h": h, "sigma": round(rng.uniform(1.5, 6.0), 3)}
    if kind == "simulate":
        return {"kind": kind, "w": w, "h": h, "photons": 10.0 ** rng.uniform(6.0, 11.0)}
    if kind == "fft":
        return {"kind": kind, "w": w, "h": h}
    if kind == "host":
        return {"kind": kind, "w": _length(rng, 64, 512), "h": _length(rng, 64, 512), "cycles": 2, "hio": 1}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(4, 40), "sizes_seed": rng.randint(0, 1 << 20),
                "cycles": 2, "hio": 2}
    return {"kind": kind, "count": rng.randint(4, 24), "sizes_seed": rng.randint(0, 1 << 20), "lo": 128,
            "hi": rng.choice([512, 1024]), "cycles": 2, "hio": 1}


def _sizes(case):
    """(w, h) of every image of a batch or a burst, from the case alone."""
    r = random.Random(case["sizes_seed"])
    if case["kind"] == "batch":
        return [(n, n) for n in (r.choice(BATCH_SIZES) for _ in range(case["count"]))]
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return [(n, n) for n in (int(round(math.exp(r.uniform(lo, hi)))) for _ in range(case["count"]))]


# ------------------------------------------------------------------ inputs
def _object(w, h, seed, shapes=6):
    """Rectangles and discs of amplitude 0.2 ... 1 in the central half of the
    frame, overlaps keeping the maximum (float64, on the GPU)."""
    r = random.Random(seed * 7919 + w * 31 + h)
    obj = torch.zeros((h, w), dtype=torch.float64, device=DEV)
    c = min(w, h) // 2
    x0, y0 = (w - c) // 2, (h - c) // 2
    yy = torch.arange(c, dtype=torch.float64, device=DEV)[:, None]
    xx = torch.arange(c, dtype=torch.float64, device=DEV)[None, :]
    part = obj[y0:y0 + c, x0:x0 + c]
    for s in range(shapes):
        cx, cy, amp = r.uniform(0, c), r.uniform(0, c), r.uniform(0.2, 1.0)
        hx, hy = r.uniform(0.04, 0.2) * c + 1, r.uniform(0.04, 0.2) * c + 1
        if s % 2 == 0:
            m = ((xx - cx).abs() <= hx) & ((yy - cy).abs() <= hy)
        else:
            m = (xx - cx) ** 2 + (yy - cy) ** 2 <= hx * hx
        part.copy_(torch.maximum(part, torch.where(m, amp, 0.0)))
    return obj


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _intensity(obj):
    f = torch.fft.fft2(obj.to(torch.complex64))
    return f.real.double() ** 2 + f.imag.double() ** 2


def _modulus(w, h, seed):
    return _intensity(_object(w, h, seed)).sqrt().float()


def _params(case):
    return im.default_params(n_cycles=case["cycles"], n_hio_cycles=case["hio"], target_error=FLT_MIN)


def _prepare_hio(case, seed):
    w, h = case["w"], case["h"]
    n = w * h
    obj = _object(w, h, seed)
    gen = _gen(seed)
    inside = obj > 0

    def near():
        # g' of a run that has nearly converged, at the unnormalized transforms' scale
        a, b, c = (torch.randn(h, w, device=DEV, generator=gen).clamp(-3, 3) for _ in range(3))
        re = obj * (1 + 0.002 * a) + torch.where(inside, 0.0, 0.0002 * b)
        return (torch.stack((re, 0.0001 * c), -1) * n).float().contiguous()

    im.check(im.lib().imresh_autotune(w, h, None, None, None))
    return {"case": case, "g": near(), "p": near(), "mask": (~inside).to(torch.uint8),
            "M": _intensity(obj).sqrt().float()}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "hio":
        return _prepare_hio(case, seed)
    if kind == "host":
        m = _modulus(case["w"], case["h"], seed).cpu().numpy()
        im.check(im.lib().imresh_autotune(case["w"], case["h"], None, None, None))
        return {"case": case, "modulus": m, "io": m.copy()}
    if kind in ("batch", "serve"):
        sizes = _sizes(case)
        mods = [_modulus(w, h, seed * 1000 + i) for i, (w, h) in enumerate(sizes)]
        for w, h in sorted(set(sizes)):
            im.check(im.lib().imresh_autotune(w, h, None, None, None))
        s = {"case": case, "moduli": mods, "io": [m.clone() for m in mods], "params": _params(case)}
        if kind == "serve":
            s["server"] = im.Server()
        return s
    if kind == "mask":
        w, h = case["w"], case["h"]
        obj, gen = _object(w, h, seed), _gen(seed)
        g = torch.stack((obj + 0.02 * torch.randn(h, w, device=DEV, generator=gen),
                         0.02 * torch.randn(h, w, device=DEV, generator=gen)), -1).float().contiguous()
        return {"case": case, "g": g, "plane": torch.empty((h, w), device=DEV)}
    if kind == "simulate":
        w, h = case["w"], case["h"]
        obj = _object(w, h, seed).float()
        return {"case": case, "obj": obj, "pattern": torch.empty_like(obj), "seed": int(seed),
                "ideal": _modulus(w, h, seed + 1), "measured": torch.empty_like(obj)}
    if kind == "fft":
        w, h, gen = case["w"], case["h"], _gen(seed)
        x = torch.randn((h, w, 2), device=DEV, generator=gen)
        return {"case": case, "x": x, "f": torch.empty_like(x), "b": torch.empty_like(x)}
    raise ValueError(kind)


# ------------------------------------------------------------------ one pass
def run(s):
    L, case = im.lib(), s["case"]
    kind = case["kind"]
    if kind == "hio":
        im.check(L.imresh_hio_iterations(s["g"].data_ptr(), s["p"].data_ptr(), s["mask"].data_ptr(),
                                         s["M"].data_ptr(), case["w"], case["h"], BETA, case["iters"], None))
        return [s["g"], s["p"]]
    if kind == "host":
        np.copyto(s["io"], s["modulus"])   # the next pattern arrives in the caller's buffer
        r = im.shrink_wrap(s["io"], n_cycles=case["cycles"], n_hio_cycles=case["hio"], target_error=FLT_MIN)
        return {"object": s["io"], "cycles": int(r.cycles_run), "masked": float(r.last_masked)}
    if kind == "batch":
        for a, b in zip(s["io"], s["moduli"]):
            a.copy_(b)
        r = im.shrink_wrap_batch_device([(a.data_ptr(), a.shape[1], a.shape[0]) for a in s["io"]], s["params"])
        return {"objects": s["io"], "masked": [float(x.last_masked) for x in r]}
    if kind == "serve":
        for a, b in zip(s["io"], s["moduli"]):
            a.copy_(b)
        torch.cuda.current_stream().synchronize()   # the server runs on streams of its own
        for a in s["io"]:
            s["server"].submit((a.data_ptr(), a.shape[1], a.shape[0]), s["params"])
        s["server"].drain()
        done = s["server"].completions()
        return {"objects": s["io"], "completed": len(done), "failed": sum(1 for c in done if c[1] != 0)}
    if kind == "mask":
        w, h = case["w"], case["h"]
        n, g, d = w * h, s["g"].data_ptr(), s["plane"].data_ptr()
        v = [im.c_float() for _ in range(4)]
        im.check(L.imresh_complex_norm(d, g, n, None))
        im.check(L.imresh_gaussian_blur(d, w, h, case["sigma"], None))
        im.check(L.imresh_vector_max(d, n, v[0], None))
        im.check(L.imresh_cutoff(d, n, 0.2 * v[0].value, 1.0, 0.0, None))
        im.check(L.imresh_calculate_hio_error(g, d, n, 0, v[1], v[2], v[3], None))
        return {"max": v[0].value, "mask": s["plane"], "error": v[1].value, "masked": v[3].value}
    if kind == "simulate":
        w, h = case["w"], case["h"]
        s["pattern"].copy_(s["obj"])
        im.check(L.imresh_diffraction_intensity_device(s["pattern"].data_ptr(), w, h, None))
        s["measured"].copy_(s["ideal"])
        im.check(L.imresh_poisson_modulus(s["measured"].data_ptr(), w, h, case["photons"], s["seed"], None))
        return {"pattern": s["pattern"], "measured": s["measured"]}
    w, h = case["w"], case["h"]
    im.check(L.imresh_fft2d(s["f"].data_ptr(), s["x"].data_ptr(), w, h, -1, None))
    im.check(L.imresh_fft2d(s["b"].data_ptr(), s["f"].data_ptr(), w, h, 1, None))
    return {"forth": s["f"], "back": s["b"]}


# ------------------------------------------------------------------ work
def _fft2_flops(w, h):
    return 5.0 * w * h * math.log2(max(2, w * h))


def work(case):
    """Each input once, each output once; the arithmetic of the transforms
    (5 n log2 n each) and of the elementwise steps."""
    kind = case["kind"]
    if kind == "hio":   # read g', gPrev, mask, modulus; write g', gPrev
        n = case["w"] * case["h"]
        return {"bytes": 37.0 * n, "flops": case["iters"] * (2 * _fft2_flops(case["w"], case["h"]) + 20.0 * n)}
    if kind in ("host", "batch", "serve"):   # modulus in, object out
        sizes = [(case["w"], case["h"])] if kind == "host" else _sizes(case)
        its = case["cycles"] * case["hio"]
        return {"bytes": float(sum(8 * w * h for w, h in sizes)),
                "flops": float(sum((2 * its + 1) * _fft2_flops(w, h)
                                   + (20 * its + 80 * case["cycles"]) * w * h for w, h in sizes))}
    n = case["w"] * case["h"]
    if kind == "mask":   # g' in, mask out; the two passes of the blur
        return {"bytes": 12.0 * n, "flops": (4.0 * (2 * math.ceil(2.885 * case["sigma"]) + 1) + 10) * n}
    if kind == "simulate":
        return {"bytes": 16.0 * n, "flops": _fft2_flops(case["w"], case["h"]) + 100.0 * n}
    return {"bytes": 32.0 * n, "flops": 2 * _fft2_flops(case["w"], case["h"])}


# ------------------------------------------------------------------ in 64 bits
def _step(g, p, mask, M):
    """One HIO iteration, unnormalized transforms."""
    p = torch.where(mask | (g.real < 0), p - float(np.float32(BETA)) * g, g)
    f = torch.fft.fft2(p)
    a = f.abs()
    f = f * (M / torch.where(a == 0, 1.0, a))
    return torch.fft.ifft2(f, norm="forward"), p


def _taps(sigma):
    r = math.ceil(2.884402748387961466 * sigma - 0.5)
    t = [math.exp(-i * i / (2 * sigma * sigma)) for i in range(-r, r + 1)]
    return [x / sum(t) for x in t], r


def _blurred(x, sigma):
    """Separable Gaussian, the edge repeated."""
    t, r = _taps(sigma)
    for dim in (1, 0):
        n = x.shape[dim]
        at = torch.arange(n, device=x.device)
        x = sum(t[k + r] * x.index_select(dim, (at + k).clamp(0, n - 1)) for k in range(-r, r + 1))
    return x


def _reconstructed(M, cycles, hio):
    """Shrink-wrap with the default parameters: (Re g', masked count)."""
    M = M.to(DEV).double()
    g = torch.fft.ifft2(M.to(torch.complex128), norm="forward")
    p, sigma, masked = g, np.float32(3.0), 0.0
    for c in range(cycles):
        b = _blurred(g.abs(), float(sigma))
        mask = b < float(np.float32(0.04 if c == 0 else 0.20)) * b.max()
        sigma = np.float32(max(np.float32(1.5), (np.float32(1) - np.float32(0.01)) * sigma))
        for _ in range(hio):
            g, p = _step(g, p, mask, M)
        masked = float(mask.sum())
    return g.real, masked


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "hio":
        g, p = (torch.view_as_complex(s[k].double()) for k in ("g", "p"))
        mask, M = s["mask"].bool(), s["M"].double()
        for _ in range(case["iters"]):
            g, p = _step(g, p, mask, M)
        return [torch.view_as_real(g), torch.view_as_real(p)]
    if kind == "host":
        return {"object": _reconstructed(torch.from_numpy(s["modulus"]), case["cycles"], case["hio"])[0],
                "cycles": None, "masked": None}
    if kind == "batch":
        return {"objects": [_reconstructed(m, case["cycles"], case["hio"])[0] for m in s["moduli"]], "masked": None}
    if kind == "serve":
        s["server"].close()
        return {"objects": [_reconstructed(m, case["cycles"], case["hio"])[0] for m in s["moduli"]],
                "completed": None, "failed": None}
    if kind == "mask":   # the cut-off decides by a last bit: the maximum alone has such a value
        top = _blurred(torch.view_as_complex(s["g"].double()).abs(), case["sigma"]).max()
        return {"max": float(top), "mask": None, "error": None, "masked": None}
    if kind == "simulate":   # the counts are random numbers
        return {"pattern": torch.fft.fft2(s["obj"].double()).abs(), "measured": None}
    x = torch.view_as_complex(s["x"].double())
    f = torch.fft.fft2(x)
    return {"forth": torch.view_as_real(f), "back": torch.view_as_real(x * (case["w"] * case["h"]))}
