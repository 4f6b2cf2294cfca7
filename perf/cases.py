"""The transforms this framework is timed on, through its public Python entry points.

Every case is what a program that uses the library does again and again: plans
(the library's plan cache, or a batch handle) and buffers are in hand, new data
arrives, one call (or a forward call and the one that undoes it) runs on it.

Kinds of case and the entry points they call:

  c2c     FFT(n).transform               batched rows, either direction
  real    RealFFT(n).forward / .inverse  real rows to a spectrum and back
  fft2    FFT2D(w, h).transform          complex images
  real2   RealFFT2D(w, h).forward / .inverse  a real image to its spectrum and back
  vert    FFTVert(n).transform           transforms down the columns of a matrix
  uneven  UnevenBatch.execute            thousands of transforms of mixed lengths
  filter  spectral_filter and its gradients
  half    fft16                          16-bit storage, FP32 arithmetic, with or without a scale
"""
import math

import numpy as np
import torch

import genfft_amd as G

_REAL = {"c64": torch.float32, "c128": torch.float64}
_CPLX = {"c64": torch.complex64, "c128": torch.complex128}
_CBYTES = {"c64": 8, "c128": 16}
_HALF = {"f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one transform per call: the latency a caller of a plan-per-call library sees (FFT_1D of the
        # reference's benchmark)
        {"name": "c64_1024_single", "kind": "c2c", "prec": "c64", "n": 1024, "batch": 1, "inverse": False},
        # frames of a recording, their number whatever the recording's length gives
        {"name": "c64_512_frames", "kind": "c2c", "prec": "c64", "n": 512, "batch": 3001, "inverse": True},
        # long rows, several hundred MiB at once (range lines of a radar scene)
        {"name": "c64_32768_rows", "kind": "c2c", "prec": "c64", "n": 32768, "batch": 2000, "inverse": False},
        # the headline: a batch of million-point transforms
        {"name": "c64_1M_batch", "kind": "c2c", "prec": "c64", "n": 1 << 20, "batch": 128, "inverse": False},
        # double precision rows (solvers), the way back
        {"name": "c128_16384_rows", "kind": "c2c", "prec": "c128", "n": 16384, "batch": 2048, "inverse": True},
        # real signals to half spectra and back (block convolution of long channels)
        {"name": "f32_65536_there_and_back", "kind": "real", "prec": "c64", "n": 65536, "batch": 1501, "half": True},
        # one large complex image (the 2D benchmark)
        {"name": "c64_image_4096", "kind": "fft2", "prec": "c64", "w": 4096, "h": 4096, "batch": 1, "pad": 0,
         "inverse": False},
        # a real image to its full spectrum and back (image filtering)
        {"name": "f32_image_2048", "kind": "real2", "prec": "c64", "w": 2048, "h": 2048, "pad": 0},
        # columns of a matrix whose width is odd (FFTVert of the reference's tests)
        {"name": "c64_columns_1024x4999", "kind": "vert", "prec": "c64", "n": 1024, "cols": 4999, "pad": 0,
         "inverse": False},
        # requests of mixed lengths gathered into one call
        {"name": "c64_mixed_lengths", "kind": "uneven", "prec": "c64", "jobs": 5000, "lo": 6, "hi": 16, "layout": 0},
        # a training step of a spectral layer: output and both gradients
        {"name": "f32_filter_16384", "kind": "filter", "prec": "c64", "n": 16384, "batch": 256},
        # half-precision storage with the automatic scale
        {"name": "f16_4096_scaled", "kind": "half", "fmt": "f16", "n": 4096, "batch": 4096, "inverse": False,
         "scale": True},
    ]


# A drawn case holds at most this many complex elements of 8 bytes (512 MiB a side).
_MOST = 1 << 26


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _batch(rng, n, most):
    """A batch of transforms of n elements: 2^10 to `most` elements in all, odd ones as often as even ones."""
    return _log(rng, max(1, (1 << 10) // n), max(1, most // n))


def draw(rng):
    kind = rng.choice(["c2c", "c2c", "c2c", "real", "real", "fft2", "real2", "vert", "uneven", "filter", "half"])
    prec = rng.choice(["c64", "c64", "c128"])
    most = _MOST if prec == "c64" else _MOST // 2
    inverse = rng.random() < 0.5
    if kind == "c2c":
        n = 1 << rng.randint(3, 22)
        return {"kind": kind, "prec": prec, "n": n, "batch": _batch(rng, n, most), "inverse": inverse}
    if kind == "real":
        n = 1 << rng.randint(4, 22)
        return {"kind": kind, "prec": prec, "n": n, "batch": _batch(rng, n, most), "half": rng.random() < 0.75}
    if kind == "fft2":
        w, h = 1 << rng.randint(5, 13), 1 << rng.randint(5, 13)
        pad = rng.choice([0, 0, 1, 8])
        # images with padded rows come one or a few at a time
        batch = rng.randint(1, 3) if pad else _batch(rng, w * h, most // 2)
        return {"kind": kind, "prec": prec, "w": w, "h": h, "batch": min(batch, max(1, most // 2 // (w * h))), "pad": pad,
                "inverse": inverse}
    if kind == "real2":
        return {"kind": kind, "prec": prec, "w": 1 << rng.randint(6, 12), "h": 1 << rng.randint(6, 12),
                "pad": rng.choice([0, 0, 1, 6])}
    if kind == "vert":
        n = 1 << rng.randint(3, 14)
        return {"kind": kind, "prec": prec, "n": n, "cols": _log(rng, 3, min(8192, most // 2 // n)),
                "pad": rng.choice([0, 0, 1, 16]), "inverse": inverse}
    if kind == "uneven":
        lo = rng.randint(4, 9)
        return {"kind": kind, "prec": prec, "jobs": _log(rng, 100, 4000), "lo": lo, "hi": rng.randint(lo + 2, 16),
                "layout": rng.randint(1, 1 << 20)}
    if kind == "filter":
        n = 1 << rng.randint(6, 14 if prec == "c64" else 13)
        return {"kind": kind, "prec": prec, "n": n, "batch": _log(rng, 2, (1 << 23) // n)}
    n = 1 << rng.randint(5, 20)
    return {"kind": "half", "fmt": rng.choice(["f16", "bf16"]), "n": n, "batch": _batch(rng, n, _MOST), "inverse": inverse,
            "scale": rng.random() < 0.5}


def _randn(shape, dtype, seed, salt):
    g = torch.Generator(device="cuda").manual_seed(seed * 1009 + salt)
    return torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _layout(case):
    """Lengths, offsets and directions of an uneven batch: a part of the case, the same for every seed."""
    r = np.random.default_rng(case["layout"])
    sizes = (1 << r.integers(case["lo"], case["hi"] + 1, case["jobs"])).astype(np.int64)
    offs = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    return sizes, offs, r.integers(0, 2, case["jobs"]).astype(bool)


def _inputs(case, seed):
    """The data of one call, made from the seed alone."""
    kind = case["kind"]
    if kind == "half":
        # pairs of 16-bit numbers; the transforms' levels lie over four decades, and
        # a program that asks for no scale keeps its spectra far inside float16's range
        x = _randn((case["batch"], case["n"], 2), torch.float32, seed, 1)
        level = 10.0 ** (_randn((case["batch"], 1, 1), torch.float32, seed, 2).clamp(-2, 2))
        x = x * level if case["scale"] else x * level / math.sqrt(case["n"])
        return {"x": x.to(_HALF[case["fmt"]])}
    real, cplx = _REAL[case["prec"]], _CPLX[case["prec"]]
    if kind == "c2c":
        return {"x": _randn((case["batch"], case["n"]), cplx, seed, 1)}
    if kind == "real":
        return {"x": _randn((case["batch"], case["n"]), real, seed, 1)}
    if kind == "fft2":
        return {"x": _randn((case["batch"], case["h"], case["w"] + case["pad"]), cplx, seed, 1)}
    if kind == "real2":
        return {"x": _randn((case["h"], case["w"] + case["pad"]), real, seed, 1)}
    if kind == "vert":
        return {"x": _randn((case["n"], case["cols"] + case["pad"]), cplx, seed, 1)}
    if kind == "uneven":
        return {"x": _randn((int(_layout(case)[0].sum()),), cplx, seed, 1)}
    return {"x": _randn((case["batch"], case["n"]), real, seed, 1), "H": _randn((case["n"] // 2 + 1,), cplx, seed, 2),
            "gy": _randn((case["batch"], case["n"]), real, seed, 3)}


def prepare(case, seed):
    s = {"case": case, **_inputs(case, seed)}
    kind, x = case["kind"], s["x"]
    if kind == "c2c":
        s["fft"], s["y"] = G.FFT(case["n"], x.dtype), torch.empty_like(x)
    elif kind == "real":
        s["fft"] = G.RealFFT(case["n"], x.dtype)
        bins = case["n"] // 2 + 1 if case["half"] else case["n"]
        s["y"] = torch.empty((case["batch"], bins), dtype=_CPLX[case["prec"]], device="cuda")
        s["z"] = torch.empty_like(x)
    elif kind == "fft2":
        s["fft"] = G.FFT2D(case["w"], case["h"], x.dtype)
        s["y"] = torch.empty((case["batch"], case["h"], case["w"]), dtype=x.dtype, device="cuda")
        if case["pad"]:  # a batch with padded rows goes image by image
            s["views"] = [(x[b], s["y"][b]) for b in range(case["batch"])]
    elif kind == "real2":
        s["fft"] = G.RealFFT2D(case["w"], case["h"], x.dtype)
        s["y"] = torch.empty((case["h"], case["w"]), dtype=_CPLX[case["prec"]], device="cuda")
        s["z"] = torch.empty((case["h"], case["w"]), dtype=x.dtype, device="cuda")
    elif kind == "vert":
        s["fft"] = G.FFTVert(case["n"], x.dtype)
        s["y"] = torch.empty((case["n"], case["cols"]), dtype=x.dtype, device="cuda")
    elif kind == "uneven":
        sizes, offs, inv = _layout(case)
        s["fft"] = G.UnevenBatch(sizes, offs, offs, inv, x.dtype)
        s["y"] = torch.empty_like(x)
    elif kind == "filter":
        x.requires_grad_(True)
        s["H"].requires_grad_(True)
    return s


def run(s):
    case = s["case"]
    kind, x = case["kind"], s["x"]
    if kind == "c2c":
        s["fft"].transform(s["y"], x, case["inverse"])
        return s["y"]
    if kind == "real":
        s["fft"].forward(s["y"], x, case["half"])
        if not case["half"]:
            return s["y"]
        s["fft"].inverse(s["z"], s["y"])
        return s["y"], s["z"]
    if kind == "fft2":
        if case["pad"]:
            for a, b in s["views"]:
                s["fft"].transform(b, case["w"], a, case["w"] + case["pad"], case["inverse"])
        else:
            s["fft"].transform(s["y"], case["w"], x, case["w"], case["inverse"], batch=case["batch"])
        return s["y"]
    if kind == "real2":
        s["fft"].forward(s["y"], case["w"], x, case["w"] + case["pad"])
        s["fft"].inverse(s["z"], case["w"], s["y"], case["w"])
        return s["y"], s["z"]
    if kind == "vert":
        s["fft"].transform(s["y"], case["cols"], x, case["cols"] + case["pad"], case["cols"], case["inverse"])
        return s["y"]
    if kind == "uneven":
        s["fft"].execute(x, s["y"])
        return s["y"]
    if kind == "filter":
        y = G.spectral_filter(x, s["H"])
        gx, gH = torch.autograd.grad(y, (x, s["H"]), s["gy"])
        return y.detach(), gx, gH
    y, scales = G.fft16(x, case["inverse"], "auto" if case["scale"] else None)
    return (y, scales) if case["scale"] else y


def work(case):
    """Each input read once and each output written once; 5 N log2 N operations a complex transform, half of it for a
    real one."""
    kind = case["kind"]
    if kind == "half":
        n, b = case["n"], case["batch"]
        return {"bytes": 8 * n * b + (4 * b if case["scale"] else 0), "flops": 5 * n * math.log2(n) * b}
    cb = _CBYTES[case["prec"]]
    if kind == "c2c":
        n, b = case["n"], case["batch"]
        return {"bytes": 2 * cb * n * b, "flops": 5 * n * math.log2(n) * b}
    if kind == "real":
        n, b = case["n"], case["batch"]
        bins = n // 2 + 1 if case["half"] else n
        passes = 2 if case["half"] else 1
        return {"bytes": passes * (n * cb // 2 + bins * cb) * b, "flops": passes * 2.5 * n * math.log2(n) * b}
    if kind == "fft2":
        n, b = case["w"] * case["h"], case["batch"]
        return {"bytes": 2 * cb * n * b, "flops": 5 * n * math.log2(n) * b}
    if kind == "real2":
        n, bins = case["w"] * case["h"], (case["w"] // 2 + 1) * case["h"]
        return {"bytes": 2 * (n * cb // 2) + n * cb + bins * cb, "flops": 5 * n * math.log2(n)}
    if kind == "vert":
        n = case["n"] * case["cols"]
        return {"bytes": 2 * cb * n, "flops": 5 * n * math.log2(case["n"])}
    if kind == "uneven":
        sizes = _layout(case)[0]
        return {"bytes": 2 * cb * int(sizes.sum()), "flops": float((5 * sizes * np.log2(sizes)).sum())}
    n, b = case["n"], case["batch"]
    bins = n // 2 + 1
    # forward: x, H -> y; backward: x, H, gy -> gx, gH; five half-cost transforms
    return {"bytes": (5 * n * cb // 2) * b + 3 * bins * cb, "flops": 5 * 2.5 * n * math.log2(n) * b}


def _dft(x, inverse, dim=-1):
    """The unscaled transform in 64 bits."""
    return torch.fft.ifft(x, dim=dim, norm="forward") if inverse else torch.fft.fft(x, dim=dim)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "half":
        v = torch.view_as_complex(d["x"].double())
        if not case["scale"]:
            return torch.view_as_real(_dft(v, case["inverse"]))
        # the largest power of two up to 1 that keeps n * max(|re| + |im|) within 2^15 (float16) or 2^120 (bfloat16)
        top = d["x"].double().abs().sum(-1).amax(-1) * case["n"] / (2.0 ** 15 if case["fmt"] == "f16" else 2.0 ** 120)
        scales = torch.exp2(-torch.ceil(torch.log2(top.clamp(min=1.0))))
        return torch.view_as_real(_dft(v, case["inverse"]) * scales[:, None]), scales
    x = d["x"].to(torch.complex128 if d["x"].is_complex() else torch.float64)
    if kind == "c2c":
        return _dft(x, case["inverse"])
    if kind == "real":
        return (torch.fft.rfft(x).contiguous(), x * case["n"]) if case["half"] else torch.fft.fft(x)
    if kind == "fft2":
        x = x[:, :, :case["w"]].contiguous()
        return _dft(_dft(x, case["inverse"]), case["inverse"], dim=-2).contiguous()
    if kind == "real2":
        x = x[:, :case["w"]].contiguous()
        return torch.fft.fft(torch.fft.fft(x), dim=0).contiguous(), x * (case["w"] * case["h"])
    if kind == "vert":
        return _dft(x[:, :case["cols"]].contiguous(), case["inverse"], dim=0).contiguous()
    if kind == "uneven":
        sizes, offs, inv = _layout(case)
        y = torch.empty_like(x)
        for n in np.unique(sizes):
            for way in (False, True):
                at = offs[(sizes == n) & (inv == way)]
                if len(at):
                    idx = torch.from_numpy(at).to(x.device)[:, None] + torch.arange(int(n), device=x.device)
                    y[idx] = _dft(x[idx], way)
        return y
    n, H, gy = case["n"], d["H"].to(torch.complex128), d["gy"].double()
    X, Y = torch.fft.rfft(x), torch.fft.rfft(gy)
    w = torch.full((n // 2 + 1,), 2.0 / n, dtype=torch.float64, device=x.device)
    w[0] = w[-1] = 1.0 / n
    # the imaginary parts of the first and last bins of a half spectrum don't count
    flat = lambda s: torch.cat([s[..., :1].real.to(s.dtype), s[..., 1:-1], s[..., -1:].real.to(s.dtype)], -1)  # noqa: E731
    y = torch.fft.irfft(flat(X * H), n)
    gx = torch.fft.irfft(flat(Y * H.conj()), n)
    return y, gx, (w * Y * X.conj()).sum(0)
