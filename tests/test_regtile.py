"""Tiles held in registers (genfft_amd/csrc/gfft_regtile.h).

Parity with the long-double oracle at the library's bounds (rel-L2 2e-7*log2 N
complex64, 1e-15*log2 N complex128) at the edges of the shapes: tiles with
missing sequences, padded pitches, the smallest batch that takes a row past
the LDS tiles, and overlapping buffers there.
"""
import ctypes
import re

import numpy as np
import pytest
import torch

import oracle_lib as O
from genfft_amd import _capi as C
from test_capi_cpu import desc, explain, field, tiles

PREC = {"c64": (C.GFFT_F32, np.complex64, torch.complex64, O.tol_c64),
        "c128": (C.GFFT_F64, np.complex128, torch.complex128, O.tol_c128)}


def _rand(shape, dt, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(dt)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,batch,pin,pout", [
    ("c64", 16, 33, 1, 0), ("c64", 32, 17, 0, 3), ("c64", 64, 9, 1, 1), ("c64", 128, 17, 0, 0), ("c64", 256, 9, 3, 0),
    ("c64", 512, 5, 0, 1), ("c64", 1024, 3, 0, 0), ("c64", 1024, 1025, 1, 0), ("c64", 2048, 3, 5, 0),
    ("c64", 4096, 2, 0, 1), ("c64", 8192, 1, 0, 0), ("c64", 8192, 5, 3, 1), ("c64", 16384, 3, 0, 7), ("c64", 32768, 96, 0, 0),
    ("c64", 32768, 97, 5, 3),
    ("c128", 16, 17, 0, 1), ("c128", 16, 4099, 0, 0), ("c128", 32, 15, 1, 0), ("c128", 64, 1, 0, 0), ("c128", 64, 4100, 3, 0),
    ("c128", 128, 9, 0, 3), ("c128", 128, 4097, 0, 0), ("c128", 256, 1, 0, 0), ("c128", 256, 13, 1, 0), ("c128", 512, 7, 0, 3), ("c128", 1024, 3, 1, 1),
    ("c128", 2048, 2, 0, 0), ("c128", 4096, 3, 3, 0), ("c128", 8192, 2, 0, 1), ("c128", 16384, 96, 0, 0),
    ("c128", 16384, 97, 1, 5)])
def test_rows_vs_oracle(gpu, prec, n, batch, pin, pout):
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    x = _rand((batch, n + pin), ndt, n + batch)
    tx = torch.from_numpy(x).to(gpu)
    plan = G.Plan(C.GFFT_C2C, n, precision=p, batch=batch, in_dist=n + pin, out_dist=n + pout)
    rows = sorted({0, 1, batch // 2, batch - 1} & set(range(batch)))
    for inv in (False, True):
        y = torch.full((batch, n + pout), 7 + 5j, dtype=tdt, device=gpu)
        plan.execute(tx, y, inverse=inv)
        h = y.cpu().numpy()
        ref = O.fft_ld(np.ascontiguousarray(x[rows, :n]).astype(np.complex128), inv)
        assert O.rel_l2_rows(h[rows, :n], ref).max() <= tol(n)
        full = np.fft.ifft(x[:, :n].astype(np.complex128)) * n if inv else np.fft.fft(x[:, :n].astype(np.complex128))
        assert O.rel_l2_rows(h[:, :n], full).max() <= tol(n)
        if pout:
            assert np.all(h[:-1, n:] == 7 + 5j)  # the gaps stay untouched


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n", [("c64", 32768), ("c128", 16384)])
def test_long_rows_on_overlapping_buffers(gpu, prec, n):
    """Exactly in place, and with the output shifted against the input by part
    of a row and by whole rows, through both execute entry points."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    batch = 97
    x = _rand((batch, n), ndt, 3)
    ref = np.fft.fft(x.astype(np.complex128))
    plan = G.Plan(C.GFFT_C2C, n, precision=p, batch=batch)
    for shift in (0, 2, n // 2, 3 * n):
        buf = torch.zeros(batch * n + shift, dtype=tdt, device=gpu)
        for at_in, at_out in ((0, shift), (shift, 0)):
            src = buf[at_in:at_in + batch * n]
            src.copy_(torch.from_numpy(x.reshape(-1)))
            out = buf[at_out:at_out + batch * n]
            plan.execute(src, out)
            assert O.rel_l2_rows(out.cpu().numpy().reshape(batch, n), ref).max() <= tol(n)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,lg", [("c64", (13, 14, 15)), ("c128", (12, 13, 14))])
@pytest.mark.parametrize("count", [3, 96])
def test_uneven_batches_of_long_rows(gpu, prec, lg, count):
    """Job tables with odd offsets through the register-held rows."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    sizes = [1 << (lg[i % 3] if count < 96 else lg[2] if i else lg[0]) for i in range(count + 1)]
    offs = np.cumsum([1] + [s + 1 for s in sizes[:-1]])
    inv = np.arange(len(sizes)) % 2 == 1
    x = _rand(int(offs[-1] + sizes[-1]), ndt, 9)
    tx = torch.from_numpy(x).to(gpu)
    y = torch.zeros_like(tx)
    b = G.UnevenBatch(sizes, offs, offs, inv, tdt)
    for mode in ("graph", "eager"):
        y.zero_()
        b.execute(tx, y, mode=mode)
        h = y.cpu().numpy()
        for o, s, i in zip(offs, sizes, inv):
            v = x[o:o + s].astype(np.complex128)
            ref = np.fft.ifft(v) * s if i else np.fft.fft(v)
            assert O.rel_l2(h[o:o + s], ref) <= tol(s)


def test_long_rows_route():
    """From 96 rows on a row past the LDS tiles is one launch; smaller batches,
    lengths beyond and a tuned split keep the four-step.  The plan's workspace
    stays the four-step's, which calls on overlapping buffers run in."""
    for prec, n in ((C.GFFT_F32, 1 << 15), (C.GFFT_F64, 1 << 14)):
        for batch, one in ((95, False), (96, True), (400, True)):
            st, text = explain(desc(prec=prec, n=n, batch=batch))
            assert st == C.GFFT_OK
            assert text.count("long_row ") == (1 if one else 0)
            assert ("on overlapping buffers" in text) == one
            assert f"scratch_bytes={batch * n * (8 << prec)}\n" in text
        st, text = explain(desc(prec=prec, n=2 * n, batch=400))
        assert st == C.GFFT_OK and "long_row" not in text


def test_layouts_past_32_bit_offsets_keep_the_lds_tiles():
    """A tile of several rows whose last row lies 2^31 bytes or more from its
    first is not register-held (its accesses are 32-bit offsets)."""
    for dist, reg in ((256, True), (1 << 24, True), (1 << 25, False)):
        st, text = explain(desc(prec=C.GFFT_F64, n=256, batch=8, ind=dist, outd=dist))
        assert st == C.GFFT_OK
        assert (field(tiles(text)[0], "rad") == "8,4,8,0") == reg


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,batch,pin,pout", [
    ("c64", 128, 9, 0, 1), ("c64", 256, 5, 2, 0), ("c64", 512, 3, 2, 2), ("c64", 512, 1, 0, 0), ("c64", 512, 8193, 0, 0), ("c64", 1024, 9, 0, 2), ("c64", 2048, 5, 0, 0), ("c64", 4096, 3, 2, 4),
    ("c64", 8192, 2, 0, 0), ("c64", 16384, 3, 4, 2), ("c64", 32768, 2, 0, 0), ("c64", 65536, 96, 0, 0),
    ("c64", 65536, 97, 2, 4), ("c128", 256, 5, 0, 1), ("c128", 512, 3, 2, 0), ("c128", 1024, 2, 0, 0),
    ("c128", 2048, 3, 0, 2), ("c128", 4096, 3, 0, 0), ("c128", 8192, 2, 2, 0),
    ("c128", 16384, 2, 0, 2), ("c128", 32768, 96, 0, 0), ("c128", 32768, 97, 2, 2)])
def test_real_rows_vs_float64(gpu, prec, n, batch, pin, pout):
    """Half and full spectra and the way back, dense and padded (pin: reals,
    pout: bins), against numpy's float64 transform at the complex bounds."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    rdt = np.float32 if prec == "c64" else np.float64
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (batch, n + pin)).astype(rdt)
    tx = torch.from_numpy(x).to(gpu)
    ref = np.fft.fft(x[:, :n].astype(np.float64))
    for half in (True, False):
        bins = n // 2 + 1 if half else n
        y = torch.full((batch, bins + pout), 7 + 5j, dtype=tdt, device=gpu)
        G.Plan(C.GFFT_R2C, n, precision=p, batch=batch, in_dist=n + pin, out_dist=bins + pout, half=half).execute(tx, y)
        h = y.cpu().numpy()
        assert O.rel_l2_rows(h[:, :bins], ref[:, :bins]).max() <= tol(n)
        if pout:
            assert np.all(h[:-1, bins:] == 7 + 5j)
    X = ref[:, :n // 2 + 1].astype(ndt)
    X[:, 0] += 3j  # ignored, as in any c2r
    X[:, -1] -= 2j
    z = torch.full((batch, n + pin), 9, dtype=torch.float32 if prec == "c64" else torch.float64, device=gpu)
    G.Plan(C.GFFT_C2R, n, precision=p, batch=batch, out_dist=n + pin).execute(torch.from_numpy(X).to(gpu), z, inverse=True)
    h = z.cpu().numpy()
    assert O.rel_l2_rows(h[:, :n] / n, x[:, :n]).max() <= 2 * tol(n)
    if pin:
        assert np.all(h[:-1, n:] == 9)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n", [("c64", 65536), ("c128", 32768)])
def test_long_real_rows_in_place(gpu, prec, n):
    """Dense half spectra over their own reals: bins of one row lie where the
    next row's reals are, so the call runs the plan's two-launch form."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    rdt = torch.float32 if prec == "c64" else torch.float64
    batch, bins = 96, n // 2 + 1
    x = np.random.default_rng(1).uniform(-1, 1, (batch, n)).astype(np.float32 if prec == "c64" else np.float64)
    buf = torch.zeros(batch * bins, dtype=tdt, device=gpu)
    reals = torch.view_as_real(buf).reshape(-1)[:batch * n]
    reals.copy_(torch.from_numpy(x.reshape(-1)))
    G.Plan(C.GFFT_R2C, n, precision=p, batch=batch, half=True).execute(reals, buf)
    h = buf.cpu().numpy().reshape(batch, bins)
    assert O.rel_l2_rows(h, np.fft.rfft(x.astype(np.float64))).max() <= tol(n)
    G.Plan(C.GFFT_C2R, n, precision=p, batch=batch).execute(buf, reals, inverse=True)
    assert O.rel_l2_rows(reals.cpu().numpy().reshape(batch, n) / n, x).max() <= 2 * tol(n)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["f16", "bf16"])
@pytest.mark.parametrize("n,batch,pin,pout", [
    (32, 33, 0, 0), (32, 5, 1, 3), (64, 17, 0, 2), (128, 9, 1, 0), (256, 5, 0, 1), (512, 3, 3, 3), (512, 5, 0, 0),
    (1024, 3, 0, 0), (2048, 2, 1, 1), (4096, 1, 0, 0), (8192, 2, 0, 5), (16384, 2, 3, 0)])
def test_half_rows_and_their_scale(gpu, fmt, n, batch, pin, pout):
    """16-bit rows with the automatic scale, a given scale and none, at padded
    pitches, both directions.  The scale is exactly the largest power of two up
    to 1 with n * max(|re| + |im|) * scale <= 2^15 (FP16) or 2^120 (BF16); the
    values are within one storage rounding plus the FP32 transform's bound."""
    import genfft_amd as G
    prec, tdt, u, top = (C.GFFT_F16, torch.float16, 2.0 ** -11, 2.0 ** 15) if fmt == "f16" else \
        (C.GFFT_BF16, torch.bfloat16, 2.0 ** -8, 2.0 ** 120)
    g = torch.Generator().manual_seed(n + batch)
    x = (torch.randn(batch, n + pin, 2, generator=g) * 10.0 ** torch.arange(batch).remainder(4).view(-1, 1, 1)).to(tdt)
    v = torch.view_as_complex(x[:, :n].double())
    l1 = x[:, :n].float().abs().sum(-1).amax(-1).double() * n / top
    auto = torch.exp2(-torch.ceil(torch.log2(l1.clamp(min=1.0))))
    plan = G.Plan(C.GFFT_C2C, n, precision=prec, batch=batch, in_dist=n + pin, out_dist=n + pout)
    tx = x.to(gpu)
    for inv in (False, True):
        ref = torch.fft.ifft(v, norm="forward") if inv else torch.fft.fft(v)
        for mode in ("auto", "given", "none"):
            y = torch.full((batch, n + pout, 2), 5.0, dtype=tdt, device=gpu)
            s = (auto / 4).float().to(gpu) if mode == "given" else torch.zeros(batch, device=gpu)
            if mode == "none":
                if fmt == "f16" and float(auto.min()) < 1:
                    continue  # would overflow
                plan.execute(tx, y, inverse=inv)
                want = torch.ones(batch, dtype=torch.float64)
            else:
                plan.execute_scaled(tx, y, s, mode == "auto", inverse=inv)
                want = s.cpu().double()
            if mode == "auto":
                assert torch.equal(want, auto)
            h = torch.view_as_complex(y.cpu()[:, :n].double().contiguous())
            r = ref * want[:, None]
            err = (h - r).abs().square().sum(-1).sqrt() / r.abs().square().sum(-1).sqrt()
            # FP16 outputs below 2^-14 round to multiples of 2^-24
            floor = 2.0 ** -25 * (2 * n) ** 0.5 / r.abs().square().sum(-1).sqrt() if fmt == "f16" else 0.0
            assert bool((err <= u + O.tol_c64(n) + floor).all())
            if pout:
                assert bool((y.cpu()[:-1, n:] == 5.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,pitch", [(4, 4, 4), (8, 16, 11), (32, 32, 32), (16, 64, 20), (2, 64, 3)])
def test_scale_of_small_images(gpu, w, h, pitch):
    """The scale pass of images of up to 1024 elements, dense and padded."""
    import genfft_amd as G
    batch = 37
    g = torch.Generator().manual_seed(w * h)
    x = (torch.randn(batch, h, pitch, 2, generator=g) * 10.0 ** torch.arange(batch).remainder(4).view(-1, 1, 1, 1)).half()
    x[:, :, w:] = 60000.0  # gaps don't count
    l1 = x[:, :, :w].float().abs().sum(-1).amax((-1, -2)).double() * (w * h) / 2.0 ** 15
    plan = G.Plan(C.GFFT_C2C_2D, w, precision=C.GFFT_F16, n2=h, batch=batch, in_stride=pitch, out_stride=w)
    y = torch.empty(batch, h, w, 2, dtype=torch.float16, device=gpu)
    s = torch.zeros(batch, device=gpu)
    plan.execute_scaled(x.to(gpu), y, s, True)
    assert torch.equal(s.cpu().double(), torch.exp2(-torch.ceil(torch.log2(l1.clamp(min=1.0)))))
    ref = torch.fft.fft2(torch.view_as_complex(x[:, :, :w].double().contiguous())) * s.cpu().double().view(-1, 1, 1)
    got = torch.view_as_complex(y.cpu().double())
    assert float((got - ref).norm() / ref.norm()) <= 2 * 2.0 ** -11 + O.tol_c64(max(2, w * h))


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,cols,pin,pout", [
    ("c64", 32, 1, 0, 0), ("c64", 32, 17, 0, 1), ("c64", 32, 16390, 0, 0), ("c64", 64, 16385, 1, 0), ("c64", 64, 32768, 0, 0),
    ("c64", 128, 8200, 0, 0), ("c64", 256, 4112, 0, 1), ("c64", 512, 4100, 0, 0),
    ("c64", 64, 3, 0, 0), ("c64", 64, 17, 1, 0), ("c64", 128, 9, 0, 1), ("c64", 256, 1, 0, 0), ("c64", 256, 15, 2, 1),
    ("c64", 512, 7, 0, 0), ("c64", 512, 4111, 0, 1), ("c64", 1024, 5, 1, 1), ("c64", 1024, 1030, 0, 0),
    ("c64", 1024, 4097, 1, 0), ("c64", 2048, 3, 0, 0), ("c64", 2048, 1027, 0, 3), ("c64", 2048, 4112, 0, 0),
    ("c64", 4096, 2, 1, 0), ("c64", 4096, 1026, 0, 0), ("c64", 4096, 3100, 0, 2),
    ("c128", 32, 1, 0, 0), ("c128", 32, 4098, 1, 0), ("c128", 32, 32768, 0, 0), ("c128", 64, 7, 0, 0), ("c128", 64, 8199, 0, 1),
    ("c128", 128, 3, 0, 1), ("c128", 128, 4100, 0, 0), ("c128", 256, 5, 1, 0), ("c128", 256, 2050, 0, 0), ("c128", 512, 3, 0, 0),
    ("c128", 512, 2056, 0, 0), ("c128", 1024, 2, 0, 1), ("c128", 1024, 2049, 0, 0), ("c128", 2048, 1, 0, 0),
    ("c128", 2048, 2049, 1, 1)])
def test_columns_vs_float64(gpu, prec, n, cols, pin, pout):
    """Column tiles with missing columns, at aligned and odd pitches, on
    aligned and shifted buffers, against numpy's float64 transform."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    x = _rand((n, cols + pin), ndt, n + cols)
    for inv, shift in ((False, 0), (True, 1)):
        src = torch.zeros(n * (cols + pin) + shift, dtype=tdt, device=gpu)[shift:]
        src.copy_(torch.from_numpy(x.reshape(-1)))
        out = torch.full((n * (cols + pout) + shift,), 7 + 5j, dtype=tdt, device=gpu)[shift:]
        G.FFTVert(n, tdt).transform(out, cols + pout, src, cols + pin, cols, inv)
        h = out.cpu().numpy().reshape(n, cols + pout)
        v = x[:, :cols].astype(np.complex128)
        ref = np.fft.ifft(v, axis=0) * n if inv else np.fft.fft(v, axis=0)
        assert O.rel_l2_rows(np.ascontiguousarray(h[:, :cols].T), np.ascontiguousarray(ref.T)).max() <= tol(n)
        if pout:
            assert np.all(h[:, cols:] == 7 + 5j)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,batch", [
    ("c64", 1 << 15, 3), ("c64", 1 << 16, 2), ("c64", 1 << 17, 3), ("c64", 1 << 19, 16), ("c64", 1 << 21, 9),
    ("c64", 1 << 22, 3), ("c64", 1 << 23, 2), ("c128", 1 << 14, 3), ("c128", 1 << 15, 2), ("c128", 1 << 17, 2),
    ("c128", 1 << 21, 3), ("c128", 1 << 22, 2)])
def test_four_step_vs_float64(gpu, prec, n, batch):
    """The splits and register-held passes of long transforms, both directions."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    x = _rand((batch, n), ndt, 11)
    tx = torch.from_numpy(x).to(gpu)
    for inv in (False, True):
        h = G.fft(tx, inverse=inv).cpu().numpy()
        v = x.astype(np.complex128)
        ref = np.fft.ifft(v) * n if inv else np.fft.fft(v)
        assert O.rel_l2_rows(h, ref).max() <= tol(n)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,w,h,batch,pad", [
    ("c64", 256, 128, 16, 0), ("c64", 1024, 128, 24, 0), ("c64", 1024, 128, 25, 0), ("c64", 512, 512, 2, 1),
    ("c128", 64, 128, 7, 0), ("c128", 64, 128, 64, 0), ("c128", 64, 128, 65, 0), ("c128", 128, 256, 9, 3)])
def test_batches_of_images(gpu, prec, w, h, batch, pad):
    """2D batches at the edges of where the row pass streams its stores and
    the columns run in its tile order, on aligned and shifted buffers."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    x = _rand((batch, h, w + pad), ndt, w + batch)
    plan = G.Plan(C.GFFT_C2C_2D, w, precision=p, n2=h, batch=batch, in_stride=w + pad, out_stride=w + pad)
    for inv, shift in ((False, 0), (True, 1)):
        src = torch.zeros(x.size + shift, dtype=tdt, device=gpu)[shift:]
        src.copy_(torch.from_numpy(x.reshape(-1)))
        out = torch.full((x.size + shift,), 7 + 5j, dtype=tdt, device=gpu)[shift:]
        plan.execute(src, out, inverse=inv)
        got = out.cpu().numpy().reshape(x.shape)
        v = x[:, :, :w].astype(np.complex128)
        ref = np.fft.ifft2(v) * (w * h) if inv else np.fft.fft2(v)
        assert O.rel_l2_rows(np.ascontiguousarray(got[:, :, :w]).reshape(batch, -1), ref.reshape(batch, -1)).max() <= tol(w * h)
        if pad:
            assert np.all(got[:, :, w:] == 7 + 5j)


@pytest.mark.parametrize("kind,prec,n,few,many,narrow,wide", [
    (C.GFFT_R2C, 0, 1 << 21, 2, 8, "8", "16"), (C.GFFT_R2C, 0, 1 << 22, 1, 4, "8", "16"),
    (C.GFFT_R2C, 1, 1 << 21, 1, 4, "4", "8"), (C.GFFT_C2C, 0, 1 << 21, 1, 4, "8", "16"),
    (C.GFFT_C2C, 1, 1 << 21, 1, 4, "4", "8")])
def test_small_batches_of_long_transforms_keep_the_narrow_columns(kind, prec, n, few, many, narrow, wide):
    """The wide 2048-row column tiles held in registers are taken once they
    number the 256 CUs (complex64 real 2^21 x 2: 67.7 us with 64 of them, 62.9
    with 128 narrow ones)."""
    for batch, m in ((few, narrow), (many, wide)):
        st, text = explain(desc(kind, prec, n, 0, batch, flags=C.GFFT_FLAG_HALF if kind == C.GFFT_R2C else 0))
        cols = [t for t in tiles(text) if field(t, "L") == "2048" and field(t, "inp") == "1"]
        assert st == 0 and [field(t, "M") for t in cols] == [m], text


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,gap,lines", [("c64", 1 << 21, 0, True), ("c64", 1 << 21, 16, True), ("c64", 1 << 21, 1, False),
                                              ("c64", 1 << 22, 5, False), ("c128", 1 << 20, 8, True), ("c128", 1 << 21, 3, False)])
def test_uneven_jobs_place_the_runs(gpu, prec, n, gap, lines):
    """The register-held column sides of a batch's four-steps know from the jobs'
    offsets whether their runs cover whole lines: odd ones are stored plain."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    count = 10
    offs = np.arange(count) * (n + gap)
    x = torch.randn(count * (n + gap), dtype=tdt, device=gpu)
    y = torch.zeros_like(x)
    plan = G.UnevenBatch([n] * count, offs.tolist(), offs.tolist(), [False] * count, tdt)
    text = plan.describe()
    for t in tiles(text):
        reg_side = field(t, "L") == "2048"  # 512- and 1024-point passes keep the LDS tiles here
        if reg_side and field(t, "outp") == "1" and field(t, "inp") == "0":
            assert (field(t, "lines"), field(t, "plain")) == (("1", "0") if lines else ("0", "1")), t
        elif reg_side:
            assert field(t, "lines") == ("1" if lines else "0"), t
    assert any(field(t, "L") == "2048" for t in tiles(text)) or n < 1 << 21
    plan.execute(x, y)
    idx = torch.from_numpy(offs[[0, count - 1]])[:, None].to(gpu) + torch.arange(n, device=gpu)
    ref = O.fft_ld(x[idx].cpu().numpy().astype(np.complex128))
    assert O.rel_l2_rows(y[idx].cpu().numpy(), ref).max() <= tol(n)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,m", [("c64", 64, 16), ("c64", 256, 8), ("c64", 1024, 4), ("c64", 2048, 4), ("c64", 4096, 4),
                                      ("c128", 128, 8), ("c128", 256, 4), ("c128", 1024, 4), ("c128", 2048, 4)])
def test_partly_filled_column_tiles(gpu, prec, n, m):
    """The last column tile with every number of columns, of infinities beside it
    none: sequences past the last one are computed on that one's elements."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    for cols in [*range(1, m), *range(2 * m + 1, 3 * m)]:
        x = torch.randn(n, cols + 1, dtype=tdt, device=gpu)
        x[:, cols] = float("inf")  # the pitch's gap
        y = torch.full((n, cols + 2), 7 + 5j, dtype=tdt, device=gpu)
        f = G.FFTVert(n, tdt)
        for inv in (False, True):
            f.transform(y, cols + 2, x, cols + 1, cols, inv)
            v = x[:, :cols].cpu().numpy().astype(np.complex128)
            ref = np.fft.ifft(v, axis=0) * n if inv else np.fft.fft(v, axis=0)
            got = y.cpu().numpy()
            assert O.rel_l2_rows(np.ascontiguousarray(got[:, :cols].T), np.ascontiguousarray(ref.T)).max() <= tol(n), cols
            assert np.all(got[:, cols:] == 7 + 5j)


@pytest.mark.parametrize("prec,n,cols,m", [
    (0, 256, 3968, "16"), (0, 256, 2560, "8"), (0, 256, 3959, "8"), (0, 512, 2816, "16"), (0, 2048, 1408, "8"),
    (0, 2048, 1403, "4"), (0, 128, 7936, "32"), (0, 64, 14336, "16"), (1, 128, 3584, "8"), (1, 1024, 1408, "8"),
    (0, 4096, 2048, "8"), (0, 4096, 1024, "4"), (0, 4096, 2052, "4"), (0, 2048, 4700, "8"), (0, 2048, 5301, "8"),
    (0, 2048, 5800, "16"), (0, 2048, 4800, "16")])
def test_column_tile_widths(prec, n, cols, m):
    """Whole columns on whole lines take the wide tile from two thirds of a round
    of the CUs on, short ones and partial lines from a full round."""
    st, text = explain(desc(C.GFFT_COLS, prec, n, cols, 1, ins=cols, outs=cols))
    t = tiles(text)
    assert st == 0 and len(t) == 1 and field(t[0], "M") == m, text


def test_half_lines_are_streamed():
    """Rows of a matrix a multiple of 64 bytes apart are stored like whole lines
    (plain=0), from 8 to 16 MiB of 32 bytes; complex64 1024 rows past 40 MiB."""
    for n, cols, plain in ((2048, 5000, "0"), (2048, 5004, "1"), (2048, 5001, "1"), (256, 5000, "0"), (256, 5004, "0"),
                           (256, 12804, "1"), (256, 5002, "1"), (1024, 5000, "1"), (1024, 5608, "0"), (512, 12808, "0")):
        st, text = explain(desc(C.GFFT_COLS, 0, n, cols, 1, ins=cols, outs=cols))
        t = tiles(text)
        assert st == 0 and [field(x, "plain") for x in t] == [plain], (n, cols, text)


def test_pitches_that_crowd_keep_neighbours_together():
    """From 256 rows on, columns whose row distance is 2, 4 or 8 times an odd
    number of 123 to 133 lines of 128 bytes take the tile order that keeps
    neighbours on one XCD (order=1)."""
    for prec, n, lines, order in ((0, 256, 500, "1"), (0, 512, 492, "1"), (0, 512, 532, "1"), (0, 256, 1000, "1"),
                                  (0, 1024, 250, "1"), (1, 512, 254, "1"), (0, 512, 484, "0"), (0, 512, 540, "0"),
                                  (0, 256, 504, "0"), (0, 256, 512, "0"), (0, 256, 501, "0"), (0, 128, 500, "0"), (0, 128, 1000, "1"),
                                  (1, 512, 256, "0"), (0, 512, 125, "0")):
        cols = lines * (8 if prec else 16)
        t = tiles(explain(desc(C.GFFT_COLS, prec, n, cols, 1, ins=cols, outs=cols))[1])
        assert [field(x, "order") for x in t] == [order], (prec, n, lines)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,cols,pin,pout", [
    ("c64", 256, 8000, 0, 0), ("c64", 512, 4063, 1, 33), ("c128", 512, 2000, 48, 0)])
def test_columns_at_those_pitches(gpu, prec, n, cols, pin, pout):
    test_columns_vs_float64(gpu, prec, n, cols, pin, pout)


def test_short_passes_by_pitch_and_size():
    """Half-line columns of 128 and 256 rows run on the LDS tiles (256 threads)
    between 8 and 20 MiB; the rows before sub-passes of 64 or 128 points are
    streamed where all of them would be dirty at the end."""
    for n, cols, nt in ((256, 9208, "256"), (256, 12808, "512"), (128, 9208, "256"), (256, 9200, "512"), (256, 9204, "512")):
        t = tiles(explain(desc(C.GFFT_COLS, 0, n, cols, 1, ins=cols, outs=cols))[1])
        assert field(t[0], "NT") == nt, (n, cols)
    for w, h, batch, plain in ((128, 8192, 2, "0"), (128, 8192, 4, "1"), (256, 8192, 1, "0"), (256, 4096, 2, "1")):
        t = tiles(explain(desc(C.GFFT_C2C_2D, 0, w, h, batch))[1])
        assert field(t[0], "plain") == plain, (w, h, batch)


@pytest.mark.parametrize("prec,n,rows,half,m", [
    (0, 1024, 40000, False, "1"), (0, 1024, 45000, False, "8"), (0, 1024, 60000, True, "1"), (0, 4096, 6000, False, "1"),
    (0, 4096, 6500, False, "2"), (0, 4096, 16000, True, "1"), (1, 1024, 12000, False, "1"), (1, 1024, 13000, False, "4"),
    (1, 1024, 30000, True, "1"), (1, 2048, 6500, False, "2"), (1, 2048, 6500, True, "1")])
def test_large_full_spectra_take_the_lds_rows(prec, n, rows, half, m):
    """Full spectra past the Infinity Cache are written in one run a row."""
    st, text = explain(desc(C.GFFT_R2C, prec, n, 0, rows, flags=C.GFFT_FLAG_HALF if half else 0))
    line = [ln for ln in text.splitlines() if ln.startswith("real_rows")]
    assert st == 0 and len(line) == 1 and field(line[0], "M") == m, text


@pytest.mark.gpu
@pytest.mark.parametrize("n,rows,full", [(4096, 6200, True), (1024, 12700, True), (2048, 6300, True), (8192, 3, True),
                                         (8192, 257, False)])
def test_f64_real_rows_at_the_limits(gpu, n, rows, full):
    """Either side of kFull, and the 8192-point rows, against numpy."""
    import genfft_amd as G
    for b in (rows - 120 if rows > 1000 else rows, rows):
        x = torch.randn(b, n, dtype=torch.float64, device=gpu)
        bins = n if full else n // 2 + 1
        y = torch.full((b, bins), 7 + 5j, dtype=torch.complex128, device=gpu)
        f = G.RealFFT(n, torch.float64)
        f.forward(y, x, not full)
        at = [0, b // 2, b - 1]
        ref = np.fft.fft(x[at].cpu().numpy())[:, :bins]
        assert O.rel_l2_rows(y[at].cpu().numpy(), np.ascontiguousarray(ref)).max() <= O.tol_c128(n)
        assert _worst_rows(y, torch.fft.fft(x)[:, :bins]) <= 2 * O.tol_c128(n)
        if not full:
            z = torch.empty_like(x)
            f.inverse(z, y)
            assert float(((z / n - x).norm(dim=1) / x.norm(dim=1)).max()) <= 2 * O.tol_c128(n)


def _worst_rows(y, ref):
    return float(((y - ref).abs().square().sum(-1) / ref.abs().square().sum(-1)).max().sqrt())


# rel-L2 against 64 bits of the radix-16 and radix-8 tiles these kernels took over from
ROUNDING = [("c2c", 4096, 64, 1.2147e-7), ("c2c", 8192, 64, 1.2520e-7), ("c2c", 16384, 64, 1.3298e-7),
            ("c2c", 32768, 100, 1.3851e-7), ("c2c", 1 << 16, 256, 1.4303e-7), ("c2c", 1 << 17, 128, 1.4741e-7),
            ("c2c", 1 << 18, 128, 1.5299e-7), ("c2c", 1 << 19, 64, 1.5703e-7), ("c2c", 1 << 20, 64, 1.6302e-7),
            ("cols", 1024, 4999, 1.0904e-7), ("cols", 2048, 2048, 1.1477e-7), ("r2c", 32768, 200, 1.3994e-7),
            ("r2c", 65536, 200, 1.4616e-7)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,count,was", ROUNDING)
def test_rounding_is_no_larger_than_before(gpu, kind, n, count, was):
    """Radix 32 has one more stage of inner twiddles than radix 16, which its
    exact constants make up for.  0.3% for the sample (2^18 values and more)."""
    import genfft_amd as G
    g = torch.Generator(device=gpu).manual_seed(1)
    if kind == "r2c":
        x = torch.randn(count, n, device=gpu, generator=g)
        y = torch.empty(count, n // 2 + 1, dtype=torch.complex64, device=gpu)
        G.RealFFT(n, torch.float32).forward(y, x, True)
        ref = torch.fft.rfft(x.double())
    elif kind == "cols":
        x = torch.randn(n, count, dtype=torch.complex64, device=gpu, generator=g)
        y = torch.empty_like(x)
        G.FFTVert(n, torch.complex64).transform(y, count, x, count, count)
        ref = torch.fft.fft(x.to(torch.complex128), dim=0)
    else:
        x = torch.randn(count, n, dtype=torch.complex64, device=gpu, generator=g)
        y = torch.empty_like(x)
        G.FFT(n, torch.complex64).forward(y, x)
        ref = torch.fft.fft(x.to(torch.complex128))
    err = float((y.to(torch.complex128) - ref).norm() / ref.norm())
    assert err <= 1.003 * was, err


def test_short_half_rows_without_a_scale():
    """The LDS tile where both sides just fill the Infinity Cache and the call
    finds no scale of its own; the register-held one finds it."""
    for n, mb, two, bf in ((32, 64, False, False), (32, 90, True, True), (64, 128, True, True), (128, 128, True, False),
                           (128, 80, False, False), (128, 160, False, False), (256, 128, False, False)):
        st, text = explain(desc(C.GFFT_C2C, C.GFFT_BF16, n, 0, (mb << 20) // (4 * n)))
        assert st == 0 and ("without an automatic scale:" in text) == bf, (n, mb)
        st, text = explain(desc(C.GFFT_C2C, C.GFFT_F16, n, 0, (mb << 20) // (4 * n)))
        assert st == 0 and ("without an automatic scale:" in text) == two, (n, mb)
        if two:
            own, given = [ln for ln in text.splitlines() if ln.startswith("tile")]
            assert field(own, "NT") != field(given, "NT") or field(own, "M") != field(given, "M")


def test_description_needs_one_buffer():
    """A buffer of the length a short one is told holds the whole text."""
    lib = C.lib()
    d = desc(C.GFFT_C2C, 0, 1 << 16, 0, 300)
    assert lib.gfft_plan_explain(ctypes.byref(d), ctypes.create_string_buffer(80), 80) != 0
    need = int(re.search(r"\((\d+) bytes needed", lib.gfft_last_error().decode()).group(1))
    buf = ctypes.create_string_buffer(need)
    assert lib.gfft_plan_explain(ctypes.byref(d), buf, need) == 0
    assert "xcd_four_step" in buf.value.decode() and "on overlapping buffers:" in buf.value.decode()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,mb", [(32, 73), (64, 100), (128, 149), (256, 101)])
def test_short_half_rows_both_ways(gpu, fmt, n, mb):
    """With no scale and the automatic one."""
    import genfft_amd as G
    batch = (mb << 20) // (4 * n)
    x = (torch.randn(batch, n, 2, device=gpu) * 0.1).to(fmt)
    v = torch.view_as_complex(x[:1000].float()).to(torch.complex128)
    ref = torch.fft.fft(v)
    eps = 2.0 ** (-10 if fmt == torch.float16 else -7)
    (plain, _), (auto, scales) = G.fft16(x), G.fft16(x, scale="auto")
    for y in (plain, auto):
        got = torch.view_as_complex(y[:1000].float()).to(torch.complex128)
        assert float((got - ref).norm() / ref.norm()) <= eps
    assert bool((scales == 1).all())
    assert float((auto.float() - plain.float()).norm() / plain.float().norm()) <= eps  # every row
