"""Four-steps that run both passes in one launch, a transform per XCD
(genfft_amd/csrc/kern_xcd.hip), against numpy's float64 transform at the
library's bounds (rel-L2 2e-7*log2 N complex64, 1e-15*log2 N complex128)."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest
import torch

import oracle_lib as O
from genfft_amd import _capi as C
from test_capi_cpu import desc, explain, field

PREC = {"c64": (C.GFFT_F32, np.complex64, torch.complex64, O.tol_c64),
        "c128": (C.GFFT_F64, np.complex128, torch.complex128, O.tol_c128)}
SHAPES = [("c64", 1 << 16, 147, 5, 3), ("c64", 1 << 16, 150, 0, 0), ("c64", 1 << 17, 82, 0, 1), ("c64", 1 << 18, 81, 1, 0),
          ("c128", 1 << 15, 98, 0, 0), ("c128", 1 << 15, 203, 1, 3), ("c128", 1 << 16, 130, 0, 0), ("c128", 1 << 17, 66, 0, 1),
          ("c64", 1 << 19, 50, 1, 0), ("c64", 1 << 20, 25, 0, 0), ("c64", 1 << 20, 33, 0, 1),
          ("c128", 1 << 18, 42, 0, 1)]


def test_route(monkeypatch):
    """Taken from where the ring fits the two launches' workspace, which stays
    what it was; by untuned complex batches only."""
    for prec, n, least in ((0, 1 << 16, 145), (0, 1 << 17, 81), (0, 1 << 18, 81), (1, 1 << 15, 97), (1, 1 << 16, 129),
                           (1, 1 << 17, 65), (0, 1 << 19, 49), (0, 1 << 20, 25), (1, 1 << 18, 41)):
        for batch in (least - 1, least + 1):
            st, text = explain(desc(C.GFFT_C2C, prec, n, 0, batch))
            head = text.split("on overlapping buffers:")
            assert st == 0 and ("xcd_four_step" in head[0]) == (batch > least)
            assert f"scratch_bytes={batch * n * (8 << prec)}\n" in head[0]
            if batch > least:
                assert "xcd" not in head[1] and head[1].count("tile L=") == 2
    for d in (desc(C.GFFT_C2C, C.GFFT_F16, 1 << 16, 0, 600), desc(C.GFFT_C2C, 0, 1 << 21, 0, 100),
              desc(C.GFFT_C2C, 0, 1 << 16, 0, 600, flags=C.GFFT_FLAG_NO_WORKSPACE)):
        assert "xcd" not in explain(d)[1]
    monkeypatch.setenv("GFFT_N1_LOG2", "7")
    assert "xcd" not in explain(desc(C.GFFT_C2C, 0, 1 << 16, 0, 600))[1]


@pytest.mark.parametrize("prec,n,batch,lens,m,ring,lag", [
    (0, 1 << 16, 300, "256,256", 16, 18, 10), (0, 1 << 17, 100, "256,512", 16, 10, 5), (0, 1 << 18, 100, "512,512", 16, 10, 6),
    (0, 1 << 19, 64, "1024,512", 16, 6, 3), (0, 1 << 20, 128, "1024,1024", 16, 4, 2), (0, 1 << 20, 26, "1024,1024", 16, 3, 1),
    (1, 1 << 15, 105, "128,256", 16, 12, 7), (1, 1 << 16, 140, "256,256", 8, 16, 10), (1, 1 << 17, 70, "256,512", 8, 8, 4),
    (1, 1 << 18, 64, "512,512", 8, 5, 2)])
def test_shape(prec, n, batch, lens, m, ring, lag):
    """The one launch a batch runs, ahead of the launches for overlapping buffers."""
    st, text = explain(desc(C.GFFT_C2C, prec, n, 0, batch))
    lines = text.split("on overlapping buffers:")[0].splitlines()[1:]
    assert st == 0 and len(lines) == 1 and lines[0].startswith("xcd_four_step ")
    assert [field(lines[0], k) for k in ("L", "M", "batch", "ring", "lag", "in", "out", "first", "last")] == [
        lens, str(m), str(batch), str(ring), str(lag), "in+0", "out+0", "1", "1"]


HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs the compiler")
def test_ring_is_read_at_agent_scope(tmp_path):
    """Row tiles read what other CUs' workgroups stored in the same launch: every
    one-launch kernel loads the ring at the scope of an agent (sc1), past its
    own CU's cache, and column stores are waited for before they are counted."""
    csrc = os.path.join(os.path.dirname(C.LIB_PATH), "csrc")
    asm = str(tmp_path / "xcd.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--offload-device-only", "-S", os.path.join(csrc, "kern_xcd.hip"), "-o", asm],
                   check=True, capture_output=True)
    kernels = re.split(r"^(?=\S*xcd_fft_kernel\S*:)", open(asm).read(), flags=re.M)[1:]
    assert len(kernels) >= 9
    for text in kernels:
        name, body = text.split(":")[0], text.split(".end_amdhsa_kernel")[0]
        loads = re.findall(r"^\s*buffer_load_dwordx([24])\b(.*)$", body, flags=re.M)
        wide = "4" if "kernelId" in name else "2"
        assert len(loads) >= 8 and all(w == wide and "sc1" in rest.split() for w, rest in loads), (name, loads[:4])
        # streamed loads are the column tiles'; the rest are twiddles
        assert "buffer_inv sc0" not in body and re.search(r"s_waitcnt vmcnt\(0\)", body), name


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,batch,pin,pout", SHAPES)
def test_vs_float64(gpu, prec, n, batch, pin, pout):
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    rng = np.random.default_rng(n + batch)
    x = (rng.uniform(-1, 1, (batch, n + pin)) + 1j * rng.uniform(-1, 1, (batch, n + pin))).astype(ndt)
    tx = torch.from_numpy(x).to(gpu)
    plan = G.Plan(C.GFFT_C2C, n, precision=p, batch=batch, in_dist=n + pin, out_dist=n + pout)
    assert "xcd_four_step" in plan.describe()
    v = x[:, :n].astype(np.complex128)
    for inv in (False, True):
        ref = np.fft.ifft(v) * n if inv else np.fft.fft(v)
        for _ in range(2):  # the counters start over
            y = torch.full((batch, n + pout), 7 + 5j, dtype=tdt, device=gpu)
            plan.execute(tx, y, inverse=inv)
            h = y.cpu().numpy()
            assert O.rel_l2_rows(np.ascontiguousarray(h[:, :n]), ref).max() <= tol(n)
            if pout:
                assert np.all(h[:-1, n:] == 7 + 5j)


@pytest.mark.gpu
@pytest.mark.parametrize("shift", [0, 1, 3 << 16])
def test_overlapping_buffers(gpu, shift):
    """In place, and with the output shifted against the input (two launches)."""
    import genfft_amd as G
    n, batch = 1 << 16, 147
    buf = torch.zeros(batch * n + shift, dtype=torch.complex64, device=gpu)
    rng = np.random.default_rng(shift)
    x = (rng.uniform(-1, 1, (batch, n)) + 1j * rng.uniform(-1, 1, (batch, n))).astype(np.complex64)
    buf[:batch * n].copy_(torch.from_numpy(x.reshape(-1)))
    out = buf[shift:shift + batch * n]
    G.Plan(C.GFFT_C2C, n, batch=batch).execute(buf[:batch * n], out)
    h = out.cpu().numpy().reshape(batch, n)
    assert O.rel_l2_rows(h, np.fft.fft(x.astype(np.complex128))).max() <= O.tol_c64(n)


@pytest.mark.gpu
def test_two_streams_and_a_graph(gpu):
    """One plan from two streams, whose calls share its ring, and replays."""
    import genfft_amd as G
    n, batch = 1 << 15, 100
    g = torch.Generator().manual_seed(3)
    x = [torch.randn(batch, n, dtype=torch.complex128, generator=g).to(gpu) for _ in range(2)]
    y = [torch.empty_like(t) for t in x]
    ref = [torch.fft.fft(t.cpu()) for t in x]
    plan = G.Plan(C.GFFT_C2C, n, precision=C.GFFT_F64, batch=batch)
    side = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for k in range(4):
        with torch.cuda.stream(side[k % 2]):
            plan.execute(x[k % 2], y[k % 2])
    torch.cuda.synchronize()
    for a, b in zip(y, ref):
        assert float(((a.cpu() - b).norm(dim=1) / b.norm(dim=1)).max()) <= O.tol_c128(n)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.execute(x[0], y[0])
    for k in range(3):
        y[0].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert float(((y[0].cpu() - ref[0]).norm(dim=1) / ref[0].norm(dim=1)).max()) <= O.tol_c128(n)


@pytest.mark.gpu
def test_in_an_uneven_batch(gpu):
    import genfft_amd as G
    rng = np.random.default_rng(9)
    sizes = np.concatenate([np.full(147, 1 << 16), np.full(20, 1 << 12), np.full(3, 1 << 17)])
    rng.shuffle(sizes)
    offs = np.concatenate([[1], 1 + np.cumsum(sizes + rng.integers(0, 3, len(sizes)))[:-1]])
    dirs = rng.integers(0, 2, len(sizes))
    total = int(offs[-1] + sizes[-1])
    x = torch.from_numpy((rng.uniform(-1, 1, total) + 1j * rng.uniform(-1, 1, total)).astype(np.complex64))
    plan = G.UnevenBatch(sizes.tolist(), offs.tolist(), offs.tolist(), [bool(d) for d in dirs], torch.complex64)
    assert "xcd_four_step" in plan.describe()
    tx = x.to(gpu)
    for _ in range(2):
        y = torch.zeros_like(tx)
        plan.execute(tx, y)
        h = y.cpu().numpy()
        for n, o, d in zip(sizes, offs, dirs):
            v = x.numpy()[o:o + n].astype(np.complex128)
            ref = np.fft.ifft(v) * n if d else np.fft.fft(v)
            assert O.rel_l2_rows(h[o:o + n][None], ref[None]).max() <= O.tol_c64(n)


@pytest.mark.gpu
def test_tuned_and_saved(gpu, tmp_path):
    """The autotuner times the one-launch form beside the others, and a saved
    choice of it loads as one."""
    import genfft_amd as G
    n, batch = 1 << 17, 82
    try:
        rep = G.autotune(n, batch, torch.complex64, reps=3)
        assert sum(c["n1_log2"] == 0 and c["row_variant"] < 0 for c in rep["candidates"]) == 1
        path = str(tmp_path / "t.json")
        G.save_tuning(path)
        C.check(C.lib().gfft_tuning_clear())
        G.load_tuning(path)
        text = G.Plan(C.GFFT_C2C, n, batch=batch).describe()
        assert ("xcd_four_step" in text) == (rep["best"]["n1_log2"] == 0)
    finally:
        C.check(C.lib().gfft_tuning_clear())


# (prec, n, batch of at least three times the ring's slots, slots, chunk limit)
WRAPS = [("c64", 1 << 16, 450, 144, 0), ("c64", 1 << 17, 250, 80, 0), ("c64", 1 << 18, 245, 80, 0),
         ("c64", 1 << 19, 150, 48, 0), ("c64", 1 << 20, 100, 32, 0), ("c64", 1 << 20, 75, 24, 200 << 20),
         ("c128", 1 << 15, 300, 96, 0), ("c128", 1 << 16, 390, 128, 0), ("c128", 1 << 17, 200, 64, 0),
         ("c128", 1 << 18, 125, 40, 0)]


def _gpu_rand(shape, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _worst(y, ref):
    return float(((y - ref).abs().square().sum(-1) / ref.abs().square().sum(-1)).max().sqrt())


@pytest.mark.gpu
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("prec,n,batch,slots,chunk", WRAPS)
def test_ring_goes_round(gpu, monkeypatch, prec, n, batch, slots, chunk, in_place):
    """Every ring reused at least three times over: each transform against the
    two launches (bound: both sides' tolerances), three of them against the
    long-double oracle."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    assert batch >= 3 * slots
    x = _gpu_rand((batch, n), tdt, n)
    if chunk:
        monkeypatch.setenv("GFFT_CHUNK_BYTES", str(chunk))
    one = G.Plan(C.GFFT_C2C, n, precision=p, batch=batch)
    assert f"batch={batch} ring={slots // 8} " in one.describe()
    monkeypatch.setenv("GFFT_DUAL", "0")
    two = G.Plan(C.GFFT_C2C, n, precision=p, batch=batch)
    assert "xcd" not in two.describe()
    ref = torch.empty_like(x)
    two.execute(x, ref)
    y = x.clone() if in_place else torch.empty_like(x)
    for k in range(1 if in_place else 2):
        one.execute(y if in_place else x, y)
        assert _worst(y, ref) <= 2 * tol(n)
    rows = [0, batch // 2, batch - 1]
    want = O.fft_ld(x[rows].cpu().numpy().astype(np.complex128))
    assert O.rel_l2_rows(y[rows].cpu().numpy(), want).max() <= tol(n)


@pytest.mark.gpu
def test_ring_goes_round_in_an_uneven_batch(gpu):
    """Two classes of it in one batch, jobs of both directions an odd number of
    elements apart, one after the other through one workspace."""
    import genfft_amd as G
    rng = np.random.default_rng(4)
    sizes = np.concatenate([np.full(450, 1 << 16), np.full(250, 1 << 17), np.full(40, 1 << 9)])
    rng.shuffle(sizes)
    offs = np.concatenate([[0], np.cumsum(sizes + rng.integers(0, 4, len(sizes)))[:-1]])
    dirs = rng.integers(0, 2, len(sizes)).astype(bool)
    x = _gpu_rand((int(offs[-1] + sizes[-1]),), torch.complex64, 4)
    y = torch.zeros_like(x)
    G.UnevenBatch(sizes.tolist(), offs.tolist(), offs.tolist(), dirs.tolist(), torch.complex64).execute(x, y)
    for n in (1 << 9, 1 << 16, 1 << 17):
        for inv in (False, True):
            at = offs[(sizes == n) & (dirs == inv)]
            idx = torch.from_numpy(at)[:, None].to(gpu) + torch.arange(n, device=gpu)
            v, got = x[idx], y[idx]
            one = G.FFT(n, torch.complex64)
            for k in range(0, len(at), 60):  # short batches: two launches
                ref = torch.empty_like(v[k:k + 60])
                one.transform(ref, v[k:k + 60].contiguous(), inv)
                assert _worst(got[k:k + 60], ref) <= 2 * O.tol_c64(n)


@pytest.mark.gpu
def test_two_plans_at_once(gpu):
    """Two plans with rings of their own on two streams at the same time."""
    import genfft_amd as G
    cases = [(torch.complex64, C.GFFT_F32, 1 << 17, 200), (torch.complex128, C.GFFT_F64, 1 << 15, 300)]
    plans = [G.Plan(C.GFFT_C2C, n, precision=p, batch=b) for _, p, n, b in cases]
    x = [_gpu_rand((b, n), dt, n) for dt, _, n, b in cases]
    ref = [torch.empty_like(t) for t in x]
    for pl, a, r in zip(plans, x, ref):
        pl.execute(a, r)
    for (dt, _, n, b), a, r in zip(cases, x, ref):
        assert O.rel_l2_rows(r[[0, b - 1]].cpu().numpy(), np.fft.fft(a[[0, b - 1]].cpu().numpy().astype(np.complex128))
                             ).max() <= (O.tol_c64(n) if dt == torch.complex64 else O.tol_c128(n))
    side = [torch.cuda.Stream(), torch.cuda.Stream()]
    y = [[torch.empty_like(t) for _ in range(3)] for t in x]
    torch.cuda.synchronize()
    for k in range(3):
        for i in (0, 1):
            with torch.cuda.stream(side[i]):
                plans[i].execute(x[i], y[i][k])
    torch.cuda.synchronize()
    for i in (0, 1):
        for k in range(3):
            assert torch.equal(y[i][k], ref[i])  # the same kernel on the same input


def test_layouts_whose_runs_share_lines():
    """Distances that leave the runs on parts of lines: taken but where the two
    launches are faster (complex64 2^18 and 2^19 with odd output distances)."""
    def one(prec, n, batch, pin, pout):
        st, text = explain(desc(C.GFFT_C2C, prec, n, 0, batch, ind=n + pin, outd=n + pout))
        assert st == 0
        return "xcd_four_step" in text
    for n, small, large in ((1 << 18, 130, 250), (1 << 19, 80, 130)):
        assert one(0, n, small, 0, 0) and one(0, n, small, 1, 0) and one(0, n, small, 0, 4)
        assert not one(0, n, small, 0, 1) and one(0, n, large, 0, 1)
        assert not one(0, n, small, 3, 5) and not one(0, n, large, 3, 5)
    for prec, n, batch in ((0, 1 << 16, 146), (0, 1 << 17, 82), (0, 1 << 20, 26), (1, 1 << 15, 98), (1, 1 << 16, 130),
                           (1, 1 << 17, 66)):
        assert one(prec, n, batch, 0, 1) and one(prec, n, batch, 3, 5)
    assert one(1, 1 << 18, 42, 0, 1) and not one(1, 1 << 18, 42, 3, 5) and one(1, 1 << 18, 70, 3, 5)


@pytest.mark.gpu
@pytest.mark.parametrize("pin,pout,shift_in,shift_out", [(1, 0, 0, 0), (0, 1, 0, 0), (3, 5, 0, 0), (4, 4, 0, 0), (0, 0, 1, 0),
                                                         (0, 0, 0, 1), (0, 0, 3, 2)])
@pytest.mark.parametrize("prec,n,batch", [("c64", 1 << 16, 150), ("c64", 1 << 17, 90), ("c64", 1 << 18, 90), ("c64", 1 << 19, 52),
                                          ("c64", 1 << 20, 28), ("c64", 1 << 20, 40), ("c128", 1 << 15, 105),
                                          ("c128", 1 << 16, 140), ("c128", 1 << 17, 70), ("c128", 1 << 18, 44)])
def test_alignments(gpu, monkeypatch, prec, n, batch, pin, pout, shift_in, shift_out):
    """Odd distances and odd base addresses, whichever kernel they take, against
    the two launches on whole lines."""
    import genfft_amd as G
    p, ndt, tdt, tol = PREC[prec]
    v = _gpu_rand((batch, n), tdt, n)
    x = torch.zeros(shift_in + batch * (n + pin), dtype=tdt, device=gpu)[shift_in:]
    x.view(batch, n + pin)[:, :n] = v
    y = torch.full((shift_out + batch * (n + pout),), 7 + 5j, dtype=tdt, device=gpu)
    out = y[shift_out:]
    plan = G.Plan(C.GFFT_C2C, n, precision=p, batch=batch, in_dist=n + pin, out_dist=n + pout)
    plan.execute(x, out)
    ref = torch.empty_like(v)
    monkeypatch.setenv("GFFT_DUAL", "0")
    G.Plan(C.GFFT_C2C, n, precision=p, batch=batch).execute(v, ref)
    got = out.view(batch, n + pout)
    assert _worst(got[:, :n], ref) <= 2 * tol(n)
    assert bool((y[:shift_out] == 7 + 5j).all()) and bool((got[:-1, n:] == 7 + 5j).all())
    # an odd output base of 2^18 and 2^19 runs as two launches
    two = shift_out and prec == "c64" and n in (1 << 18, 1 << 19)
    if not pin and not pout:
        assert len(plan.profile(x, out)) == (2 if two else 1)


@pytest.mark.gpu
def test_untuned_candidate_is_listed_once(gpu):
    """2^20 has two rings; the autotuner times its untuned plan once."""
    import genfft_amd as G
    try:
        rep = G.autotune(1 << 20, 26, torch.complex64, reps=1)
        assert sum(c["n1_log2"] == 0 and c["row_variant"] < 0 for c in rep["candidates"]) == 1
    finally:
        C.check(C.lib().gfft_tuning_clear())
