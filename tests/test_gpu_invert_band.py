"""cg_invert's band-limited passes (large grids whose inverted planes are few): only the inverted
frequencies go through the x and y passes, the update comes back and is added to the prior mean.
Against the drop-in sequence on the runtime-plan FFT engine, which computes every wavenumber: odd
and even lengths on every axis, lengths with and without a two-radix split, the longest tables,
planes that are their own mirror, inverted planes whose mirror is not, tables without Hermitian
symmetry (the half-complex inverse keeps the Hermitian part), FP64 re-solves, failures, one and two
angles (updates sharing a work grid), realisations.

Covariances depend on the tables alone: bit for bit.  Means: both sides are FP32 transforms of the
same data, each within about 3e-7 of its largest part; the updates are as large as the means here,
so 5e-6 of the update covers both."""
import numpy as np
import pytest

import crava_amd as C
import problem as P
from conftest import rel_l2

pytestmark = pytest.mark.gpu

CASES = {
    "even": dict(shape=(256, 250, 200), nt=3, nreal=2),
    "odd": dict(shape=(245, 225, 243), nt=5),
    "odd x, even z, one angle": dict(shape=(375, 189, 180), nt=1, high=25.0),
    "two angles": dict(shape=(240, 243, 216), nt=2, nreal=1),
    "long": dict(shape=(1152, 10, 1120), nt=4),
    "long odd": dict(shape=(735, 27, 675), nt=3),
    "eight angles": dict(shape=(280, 216, 225), nt=8, precision=C.PREC_REFERENCE),
    "self-mirrored planes": dict(shape=(252, 240, 210), nt=3, planes=(0, 105, 1, 209, 30, 180)),
    "one-sided planes": dict(shape=(250, 256, 200), nt=3, planes=(20, 21, 190, 100)),
    "re-solves": dict(shape=(256, 250, 200), nt=5, sn=1e8),
    # 72% of the planes: the FP64 list does not fit past the band in a work grid
    "re-solves, wide band": dict(shape=(256, 250, 200), nt=5, sn=1e8, few=4, planes=tuple(range(1, 73)) + tuple(range(128, 200))),
    "failures": dict(shape=(240, 250, 210), nt=3, precision=C.PREC_REFERENCE, fail=True),
}


def _problem(nt, shape, high=55.0, planes=None, sn=5.0, fail=False, **_):
    nxp, nyp, nzp = shape
    p = P.make_problem(14, 3, int(nzp * 0.8), nxp=16, nyp=4, nzp=nzp, angles_deg=tuple(np.linspace(0.0, 40.0, nt)),
                       high_cut=high, sn=sn, seed=nzp)
    rng = np.random.default_rng(nxp)
    p.update(nx=nxp - 3, ny=max(nyp - 3, 1), nxp=nxp, nyp=nyp)
    lateral = np.exp(rng.uniform(-3.0, 1.0, (nyp, nxp // 2 + 1))).astype(np.float32)  # no symmetry
    p["rxy"], p["lam2d"] = lateral, lateral
    p["mean_real"] = rng.standard_normal((3, nzp, nyp, nxp), dtype=np.float32)
    p["seis_real"] = rng.standard_normal((nt, nzp, nyp, nxp), dtype=np.float32)
    if planes is not None:
        inv = np.zeros(nzp, np.int32)
        inv[list(planes)] = 1
        p["invert"] = inv
    if fail:
        p.update(sigma0e=-10.0 * np.abs(p["sigma0e"]) - 1.0, prior_var0=p["prior_var0"] * 1e-12)
    return p


def _z_launches(p, nt):
    """The band sequence's z launches: runs of as many grids as have 96 MB of band planes, forward and
    inverse.  (The shared launches and the drop-in calls have other numbers, which is checked too.)"""
    nxp, nyp, nzp = p["nxp"], p["nyp"], p["nzp"]
    cnxp, n = nxp // 2 + 1, 3 + nt
    both = np.asarray(p["invert"], bool) | np.roll(np.asarray(p["invert"], bool)[::-1], 1)
    cells = int(both[: nzp // 2 + 1].sum()) * 2 * cnxp * nyp
    runs = lambda k, size: -(-k // min(16, max(1, (96 << 20) // size)))
    count = runs(n, 8 * cells) + runs(3, 8 * cells)
    assert 8 * cnxp * nyp * nzp > 48 << 20 and count not in (n + 3, runs(n, 8 * cnxp * nyp * nzp) + runs(3, 8 * cnxp * nyp * nzp))
    return count


@pytest.mark.parametrize("name", list(CASES))
def test_band_matches_dropin(ctx, name):
    kw = CASES[name]
    nt, nreal, prec = kw["nt"], kw.get("nreal", 0), kw.get("precision", C.PREC_MIXED)
    print("band", name, kw, flush=True)
    p = _problem(**kw)
    mk = lambda ct, n: [C.FFTGrid(ctx, p["nx"], p["ny"], p["nz"], p["nxp"], p["nyp"], p["nzp"], ct) for _ in range(n)]
    it = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=5, mean_in=mk(C.PARAMETER, 3),
              seis_in=mk(C.DATA, nt), mean=mk(C.PARAMETER, 3), data=mk(C.DATA, nt), cov=mk(C.COVARIANCE, 6),
              out=[mk(C.PARAMETER, 3) for _ in range(nreal)])
    for g, r in zip(it["mean_in"] + it["seis_in"], list(p["mean_real"]) + list(p["seis_real"])):
        g.upload_real(r)
    res = {}
    for engine in (C.FFT_GENERIC, C.FFT_AUTO):
        ctx.set_fft_engine(engine)
        ctx.set_profiling(True)
        ctx.reset_kernel_time()
        try:
            stats = C.invert(ctx, it, precision=prec, stats=True)
            ctx.sync()
            passes = ctx.kernel_time(C.K_FFT_Z)[0]
        finally:
            ctx.set_profiling(False)
            ctx.set_fft_engine(C.FFT_AUTO)
        res[engine] = (np.stack([g.download_real(padded=True) for g in it["mean"]]),
                       [g.download_complex() for g in it["cov"]],
                       [np.stack([g.download_real() for g in r]) for r in it["out"]], stats, passes)
    (m0, c0, o0, s0, _), (m1, c1, o1, s1, z1) = res[C.FFT_GENERIC], res[C.FFT_AUTO]
    assert s1 == s0
    if not nreal:  # the realisations of a split-z length have z passes of their own
        assert z1 == _z_launches(p, nt)
    if kw.get("sn"):
        assert s1[2] > s1[0] // kw.get("few", 2)  # the wide band's outer planes are well conditioned
    if kw.get("fail"):
        assert s1[0] == s1[1] > 0
    assert all(np.array_equal(a, b) for a, b in zip(c0, c1))
    nxp = p["nxp"]
    assert not np.any(m1[..., nxp:])  # the row padding is zero, as the inverse transform leaves it
    base = p["mean_real"]
    if kw.get("fail"):
        assert np.array_equal(m1[..., :nxp], base)  # no update: the prior mean as it was
        assert rel_l2(m0[..., :nxp], base) < 1e-6
    else:
        e = rel_l2(m1[..., :nxp] - base, m0[..., :nxp] - base)
        print("band %s: mean update %.2e, stats %s, z launches %d" % (name, e, s1, z1), flush=True)
        # re-solved wavenumbers amplify the rounding of the data (S/N 1e8)
        assert e < (5e-3 if kw.get("sn") else 5e-6)
    for a, b in zip(o0, o1):
        assert rel_l2(b, a) < 5e-6
    for g in it["mean_in"] + it["seis_in"] + it["mean"] + it["data"] + it["cov"] + [g for r in it["out"] for g in r]:
        g.close()


@pytest.mark.parametrize("nt", [1, 2, 5])
def test_work_grid_contents_do_not_matter(ctx, nt):
    """The outputs and the work grids may hold anything before the call: the results have the same
    bits after zeros and after NaN.  Odd rows: the columns past the row belong to no pair of traces."""
    print("work grids", nt, flush=True)
    p = _problem(nt, (375, 189, 180), high=25.0)
    mk = lambda ct, n: [C.FFTGrid(ctx, p["nx"], p["ny"], p["nz"], p["nxp"], p["nyp"], p["nzp"], ct) for _ in range(n)]
    it = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=5, mean_in=mk(C.PARAMETER, 3),
              seis_in=mk(C.DATA, nt), mean=mk(C.PARAMETER, 3), data=mk(C.DATA, nt), cov=mk(C.COVARIANCE, 6), out=[])
    for g, r in zip(it["mean_in"] + it["seis_in"], list(p["mean_real"]) + list(p["seis_real"])):
        g.upload_real(r)
    res = []
    for value in (0.0, np.nan):
        before = np.full((p["nzp"], p["nyp"], p["nxp"] // 2 + 1), value + 1j * value, np.complex64)
        for g in it["mean"] + it["data"] + it["cov"]:
            g.upload_complex(before)
        C.invert(ctx, it)
        res.append([g.download_real(padded=True) for g in it["mean"]] + [g.download_complex() for g in it["cov"]])
    for a, b in zip(*res):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
    for g in it["mean_in"] + it["seis_in"] + it["mean"] + it["data"] + it["cov"]:
        g.close()


def test_deferral_list_needs_no_memory():
    """On the split-z geometries a call holds no list of 4 bytes per inverted wavenumber (11 MB here, 409 MB
    at 1152 x 1152 x 384): a budget for the grids and 4 MB more takes another grid after it."""
    nt, shape = 5, (576, 72, 320)
    p = _problem(nt, shape, sn=1e8)
    dims = (p["nx"], p["ny"], p["nz"], *shape)
    grid = C.lib().cg_arena_grid_bytes(*shape)
    with C.Context(0, hbm_budget=23 * grid + (4 << 20)) as own:
        mk = lambda ct, n: [C.FFTGrid(own, *dims, ct) for _ in range(n)]
        it = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=5, mean_in=mk(C.PARAMETER, 3),
                  seis_in=mk(C.DATA, nt), mean=mk(C.PARAMETER, 3), data=mk(C.DATA, nt), cov=mk(C.COVARIANCE, 6), out=[])
        for g, r in zip(it["mean_in"] + it["seis_in"], list(p["mean_real"]) + list(p["seis_real"])):
            g.upload_real(r)
        stats = C.invert(own, it, stats=True)
        print("deferral list", stats, own.memory(), 22 * grid, flush=True)
        assert stats[2] > stats[0] // 2
        C.FFTGrid(own, *dims, C.DATA).close()


def test_alone_and_in_a_batch(ctx):
    """Above the size of the band sequence cg_invert and a batch, which transforms every wavenumber, agree
    to the FP32 rounding of two transform sequences (3e-7 of the means' largest part each; 2e-6 of the
    updates, which are as large); covariances, which depend on the tables alone, bit for bit."""
    p = _problem(5, (256, 250, 200))
    mk = lambda ct, n: [C.FFTGrid(ctx, p["nx"], p["ny"], p["nz"], p["nxp"], p["nyp"], p["nzp"], ct) for _ in range(n)]
    it = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=5, mean_in=mk(C.PARAMETER, 3),
              seis_in=mk(C.DATA, 5), mean=mk(C.PARAMETER, 3), data=mk(C.DATA, 5), cov=mk(C.COVARIANCE, 6),
              out=[mk(C.PARAMETER, 3)])
    for g, r in zip(it["mean_in"] + it["seis_in"], list(p["mean_real"]) + list(p["seis_real"])):
        g.upload_real(r)
    results = lambda: (np.stack([g.download_real() for g in it["mean"]]), [g.download_complex() for g in it["cov"]],
                       np.stack([g.download_real() for g in it["out"][0]]))
    C.invert(ctx, it)
    alone = results()
    b = C.Batch(ctx, [it])
    b.run()
    b.wait()
    batched = results()
    b.close()
    prior = p["mean_real"]
    e = rel_l2(alone[0] - prior, batched[0] - prior), rel_l2(alone[2], batched[2])
    print("alone / in a batch: updates %.2e, realisation %.2e" % e, flush=True)
    assert max(e) < 2e-6
    assert all(np.array_equal(x, y) for x, y in zip(alone[1], batched[1]))
    for g in it["mean_in"] + it["seis_in"] + it["mean"] + it["data"] + it["cov"] + it["out"][0]:
        g.close()


def _factorable(n):
    for q in (2, 3, 5, 7):
        while n % q == 0:
            n //= q
    return n == 1


LENGTHS = [n for n in range(10, 1153) if _factorable(n)]  # shorter z axes do not make a grid of 48 MB


@pytest.mark.parametrize("part", range(6))
def test_every_band_length(ctx, part):
    """z passes of every compiled length (10 .. 1152), x passes of the same, paired so that the grids are
    large enough for the band sequence: against the runtime-plan engine over all wavenumbers, compared
    on the device.  60% of the planes are inverted, with the tables of in-band planes on all of them."""
    base = P.make_problem(14, 3, 50, nxp=16, nyp=4, nzp=64, angles_deg=(0.0, 15.0, 30.0), seed=4)
    inband = np.nonzero(base["invert"])[0]
    worst = 0.0
    for i in range(part, len(LENGTHS), 6):
        nzp, nxp = LENGTHS[i], LENGTHS[-1 - i]
        nyp = next(n for n in range(1, 1153) if _factorable(n) and 8 * (nxp // 2 + 1) * n * nzp > 48 << 20)
        print("band lengths", (nxp, nyp, nzp), flush=True)
        p = dict(base, nx=nxp, ny=nyp, nz=nzp, nxp=nxp, nyp=nyp, nzp=nzp)
        for name in ("K", "e1", "e2", "e3"):
            p[name] = base[name][inband[np.arange(nzp) % len(inband)]]
        p["rt"] = np.full(nzp, base["rt"][inband[0]], np.float32)
        p["invert"] = np.zeros(nzp, np.int32)
        m = int(0.3 * nzp)
        p["invert"][1 : m + 1] = p["invert"][nzp - m :] = 1
        lateral = np.exp(np.random.default_rng(i).uniform(-3.0, 1.0, (nyp, nxp // 2 + 1))).astype(np.float32)
        mk = lambda ct, n: [C.FFTGrid(ctx, nxp, nyp, nzp, nxp, nyp, nzp, ct) for _ in range(n)]
        inputs = dict(mean_in=mk(C.PARAMETER, 3), seis_in=mk(C.DATA, 3))
        for k, g in enumerate(inputs["mean_in"] + inputs["seis_in"]):
            g.add_white_noise(1.0, 10 * i + k)
        res = {}
        for engine in (C.FFT_GENERIC, C.FFT_AUTO):
            it = dict(inputs, tables=p, rxy=lateral, rt=p["rt"], lam2d=lateral, seed=5, mean=mk(C.PARAMETER, 3),
                      data=mk(C.DATA, 3), cov=mk(C.COVARIANCE, 6), out=[])
            ctx.set_fft_engine(engine)
            ctx.set_profiling(True)
            ctx.reset_kernel_time()
            try:
                C.invert(ctx, it)
                ctx.sync()
                launches = ctx.kernel_time(C.K_FFT_Z)[0]
            finally:
                ctx.set_profiling(False)
                ctx.set_fft_engine(C.FFT_AUTO)
            res[engine] = it
        assert launches == _z_launches(p, 3)
        want, got = res[C.FFT_GENERIC], res[C.FFT_AUTO]
        assert np.array_equal(got["cov"][i % 6].download_complex(), want["cov"][i % 6].download_complex())
        for prior, w, g in zip(inputs["mean_in"], want["mean"], got["mean"]):
            prior.multiplyByScalar(-1.0)
            prior.add(w)  # the update
            w.multiplyByScalar(-1.0)
            w.add(g)
            e = (w.sum_squares(True) / prior.sum_squares(True)) ** 0.5
            worst = max(worst, e)
            assert e < 5e-6, (nxp, nyp, nzp, e)
        for it in (want, got):
            for g in it["mean"] + it["data"] + it["cov"]:
                g.close()
        for g in inputs["mean_in"] + inputs["seis_in"]:
            g.close()
    print("band lengths, part %d: worst error of the update %.2e" % (part, worst), flush=True)
