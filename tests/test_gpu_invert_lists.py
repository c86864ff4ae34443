"""cg_invert on small grids runs each FFT pass of its grids in shared launches: odd and even lengths,
single rows and planes, more grids than one launch holds, an odd and an even number of realisations,
and the means' work grids being the inputs themselves (which the shared launches do not take).
Against the drop-in calls: bit for bit where they run the same kernels (odd row lengths, and the
covariances, which depend on the tables alone); even row lengths take another forward x pass, whose
FP32 rounding (3e-7 of the largest part on either side) the results then carry."""
import numpy as np
import pytest

import crava_amd as C
import problem as P
from conftest import rel_l2

pytestmark = pytest.mark.gpu

# (nxp, nyp, nzp), angles, realisations; the fifth has 36 MB grids: two to a launch, five in all
CASES = [((12, 10, 16), 3, 2), ((9, 7, 15), 5, 1), ((14, 1, 20), 8, 0), ((15, 6, 21), 4, 3), ((250, 180, 200), 2, 1)]


def _problem(shape, nt):
    nxp, nyp, nzp = shape
    small = nxp * nyp * nzp < 1 << 16
    p = P.make_problem(max(nxp - 2, 1), max(nyp - 2, 1), max(nzp - 4, 1), nxp=nxp, nyp=nyp if small else 2, nzp=nzp,
                       angles_deg=tuple(np.linspace(0.0, 40.0, nt)), seed=nxp)
    if not small:  # the tables of a thin slab, laid over random cubes of the whole size
        rng = np.random.default_rng(1)
        p["nyp"], p["ny"] = nyp, nyp - 2
        for name in ("rxy", "lam2d"):
            p[name] = np.abs(rng.standard_normal((nyp, nxp // 2 + 1))).astype(np.float32)
        p["mean_real"] = rng.standard_normal((3, nzp, nyp, nxp), dtype=np.float32)
        p["seis_real"] = rng.standard_normal((nt, nzp, nyp, nxp), dtype=np.float32)
    return p


def _grids(ctx, p, n, ct, real=None):
    out = [C.FFTGrid(ctx, p["nx"], p["ny"], p["nz"], p["nxp"], p["nyp"], p["nzp"], ct) for _ in range(n)]
    for g, r in zip(out, real if real is not None else ()):
        g.upload_real(r)
    return out


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("in_place", [False, True])
def test_shared_launches_equal_dropin_calls(ctx, case, in_place):
    shape, nt, nreal = CASES[case]
    print("shared launches", shape, nt, nreal, in_place, flush=True)
    p = _problem(shape, nt)
    mean_in, seis_in = _grids(ctx, p, 3, C.PARAMETER, p["mean_real"]), _grids(ctx, p, nt, C.DATA, p["seis_real"])
    mean, data, cov = (_grids(ctx, p, n, t) for n, t in ((3, C.PARAMETER), (nt, C.DATA), (6, C.COVARIANCE)))
    outs = [_grids(ctx, p, 3, C.PARAMETER) for _ in range(nreal)]
    for g, s in zip(mean + data, mean_in + seis_in):
        g.fft_from(s)
    want_stats = C.posterior(ctx, p, mean, data, cov, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], want_residual=False,
                             precision=C.PREC_MIXED)
    for g in mean:
        g.invFFTInPlace()
    for r in range(0, nreal, 2):
        C.simulate(ctx, cov, mean, outs[r], seed=9, realisation=r, next_out=outs[r + 1] if r + 1 < nreal else None)
    want = [g.download_real() for g in mean] + [g.download_complex() for g in cov] + \
           [g.download_real() for r in outs for g in r]
    item = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=9, mean_in=mean_in, seis_in=seis_in,
                mean=mean_in if in_place else mean, data=data, cov=cov, out=outs)
    stats = C.invert(ctx, item, stats=True)
    got = [g.download_real() for g in item["mean"]] + [g.download_complex() for g in cov] + \
          [g.download_real() for r in outs for g in r]
    assert stats == want_stats
    for k, (w, g) in enumerate(zip(want, got)):
        if shape[0] % 2 or in_place or 3 <= k < 9:
            assert np.array_equal(w, g)
        else:
            assert rel_l2(g, w) < 2e-6
    for g in mean_in + seis_in + mean + data + cov + [g for r in outs for g in r]:
        g.close()


def test_every_even_row_length(ctx):
    """The shared launches' x passes (forward, inverse, inverse with the added mean) at every even row
    length that has a plan, 45 rows (no multiple of the rows of any workgroup but the smallest): against
    the runtime-plan engine."""
    def factorable(n):
        for q in (2, 3, 5, 7):
            while n % q == 0:
                n //= q
        return n == 1

    base = P.make_problem(14, 2, 12, nxp=16, nyp=3, nzp=15, angles_deg=(0.0, 20.0), seed=3)
    worst = 0.0
    for nxp in [2 * n for n in range(2, 577) if factorable(n)]:
        rng = np.random.default_rng(nxp)
        p = dict(base, nx=nxp, ny=2, nxp=nxp)
        p["rxy"] = p["lam2d"] = np.exp(rng.uniform(-3.0, 1.0, (3, nxp // 2 + 1))).astype(np.float32)
        real = rng.standard_normal((5, 15, 3, nxp), dtype=np.float32)
        mean_in, seis_in = _grids(ctx, p, 3, C.PARAMETER, real[:3]), _grids(ctx, p, 2, C.DATA, real[3:])
        mean, data, cov = (_grids(ctx, p, n, t) for n, t in ((3, C.PARAMETER), (2, C.DATA), (6, C.COVARIANCE)))
        out = [_grids(ctx, p, 3, C.PARAMETER) for _ in range(2)]
        item = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=9, mean_in=mean_in, seis_in=seis_in,
                    mean=mean, data=data, cov=cov, out=out)
        res = []
        for engine in (C.FFT_GENERIC, C.FFT_AUTO):
            ctx.set_fft_engine(engine)
            try:
                C.invert(ctx, item)
                res.append([g.download_real(padded=True) for g in mean + out[0] + out[1]])
            finally:
                ctx.set_fft_engine(C.FFT_AUTO)
        for want, got in zip(*res):
            e = rel_l2(got, want)
            worst = max(worst, e)
            assert e < 2e-6, (nxp, e)
        for g in mean_in + seis_in + mean + data + cov + [g for r in out for g in r]:
            g.close()
    print("even row lengths: worst rel L2 %.2e" % worst, flush=True)
