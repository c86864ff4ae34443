"""A batch of several larger inversions runs in parts on side streams, small ones and ones of equal
size share their launches.  Every inversion equals a batch of
one bit for bit, with launches and replayed as a graph, for one to six inversions of uneven sizes;
and inversions that pass grids to each other (one's realisation is another's seismic input, which
every forward transform reads before a result is written) keep that order."""
import numpy as np
import pytest

import crava_amd as C
import problem as P

pytestmark = pytest.mark.gpu

SIZES = [(20, 18, 40), (9, 11, 30), (30, 12, 25), (12, 12, 60), (16, 25, 35), (8, 7, 45)]


def _item(ctx, k, nreal, sizes=SIZES):
    p = P.make_problem(*sizes[k], seed=100 + k, angles_deg=tuple(np.linspace(0.0, 30.0, 2 + k % 3)))
    mk = lambda ct, n: [C.FFTGrid(ctx, p["nx"], p["ny"], p["nz"], p["nxp"], p["nyp"], p["nzp"], ct) for _ in range(n)]
    nt = p["ntheta"]
    it = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=k, mean_in=mk(C.PARAMETER, 3),
              seis_in=mk(C.DATA, nt), mean=mk(C.PARAMETER, 3), data=mk(C.DATA, nt), cov=mk(C.COVARIANCE, 6),
              out=[mk(C.PARAMETER, 3) for _ in range(nreal)])
    for g, r in zip(it["mean_in"] + it["seis_in"], list(p["mean_real"]) + list(p["seis_real"])):
        g.upload_real(r)
    return it


def _results(it):
    return [g.download_real() for g in it["mean"]] + [g.download_complex() for g in it["cov"]] + \
           [g.download_real() for r in it["out"] for g in r]


def _close(items):
    for it in items:
        for g in it["mean_in"] + it["seis_in"] + it["mean"] + it["data"] + it["cov"] + [g for r in it["out"] for g in r]:
            g.close()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6])
def test_parts_equal_batches_of_one(ctx, n):
    print("parts", n, flush=True)
    items = [_item(ctx, k, k % 3) for k in range(n)]
    want = []
    for it in items:
        b = C.Batch(ctx, [it])
        b.run()
        b.wait()
        want.append(_results(it))
        b.close()
    b = C.Batch(ctx, items)
    for rep in range(3):
        if rep == 1:
            b.use_graph()
        for it in items:
            for g in it["mean"] + it["cov"]:
                g.fillInConstant(-1.0)
        b.run()
        b.wait()
        for it, w in zip(items, want):
            assert all(np.array_equal(x, y) for x, y in zip(_results(it), w)), (n, rep)
    b.close()
    _close(items)


def test_grids_handed_on_keep_the_pass_order(ctx):
    a, c = _item(ctx, 0, 1), _item(ctx, 0, 0)
    b1 = C.Batch(ctx, [c])
    b1.run()
    b1.wait()
    want = _results(c)
    b1.close()
    seis = c["seis_in"][0].download_real(padded=True)
    a["out"][0][0].setType(C.DATA)  # the realisation grid holds the other's seismic cube first
    a["out"][0][0].upload_real(seis)
    shared = dict(c, seis_in=[a["out"][0][0]] + c["seis_in"][1:])
    b = C.Batch(ctx, [a, shared])
    b.run()
    b.wait()
    assert all(np.array_equal(x, y) for x, y in zip(_results(shared), want))
    b.close()
    _close([a, c])


LARGE = [(70, 60, 80), (75, 48, 100), (60, 80, 70), (72, 64, 90), (70, 60, 80)]  # over 2^18 padded cells each


@pytest.mark.parametrize("sizes", [LARGE[:2], LARGE, LARGE[:1] * 3, SIZES[:2], SIZES, SIZES[:1] * 4],
                         ids=["large two", "large five", "large equal", "small two", "small six", "small equal"])
def test_shared_launches(ctx, sizes):
    """x launches of a run: together, each pass (forward, means, realisations) has one per row length;
    parts have their own.  The results are those of batches of one either way."""
    print("launches", sizes, flush=True)
    items = [_item(ctx, k, 1, sizes) for k in range(len(sizes))]
    want = []
    for it in items:
        b = C.Batch(ctx, [it])
        b.run()
        b.wait()
        want.append(_results(it))
        b.close()
    b = C.Batch(ctx, items)
    ctx.set_profiling(True)
    ctx.reset_kernel_time()
    b.run()
    b.wait()
    launches = ctx.kernel_time(C.K_FFT_X)[0]
    ctx.set_profiling(False)
    got = [_results(it) for it in items]
    b.use_graph()
    b.run()
    b.wait()
    for it, w, g in zip(items, want, got):
        assert all(np.array_equal(x, y) for x, y in zip(g, w))
        assert all(np.array_equal(x, y) for x, y in zip(_results(it), w))
    lengths = len({it["mean"][0].nxp for it in items})
    geometries = len({(it["mean"][0].nxp, it["mean"][0].nyp, it["mean"][0].nzp) for it in items})
    print("%d inversions, %d geometries, %d row lengths: %d x launches" % (len(items), geometries, lengths, launches))
    if sizes[0] in LARGE and geometries > 1:
        assert launches == 3 * geometries  # at most four geometries: a part each
    else:
        assert launches == 3 * lengths
    b.close()
    _close(items)


def test_a_part_that_cannot_be_planned(ctx):
    """The second part's z axis is too long for a workgroup's LDS: the batch is refused, what the first
    part held is given back once its copy to the device is over, and other batches run as before."""
    good = _item(ctx, 0, 0, LARGE)
    p = P.make_problem(2, 2, 50, nxp=4, nyp=4, nzp=64, angles_deg=(0.0,))
    for name in ("K", "e1", "e2", "e3", "invert", "rt"):
        p[name] = np.resize(p[name], (7000,) + p[name].shape[1:])
    p.update(nz=6000, nzp=7000)
    mk = lambda ct, n: [C.FFTGrid(ctx, p["nx"], p["ny"], p["nz"], p["nxp"], p["nyp"], p["nzp"], ct) for _ in range(n)]
    bad = dict(tables=p, rxy=p["rxy"], rt=p["rt"], lam2d=p["lam2d"], seed=1, mean_in=mk(C.PARAMETER, 3),
               seis_in=mk(C.DATA, 1), mean=mk(C.PARAMETER, 3), data=mk(C.DATA, 1), cov=mk(C.COVARIANCE, 6), out=[])
    b = C.Batch(ctx, [good])
    b.run()
    b.wait()
    want = _results(good)
    b.close()
    held = ctx.memory()[0]
    for _ in range(3):
        with pytest.raises(C.CravaError, match="too long"):
            C.Batch(ctx, [good, bad])
        assert ctx.memory()[0] == held
    b = C.Batch(ctx, [good])
    b.run()
    b.wait()
    assert all(np.array_equal(x, y) for x, y in zip(_results(good), want))
    b.close()
    _close([good, bad])
