"""Which kernel a pass takes (tos_pairs_last_pass): the comparisons of
test_gpu_tile.py hold the pass on the ladder against the general kernel, so
the default run has to be on the ladder there, and off it where a catalogue
has none."""
import ctypes

import numpy as np
import pytest

import tos_amd
from tos_amd import GridSpec, _lib, synth
from test_gpu_tile import CART, GRIDS, OBS, POLAR_GRIDS, close, masked

ALL = GRIDS + [(tos_amd.POLAR,) + s for s in POLAR_GRIDS]


def test_last_pass_refuses_invalid_arguments():
    k = ctypes.c_int32(0)
    assert _lib.lib().tos_pairs_last_pass(None, ctypes.byref(k)) == 1


@pytest.fixture(scope="module")
def lists(dev):
    """The catalogue of test_gpu_tile.py and its pair list for each grid type."""
    cat = masked(synth.lya_catalog(520, area_deg2=40.0, seed=71), 0.05)
    dcat = dev.upload(cat)
    wide = {CART: GridSpec.cartesian(), OBS: GridSpec.observing(), tos_amd.POLAR: GridSpec.polar()}
    out = {t: dcat.pairs(g.max_angular_scale(cat.scale), order=3, nthreads=8) for t, g in wide.items()}
    yield cat, dcat, out
    for p in out.values():
        p.free()
    dcat.free()


@pytest.mark.gpu
@pytest.mark.parametrize("spec", ALL, ids=[f"{s[0]}-{s[1]}-{s[2]}-{s[3][-1]}" for s in ALL])
def test_survey_catalogues_take_the_ladder(dev, lists, spec):
    pairs, grid = lists[2][spec[0]], GridSpec.from_specs(*spec)
    print(f"case: grid {grid.specs} type {grid.type}", flush=True)
    for prec in (tos_amd.FP64, tos_amd.FP32C):
        pairs.run(grid, precision=prec, flags=tos_amd.XI_NO_ZCONST)
        assert pairs.last_pass() == tos_amd.PASS_GENERAL
        pairs.run(grid, precision=prec)
        assert pairs.last_pass() == tos_amd.PASS_LADDER
    pairs.run(grid, precision=tos_amd.FP64, accum=tos_amd.ACC_ALL)
    assert pairs.last_pass() == tos_amd.PASS_LADDER


@pytest.mark.gpu
def test_batches_and_sky_bins(dev, lists):
    pairs, grid = lists[2][CART], GridSpec.cartesian()
    pairs.run_per_skybin(grid, precision=tos_amd.FP32C)
    assert pairs.last_pass() == tos_amd.PASS_GENERAL
    jobs = [(lists[2][t], g, p) for t, g, p in ((CART, grid, tos_amd.FP64), (OBS, GridSpec.observing(), tos_amd.FP32C),
                                                 (tos_amd.POLAR, GridSpec.polar(), tos_amd.FP32C))]
    dev.batch_run(jobs)
    assert [p.last_pass() for p, _, _ in jobs] == [tos_amd.PASS_LADDER] * 3


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["off_ladder", "two_wavelengths", "descending", "overflow", "few_pairs", "shape",
                                    "both_signs"])
def test_passes_without_a_ladder(dev, lists, change):
    cat = lists[0]
    kw = {k: getattr(cat, k).copy() for k in ("value", "loglam", "weight", "distance")}
    n, a, b = cat.n_pix, cat.offsets[40], cat.offsets[41]
    if change == "off_ladder":
        kw["distance"] += np.repeat(np.arange(cat.n_los), cat.counts()).astype(np.float32) * np.float32(1e-2)
    elif change == "two_wavelengths":
        kw["loglam"][n // 2] += np.float32(1e-5)
    elif change == "descending":
        for k in ("distance", "loglam"):
            kw[k][a:b] = kw[k][a:b][::-1]
    elif change == "both_signs":    # half of the ladder behind the origin
        kw["distance"] -= np.float32(np.median(kw["distance"])) + np.float32(0.37)
    elif change == "overflow":
        kw["weight"][n // 3] = kw["value"][n // 3] = 1e30
    c = synth.Catalog(cat.ra, cat.dec, cat.offsets, kw["value"], kw["loglam"], kw["weight"], kw["distance"], cat.zq,
                      cat.scale)
    if change == "few_pairs":
        c = c.subset(np.arange(20))
    grid = GridSpec.cartesian()
    dcat = dev.upload(c)
    pairs = dcat.pairs(grid.max_angular_scale(c.scale), order=3, nthreads=8)
    assert pairs.last_pass() == tos_amd.PASS_NONE
    print(f"case: {change}", flush=True)
    for _ in range(2):
        pairs.run(grid, precision=tos_amd.FP32C, block_size=512 if change == "shape" else 0)
        assert pairs.last_pass() == tos_amd.PASS_GENERAL
    if change != "shape":
        dev.batch_run([(pairs, grid, tos_amd.FP32C)])
        assert pairs.last_pass() == tos_amd.PASS_GENERAL
    pairs.free()
    dcat.free()


@pytest.mark.gpu
@pytest.mark.parametrize("unit", [1e-3, 0.05, 1.0, 10.0])
@pytest.mark.parametrize("polar", [False, True], ids=["cartesian", "polar"])
def test_distances_in_other_units(dev, lists, unit, polar):
    """Edges are tracked from a squared separation on that scales with the
    distances: few pixel pairs take the reference arithmetic in any unit."""
    cat, u = lists[0], np.float32(unit)
    c = synth.Catalog(cat.ra, cat.dec, cat.offsets, cat.value, cat.loglam, cat.weight, cat.distance * u, cat.zq,
                      cat.scale * float(u))
    top = 200.0 * float(u)
    grid = GridSpec.from_specs(tos_amd.POLAR if polar else CART, f"[0:{top!r}]*50",
                               "[0:1]*20" if polar else f"[0:{top!r}]*50", "[3.556:3.735]*1")
    dcat = dev.upload(c)
    pairs = dcat.pairs(grid.max_angular_scale(c.scale), order=3, nthreads=8)
    print(f"case: unit {unit} polar {polar}", flush=True)
    h = pairs.run(grid, precision=tos_amd.FP32C)
    assert pairs.last_pass() == tos_amd.PASS_LADDER
    close(h, *(lambda r: (r.num_pairs, {"didj": r.didj, "wgt": r.wgt}))(
        pairs.run(grid, precision=tos_amd.FP64, flags=tos_amd.XI_NO_ZCONST)))
    # r < 2 Mpc/h of 200 is 1e-4 of the pairs of a uniform sky, and some 1e-4
    # of the rest lie within the error bound of an edge
    assert h.num_guard_rechecks < 0.01 * h.num_pairs_evaluated
    pairs.free()
    dcat.free()


def thinned(cat, keep):
    owner = np.repeat(np.arange(cat.n_los), cat.counts())
    off = np.zeros(cat.n_los + 1, np.int64)
    np.cumsum(np.bincount(owner[keep], minlength=cat.n_los), out=off[1:])
    return synth.Catalog(cat.ra, cat.dec, off, cat.value[keep], cat.loglam[keep], cat.weight[keep],
                         cat.distance[keep], cat.zq, cat.scale)


def passes(dev, cat, grid, n, prec=tos_amd.FP32C):
    """The kernels of n passes over a new pair list, whose results must agree
    with the general kernel's."""
    dcat = dev.upload(cat)
    pairs = dcat.pairs(grid.max_angular_scale(cat.scale), order=3, nthreads=8)
    assert pairs.stats()["num_sightline_pairs_used"] >= 400
    out = []
    for k in range(n):
        print(f"case: {cat.n_los} sightlines {cat.n_pix} pixels grid {grid.specs} pass {k}", flush=True)
        h = pairs.run(grid, precision=prec)
        out.append(pairs.last_pass())
        if k in (0, n - 1):
            ref = pairs.run(grid, precision=tos_amd.FP64, flags=tos_amd.XI_NO_ZCONST)
            close(h, ref.num_pairs, {"didj": ref.didj, "wgt": ref.wgt})
    pairs.free()
    dcat.free()
    return out


# Forms whose visits cost more than the pixel pairs they hold: thinned spectra,
# bins far narrower than the pairs' separations differ, pairs too close to track
COSTLY = {
    "masked": lambda: (thinned(c := synth.lya_catalog(400, area_deg2=130.0, seed=3),
                               np.random.default_rng(5).random(c.n_pix) < 0.03), GridSpec.cartesian()),
    "every_25th": lambda: (thinned(c := synth.lya_catalog(700, area_deg2=100.0, seed=3),
                                   (np.arange(c.n_pix) - np.repeat(c.offsets[:-1], c.counts())) % 25 == 0),
                           GridSpec.cartesian()),
    "narrow_bins": lambda: (synth.lya_catalog(120, area_deg2=40.0, seed=3),
                            GridSpec.from_specs(CART, "[0:200]*2", "[0:200]*4000", "[3.556:3.735]*1")),
    "close_pairs": lambda: (synth.lya_catalog(800, area_deg2=0.2, seed=3),
                            GridSpec.from_specs(CART, "[0:2]*10", "[0:2]*10", "[3.556:3.735]*1")),
}


@pytest.mark.gpu
@pytest.mark.parametrize("form", list(COSTLY))
def test_forms_that_the_ladder_makes_slower(dev, form):
    cat, grid = COSTLY[form]()
    assert passes(dev, cat, grid, 8) == [tos_amd.PASS_GENERAL] * 8


@pytest.mark.gpu
def test_a_small_list_gets_its_plan_once_it_has_paid(dev):
    """The plan of a small, thinned list costs more than a pass gains: the
    first passes go without, later ones have it, for good."""
    cat = synth.lya_catalog(60, area_deg2=5.0, seed=3)
    cat = thinned(cat, np.random.default_rng(5).random(cat.n_pix) < 0.3)
    p = passes(dev, cat, GridSpec.cartesian(), 12)
    assert p[0] == tos_amd.PASS_GENERAL and p[-1] == tos_amd.PASS_LADDER
    assert p == sorted(p)


@pytest.mark.gpu
def test_batches_choose_as_a_whole(dev):
    """Jobs too small for a plan each share the launch's choice, and a sparse
    job stays on the general kernel among full ones."""
    grid = GridSpec.cartesian()
    full = synth.lya_catalog(700, area_deg2=100.0, seed=4)
    sparse = thinned(full, (np.arange(full.n_pix) - np.repeat(full.offsets[:-1], full.counts())) % 25 == 0)
    made = []
    for cat in (full, sparse, synth.lya_catalog(30, area_deg2=3.0, seed=5)):
        dcat = dev.upload(cat)
        made.append((dcat, dcat.pairs(grid.max_angular_scale(cat.scale), order=3, nthreads=8)))
    jobs = [(p, grid, tos_amd.FP32C) for _, p in made]
    for graph in (False, True, True):
        res = dev.batch_run(jobs, use_graph=graph)[0]
        assert [p.last_pass() for _, p in made][:2] == [tos_amd.PASS_LADDER, tos_amd.PASS_GENERAL]
        for (_, p), h in zip(made, res):
            ref = p.run(grid, precision=tos_amd.FP64, flags=tos_amd.XI_NO_ZCONST)
            close(h, ref.num_pairs, {"didj": ref.didj, "wgt": ref.wgt})
            p.run(grid, precision=tos_amd.FP32C)
    for dcat, p in made:
        p.free()
        dcat.free()


@pytest.mark.gpu
def test_catalogue_bytes_count_the_ladder(dev):
    cat = synth.lya_catalog(500, area_deg2=40.0, seed=3)
    grid = GridSpec.cartesian()
    dcat = dev.upload(cat)
    pairs = dcat.pairs(grid.max_angular_scale(cat.scale), order=3, nthreads=8)

    def held():
        n = ctypes.c_int64(0)
        assert _lib.lib().tos_catalog_info(dcat.h, None, None, ctypes.byref(n)) == 0
        return n.value

    before = held()
    pairs.run(grid, precision=tos_amd.FP32C)
    assert pairs.last_pass() == tos_amd.PASS_LADDER
    # three floats a step of a block, and a place for each sightline
    assert held() >= before + 12 * cat.n_pix + 8 * cat.n_los
    pairs.free()
    dcat.free()


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [3e-21, 1e-22, 1e-30])
def test_products_below_the_normal_floats(dev, ora, lists, scale):
    """w1 w2 and (w d)1 (w d)2 round to subnormal floats like the reference's
    (types.h:77-87), and to zero below them."""
    cat = lists[0]
    c = synth.Catalog(cat.ra, cat.dec, cat.offsets, cat.value, cat.loglam, cat.weight * np.float32(scale),
                      cat.distance, cat.zq, cat.scale)
    if scale > 1e-30:
        p = np.float64(np.median(c.weight)) ** 2
        assert 2.0 ** -149 < p < 2.0 ** -126
    grid = GridSpec.cartesian()
    ref = ora.xi_run(c, grid, c.scale, order=3, nthreads=8)["raw"]
    dcat = dev.upload(c)
    pairs = dcat.pairs(grid.max_angular_scale(c.scale), order=3, nthreads=8)
    print(f"case: weights times {scale}", flush=True)
    h = pairs.run(grid, precision=tos_amd.FP64)
    assert pairs.last_pass() == tos_amd.PASS_LADDER
    close(h, ref["num_pairs"], ref)
    assert (scale == 1e-30) == (h.wgt.max() == 0.0)
    a = pairs.run(grid, precision=tos_amd.FP64, accum=tos_amd.ACC_ALL)
    assert pairs.last_pass() == tos_amd.PASS_LADDER
    close(a, ref["num_pairs"], ref)
    pairs.free()
    dcat.free()
