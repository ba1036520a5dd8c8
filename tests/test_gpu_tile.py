"""The pass on a pixel ladder (csrc/tos_tilepass.hip: catalogues whose pixels
share one set of (distance, loglam) steps) against the CPU oracle and against
the general pair kernel on the same pair list (a work-scheme flag selects
it): counts bit-exact, sums within 1e-10 relative (both add the reference's
f32 products in FP64; the orders differ).

The grids are those where the tiles' edge tracking can go wrong: axis-1 bins
narrower than the spread of a tile, axes starting above 0 or below it, an axis
that ends far inside the pair list, z axes with several bins and one that
leaves its axis, more bins than one LDS histogram holds (bands of axis-0
rows), theta bins below and past the axis."""
import numpy as np
import pytest

import tos_amd
from tos_amd import GridSpec, synth
from conftest import SUM_RTOL, rel_err, signed_sum_err

pytestmark = pytest.mark.gpu

CART, OBS = tos_amd.CARTESIAN, tos_amd.OBSERVING


def masked(cat, fraction, seed=5):
    """Pixels taken out at random, every tenth sightline reduced to 1 pixel."""
    rng = np.random.default_rng(seed)
    keep = rng.random(cat.n_pix) >= fraction
    owner = np.repeat(np.arange(cat.n_los), cat.counts())
    first = np.zeros(cat.n_pix, bool)
    first[cat.offsets[:-1]] = True
    keep = np.where(owner % 10 == 3, first, keep)
    off = np.zeros(cat.n_los + 1, np.int64)
    np.cumsum(np.bincount(owner[keep], minlength=cat.n_los), out=off[1:])
    return synth.Catalog(cat.ra, cat.dec, off, cat.value[keep], cat.loglam[keep], cat.weight[keep],
                         cat.distance[keep], cat.zq, cat.scale)


@pytest.fixture(scope="module")
def dev():
    with tos_amd.Device(0) as d:
        yield d


@pytest.fixture(scope="module")
def field():
    cat = masked(synth.lya_catalog(520, area_deg2=40.0, seed=71), 0.05)
    # coincident and nearly coincident sightlines (K = 2 (1 - c) of 0 and ~1e-12)
    cat.ra[7], cat.dec[7] = cat.ra[6], cat.dec[6]
    cat.ra[9], cat.dec[9] = cat.ra[8] + 1e-6, cat.dec[8]
    return cat


def close(h, ref_cnt, ref):
    assert np.array_equal(h.num_pairs.astype(np.int64), np.asarray(ref_cnt).astype(np.int64))
    assert signed_sum_err(h.didj, ref["didj"], ref["wgt"]) <= SUM_RTOL
    assert rel_err(h.wgt, ref["wgt"]) <= SUM_RTOL


GRIDS = [
    (CART, "[0:200]*50", "[0:200]*50", "[3.556:3.735]*1"),
    (CART, "[0:200]*50", "[0:200]*50", "[3.556:3.735]*3"),
    (CART, "[0:100]*7", "[0:200]*400", "[3.556:3.735]*1"),
    (CART, "[10:150]*11", "[35:90]*13", "[3.556:3.735]*2"),
    (CART, "[-5:60]*13", "[-30:160]*19", "[3.556:3.735]*1"),
    (CART, "[0:3]*2", "[0:1]*5", "[3.556:3.735]*1"),
    (CART, "[0:200]*100", "[0:200]*100", "[3.556:3.735]*1"),
    (CART, "[0:200]*20", "[0:200]*20", "[0.6:3.0]*3"),
    (CART, "[0:200]*20", "[0:200]*20", "[4.6:5.0]*2"),
    (OBS, "[0:0.02]*20", "[0:0.06]*6", "[3.556:3.735]*1"),
    (OBS, "[0:0.05]*50", "[0.01:0.04]*30", "[3.556:3.735]*2"),
    (OBS, "[0.001:0.02]*200", "[0:0.06]*60", "[0.6:3.0]*3"),
]


@pytest.mark.parametrize("spec", GRIDS, ids=[f"{s[0]}-{s[1]}-{s[2]}-{s[3][-1]}" for s in GRIDS])
def test_tile_pass_equals_the_general_kernel(dev, field, spec):
    grid = GridSpec.from_specs(*spec)
    wide = GridSpec.cartesian() if spec[0] == CART else GridSpec.observing()
    dcat = dev.upload(field)
    pairs = dcat.pairs(wide.max_angular_scale(field.scale), order=3, nthreads=8)
    assert pairs.stats()["num_sightline_pairs_used"] > 20000
    for prec in (tos_amd.FP64, tos_amd.FP32C):
        print(f"case: grid {grid.specs} type {grid.type} precision {prec}", flush=True)
        ref = pairs.run(grid, precision=prec, flags=tos_amd.XI_NO_ZCONST)
        h = pairs.run(grid, precision=prec)
        close(h, ref.num_pairs, {"didj": ref.didj, "wgt": ref.wgt})
        assert h.num_pixel_pairs_used == ref.num_pixel_pairs_used
    pairs.free()
    dcat.free()


@pytest.mark.parametrize("spec", [GRIDS[0], GRIDS[3], GRIDS[10]], ids=["cartesian", "offset", "observing"])
def test_tile_pass_against_the_oracle(dev, field, spec):
    from oracle import oracle as ora
    grid = GridSpec.from_specs(*spec)
    wide = GridSpec.cartesian() if spec[0] == CART else GridSpec.observing()
    ref = ora.xi_run(field, wide if spec[0] == CART and spec != GRIDS[3] else grid, field.scale, order=3, nthreads=8)
    dcat = dev.upload(field)
    pairs = dcat.pairs((wide if spec[0] == CART and spec != GRIDS[3] else grid).max_angular_scale(field.scale),
                       order=3, nthreads=8)
    for prec in (tos_amd.FP64, tos_amd.FP32C):
        print(f"case: grid {grid.specs} precision {prec}", flush=True)
        close(pairs.run(grid, precision=prec), ref["raw"]["num_pairs"], ref["raw"])
    pairs.free()
    dcat.free()


@pytest.mark.parametrize("change", ["off_ladder", "two_wavelengths", "descending"])
def test_catalogues_without_a_ladder(dev, field, change):
    """Pixels off any common ladder take the general kernel, same results."""
    cat = synth.Catalog(field.ra, field.dec, field.offsets, field.value, field.loglam.copy(), field.weight,
                        field.distance.copy(), field.zq, field.scale)
    n = cat.n_pix
    if change == "off_ladder":      # every sightline its own distances
        cat.distance += np.repeat(np.arange(cat.n_los), cat.counts()).astype(np.float32) * np.float32(1e-2)
    elif change == "two_wavelengths":
        cat.loglam[n // 2] += np.float32(1e-5)
    else:
        a, b = cat.offsets[40], cat.offsets[41]
        cat.distance[a:b] = cat.distance[a:b][::-1]
        cat.loglam[a:b] = cat.loglam[a:b][::-1]
    grid = GridSpec.cartesian(rpar="[0:200]*20", rperp="[0:200]*20")
    dcat = dev.upload(cat)
    pairs = dcat.pairs(grid.max_angular_scale(cat.scale), order=3, nthreads=8)
    print(f"case: {change}", flush=True)
    ref = pairs.run(grid, precision=tos_amd.FP64, flags=tos_amd.XI_NO_ZCONST | tos_amd.XI_NO_WINDOW)
    h = pairs.run(grid, precision=tos_amd.FP32C)
    close(h, ref.num_pairs, {"didj": ref.didj, "wgt": ref.wgt})
    pairs.free()
    dcat.free()


def test_a_weighted_value_that_overflows(dev, field):
    """A w d beyond the float range reaches the bins of its own pairs only."""
    cat = synth.Catalog(field.ra, field.dec, field.offsets, field.value.copy(), field.loglam, field.weight.copy(),
                        field.distance, field.zq, field.scale)
    for k, v in ((cat.n_pix // 3, 1e30), (cat.n_pix // 2, -1e30)):
        cat.weight[k], cat.value[k] = 1e30, v
    grid = GridSpec.cartesian()
    dcat = dev.upload(cat)
    pairs = dcat.pairs(grid.max_angular_scale(cat.scale), order=3, nthreads=8)
    ref = pairs.run(grid, precision=tos_amd.FP64, flags=tos_amd.XI_NO_ZCONST)
    h = pairs.run(grid, precision=tos_amd.FP64)
    assert np.array_equal(h.num_pairs, ref.num_pairs)
    assert 0 < np.sum(~np.isfinite(ref.didj)) < ref.didj.size
    assert np.array_equal(np.isnan(h.didj), np.isnan(ref.didj))
    assert np.array_equal(np.isinf(h.didj), np.isinf(ref.didj))
    assert rel_err(h.wgt, ref.wgt) <= SUM_RTOL
    pairs.free()
    dcat.free()


@pytest.mark.parametrize("spec", [GRIDS[k] for k in (0, 1, 3, 4, 8, 9, 11)],
                         ids=[f"{GRIDS[k][0]}-{GRIDS[k][1]}-{GRIDS[k][3]}" for k in (0, 1, 3, 4, 8, 9, 11)])
def test_seven_sums_equal_the_general_kernel(dev, field, spec):
    grid = GridSpec.from_specs(*spec)
    wide = GridSpec.cartesian() if spec[0] == CART else GridSpec.observing()
    dcat = dev.upload(field)
    pairs = dcat.pairs(wide.max_angular_scale(field.scale), order=3, nthreads=8)
    print(f"case: grid {grid.specs} type {grid.type}", flush=True)
    ref = pairs.run(grid, precision=tos_amd.FP64, accum=tos_amd.ACC_ALL, flags=tos_amd.XI_NO_ZCONST)
    h = pairs.run(grid, precision=tos_amd.FP64, accum=tos_amd.ACC_ALL)
    close(h, ref.num_pairs, {"didj": ref.didj, "wgt": ref.wgt})
    for k in ("wi", "wj", "z"):
        assert rel_err(h.extra[k], ref.extra[k]) <= SUM_RTOL, k
    # signed: against the weights of the same pixels
    assert signed_sum_err(h.extra["di"], ref.extra["di"], ref.extra["wi"]) <= SUM_RTOL
    assert signed_sum_err(h.extra["dj"], ref.extra["dj"], ref.extra["wj"]) <= SUM_RTOL
    pairs.free()
    dcat.free()


# mu axes that end inside [0, 1], start above 0 or below it, finer than the
# r axis; r axes that start above 0 or below it, narrower than a tile's
# spread, in several LDS bands; z axes with several bins or left
POLAR_GRIDS = [
    ("[0:200]*50", "[0:1]*20", "[3.556:3.735]*1"),
    ("[0:200]*50", "[0:1]*20", "[3.556:3.735]*3"),
    ("[20:150]*13", "[0.1:0.9]*7", "[3.556:3.735]*2"),
    ("[-5:90]*19", "[-0.3:0.5]*8", "[3.556:3.735]*1"),
    ("[0:200]*3", "[0:1]*500", "[3.556:3.735]*1"),
    ("[0:200]*400", "[0:1]*3", "[3.556:3.735]*1"),
    ("[0:200]*100", "[0:1]*100", "[3.556:3.735]*1"),
    ("[0:1.5]*3", "[0:1]*4", "[3.556:3.735]*1"),
    ("[0:200]*20", "[0:1]*1", "[0.6:3.0]*3"),
    ("[0:200]*20", "[0.5:0.9]*1", "[4.6:5.0]*2"),
    ("[0:200]*64", "[0:1.5]*16", "[3.556:3.735]*1"),
]


@pytest.mark.parametrize("spec", POLAR_GRIDS, ids=["-".join(s) for s in POLAR_GRIDS])
def test_polar_tile_pass_equals_the_general_kernel(dev, field, spec):
    grid = GridSpec.from_specs(tos_amd.POLAR, *spec)
    dcat = dev.upload(field)
    pairs = dcat.pairs(GridSpec.polar().max_angular_scale(field.scale), order=3, nthreads=8)
    assert pairs.stats()["num_sightline_pairs_used"] > 20000
    for prec in (tos_amd.FP64, tos_amd.FP32C):
        print(f"case: polar grid {grid.specs} precision {prec}", flush=True)
        ref = pairs.run(grid, precision=prec, flags=tos_amd.XI_NO_ZCONST)
        h = pairs.run(grid, precision=prec)
        close(h, ref.num_pairs, {"didj": ref.didj, "wgt": ref.wgt})
        assert h.num_pixel_pairs_used == ref.num_pixel_pairs_used
    ref = pairs.run(grid, precision=tos_amd.FP64, accum=tos_amd.ACC_ALL, flags=tos_amd.XI_NO_ZCONST)
    h = pairs.run(grid, precision=tos_amd.FP64, accum=tos_amd.ACC_ALL)
    close(h, ref.num_pairs, {"didj": ref.didj, "wgt": ref.wgt})
    for k in ("wi", "wj", "z"):
        assert rel_err(h.extra[k], ref.extra[k]) <= SUM_RTOL, k
    pairs.free()
    dcat.free()


def test_polar_tile_pass_against_the_oracle(dev, field):
    from oracle import oracle as ora
    grid = GridSpec.from_specs(tos_amd.POLAR, *POLAR_GRIDS[1])
    ref = ora.xi_run(field, grid, field.scale, order=3, nthreads=8)
    dcat = dev.upload(field)
    pairs = dcat.pairs(grid.max_angular_scale(field.scale), order=3, nthreads=8)
    for prec in (tos_amd.FP64, tos_amd.FP32C):
        print(f"case: polar grid {grid.specs} precision {prec}", flush=True)
        close(pairs.run(grid, precision=prec), ref["raw"]["num_pairs"], ref["raw"])
    jobs = [(pairs, grid, tos_amd.FP64), (pairs, GridSpec.polar(), tos_amd.FP32C)]
    h = dev.batch_run(jobs)[0]
    close(h[0], ref["raw"]["num_pairs"], ref["raw"])
    one = pairs.run(GridSpec.polar(), precision=tos_amd.FP64, flags=tos_amd.XI_NO_ZCONST)
    close(h[1], one.num_pairs, {"didj": one.didj, "wgt": one.wgt})
    pairs.free()
    dcat.free()
