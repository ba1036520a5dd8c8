// tos_tile.cpp -- host side of the tile path (tos_tileplan.hip,
// tos_tilepass.hip): when a job takes it, the catalogue's ladder and the pair
// list's plan, both built once on first use.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "tos_capi_impl.h"

namespace tos {

namespace {

struct Scratch {   // released on every return
    DevBuf b[7];
    ~Scratch()
    {
        for (DevBuf &x : b) x.release();
    }
};

int copy_back(tos_ctx *ctx, void *dst, const void *src, size_t n, const char *what)
{
    hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    return e == hipSuccess ? TOS_OK : hip_fail(ctx, e, what);
}

}  // namespace

void Ladder::release()
{
    for (DevBuf *x : {&pix, &d, &l, &place}) x->release();
}

void TilePlan::release()
{
    for (DevBuf *x : {&masks, &rec, &batch_ptr, &visits}) x->release();
    state = 0;
}

// The catalogue on its ladder, or state 2 when it has none (or no memory).
int ensure_ladder(tos_ctx *ctx, tos_catalog *cat)
{
    Ladder &L = cat->ladder;
    if (L.state) return TOS_OK;
    L.state = 2;
    if (cat->n_los == 0 || cat->n_pix == 0 || !(cat->dmin > 1e-3) || !cat->d_sorted || !cat->l_sorted) return TOS_OK;
    // the table and the state in the context's scratch: a catalogue without a
    // ladder costs no allocation
    constexpr size_t kTableBytes = (size_t)kLadderTable * 8;
    uint32_t st[3] = {0, 0, 0};
    if (ctx->scratch_a.reserve(kTableBytes + sizeof(st)) != TOS_OK) return TOS_OK;
    int rc;
    LadderArgs a{};
    a.pix = (const float4 *)cat->pix.ptr;
    a.los = (const LosInfo *)cat->los.ptr;
    a.n_los = cat->n_los;
    a.n_pix = cat->n_pix;
    a.table = (uint64_t *)ctx->scratch_a.ptr;
    a.state = (uint32_t *)((char *)ctx->scratch_a.ptr + kTableBytes);
    int e = launch_ladder_collect(a, ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, (hipError_t)e, "ladder collection");
    if ((rc = copy_back(ctx, st, a.state, sizeof(st), "ladder state copy")) != TOS_OK) return rc;
    if (st[0]) return TOS_OK;
    std::vector<uint64_t> tab(kLadderTable);
    if ((rc = copy_back(ctx, tab.data(), a.table, kTableBytes, "ladder table copy")) != TOS_OK) return rc;
    Scratch sc;
    DevBuf &step = sc.b[0], &nblk_of = sc.b[1];
    if (step.reserve(kLadderTable * 2) != TOS_OK || nblk_of.reserve((size_t)cat->n_los * 4) != TOS_OK ||
        L.place.reserve((size_t)cat->n_los * sizeof(LadderLos)) != TOS_OK) {
        L.release();
        return TOS_OK;
    }
    a.step = (const uint16_t *)step.ptr;
    a.place = (LadderLos *)L.place.ptr;
    a.nblk_of = (uint32_t *)nblk_of.ptr;
    // the steps in ascending distance; wavelengths must ascend with them
    struct Step {
        float d, l;
        int slot;
    };
    std::vector<Step> steps;
    for (int k = 0; k < kLadderTable; ++k) {
        if (tab[(size_t)k] == ~0ull) continue;
        const uint32_t db = (uint32_t)tab[(size_t)k], lb = (uint32_t)(tab[(size_t)k] >> 32);
        Step s;
        std::memcpy(&s.d, &db, 4);
        std::memcpy(&s.l, &lb, 4);
        s.slot = k;
        steps.push_back(s);
    }
    std::sort(steps.begin(), steps.end(), [](const Step &x, const Step &y) { return x.d < y.d; });
    bool ok = !steps.empty() && steps.size() <= (size_t)kMaxLadder;
    for (size_t k = 1; ok && k < steps.size(); ++k) ok = steps[k].d > steps[k - 1].d && steps[k].l > steps[k - 1].l;
    if (!ok) {
        L.release();
        return TOS_OK;
    }
    L.nblk = (int)((steps.size() + kBlockSteps - 1) / kBlockSteps);
    std::vector<uint16_t> step_of(kLadderTable, 0);
    L.h_d.assign((size_t)L.nblk * kBlockSteps, steps.back().d);
    L.h_l.assign((size_t)L.nblk * kBlockSteps, steps.back().l);
    for (size_t k = 0; k < steps.size(); ++k) {
        step_of[(size_t)steps[k].slot] = (uint16_t)k;
        L.h_d[k] = steps[k].d;
        L.h_l[k] = steps[k].l;
    }
    if ((rc = upload(ctx, step, step_of.data(), step_of.size() * 2, "ladder steps")) != TOS_OK ||
        (rc = upload(ctx, L.d, L.h_d.data(), L.h_d.size() * 4, "ladder distances")) != TOS_OK ||
        (rc = upload(ctx, L.l, L.h_l.data(), L.h_l.size() * 4, "ladder wavelengths")) != TOS_OK)
        return rc;
    e = launch_ladder_place(a, ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, (hipError_t)e, "ladder placement");
    if ((rc = copy_back(ctx, st, a.state, sizeof(st), "ladder block count")) != TOS_OK) return rc;
    if (st[0] || st[2] >= (1u << 24) ||   // 32-bit byte offsets
        L.pix.reserve((size_t)st[2] * kBlockBytes) != TOS_OK) {
        L.release();
        return TOS_OK;
    }
    a.out = (float *)L.pix.ptr;
    e = launch_ladder_fill(a, st[2], ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, (hipError_t)e, "ladder fill");
    if ((rc = copy_back(ctx, st, a.state, sizeof(st), "ladder state copy")) != TOS_OK) return rc;
    if (st[0]) {
        L.release();
        return TOS_OK;
    }
    L.state = 1;
    return TOS_OK;
}

// Pairs per batch.  A group's batches split its range of separations, so a
// short batch costs no more bin edges, only tiles: each is drawn from one
// counter (some 10 ns a draw) and starts its cells anew.  Long ones make large
// last tiles.  Measured, ms per pass at n / 64 pairs a batch (8192 at most) /
// n / 128 / n / 256 / n / 512: 141,344 pairs in four bands 3.7 / 4.0 / 7.0 /
// 13.4; 1.47 million pairs 5.3 / 5.4 / 5.2 / 5.3 (16384 a batch: 5.9); twelve
// jobs of 2,000 to 12,000 sightlines - / 27.4 / 30.6 / 37.3; 3,450 pairs at
// 512 / 1024 a batch 0.256 / 0.286; 37 million at 8192 / 16384 122 / 120.
static int64_t batch_pairs(int64_t n_pairs)
{
    const int64_t q = std::max<int64_t>(std::min<int64_t>(n_pairs / 64, 8192), n_pairs / 1024);
    return std::max<int64_t>(512, std::min<int64_t>(kMaxBatch, q));
}

// [0, n) in the fewest equal parts of at most `most`, appended from `first`.
static void cut_equal(std::vector<int32_t> &ptr, int64_t first, int64_t n, int64_t most)
{
    const int64_t parts = (n + most - 1) / most;
    for (int64_t k = 0; k < parts; ++k) ptr.push_back((int32_t)(first + n * k / parts));
}

int ensure_tile_plan(tos_ctx *ctx, tos_pairs *p)
{
    TilePlan &T = p->tiles;
    if (T.state) return TOS_OK;
    T.state = 2;
    tos_catalog *cat = const_cast<tos_catalog *>(p->cat);
    int rc = ensure_ladder(ctx, cat);
    if (rc != TOS_OK) return rc;
    const Ladder &L = cat->ladder;
    if (L.state != 1 || p->n_pairs == 0) return TOS_OK;
    std::vector<int32_t> gp, bp;
    cut_equal(gp, 0, p->n_pairs, kMaxGroup);
    gp.push_back((int32_t)p->n_pairs);
    int32_t max_group = 0;
    for (size_t k = 0; k + 1 < gp.size(); ++k) {
        max_group = std::max(max_group, gp[k + 1] - gp[k]);
        cut_equal(bp, gp[k], gp[k + 1] - gp[k], batch_pairs(p->n_pairs));
    }
    bp.push_back((int32_t)p->n_pairs);
    int32_t q = 0;
    for (size_t k = 0; k + 1 < bp.size(); ++k) q = std::max(q, bp[k + 1] - bp[k]);
    T.n_batches = (int)bp.size() - 1;
    if ((int64_t)T.n_batches * L.nblk * (2 * L.nblk + 1) >= (1ll << 31)) return TOS_OK;
    Scratch sc;
    DevBuf &rlos = sc.b[0], &rptr = sc.b[1], &state = sc.b[2], &cover = sc.b[3], &keys = sc.b[4], &groups = sc.b[5], &keys2 = sc.b[6];
    T.words = (int)((q + 63) / 64);
    const size_t np = (size_t)p->n_pairs, rows = (size_t)T.n_batches * L.nblk;
    if (cover.reserve(np * 4) != TOS_OK || T.masks.reserve(rows * 2 * T.words * 8) != TOS_OK || T.rec.reserve(np * 16) != TOS_OK ||
        T.visits.reserve(rows * L.nblk * 4) != TOS_OK ||
        state.reserve(16) != TOS_OK || (max_group > kSortRun && (keys.reserve(np * 8) != TOS_OK || keys2.reserve(np * 8) != TOS_OK))) {
        T.release();
        T.state = 2;
        return TOS_OK;
    }
    uint64_t st[2] = {0, 0};
    if ((rc = upload(ctx, T.batch_ptr, bp.data(), bp.size() * 4, "tile batches")) != TOS_OK ||
        (rc = upload(ctx, groups, gp.data(), gp.size() * 4, "tile groups")) != TOS_OK ||
        (rc = upload(ctx, rlos, p->h.row_los.data(), p->h.row_los.size() * 4, "tile rows")) != TOS_OK ||
        (rc = upload(ctx, rptr, p->h.row_ptr.data(), p->h.row_ptr.size() * 8, "tile row offsets")) != TOS_OK ||
        (rc = upload(ctx, state, st, sizeof(st), "tile state")) != TOS_OK)
        return rc;
    TilePlanArgs a{};
    a.row_los = (const int32_t *)rlos.ptr;
    a.row_ptr = (const int64_t *)rptr.ptr;
    a.other = (const int32_t *)p->other.ptr;
    a.csep = (const double *)p->csep.ptr;
    a.place = (const LadderLos *)L.place.ptr;
    a.n_rows = p->n_rows;
    a.n_batches = T.n_batches;
    a.max_batch = q;
    a.n_groups = (int32_t)gp.size() - 1;
    a.max_group = max_group;
    a.group_ptr = (const int32_t *)groups.ptr;
    a.nblk = L.nblk;
    a.batch_ptr = (const int32_t *)T.batch_ptr.ptr;
    a.words = T.words;
    a.keys = (uint64_t *)keys.ptr;
    a.keys2 = (uint64_t *)keys2.ptr;
    a.cover = (uint32_t *)cover.ptr;
    a.masks = (uint64_t *)T.masks.ptr;
    a.rec = (uint4 *)T.rec.ptr;
    a.visits = (uint32_t *)T.visits.ptr;
    a.state = (unsigned long long *)state.ptr;
    const int e = launch_tile_plan(a, ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, (hipError_t)e, "tile plan");
    if ((rc = copy_back(ctx, st, state.ptr, sizeof(st), "tile state copy")) != TOS_OK) return rc;
    if (st[0]) {
        T.release();
        T.state = 2;
        return TOS_OK;
    }
    T.total = st[1];
    T.state = 1;
    return TOS_OK;
}

// Fewer candidate pairs than this take the general path.  Measured, general
// / tile, us per pass on a 200 x 200 Mpc/h grid of 50 x 50 bins: 426 pairs
// 535 / 260; 1,259 pairs 547 / 257; 9,061 pairs 770 / 383; 6.2 million pairs
// 53,500 / 25,400.  Below, a launch is a few tiles and the plan of a first
// pass costs what it saves.
constexpr int64_t kTileMinPairs = 400;

bool tile_job(const tos_catalog *cat, const tos_pairs *p, const tos_grid &g)
{
    if (p->n_pairs < kTileMinPairs) return false;
    if (cat->ladder.state == 2 || p->tiles.state == 2) return false;
    // the edge bound needs squared separations well above their rounding
    if (!(cat->dmin > 1e-3) || cat->dmax > 1e5) return false;
    // bins far past an axis stay there: the reference's cast wraps only
    // beyond 2^31 of them
    auto wraps = [&](double top, int k) { return (top + std::fabs(g.min[k])) / g.width[k] > 1e9; };
    if (g.type == TOS_CARTESIAN) return !wraps(2.0 * cat->dmax, 1);
    // Polar: |d1 - d2| exact, a table of the edges in LDS
    if (g.type == TOS_POLAR)
        return cat->dmax <= 2.0 * cat->dmin && tile_edges(g) <= kTileMaxEdges && !wraps(2.0 * cat->dmax, 0) &&
               !wraps(1.0, 1);
    return true;
}

bool tile_args(const tos_pairs *p, const tos_grid &g, TileArgs &t)
{
    const tos_catalog *cat = p->cat;
    const Ladder &L = cat->ladder;
    const TilePlan &T = p->tiles;
    t = TileArgs{};
    t.pix = (const float *)L.pix.ptr;
    t.d = (const float *)L.d.ptr;
    t.l = (const float *)L.l.ptr;
    t.masks = (const uint64_t *)T.masks.ptr;
    t.words = T.words;
    t.rec = (const uint4 *)T.rec.ptr;
    t.batch_ptr = (const int32_t *)T.batch_ptr.ptr;
    t.visits = (const uint32_t *)T.visits.ptr;
    t.nblk = L.nblk;
    t.n_batches = T.n_batches;
    t.width0 = g.width[0];
    t.width1 = g.width[1];
    // tiles whose steps all differ by less than the axis-0 window
    const std::vector<float> &key = g.type == TOS_OBSERVING ? L.h_l : L.h_d;
    const double X = grid_window_half(g, cat->dmax, g.type == TOS_OBSERVING ? cat->lmax_abs : cat->dmax);
    int band = L.nblk - 1;
    if (X > 0) {
        band = 0;
        for (int b1 = 0; b1 < L.nblk; ++b1)
            for (int b2 = b1 + band + 1; b2 < L.nblk; ++b2) {
                if (!((double)key[(size_t)b2 * kBlockSteps] - (double)key[(size_t)b1 * kBlockSteps + kBlockSteps - 1] < X)) break;
                band = b2 - b1;
            }
    }
    t.band = band;
    // K of an edge at squared separation s >= s_min is known within a relative
    //   2^-24 (f32 K) + 3 2^-24 (f32 threshold: the squared edge, 1 / (d1 d2)
    //   and their product)
    //   + (7e-15 dmax^2 (the reference's FP64 rounding of r^2) + 2^-24 base) / s_min,
    // base <= ulp32(dmax^2) + 2 * 2^-24 dmax * axis-0 range; doubled
    // (Polar: base <= ulp32(dmax^2), six more roundings in the threshold, and
    // r^2 = r_par^2 / mu^2 as the reference's rounded mu, of at least (smallest
    // step) / R, has it).
    // s_min is 4 (Mpc/h)^2 for the distances of a survey and goes down with
    // dmax^2, like the errors: in Gpc/h every pair would lie below 4, and each
    // takes the reference arithmetic there (400,000 sightline pairs 29 ms, the
    // general kernel 23, this 1.9).
    const double u = std::ldexp(1.0, -24);
    const double scale = std::min(1.0, cat->dmax / 5000.0);
    t.s_min = 4.0 * scale * scale;
    double base = 2.0 * u * cat->dmax * cat->dmax + 4.0 * u * cat->dmax * std::fabs(g.max[0]);
    double ops = 4.0, abs_err = 7e-15 * cat->dmax * cat->dmax;
    if (g.type == TOS_POLAR) {
        base = 2.0 * u * cat->dmax * cat->dmax;
        ops = 10.0;
        double step = INFINITY;
        for (size_t k = 1; k < L.h_d.size(); ++k)
            if (L.h_d[k] > L.h_d[k - 1]) step = std::min(step, (double)L.h_d[k] - (double)L.h_d[k - 1]);
        const double R = std::fabs(g.min[0]) + g.nbins[0] * g.width[0];
        const double M = 1.0 + std::fabs(g.min[1]) + g.nbins[1] * g.width[1];
        abs_err += 1e-15 * R * R * (4.0 + M * R / step);
    }
    t.eps = 2.0 * (ops * u + (abs_err + u * base) / t.s_min);
    t.ulps = (uint32_t)std::ceil(2.2 * t.eps / u) + 2;
    return t.eps < 1e-4;
}

int tile_workgroups(const tos_pairs *p, const TileArgs &a, int want, int block)
{
    const int64_t tiles = (int64_t)a.n_batches * a.nblk * (2 * a.band + 1);
    const int64_t waves = block / 64;
    const int64_t n = std::min<int64_t>(want, (tiles + 2 * waves - 1) / (2 * waves));
    // enough that not all of them can run out of counts (kTileVisits)
    return (int)std::max<int64_t>(n, (int64_t)(p->tiles.total / kTileVisits) + 1);
}

}  // namespace tos
