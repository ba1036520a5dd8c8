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

// Places in one allocation (an allocation takes some 10 to 100 us, a plan and
// a ladder were 17 of them).
struct Carve {
    size_t bytes = 0;
    size_t add(size_t n)
    {
        const size_t at = (bytes + 255) & ~(size_t)255;
        bytes = at + n;
        return at;
    }
};
// A plan's temporaries up to this size lie in the context's scratch, which
// stays; larger ones are allocated for it.
constexpr size_t kKeepScratch = (size_t)32 << 20;

int copy_back(tos_ctx *ctx, void *dst, const void *src, size_t n, const char *what)
{
    hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    return e == hipSuccess ? TOS_OK : hip_fail(ctx, e, what);
}

}  // namespace

void Ladder::release()
{
    pix.release();
    mem.release();
}

void TilePlan::release()
{
    mem.release();
    state = 0;
}

constexpr size_t kTableBytes = (size_t)kLadderTable * 8;
constexpr size_t kStateWords = 2, kStepWords = kLadderTable / 4;   // behind the table

static LadderArgs ladder_args(const tos_catalog *cat)
{
    LadderArgs a{};
    a.pix = (const float4 *)cat->pix.ptr;
    a.los = (const LosInfo *)cat->los.ptr;
    a.n_los = cat->n_los;
    a.n_pix = cat->n_pix;
    return a;
}

// Looks for the catalogue's ladder: state 3 (its steps are known) or 2 (none,
// or no memory).
static int survey_ladder(tos_ctx *ctx, tos_catalog *cat)
{
    Ladder &L = cat->ladder;
    if (L.state) return TOS_OK;
    L.state = 2;
    if (cat->n_los == 0 || cat->n_pix == 0 || !(cat->dmin > 1e-3) || !cat->d_sorted || !cat->l_sorted) return TOS_OK;
    // the table and the state in the context's scratch: a catalogue without a
    // ladder costs no allocation
    uint32_t st[3] = {0, 0, 0};
    if (ctx->scratch_a.reserve(kTableBytes + 8 * (kStateWords + kStepWords)) != TOS_OK) return TOS_OK;
    int rc;
    LadderArgs a = ladder_args(cat);
    a.table = (uint64_t *)ctx->scratch_a.ptr;
    a.state = (uint32_t *)((char *)ctx->scratch_a.ptr + kTableBytes);
    int e = launch_ladder_collect(a, ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, (hipError_t)e, "ladder collection");
    if ((rc = copy_back(ctx, st, a.state, sizeof(st), "ladder state copy")) != TOS_OK) return rc;
    if (st[0]) return TOS_OK;
    std::vector<uint64_t> tab(kLadderTable);
    if ((rc = copy_back(ctx, tab.data(), a.table, kTableBytes, "ladder table copy")) != TOS_OK) return rc;
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
    // (K of an edge is formed with 1 / (d1 d2), which must not change sign)
    bool ok = !steps.empty() && steps.size() <= (size_t)kMaxLadder && steps[0].d > 0.0f;
    for (size_t k = 1; ok && k < steps.size(); ++k) ok = steps[k].d > steps[k - 1].d && steps[k].l > steps[k - 1].l;
    if (!ok) return TOS_OK;
    L.n_steps = (int)steps.size();
    L.nblk = (int)((steps.size() + kBlockSteps - 1) / kBlockSteps);
    tab.resize(kLadderTable + kStateWords + kStepWords, 0);
    uint16_t *step_of = (uint16_t *)(tab.data() + kLadderTable + kStateWords);
    L.h_d.assign((size_t)L.nblk * kBlockSteps, steps.back().d);
    L.h_l.assign((size_t)L.nblk * kBlockSteps, steps.back().l);
    for (size_t k = 0; k < steps.size(); ++k) {
        step_of[steps[k].slot] = (uint16_t)k;
        L.h_d[k] = steps[k].d;
        L.h_l[k] = steps[k].l;
    }
    L.table.swap(tab);
    // mean blocks of a sightline, from some of them
    const int64_t every = std::max<int64_t>(1, cat->n_los / 512);
    int64_t n = 0, blocks = 0;
    for (int64_t k = 0; k < cat->n_los; k += every) {
        const LosInfo &li = cat->h_los[(size_t)k];
        if (li.n == 0) continue;
        auto at = [&](float l) { return (std::lower_bound(L.h_l.begin(), L.h_l.begin() + L.n_steps, l) - L.h_l.begin()) / kBlockSteps; };
        blocks += at(li.lmax) - at(li.lmin) + 1;
        ++n;
    }
    L.mean_nb = n > 0 ? (double)blocks / (double)n : 0.0;
    L.state = 3;
    return TOS_OK;
}

// What a step of building a ladder or a plan left undone: its memory is given
// back, and a lack of memory is no error, the job takes the general path.
template <typename T>
static int give_up(T &built, int rc)
{
    built.release();
    built.state = 2;
    return rc == TOS_ERR_NOMEM ? TOS_OK : rc;
}

// A surveyed catalogue's pixels laid out on the ladder (state 1; 2: none, or
// no memory).
static int build_ladder(tos_ctx *ctx, tos_catalog *cat)
{
    Ladder &L = cat->ladder;
    if (L.state != 3) return TOS_OK;
    uint32_t st[3] = {0, 0, 0};
    int rc;
    Carve c;
    const size_t key_bytes = L.h_d.size() * 4, at_keys = c.add(2 * key_bytes), at_place = c.add((size_t)cat->n_los * sizeof(LadderLos));
    if (ctx->scratch_b.reserve((size_t)cat->n_los * 4) != TOS_OK || L.mem.reserve(c.bytes) != TOS_OK)
        return give_up(L, TOS_ERR_NOMEM);
    L.d = (float *)((char *)L.mem.ptr + at_keys);
    L.l = L.d + L.h_d.size();
    L.place = (LadderLos *)((char *)L.mem.ptr + at_place);
    std::vector<float> keys(L.h_d);
    keys.insert(keys.end(), L.h_l.begin(), L.h_l.end());
    if ((rc = upload(ctx, ctx->scratch_a, L.table.data(), L.table.size() * 8, "ladder table")) != TOS_OK ||
        (rc = upload(ctx, L.mem, keys.data(), keys.size() * 4, "ladder steps")) != TOS_OK)
        return give_up(L, rc);
    LadderArgs a = ladder_args(cat);
    a.table = (uint64_t *)ctx->scratch_a.ptr;
    a.state = (uint32_t *)((char *)ctx->scratch_a.ptr + kTableBytes);
    a.step = (const uint16_t *)((char *)ctx->scratch_a.ptr + kTableBytes + 8 * kStateWords);
    a.place = L.place;
    a.nblk_of = (uint32_t *)ctx->scratch_b.ptr;
    int e = launch_ladder_place(a, ctx->stream);
    if (e != hipSuccess) return give_up(L, hip_fail(ctx, (hipError_t)e, "ladder placement"));
    if ((rc = copy_back(ctx, st, a.state, sizeof(st), "ladder block count")) != TOS_OK) return give_up(L, rc);
    if (st[0] || st[2] >= (1u << 24) ||   // 32-bit byte offsets
        L.pix.reserve((size_t)st[2] * kBlockBytes) != TOS_OK)
        return give_up(L, TOS_ERR_NOMEM);
    a.out = (float *)L.pix.ptr;
    e = launch_ladder_fill(a, st[2], ctx->stream);
    if (e != hipSuccess) return give_up(L, hip_fail(ctx, (hipError_t)e, "ladder fill"));
    if ((rc = copy_back(ctx, st, a.state, sizeof(st), "ladder state copy")) != TOS_OK) return give_up(L, rc);
    if (st[0]) return give_up(L, TOS_OK);
    L.state = 1;
    L.table = std::vector<uint64_t>();
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

// The list's tile plan: T.state 1, or 2 (none, or no memory).
static int ensure_tile_plan(tos_ctx *ctx, tos_pairs *p)
{
    TilePlan &T = p->tiles;
    if (T.state) return TOS_OK;
    T.state = 2;
    tos_catalog *cat = const_cast<tos_catalog *>(p->cat);
    int rc = build_ladder(ctx, cat);
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
    T.words = (int)((q + 63) / 64);
    const size_t np = (size_t)p->n_pairs, rows = (size_t)T.n_batches * L.nblk;
    Carve c, tmp;
    const size_t at_masks = c.add(rows * 2 * T.words * 8), at_rec = c.add(np * 16), at_visits = c.add(rows * L.nblk * 4),
                 at_batches = c.add(bp.size() * 4);
    const HostPairs &h = p->h;
    const size_t at_state = tmp.add(16), at_groups = tmp.add(gp.size() * 4), at_rlos = tmp.add(h.row_los.size() * 4),
                 at_rptr = tmp.add(h.row_ptr.size() * 8), head = tmp.bytes, at_cover = tmp.add(np * 4),
                 sorted = max_group > kSortRun ? np * 8 : 0, at_keys = tmp.add(sorted), at_keys2 = tmp.add(sorted);
    struct Local {
        DevBuf b;
        ~Local() { b.release(); }
    } local;
    DevBuf &work = tmp.bytes <= kKeepScratch ? ctx->scratch_c : local.b;
    if (T.mem.reserve(c.bytes) != TOS_OK || work.reserve(tmp.bytes) != TOS_OK) return give_up(T, TOS_ERR_NOMEM);
    char *const mem = (char *)T.mem.ptr, *const w = (char *)work.ptr;
    T.masks = (uint64_t *)(mem + at_masks);
    T.rec = (uint4 *)(mem + at_rec);
    T.visits = (uint32_t *)(mem + at_visits);
    T.batch_ptr = (int32_t *)(mem + at_batches);
    std::vector<char> up(head, 0);
    std::memcpy(up.data() + at_groups, gp.data(), gp.size() * 4);
    std::memcpy(up.data() + at_rlos, h.row_los.data(), h.row_los.size() * 4);
    std::memcpy(up.data() + at_rptr, h.row_ptr.data(), h.row_ptr.size() * 8);
    hipError_t he = hipMemcpyAsync(w, up.data(), head, hipMemcpyHostToDevice, ctx->stream);
    if (he == hipSuccess)
        he = hipMemcpyAsync(T.batch_ptr, bp.data(), bp.size() * 4, hipMemcpyHostToDevice, ctx->stream);
    if (he != hipSuccess) return give_up(T, hip_fail(ctx, he, "tile plan tables"));
    uint64_t st[2] = {0, 0};
    TilePlanArgs a{};
    a.row_los = (const int32_t *)(w + at_rlos);
    a.row_ptr = (const int64_t *)(w + at_rptr);
    a.other = (const int32_t *)p->other.ptr;
    a.csep = (const double *)p->csep.ptr;
    a.place = L.place;
    a.n_rows = p->n_rows;
    a.n_batches = T.n_batches;
    a.max_batch = q;
    a.n_groups = (int32_t)gp.size() - 1;
    a.max_group = max_group;
    a.group_ptr = (const int32_t *)(w + at_groups);
    a.nblk = L.nblk;
    a.batch_ptr = T.batch_ptr;
    a.words = T.words;
    a.keys = (uint64_t *)(w + at_keys);
    a.keys2 = (uint64_t *)(w + at_keys2);
    a.cover = (uint32_t *)(w + at_cover);
    a.masks = T.masks;
    a.rec = T.rec;
    a.visits = T.visits;
    a.state = (unsigned long long *)(w + at_state);
    const int e = launch_tile_plan(a, ctx->stream);
    if (e != hipSuccess) return give_up(T, hip_fail(ctx, (hipError_t)e, "tile plan"));
    if ((rc = copy_back(ctx, st, a.state, sizeof(st), "tile state copy")) != TOS_OK) return give_up(T, rc);
    if (st[0]) return give_up(T, TOS_OK);
    T.total = st[1];
    T.state = 1;
    return TOS_OK;
}

// Fewer candidate pairs than this take the general path.  Measured, general
// / tile, us per pass on a 200 x 200 Mpc/h grid of 50 x 50 bins: 426 pairs
// 535 / 260; 1,259 pairs 547 / 257; 9,061 pairs 770 / 383.  Below, a launch is
// a few tiles.
constexpr int64_t kTileMinPairs = 400;

// Whether the tile path can do a job of the list at all.
static bool tile_able(const tos_pairs *p, const tos_grid &g)
{
    const tos_catalog *cat = p->cat;
    // the plan's kernels step past a group's last pair in 32 bits
    if (p->n_pairs > INT32_MAX - kMaxGroup) return false;
    if (p->n_pairs < kTileMinPairs || cat->ladder.state == 2 || p->tiles.state == 2 || !(cat->l_step > 0)) return false;
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

// Blocks apart that two steps inside the axis-0 window can lie (all, without
// a window).
static int tile_band(const tos_catalog *cat, const tos_grid &g)
{
    const Ladder &L = cat->ladder;
    const std::vector<float> &key = g.type == TOS_OBSERVING ? L.h_l : L.h_d;
    const double X = grid_window_half(g, cat->dmax, g.type == TOS_OBSERVING ? cat->lmax_abs : cat->dmax);
    if (!(X > 0)) return L.nblk - 1;
    int band = 0;
    for (int b1 = 0; b1 < L.nblk; ++b1)
        for (int b2 = b1 + band + 1; b2 < L.nblk; ++b2) {
            if (!((double)key[(size_t)b2 * kBlockSteps] - (double)key[(size_t)b1 * kBlockSteps + kBlockSteps - 1] < X)) break;
            band = b2 - b1;
        }
    return band;
}

// From this squared separation up the edges are tracked (see tile_args).
static double tile_s_min(const tos_catalog *cat)
{
    const double scale = std::min(1.0, cat->dmax / 5000.0);
    return 4.0 * scale * scale;
}

// What the passes of a launch's jobs are expected to take, in us.
struct PassCost {
    int jobs = 0;
    // general path: the longest chain of one work item, the sightline pairs'
    // work, and that of N pixel pairs (w_pix: weighted)
    double gen_lat = 0, gen_pairs = 0, w_pix = 0, N = 0;
    // tile path: start, the visits' work, the longest chain of edges, of close
    // pairs; the plan
    double base = 140, tile = 0, edges = 0, near = 0, plan = 0;
    double general() const
    {
        const double pix = N > 0 ? std::min(2e-6 * w_pix, 3000.0 * w_pix / N + 3e-7 * w_pix) : 0.0;
        return 150 + (jobs > 1 ? 15.0 * jobs : 0.0) + std::hypot(gen_lat, gen_pairs + pix);
    }
    // (many jobs fill the device better than one that starts and ends alone)
    double tiles() const { return base + std::max(jobs > 1 ? 300 + 0.6 * tile : tile, edges) + near; }
    // (and their plans' memory is not that of a list just freed)
    double plans() const { return jobs > 1 ? 1.35 * plan : plan; }
    void add(const PassCost &o)
    {
        jobs += o.jobs;
        gen_lat = std::max(gen_lat, o.gen_lat);
        gen_pairs += o.gen_pairs;
        w_pix += o.w_pix;
        N += o.N;
        base = std::max(base, o.base);
        tile += o.tile;
        edges = std::max(edges, o.edges);
        near = std::max(near, o.near);
        plan += o.plan;
    }
};

// A visit costs the same whether its 256 pixel pairs exist or not, so sparse
// sightlines make the tile path the slower one; bins that are narrow for the
// pairs there are, and pairs too close to track, cost it as much; and a first
// pass pays for the plan.  The coefficients are a fit to 594 measured forms:
// 40 to 12,000 sightlines; 2 to 95 % of the pixels masked, sightlines cut to 3,
// 12 and 40 pixels or thinned 8 and 25 times; all grids, windows of 2 to 200
// Mpc/h, 50 to 4000 axis-1 bins; both precisions, two and seven sums.  Of
// the forms that the tile path makes slower by a tenth or more (780 pairs with
// 4000 bins 1.4 / 9.4 ms, 144,000 pairs thinned 25 times 0.67 / 0.78, 4,700
// pairs within 2 Mpc/h 0.58 / 0.87) the rule takes none.  Before the ladder is
// surveyed its size is that of the sampled spectra.
static PassCost pass_cost(const tos_ctx *ctx, const tos_pairs *p, const tos_grid &g, int prec, int accum)
{
    const tos_catalog *cat = p->cat;
    const Ladder &L = cat->ladder;
    const bool all = accum == TOS_ACC_ALL, polar = g.type == TOS_POLAR, obs = g.type == TOS_OBSERVING;
    const double P = (double)p->n_pairs, N = (double)p->h.stats.num_pixel_pairs;
    GridExact ge;
    grid_exact_consts(g, ge);
    const bool fixed = tile_fixed((int)ge.nslots);
    // the ladder's blocks, those of a sightline, the axis-0 band, and the share
    // of a pair's pixel pairs inside the axis-0 window
    const double X = grid_window_half(g, cat->dmax, obs ? cat->lmax_abs : cat->dmax);
    const double key_range = obs ? cat->l_range : cat->dmax - cat->dmin;
    const double steps = L.state ? (double)L.n_steps : cat->l_range / cat->l_step + 1.0;
    const double nblk = std::ceil(steps / kBlockSteps);
    const double nb = L.state ? L.mean_nb : std::min(nblk, cat->l_span / (cat->l_step * kBlockSteps) + 1.0);
    const double block = std::max(1e-300, key_range / std::max(1.0, nblk));
    const double band = X > 0 ? std::min(nblk - 1.0, std::floor(X / block) + 1.0) : nblk - 1.0;
    const double w = X > 0 ? std::min(1.0, 2.0 * X / (nb * block)) : 1.0;
    PassCost c;
    // general path; beyond the fixed layout LDS holds fewer wavefronts, and
    // too large a grid takes a pass for each band
    double f = all ? 3.5 : prec == TOS_FP64 ? 1.6 : 1.0;
    if (g.type != TOS_CARTESIAN) f *= 1.15;
    const uint32_t rows = std::max(1u, band_rows_for(ctx, accum, g));
    const double bands = (double)((ge.n[0] + rows - 1) / rows);
    const double Nw = N * (0.3 + 0.7 * w);
    const double partners = P / (double)std::max<int64_t>(1, p->n_rows), pix = std::sqrt(N / P);
    const double item = std::max(pix * std::sqrt(partners), partners * std::min(4.8, 0.25 * pix));
    c.gen_lat = (all ? 2.0 : f) * (fixed ? 1.0 : 1.6 * bands) * std::min(380.0, item) * (0.2 + 0.75 * w);
    const double g_all = f * bands * (fixed ? 1.0 : prec == TOS_FP64 ? 1.9 : 3.5);
    c.jobs = 1;
    c.gen_pairs = g_all * 2e-3 * P;
    c.w_pix = g_all * Nw;
    c.N = Nw;
    // tile path
    if (polar) c.base = 245;
    if (p->tiles.state == 0) c.plan = 190 + 11e-3 * std::min(P, 16384.0) + 0.8e-3 * P;
    const double all_visits = p->tiles.state == 1 ? (double)p->tiles.total : P * nb * nb;
    const double visits = std::max(1.0, all_visits * std::min(1.0, (2.0 * band + 1.0) / std::max(1.0, nb)));
    const double tiles = nblk * (2.0 * band + 1.0), bins = polar ? (double)tile_edges(g) : (double)ge.n[1];
    const double batch = (double)std::min<int64_t>(batch_pairs(p->n_pairs), p->n_pairs), batches = P / batch;
    // edges a cell passes per visit: each group of pairs takes a tile's cells
    // through all bins
    const double e = bins * tiles * std::ceil(P / kMaxGroup) / visits;
    c.tile = 0.8e-3 * P + visits * 1e-3 * (0.02 + 0.7 * std::max(std::sqrt(e), 2.0 * e)) * (all ? 2.5 : fixed ? 1.0 : P < 3e5 ? 1.25 : 2.7);
    if (obs) return c;
    c.edges = std::max(0.0, (polar ? 9.0 : 5.0) * (bins / std::sqrt(batches) - 30.0));
    // pairs too close to track, in one batch or a few
    const double reach = std::max(p->max_ang, 1e-9);
    const double close = std::min(1.0, tile_s_min(cat) / (cat->dmin * cat->dmin * reach * reach));
    const double cover = std::min(1.0, nb / nblk);
    c.near = (polar ? 25.0 : 17.0) * std::min(close * P, batch) * cover * cover + 0.75e-3 * close * visits;
    return c;
}

// The plan must pay for itself on this pass, or have paid on the passes that
// went without it: a list that is used again and again gets one at last.
static bool tiles_pay(const PassCost &c, int32_t passes_before)
{
    return (c.general() - c.tiles()) * (passes_before + 1.0) >= c.plans();
}

int choose_tiles(tos_ctx *ctx, int n, const TileJob *jobs, char *take)
{
    int rc;
    std::vector<PassCost> cost((size_t)n);
    auto price = [&](int j) { cost[(size_t)j] = pass_cost(ctx, jobs[j].p, *jobs[j].g, jobs[j].prec, jobs[j].accum); };
    auto pays = [&] {
        PassCost c;
        int32_t before = INT32_MAX;
        for (int j = 0; j < n; ++j) {
            if (!take[j]) continue;
            c.add(cost[(size_t)j]);
            if (jobs[j].p->tiles.state == 0) before = std::min(before, jobs[j].p->passes_before_plan);
        }
        return tiles_pay(c, before);
    };
    bool any = false;
    for (int j = 0; j < n; ++j) {
        if (!(take[j] = tile_able(jobs[j].p, *jobs[j].g))) continue;
        any = true;
        price(j);
    }
    if (!any) return TOS_OK;
    bool pay = pays();
    if (pay) {
        for (int j = 0; j < n; ++j) {
            if (!take[j]) continue;
            const int known = jobs[j].p->cat->ladder.state;
            if ((rc = survey_ladder(ctx, const_cast<tos_catalog *>(jobs[j].p->cat))) != TOS_OK) return rc;
            if (!(take[j] = jobs[j].p->cat->ladder.state != 2)) continue;
            if (known == 0) price(j);
            take[j] = cost[(size_t)j].tiles() < cost[(size_t)j].general();
        }
        pay = pays();
    }
    for (int j = 0; j < n; ++j) {
        if (!take[j]) continue;
        if (!pay) {
            if (jobs[j].p->passes_before_plan < 1000) ++jobs[j].p->passes_before_plan;
        } else if ((rc = ensure_tile_plan(ctx, jobs[j].p)) != TOS_OK) {
            return rc;
        }
        take[j] = pay && jobs[j].p->tiles.state == 1;
    }
    return TOS_OK;
}

bool drop_tiles(tos_ctx *ctx, tos_pairs *p)
{
    Ladder &L = const_cast<tos_catalog *>(p->cat)->ladder;
    if (p->tiles.state != 1 && L.state != 1) return false;
    (void)hipStreamSynchronize(ctx->stream);
    (void)give_up(p->tiles, TOS_OK);
    (void)give_up(L, TOS_OK);   // other lists of the catalogue: see tile_able
    return true;
}

bool tile_args(const tos_pairs *p, const tos_grid &g, TileArgs &t)
{
    const tos_catalog *cat = p->cat;
    const Ladder &L = cat->ladder;
    const TilePlan &T = p->tiles;
    t = TileArgs{};
    t.pix = (const float *)L.pix.ptr;
    t.d = L.d;
    t.l = L.l;
    t.masks = T.masks;
    t.words = T.words;
    t.rec = T.rec;
    t.batch_ptr = T.batch_ptr;
    t.visits = T.visits;
    t.nblk = L.nblk;
    t.n_batches = T.n_batches;
    t.width0 = g.width[0];
    t.width1 = g.width[1];
    t.band = tile_band(cat, g);
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
    t.s_min = tile_s_min(cat);
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
