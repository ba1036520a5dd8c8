// tos_tilepass.hip -- the pixel-pair pass on a ladder (tos_tileplan.hip).
//
// A tile is 16 x 16 pairs of ladder steps (k1, k2).  One wavefront walks the
// sightline pairs of a batch that cover a tile, in ascending K = 2 (1 - c):
// 256 pixel pairs per step, one running sum per (k1, k2) in registers.
//   products  one v_mfma_f32_16x16x1_4b per sightline pair: its four blocks
//             are the outer products w1 w2, (w d)1 (w d)2, 1 1 and one not used.  With
//             C = 0 a product rounds once, to the reference's own f32
//             product (types.h:77-87); the third block is 1 where both
//             sightlines have the pixel.
//   sums      each product is converted and added in FP64, as the reference
//             does.
//   bins      axis 0 depends on (k1, k2) alone and is evaluated once per
//             tile; axis 1 moves up one bin when K passes the edge's value,
//             held per lane in `thr`.  Only then are the sums added to the
//             workgroup's LDS histogram.  A pair whose K is within the error
//             bound of an edge, or whose separation is too small for the
//             bound, is binned with the reference arithmetic (slow_bin).
// So 64 pixel pairs cost some 9 VALU instructions (two conversions, two FP64
// additions and one count each, and a share of the scan and the edges) in
// place of 26 and three LDS atomics (xi_pairs_kernel).  VALU issue (0.82 of its
// peak for 37 million sightline pairs) and, for large catalogues, L2 misses on
// the sightlines' blocks (7.4e11 bytes at 6.5 TB/s there) bound the pass: 23
// instructions a visit of 256 pairs of steps and some 115 where an edge is
// passed.  Sorting larger groups (kMaxGroup) makes edges rarer: 46
// instructions a visit at 16384 pairs, 39 at 65536, 33 at 1048576 (Polar 41).
// 0.89 of a visit's 256 are pixel pairs, the rest covers ends of sightlines.
//
// Polar grids have both their axes move with K, at a K of its own for each
// pair of steps; the edges come from a table in LDS, so one formula serves
// both axes.  Where a tile's next pair has passed several edges of a cell the
// cell moves up again, without the reference arithmetic.
//
// 16 x 16 is the matrix instruction's tile and four cells a lane: with the
// running sums, two visits' operands and the edges it takes 128 vector
// registers, which keeps 16 wavefronts on a CU.  Wavefronts draw tiles from
// one counter; ranges of tiles of equal visits cut beforehand were 20 % slower
// (8.5 against 7.1 ms for 1.47 million sightline pairs), since the time of a
// visit varies with the edges it meets.
//
// Measured, us per pass, general kernel / this one: 3,450 sightline pairs 566
// / 218; 1.47 million (1.3e10 pixel pairs) FP64 25040 / 5130, Polar 16860 /
// 4790; 37 million (3.3e11) 335,000 / 115,400; Observing, 1.3 million pairs
// 13930 / 3690.
//
// With seven sums a second instruction forms (w d)1, (w d)2, w1 and w2 as
// products by 1, exactly; the mean wavelength is one number per cell.  141,344
// pairs, 50 x 50 x 3 bins in four bands: 64,240 / 3,390 us (the general kernel
// makes three full passes with eight atomics per pixel pair; here a band takes
// the tiles it has cells in).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "tos_binning.h"
#include "tos_internal.h"

namespace tos {
namespace {

constexpr int kWave = 64;
constexpr int kRun = 64;               // entries processed per run
constexpr int kChunk = 2 * kWave;      // pairs scanned at a time
constexpr int kQueue = kRun + kChunk;  // queue entries per wavefront

typedef float float16_v __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_v __attribute__((ext_vector_type(4)));

// A pointer into global memory: where the arguments are read from memory
// (tile_batch_kernel) the compiler would otherwise make every access a flat
// one.
#define TOS_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const TOS_GLOBAL T *global(const void *p)
{
    return (const TOS_GLOBAL T *)p;
}

// Orders a wavefront's LDS accesses before and after it, for its queue, which
// other lanes read than wrote it.  LDS serves a wavefront's accesses in order,
// so this holds the compiler only.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The workgroup's control words, after its histogram in LDS.
struct TileCtl {
    unsigned long long recheck;
    unsigned long long eval;
    uint32_t visits;                   // of the tiles taken so far
    int32_t pad;
};
constexpr size_t kTileCtlBytes = (sizeof(TileCtl) + 15) & ~(size_t)15;

// K of axis-1 edge e (in bins) of a pair of steps, lowered by its error
// bound (inv = (1 - eps) / (d1 d2)): r_perp^2 = K d1 d2 + base.
__device__ __forceinline__ float edge_k(double min1, double width1, float e, float base, float inv)
{
    const double s = __builtin_fma((double)e, width1, min1);
    return (float)__builtin_fma(s, s, -(double)base) * inv;
}

// r_perp^2 of a pair of steps at K, in the reference arithmetic
// (XiEstimator.cc:237-243): K d1 d2 + base up to rounding.
__device__ __forceinline__ float pair_base(float d1, float d2)
{
    const double a = (double)d1, b = (double)d2, rpar = (double)fabsf(d1 - d2);
    return (float)(((double)(d1 * d1) + b * b) - 2.0 * a * b - rpar * rpar);
}

__device__ __forceinline__ float pair_inv(float d1, float d2, double eps)
{
    return (float)((1.0 - eps) / ((double)d1 * (double)d2));
}

struct SlowBin {
    uint32_t off8;
    float edge, thr;
};

// The reference's bin of one pixel pair, and the K up to which it holds for
// its pair of steps (thr < 0: this pair only).  Out of line: it runs for a
// tile's first pair and for the rare pairs next to an edge.
__device__ __forceinline__ SlowBin slow_cart(const GridExact &ge, double width1, uint32_t band_lo8, float d1, float l1, float d2,
                                             float l2, double c, double eps, double s_min, float K, float k_safe)
{
    const double d2d = (double)d2;
    const double r1_sq = (double)(d1 * d1), two = (double)(2.0f * d1) * c;
    const uint32_t slot = exact_bin_cart(ge, d1, l1, r1_sq, two, d2, l2, false, 0);
    const double rpar = (double)fabsf(d1 - d2);
    const float base = pair_base(d1, d2);
    const float inv = pair_inv(d1, d2, eps);
    const double rp2 = fabs(r1_sq + (d2d - two) * d2d - rpar * rpar);
    const double t = (sqrt_no_tiny(rp2) - ge.min[1]) * ge.inv[1];
    const double n1 = (double)ge.n[1];
    // the edges around t (the cast truncates: (-1, 1) is one bin)
    const double lo = t >= n1 ? n1 : t >= 1.0 ? floor(t) : -1.0;
    const double up = t <= -1.0 ? -1.0 : floor(t < 0.0 ? 0.0 : t) + 1.0;
    const float k_up = edge_k(ge.min[1], width1, (float)up, base, inv);
    const bool no_lo = t <= -1.0 || __builtin_fma(lo, width1, ge.min[1]) <= 0.0;
    const float k_lo = no_lo ? -1.0f : edge_k(ge.min[1], width1, (float)lo, base, inv);
    const bool settled = rp2 >= s_min && k_lo <= k_safe && (t >= n1 || K < k_up) && z_bin_exact(ge, l1, l2) < ge.n[2];
    SlowBin s;
    s.off8 = slot == kReject ? kReject : (slot << 3) - band_lo8;
    s.edge = (float)up;
    s.thr = !settled || t <= -1.0 ? -1.0f : t >= n1 ? __builtin_inff() : k_up;
    return s;
}

// Polar: r^2 = K d1 d2 + r_par^2 + base, where base = f32(d1^2) - d1^2 since
// |d1 - d2| is exact (tile_job asks for dmax <= 2 dmin).  Each (k1, k2) meets
// the edges of r upwards and those of mu = r_par / r downwards: at
// r^2 = table[e], r edge e <= n0, and r^2 = r_par^2 table[n0 + 1 + j] with
// 1 / mu^2 of mu edge j (of the bins' lower edges; bin 0 ends at t = -1,
// where the cast truncates).
struct PolarStep {
    double rr, rrb;                    // r_par^2, r_par^2 + base
    float rpar, inv;                   // inv = (1 - eps) / (d1 d2)
};

__device__ __forceinline__ float polar_inv(float d1, float d2, float keep) { return keep * __builtin_amdgcn_rcpf(d1 * d2); }

__device__ __forceinline__ PolarStep polar_step(float d1, float d2, float inv)
{
    PolarStep p;
    const float sq = d1 * d1;
    p.rpar = fabsf(d1 - d2);
    p.rr = (double)p.rpar * (double)p.rpar;
    p.rrb = p.rr - (double)__builtin_fmaf(d1, d1, -sq);
    p.inv = inv;
    return p;
}

// K at r^2 = f t, lowered by its error bound
__device__ __forceinline__ float polar_k(const PolarStep &p, double f, double t)
{
    return (float)__builtin_fma(f, t, -p.rrb) * p.inv;
}

__device__ __forceinline__ double polar_edge(const GridExact &ge, const TileArgs &w, uint32_t i)
{
    if (i <= ge.n[0]) {
        const double r = __builtin_fma((double)i, w.width0, ge.min[0]);
        return r * r;
    }
    const uint32_t j = i - ge.n[0] - 1;
    const double mu = __builtin_fma(j > 0 ? (double)j : -1.0, w.width1, ge.min[1]);
    return mu > 0.0 ? 1.0 / (mu * mu) : (double)__builtin_inff();
}

struct SlowPolar {
    uint32_t off8, edges;
    float kr, km;
};

__device__ __forceinline__ SlowPolar slow_polar(const GridExact &ge, double width0, const double *table, uint32_t band_lo8,
                                                float d1, float l1, float d2, float l2, double c, float inv,
                                                double s_min, float K, float k_safe)
{
    const double d2d = (double)d2;
    const double r1_sq = (double)(d1 * d1), two = (double)(2.0f * d1) * c;
    const uint32_t slot = exact_bin_polar(ge, d1, l1, r1_sq, two, d2, l2, false, 0);
    const PolarStep p = polar_step(d1, d2, inv);
    const double r_sq = r1_sq + (d2d - two) * d2d;
    const double r = sqrt_no_tiny(r_sq);
    const double t0 = (r - ge.min[0]) * ge.inv[0], t1 = ((double)p.rpar / r - ge.min[1]) * ge.inv[1];
    const double n0 = (double)ge.n[0], n1 = (double)ge.n[1];
    // bins and edges around t0 and t1 (the cast truncates: (-1, 1) is one bin)
    const uint32_t i0 = t0 >= n0 ? ge.n[0] : t0 >= 1.0 ? (uint32_t)(int32_t)t0 : 0u;
    const uint32_t i1 = t1 >= n1 ? ge.n[1] : t1 >= 1.0 ? (uint32_t)(int32_t)t1 : 0u;
    const uint32_t mu0 = ge.n[0] + 1u;
    const double r_below = ge.min[0] - width0;
    const float k0 = i0 > 0u ? polar_k(p, 1.0, table[i0]) : r_below > 0.0 ? polar_k(p, r_below, r_below) : -1.0f;
    const bool no_mu = p.rpar == 0.0f;   // mu = 0 at any K
    const float k1 = t1 >= n1 || no_mu ? -1.0f : polar_k(p, p.rr, table[mu0 + (t1 <= -1.0 ? 0u : i1 + 1u)]);
    const float kr = polar_k(p, 1.0, table[min(i0 + 1u, ge.n[0])]);
    const float km = no_mu ? __builtin_inff() : polar_k(p, p.rr, table[mu0 + i1]);
    const bool dead = t0 >= n0 || t1 <= -1.0;
    const uint32_t iz = z_bin_exact(ge, l1, l2);
    const bool settled = r_sq - p.rr >= s_min && t0 > -1.0 && k0 <= k_safe && k1 <= k_safe && iz < ge.n[2] &&
                         (dead || (K < kr && K < km));
    SlowPolar s;
    s.edges = 0u;                      // in the mu axis
    if (!settled) {
        s.off8 = slot == kReject ? kReject : (slot << 3) - band_lo8;
        s.kr = -1.0f;
        s.km = __builtin_inff();
    } else if (dead) {
        s.off8 = kReject;
        s.kr = s.km = __builtin_inff();
    } else {
        // above the mu axis (i1 = n1) the slot is that of a bin past the row
        s.off8 = (slot3(ge, i0, i1, iz) << 3) - band_lo8;
        s.edges = (i0 + 1u) | (i1 << 16);
        s.kr = kr;
        s.km = km;
    }
    return s;
}

template <int NSUM, bool POLAR>
struct Cell {                          // one (k1, k2) of a lane
    double dd, ww;                     // running sums
    double x[NSUM == 7 ? 4 : 1];       // (w d)1, (w d)2, w1, w2
    float n;                           // pairs in them (exact: below 2^24)
    uint32_t off8;                     // LDS byte offset of their slot, kReject: none
    float thr;                         // K of the next edge (lower bound; Polar: of r); < 0: bin every pair exactly
    float edge;                        // that edge, in bins
    float km;                          // Polar: K of the next edge of mu
    uint32_t edges;                    // Polar: the next edges e | j << 16

    __device__ __forceinline__ float at() const { return POLAR ? fminf(thr, km) : thr; }
    // the running sums have a slot (Polar: mu is not above its axis)
    __device__ __forceinline__ bool in_axis(const GridExact &ge) const { return !POLAR || (edges >> 16) < ge.n[1]; }
};

template <int COORD, int NSUM, bool FIXED>
__device__ __forceinline__ void tile_block(const XiKernelArgs &a, const TileArgs &t, size_t part_row)
{
    constexpr bool POLAR = COORD == TOS_POLAR;
    using CellT = Cell<NSUM, POLAR>;
    const GridExact &ge = a.ge;
    const float keep = (float)(1.0 - t.eps);
    extern __shared__ double lds_tile[];
    const uint32_t nslots = FIXED ? ge.nslots : a.band_len8 / 8u;
    const Hist<NSUM, FIXED> H(lds_tile, nslots);
    char *after = reinterpret_cast<char *>(lds_tile) + ((hist_bytes<NSUM, FIXED>(nslots) + 15u) & ~15u);
    TileCtl &ctl = *reinterpret_cast<TileCtl *>(after);
    const int lane = threadIdx.x & (kWave - 1);
    uint4 *queue = reinterpret_cast<uint4 *>(after + kTileCtlBytes) + (threadIdx.x / kWave) * kQueue;
    double *table = reinterpret_cast<double *>(after + kTileCtlBytes + (blockDim.x / kWave) * (kQueue * sizeof(uint4)));
    if constexpr (POLAR)
        for (uint32_t i = threadIdx.x; i < ge.n[0] + ge.n[1] + 2u; i += blockDim.x) table[i] = polar_edge(ge, t, i);
    {
        const int ns = (int)H.stride();
        for (int b = threadIdx.x; b < ns * NSUM; b += blockDim.x) H.hs[b] = 0.0;
        for (int b = threadIdx.x; b < ns; b += blockDim.x) H.hc[b] = 0u;
    }
    if (threadIdx.x == 0) {
        ctl.visits = 0;
        ctl.recheck = 0ull;
        ctl.eval = 0ull;
    }
    __syncthreads();

    const int g = lane >> 4, col = lane & 15;
    // this lane's operand element: block (channel) g of row / column col;
    // row rho of the A operand is step 4 (rho mod 4) + rho / 4, so that
    // register r of the result holds the steps 4 r + g of its four lane groups
    const uint32_t at_a = 4u * col, at_b = 4u * col;
    // (the fourth block's result is not used)
    const uint32_t lane_a = at_a + kChannelBytes * min(g, 2), lane_b = at_b + kChannelBytes * min(g, 2);
    // the second instruction's blocks: (w d)1 1, 1 (w d)2, w1 1, 1 w2
    const uint32_t lane_a2 = at_a + kChannelBytes * (g == 0 ? 1 : g == 2 ? 0 : 2);
    const uint32_t lane_b2 = at_b + kChannelBytes * (g == 1 ? 1 : g == 3 ? 0 : 2);
    const TOS_GLOBAL char *pixels = global<char>(t.pix);
    const TOS_GLOBAL float *step_d = global<float>(t.d), *step_l = global<float>(t.l);
    const TOS_GLOBAL uint4_v *records = global<uint4_v>(t.rec);
    const int32_t wide = 2 * t.band + 1;
    uint32_t nre = 0;
    uint32_t neval = 0;                // a lane's share of a workgroup's pairs, below 2^32

    const uint32_t n_tiles = (uint32_t)(t.n_batches * t.nblk * wide);
    for (;;) {
        // the launch's next tile (drawn one at a time: 6.2 million
        // sightline pairs took no less with draws of 16), unless the
        // workgroup's u32 counts could overflow: kTileVisits visits of 256
        // pairs, and one tile of at most kMaxBatch visits more for each of its
        // wavefronts
        uint32_t id = ~0u;
        if (lane == 0 && __hip_atomic_load(&ctl.visits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < kTileVisits)
            id = __hip_atomic_fetch_add((TOS_GLOBAL uint32_t *)t.next, 1u, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
        id = (uint32_t)__builtin_amdgcn_readfirstlane((int)id);
        if (id >= n_tiles) break;
        const int32_t row = (int32_t)id / wide;
        const int32_t batch = row / t.nblk;
        const int32_t b1 = row - batch * t.nblk, b2 = b1 - t.band + ((int32_t)id - row * wide);
        if (b2 < 0 || b2 >= t.nblk) continue;
        const uint32_t visits = global<uint32_t>(t.visits)[(size_t)row * t.nblk + b2];
        if (visits == 0) continue;

        // the lane's four cells
        const float d2 = step_d[16 * b2 + block_place(col)], l2 = step_l[16 * b2 + block_place(col)];
        float inv_dd[4];               // Cartesian: (1 - eps) / (d1 d2), pair_base
        float base[4];
        float dist1[4];                // Polar: distances of the rows
        uint32_t f0[4];                // Observing: flat bin of the cell at theta bin 0
        float lsum[4];                 // seven sums: loglam1 + loglam2
        CellT cell[4];
        bool any = false;
        auto clear = [](CellT &c) {
            c.dd = c.ww = 0.0;
            if constexpr (NSUM == 7) c.x[0] = c.x[1] = c.x[2] = c.x[3] = 0.0;
            c.n = 0.0f;
        };
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float d1 = step_d[16 * b1 + block_place(4 * g + r)], l1 = step_l[16 * b1 + block_place(4 * g + r)];
            clear(cell[r]);
            if constexpr (NSUM == 7) lsum[r] = l1 + l2;
            cell[r].off8 = kReject;
            cell[r].edge = 0.0f;
            if constexpr (POLAR) {
                // r >= r_par, up to rounding: past the window none is in range
                dist1[r] = d1;
                inv_dd[r] = polar_inv(d1, d2, keep);
                const bool live = !a.window || (double)fabsf(d1 - d2) < a.win_half;
                cell[r].edges = 0u;
                cell[r].thr = live ? -1.0f : __builtin_inff();
                cell[r].km = __builtin_inff();
                any |= live;
                continue;
            }
            const double x0 = (double)(COORD == TOS_OBSERVING ? fabsf(l1 - l2) : fabsf(d1 - d2));
            const uint32_t i0 = axis_checked((x0 - ge.min[0]) * ge.inv[0], ge.n[0]);
            // dead cells: outside axis 0, or (Cartesian, with a regular z bin)
            // outside the band of axis-0 rows
            const uint32_t iz = z_bin_exact(ge, l1, l2);
            const bool live = i0 != kReject && (FIXED || COORD == TOS_OBSERVING || iz >= ge.n[2] ||
                                                i0 * ge.row8 - a.band_lo8 < a.band_len8);
            cell[r].thr = live ? -1.0f : __builtin_inff();
            any |= live;
            if constexpr (COORD == TOS_OBSERVING) {
                f0[r] = iz + i0 * ge.rowlen;
            } else if constexpr (COORD == TOS_CARTESIAN) {
                base[r] = pair_base(d1, d2);
                inv_dd[r] = pair_inv(d1, d2, t.eps);
            }
        }
        if (!__any(any)) continue;
        if (lane == 0) __hip_atomic_fetch_add(&ctl.visits, visits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        float next = -1.0f;            // Cartesian, Polar: K of the first edge of the lane's cells
        bool fresh = true;             // Observing: theta, the running sums' theta bin, is not set
        uint32_t theta = 0;

        auto empty = [&](CellT &c, uint32_t n) {
            neval += n;
            clear(c);
        };
        auto add = [&](const CellT &c, uint32_t n, float ls) {
            H.add8n(c.off8, n, c.dd, c.ww);
            // every pair of a cell has the same mean wavelength
            if constexpr (NSUM == 7)
                H.add8n_more(c.off8, c.x[0], c.x[1], c.x[2], c.x[3], (double)n * (0.5 * (double)ls));
        };
        auto flush = [&](CellT &c, float ls) {
            const uint32_t n = (uint32_t)c.n;
            if (n > 0u && c.off8 < a.band_len8 && c.in_axis(ge)) add(c, n, ls);
            empty(c, n);
        };
        // K reaches the threshold of some cell of the wavefront: cells that
        // pass one edge for certain move up one bin; any other one takes the
        // reference's bin at the pair's own c and the K up to which it holds
        auto cross = [&](float K, uint32_t p) {
            const uint32_t kb = __float_as_uint(K);
            const uint32_t kb_safe = kb > t.ulps ? kb - t.ulps : 0u;
            bool again;
            do {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    CellT &c = cell[r];
                    // as unsigned bits a negative thr is above every K
                    if (c.at() <= K && __float_as_uint(c.at()) <= kb_safe) {
                        const uint32_t n = (uint32_t)c.n;
                        // (a band of a larger grid holds a part of the slots)
                        if ((FIXED || c.off8 < a.band_len8) && c.in_axis(ge)) add(c, n, lsum[r]);
                        empty(c, n);
                        if constexpr (POLAR) {
                            float d1 = dist1[r];
                            asm volatile("" : "+v"(d1));   // its terms are formed here, not kept
                            const PolarStep p = polar_step(d1, d2, inv_dd[r]);
                            const bool of_r = !(c.km < c.thr);
                            // past the last r bin, or mu below its axis: for good
                            const bool out = of_r ? (c.edges & 0xffffu) >= ge.n[0] : c.edges < 0x10000u;
                            c.edges += of_r ? 1u : 0xffff0000u;
                            const uint32_t i = of_r ? c.edges & 0xffffu : ge.n[0] + 1u + (c.edges >> 16);
                            const float k = polar_k(p, of_r ? 1.0 : p.rr, table[out ? 0u : i]);
                            c.off8 = out ? kReject : c.off8 + (of_r ? ge.row8 : 0u - ge.nz8);
                            c.thr = out ? __builtin_inff() : of_r ? k : c.thr;
                            c.km = out ? __builtin_inff() : of_r ? c.km : k;
                            continue;
                        }
                        const bool out = c.edge >= (float)ge.n[1];
                        c.off8 = out ? kReject : c.off8 + ge.nz8;
                        c.edge += 1.0f;
                        float bs = base[r];
                        asm volatile("" : "+v"(bs));   // converted here, not kept as a double
                        c.thr = out ? __builtin_inff() : edge_k(ge.min[1], t.width1, c.edge, bs, inv_dd[r]);
                    }
                }
                next = fminf(fminf(cell[0].at(), cell[1].at()), fminf(cell[2].at(), cell[3].at()));
                // several edges passed since the tile's last pair: once more
                again = next <= K && __float_as_uint(next) <= kb_safe;
            } while (__any(again));
            if (__any(next <= K)) {
                const double cs = global<double>(a.csep)[p];
                uint32_t slow = 0;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (cell[r].at() <= K) {
                        slow |= 1u << r;
                        flush(cell[r], lsum[r]);
                    }
                // one copy of the code for the four cells
#pragma unroll 1
                for (int r = 0; r < 4; ++r) {
                    if ((slow >> r) & 1u) {
                        const int k1 = 16 * b1 + block_place(4 * g + r);
                        if constexpr (POLAR) {
                            const float d1 = step_d[k1];
                            const SlowPolar s = slow_polar(ge, t.width0, table, a.band_lo8, d1, step_l[k1], d2, l2, cs,
                                                           polar_inv(d1, d2, keep), t.s_min, K,
                                                           __uint_as_float(kb_safe));
                            nre += s.kr < 0.0f ? 1u : 0u;
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                cell[q].off8 = r == q ? s.off8 : cell[q].off8;
                                cell[q].edges = r == q ? s.edges : cell[q].edges;
                                cell[q].thr = r == q ? s.kr : cell[q].thr;
                                cell[q].km = r == q ? s.km : cell[q].km;
                            }
                            continue;
                        }
                        const SlowBin s = slow_cart(ge, t.width1, a.band_lo8, step_d[k1], step_l[k1], d2, l2, cs, t.eps,
                                                    t.s_min, K, __uint_as_float(kb_safe));
                        nre += s.thr < 0.0f ? 1u : 0u;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            cell[q].off8 = r == q ? s.off8 : cell[q].off8;
                            cell[q].edge = r == q ? s.edge : cell[q].edge;
                            cell[q].thr = r == q ? s.thr : cell[q].thr;
                        }
                    }
                }
                next = fminf(fminf(cell[0].at(), cell[1].at()), fminf(cell[2].at(), cell[3].at()));
                // nothing of this branch in flight where it joins the visits
                __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
            }
        };
        // Observing grid: another theta bin (XiEstimator.cc:273, unchecked: it
        // can carry into axis 0), the same one for every cell
        auto turn = [&](uint32_t th) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                flush(cell[r], lsum[r]);
                const uint32_t f = f0[r] + th * ge.n[2];
                cell[r].off8 = cell[r].thr < 0.0f && f < ge.ntot ? 8u * slot_of(ge, f) - a.band_lo8 : kReject;
            }
            theta = th;
        };
        auto visit = [&](float A, float B, float A2, float B2) {
            const float16_v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            const float16_v D = __builtin_amdgcn_mfma_f32_16x16x1f32(A, B, zero, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                cell[r].ww += (double)D[r];
                cell[r].dd += (double)D[4 + r];
                cell[r].n += D[8 + r];
            }
            if constexpr (NSUM == 7) {
                const float16_v E = __builtin_amdgcn_mfma_f32_16x16x1f32(A2, B2, zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int j = 0; j < 4; ++j) cell[r].x[j] += (double)E[4 * j + r];
            }
        };
        auto load_a = [&](uint32_t off) { return *(const TOS_GLOBAL float *)(pixels + (off + lane_a)); };
        auto load_a2 = [&](uint32_t off) { return NSUM == 7 ? *(const TOS_GLOBAL float *)(pixels + (off + lane_a2)) : 0.f; };
        auto load_b2 = [&](uint32_t off) { return NSUM == 7 ? *(const TOS_GLOBAL float *)(pixels + (off + lane_b2)) : 0.f; };
        auto load_b = [&](uint32_t off) { return *(const TOS_GLOBAL float *)(pixels + (off + lane_b)); };

        // the batch's pairs that cover the tile: the words of 64 pairs whose
        // masks for both blocks meet, 64 words at a time on the lanes
        const int32_t p0 = global<int32_t>(t.batch_ptr)[batch];
        const int n_words = (global<int32_t>(t.batch_ptr)[batch + 1] - p0 + kWave - 1) / kWave;
        const TOS_GLOBAL uint64_t *mask1 = global<uint64_t>(t.masks) + ((size_t)(2 * batch) * t.nblk + b1) * t.words;
        const TOS_GLOBAL uint64_t *mask2 = global<uint64_t>(t.masks) + ((size_t)(2 * batch + 1) * t.nblk + b2) * t.words;
        const uint32_t add1 = kBlockBytes * (uint32_t)b1, add2 = kBlockBytes * (uint32_t)b2;
        int w0 = -kWave;               // first word of the lanes' words
        uint64_t word = 0, left = 0;   // the lane's word; words still to queue
        int fill = 0;                  // queued entries (wave-uniform)
        // pairs of the next word, or 0 when there is none
        auto take = [&](int &w) -> uint64_t {
            while (left == 0) {
                w0 += kWave;
                if (w0 >= n_words) {
                    w0 = n_words;
                    return 0;
                }
                word = w0 + lane < n_words ? mask1[w0 + lane] & mask2[w0 + lane] : 0ull;
                left = __ballot(word != 0);
            }
            const int q = __ffsll((unsigned long long)left) - 1;
            left &= left - 1;
            w = w0 + q;
            return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(word >> 32), q) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)word, q);
        };
        for (;;) {
            bool done = false;
            while (fill < kRun && !done) {
                int wa = 0, wb = 0;
                const uint64_t ma = take(wa), mb = take(wb);
                done = mb == 0;
                const uint64_t below = (1ull << lane) - 1ull;
                const bool ia = (ma >> lane) & 1ull, ib = (mb >> lane) & 1ull;
                uint4_v ea = {0, 0, 0, 0}, eb = ea;
                if (ia) ea = records[p0 + wa * kWave + lane];
                if (ib) eb = records[p0 + wb * kWave + lane];
                if constexpr (COORD == TOS_OBSERVING) {   // the pair's theta bin in the place of K
                    if (ia) ea.z = global<uint32_t>(a.theta_bin)[ea.w];
                    if (ib) eb.z = global<uint32_t>(a.theta_bin)[eb.w];
                }
                if (ia) queue[fill + __popcll(ma & below)] = make_uint4(ea.x + add1, ea.y + add2, ea.z, ea.w);
                fill += __popcll(ma);
                if (ib) queue[fill + __popcll(mb & below)] = make_uint4(eb.x + add1, eb.y + add2, eb.z, eb.w);
                fill += __popcll(mb);
            }
            if (fill == 0) break;
            wave_lds_fence();
            int n = kRun;
            if (fill < kRun) {
                // padding entries read the zero block and repeat the last K
                n = (fill + 3) & ~3;
                const uint4 last = queue[fill - 1];
                if (lane < n - fill) queue[fill + lane] = make_uint4(0u, 0u, last.z, last.w);
                wave_lds_fence();
            }
            // four entries at a time; each operand register is loaded for the
            // entry four ahead as soon as its visit is done
            float A[4], B[4], A2[4], B2[4];
            uint32_t Z[4];             // K, or the theta bin
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                A[q] = load_a(queue[q].x);
                B[q] = load_b(queue[q].y);
                A2[q] = load_a2(queue[q].x);
                B2[q] = load_b2(queue[q].y);
                Z[q] = queue[q].z;
            }
            if (COORD == TOS_OBSERVING && fresh) {
                theta = ~Z[0];
                fresh = false;
            }
            for (int k = 0; k < n; k += 4) {
                const uint4 *ahead = queue + (k + 4 < n ? k + 4 : 0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t xa = ahead[q].x, xb = ahead[q].y, xk = ahead[q].z;
                    if constexpr (COORD == TOS_OBSERVING) {
                        if (__any(Z[q] != theta)) turn(Z[q]);
                    } else {
                        if (__any(next <= __uint_as_float(Z[q]))) cross(__uint_as_float(Z[q]), queue[k + q].w);
                    }
                    visit(A[q], B[q], A2[q], B2[q]);
                    A[q] = load_a(xa);
                    B[q] = load_b(xb);
                    A2[q] = load_a2(xa);
                    B2[q] = load_b2(xb);
                    Z[q] = xk;
                }
            }
            const int rest = fill > kRun ? fill - kRun : 0;   // at most kChunk
            wave_lds_fence();          // the visits' reads
            if (rest > 0) {
                const uint4 x = queue[kRun + lane], y = queue[kRun + (kWave + lane < kChunk ? kWave + lane : lane)];
                wave_lds_fence();
                queue[lane] = x;
                queue[kWave + lane] = y;
            }
            fill = rest;
            // past the last edge of every cell
            if (COORD != TOS_OBSERVING && !__any(next < __builtin_inff())) break;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) flush(cell[r], lsum[r]);
    }

    if (nre) __hip_atomic_fetch_add(&ctl.recheck, (unsigned long long)nre, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_WORKGROUP);
    if (neval) __hip_atomic_fetch_add(&ctl.eval, (unsigned long long)neval, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    const size_t out = part_row * (size_t)a.nbins;
    const uint32_t st = H.stride();
    const uint32_t band_slot0 = FIXED ? 0u : a.band_lo8 / 8u;
    for (int b = threadIdx.x; b < a.nbins; b += blockDim.x) {
        const uint32_t sl = slot_of(ge, (uint32_t)((FIXED ? 0 : a.band_bin0) + b)) - band_slot0;
        a.part_cnt[out + b] = H.hc[sl];
#pragma unroll
        for (int k = 0; k < NSUM; ++k) a.part_sum[(out + b) * NSUM + k] = H.hs[(size_t)k * st + sl];
    }
    if (threadIdx.x == 0) {
        if (ctl.recheck) __hip_atomic_fetch_add(&a.n_recheck[0], ctl.recheck, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (ctl.eval) __hip_atomic_fetch_add(&a.n_recheck[1], ctl.eval, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The seven sums take twice the vector registers and their histogram leaves
// room for one workgroup of eight wavefronts on a CU.
template <int COORD, int NSUM, bool FIXED>
__global__ void __launch_bounds__(NSUM == 7 ? 512 : kTileBlockMax)
__attribute__((amdgpu_waves_per_eu(NSUM == 7 ? 2 : 4, NSUM == 7 ? 2 : 4))) tile_pass_kernel(TileKernelArgs a)
{
    tile_block<COORD, NSUM, FIXED>(a.xi, a.tile, blockIdx.x);
}

// Many jobs in one launch: workgroup w serves job b.wg[w].job and writes its
// partial row b.wg[w].row.
template <int COORD, int NSUM, bool FIXED>
__global__ void __launch_bounds__(kTileBlockMax) __attribute__((amdgpu_waves_per_eu(4, 4)))
tile_batch_kernel(TileBatchArgs b)
{
    const XiWgTask w = b.wg[blockIdx.x];
    // a copy taken before the kernel writes anything: scalar loads
    const TileKernelArgs a = b.jobs[w.job];
    tile_block<COORD, NSUM, FIXED>(a.xi, a.tile, (size_t)w.row);
}

// n_wg == 0 only raises the kernel's dynamic LDS limit.
template <typename A>
hipError_t launch_one(void (*fn)(A), const A &a, int n_wg, int block, size_t lds, hipStream_t st)
{
    const hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess || n_wg == 0) return e;
    hipLaunchKernelGGL(fn, dim3(n_wg), dim3(block), lds, st, a);
    return hipGetLastError();
}

}  // namespace

bool tile_fixed(int nslots) { return (uint32_t)nslots <= kFixedSlots; }

int tile_threads_per_cu(int nsum) { return nsum == 7 ? 512 : 1024; }

// 512 threads where two workgroups share a CU's LDS, else 1024: 16
// wavefronts per CU either way (128 vector registers); 512 with seven sums.
int tile_block_size(int nsum, int nslots) { return nsum == 7 || tile_fixed(nslots) ? 512 : 1024; }

// n_edges: bins of both axes of a Polar grid, 0 on the others
size_t tile_lds_bytes(int nsum, int nslots, int n_edges)
{
    const size_t hist = nsum == 7           ? hist_bytes<7, false>(nslots)
                        : tile_fixed(nslots) ? hist_bytes<2, true>(nslots)
                                             : hist_bytes<2, false>(nslots);
    return ((hist + 15) & ~(size_t)15) + kTileCtlBytes +
           (size_t)(tile_block_size(nsum, nslots) / kWave) * kQueue * sizeof(uint4) +
           (n_edges > 0 ? (size_t)(n_edges + 2) * sizeof(double) : 0);
}

int launch_tile_pass(int coord, int nsum, const TileKernelArgs &a, int n_wg, int block, size_t lds, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    const bool fixed = !a.xi.banded && tile_fixed((int)a.xi.ge.nslots);
    void (*fn)(TileKernelArgs);
    if (nsum == 7)
        fn = coord == TOS_OBSERVING ? tile_pass_kernel<TOS_OBSERVING, 7, false>
             : coord == TOS_POLAR   ? tile_pass_kernel<TOS_POLAR, 7, false>
                                    : tile_pass_kernel<TOS_CARTESIAN, 7, false>;
    else if (coord == TOS_POLAR)
        fn = fixed ? tile_pass_kernel<TOS_POLAR, 2, true> : tile_pass_kernel<TOS_POLAR, 2, false>;
    else if (coord == TOS_OBSERVING)
        fn = fixed ? tile_pass_kernel<TOS_OBSERVING, 2, true> : tile_pass_kernel<TOS_OBSERVING, 2, false>;
    else
        fn = fixed ? tile_pass_kernel<TOS_CARTESIAN, 2, true> : tile_pass_kernel<TOS_CARTESIAN, 2, false>;
    return (int)launch_one(fn, a, n_wg, block, lds, st);
}

int launch_tile_batch(int coord, bool fixed, const TileBatchArgs &b, int n_wg, int block, size_t lds, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    if (coord == TOS_OBSERVING)
        return (int)(fixed ? launch_one(tile_batch_kernel<TOS_OBSERVING, 2, true>, b, n_wg, block, lds, st)
                           : launch_one(tile_batch_kernel<TOS_OBSERVING, 2, false>, b, n_wg, block, lds, st));
    if (coord == TOS_POLAR)
        return (int)(fixed ? launch_one(tile_batch_kernel<TOS_POLAR, 2, true>, b, n_wg, block, lds, st)
                           : launch_one(tile_batch_kernel<TOS_POLAR, 2, false>, b, n_wg, block, lds, st));
    return (int)(fixed ? launch_one(tile_batch_kernel<TOS_CARTESIAN, 2, true>, b, n_wg, block, lds, st)
                       : launch_one(tile_batch_kernel<TOS_CARTESIAN, 2, false>, b, n_wg, block, lds, st));
}

}  // namespace tos
