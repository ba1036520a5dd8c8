// tos_binning.h -- device code shared by the pair kernels: the reference's
// bin arithmetic, operation by operation, and the LDS histogram.  The files
// that include it are built with -ffp-contract=off.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "tos_internal.h"

namespace tos {
namespace {

// x86-64 cvttsd2si r64 then the low 32 bits: NaN / out of int64 range -> 0.
__device__ __forceinline__ uint32_t cvt_x86_slow(double t)
{
    if (!(t >= -9223372036854775808.0 && t < 9223372036854775808.0)) return 0u;
    return (uint32_t)(uint64_t)(int64_t)t;
}

// static_cast<unsigned>(t), rejected when >= n (n < 2^24).  For t in
// (-1, n) the cast is trunc(t); for t in [-4e9, -1] or [n, 4e9] the x86
// result is >= n; anything else (NaN, huge values) takes the exact path.
__device__ __forceinline__ uint32_t axis_checked(double t, uint32_t n)
{
    if (t > -1.0 && t < (double)n) return (uint32_t)(int32_t)t;
    if (fabs(t) < 4.0e9) return kReject;
    const uint32_t b = cvt_x86_slow(t);
    return b < n ? b : kReject;
}

// static_cast<unsigned>(t) without a range check (the z axis,
// XiEstimator.cc:200,253,287).
__device__ __forceinline__ uint32_t axis_unchecked(double t)
{
    if (t > -1.0 && t < 2147483647.0) return (uint32_t)(int32_t)t;
    return cvt_x86_slow(t);
}

__device__ __forceinline__ uint32_t z_bin_exact(const GridExact &g, float l1, float l2)
{
    const float lsum = l1 + l2;
    const double zc = 0.5 * (double)lsum;
    return axis_unchecked((zc - g.min[2]) * g.inv[2]);
}

// LDS slot of flat bin f < ntot (see GridExact::pad).
__device__ __forceinline__ uint32_t slot_of(const GridExact &g, uint32_t f)
{
    return f + (f / g.rowlen) * g.pad;
}

// Slot of the in-range triple (i0 < n0, i1 < n1, iz < n2): 24-bit
// multiply-adds (all factors are below 2^24).
__device__ __forceinline__ uint32_t slot3(const GridExact &g, uint32_t i0, uint32_t i1, uint32_t iz)
{
    return __umul24(i0, g.rowlen + g.pad) + __umul24(i1, g.n[2]) + iz;
}

// a * b + c for a, b < 2^24 (b wave-uniform, in an SGPR): one v_mad_u32_u24,
// where the compiler would otherwise emit two multiplies and a three-way add.
__device__ __forceinline__ uint32_t mad_u24(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

// Flat bin (reference order, u32 arithmetic) -> LDS slot or kReject.  When
// the z bin is the sightline pair's constant izc < n_z the flat bin is in
// range and its row is i0.
__device__ __forceinline__ uint32_t finish_bin(const GridExact &g, uint32_t i0, uint32_t i1, bool zc, uint32_t izc,
                                               float l1, float l2)
{
    if (zc) return slot3(g, i0, i1, izc);
    const uint32_t f = z_bin_exact(g, l1, l2) + (i1 + i0 * g.n[1]) * g.n[2];
    return f < g.ntot ? slot_of(g, f) : kReject;
}

// sqrt(x), correctly rounded, for x = +-0, +inf, NaN, x < 0 (NaN) and every
// x >= 2^-767: the hardware reciprocal square root refined by two
// Newton-Raphson (Goldschmidt) steps on g ~ sqrt(x) and h ~ 1/(2 sqrt(x)),
// the sequence the AMDGPU backend emits for sqrt(double) without its
// rescaling of inputs below 2^-767.  The squared separations binned here
// are built from FP32 distances: a nonzero one is at least ~1e-106.
__device__ __forceinline__ double sqrt_no_tiny(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    return (x == 0.0 || x == __builtin_inf()) ? x : g;
}

// Cartesian branch, XiEstimator.cc:226-259.
__device__ __forceinline__ uint32_t exact_bin_cart(const GridExact &g, float d1, float l1, double r1_sq,
                                                   double two_r1_cos12, float d2, float l2, bool zc,
                                                   uint32_t izc)
{
    const float adiff = fabsf(d1 - d2);
    const double r_para = (double)adiff;
    const uint32_t ipar = axis_checked((r_para - g.min[0]) * g.inv[0], g.n[0]);
    if (ipar == kReject) return kReject;
    const double d2d = (double)d2;
    const double r_sq = r1_sq + (d2d - two_r1_cos12) * d2d;
    const double rp2 = fabs(r_sq - r_para * r_para);
    const uint32_t iperp = axis_checked((sqrt_no_tiny(rp2) - g.min[1]) * g.inv[1], g.n[1]);
    if (iperp == kReject) return kReject;
    return finish_bin(g, ipar, iperp, zc, izc, l1, l2);
}

// Polar branch, XiEstimator.cc:168-225.
__device__ __forceinline__ uint32_t exact_bin_polar(const GridExact &g, float d1, float l1, double r1_sq,
                                                    double two_r1_cos12, float d2, float l2, bool zc,
                                                    uint32_t izc)
{
    const double d2d = (double)d2;
    const double r_sq = r1_sq + (d2d - two_r1_cos12) * d2d;
    const double r = sqrt_no_tiny(r_sq);
    const uint32_t ir = axis_checked((r - g.min[0]) * g.inv[0], g.n[0]);
    if (ir == kReject) return kReject;
    if (r == 0) return kReject;
    const float adiff = fabsf(d1 - d2);
    const double mu = (double)adiff / r;
    const uint32_t imu = axis_checked((mu - g.min[1]) * g.inv[1], g.n[1]);
    if (imu == kReject) return kReject;
    return finish_bin(g, ir, imu, zc, izc, l1, l2);
}

// Observing branch, XiEstimator.cc:261-294 (theta bin per sightline pair).
__device__ __forceinline__ uint32_t exact_bin_obs(const GridExact &g, float l1, float l2, uint32_t ith,
                                                  bool zc, uint32_t izc)
{
    const float adl = fabsf(l1 - l2);
    const uint32_t idl = axis_checked(((double)adl - g.min[0]) * g.inv[0], g.n[0]);
    if (idl == kReject) return kReject;
    // the theta bin is not range checked (XiEstimator.cc:273,283): it can
    // carry into the axis-0 index, so then the slot comes from the flat bin
    if (zc && ith < g.n[1]) return slot3(g, idl, ith, izc);
    const uint32_t iz = zc ? izc : z_bin_exact(g, l1, l2);
    const uint32_t f = iz + (ith + idl * g.n[1]) * g.n[2];
    return f < g.ntot ? slot_of(g, f) : kReject;
}

// The workgroup's LDS histogram: NSUM double arrays and one u32 count array
// of nslots entries.  FIXED: the arrays sit at compile-time offsets sized for
// kFixedSlots, so every update needs a single address computation.
constexpr uint32_t kFixedSlots = 2560;

template <int NSUM, bool FIXED>
struct Hist {
    double *hs;
    uint32_t *hc;
    uint32_t ns;      // runtime array stride (nslots) when !FIXED

    __device__ __forceinline__ Hist(double *base, uint32_t nslots)
        : hs(base), hc(reinterpret_cast<uint32_t *>(base + (size_t)(FIXED ? kFixedSlots : nslots) * NSUM)),
          ns(FIXED ? kFixedSlots : nslots)
    {
    }
    __device__ __forceinline__ uint32_t stride() const { return FIXED ? kFixedSlots : ns; }

    // n pixel pairs with summed terms into the slot at byte offset off8.
    __device__ __forceinline__ void add8n(uint32_t off8, uint32_t n, double didj, double ww) const
    {
        const uint32_t st8 = 8u * stride();
        char *bs = reinterpret_cast<char *>(hs);
        char *bc = reinterpret_cast<char *>(hc);
        __hip_atomic_fetch_add(reinterpret_cast<uint32_t *>(bc + (off8 >> 1)), n, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8), didj);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + st8), ww);
    }

    // The other five sums of the seven.
    __device__ __forceinline__ void add8n_more(uint32_t off8, double wd1, double wd2, double w1, double w2,
                                               double z) const
    {
        const uint32_t st8 = 8u * stride();
        char *bs = reinterpret_cast<char *>(hs);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 2 * st8), wd1);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 3 * st8), wd2);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 4 * st8), w1);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 5 * st8), w2);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 6 * st8), z);
    }

    // One pixel pair into the slot at byte offset off8 = 8 * slot of the
    // FP64 arrays (the count sits at off8 / 2 of the u32 array), so one
    // address register serves every array through immediate offsets.
    __device__ __forceinline__ void add8(uint32_t off8, float wd1, float w1, float l1, float wd2, float w2,
                                         float l2) const
    {
        const uint32_t st8 = 8u * stride();
        char *bs = reinterpret_cast<char *>(hs);
        char *bc = reinterpret_cast<char *>(hc);
        __hip_atomic_fetch_add(reinterpret_cast<uint32_t *>(bc + (off8 >> 1)), 1u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        const float didj = wd1 * wd2;
        const float ww = w1 * w2;
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8), (double)didj);
        unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + st8), (double)ww);
        if constexpr (NSUM == 7) {
            const float lsum = l1 + l2;
            unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 2 * st8), (double)wd1);
            unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 3 * st8), (double)wd2);
            unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 4 * st8), (double)w1);
            unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 5 * st8), (double)w2);
            unsafeAtomicAdd(reinterpret_cast<double *>(bs + off8 + 6 * st8), 0.5 * (double)lsum);
        }
    }
};

// Bytes of the histogram arrays, rounded up to 8; the workgroup's control
// words (item counter, two u64 tallies) follow them, so the histogram
// itself starts at LDS address 0 and every slot address is a plain
// register plus an immediate offset.
template <int NSUM, bool FIXED>
__host__ __device__ constexpr uint32_t hist_bytes(uint32_t nslots)
{
    return (((FIXED ? kFixedSlots : nslots) * (8u * NSUM + 4u)) + 7u) & ~7u;
}

}  // namespace
}  // namespace tos
