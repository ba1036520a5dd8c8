// tos_distance.hip -- the per-pixel distance transform of h5healxi.cc:196-216
// on the device: the FP64 line-of-sight comoving distance of every pixel's
// wavelength (tos_cosmo.h, the same arithmetic as the host's
// tos_cosmo_distances), rounded to the pixel's float.
//
// One integral is 512 terms of some 60 FP64 instructions, 1.4 ns of the whole
// device; a pixel is 8 bytes.  Pixels of a survey share one wavelength grid,
// so the integral is evaluated once per distinct loglam of the call:
//   collect  every loglam into a hash table, new ones into a list,
//   eval     one wavefront per listed value: lanes evaluate the terms, which
//            are then added in the host's order (the same bits),
//   look up  the table's float for every pixel.
// A call of about as many distinct values as the list holds, or more,
// evaluates one pixel per thread instead: the host samples the call, and where
// that has guessed too few the kernels decide by a device flag, without a
// copy back.
//
// Measured, one pixel per thread / this: kernels for 1.5 million pixels of 719
// wavelengths 2174 / 91 us (56 collecting); the call 2413 / 617 us, the rest
// copies of 12 MB; 12 million pixels 23.2 / 6.8 ms; 1 pixel 145 / 40 us, 1000
// pixels 134 / 48 us (the lanes share an integral).  All pixels distinct:
// 4096 pixels 144 / 74 us, 20,000 pixels 142 / 142, 1 million 1439 / 1442.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "tos_capi_impl.h"
#include "tos_cosmo.h"

using namespace tos;

namespace tos {
namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int kCollectBlock = 1024;
// 16 wavefronts on each of 256 CUs; the table is a quarter full at most, so
// that probes stay short.  Values beyond the list cost as much as pixels
// evaluated one per thread.
constexpr uint32_t kMaxValues = 4096;
constexpr uint32_t kSlots = 4 * kMaxValues;
constexpr uint32_t kMaxProbe = 64;           // at a quarter full a run this long does not occur by chance
constexpr uint32_t kNoValue = 0xffffffffu;   // a NaN

struct ValueTable {
    uint32_t key[kSlots];          // loglam bits, kNoValue: empty
    float dist[kSlots];
    uint32_t list[kMaxValues];     // slots taken
    uint32_t n;                    // of them
    uint32_t direct;               // more values than the list holds
};

struct DistanceArgs {
    const float *loglam;
    int64_t n;
    double ol, om, log_lya;
    ValueTable *t;
    float *out;
};

__device__ __forceinline__ uint32_t value_slot(uint32_t bits) { return (bits * 2654435761u) >> 18; }
static_assert(kSlots == 1u << 14, "value_slot takes the top 14 bits");

// The value's key: its bits (the NaN that marks empty slots takes those of
// another one).
__device__ __forceinline__ uint32_t value_key(float x)
{
    const uint32_t bits = __float_as_uint(x);
    return bits == kNoValue ? kNoValue - 1u : bits;
}

__global__ void __launch_bounds__(kCollectBlock) clear_table(DistanceArgs a)
{
    const uint32_t i = blockIdx.x * kCollectBlock + threadIdx.x;
    if (i < kSlots) a.t->key[i] = kNoValue;
    if (i == 0) a.t->n = a.t->direct = 0;
}

__device__ __forceinline__ void collect_value(ValueTable *t, uint32_t bits)
{
    uint32_t h = value_slot(bits);
    for (uint32_t probe = 0; probe < kMaxProbe; ++probe) {
        uint32_t k = __hip_atomic_load(&t->key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (k == kNoValue &&
            __hip_atomic_compare_exchange_strong(&t->key[h], &k, bits, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT)) {
            const uint32_t at = __hip_atomic_fetch_add(&t->n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (at >= kMaxValues) break;
            t->list[at] = h;
            return;
        }
        if (k == bits) return;
        h = (h + 1) & (kSlots - 1);
    }
    __hip_atomic_store(&t->direct, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The workgroup's last value of each slot, in LDS, keeps all but the first of
// its equal pixels off the table (a few hundred words that every wavefront
// of the device would read at once).
__global__ void __launch_bounds__(kCollectBlock) collect_values(DistanceArgs a)
{
    __shared__ uint32_t seen[kSlots];
    for (uint32_t i = threadIdx.x; i < kSlots; i += kCollectBlock) seen[i] = kNoValue;
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * kCollectBlock;
    for (int64_t i = (int64_t)blockIdx.x * kCollectBlock + threadIdx.x; i < a.n; i += stride) {
        const uint32_t bits = value_key(a.loglam[i]);
        const uint32_t h = value_slot(bits);
        if (__hip_atomic_load(&seen[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == bits) continue;
        if (__hip_atomic_load(&a.t->direct, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
        collect_value(a.t, bits);
        __hip_atomic_store(&seen[h], bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// One wavefront per listed value.
__global__ void __launch_bounds__(kBlock) eval_values(DistanceArgs a)
{
    __shared__ double term[kBlock / kWave][kLosTerms];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint32_t v = blockIdx.x * (kBlock / kWave) + wave;
    if (a.t->direct || blockIdx.x * (kBlock / kWave) >= a.t->n) return;   // the whole workgroup
    const bool on = v < a.t->n;
    const uint32_t slot = on ? a.t->list[v] : 0u;
    const double z = on ? pixel_redshift(a.log_lya, __uint_as_float(a.t->key[slot])) : 0.0;
    const double h = log1p_rn(z) / kLosPanels;
    for (int q = lane; q < kLosTerms; q += kWave) term[wave][q] = los_term(a.ol, a.om, h, q);
    __syncthreads();
    double acc = 0;
    for (int q = 0; q < kLosTerms; ++q) acc += term[wave][q];
    if (on && lane == 0) a.t->dist[slot] = z == 0 ? 0.0f : (float)(kLosScale * acc * 0.5 * h);
}

__global__ void __launch_bounds__(kBlock) look_up(DistanceArgs a)
{
    if (a.t->direct) return;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < a.n; i += stride) {
        const uint32_t bits = value_key(a.loglam[i]);
        uint32_t h = value_slot(bits);
        for (uint32_t probe = 1; probe < kMaxProbe && a.t->key[h] != bits; ++probe) h = (h + 1) & (kSlots - 1);
        a.out[i] = a.t->dist[h];
    }
}

__global__ void __launch_bounds__(kBlock) direct_distances(DistanceArgs a)
{
    if (a.t && !a.t->direct) return;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= a.n) return;
    a.out[i] = pixel_distance(a.ol, a.om, a.log_lya, a.loglam[i]);
}

// Whether a call has about as many distinct values as the list holds, or more:
// Chao's estimate from kSample pixels spread over it, which is 10 % off (one
// standard deviation) for equally frequent values.  Such a call is one launch,
// as if there were no table: finding it out on the device took 12 us with a
// sample there and 65 by filling the list.  The line lies at 0.85 of the list:
// 4500 values are taken for fewer once in 400 calls, 3000 for more once in 20.
constexpr int64_t kSample = 1024;

bool many_values(const float *loglam, int64_t n)
{
    if (n <= (int64_t)kMaxValues) return false;
    uint32_t key[2 * kSample], bits[kSample];
    uint16_t count[2 * kSample] = {};
    for (int64_t q = 0; q < kSample; ++q) std::memcpy(&bits[q], loglam + q * n / kSample, 4);
    int64_t seen = 0, once = 0, twice = 0;
    for (const uint32_t b : bits) {
        uint32_t h = (b * 2654435761u) >> 21;
        while (count[h] && key[h] != b) h = (h + 1) & (2 * kSample - 1);
        key[h] = b;
        const uint16_t c = ++count[h];
        seen += c == 1;
        once += c == 1 ? 1 : c == 2 ? -1 : 0;
        twice += c == 2 ? 1 : c == 3 ? -1 : 0;
    }
    const double distinct = (double)seen + (double)once * (double)once / (2.0 * std::max(0.5, (double)twice));
    return distinct > 0.85 * kMaxValues;
}
static_assert(2 * kSample == 1 << 11, "the sample's table takes the top 11 bits");

}  // namespace
}  // namespace tos

extern "C" int tos_pixel_distances(tos_ctx *ctx, double omega_lambda, double omega_matter, int64_t n,
                                   const float *loglam, float *distance)
{
    if (!ctx) return TOS_ERR_INVALID;
    if (n < 0 || (n > 0 && (!loglam || !distance)) || !std::isfinite(omega_lambda) || !std::isfinite(omega_matter)) {
        set_err(ctx, "tos_pixel_distances: invalid argument");
        return TOS_ERR_INVALID;
    }
    if (n == 0) return TOS_OK;
    if (omega_matter == 0) omega_matter = 1 - omega_lambda;   // h5healxi.cc:124
    hipSetDevice(ctx->device);
    const size_t nb = (size_t)n * sizeof(float);
    int rc;
    if ((rc = upload(ctx, ctx->scratch_a, loglam, nb, "pixel loglam")) != TOS_OK) return rc;
    const bool direct = many_values(loglam, n);
    if (ctx->scratch_b.reserve(nb) != TOS_OK || (!direct && ctx->scratch_c.reserve(sizeof(ValueTable)) != TOS_OK)) {
        set_err(ctx, "tos_pixel_distances: device allocation failed");
        return TOS_ERR_NOMEM;
    }
    const int64_t blocks = (n + kBlock - 1) / kBlock;
    if (blocks > 0x7fffffff) {
        set_err(ctx, "tos_pixel_distances: too many pixels for one launch");
        return TOS_ERR_INVALID;
    }
    DistanceArgs a{};
    a.loglam = (const float *)ctx->scratch_a.ptr;
    a.n = n;
    a.ol = omega_lambda;
    a.om = omega_matter;
    a.log_lya = std::log10(1216.0);   // constants.h:9-10 (lyA, logLyA)
    a.t = direct ? nullptr : (ValueTable *)ctx->scratch_c.ptr;
    a.out = (float *)ctx->scratch_b.ptr;
    if (!direct) {
        const unsigned some = (unsigned)std::min<int64_t>(blocks, 2048);
        const unsigned values = (unsigned)std::min<int64_t>(n, kMaxValues);
        hipLaunchKernelGGL(clear_table, dim3(kSlots / kCollectBlock), dim3(kCollectBlock), 0, ctx->stream, a);
        // two workgroups of 64 KiB on a CU
        const unsigned collect = (unsigned)std::min<int64_t>((n + kCollectBlock - 1) / kCollectBlock, 2 * ctx->ncu);
        hipLaunchKernelGGL(collect_values, dim3(collect), dim3(kCollectBlock), 0, ctx->stream, a);
        hipLaunchKernelGGL(eval_values, dim3((values + 3) / 4), dim3(kBlock), 0, ctx->stream, a);
        hipLaunchKernelGGL(look_up, dim3(some), dim3(kBlock), 0, ctx->stream, a);
    }
    hipLaunchKernelGGL(direct_distances, dim3((unsigned)blocks), dim3(kBlock), 0, ctx->stream, a);
    hipError_t he = hipGetLastError();
    if (he == hipSuccess) he = hipMemcpyAsync(distance, ctx->scratch_b.ptr, nb, hipMemcpyDeviceToHost, ctx->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(ctx->stream);
    if (he != hipSuccess) return hip_fail(ctx, he, "tos_pixel_distances");
    return TOS_OK;
}
