// tos_tileplan.hip -- plan of the tile path: the catalogue's ladder of
// (distance, loglam) steps, its pixels laid out on it, and the candidate
// pairs in batches sorted by separation.
//
// Survey spectra are resampled to one wavelength grid, so the distances of a
// catalogue's pixels take a few hundred values (the ladder).  On the ladder
// the axis-0 bin of a pixel pair depends on its two steps only, whatever the
// sightlines, and its axis-1 bin rises with the separation measure
// K = 2 (1 - c) of the sightline pair; tos_tilepass.hip walks the pairs of a
// batch in ascending K and keeps one running sum per pair of steps.
//
// A group of neighbouring pairs is sorted by K and cut into batches, so that
// a batch spans a part of the K range only: its tiles meet fewer bin edges
// than those of a batch of as many pairs cut out of the list.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "tos_internal.h"

namespace tos {
namespace {

constexpr int kWave = 64;
constexpr uint64_t kEmpty = ~0ull;

__device__ __forceinline__ uint32_t slot_hash(uint32_t dbits)
{
    return (dbits * 2654435761u) >> 19;   // 13 bits: kLadderTable slots
}

__device__ __forceinline__ uint64_t step_key(const float4 &p)
{
    return ((uint64_t)__float_as_uint(p.y) << 32) | __float_as_uint(p.x);
}

// Table slot of a key known to be present, or -1.
__device__ __forceinline__ int find_step(const uint64_t *table, uint64_t key)
{
    uint32_t h = slot_hash((uint32_t)key);
    for (int probe = 0; probe < kLadderTable; ++probe) {
        const uint64_t k = table[h];
        if (k == key) return (int)h;
        if (k == kEmpty) return -1;
        h = (h + 1) & (kLadderTable - 1);
    }
    return -1;
}

// Clears the table.  The last workgroup looks at kSample pixels spread over
// the catalogue: a distance with two wavelengths, or more than kMaxLadder
// distances, and there is no ladder (state[0]).  Finding that out by filling
// the table took 2 ms for 16,000 pixels off any ladder and 14 ms for 440,000
// (every thread of the device inserts, and probes an overfull table); this
// and its read-back take 20 to 30 us.
constexpr uint32_t kSample = 4096;
constexpr int kMaxProbe = 64;   // the tables are a quarter and half full at most
static_assert(kSample >= 2 * kMaxLadder && (kSample & (kSample - 1)) == 0, "slots of the sample's table");
__global__ void __launch_bounds__(1024) ladder_clear(LadderArgs a)
{
    __shared__ unsigned long long seen[kSample];
    __shared__ uint32_t distinct, bad;
    const int32_t i = (int32_t)(blockIdx.x * 1024 + threadIdx.x);
    if (i < kLadderTable) {   // whole workgroups: kLadderTable is a multiple of 1024
        a.table[i] = kEmpty;
        return;
    }
    for (uint32_t q = threadIdx.x; q < kSample; q += 1024) seen[q] = kEmpty;
    if (threadIdx.x == 0) distinct = bad = 0;
    __syncthreads();
    const int64_t n = min(a.n_pix, (int64_t)kSample), step = a.n_pix / n;
    for (uint32_t q = threadIdx.x; q < n; q += 1024) {
        const uint64_t key = step_key(a.pix[q * step]);
        uint32_t h = slot_hash((uint32_t)key) & (kSample - 1);
        for (int probe = 0; probe < kMaxProbe; ++probe) {
            // decided: no more of the probes, which get long
            if (__hip_atomic_load(&distinct, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > (uint32_t)kMaxLadder) break;
            const uint64_t k = atomicCAS(&seen[h], (unsigned long long)kEmpty, (unsigned long long)key);
            if (k == kEmpty) atomicAdd(&distinct, 1u);
            else if (k != key && (uint32_t)k == (uint32_t)key) bad = 1;
            if (k == kEmpty || (uint32_t)k == (uint32_t)key) break;
            if (probe + 1 == kMaxProbe) bad = 1;
            h = (h + 1) & (kSample - 1);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a.state[0] = bad || distinct > (uint32_t)kMaxLadder ? 1u : 0u;
        a.state[1] = a.state[2] = 0u;
    }
}
static_assert(kLadderTable % 1024 == 0, "ladder_clear's workgroups clear or sample as a whole");

// Every distinct (distance, loglam) of the catalogue into the hash table; a
// distance with two wavelengths, or more than kMaxLadder of them, ends the
// collection (state[0]).  The table is read before it is written, and almost
// every pixel finds its entry: 23.3 M pixels are read once, at L2 hit cost
// per probe.
__global__ void __launch_bounds__(256) ladder_collect(LadderArgs a)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    uint64_t last = kEmpty;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n_pix; i += stride) {
        if (__hip_atomic_load(&a.state[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
        const uint64_t key = step_key(a.pix[i]);
        if (key == last) continue;
        last = key;
        uint32_t h = slot_hash((uint32_t)key);
        for (int probe = 0;; ++probe) {
            if (probe == kMaxProbe) {
                a.state[0] = 1;
                break;
            }
            uint64_t k = __hip_atomic_load(&a.table[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (k == kEmpty) {
                if (__hip_atomic_compare_exchange_strong(&a.table[h], &k, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT)) {
                    const uint32_t n = __hip_atomic_fetch_add(&a.state[1], 1u, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_AGENT);
                    if (n >= (uint32_t)kMaxLadder) a.state[0] = 1;
                    break;
                }
            }
            if (k == key) break;
            if ((uint32_t)k == (uint32_t)key) {   // one distance, two wavelengths
                a.state[0] = 1;
                break;
            }
            h = (h + 1) & (kLadderTable - 1);
        }
    }
}

// First and last ladder step of each sightline: its blocks.
__global__ void __launch_bounds__(256) ladder_place(LadderArgs a)
{
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= a.n_los) return;
    const LosInfo li = a.los[s];
    uint32_t b0 = 0, nb = 0;
    if (li.n > 0) {
        const int h0 = find_step(a.table, step_key(a.pix[li.off]));
        const int h1 = find_step(a.table, step_key(a.pix[li.off + li.n - 1]));
        if (h0 < 0 || h1 < 0 || a.step[h1] < a.step[h0]) {
            a.state[0] = 1;
        } else {
            b0 = a.step[h0] / kBlockSteps;
            nb = a.step[h1] / kBlockSteps + 1 - b0;
        }
    }
    a.place[s].b0_nb = b0 | (nb << 8);
    a.nblk_of[s] = nb;
}

// Exclusive prefix of n counts in place, plus `base`; *total = base + sum.
__global__ void __launch_bounds__(1024) scan_u32(uint32_t *v, int64_t n, uint32_t base, uint32_t *total)
{
    __shared__ uint32_t part[1024];
    const int64_t per = (n + 1023) / 1024;
    const int64_t i0 = min(n, (int64_t)threadIdx.x * per), i1 = min(n, i0 + per);
    uint32_t s = 0;
    for (int64_t i = i0; i < i1; ++i) s += v[i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const uint32_t t = ((int)threadIdx.x >= off) ? part[threadIdx.x - off] : 0u;
        __syncthreads();
        part[threadIdx.x] += t;
        __syncthreads();
    }
    uint32_t acc = base + part[threadIdx.x] - s;
    for (int64_t i = i0; i < i1; ++i) {
        const uint32_t c = v[i];
        v[i] = acc;
        acc += c;
    }
    if (threadIdx.x == 1023) *total = base + part[1023];
}

__global__ void __launch_bounds__(256) zero_f4(float4 *p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// One wavefront per sightline: its pixels onto the ladder.  The steps must
// ascend within the sightline and the weights be finite (state[0] otherwise):
// where one of two sightlines has no pixel the pass multiplies by zero.
__global__ void __launch_bounds__(256) ladder_fill(LadderArgs a)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    if (s >= a.n_los) return;
    const LosInfo li = a.los[s];
    const uint32_t b0 = a.place[s].b0_nb & 255u, nb = a.place[s].b0_nb >> 8;
    const uint32_t first = a.nblk_of[s];
    if (lane == 0) a.place[s].off = kBlockBytes * (first - b0);
    int prev = -1;   // wave-uniform: the last step of the pixels before
    for (int32_t p0 = 0; p0 < li.n; p0 += kWave) {
        const int32_t p = p0 + lane;
        const bool in = p < li.n;
        int st = 0x7fffffff;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (in) {
            v = a.pix[li.off + p];
            const int h = find_step(a.table, step_key(v));
            st = h >= 0 ? (int)a.step[h] : -1;
        }
        int before = __shfl_up(st, 1);
        if (lane == 0) before = prev;
        const uint32_t at = (uint32_t)st - b0 * kBlockSteps;
        const bool ok = !in || (st > before && at < nb * kBlockSteps && __builtin_isfinite(v.z) &&
                                __builtin_isfinite(v.w));
        if (!ok) a.state[0] = 1;
        if (in && ok) {
            constexpr uint32_t ch = kChannelBytes / 4;
            float *o = a.out + (size_t)(first + at / kBlockSteps) * (3 * ch) + block_place(at % kBlockSteps);
            o[0] = v.z;
            o[ch] = v.w;
            o[2 * ch] = 1.0f;
        }
        prev = __shfl(st, kWave - 1);
    }
}

// The record of the group's pair `key` (K bits << 32 | index in the group) at
// its place `at` in ascending K.
__device__ __forceinline__ void put_record(const TilePlanArgs &a, int32_t p0, int32_t at, uint64_t key, int64_t r0,
                                           int64_t r1)
{
    const int32_t p = p0 + (int32_t)(uint32_t)key;
    while (r0 < r1) {   // last row with row_ptr <= p
        const int64_t mid = r0 + (r1 - r0 + 1) / 2;
        if (a.row_ptr[mid] <= p) r0 = mid;
        else r1 = mid - 1;
    }
    const LadderLos li = a.place[a.row_los[r0]], lj = a.place[a.other[p]];
    a.rec[p0 + at] = make_uint4(li.off, lj.off, (uint32_t)(key >> 32), (uint32_t)p);
    a.cover[p0 + at] = (li.b0_nb & 0xffffu) | (lj.b0_nb << 16);
}

// One workgroup per run of kSortRun pairs of a group: the run sorted by
// K = f32(2 (1 - c)) (a bitonic network over {K, index} in LDS).  A group of
// one run gets its records at once, the runs of a longer one go to a.keys.
// A coincident pair's c may exceed 1 by a rounding; its K is taken as 0.
__global__ void __launch_bounds__(1024) tile_sort(TilePlanArgs a)
{
    extern __shared__ uint64_t key[];
    const int32_t p0 = a.group_ptr[blockIdx.x], p1 = a.group_ptr[blockIdx.x + 1];
    const int32_t s0 = p0 + (int32_t)blockIdx.y * kSortRun;
    if (s0 >= p1) return;
    const int32_t n = min(p1 - s0, kSortRun);
    int32_t m = 2;
    while (m < n) m <<= 1;
    for (int32_t t = threadIdx.x; t < m; t += blockDim.x) {
        uint64_t k = kEmpty;
        if (t < n) {
            const double kd = 2.0 * (1.0 - a.csep[s0 + t]);
            if (!(kd > -1e-9 && kd < 4.5)) a.state[0] = 1;
            const float kf = kd > 0.0 ? (float)kd : 0.0f;
            k = ((uint64_t)__float_as_uint(kf) << 32) | (uint32_t)(s0 - p0 + t);
        }
        key[t] = k;
    }
    __syncthreads();
    for (int32_t k = 2; k <= m; k <<= 1) {
        for (int32_t j = k >> 1; j > 0; j >>= 1) {
            for (int32_t t = threadIdx.x; t < m / 2; t += blockDim.x) {
                const int32_t i = 2 * (t & ~(j - 1)) + (t & (j - 1));
                const uint64_t x = key[i], y = key[i + j];
                if ((x > y) == ((i & k) == 0)) {
                    key[i] = y;
                    key[i + j] = x;
                }
            }
            __syncthreads();
        }
    }
    const bool whole = p1 - p0 <= kSortRun;
    for (int32_t t = threadIdx.x; t < n; t += blockDim.x) {
        if (whole) put_record(a, p0, t, key[t], 0, a.n_rows - 1);
        else a.keys[s0 + t] = key[t];
    }
}

// Merges neighbouring runs of `width` keys of each group, from `src` to `dst`:
// a key's place is its index in its own run plus the number of smaller keys in
// the other (keys differ).  The last merge, of a whole group, writes the
// records.
__global__ void __launch_bounds__(256) tile_merge(TilePlanArgs a, const uint64_t *src, uint64_t *dst, int32_t width)
{
    const int32_t p0 = a.group_ptr[blockIdx.x], n = a.group_ptr[blockIdx.x + 1] - p0;
    const int32_t t = (int32_t)(blockIdx.y * blockDim.x + threadIdx.x);
    if (n <= kSortRun || t >= n) return;
    const uint64_t *keys = src + p0;
    const uint64_t mine = keys[t];
    const int32_t run = t / width, other = run ^ 1;
    const int32_t first = min(n, other * width);
    int32_t lo = first, hi = min(n, first + width);
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo) / 2;
        if (keys[mid] < mine) lo = mid + 1;
        else hi = mid;
    }
    const int32_t at = min(run, other) * width + (t - run * width) + (lo - first);
    if (dst) dst[p0 + at] = mine;
    else put_record(a, p0, at, mine, 0, a.n_rows - 1);
}

// Pairs covering each tile of a batch: corner counts of the covered
// rectangles, summed along both axes.
__global__ void __launch_bounds__(256) tile_visits(TilePlanArgs a)
{
    extern __shared__ int32_t cnt[];   // [(nblk + 1)][(nblk + 1)]
    const int32_t w = a.nblk + 1;
    for (int32_t t = threadIdx.x; t < w * w; t += blockDim.x) cnt[t] = 0;
    __syncthreads();
    for (int32_t p = a.batch_ptr[blockIdx.x] + threadIdx.x; p < a.batch_ptr[blockIdx.x + 1]; p += blockDim.x) {
        const uint32_t c = a.cover[p];
        const int32_t i0 = c & 255, i1 = i0 + ((c >> 8) & 255), j0 = (c >> 16) & 255, j1 = j0 + (c >> 24);
        atomicAdd(&cnt[i0 * w + j0], 1);
        atomicAdd(&cnt[i1 * w + j0], -1);
        atomicAdd(&cnt[i0 * w + j1], -1);
        atomicAdd(&cnt[i1 * w + j1], 1);
    }
    __syncthreads();
    for (int32_t i = threadIdx.x; i < w; i += blockDim.x)
        for (int32_t j = 1; j < w; ++j) cnt[i * w + j] += cnt[i * w + j - 1];
    __syncthreads();
    for (int32_t j = threadIdx.x; j < w; j += blockDim.x)
        for (int32_t i = 1; i < w; ++i) cnt[i * w + j] += cnt[(i - 1) * w + j];
    __syncthreads();
    uint32_t *out = a.visits + (size_t)blockIdx.x * a.nblk * a.nblk;
    uint64_t sum = 0;
    for (int32_t t = threadIdx.x; t < a.nblk * a.nblk; t += blockDim.x) {
        const uint32_t v = (uint32_t)cnt[(t / a.nblk) * w + t % a.nblk];
        out[t] = v;
        sum += v;
    }
    for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if ((threadIdx.x & (kWave - 1)) == 0) atomicAdd(&a.state[1], (unsigned long long)sum);
}

// Masks of the pairs whose sightlines cover each block: one wavefront per 64
// pairs, lane b keeping the words of blocks b and b + 64.
__global__ void __launch_bounds__(256) tile_masks(TilePlanArgs a)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int w = blockIdx.y * 4 + threadIdx.x / kWave;
    const int32_t p0 = a.batch_ptr[blockIdx.x], p1 = a.batch_ptr[blockIdx.x + 1];
    if (w * kWave >= p1 - p0) return;
    const int32_t p = p0 + w * kWave + lane;
    const uint32_t c = p < p1 ? a.cover[p] : 0u;
    for (int side = 0; side < 2; ++side) {
        const int b0 = (c >> (16 * side)) & 255, nb = (c >> (16 * side + 8)) & 255;
        uint64_t m0 = 0, m1 = 0;
        for (int b = 0; b < a.nblk; ++b) {
            const uint64_t m = __ballot((uint32_t)(b - b0) < (uint32_t)nb);
            if (lane == (b & 63)) (b < 64 ? m0 : m1) = m;
        }
        uint64_t *out = a.masks + ((size_t)(2 * blockIdx.x + side) * a.nblk) * a.words + w;
        if (lane < a.nblk) out[(size_t)lane * a.words] = m0;
        if (lane + 64 < a.nblk) out[(size_t)(lane + 64) * a.words] = m1;
    }
}

}  // namespace

int launch_ladder_collect(const LadderArgs &a, void *stream)
{
    if (a.n_pix <= 0) return 0;
    const int64_t blocks = (a.n_pix + 255) / 256;
    hipLaunchKernelGGL(ladder_clear, dim3(kLadderTable / 1024 + 1), dim3(1024), 0, (hipStream_t)stream, a);
    hipLaunchKernelGGL(ladder_collect, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0,
                       (hipStream_t)stream, a);
    return (int)hipGetLastError();
}

int launch_ladder_place(const LadderArgs &a, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    if (a.n_los <= 0) return 0;
    hipLaunchKernelGGL(ladder_place, dim3((unsigned)((a.n_los + 255) / 256)), dim3(256), 0, st, a);
    // block 0 is the zero block that padding entries of the pass read
    hipLaunchKernelGGL(scan_u32, dim3(1), dim3(1024), 0, st, a.nblk_of, a.n_los, 1u, a.state + 2);
    return (int)hipGetLastError();
}

int launch_ladder_fill(const LadderArgs &a, int64_t n_blocks, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    if (a.n_los <= 0) return 0;
    const int64_t n = n_blocks * (kBlockBytes / sizeof(float4));
    hipLaunchKernelGGL(zero_f4, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (float4 *)a.out, n);
    hipLaunchKernelGGL(ladder_fill, dim3((unsigned)((a.n_los + 3) / 4)), dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

int launch_tile_plan(const TilePlanArgs &a, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    if (a.n_batches <= 0) return 0;
    int32_t m = 2;
    while (m < a.max_group && m < kSortRun) m <<= 1;
    const size_t lds_sort = (size_t)m * 8, lds_cnt = (size_t)(a.nblk + 1) * (a.nblk + 1) * 4;
    hipError_t e = hipFuncSetAttribute((const void *)tile_sort, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds_sort);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)tile_visits, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_cnt);
    if (e != hipSuccess) return (int)e;
    const unsigned ng = (unsigned)a.n_groups, runs = (unsigned)((a.max_group + kSortRun - 1) / kSortRun);
    hipLaunchKernelGGL(tile_sort, dim3(ng, runs), dim3(1024), lds_sort, st, a);
    const uint64_t *src = a.keys;
    uint64_t *dst = a.keys2;
    for (int32_t width = kSortRun; width < a.max_group; width *= 2) {
        const bool last = 2 * width >= a.max_group;
        hipLaunchKernelGGL(tile_merge, dim3(ng, (unsigned)((a.max_group + 255) / 256)), dim3(256), 0, st, a, src,
                           last ? nullptr : dst, width);
        uint64_t *const t = dst;
        dst = const_cast<uint64_t *>(src);
        src = t;
    }
    hipLaunchKernelGGL(tile_masks, dim3((unsigned)a.n_batches, (unsigned)((a.words + 3) / 4)), dim3(256), 0, st, a);
    hipLaunchKernelGGL(tile_visits, dim3((unsigned)a.n_batches), dim3(256), lds_cnt, st, a);
    return (int)hipGetLastError();
}

}  // namespace tos
