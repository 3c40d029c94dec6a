// Stable LSD radix sort of u32 keys with u32 values ("onesweep" form),
// written for CDNA wave64.  Replaces the reference's 32 passes of 1-bit
// splits (engine/algorithms/radixSortKernels.cu:85-123), each of which runs a
// flag kernel, two multi-level scans, a split kernel and two gathers.
//
// Per sort:
//   1. one histogram kernel counts the 8-bit digits of every pass at once
//      and clears the look-back words;
//   2. one kernel per pass: each tile (256 lanes x 4..32 keys) ranks its keys by digit with
//      64-lane ballot matching (stable within the wave), publishes its digit
//      counts, resolves its global digit bases by the exclusive scan of the
//      pass's counts and per-digit decoupled look-back over earlier tiles,
//      stages the keys in LDS in sorted order and writes them out in digit
//      runs.
// Up to 8192 keys are sorted by one workgroup in one launch, all passes in
// its LDS (sort_small_kernel).
// A stable LSD sort has a unique output, so keys and the permutation match
// the reference's bit for bit.
#include "sort.hpp"

#include "scan_impl.hpp"

namespace flip2 {

namespace {

constexpr int kSortThreads = 256;             // 4 waves
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kRadix = 256;
constexpr int kHistThreads = 256;
constexpr int kLookback = 16;                 // earlier tiles whose status a digit loads per step
constexpr uint32_t kDigitFlagShift = 30;
constexpr uint32_t kDigitValueMask = (1u << kDigitFlagShift) - 1u;
constexpr uint32_t kDigitAggregate = 1u << kDigitFlagShift;
constexpr uint32_t kDigitInclusive = 2u << kDigitFlagShift;
constexpr int kMaxPasses = 4;

// Keys per lane of a digit-pass tile.  Large sorts: fewer tiles and
// look-backs, longer digit runs (32 measured fastest at millions of keys).
// Small ones are a chain of latencies, and a tile's ranking is a chain over
// its keys per lane: more, shorter tiles, as long as a look-back reaches the
// first in a few steps (24 bits: 65536 keys 33 us with 4 keys per lane, 40
// with 8, 49 with 16; 262144 keys 52, 53 and 57; 524288 keys 80, 63 and 64).
constexpr int kManyKeys = 1 << 20, kFewKeys = 1 << 18;
int sort_items(uint32_t n) { return n >= (uint32_t)kManyKeys ? 32 : n >= (uint32_t)kFewKeys ? 16 : 4; }

constexpr int kSmallThreads = 1024;
// Most keys of the one-workgroup sort: with 16 keys per lane it takes 52 us at
// 16384 keys over 32 bits, the digit kernels 34.
constexpr uint32_t kSmallKeys = 8 * kSmallThreads;

struct SortLayout {
    uint32_t passes;
    size_t histOff, counterOff, statusOff, total;
};

SortLayout sort_layout(uint32_t n, uint32_t beginBit, uint32_t endBit, int items) {
    SortLayout L{};
    L.passes = (endBit > beginBit) ? ceil_div(endBit - beginBit, 8) : 0;
    const uint32_t tiles = ceil_div(n ? n : 1, (uint32_t)items * kSortThreads);
    size_t off = 0;
    L.histOff = off; off += (size_t)kMaxPasses * kRadix * sizeof(uint32_t);
    L.counterOff = off; off += 256;
    L.statusOff = off; off += (size_t)L.passes * tiles * kRadix * sizeof(uint32_t);
    L.total = off + 256;
    return L;
}

__device__ inline uint32_t digit_of(uint32_t key, uint32_t shift, uint32_t mask) {
    return (key >> shift) & mask;
}

// Clears the digit histograms and the tile counters.
__global__ void sort_clear_kernel(uint32_t* words, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) words[i] = 0;
}

// Digit histograms of every pass.  A workgroup counts one chunk of 256 ITEMS
// keys in LDS (all of a thread's loads issued before its counting) and adds its
// counts to the global histogram, one atomic per non-empty bin.  The same
// launch clears the look-back status words of the passes.
template <int ITEMS>
__global__ void __launch_bounds__(kHistThreads)
sort_histogram_kernel(const uint32_t* __restrict__ keys, uint32_t n, uint32_t beginBit, uint32_t endBit,
                      uint32_t passes, uint32_t* __restrict__ hist, uint32_t* __restrict__ clearWords,
                      uint32_t clearCount) {
    __shared__ uint32_t s_hist[kMaxPasses * kRadix];
    for (int i = threadIdx.x; i < kMaxPasses * kRadix; i += kHistThreads) s_hist[i] = 0;
    for (uint32_t i = blockIdx.x * kHistThreads + threadIdx.x; i < clearCount; i += gridDim.x * kHistThreads)
        clearWords[i] = 0;
    constexpr uint32_t kChunk = kHistThreads * ITEMS;
    const uint32_t base = blockIdx.x * kChunk;
    const bool vec = (reinterpret_cast<uintptr_t>(keys) & 15u) == 0 && base + kChunk <= n;
    uint32_t key[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS / 4; ++k) {
        const uint32_t i = base + ((uint32_t)k * kHistThreads + threadIdx.x) * 4u;
        if (vec) {
            const uint4 v = *reinterpret_cast<const uint4*>(keys + i);
            key[4 * k] = v.x; key[4 * k + 1] = v.y; key[4 * k + 2] = v.z; key[4 * k + 3] = v.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) key[4 * k + e] = (i + e < n) ? keys[i + e] : 0u;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS / 4; ++k) {
        const uint32_t i = base + ((uint32_t)k * kHistThreads + threadIdx.x) * 4u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (i + e >= n) break;
            const uint64_t act = __ballot(true);
            const uint32_t lead = (uint32_t)__ffsll((unsigned long long)act) - 1u;
            for (uint32_t p = 0; p < passes; ++p) {
                const uint32_t shift = beginBit + 8u * p;
                const uint32_t bits = min(8u, endBit - shift);
                const uint32_t d = digit_of(key[4 * k + e], shift, (1u << bits) - 1u);
                // Keys that arrive nearly sorted (a FLIP step's particles,
                // sorted the step before) share their upper digits across a
                // wave, and 64 atomics on one LDS word serialise: a wave
                // whose digits agree adds its count with one atomic.
                const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
                if (__ballot(d == d0) == act) {
                    if ((threadIdx.x & 63u) == lead) atomicAdd(&s_hist[p * kRadix + d0], (uint32_t)__popcll(act));
                } else {
                    atomicAdd(&s_hist[p * kRadix + d], 1u);
                }
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < passes * kRadix; i += kHistThreads) {
        const uint32_t c = s_hist[i];
        if (c) atomicAdd(&hist[i], c);
    }
}

__device__ inline uint32_t digit_status_load(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void digit_status_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int ITEMS>
__global__ void __launch_bounds__(kSortThreads)
sort_pass_kernel(const uint32_t* __restrict__ keysIn, const uint32_t* __restrict__ valsIn,
                 uint32_t* __restrict__ keysOut, uint32_t* __restrict__ valsOut, uint32_t n,
                 uint32_t shift, uint32_t mask, const uint32_t* __restrict__ digitCounts,
                 uint32_t* __restrict__ status, uint32_t* __restrict__ counter) {
    __shared__ uint32_t s_keys[(ITEMS * kSortThreads)];
    __shared__ uint32_t s_vals[(ITEMS * kSortThreads)];
    __shared__ uint32_t s_wave[kSortWaves][kRadix];  // counts, then exclusive offsets across waves
    __shared__ uint32_t s_tileExcl[kRadix];
    __shared__ uint32_t s_globalBase[kRadix];
    __shared__ uint32_t s_scanTmp[2][kSortWaves];
    __shared__ uint32_t s_tile;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    if (tid == 0) s_tile = atomicAdd(counter, 1u);
    for (int i = tid; i < kSortWaves * kRadix; i += kSortThreads) (&s_wave[0][0])[i] = 0;
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t tileBase = tile * (uint32_t)(ITEMS * kSortThreads);
    const uint32_t waveBase = tileBase + (uint32_t)wave * (64u * ITEMS);

    uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t i = waveBase + (uint32_t)k * 64u + (uint32_t)lane;
        const bool valid = i < n;
        key[k] = valid ? keysIn[i] : 0xffffffffu;
        val[k] = valid ? (valsIn ? valsIn[i] : i) : 0u;
    }

    const uint64_t ltMask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t i = waveBase + (uint32_t)k * 64u + (uint32_t)lane;
        const bool valid = i < n;
        const uint32_t d = digit_of(key[k], shift, mask);
        uint64_t m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t bm = __ballot((d >> b) & 1u);
            m &= ((d >> b) & 1u) ? bm : ~bm;
        }
        const uint64_t lower = m & ltMask;
        const uint32_t before = s_wave[wave][d];
        __builtin_amdgcn_wave_barrier();
        if (valid && lower == 0) s_wave[wave][d] = before + (uint32_t)__popcll(m);
        __builtin_amdgcn_wave_barrier();
        rank[k] = before + (uint32_t)__popcll(lower);
    }
    __syncthreads();

    // Thread d: tile count of digit d and the wave-exclusive offsets.
    const uint32_t d = (uint32_t)tid;
    uint32_t tileCount = 0;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
        const uint32_t c = s_wave[w][d];
        s_wave[w][d] = tileCount;
        tileCount += c;
    }
    uint32_t* myStatus = status + (size_t)tile * kRadix + d;
    digit_status_store(myStatus, (tile == 0 ? kDigitInclusive : kDigitAggregate) | tileCount);

    // Exclusive scans over the 256 digits of the tile's counts and of the
    // whole pass's (the digits' offsets in the output).
    uint32_t digitOffset = 0;
    {
        const uint32_t incl = wave_inclusive_scan(tileCount);
        const uint32_t all = digitCounts[d], allIncl = wave_inclusive_scan(all);
        if (lane == 63) {
            s_scanTmp[0][wave] = incl;
            s_scanTmp[1][wave] = allIncl;
        }
        __syncthreads();
        uint32_t waveOff = 0;
        for (int w = 0; w < wave; ++w) {
            waveOff += s_scanTmp[0][w];
            digitOffset += s_scanTmp[1][w];
        }
        s_tileExcl[d] = waveOff + incl - tileCount;
        digitOffset += allIncl - all;
    }

    // Per-digit look-back over the earlier tiles, kLookback tiles per step:
    // their status loads are issued together, then consumed nearest first
    // until an inclusive prefix is found.  Inclusive prefixes then advance
    // kLookback tiles per status round trip.
    uint32_t prefix = 0;
    if (tile > 0) {
        int64_t j = (int64_t)tile - 1;
        for (;;) {
            uint32_t st[kLookback];
#pragma unroll
            for (int q = 0; q < kLookback; ++q)
                st[q] = (j - q >= 0) ? digit_status_load(status + (size_t)(j - q) * kRadix + d) : kDigitInclusive;
            bool done = false;
#pragma unroll
            for (int q = 0; q < kLookback; ++q) {
                if (!done) {
                    while ((st[q] >> kDigitFlagShift) == 0) {
                        __builtin_amdgcn_s_sleep(1);
                        st[q] = digit_status_load(status + (size_t)(j - q) * kRadix + d);
                    }
                    prefix += st[q] & kDigitValueMask;
                    done = (st[q] >> kDigitFlagShift) == 2u;
                }
            }
            if (done) break;
            j -= kLookback;
        }
        digit_status_store(myStatus, kDigitInclusive | (prefix + tileCount));
    }
    __syncthreads();
    s_globalBase[d] = digitOffset + prefix - s_tileExcl[d];

    // Stage in LDS in tile-sorted order.
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t i = waveBase + (uint32_t)k * 64u + (uint32_t)lane;
        if (i < n) {
            const uint32_t dk = digit_of(key[k], shift, mask);
            const uint32_t pos = s_tileExcl[dk] + s_wave[wave][dk] + rank[k];
            s_keys[pos] = key[k];
            s_vals[pos] = val[k];
        }
    }
    __syncthreads();

    const uint32_t valid = (n > tileBase) ? min((uint32_t)(ITEMS * kSortThreads), n - tileBase) : 0u;
    for (uint32_t j = (uint32_t)tid; j < valid; j += kSortThreads) {
        const uint32_t k = s_keys[j];
        const uint32_t o = s_globalBase[digit_of(k, shift, mask)] + j;
        if (o < n) {
            keysOut[o] = k;
            valsOut[o] = s_vals[j];
        }
    }
}

// Every pass of a sort of at most 1024 ITEMS keys by one workgroup: keys and
// values in registers, ranked as in sort_pass_kernel, scattered through LDS.
// A chain of latencies: 4099 keys over 32 bits take 26 us in one launch, the
// digit kernels' seven launches took 52.
template <int ITEMS>
__global__ void __launch_bounds__(kSmallThreads)
sort_small_kernel(const uint32_t* __restrict__ keysIn, const uint32_t* __restrict__ valsIn,
                  uint32_t* __restrict__ keysOut, uint32_t* __restrict__ valsOut, uint32_t n, uint32_t beginBit,
                  uint32_t endBit) {
    constexpr int kWaves = kSmallThreads / 64;
    __shared__ uint32_t s_kv[2][ITEMS * kSmallThreads];
    __shared__ uint32_t s_wave[kWaves][kRadix];
    __shared__ uint32_t s_scanTmp[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t waveBase = (uint32_t)wave * (64u * ITEMS) + (uint32_t)lane;
    uint32_t key[ITEMS], val[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t i = waveBase + 64u * (uint32_t)k;
        key[k] = i < n ? keysIn[i] : 0xffffffffu;
        val[k] = i < n ? (valsIn ? valsIn[i] : i) : 0u;
    }
    const uint64_t ltMask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (uint32_t shift = beginBit; shift < endBit; shift += 8u) {
        const uint32_t mask = (1u << min(8u, endBit - shift)) - 1u;
        for (int i = tid; i < kWaves * kRadix; i += kSmallThreads) (&s_wave[0][0])[i] = 0;
        __syncthreads();
        uint32_t rank[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const bool valid = waveBase + 64u * (uint32_t)k < n;
            const uint32_t d = digit_of(key[k], shift, mask);
            uint64_t m = __ballot(valid);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const uint64_t bm = __ballot((d >> b) & 1u);
                m &= ((d >> b) & 1u) ? bm : ~bm;
            }
            const uint64_t lower = m & ltMask;
            const uint32_t before = s_wave[wave][d];
            __builtin_amdgcn_wave_barrier();
            if (valid && lower == 0) s_wave[wave][d] = before + (uint32_t)__popcll(m);
            __builtin_amdgcn_wave_barrier();
            rank[k] = before + (uint32_t)__popcll(lower);
        }
        __syncthreads();
        // thread d < 256: the waves' exclusive offsets of digit d, after all
        // smaller digits
        uint32_t count = 0, incl = 0;
        if (tid < kRadix) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const uint32_t c = s_wave[w][tid];
                s_wave[w][tid] = count;
                count += c;
            }
            incl = wave_inclusive_scan(count);
            if (lane == 63) s_scanTmp[wave] = incl;
        }
        __syncthreads();
        if (tid < kRadix) {
            uint32_t off = incl - count;
            for (int w = 0; w < wave; ++w) off += s_scanTmp[w];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) s_wave[w][tid] += off;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            if (waveBase + 64u * (uint32_t)k < n) {
                const uint32_t pos = s_wave[wave][digit_of(key[k], shift, mask)] + rank[k];
                s_kv[0][pos] = key[k];
                s_kv[1][pos] = val[k];
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t i = waveBase + 64u * (uint32_t)k;
            if (i < n) {
                key[k] = s_kv[0][i];
                val[k] = s_kv[1][i];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t i = waveBase + 64u * (uint32_t)k;
        if (i < n) {
            keysOut[i] = key[k];
            valsOut[i] = val[k];
        }
    }
}

}  // namespace

uint32_t sort_passes(uint32_t beginBit, uint32_t endBit) {
    return (endBit > beginBit) ? ceil_div(endBit - beginBit, 8) : 0;
}

size_t sort_workspace_bytes(uint32_t n, uint32_t beginBit, uint32_t endBit) {
    if (endBit > 32) endBit = 32;
    // status words of 4096-key tiles, the shortest but for few keys, and enough
    // for every smaller sort (a workspace outlives one length)
    return std::max(sort_layout(n, beginBit, endBit, 16).total,
                    sort_layout(std::min<uint32_t>(n, kFewKeys - 1), beginBit, endBit, 4).total);
}

void sort_pairs_u32(const uint32_t* keysIn, const uint32_t* valsIn, uint32_t* keysOut, uint32_t* valsOut,
                    uint32_t* keysAlt, uint32_t* valsAlt, uint32_t n, uint32_t beginBit, uint32_t endBit,
                    void* ws, size_t wsBytes, hipStream_t stream, hipEvent_t* passEvents, int itemsPerThread) {
    int items = itemsPerThread ? itemsPerThread : sort_items(n);
    // (a workspace that holds only the status words of 4096-key tiles will do)
    if (!itemsPerThread && items == 4 && wsBytes < sort_layout(n, beginBit, endBit, 4).total) items = 16;
    FLIP2_REQUIRE(items == 4 || items == 16 || items == 24 || items == 32, kErrArgument,
                  "sort: 4, 16, 24 or 32 keys per lane");
    FLIP2_REQUIRE(endBit <= 32 && beginBit <= endBit, kErrArgument, "sort: bad bit range");
    FLIP2_REQUIRE(n < (1u << kDigitFlagShift), kErrRange, "sort: n must be below 2^30");
    FLIP2_REQUIRE(keysIn && keysOut && valsOut, kErrArgument, "sort: null buffer");
    FLIP2_REQUIRE(keysIn != keysOut && keysIn != keysAlt && (!valsIn || (valsIn != valsOut && valsIn != valsAlt)),
                  kErrArgument, "sort: inputs must not alias outputs");
    if (n == 0) return;
    const SortLayout L = sort_layout(n, beginBit, endBit, items);
    FLIP2_REQUIRE(ws && wsBytes >= L.total, kErrArgument, "sort: workspace too small");
    if (L.passes == 0) {
        FLIP2_HIP(hipMemcpyAsync(keysOut, keysIn, (size_t)n * 4, hipMemcpyDeviceToDevice, stream));
        if (valsIn) {
            FLIP2_HIP(hipMemcpyAsync(valsOut, valsIn, (size_t)n * 4, hipMemcpyDeviceToDevice, stream));
        } else {
            // identity permutation via a one-pass "sort" on an all-zero digit
            // range is overkill; the caller asked for no bits, so write iota.
            FLIP2_REQUIRE(false, kErrArgument, "sort: empty bit range needs explicit values");
        }
        return;
    }
    FLIP2_REQUIRE(L.passes == 1 || (keysAlt && valsAlt), kErrArgument, "sort: alternate buffers required");
    if (n <= kSmallKeys && !itemsPerThread) {
        if (passEvents) FLIP2_HIP(hipEventRecord(passEvents[0], stream));
        if (n <= 4u * kSmallThreads)
            FLIP2_KERNEL(sort_small_kernel<4>, dim3(1), dim3(kSmallThreads), 0, stream, keysIn, valsIn, keysOut,
                         valsOut, n, beginBit, endBit);
        else
            FLIP2_KERNEL(sort_small_kernel<8>, dim3(1), dim3(kSmallThreads), 0, stream, keysIn, valsIn, keysOut,
                         valsOut, n, beginBit, endBit);
        FLIP2_LAUNCH_CHECK();
        if (passEvents)
            for (uint32_t p = 0; p < L.passes; ++p) FLIP2_HIP(hipEventRecord(passEvents[p + 1], stream));
        return;
    }
    char* w = reinterpret_cast<char*>(ws);
    uint32_t* hist = reinterpret_cast<uint32_t*>(w + L.histOff);
    uint32_t* counters = reinterpret_cast<uint32_t*>(w + L.counterOff);
    uint32_t* status = reinterpret_cast<uint32_t*>(w + L.statusOff);

    // Histograms and tile counters are cleared first; the status words of the
    // passes (packed at this tile size) by the histogram kernel.
    const uint32_t tiles = ceil_div(n, (uint32_t)items * kSortThreads);
    const size_t passStride = (size_t)tiles * kRadix;
    const uint32_t headWords = (uint32_t)(L.statusOff / 4);
    FLIP2_KERNEL(sort_clear_kernel, dim3(ceil_div(headWords, 256)), dim3(256), 0, stream,
                       reinterpret_cast<uint32_t*>(w), headWords);
    FLIP2_LAUNCH_CHECK();
    // chunks of 8192 keys, of 1024 for small sorts (whose time is a chunk's)
    if (items > 4)
        FLIP2_KERNEL(sort_histogram_kernel<32>, dim3(ceil_div(n, 32u * kHistThreads)), dim3(kHistThreads), 0, stream,
                     keysIn, n, beginBit, endBit, L.passes, hist, status, (uint32_t)(L.passes * passStride));
    else
        FLIP2_KERNEL(sort_histogram_kernel<4>, dim3(ceil_div(n, 4u * kHistThreads)), dim3(kHistThreads), 0, stream,
                     keysIn, n, beginBit, endBit, L.passes, hist, status, (uint32_t)(L.passes * passStride));
    FLIP2_LAUNCH_CHECK();
    if (passEvents) FLIP2_HIP(hipEventRecord(passEvents[0], stream));

    // Ping-pong so that the last pass writes keysOut/valsOut.
    const uint32_t* srcK = keysIn;
    const uint32_t* srcV = valsIn;
    for (uint32_t p = 0; p < L.passes; ++p) {
        const bool toOut = ((L.passes - 1 - p) % 2) == 0;
        uint32_t* dstK = toOut ? keysOut : keysAlt;
        uint32_t* dstV = toOut ? valsOut : valsAlt;
        const uint32_t shift = beginBit + 8u * p;
        const uint32_t bits = std::min(8u, endBit - shift);
        const uint32_t mask = (1u << bits) - 1u;
        uint32_t* st = status + (size_t)p * passStride;
        if (items == 32)
            FLIP2_KERNEL(sort_pass_kernel<32>, dim3(ceil_div(n, 32u * kSortThreads)), dim3(kSortThreads), 0,
                               stream, srcK, srcV, dstK, dstV, n, shift, mask, hist + p * kRadix, st, counters + p);
        else if (items == 24)
            FLIP2_KERNEL(sort_pass_kernel<24>, dim3(ceil_div(n, 24u * kSortThreads)), dim3(kSortThreads), 0,
                               stream, srcK, srcV, dstK, dstV, n, shift, mask, hist + p * kRadix, st, counters + p);
        else if (items == 4)
            FLIP2_KERNEL(sort_pass_kernel<4>, dim3(ceil_div(n, 4u * kSortThreads)), dim3(kSortThreads), 0,
                               stream, srcK, srcV, dstK, dstV, n, shift, mask, hist + p * kRadix, st, counters + p);
        else
            FLIP2_KERNEL(sort_pass_kernel<16>, dim3(ceil_div(n, 16u * kSortThreads)), dim3(kSortThreads), 0,
                               stream, srcK, srcV, dstK, dstV, n, shift, mask, hist + p * kRadix, st, counters + p);
        FLIP2_LAUNCH_CHECK();
        if (passEvents) FLIP2_HIP(hipEventRecord(passEvents[p + 1], stream));
        srcK = dstK;
        srcV = dstV;
    }
}

}  // namespace flip2
