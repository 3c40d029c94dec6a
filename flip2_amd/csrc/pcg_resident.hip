// The whole inner PCG of one refinement (Jacobi or brick-local MIC(0)) in one
// kernel, the Krylov vectors resident in registers and LDS.
//
// What it replaces and why.  With two kernels per iteration every iteration
// streams ~50 bytes per cell through the caches and pays two launches (and,
// for large systems, two summing kernels).  The vectors of up to ~11000 slots
// fit the chip's registers and LDS, so here an iteration moves only the
// slots' faces (1.5 KB out and in per slot) and two grid-wide sums.  Per
// iteration of a solve, two-kernel form -> this one: 160 slots Jacobi 14.5 ->
// 4.3 us, MIC(0) 18.9 -> 6.7; 960 slots 18.5 -> 5.5 and 22.6 -> 7.7; 2383
// slots 21.9 -> 6.9 and 31.7 -> 9.9; 4122 slots 33.6 -> 10.1 and 45.4 -> 13.7;
// 9196 slots 54.5 -> 21.6 and 68.6 -> 22.6.
// What bounds it: up to ~2000 slots the latency of the two sums (a write
// and a read through memory each, ~1.5 us) and, with MIC(0), the chain of the
// sweeps' 44 steps; above, instruction issue beside the same waits: ~2500
// instructions per wave and iteration for four slots with MIC(0), half of them
// the sweeps.  2383 slots (one wave per SIMD): 4.2 of the 9.9 us at four clocks
// each; 9196 slots (nine waves per CU, three on one of its SIMDs): 12.5 of the
// 22.6 us, and waves wait for 65% of their time, among others for the registers
// that do not fit (see below).
//
// Layout of large systems (pcg_resident_kernel; pcg_wide_kernel, one slot per
// wave, has its own below).  A wave holds four slots, one per row of 16 lanes.  Lane 8 J + i of
// a row holds the cells (i, j = 4 J + b, k), b = 0..3, k = 0..7, of its slot:
// 32 cells per vector.  Register [b][m] holds k = (m - i - j) mod 8, so cells
// with the same i + j + k (mod 8) -- one anti-diagonal plane of the MIC(0)
// sweeps -- sit in the same register of every lane, and every neighbour of a
// cell is at a fixed register: (b, m -+ 1) for x and z, (b -+ 1, m -+ 1) for
// y, in the own lane or one DPP row shift away (by 1 for x, by 8 for y).
// The sweeps therefore run in registers (the two-kernel form exchanges every
// plane through LDS and is bound by it: ~260 LDS instructions per slot).
// Registers hold r, p, the factors and z / q; LDS holds e and the slot's six
// faces of p (neighbours' cells).  That takes 218 registers (MIC(0)) and 241
// (Jacobi), which up to eight waves per workgroup have; from nine on a lane has
// 168, and 50 and 81 of them go to scratch memory and back in an iteration (25
// reads and 8 writes per wave with MIC(0)).
//
// Per iteration: z = M^-1 r; the faces of z go out; sum r.z, r.r over the
// grid; p = z + beta p for the own cells and, with the neighbours' faces of
// z, for the face cells; q = A p; sum p.q over the grid; e += alpha p,
// r -= alpha q.
//
// Grid-wide sums.  Every workgroup publishes its sums as 64-bit words that
// carry 32 bits of a double and the sum's number, with relaxed agent-scope
// stores (written through to memory: L2 is per XCD), and reads all the
// others' until their numbers match; it adds them in workgroup order, so all
// get the same double.  The words are published in eight copies, one for the
// workgroups of each XCD: 256 workgroups reading the same lines wait for each
// other (960 slots, Jacobi: 6.2 -> 5.7 us per iteration).  The faces are
// written through and waited for before the words that announce them.  A
// workgroup waits for all others, so the launch needs every workgroup on the
// chip at once: the grid is one workgroup per CU at most, launches of one
// process take turns (resident_mutex), and every wait is bounded -- if it
// runs out (another process holds CUs), the kernel ends, reports it, and the
// caller solves with the two-kernel form.
#include "ns_solver.hpp"

#include <cstddef>

namespace flip2 {
namespace ns {

namespace {

constexpr int kRowSlots = 4;                // slots per wave
constexpr uint32_t kWideMaxWaves = 12;      // of a workgroup with one slot per wave
constexpr uint32_t kSumCopies = 8;          // of a sum's words, one per XCD
constexpr uint32_t kSumWords = kSumCopies * 256u * 4u;
constexpr uint32_t kFaceFloats = 384;       // floats of a slot's six faces

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Cache policy of the faces' accesses: sc1 (agent scope) -- stores write
// through the XCD's L2, loads do not hit in it.
constexpr int kAgent = 16;

constexpr int kRowShr1 = 0x111, kRowShr8 = 0x118, kRowShl1 = 0x101, kRowShl8 = 0x108;

// The value of the lane CTRL's row shift away, 0 where it lies outside the row.
template <int CTRL>
__device__ inline float row_shift(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// The same for the lanes of BANKS (groups of four lanes); the others get `other`.
template <int CTRL, int BANKS>
__device__ inline float row_shift_or(float other, float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(other), __float_as_int(v), CTRL, 0xf, BANKS, false));
}
// The value of the first lane of the row's quads 0 and 2 and of the last of
// quads 1 and 3 (lanes 0, 7, 8, 15: the cells with i = 0 and 7), in the quad.
__device__ inline float quad_edge(float v) {
    const int first = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x00, 0xf, 0xf, false);
    return __int_as_float(__builtin_amdgcn_update_dpp(first, __float_as_int(v), 0xff, 0xf, 0xa, false));
}
template <int CTRL>
__device__ inline double row_shift(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// a in the lanes of `lanes`, else b (a select that stays one: left to itself
// the compiler puts the selected value's computation under a branch, and the
// four columns' chains then no longer overlap).
__device__ inline float lanes_or(uint64_t lanes, float a, float b) {
    float o;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(o) : "v"(b), "v"(a), "s"(lanes));
    return o;
}
// Sum over the 16 lanes of a row, valid in its last lane (fixed order).
__device__ inline double row_sum(double v) {
    v += row_shift<0x111>(v);
    v += row_shift<0x112>(v);
    v += row_shift<0x114>(v);
    v += row_shift<0x118>(v);
    return v;
}

// v of one lane, for all.
__device__ inline double lane_value(double v, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Lanes (bit set) of every row whose cell of step t, column b lies in the
// brick: 0 <= t - b - i - 4 J <= 7.
constexpr uint64_t step_lanes(int t, int b) {
    uint32_t row = 0;
    for (int l = 0; l < 16; ++l) {
        const int k = t - b - (l & 7) - 4 * (l >> 3);
        if (k >= 0 && k <= 7) row |= 1u << l;
    }
    return (uint64_t)(row | (row << 16)) * 0x100000001ull;
}
// Lanes whose register m of column b holds plane k.
constexpr uint64_t plane_lanes(int m, int b, int k) {
    uint32_t row = 0;
    for (int l = 0; l < 16; ++l)
        if (((m - b - (l & 7) - 4 * (l >> 3)) & 7) == k) row |= 1u << l;
    return (uint64_t)(row | (row << 16)) * 0x100000001ull;
}

// One slot per wave: the lanes (8 j + i) with a cell of step t, and those whose
// register m holds plane k.
constexpr uint64_t wide_lanes(int t) {
    uint64_t o = 0;
    for (int l = 0; l < 64; ++l) {
        const int k = t - (l & 7) - (l >> 3);
        if (k >= 0 && k <= 7) o |= 1ull << l;
    }
    return o;
}
constexpr uint64_t wide_plane(int m, int k) {
    uint64_t o = 0;
    for (int l = 0; l < 64; ++l)
        if (((m - (l & 7) - (l >> 3)) & 7) == k) o |= 1ull << l;
    return o;
}
// The value of the lane 8 below / above (any in the lanes that have none).
// Half a row's neighbours are in its other half; the others come from the
// next row: rows are exchanged by the swaps of 16 and of 32 lanes.
__device__ inline float lane_up8(float v) {
    const unsigned u = (unsigned)__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true);  // halves swapped
    const auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);            // rows 0 0 2 2, 1 1 3 3
    const auto s32 = __builtin_amdgcn_permlane32_swap(s16[0], s16[1], false, false);  // rows 0 0 1 1, 2 2 3 3
    const float low = lanes_or(0xffff000000000000ull, __uint_as_float(s16[0]), __uint_as_float(s32[0]));
    return row_shift_or<kRowShr8, 0xc>(low, v);
}
__device__ inline float lane_down8(float v) {
    const unsigned u = (unsigned)__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true);
    const auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const auto s32 = __builtin_amdgcn_permlane32_swap(s16[0], s16[1], false, false);
    const float high = lanes_or(0x000000000000ffffull, __uint_as_float(s16[1]), __uint_as_float(s32[1]));
    return row_shift_or<kRowShl8, 0x3>(high, v);
}

// Forward and backward sweep of the MIC(0) factors pc: z = M^-1 z in place.
// Step t handles the plane i + j + k = t; the carried values of the previous
// step (0 in lanes without a cell) are the x, y and z neighbours'.  Off the
// fluid pc = 0, so such cells carry 0 (the coupling bits of the coefficients
// are not needed: two fluid neighbours are always coupled).  in0 / in7: 0 in
// the lanes whose x neighbour below / above lies in another row, else 1.
__device__ inline void mic_sweeps(float (&z)[4][8], const float (&pc)[4][8], float in0, float in7) {
    float w[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 22; ++t) {
        float wn[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int m = t & 7;
            if (t < b || t > b + 18) {  // no lane has a cell
                wn[b] = 0.f;
                continue;
            }
            float acc = z[b][m];
            acc = fmaf(row_shift<kRowShr1>(w[b]), in0, acc);
            acc += b ? w[b > 0 ? b - 1 : 0] : row_shift<kRowShr8>(w[3]);
            acc += w[b];
            const float q = acc * pc[b][m];
            z[b][m] = lanes_or(step_lanes(t, b), q, z[b][m]);
            wn[b] = lanes_or(step_lanes(t, b), q * pc[b][m], 0.f);
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) w[b] = wn[b];
    }
    float u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 21; t >= 0; --t) {
        float un[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int m = t & 7;
            if (t < b || t > b + 18) {
                un[b] = 0.f;
                continue;
            }
            const float f = pc[b][m];
            float acc = z[b][m];
            acc = fmaf(f, row_shift<kRowShl1>(u[b]) * in7, acc);
            acc = fmaf(f, b < 3 ? u[b < 3 ? b + 1 : 3] : row_shift<kRowShl8>(u[0]), acc);
            acc = fmaf(f, u[b], acc);
            const float x = acc * f;
            z[b][m] = lanes_or(step_lanes(t, b), x, z[b][m]);
            un[b] = lanes_or(step_lanes(t, b), x, 0.f);
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) u[b] = un[b];
    }
}

// v[k's register] per column: the values of plane K (0 or 7) in this lane.
template <int K>
__device__ inline float plane_value(const float (&v)[8], int b, int d0) {
    const int m = (K + b + d0) & 7;
    const float a0 = (m & 1) ? v[1] : v[0], a1 = (m & 1) ? v[3] : v[2], a2 = (m & 1) ? v[5] : v[4],
                a3 = (m & 1) ? v[7] : v[6];
    const float c0 = (m & 2) ? a1 : a0, c1 = (m & 2) ? a3 : a2;
    return (m & 4) ? c1 : c0;
}

// The operator's diagonal of cell (b, m), from its byte.
__device__ inline float diagonal(const uint32_t (&dg)[8], int b, int m) {
    return (float)((dg[2 * b + (m >> 2)] >> (8 * (m & 3))) & 0xffu);
}

__device__ inline v4u pack4(float a, float b, float c, float d) {
    v4u v;
    v.x = __float_as_uint(a);
    v.y = __float_as_uint(b);
    v.z = __float_as_uint(c);
    v.w = __float_as_uint(d);
    return v;
}

// One 64-bit word of a published sum: `half` (0 low, 1 high) of v's bits
// above the sum's number.
__device__ inline void publish(uint64_t* word, double v, int half, uint32_t number) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    const uint32_t part = half ? (uint32_t)(bits >> 32) : (uint32_t)bits;
    __hip_atomic_store(word, ((uint64_t)part << 32) | number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Orders a wave's LDS accesses between its lanes (they execute in order).
__device__ inline void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// What the workgroup shares besides e and the faces.
struct Shared {
    double slot[2][4 * kWideMaxWaves];  // per-slot sums
    double part[2][16];                     // row sums of the published values
    uint32_t bad;
};

// Grid-wide sums of a and (N == 2) b.  Words: N * 2 of 4 per workgroup and copy.
// False when a wait ran out.  Every thread of every workgroup gets the sums.
template <int N>
__device__ inline bool grid_sum(Shared& sh, double a, double b, const CgResident& c, uint64_t* words,
                                uint32_t number, double& sa, double& sb) {
    const uint32_t groups = c.groups;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, waves = blockDim.x >> 6;
    a = row_sum(a);
    if (N == 2) b = row_sum(b);
    if ((lane & 15u) == 15u) {
        sh.slot[0][wave * 4u + (lane >> 4)] = a;
        if (N == 2) sh.slot[1][wave * 4u + (lane >> 4)] = b;
    }
    // the faces written before this sum are in memory before it is announced
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (wave == 0) {
        const bool have = lane < 4u * waves;
        double x = have ? sh.slot[0][lane] : 0.0, y = (N == 2 && have) ? sh.slot[1][lane] : 0.0;
        x = row_sum(x);
        if (N == 2) y = row_sum(y);
        double tx = 0.0, ty = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            tx += lane_value(x, 16 * r + 15);
            if (N == 2) ty += lane_value(y, 16 * r + 15);
        }
        if (groups > 1u) {
            const uint32_t copy = lane / (2u * N), q = lane % (2u * N);
            if (copy < kSumCopies)
                publish(words + (copy * 256u + blockIdx.x) * 4u + q, q < 2u ? tx : ty, (int)(q & 1u), number);
        } else if (lane == 0) {
            sh.part[0][0] = tx;
            if (N == 2) sh.part[1][0] = ty;
        }
    }
    if (groups > 1u) {
        if (tid < 256u) {
            double x = 0.0, y = 0.0;
            if (tid < groups) {
                const uint64_t* w = words + ((blockIdx.x & (kSumCopies - 1u)) * 256u + tid) * 4u;
                uint64_t v[2 * N] = {};
                for (uint32_t t = 0; t < c.pause; ++t) __builtin_amdgcn_s_sleep(1);
                for (uint32_t poll = 0;; ++poll) {
                    if (poll >= c.polls) {
                        sh.bad = 1u;
                        break;
                    }
                    bool all = true;
#pragma unroll
                    for (int q = 0; q < 2 * N; ++q)
                        v[q] = __hip_atomic_load(w + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int q = 0; q < 2 * N; ++q) all = all && (uint32_t)v[q] == number;
                    if (all) break;
                }
                x = __builtin_bit_cast(double, (v[1] & 0xffffffff00000000ull) | (v[0] >> 32));
                if (N == 2) y = __builtin_bit_cast(double, (v[2 * N - 1] & 0xffffffff00000000ull) | (v[2 * N - 2] >> 32));
            }
            x = row_sum(x);
            if (N == 2) y = row_sum(y);
            if ((lane & 15u) == 15u) {
                sh.part[0][tid >> 4] = x;
                if (N == 2) sh.part[1][tid >> 4] = y;
            }
        }
        __syncthreads();
        if (sh.bad) return false;
        sa = sh.part[0][0];
        if (N == 2) sb = sh.part[1][0];
        const uint32_t rows = (groups + 15u) >> 4;
        for (uint32_t r = 1; r < rows; ++r) {
            sa += sh.part[0][r];
            if (N == 2) sb += sh.part[1][r];
        }
    } else {
        __syncthreads();
        sa = sh.part[0][0];
        if (N == 2) sb = sh.part[1][0];
    }
    return true;
}

}  // namespace

// LDS: Shared, then per wave e (8 x 64 float4) and the neighbours' faces of
// p (6 x 64 float4: -x, +x, y in two halves, -z, +z), laid out as a lane
// loads them.
constexpr uint32_t kWaveLds = (8u + 6u) * 64u * 16u;
constexpr uint32_t kWideLds = 80u * 32u;  // one slot per wave: p of its rows j = -1 .. 8

template <int MIC, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
pcg_resident_kernel(CgResident c) {
    extern __shared__ __align__(16) unsigned char s_raw[];
    Shared& sh = *reinterpret_cast<Shared*>(s_raw);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    float4* s_e = reinterpret_cast<float4*>(s_raw + ((sizeof(Shared) + 15u) & ~15u) + wave * kWaveLds) + lane;
    float4* s_h = s_e + 8 * 64;
    const uint32_t i = lane & 7u, J = (lane >> 3) & 1u;
    const int d0 = (int)(i + 4u * J);
    const uint32_t slotRaw = (blockIdx.x * waves + wave) * kRowSlots + (lane >> 4);
    const bool live = slotRaw < c.na;
    const uint32_t slot = live ? slotRaw : 0u;
    const float in0 = i == 0u ? 0.f : 1.f, in7 = i == 7u ? 0.f : 1.f;  // x neighbour in the lane next door
    const float out0 = -(1.f - in0), out7 = -(1.f - in7);
    // the x face cells that lanes with i = 0 and i = 7 meet (the others read
    // the former's)
    const float4* s_x = s_h - lane + (i == 7u ? 64u : 0u) + (lane & 48u) + 8u * J;
    if (threadIdx.x == 0) sh.bad = 0u;

    // The slot's cells.  cell address of (b, m): base + 64 ((m - b - d0) & 7) + 8 b
    const uint32_t base = slot * 512u + 32u * J + i;
    float r[4][8], p[4][8], pc[4][8], z[4][8];
    uint32_t dg[8];  // diagonal of cell 4 w + byte, w = 2 b + (m >> 2)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        // (every load before the first use, none under a condition; a padding
        // row reads slot 0 and keeps nothing of it)
        uint32_t cf[8];
        double r0[8];
        float f[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const uint32_t v = base + 64u * (uint32_t)((m - b - d0) & 7) + 8u * (uint32_t)b;
            cf[m] = c.coef[v];
            r0[m] = c.r64[v];
            f[m] = MIC ? c.precon[v] : 0.f;
        }
        dg[2 * b] = dg[2 * b + 1] = 0u;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const uint32_t keep = live && cf[m] != 0u ? 0xffffffffu : 0u, diag = cf[m] & keep & 7u;
            dg[2 * b + (m >> 2)] |= diag << (8 * (m & 3));
            if (!MIC) f[m] = 1.f / (float)max(diag, 1u);
            r[b][m] = __uint_as_float(__float_as_uint((float)r0[m]) & keep);
            pc[b][m] = __uint_as_float(__float_as_uint(f[m]) & keep);
            p[b][m] = 0.f;
        }
    }
#pragma unroll
    for (int w = 0; w < 8; ++w) s_e[64 * w] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < 6; ++w) s_h[64 * w] = make_float4(0.f, 0.f, 0.f, 0.f);

    // Faces in memory: slot, then face (-x, +x, -y, +y, -z, +z), 64 floats
    // each, in the owner's register order: x faces [J][m / 4][b][m % 4], y
    // faces [m / 4][i][m % 4], z faces [lane of the row][b].  Offsets past
    // the buffer (no such slot) read 0 and store nothing.
    constexpr uint32_t kNone = 0x80000000u;
    const __amdgpu_buffer_rsrc_t faces =
        __builtin_amdgcn_make_buffer_rsrc(c.faces, 0, c.na * kFaceFloats * 4u, 0x00027000);
    const uint32_t mine = live ? slot * (kFaceFloats * 4u) : kNone;
    // lane 4 Q + b of a row stores column b of an x face: lane 0's (Q = 0:
    // -x, J = 0), 7's (1: +x, J = 0), 8's (2: -x, J = 1) or 15's (3: +x, J = 1)
    const uint32_t outX = mine + ((lane & 4u) ? 256u : 0u) + 128u * J + 16u * (lane & 3u);
    const uint32_t outY = mine + (J ? 768u : 512u) + 16u * i;
    const uint32_t outZ = mine + 1024u + 16u * (lane & 15u);
    auto nbr = [&](uint32_t d, uint32_t face, uint32_t add) {  // the neighbour's face towards this slot
        const int32_t s = live ? c.nbrSlot[slot * 6u + d] : -1;
        return s < 0 ? kNone : (uint32_t)s * (kFaceFloats * 4u) + 256u * face + add;
    };
    const uint32_t l16 = 16u * (lane & 15u);
    const uint32_t inX0 = nbr(0, 1, l16), inX1 = nbr(1, 0, l16);
    const uint32_t inY = J ? nbr(3, 2, 16u * i) : nbr(2, 3, 16u * i);
    const uint32_t inZ0 = nbr(4, 5, l16), inZ1 = nbr(5, 4, l16);
    // (kNone plus the offsets added below stays past the buffer: it has less
    // than 2^31 bytes)

    uint64_t* words = c.words;
    double rzOld = 0.0;
    uint32_t it = 0;
    bool failed = false;
    for (;; ++it) {
        // what the loop derives from these is derived again in every
        // iteration (kept across it, it would not fit the registers)
#pragma unroll
        for (int w = 0; w < 8; ++w) asm volatile("" : "+v"(dg[w]));
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int m = 0; m < 8; ++m) asm volatile("" : "+v"(pc[b][m]));
        // z = M^-1 r and its sums
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                z[b][m] = r[b][m];
                if (!MIC) {  // r / diagonal, rounded as the quotient (r times the rounded reciprocal costs iterations)
                    const float q = r[b][m] * pc[b][m];
                    z[b][m] = fmaf(fmaf(-q, diagonal(dg, b, m), r[b][m]), pc[b][m], q);
                }
            }
        if (MIC) mic_sweeps(z, pc, in0, in7);
        // the faces go out first: they are on their way during the sums
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = 4 * h + e;
                v[e] = lanes_or(0x1111111111111111ull, quad_edge(z[0][m]), quad_edge(z[1][m]));
                v[e] = lanes_or(0x3333333333333333ull, v[e], lanes_or(0x4444444444444444ull, quad_edge(z[2][m]), quad_edge(z[3][m])));
            }
            __builtin_amdgcn_raw_buffer_store_b128(pack4(v[0], v[1], v[2], v[3]), faces, outX + (uint32_t)(64 * h), 0,
                                                   kAgent);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = J ? z[3][4 * h + e] : z[0][4 * h + e];
            __builtin_amdgcn_raw_buffer_store_b128(pack4(v[0], v[1], v[2], v[3]), faces, outY + (uint32_t)(128 * h), 0,
                                                   kAgent);
        }
        __builtin_amdgcn_raw_buffer_store_b128(pack4(plane_value<0>(z[0], 0, d0), plane_value<0>(z[1], 1, d0),
                                                     plane_value<0>(z[2], 2, d0), plane_value<0>(z[3], 3, d0)),
                                               faces, outZ, 0, kAgent);
        __builtin_amdgcn_raw_buffer_store_b128(pack4(plane_value<7>(z[0], 0, d0), plane_value<7>(z[1], 1, d0),
                                                     plane_value<7>(z[2], 2, d0), plane_value<7>(z[3], 3, d0)),
                                               faces, outZ + 256u, 0, kAgent);
        double srz = 0.0, srr = 0.0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                srz += (double)r[b][m] * (double)z[b][m];
                srr += (double)r[b][m] * (double)r[b][m];
            }
        double rz, rr;
        if (!grid_sum<2>(sh, srz, srr, c, words, c.number + 2u * it, rz, rr)) {
            failed = true;
            break;
        }
        if (rr <= c.thr2 || !(rr == rr) || it == c.limit) break;  // the same decision everywhere
        const float beta = it == 0u ? 0.f : rzOld != 0.0 ? (float)(rz / rzOld) : 0.f;
        rzOld = rz;

        // p = z + beta p, own cells and the neighbours' face cells
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int m = 0; m < 8; ++m) p[b][m] = fmaf(beta, p[b][m], z[b][m]);
        __builtin_amdgcn_sched_barrier(0);  // z's registers are free for the faces
        float4 h4[6];
#pragma unroll
        for (int w = 0; w < 6; ++w) {
            const uint32_t off =
                w == 0 ? inX0 : w == 1 ? inX1 : w < 4 ? inY + (uint32_t)(128 * (w - 2)) : w == 4 ? inZ0 : inZ1;
            h4[w] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(faces, off, 0, kAgent));
        }
#pragma unroll
        for (int w = 0; w < 6; ++w) {
            const float4 o = s_h[64 * w];
            s_h[64 * w] = make_float4(fmaf(beta, o.x, h4[w].x), fmaf(beta, o.y, h4[w].y), fmaf(beta, o.z, h4[w].z),
                                      fmaf(beta, o.w, h4[w].w));
        }
        __builtin_amdgcn_sched_barrier(0);
        wave_lds_order();

        // q = A p (in z)
        double spq = 0.0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            __builtin_amdgcn_sched_barrier(0);  // one column's faces in registers at a time
            const float zl = reinterpret_cast<const float*>(s_h + 256)[b], zh = reinterpret_cast<const float*>(s_h + 320)[b];
            float yh[8];
            if (b == 0 || b == 3) {
                const float4 y0 = s_h[128], y1 = s_h[192];
                yh[0] = y0.x; yh[1] = y0.y; yh[2] = y0.z; yh[3] = y0.w;
                yh[4] = y1.x; yh[5] = y1.y; yh[6] = y1.z; yh[7] = y1.w;
            }
            float xh[8];
            const float4 x0 = s_x[b], x1 = s_x[4 + b];
            xh[0] = x0.x; xh[1] = x0.y; xh[2] = x0.z; xh[3] = x0.w;
            xh[4] = x1.x; xh[5] = x1.y; xh[6] = x1.z; xh[7] = x1.w;
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const int lo = (m + 7) & 7, hi = (m + 1) & 7;
                float s = diagonal(dg, b, m) * p[b][m];
                s = fmaf(row_shift<kRowShr1>(p[b][lo]), -in0, s);
                s = fmaf(xh[lo], out0, s);
                s = fmaf(row_shift<kRowShl1>(p[b][hi]), -in7, s);
                s = fmaf(xh[hi], out7, s);
                s -= b > 0 ? p[b > 0 ? b - 1 : 0][lo] : row_shift_or<kRowShr8, 0xc>(yh[lo], p[3][lo]);
                s -= b < 3 ? p[b < 3 ? b + 1 : 3][hi] : row_shift_or<kRowShl8, 0x3>(yh[hi], p[0][hi]);
                s -= lanes_or(plane_lanes(m, b, 0), zl, p[b][lo]);
                s -= lanes_or(plane_lanes(m, b, 7), zh, p[b][hi]);
                const float q = pc[b][m] != 0.f ? s : 0.f;  // (pc is not 0 on the fluid)
                z[b][m] = q;
                spq += (double)p[b][m] * (double)q;
            }
        }
        double pq, unused;
        if (!grid_sum<1>(sh, spq, 0.0, c, words + kSumWords, c.number + 2u * it + 1u, pq, unused)) {
            failed = true;
            break;
        }
        const float alpha = pq != 0.0 ? (float)(rz / pq) : 0.f;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float4 e = s_e[64 * (2 * b + h)];
                e.x = fmaf(alpha, p[b][4 * h], e.x);
                e.y = fmaf(alpha, p[b][4 * h + 1], e.y);
                e.z = fmaf(alpha, p[b][4 * h + 2], e.z);
                e.w = fmaf(alpha, p[b][4 * h + 3], e.w);
                s_e[64 * (2 * b + h)] = e;
#pragma unroll
                for (int k = 0; k < 4; ++k) r[b][4 * h + k] = fmaf(-alpha, z[b][4 * h + k], r[b][4 * h + k]);
            }
    }

    // x += e on the fluid cells; the result for the host
    if (!failed && live) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const float4 e0 = s_e[64 * (2 * b)], e1 = s_e[64 * (2 * b + 1)];
            const float e[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
            double x[8];
#pragma unroll
            for (int m = 0; m < 8; ++m) x[m] = c.x64[base + 64u * (uint32_t)((m - b - d0) & 7) + 8u * (uint32_t)b];
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const uint32_t v = base + 64u * (uint32_t)((m - b - d0) & 7) + 8u * (uint32_t)b;
                if (pc[b][m] != 0.f) c.x64[v] = x[m] + (double)e[m];
            }
        }
    }
    if (threadIdx.x == 0) {
        if (blockIdx.x == 0) c.result[0] = it;
        if (failed) c.result[1] = c.number;
    }
}

// One slot per wave, for systems that leave the chip idle with four: lane
// 8 j + i holds the column (i, j) of its slot, register m its k = (m - i - j)
// mod 8 (as above, neighbours are at fixed registers; lanes 8 apart are
// exchanged by row swaps in the sweeps and through LDS in the product), and
// the correction e stays in registers.  A quarter of the instructions per
// wave: 160 slots, Jacobi 6.5 -> 5.2 us per iteration, MIC(0) 9.1 -> 7.6
// (before the sums' copies and pauses).
template <int MIC>
__global__ void __launch_bounds__(64 * kWideMaxWaves)
pcg_wide_kernel(CgResident c) {
    extern __shared__ __align__(16) unsigned char s_raw[];
    Shared& sh = *reinterpret_cast<Shared*>(s_raw);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    // p of rows j = -1 .. 8 (8 lanes of 8 registers each)
    float4* s_p = reinterpret_cast<float4*>(s_raw + ((sizeof(Shared) + 15u) & ~15u) + wave * kWideLds) + 16 + 2 * lane;
    const uint32_t i = lane & 7u, j = lane >> 3;
    const int d0 = (int)(i + j);
    const uint32_t slotRaw = blockIdx.x * waves + wave;
    const bool live = slotRaw < c.na;
    const uint32_t slot = live ? slotRaw : 0u;
    const float in0 = i == 0u ? 0.f : 1.f, in7 = i == 7u ? 0.f : 1.f;
    const float jn0 = j == 0u ? 0.f : 1.f, jn7 = j == 7u ? 0.f : 1.f;
    if (threadIdx.x == 0) sh.bad = 0u;

    const uint32_t base = slot * 512u + lane;
    float r[8], p[8], pc[8], z[8], e[8], dg[8];
    float xh[8], yh[8], zl = 0.f, zh = 0.f;  // the neighbours' faces of p (x: lanes i = 0, 7; y: j = 0, 7)
    {
        uint32_t cf[8];
        double r0[8];
        float f[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const uint32_t v = base + 64u * (uint32_t)((m - d0) & 7);
            cf[m] = c.coef[v];
            r0[m] = c.r64[v];
            f[m] = MIC ? c.precon[v] : 0.f;
        }
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const uint32_t keep = live && cf[m] != 0u ? 0xffffffffu : 0u, diag = cf[m] & keep & 7u;
            dg[m] = (float)diag;
            if (!MIC) f[m] = 1.f / (float)max(diag, 1u);
            r[m] = __uint_as_float(__float_as_uint((float)r0[m]) & keep);
            pc[m] = __uint_as_float(__float_as_uint(f[m]) & keep);
            p[m] = e[m] = xh[m] = yh[m] = 0.f;
        }
    }

    constexpr uint32_t kNone = 0x80000000u;
    const __amdgpu_buffer_rsrc_t faces =
        __builtin_amdgcn_make_buffer_rsrc(c.faces, 0, c.na * kFaceFloats * 4u, 0x00027000);
    // x faces [j][m], y faces [i][m] in the owner's register order, z faces [j][i]
    const uint32_t mine = live ? slot * (kFaceFloats * 4u) : kNone;
    const uint32_t outX = i == 0u ? mine + 32u * j : i == 7u ? mine + 256u + 32u * j : kNone;
    const uint32_t outY = j == 0u ? mine + 512u + 32u * i : j == 7u ? mine + 768u + 32u * i : kNone;
    const uint32_t outZ = mine + 1024u + 4u * lane;
    auto nbr = [&](uint32_t d, uint32_t face, uint32_t add) {
        const int32_t s = live ? c.nbrSlot[slot * 6u + d] : -1;
        return s < 0 ? kNone : (uint32_t)s * (kFaceFloats * 4u) + 256u * face + add;
    };
    const uint32_t inX = i == 0u ? nbr(0, 1, 32u * j) : i == 7u ? nbr(1, 0, 32u * j) : kNone;
    const uint32_t inY = j == 0u ? nbr(2, 3, 32u * i) : j == 7u ? nbr(3, 2, 32u * i) : kNone;
    const uint32_t inZ0 = nbr(4, 5, 4u * lane), inZ1 = nbr(5, 4, 4u * lane);

    uint64_t* words = c.words;
    double rzOld = 0.0;
    uint32_t it = 0;
    bool failed = false;
    for (;; ++it) {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            z[m] = r[m];
            if (!MIC) {
                const float q = r[m] * pc[m];
                z[m] = fmaf(fmaf(-q, dg[m], r[m]), pc[m], q);
            }
        }
        if (MIC) {
            float w = 0.f;
#pragma unroll
            for (int t = 0; t < 22; ++t) {
                const int m = t & 7;
                float acc = z[m] + w;
                acc = fmaf(row_shift<kRowShr1>(w), in0, acc);
                acc = fmaf(lane_up8(w), jn0, acc);
                const float q = acc * pc[m];
                z[m] = lanes_or(wide_lanes(t), q, z[m]);
                w = lanes_or(wide_lanes(t), q * pc[m], 0.f);
            }
            float u = 0.f;
#pragma unroll
            for (int t = 21; t >= 0; --t) {
                const int m = t & 7;
                const float f = pc[m];
                float acc = fmaf(f, u, z[m]);
                acc = fmaf(f, row_shift<kRowShl1>(u) * in7, acc);
                acc = fmaf(f, lane_down8(u) * jn7, acc);
                const float x = acc * f;
                z[m] = lanes_or(wide_lanes(t), x, z[m]);
                u = lanes_or(wide_lanes(t), x, 0.f);
            }
        }
        __builtin_amdgcn_raw_buffer_store_b128(pack4(z[0], z[1], z[2], z[3]), faces, outX, 0, kAgent);
        __builtin_amdgcn_raw_buffer_store_b128(pack4(z[4], z[5], z[6], z[7]), faces, outX + 16u, 0, kAgent);
        __builtin_amdgcn_raw_buffer_store_b128(pack4(z[0], z[1], z[2], z[3]), faces, outY, 0, kAgent);
        __builtin_amdgcn_raw_buffer_store_b128(pack4(z[4], z[5], z[6], z[7]), faces, outY + 16u, 0, kAgent);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(plane_value<0>(z, 0, d0)), faces, outZ, 0, kAgent);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(plane_value<7>(z, 0, d0)), faces, outZ + 256u, 0, kAgent);
        double srz = 0.0, srr = 0.0;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            srz += (double)r[m] * (double)z[m];
            srr += (double)r[m] * (double)r[m];
        }
        double rz, rr;
        if (!grid_sum<2>(sh, srz, srr, c, words, c.number + 2u * it, rz, rr)) {
            failed = true;
            break;
        }
        if (rr <= c.thr2 || !(rr == rr) || it == c.limit) break;  // the same decision everywhere
        const float beta = it == 0u ? 0.f : rzOld != 0.0 ? (float)(rz / rzOld) : 0.f;
        rzOld = rz;
        v4u h4[4];
        uint32_t h1[2];
        h4[0] = __builtin_amdgcn_raw_buffer_load_b128(faces, inX, 0, kAgent);
        h4[1] = __builtin_amdgcn_raw_buffer_load_b128(faces, inX + 16u, 0, kAgent);
        h4[2] = __builtin_amdgcn_raw_buffer_load_b128(faces, inY, 0, kAgent);
        h4[3] = __builtin_amdgcn_raw_buffer_load_b128(faces, inY + 16u, 0, kAgent);
        h1[0] = __builtin_amdgcn_raw_buffer_load_b32(faces, inZ0, 0, kAgent);
        h1[1] = __builtin_amdgcn_raw_buffer_load_b32(faces, inZ1, 0, kAgent);
#pragma unroll
        for (int m = 0; m < 8; ++m) p[m] = fmaf(beta, p[m], z[m]);
        s_p[0] = make_float4(p[0], p[1], p[2], p[3]);
        s_p[1] = make_float4(p[4], p[5], p[6], p[7]);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const v4u hx = h4[m >> 2], hy = h4[2 + (m >> 2)];
            xh[m] = fmaf(beta, xh[m], __uint_as_float(hx[m & 3]));
            yh[m] = fmaf(beta, yh[m], __uint_as_float(hy[m & 3]));
        }
        zl = fmaf(beta, zl, __uint_as_float(h1[0]));
        zh = fmaf(beta, zh, __uint_as_float(h1[1]));
        if (j == 0u || j == 7u) {
            float4* o = s_p + (j == 0u ? -16 : 16);
            o[0] = make_float4(yh[0], yh[1], yh[2], yh[3]);
            o[1] = make_float4(yh[4], yh[5], yh[6], yh[7]);
        }
        wave_lds_order();
        const float4 a0 = s_p[-16], a1 = s_p[-15], b0 = s_p[16], b1 = s_p[17];
        const float ym[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        const float yp[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
        double spq = 0.0;
        float q[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int lo = (m + 7) & 7, hi = (m + 1) & 7;
            float s = dg[m] * p[m];
            s -= lanes_or(0x0101010101010101ull, xh[lo], row_shift<kRowShr1>(p[lo]));
            s -= lanes_or(0x8080808080808080ull, xh[hi], row_shift<kRowShl1>(p[hi]));
            s -= ym[lo];
            s -= yp[hi];
            s -= lanes_or(wide_plane(m, 0), zl, p[lo]);
            s -= lanes_or(wide_plane(m, 7), zh, p[hi]);
            q[m] = pc[m] != 0.f ? s : 0.f;
            spq += (double)p[m] * (double)q[m];
        }
        wave_lds_order();  // the next iteration's writes come after these reads
        double pq, unused;
        if (!grid_sum<1>(sh, spq, 0.0, c, words + kSumWords, c.number + 2u * it + 1u, pq, unused)) {
            failed = true;
            break;
        }
        const float alpha = pq != 0.0 ? (float)(rz / pq) : 0.f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            e[m] = fmaf(alpha, p[m], e[m]);
            r[m] = fmaf(-alpha, q[m], r[m]);
        }
    }

    if (!failed && live) {
        double x[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) x[m] = c.x64[base + 64u * (uint32_t)((m - d0) & 7)];
#pragma unroll
        for (int m = 0; m < 8; ++m)
            if (pc[m] != 0.f) c.x64[base + 64u * (uint32_t)((m - d0) & 7)] = x[m] + (double)e[m];
    }
    if (threadIdx.x == 0) {
        if (blockIdx.x == 0) c.result[0] = it;
        if (failed) c.result[1] = c.number;
    }
}

namespace {
using ResidentKernel = void (*)(CgResident);
ResidentKernel resident_kernel(bool mic, const ResidentShape& s) {
    if (s.wide) {
        return mic ? pcg_wide_kernel<1> : pcg_wide_kernel<0>;
    }
    // up to eight waves (two per SIMD) a lane may use 256 registers, above 168
    // (which spills; the slots of nine to eleven waves have no other room)
    if (s.waves <= 8u) return mic ? pcg_resident_kernel<1, 8> : pcg_resident_kernel<0, 8>;
    return mic ? pcg_resident_kernel<1, kResidentMaxWaves> : pcg_resident_kernel<0, kResidentMaxWaves>;
}
size_t resident_lds(const ResidentShape& s) {
    return ((sizeof(Shared) + 15u) & ~(size_t)15u) + (size_t)s.waves * (s.wide ? kWideLds : kWaveLds);
}
}  // namespace

ResidentShape resident_shape(uint32_t na, bool mic) {
    ResidentShape s{};
    if (!na) return s;
    int dev = 0, cus = 0, lds = 0;
    FLIP2_HIP(hipGetDevice(&dev));
    FLIP2_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    FLIP2_HIP(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const uint32_t most = std::min<uint32_t>(256u, (uint32_t)cus);
    // One slot per wave as long as the CUs hold the waves with the registers
    // they need (per iteration, four slots per wave -> one: 960 slots Jacobi
    // 7.3 -> 5.5 us, 1370 slots 7.3 -> 5.9 and MIC(0) 10.2 -> 9.2, 2508 slots
    // Jacobi 8.0 -> 7.4).  With MIC(0) only up to two waves per SIMD: beyond,
    // its sweeps, which keep four columns per lane busy in the other layout
    // and one here, are bound by instruction issue (2383 slots 9.9 against
    // 10.3 us).  At least four waves, one per SIMD: an iteration of a wave is
    // a chain of instructions, and fewer workgroups have fewer sums.
    s.wide = na <= (mic ? 8u : kWideMaxWaves) * most;
    const uint32_t all = s.wide ? na : ceil_div(na, kRowSlots);
    s.waves = std::max(4u, ceil_div(all, most));
    if ((!s.wide && s.waves > (uint32_t)kResidentMaxWaves) || resident_lds(s) > (size_t)lds) return s;
    int per = 0;
    FLIP2_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, resident_kernel(mic, s), 64 * (int)s.waves,
                                                           resident_lds(s)));
    if (per >= 1) s.groups = ceil_div(all, s.waves);
    return s;
}

size_t resident_words() { return 2u * kSumWords; }
size_t resident_face_floats(uint32_t na) { return (size_t)na * kFaceFloats; }

std::mutex& resident_mutex(int device) {
    static std::mutex m[64];
    return m[device & 63];
}

void launch_pcg_resident(const CgResident& c, const ResidentShape& shape, bool mic, hipStream_t s) {
    FLIP2_REQUIRE(c.na && c.na <= (1u << 20) && shape.groups && c.groups == shape.groups && shape.groups <= 256u &&
                      (uint64_t)shape.groups * shape.waves * (shape.wide ? 1u : kRowSlots) >= c.na,
                  kErrArgument, "resident PCG: the grid does not hold the slots");
    const size_t lds = resident_lds(shape);
    const ResidentKernel pcg_resident_kernel = resident_kernel(mic, shape);
    CgResident k = c;
    // The words arrive after the latency of a write and a read.  Reads that
    // come earlier find nothing and hold up the others' writes and faces, the
    // more workgroups the worse; a pause that is too long is paid in full.
    // Per iteration without / with a pause (64 clocks each): 12 slots 4.66 ->
    // 4.58 us with 4 (5.25 with 18), 160 slots 4.70 -> 4.28 with 10 (4.69 with
    // 18), 960 slots 7.72 -> 5.47 with 18 (5.96 with 10), 9196 slots MIC(0)
    // 25.0 -> 22.6 with 36 (22.7 with 40, 24.2 with 18).
    k.pause = shape.groups <= 16u ? 4u : shape.groups <= 64u ? 10u : shape.waves <= 8u || shape.wide ? 18u : 36u;
    // (a timer knows both layouts' kernels by this variable's name)
    FLIP2_KERNEL(pcg_resident_kernel, dim3(shape.groups), dim3(64 * shape.waves), lds, s, k);
    FLIP2_LAUNCH_CHECK();
}

}  // namespace ns
}  // namespace flip2
