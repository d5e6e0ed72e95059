// W4A8 tile GEMM for CDNA4 int8 MFMA on the re-laid-out int4 weight.
//
//   sum_g  = sum_{k in group g} xq[m,k] * (code(n,k) - 8)     int32, exact
//   total  = fma((float)sum_g, ws[n,g], total)                 g = 0,1,.. from 0.f
//   y[m,n] = bf16(total * xs[m])
//
// Same bits as the W4A8 GEMV for every m: the integer part is exact and the fp32 part is the one chain
// over the groups in ascending order.
//
// What bounds it.  Per 128 k a 64 x 64 piece of the output needs 512 clocks of matrix pipe and, per group, one
// convert and one multiply-add for each of its elements: 128 vector instructions a wavefront, which mostly run
// beside the MFMAs of the SIMD's other wavefront.  The earlier two-stage kernel (widened weight through LDS: a
// write, a barrier and a read more per step) took 1.7 us for two 128 x 128 tiles of a CU; this one takes
// 1.3.  Pieces taken out of a copy (1024 x 51200 x 5120, 326 us): MFMAs alone 160 us (3.4 POP/s -- what the
// clock leaves of the peak under random operands), + flush 233, operand requests 90, LDS reads 15..40,
// widening 20: they add up instead of hiding, as for a launch bound by power, so what helps is fewer bytes moved
// and fewer instructions, not deeper prefetch (four to six stages, double-buffered fragments and 32x32x32 MFMAs
// all measured the same or slower; under random operands 16x16x64 sustains 12 % more than 32x32x32).
//
// Design:
//   - activations and the *packed* weight go global -> LDS directly (buffer_load_dwordx4 ... lds; rows past the
//     matrix and steps past K read zeros), NST steps in flight, one barrier per step;
//   - a wavefront reads packed rows in the MFMA arrangement and widens them itself, three vector instructions
//     per eight codes: 16 (code - 8) is the code with its top bit flipped in the high nibble of a byte.  The
//     sums are 16 times too large, exactly, and the flush multiplies by scale / 16, which is exact for scales from
//     2^-122 up.  The encoder's are above 1e-9; a wavefront that meets a smaller one (a running minimum, 0..2 % of
//     the launch: 1024 x 51200 x 5120 344 -> 348 us; a compare and branch per flush took 5 % and made 128 x 160
//     spill) forms its results anew at the end, element by element;
//   - the output is walked column tile by column tile: while column j multiplies, the sums of column j - 1 are
//     flushed and column j + 1 is widened, in slots of one MFMA and the vector instructions beside it (left to
//     itself the compiler clumps them, 6 % slower);
//   - the activation is the MFMA row operand and the weight the column operand: a lane owns one n per tile, so a
//     tile needs one scale per lane and group, fetched four steps at a time straight into registers (a scale a
//     step is a gather of one cache line per row).
#include "common.hpp"
#include "gemm_tiles.hpp"

#include <cmath>
#include <type_traits>

namespace {

using namespace cmi;

constexpr int BK = 128;  // k of a step

struct Args {
    const int8_t *xq;
    const uint8_t *w4;
    const float *xs;
    const float *ws;  // [N, G]
    uint16_t *y;
    int M, N, K, G;
    int tiles_m, tiles_n;
};

typedef __attribute__((address_space(3))) void *lds_ptr_t;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int v2i32 __attribute__((ext_vector_type(2)));

template <int WM, int WN, int TM, int TN, int NST>
struct Cfg {
    static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
    static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;  // WM x WN wavefronts of 16 TM x 16 TN
    static constexpr int X_BYTES = BM * BK, P_BYTES = BN * BK / 2, STAGE = X_BYTES + P_BYTES;
    static constexpr int XL = (BM / 8 + WAVES - 1) / WAVES, PL = (BN / 16 + WAVES - 1) / WAVES;  // requests per wavefront
    static constexpr int LOADS = XL + PL;
    static constexpr int YPITCH = 2 * BN + 16;  // bytes per row of the parked result
    static constexpr int LDS_BYTES = NST * STAGE > BM * YPITCH ? NST * STAGE : BM * YPITCH;
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// One element's sum over the groups, from memory: the statement at the head of this file as it stands.  A word of the
// packed weight holds k 0..3 in its low nibbles and k 4..7 in its high ones.
template <int LG>
__device__ __forceinline__ float total_of(const Args &a, int m, int n) {
    const int8_t *x = a.xq + (size_t)m * a.K;
    const uint8_t *w = a.w4 + (size_t)n * (a.K / 2);
    float total = 0.f;
    for (int g = 0; g < a.G; ++g) {
        int sum = 0;
        for (int k = g * (32 << LG); k < (g + 1) * (32 << LG); ++k) {
            const int b = k % 8;
            sum += x[k] * (((w[k / 8 * 4 + b % 4] >> (b / 4 * 4)) & 15) - 8);
        }
        total = fmaf((float)sum, a.ws[(size_t)n * a.G + g], total);
    }
    return total;
}

// y[m,n] = bf16(total * xs[m]) of a wavefront's TM x TN tiles of 16 x 16 at (mw, nw) of its workgroup's, into LDS.
// inexact: lanes that met a scale below 2^-122; the wavefront's results are formed anew.
template <int TM, int TN, int YPITCH, int LG>
__device__ __forceinline__ void park_results(const Args &a, const float (&total)[TM][TN][4], uint64_t inexact, uint16_t *park, int m0,
                                             int n0, int mw, int nw, int lane) {
    const int fr = lane & 15, fc = lane >> 4;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int ml = mw + i * 16 + fc * 4 + r;
            const float xm = a.xs[min(m0 + ml, a.M - 1)];
#pragma unroll
            for (int j = 0; j < TN; ++j) park[ml * (YPITCH / 2) + nw + j * 16 + fr] = (uint16_t)f32_to_bf16_bits(total[i][j][r] * xm);
        }
    if (inexact)
        for (int e = lane; e < 16 * TM * 16 * TN; e += 64) {
            const int ml = mw + e / (16 * TN), nl = nw + e % (16 * TN);
            if (m0 + ml < a.M && n0 + nl < a.N)
                park[ml * (YPITCH / 2) + nl] = (uint16_t)f32_to_bf16_bits(total_of<LG>(a, m0 + ml, n0 + nl) * a.xs[m0 + ml]);
        }
}

// The results of a BM x BN tile, parked in LDS in rows of YPITCH bytes, leave as whole 16-byte pieces of rows.
template <int BM, int BN, int YPITCH, int THREADS>
__device__ __forceinline__ void store_parked(const Args &a, const uint16_t *park, int m0, int n0) {
    const int rows = min(a.M - m0, BM), cols = min(a.N - n0, BN);
    if (a.N % 8 == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0) {
        constexpr int CH = BN / 8;
        for (int t = threadIdx.x; t < rows * CH; t += THREADS) {
            const int m = t / CH, c = t - m * CH;
            const uint4 v = *reinterpret_cast<const uint4 *>(reinterpret_cast<const int8_t *>(park) + m * YPITCH + c * 16);
            uint16_t *dst = a.y + (size_t)(m0 + m) * a.N + n0 + c * 8;
            if (c * 8 + 8 <= cols) {
                *reinterpret_cast<uint4 *>(dst) = v;
            } else {
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (c * 8 + k < cols) dst[k] = (uint16_t)(w[k / 2] >> (16 * (k & 1)));
            }
        }
    } else {  // rows that are not 16-byte aligned: element by element, a wavefront's stores side by side
        for (int t = threadIdx.x; t < rows * BN; t += THREADS) {
            const int m = t / BN, c = t - m * BN;
            if (c < cols) a.y[(size_t)(m0 + m) * a.N + n0 + c] = park[m * (YPITCH / 2) + c];
        }
    }
}

// LG: log2(group size / 32).  2: a step is a group.  3: a group is two steps, the first one's sums are kept.  1: a
// step holds two groups, one MFMA each.
template <int WM, int WN, int TM, int TN, int NST, int LG>
__global__ void __launch_bounds__(64 * WM * WN, 2) gemm_w4a8_tile_kernel(const Args a) {
    using C = Cfg<WM, WN, TM, TN, NST>;
    extern __shared__ __align__(16) int8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, wm = wave / WN;
    int tm, tn;
    banded_tile(a.tiles_m, a.tiles_n, blockIdx.x, tm, tn);
    const int m0 = tm * C::BM, n0 = tn * C::BN;

    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t *>(a.xq) + (size_t)m0 * a.K, 0, min(a.M - m0, C::BM) * a.K, 0x00020000);
    const __amdgpu_buffer_rsrc_t pres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(a.w4) + (size_t)n0 * (a.K / 2), 0, min(a.N - n0, C::BN) * (a.K / 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.ws) + (size_t)n0 * a.G, 0, min(a.N - n0, C::BN) * a.G * 4, 0x00020000);

    // Requests of a step.  Activations: 8 rows x 128 B each, chunk index XOR (row / 2) % 8; packed weight: 16
    // rows x 64 B each, piece index XOR (row / 4) % 4.
    const int xoff = (lane >> 3) * a.K + ((lane & 7) ^ (lane >> 4)) * 16;
    const int poff = (lane >> 2) * (a.K / 2) + ((lane & 3) ^ ((lane >> 4) & 3)) * 16;
    auto issue = [&](int slot, int ks) {
        int8_t *base = lds + slot * C::STAGE;
#pragma unroll
        for (int h = 0; h < C::XL; ++h) {
            // rows 8g .. 8g + 7: (row / 2) % 8 = 4 (g % 2) + lane / 16
            const int g = min(C::XL * wave + h, C::BM / 8 - 1);  // past the last: the last again, same bytes
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (lds_ptr_t)(base + g * 1024), 16, xoff ^ ((g & 1) * 64),
                                                     ks * BK + g * 8 * a.K, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < C::PL; ++h) {
            const int p = min(C::WAVES * h + wave, C::BN / 16 - 1);  // past the last: the last again, same bytes
            __builtin_amdgcn_raw_ptr_buffer_load_lds(pres, (lds_ptr_t)(base + C::X_BYTES + p * 1024), 16, poff,
                                                     ks * (BK / 2) + p * 16 * (a.K / 2), 0, 0);
        }
    };

    // Fragments of 16x16x64: lane l holds row l % 16 and 16 of an MFMA's 64 k, the same ones of both operands.  With
    // c = l / 16, MFMA e of a step takes the e-th half of piece c of the packed row and 16-byte chunk 2c + e of the
    // activation row; with groups of 64 it has to stay inside one: half c % 2 of piece 2e + c / 2, chunk 4e + c.
    const int fr = lane & 15, fc = lane >> 4, fsw = (fr >> 1) & 7;
    int xf[2], pf[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        xf[e] = (wm * 16 * TM + fr) * BK + ((LG == 1 ? 4 * e + fc : 2 * fc + e) ^ fsw) * 16;
        const int piece = LG == 1 ? 2 * e + (fc >> 1) : fc;
        pf[e] = C::X_BYTES + (wn * 16 * TN + fr) * 64 + (piece ^ ((fr >> 2) & 3)) * 16 + (LG == 1 ? (fc & 1) : e) * 8;
    }
    const int soff = (wn * 16 * TN + fr) * a.G * 4;

    v4i32 x[TM][2];
    v4i32 packed[TN];  // words 0, 1 belong to MFMA 0 and words 2, 3 to MFMA 1
    auto read_x = [&](int slot, int i, int e) {
        return *reinterpret_cast<const v4i32 *>(lds + slot * C::STAGE + xf[e] + i * 16 * BK);
    };
    auto read_p = [&](int slot, int j) {
        const int8_t *p = lds + slot * C::STAGE + j * 16 * 64;
        if constexpr (LG != 1) return *reinterpret_cast<const v4i32 *>(p + pf[0]);
        const v2i32 a0 = *reinterpret_cast<const v2i32 *>(p + pf[0]), a1 = *reinterpret_cast<const v2i32 *>(p + pf[1]);
        return v4i32{a0.x, a0.y, a1.x, a1.y};
    };
    // scales of the groups of four steps, the next four requested a chunk ahead: four groups (LG 2), two (LG 3; two
    // more come along) or eight (LG 1)
    constexpr int SV = LG == 1 ? 2 : 1;
    f32x4 sc[TN][SV], sc_next[TN][SV];
    auto load_s = [&](int j, int v, int chunk) {
        const int first = LG == 3 ? chunk * 8 : chunk * 16 * SV + v * 16;
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(sres, soff, first + j * 16 * a.G * 4, 0));
    };

    // Four codes as int8 16 (code - 8): the code's top bit flipped, moved to the high nibble.  Low nibbles of a
    // word are k 0..3, high nibbles k 4..7.
    auto nibbles = [](int word, int high) {
        return (int)(((high ? (uint32_t)word : (uint32_t)word << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
    };
    v4i32 w[2];  // the column about to be multiplied, widened

    float total[TM][TN][4];
    constexpr int PG = LG == 1 ? 2 : 1;  // groups a step closes in a column
    v4i32 pend[PG][TM];                  // the latest closed column's sums, flushed under the next column's MFMAs
    float pend_scale[PG];
    // The smallest magnitude of a scale so far but zero, as 2 * bits - 1, and the lanes where it was below 2^-122.
    constexpr uint32_t TINY = 2 * (5u << 23) - 1;
    uint32_t least = ~0u;
    uint64_t inexact = 0;
    v4i32 part[LG == 3 ? TN : 1][TM];    // LG 3: sums of the first half of a group
#pragma unroll
    for (int g = 0; g < PG; ++g) {
        pend_scale[g] = 0.f;
#pragma unroll
        for (int i = 0; i < TM; ++i) pend[g][i] = v4i32{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) total[i][j][r] = 0.f;

    const int ksteps = a.K / BK;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < SV; ++v) sc[j][v] = load_s(j, v, 0);
#pragma unroll
    for (int s = 0; s < NST; ++s) issue(s, s);
    wait_vmcnt<(NST - 1) * C::LOADS>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) x[i][e] = read_x(0, i, e);
#pragma unroll
    for (int j = 0; j < TN; ++j) packed[j] = read_p(0, j);
#pragma unroll
    for (int h = 0; h < 8; ++h) w[h / 4][h % 4] = nibbles(packed[0][h / 2], h & 1);

    // Step ks enters with its activations and packed weights in registers (requested from LDS during step ks - 1), its
    // first column widened.  Behind the barrier stage ks + 1 is complete and the slot of stage ks, which every
    // wavefront has read, takes the requests of stage ks + NST.
    int slot = 0;
    auto step = [&](auto u_tag, int ks) {
        constexpr int U = decltype(u_tag)::value;  // place of the step in its chunk of four
        constexpr bool OPENS = LG != 3 || (U & 1) == 0, CLOSES = LG != 3 || (U & 1) == 1;
        const int next = slot + 1 == NST ? 0 : slot + 1;
        // in flight behind stage ks + 1: NST - 2 stages and, from the step after they were requested until they are
        // older than that stage, the chunk's scales
        wait_vmcnt<(NST - 2) * C::LOADS + (U >= 1 && U < NST ? TN * SV : 0)>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(slot, ks + NST);
        if constexpr (U == 0) {
            asm volatile("" ::: "memory");  // behind the stage's requests: the counted waits rely on it
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < SV; ++v) sc_next[j][v] = load_s(j, v, (ks >> 2) + 1);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int jp = j ? j - 1 : TN - 1, jn = j + 1 < TN ? j + 1 : 0;
            // whether pend holds sums: the column before closed its group (column 0 follows the step before)
            const bool flush = LG != 3 || (j ? CLOSES : !CLOSES);
            const v4i32 zero = {0, 0, 0, 0};
            v4i32 acc[PG][TM], wide[2];
            constexpr int SLOTS = 2 * TM;
#pragma unroll
            for (int t = 0; t < SLOTS; ++t) {
                const int i = t % TM, e = t / TM, g = PG == 2 ? e : 0;
                const v4i32 from = PG == 1 && e ? acc[0][i] : OPENS ? zero : part[LG == 3 ? j : 0][i];
                acc[g][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[i][e], w[e], from, 0, 0, 0);
                // the step's last use of these activations: the next step's take their registers
                if (j == TN - 1) x[i][e] = read_x(next, i, e);
                if (t == 0) packed[j] = read_p(next, j);
                if (flush) {
#pragma unroll
                    for (int f = 4 * TM * PG * t / SLOTS; f < 4 * TM * PG * (t + 1) / SLOTS; ++f) {
                        const int fg = f / (4 * TM), fi = f / 4 % TM, r = f % 4;  // groups ascending
                        total[fi][jp][r] = fmaf((float)pend[fg][fi][r], pend_scale[fg], total[fi][jp][r]);
                    }
                }
#pragma unroll
                for (int h = 8 * t / SLOTS; h < 8 * (t + 1) / SLOTS; ++h) wide[h / 4][h % 4] = nibbles(packed[jn][h / 2], h & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!CLOSES) {
#pragma unroll
                for (int i = 0; i < TM; ++i) part[LG == 3 ? j : 0][i] = acc[0][i];
            } else {
#pragma unroll
                for (int g = 0; g < PG; ++g) {
#pragma unroll
                    for (int i = 0; i < TM; ++i) pend[g][i] = acc[g][i];
                    const int at = LG == 3 ? U >> 1 : LG == 1 ? 2 * U + g : U;
                    pend_scale[g] = sc[j][at / 4][at % 4] * 0.0625f;
                }
            }
            w[0] = wide[0];
            w[1] = wide[1];
        }
        slot = next;
    };
    for (int c = 0; 4 * c < ksteps; ++c) {
        if constexpr (LG == 3) least = ~0u;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < SV; ++v)
#pragma unroll
                for (int i = 0; i < (LG == 3 ? 2 : 4); ++i) least = min(least, 2 * __float_as_uint(sc[j][v][i]) - 1);
        if constexpr (LG == 3) inexact |= __builtin_amdgcn_ballot_w64(least < TINY);  // no vector register to spare
        step(std::integral_constant<int, 0>{}, 4 * c);
        if (4 * c + 1 < ksteps) step(std::integral_constant<int, 1>{}, 4 * c + 1);
        if (4 * c + 2 < ksteps) step(std::integral_constant<int, 2>{}, 4 * c + 2);
        if (4 * c + 3 < ksteps) step(std::integral_constant<int, 3>{}, 4 * c + 3);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < SV; ++v) sc[j][v] = sc_next[j][v];
    }
#pragma unroll
    for (int g = 0; g < PG; ++g)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                total[i][TN - 1][r] = fmaf((float)pend[g][i][r], pend_scale[g], total[i][TN - 1][r]);
    if constexpr (LG != 3) inexact = __builtin_amdgcn_ballot_w64(least < TINY);
    wait_vmcnt<0>();  // requests past the last step (they read zeros or the next rows)

    // y[m,n] = bf16(total * xs[m]), parked in LDS so that whole 16-byte pieces of rows leave
    __syncthreads();
    uint16_t *park = reinterpret_cast<uint16_t *>(lds);
    park_results<TM, TN, C::YPITCH, LG>(a, total, inexact, park, m0, n0, wm * 16 * TM, wn * 16 * TN, lane);
    __syncthreads();
    store_parked<C::BM, C::BN, C::YPITCH, C::THREADS>(a, park, m0, n0);
}

// ---------------------------------------------------------------------------
// Few tiles, or few rows (2 .. several hundred): a step of four groups.
//
// What bounds it.  With a tile or two per CU the kernel above is a chain of K / 128 steps of 0.27 us whatever is in them:
// the barrier, the trip to LDS for the next fragments and one wavefront per SIMD with 40 vector instructions to issue.
// Here a barrier buys four groups: 0.6 .. 0.9 us per step of 512 k, of which, taken apart for 100 rows of 9728 -> 2560 (32
// x 64 tiles, 20.1 us in all with the quantiser), the operands' way from L2 to LDS takes 10 us (62 B/ns per CU of the 75 that
// such loads reach) and fragments and arithmetic 10, half of it hidden under the other.
//
// A row's 512 (activations) or 256 (packed weight) bytes of a step are requested together and lie together in LDS, 16-byte
// piece index XOR row % 16; the step's scales come the same way.  A wavefront reads its fragments of all four groups behind
// the barrier and has no others in flight (reading them a step ahead measured 2..5 % slower: registers and the same
// LDS time).  NST = 2 stages leave room for two or three workgroups per CU, which hide each other's trips; 3 or 4 are
// for launches of one per CU.  A wavefront on 16 rows at a time widens every code again for the next 16: the 32- and 48-row
// tiles of wavefronts side by side do it once.  Sharing K among wavefronts that hand their sums over through LDS was built
// first and took 32 us for that shape: operands straight into registers in the MFMA arrangement come at 16 bytes a clock.
//
// Groups of 64 and 256: a stage is eight or two groups; 64 close one after each MFMA (operand pieces as above), 256 after
// every second 128.
//
// ONCE: a single tile of rows, so that every weight byte is read by one workgroup and need not stay in the caches.
//
// Cold weights, with the quantiser in front (2.5 us at 16 x 4096, 4.7 at 100 x 9728): 100 rows of 9728 -> 2560 28.7 -> 20.1 us, 40
// rows 23.3 -> 16.3, 200 rows 33.7 -> 26.4; 100 rows of 4096 -> 2560 15.1 -> 11.6; 40 rows of 25600 -> 5120 59.5 -> 38.4; 16 rows of
// 2560 -> 151936 54.6 -> 51.3, of 4096 -> 12288 14.6 -> 12.9 (both against the matrix-pipe GEMV); groups of 256, 100 rows of 9728 ->
// 2560 28.4 -> 19.8, 24 rows of 14336 -> 4096 32.1 -> 21.0.
constexpr int NT = 2;  // cache policy of a load: nontemporal
constexpr int U = 4, X_ROW = U * BK, P_ROW = U * BK / 2;  // 128s of a stage; bytes of a row in it: 512 and 256

template <int WM, int WN, int TM, int TN, int NST, int LG>
struct DeepCfg {
    static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
    static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    static constexpr int X_BYTES = BM * X_ROW, P_BYTES = BN * P_ROW;
    static constexpr int SU = (U * 4) >> LG;  // groups of a stage: 8, 4, 2
    static constexpr int S_BYTES = BN * SU * 4, STAGE = X_BYTES + P_BYTES + S_BYTES;
    static constexpr int XL = X_BYTES / 1024 / WAVES, PL = P_BYTES / 1024 / WAVES;  // requests per wavefront and stage
    static constexpr int SL = (BN * SU / 64 + WAVES - 1) / WAVES;
    static constexpr int LOADS = XL + PL + SL;
    static constexpr int YPITCH = 2 * BN + 16;
    static constexpr int LDS_BYTES = NST * STAGE;
    static_assert(BM % (2 * WAVES) == 0 && BN % (4 * WAVES) == 0, "whole requests per wavefront");
    static_assert(BM * YPITCH <= LDS_BYTES, "result does not fit");
};

template <int WM, int WN, int TM, int TN, int NST, int LG, bool ONCE>
__global__ void __launch_bounds__(64 * WM * WN, 2) gemm_w4a8_deep_kernel(const Args a) {
    using C = DeepCfg<WM, WN, TM, TN, NST, LG>;
    extern __shared__ __align__(16) int8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, wm = wave / WN;
    int tm, tn;
    banded_tile(a.tiles_m, a.tiles_n, blockIdx.x, tm, tn);
    const int m0 = tm * C::BM, n0 = tn * C::BN;

    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t *>(a.xq) + (size_t)m0 * a.K, 0, min(a.M - m0, C::BM) * a.K, 0x00020000);
    const __amdgpu_buffer_rsrc_t pres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(a.w4) + (size_t)n0 * (a.K / 2), 0, min(a.N - n0, C::BN) * (a.K / 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.ws) + (size_t)n0 * a.G, 0, min(a.N - n0, C::BN) * a.G * 4, 0x00020000);

    // Requests of a stage: two rows x 512 B of activations, four rows x 256 B of packed weight each, 16-byte piece index
    // XOR row % 16; then the scales, [column][SU].
    int xoff[C::XL], poff[C::PL];
#pragma unroll
    for (int h = 0; h < C::XL; ++h) xoff[h] = (lane >> 5) * a.K + ((lane & 31) ^ ((2 * (C::XL * wave + h) + (lane >> 5)) & 15)) * 16;
#pragma unroll
    for (int h = 0; h < C::PL; ++h) poff[h] = (lane >> 4) * (a.K / 2) + ((lane & 15) ^ ((4 * (C::PL * wave + h) + (lane >> 4)) & 15)) * 16;
    const int soff = (lane / C::SU) * a.G * 4 + (lane % C::SU) * 4;
    auto issue = [&](int slot, int stage) {
        int8_t *base = lds + slot * C::STAGE;
#pragma unroll
        for (int h = 0; h < C::PL; ++h) {
            const int q = C::PL * wave + h, off = poff[h];
            __builtin_amdgcn_raw_ptr_buffer_load_lds(pres, (lds_ptr_t)(base + C::X_BYTES + q * 1024), 16, off,
                                                     stage * P_ROW + q * 4 * (a.K / 2), 0, ONCE ? NT : 0);
        }
#pragma unroll
        for (int h = 0; h < C::XL; ++h) {
            const int q = C::XL * wave + h, off = xoff[h];
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (lds_ptr_t)(base + q * 1024), 16, off, stage * X_ROW + q * 2 * a.K, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < C::SL; ++h) {
            const int r = min(C::SL * wave + h, C::BN * C::SU / 64 - 1);  // past the last: the last again, same bytes
            __builtin_amdgcn_raw_ptr_buffer_load_lds(sres, (lds_ptr_t)(base + C::X_BYTES + C::P_BYTES + r * 256), 4, soff,
                                                     stage * C::SU * 4 + r * (64 / C::SU) * a.G * 4, 0, 0);
        }
    };
    // a lane's pieces: row fr of a tile, piece u * 4 + fc of the packed row and pieces u * 8 + 2 fc + e of the activations;
    // with groups of 64, half fc % 2 of piece u * 4 + 2 e + fc / 2 and piece u * 8 + 4 e + fc (as above)
    const int fr = lane & 15, fc = lane >> 4;
    int xf[2][2], pf[U][LG == 1 ? 2 : 1];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 2; ++e) xf[h][e] = (wm * 16 * TM + fr) * X_ROW + ((8 * h + (LG == 1 ? 4 * e + fc : 2 * fc + e)) ^ fr) * 16;  // u = h, h + 2: 256 B on
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int row = C::X_BYTES + (wn * 16 * TN + fr) * P_ROW;
        if constexpr (LG != 1) {
            pf[u][0] = row + ((4 * u + fc) ^ fr) * 16;
        } else {
#pragma unroll
            for (int e = 0; e < 2; ++e) pf[u][e] = row + ((4 * u + 2 * e + (fc >> 1)) ^ fr) * 16 + (fc & 1) * 8;
        }
    }
    const int sf = C::X_BYTES + C::P_BYTES + (wn * 16 * TN + fr) * (C::SU * 4);
    auto read_p = [&](const int8_t *base, int u, int j) {
        const int8_t *row = base + j * 16 * P_ROW;
        if constexpr (LG != 1) {
            return *reinterpret_cast<const v4i32 *>(row + pf[u][0]);
        } else {
            const v2i32 p0 = *reinterpret_cast<const v2i32 *>(row + pf[u][0]), p1 = *reinterpret_cast<const v2i32 *>(row + pf[u][1]);
            return v4i32{p0.x, p0.y, p1.x, p1.y};
        }
    };
    auto nibbles = [](int word, int high) {
        return (int)(((high ? (uint32_t)word : (uint32_t)word << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
    };

    float total[TM][TN][4];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) total[i][j][r] = 0.f;
    constexpr uint32_t TINY = 2 * (5u << 23) - 1;  // as above
    uint32_t least = ~0u;

#pragma unroll
    for (int s = 0; s < NST - 1; ++s) issue(s, s);
    const int ksteps = a.K / BK;
    int slot = 0;
    auto stage = [&](auto whole_tag, int s) {
        constexpr bool WHOLE = decltype(whole_tag)::value;
        wait_vmcnt<(NST - 2) * C::LOADS>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // the slot that the stage before was read from
        issue(slot == 0 ? NST - 1 : slot - 1, s + NST - 1);
        const int8_t *base = lds + slot * C::STAGE;
        typedef float scales_t __attribute__((ext_vector_type(C::SU)));
        scales_t sc[TN];
        v4i32 x[U][TM][2], p[U][TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) sc[j] = *reinterpret_cast<const scales_t *>(base + sf + j * 16 * C::SU * 4);
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int j = 0; j < TN; ++j) p[u][j] = read_p(base, u, j);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    x[u][i][e] = *reinterpret_cast<const v4i32 *>(base + xf[u & 1][e] + (u >> 1) * 256 + i * 16 * X_ROW);
            __builtin_amdgcn_sched_barrier(0);
        }
        v4i32 acc[TN][TM];  // (groups of 256: kept over two u)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!WHOLE && s * U + u >= ksteps) break;  // uniform
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                v4i32 w[2];
#pragma unroll
                for (int h = 0; h < 8; ++h) w[h / 4][h % 4] = nibbles(p[u][j][h / 2], h & 1);
                const auto flush = [&](int g) {
                    least = min(least, 2 * __float_as_uint(sc[j][g]) - 1);
                    const float scale = sc[j][g] * 0.0625f;
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) total[i][j][r] = fmaf((float)acc[j][i][r], scale, total[i][j][r]);
                };
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const bool opens = LG == 1 || (e == 0 && (LG == 2 || u % 2 == 0)), closes = LG == 1 || (e == 1 && (LG == 2 || u % 2 == 1));
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        const v4i32 from = opens ? v4i32{0, 0, 0, 0} : acc[j][i];
                        acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[u][i][e], w[e], from, 0, 0, 0);
                    }
                    if (closes) flush(LG == 1 ? 2 * u + e : LG == 2 ? u : u / 2);
                }
            }
        }
        slot = slot + 1 == NST ? 0 : slot + 1;
    };
    const int whole = ksteps / U;
    for (int s = 0; s < whole; ++s) stage(std::true_type{}, s);
    if (whole * U < ksteps) stage(std::false_type{}, whole);
    const uint64_t inexact = __builtin_amdgcn_ballot_w64(least < TINY);
    wait_vmcnt<0>();
    __syncthreads();
    uint16_t *park = reinterpret_cast<uint16_t *>(lds);
    park_results<TM, TN, C::YPITCH, LG>(a, total, inexact, park, m0, n0, wm * 16 * TM, wn * 16 * TN, lane);
    __syncthreads();
    store_parked<C::BM, C::BN, C::YPITCH, C::THREADS>(a, park, m0, n0);
}

template <int WM, int WN, int TM, int TN, int NST, int LG>
int launch_deep(Args &a, hipStream_t st) {
    using C = DeepCfg<WM, WN, TM, TN, NST, LG>;
    a.tiles_m = (a.M + C::BM - 1) / C::BM;
    a.tiles_n = (a.N + C::BN - 1) / C::BN;
    // the tile's operand offsets are 32-bit
    CMI_REQUIRE((size_t)(C::BM > C::BN ? C::BM : C::BN) * (a.K + NST * X_ROW) < ((size_t)1 << 31), CMI_E_UNSUPPORTED,
                "cmi_gemm_w4a8: K=%d too long", a.K);
    static std::atomic<uint64_t> devices[2];
    const auto run = [&](auto kernel, std::atomic<uint64_t> &done) {
        if (const int rc = reserve_lds(reinterpret_cast<const void *>(kernel), C::LDS_BYTES, done, "cmi_gemm_w4a8")) return rc;
        kernel<<<dim3(a.tiles_m * a.tiles_n), dim3(C::THREADS), C::LDS_BYTES, st>>>(a);
        return check_launch("cmi_gemm_w4a8");
    };
    if (a.tiles_m == 1) return run(gemm_w4a8_deep_kernel<WM, WN, TM, TN, NST, LG, true>, devices[1]);
    if constexpr (LG != 1) return run(gemm_w4a8_deep_kernel<WM, WN, TM, TN, NST, LG, false>, devices[0]);
    return fail(CMI_E_UNSUPPORTED, "cmi_gemm_w4a8: internal dispatch");  // groups of 64: up to 16 rows (gemm_w4a8_tile_us)
}

template <int WM, int WN, int TM, int TN, int NST, int LG>
int launch(Args &a, hipStream_t st) {
    using C = Cfg<WM, WN, TM, TN, NST>;
    a.tiles_m = (a.M + C::BM - 1) / C::BM;
    a.tiles_n = (a.N + C::BN - 1) / C::BN;
    // the tile's operand offsets are 32-bit
    CMI_REQUIRE((size_t)(C::BM > C::BN ? C::BM : C::BN) * (a.K + NST * BK) < ((size_t)1 << 31), CMI_E_UNSUPPORTED,
                "cmi_gemm_w4a8: K=%d too long", a.K);
    static std::atomic<uint64_t> devices{0};
    if (const int rc = reserve_lds(reinterpret_cast<const void *>(gemm_w4a8_tile_kernel<WM, WN, TM, TN, NST, LG>), C::LDS_BYTES,
                                   devices, "cmi_gemm_w4a8"))
        return rc;
    gemm_w4a8_tile_kernel<WM, WN, TM, TN, NST, LG><<<dim3(a.tiles_m * a.tiles_n), dim3(C::THREADS), C::LDS_BYTES, st>>>(a);
    return check_launch("cmi_gemm_w4a8");
}

// The tiles (rows x columns).  Two workgroups of four wavefronts share a CU; 128 x 160 exists for the tile count
// (1024 x 5120: 256 tiles, one per CU).
// (D: of four groups a step, L with more stages)
enum Tile { T128x160, T128x128, T64x128, T64x96, T64x64, T32x64, T32x128, T16x32, D16x64, D16x64L, D32x32, D32x32L, D32x64, D32x64L, D48x64, TILES };

template <int LG>
int launch_tile(Args &a, Tile tile, hipStream_t st) {
    if constexpr (LG == 2) {
        switch (tile) {
            case T128x160: return launch<2, 2, 4, 5, 3, 2>(a, st);
            case T128x128: return launch<2, 2, 4, 4, 3, 2>(a, st);
            case T64x96: return launch<2, 2, 2, 3, 3, 2>(a, st);
            case T32x128: return launch<1, 4, 2, 2, 4, 2>(a, st);
            default: break;
        }
    }
    switch (tile) {
        case T64x128: return launch<2, 2, 2, 4, 3, LG>(a, st);
        case T64x64: return launch<2, 2, 2, 2, 4, LG>(a, st);
        case T32x64: return launch<2, 2, 1, 2, 4, LG>(a, st);
        case T16x32: return launch<1, 2, 1, 1, 4, LG>(a, st);
        case D16x64: return launch_deep<1, 4, 1, 1, 2, LG>(a, st);
        case D16x64L: return launch_deep<1, 4, 1, 1, 4, LG>(a, st);
        case D32x32: return launch_deep<2, 2, 1, 1, 2, LG>(a, st);
        case D32x32L: return launch_deep<2, 2, 1, 1, 4, LG>(a, st);
        case D32x64: return launch_deep<1, 4, 2, 1, 2, LG>(a, st);
        case D32x64L: return launch_deep<2, 4, 1, 1, 3, LG>(a, st);
        case D48x64: return launch_deep<1, 4, 3, 1, 2, LG>(a, st);
        default: return CMI_E_UNSUPPORTED;
    }
}

// Time of a tile's launch in us: fixed part, then per step a share of every tile its CU holds (an odd one of two
// costs more) and of the cold weight.  Fitted to cold-weight sweeps of every tile on sixteen layer shapes x 23
// batch sizes (17..8192 rows): the choice takes 1.5 % more than the best tile of each point, at most 18 %.
struct Cost {
    int bm, bn;
    double fixed, step, tile, odd, n;
    bool any_group;  // built for groups of 64 and 256 too
};
const Cost COSTS[D16x64] = {
    {128, 160, 6.82, 0.0000, 0.7856, 0.0163, 0.0024, false},
    {128, 128, 5.36, 0.0000, 0.6325, 0.0240, 0.0059, false},
    {64, 128, 4.18, 0.0071, 0.3823, 0.0521, 0.0376, true},
    {64, 96, 3.85, 0.0000, 0.3145, 0.0590, 0.0481, false},
    {64, 64, 3.50, 0.0000, 0.2262, 0.0434, 0.0490, true},
    {32, 64, 3.04, 0.0095, 0.1537, 0.0443, 0.0723, true},
    {32, 128, 3.44, 0.0000, 0.2513, 0.0209, 0.0682, false},
    {16, 32, 2.76, 0.0342, 0.0615, 0.0152, 0.0926, true},
};

// The same for the tiles of four groups a step: fixed part, per step a share of every tile the CU holds, of every round
// of the workgroups it can hold at a time and of the cold weight, and what a tile and a round cost beside their steps.  Fitted to
// cold-weight sweeps on fifteen layer shapes x 21 batch sizes (17..1024 rows) and twenty x five (2..16).
struct DeepCost {
    int bm, bn, per_cu, code;  // code: cmi_set_option("w4_gemm_deep"), rows x 100 + columns, one more for more stages
    double fixed, tile, round, n, tiles, rounds;
};
const DeepCost DEEP_COSTS[TILES - D16x64] = {
    {16, 64, 3, 1664, 1.84, 0.196, 0.297, 0.289, 0.41, 0.28}, {16, 64, 1, 1665, 1.40, 0.463, 0.0, 0.219, 0.0, 1.57},
    {32, 32, 3, 3232, 1.84, 0.198, 0.273, 0.222, 0.28, 0.52}, {32, 32, 1, 3233, 1.47, 0.452, 0.0, 0.121, 0.0, 1.53},
    {32, 64, 2, 3264, 1.64, 0.266, 0.412, 0.203, 0.31, 0.93}, {32, 64, 1, 3265, 1.41, 0.420, 0.188, 0.165, 0.0, 1.65},
    {48, 64, 1, 4864, 1.37, 0.865, 0.0, 0.180, 0.0, 1.88},
};

// Both for groups of 256, beyond 16 rows: they flush half as often, which shortens the steps of the wide tiles of one 128 more than the
// others.  Fitted to sweeps of 52 layer shapes x 16 batch sizes (17..1024 rows, rows quantised in front, every weight cold).
constexpr int ANY_GROUP = 4;
const struct { Tile tile; Cost cost; } COSTS_256[ANY_GROUP] = {
    {T64x128, {64, 128, 4.7938, 0.0351, 0.3903, 0.0588, 0.0133, true}}, {T64x64, {64, 64, 3.9387, 0.0301, 0.2420, 0.0552, 0.0144, true}},
    {T32x64, {32, 64, 3.3359, 0.0639, 0.1595, 0.0522, 0.0380, true}},   {T16x32, {16, 32, 2.8913, 0.0966, 0.0642, 0.0302, 0.0699, true}},
};
const DeepCost DEEP_COSTS_256[TILES - D16x64] = {
    {16, 64, 3, 1664, 2.048, 0.158, 0.565, 0.347, 0.558, 0.0}, {16, 64, 1, 1665, 1.568, 0.0, 0.520, 0.196, 0.719, 0.948},
    {32, 32, 2, 3232, 2.469, 0.070, 0.618, 0.179, 0.365, 0.0}, {32, 32, 1, 3233, 1.575, 0.0, 0.491, 0.076, 1.499, 0.194},
    {32, 64, 2, 3264, 2.101, 0.181, 0.674, 0.170, 0.973, 0.0}, {32, 64, 1, 3265, 1.590, 0.0, 0.681, 0.142, 1.742, 0.0},
    {48, 64, 1, 4864, 1.385, 0.366, 0.561, 0.079, 2.233, 0.0},
};

Tile deep_tile(int code) {
    int t = 0;
    while (t < TILES - D16x64 && DEEP_COSTS[t].code != code) ++t;
    return static_cast<Tile>(D16x64 + t);
}

// (Beyond 16 rows a third workgroup of the smallest tiles fits beside two, but between two and three tiles to a CU it takes as long as a round
// of its own: 256 rows of 11008 -> 2700, 680 tiles of 32 x 32, 41.5 us, modelled 23.6 with three to a round, 38.8 on 64-row tiles.  Up to 16
// rows it does so at some sizes and not at others -- 9 rows of 4096 -> 37022 20.2 us as modelled, of 7296 -> 34372 43 (GEMV 25 and 39).)
double cost(const DeepCost &c, int M, int N, int K) {
    const double steps = (K + U * BK - 1) / (U * BK), r = (double)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) / 256.0;
    const double held = r <= 6 ? ceil(r) : r + 0.5, rounds = fmax(ceil(r / c.per_cu), M > 16 ? fmin(2.0, ceil(r / 2)) : 1.0);
    return c.fixed + steps * (c.tile * held + c.round * rounds + c.n * N * 1e-4) + c.tiles * held + c.rounds * rounds;
}

double cost(const Cost &c, int M, int N, int K) {
    const double steps = K / 128.0, r = (double)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) / 256.0;
    const double held = r <= 6 ? ceil(r) : r + 0.5;
    const double odd = r > 6 ? 0.5 : fmod(held, 2.0);
    return c.fixed + steps * (c.step + c.tile * held + c.odd * odd + c.n * N * 1e-4);
}

}  // namespace

namespace cmi {

static double deep_us(const DeepCost *costs, int tiles, int M, int N, int K, int *tile) {
    const int option = option_w4_gemm_deep();
    if (option > 1) {
        *tile = deep_tile(option);
        return 0.0;
    }
    double best = 1e30;
    for (int t = 0; option == 0 && K <= 1 << 24 && t < tiles; ++t) {  // (longer rows: the tile's offsets are 32-bit)
        const double us = cost(costs[t], M, N, K);
        if (us < best) best = us, *tile = D16x64 + t;
    }
    return best;
}

double gemm_w4a8_deep_us(int M, int N, int K, int *tile) { return deep_us(DEEP_COSTS, TILES - D16x64, M, N, K, tile); }

double gemm_w4a8_tile_us(int M, int N, int K, int gs, int *tile) {
    double best = 1e30;
    for (int t = 0; t < D16x64; ++t) {
        if (gs != BK && !COSTS[t].any_group) continue;
        const double us = cost(COSTS[t], M, N, K);
        if (us < best) best = us, *tile = t;
    }
    // Four groups a step where they are modelled to gain at least 5 %, or to lose at most 5 % on 16 x 32 tiles, which take up to 1.5
    // times their model at long rows (35 rows of 17920 -> 1582 38.6 us against 25.1): of 480 sizes (24 layer shapes x 17..1024 rows, rows
    // quantised in front, every weight cold) 19128 us without them, 17929 with, 17749 with the best of every size, none more than 2 %
    // slower.  Groups of 256 by costs of their own, with 3 % up to 200 rows and 7 % beyond (416 sizes 20221 -> 18160, 17970
    // with the best of every size; by the costs above 19067 and up to 30 % slower, 80 rows of 2048 -> 11008 13.5 -> 17.5).  Groups of 64
    // flush twice as often, which costs these tiles 1.35 times their model and the others 1.17: up to 16 rows, where they
    // are modelled to gain more than that (1106 us in all, 1095 with the best of every size, 1230 without them; 16 rows of
    // 5120 -> 32768 28.3 -> 21.1); beyond, the gain is 2 % in all and the model does not find it.
    int deep = 0;
    if (gs == 256 && M > 16) {
        for (const auto &c : COSTS_256)
            if (c.tile == *tile) best = cost(c.cost, M, N, K);
        // (48 x 64, the last: beyond 150 rows up to 21 % slower than modelled where rows are long, 300 rows of 17920 -> 6617)
        const double us = deep_us(DEEP_COSTS_256, TILES - D16x64 - (M > 150 && K > 10240), M, N, K, &deep);
        if (us < (M <= 200 ? 0.97 : 0.93) * best) best = us, *tile = deep;
        return best;
    }
    const double us = gs == 64 && M > 16 ? 1e30 : gemm_w4a8_deep_us(M, N, K, &deep);
    if (us < (gs == 64 ? 0.82 : M > 16 && *tile == T16x32 ? 1.05 : 0.95) * best) best = us, *tile = deep;
    return best;
}

int gemm_w4a8_forced_tile(int option, int gs) {
    static const struct { int option; Tile tile; } names[] = {{64, T32x64},   {128, T128x128}, {192, T64x96},  {128192, T64x128},
                                                              {256, T32x128}, {320, T128x160}, {321, T16x32}, {322, T64x64},
                                                              {6464, T64x64}};
    for (const auto &e : names)
        if (e.option == option && (gs == BK || COSTS[e.tile].any_group)) return e.tile;
    return T64x64;
}

bool gemm_w4a8_deep_code(int code) { return deep_tile(code) < TILES; }

int gemm_w4a8_tile(const uint8_t *w4, const float *ws, const int8_t *xq, const float *xs, void *y, int M, int N, int K,
                   int gs, int tile, void *stream) {
    Args a{xq, w4, xs, ws, static_cast<uint16_t *>(y), M, N, K, K / gs, 0, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    const Tile t = static_cast<Tile>(tile);
    return gs == 64 ? launch_tile<1>(a, t, st) : gs == 256 ? launch_tile<3>(a, t, st) : launch_tile<2>(a, t, st);
}

}  // namespace cmi
