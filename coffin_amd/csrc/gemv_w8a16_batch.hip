// int8 weight-only GEMV for 2..16 activation rows, in the canonical summation order of gemv_w8a16.hip: row r has the bits of the
// single-row call on it.
//
// v_mfma_f32_4x4x4_16b_bf16 adds, in each of 16 blocks of four lanes, four products of four weight rows with four activation rows
// to 4 x 4 sums: with the chunk that a chain of the canonical order owns in each block, the MFMA steps of the single-row kernels
// form the chains of up to four activation rows in one instruction, and every int8 is widened once for all of them.  The
// dot-product kernel that this replaces issued eight v_dot2 per 16 weight bytes and activation row: 16 rows ran at a fifth of the
// memory rate.  What bounds these kernels now: at one group of four activation rows the bytes of the weight (launch floors below 10 MB);
// at four groups the vector ALU and LDS reads of the activations, 2 KiB per group and KiB of weight.
//
// Two kernels, us before -> after of a dependent launch on cold weights:
//   stream    one workgroup per CU keeps the activations in LDS and its wavefronts walk row blocks (four weight rows), the next
//             block's loads requested segment by segment as registers free up.  2560 -> 151936 at 4 / 8 / 16 rows
//             76 -> 66 / 119 -> 67 / 224 -> 81 (one row 57), 2560 -> 19456 at 16 rows 37 -> 16, 5120 -> 51200 at 16 rows 207 -> 60.
//   quarters  a wavefront holds a quarter of the chunks of a row block, so a block is four wavefronts (more where units of K are
//             dealt to several sets of four): few outputs then still are many wavefronts with few instructions each, which is what
//             a launch of under 10 us is made of.  2560 -> 6144 at 4 / 16 rows 6.3 -> 5.5 / 13.7 -> 7.8, 4096 -> 2560 5.6 -> 4.4 / 10.8 -> 7.5,
//             9728 -> 2560 9.1 -> 9.0 / 35 -> 15, 1024 outputs of 2560 3.4 -> 3.0 / 8.5 -> 4.7.
// Rows of K that do not fit LDS go through it in windows of whole units (25600 -> 5120 at 4 / 16 rows 107 -> 37 / 403 -> 62; the
// dot-product kernel split the batch until each part fit and read the weight once for each).

#include "gemv_w8a16_math.hpp"

namespace {

using namespace cmi;

struct BatchArgs {
    const int8_t *wq;
    const float *ws;
    const uint16_t *x;
    uint16_t *y;
    int M, N, K;
    int nchunks;    // K / 16
    int segs;       // ceil(nchunks / 64)
    int quarters;   // ceil(nchunks / 16)
    int units;      // of the canonical order
    int items;      // ceil(N / 4)
    int teams;      // quarters kernel: row blocks per workgroup
    int sets;       // quarters kernel: wavefronts that share a quarter of a row block by its units (1 for windows)
    uint32_t sets_rcp;   // ceil(2^16 / sets)
    uint32_t xvecs_rcp;  // ceil(2^32 / (K/8))
};

// Activation row (of four) that lane l holds: blocks of odd number hold them in reverse, so that the lanes l ^ 7 and l ^ 15,
// which DPP adds in one instruction, hold the same one.
__device__ __forceinline__ int lane_row(int lane) { return (lane & 4) ? 3 - (lane & 3) : lane & 3; }

// Where chunk c (of a segment's 64) of activation row j of four lies in the LDS copy, in 16-byte slots of its segment: blocks of 128
// slots per 16 chunks that one MFMA step takes, the halves of the chunks apart.  WHOLE: a step takes every fourth chunk, else sixteen
// in a row.  A wavefront reads whole halves; the xor keeps the writes, which come in memory order, free of conflicts.
template <bool WHOLE>
__device__ __forceinline__ int x_step(int c) { return WHOLE ? c & 3 : c >> 4; }
template <bool WHOLE>
__device__ __forceinline__ int x_slot(int c, int j, int half) {
    if constexpr (WHOLE) return half * 64 + ((c >> 2) ^ (half << 1)) * 4 + (j ^ (c & 3));
    return half * 64 + (c & 15) * 4 + (j ^ (((c >> 2) & 1) | (half << 1)));
}

// 4 x 4 transpose within every four lanes: register r of lane i becomes register i of lane r.
__device__ __forceinline__ void quad_transpose(u32x4 (&w)[4]) {
#pragma unroll
    for (int d = 0; d < 4; d += 2) {
        uint32_t t0, t1, t2, t3, u0, u1, u2, u3;
        uint32_t a0 = w[0][d], a1 = w[1][d], a2 = w[2][d], a3 = w[3][d];
        uint32_t b0 = w[0][d + 1], b1 = w[1][d + 1], b2 = w[2][d + 1], b3 = w[3][d + 1];
        asm("s_mov_b64 vcc, %16\n\ts_nop 1\n\t"
            "v_cndmask_b32_dpp %0, %9, %8, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %2, %11, %10, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %4, %13, %12, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %6, %15, %14, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "s_not_b64 vcc, vcc\n\t"
            "v_cndmask_b32_dpp %1, %8, %9, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %3, %10, %11, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %5, %12, %13, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %7, %14, %15, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
            : "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3), "=&v"(u0), "=&v"(u1), "=&v"(u2), "=&v"(u3)
            : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "v"(b0), "v"(b1), "v"(b2), "v"(b3), "s"(0x5555555555555555ull)
            : "vcc", "scc");
        asm("s_mov_b64 vcc, %16\n\ts_nop 1\n\t"
            "v_cndmask_b32_dpp %0, %10, %8, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %1, %11, %9, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %4, %14, %12, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %5, %15, %13, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "s_not_b64 vcc, vcc\n\t"
            "v_cndmask_b32_dpp %2, %8, %10, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %3, %9, %11, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %6, %12, %14, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_cndmask_b32_dpp %7, %13, %15, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
            : "=&v"(a0), "=&v"(a1), "=&v"(a2), "=&v"(a3), "=&v"(b0), "=&v"(b1), "=&v"(b2), "=&v"(b3)
            : "v"(t0), "v"(t1), "v"(t2), "v"(t3), "v"(u0), "v"(u1), "v"(u2), "v"(u3), "s"(0x3333333333333333ull)
            : "vcc", "scc");
        w[0][d] = a0, w[1][d] = a1, w[2][d] = a2, w[3][d] = a3;
        w[0][d + 1] = b0, w[1][d + 1] = b1, w[2][d + 1] = b2, w[3][d + 1] = b3;
    }
}

// Sums over the 16 blocks of a wavefront of 4 MG values a lane (value 4 * group + weight row), pairing blocks b ^ 1, b ^ 2, b ^ 4,
// b ^ 8 in this order.  Lanes l ^ 7 and l ^ 15 are the pairs of the first two levels (see lane_row; the half that a lane keeps is chosen
// so that its partner at the next level keeps the same one), then rows and halves of the wavefront.  While values are left to
// choose from, a level halves them; the total of value quarter_index(l) for activation row lane_row(l) ends in lane l.
template <int MG>
__device__ __forceinline__ float quarter_sum(const v4f32 (&acc)[MG], int lane) {
    constexpr int NV = 4 * MG;
    float v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = acc[i / 4][i % 4];
    const bool s1 = (((lane >> 2) ^ (lane >> 3)) & 1) != 0, s2 = ((lane >> 3) & 1) != 0;
    float a[NV / 2], b[NV / 4];
    transposed_level<0x141, NV / 2>(v, a, s1);
    transposed_level<0x140, NV / 4>(a, b, s2);
    if constexpr (MG == 4) {
        return swap32_add(swap16_add(b[0], b[2]), swap16_add(b[1], b[3]));
    } else if constexpr (MG == 2) {
        const float c = swap16_add(b[0], b[1]);
        return swap32_add(c, c);
    } else {
        const float c = swap16_add(b[0], b[0]);
        return swap32_add(c, c);
    }
}
template <int MG>
__device__ __forceinline__ int quarter_index(int lane) {
    const int s1 = ((lane >> 2) ^ (lane >> 3)) & 1, s2 = (lane >> 3) & 1, b4 = (lane >> 4) & 1, b5 = (lane >> 5) & 1;
    if constexpr (MG == 4) return s1 * 8 + s2 * 4 + b4 * 2 + b5;
    else if constexpr (MG == 2) return s1 * 4 + s2 * 2 + b4;
    else return s1 * 2 + s2;
}

// Activations on their way to LDS, XV 16-byte vectors a thread in memory order.
template <int XV>
__device__ __forceinline__ void request_x(uint4 (&xs)[XV], const BatchArgs &a, int threads) {
    const uint4 *xg = reinterpret_cast<const uint4 *>(a.x);
    const int total = a.M * (a.K / 8);
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int idx = threadIdx.x + j * threads;
        xs[j] = idx < total ? xg[idx] : make_uint4(0, 0, 0, 0);
    }
}

template <int MG, bool WHOLE>
__device__ __forceinline__ int x_at(int chunk, int m, int half) {
    return (((chunk >> 6) * 4 + x_step<WHOLE>(chunk & 63)) * MG + (m >> 2)) * 128 + x_slot<WHOLE>(chunk & 63, m & 3, half);
}

// ... into LDS, zeros past K up to the end of the last segment (WHOLE) or quarter.
template <int MG, bool WHOLE, int XV>
__device__ __forceinline__ void keep_x(uint4 *smem, const uint4 (&xs)[XV], const BatchArgs &a, int threads) {
    const int xvecs = a.K / 8, total = a.M * xvecs;
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int idx = threadIdx.x + j * threads;
        const int m = __umulhi((uint32_t)idx, a.xvecs_rcp), v = idx - m * xvecs;
        if (idx < total) smem[x_at<MG, WHOLE>(v >> 1, m, v & 1)] = xs[j];
    }
    const int end = WHOLE ? a.segs * 64 : a.quarters * 16;
    for (int i = threadIdx.x; i < (end - a.nchunks) * 8 * MG; i += threads) {
        const int r = i % (8 * MG);
        smem[x_at<MG, WHOLE>(a.nchunks + i / (8 * MG), r >> 1, r & 1)] = make_uint4(0, 0, 0, 0);
    }
}

// One MFMA step (16 chunks of four weight rows) onto the chains of all activation groups.
template <int MG>
__device__ __forceinline__ void add_step(v4f32 (&acc)[MG], const u32x4 &d, const uint4 (&x)[MG][2], bool from_zero) {
    const Chunk w = widen_chunk(d);
#pragma unroll
    for (int g = 0; g < MG; ++g) acc[g] = chain_chunk(from_zero ? v4f32{0.f, 0.f, 0.f, 0.f} : acc[g], w, x[g][0], x[g][1]);
}

// MG: groups of four activation rows; U: segments of a unit; XV: 16-byte vectors of activations a thread carries to LDS.
// A load takes 1 KiB of one weight row, whole lines in order; four of them, one for each row of the block, become the MFMA
// arrangement by a transpose within every four lanes (step q then holds chunks 4t + q in block t).  Loaded in that arrangement
// directly, four rows' 16-byte pieces alternate in neighbouring lanes, and 2560 -> 151936 at four rows took 74 us instead of 62.
// The four steps' sums meet in the lane, (0 + 1) + (2 + 3): the tree's levels c ^ 1 and c ^ 2.
template <int MG, int U, int XV, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
gemv_w8a16_stream_kernel(const BatchArgs a) {
    extern __shared__ uint4 smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint4 xs[XV];
    request_x(xs, a, 64 * WAVES);
    const XcdItems blocks = xcd_items(a.items, wave, WAVES);  // of four weight rows
    const int end = blocks.end, step = blocks.step;
    int item = blocks.next, u = 0;

    u32x4 w[U][4];
    auto load_seg = [&](int it, int unit, int s) {
        const uint32_t off = (uint32_t)min((unit * U + s) * 64 + lane, a.nchunks - 1) * 16u;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            w[s][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(a.wq + (size_t)min(it * 4 + r, a.N - 1) * a.K + off));
    };
    if (item < end) {
#pragma unroll
        for (int s = 0; s < U; ++s) load_seg(item, 0, s);
    }
    keep_x<MG, true>(smem, xs, a, 64 * WAVES);
    __syncthreads();

    const int vi = quarter_index<MG>(lane);
    const int row = vi % 4, xrow = lane_row(lane), m = (vi / 4) * 4 + xrow;
    const bool mine = (MG == 4 || (lane & (MG == 2 ? 32 : 48)) == 0) && m < a.M;
    const int slot0 = x_slot<true>(lane & 60, xrow, 0), slot1 = x_slot<true>(lane & 60, xrow, 1);
    float scale = 0.f, total = 0.f;
#pragma unroll 1
    while (item < end) {
        const bool last = u + 1 == a.units;
        const int next = last ? item + step : item, next_u = last ? 0 : u + 1;
        if (u == 0) scale = a.ws[min(item * 4 + row, a.N - 1)];
        v4f32 acc[4][MG];
#pragma unroll
        for (int s = 0; s < U; ++s) {
            if (s == 0 || u * U + s < a.segs) {
                quad_transpose(w[s]);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint4 x[MG][2];
                    const uint4 *at = smem + ((u * U + s) * 4 + q) * MG * 128;
#pragma unroll
                    for (int g = 0; g < MG; ++g) x[g][0] = at[g * 128 + (slot0 ^ q)], x[g][1] = at[g * 128 + (slot1 ^ q)];
                    add_step<MG>(acc[q], w[s][q], x, s == 0);
                }
            }
            if (next < end) load_seg(next, next_u, s);
        }
        v4f32 sum[MG];
#pragma unroll
        for (int g = 0; g < MG; ++g) sum[g] = (acc[0][g] + acc[1][g]) + (acc[2][g] + acc[3][g]);
        const float t = quarter_sum<MG>(sum, lane);
        total = u == 0 ? t : total + t;
        const int n = item * 4 + row;
        if (last && mine && n < a.N) a.y[(size_t)m * a.N + n] = (uint16_t)f32_to_bf16_bits(scale * total);
        item = next, u = next_u;
    }
}

// The activations of SEGS segments of K from first_seg on, on their way to LDS (1024 threads) and into it, zeros past K.
template <int MG, int SEGS, int XV>
__device__ __forceinline__ void request_window(uint4 (&xs)[XV], const BatchArgs &a, int first_seg) {
    const uint4 *xg = reinterpret_cast<const uint4 *>(a.x);
    const int xvecs = a.K / 8;
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int idx = threadIdx.x + j * 1024, m = idx / (SEGS * 128), v = first_seg * 128 + idx % (SEGS * 128);
        xs[j] = m < a.M && v < xvecs ? xg[(size_t)m * xvecs + v] : make_uint4(0, 0, 0, 0);
    }
}
template <int MG, int SEGS, int XV>
__device__ __forceinline__ void keep_window(uint4 *smem, const uint4 (&xs)[XV], const BatchArgs &a) {
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int idx = threadIdx.x + j * 1024, m = idx / (SEGS * 128), v = idx % (SEGS * 128);
        if (m < a.M) smem[x_at<MG, false>(v >> 1, m, v & 1)] = xs[j];
    }
}

// RG: row blocks a wavefront shares the activation fragments between.  SETS: sets of four wavefronts that share a row block by its
// units (0: a.sets).  ONE: K is one unit.  WINDOW: LDS holds the activations of SETS units at a time.
// A lane loads its own row of the MFMA arrangement, 256 bytes of four rows a load: a transpose would need all four quarters in one
// wavefront.  The tree's levels c ^ 1 .. c ^ 8 are the blocks of the wavefront, c ^ 16 and c ^ 32 the quarters, which meet in LDS.
template <int MG, int RG, int U, int SETS, bool ONE, bool WINDOW, int XV>
__global__ void __launch_bounds__(1024)
gemv_w8a16_quarters_kernel(const BatchArgs a) {
    extern __shared__ uint4 smem[];
    constexpr int OUT = 16 * MG;  // outputs of four weight rows
    // The next unit's weights are asked for behind this one's sums: segment by segment as registers free up measured 5..20 % slower
    // (two rows of 5120 -> 7168 12.4 against 10.3 us, 16 of 25600 -> 5120 77 against 62) except between windows with two blocks (41 against 39).
    constexpr bool AS_FREED = WINDOW && RG == 2;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sets = SETS ? SETS : a.sets, threads = a.teams * sets * 256;
    const int q = wave & 3, team = SETS ? (wave >> 2) / SETS : (int)(((uint32_t)(wave >> 2) * a.sets_rcp) >> 16), set = (wave >> 2) - team * sets;
    const int n0 = (xcd_contiguous_block(blockIdx.x, gridDim.x) * a.teams + team) * 4 * RG;
    uint4 xs[XV];
    if constexpr (WINDOW) request_window<MG, SETS * U>(xs, a, 0);
    else request_x(xs, a, threads);

    const int row = lane & 3, chunk0 = q * 16 + (lane >> 2), xrow = lane_row(lane);
    u32x4 w[U][RG];
    auto load_seg = [&](int unit, int s) {
        const uint32_t off = (uint32_t)min((unit * U + s) * 64 + chunk0, a.nchunks - 1) * 16u;
#pragma unroll
        for (int r = 0; r < RG; ++r)
            w[s][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(a.wq + (size_t)min(n0 + 4 * r + row, a.N - 1) * a.K + off));
    };
#pragma unroll
    for (int s = 0; s < U; ++s) load_seg(set, s);
    // the output that this thread adds up, scales and stores
    const int ft = (int)threadIdx.x - team * sets * 256, fr = ft / OUT, fo = ft % OUT;
    const int fm = (fo / 16) * 4 + fo % 4, fn = n0 + 4 * fr + (fo / 4) % 4;
    const float scale = a.ws[min(fn, a.N - 1)];
    if constexpr (WINDOW) keep_window<MG, SETS * U>(smem, xs, a);
    else keep_x<MG, false>(smem, xs, a, threads);
    __syncthreads();
    // quarter totals [row block][weight rows][unit (WINDOW: those in hand)][quarter][output]
    const int units = ONE ? 1 : a.units, kept = WINDOW ? SETS : units;
    float *totals = reinterpret_cast<float *>(smem + (WINDOW ? SETS * 4 * U : a.quarters) * MG * 128) + team * kept * (4 * RG * OUT);
    float total = 0.f;
    auto add_unit = [&](int u) {  // thread of output fo: the quarters of a unit meet as in the single-row tree, then the units in order
        if (fr >= RG) return;
        const float *t = totals + ((fr * kept + (WINDOW ? u % SETS : u)) * 4) * OUT + fo;
        const float s = (t[0] + t[OUT]) + (t[2 * OUT] + t[3 * OUT]);
        total = u == 0 ? s : total + s;
    };
    const int slot0 = x_slot<false>(chunk0, xrow, 0), slot1 = x_slot<false>(chunk0, xrow, 1);
    const int vi = quarter_index<MG>(lane);
    const bool mine = MG == 4 || (lane & (MG == 2 ? 32 : 48)) == 0;
#pragma unroll 1
    for (int trip = 0; trip < units; trip += sets) {
        const int u = trip + set;  // (past the last unit in the last trip of some sets: nothing is live there)
        const bool more = trip + sets < units;
        if constexpr (WINDOW)
            if (more) request_window<MG, SETS * U>(xs, a, (trip + sets) * U);
        v4f32 acc[RG][MG];
#pragma unroll
        for (int r = 0; r < RG; ++r)
#pragma unroll
            for (int g = 0; g < MG; ++g) acc[r][g] = v4f32{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < U; ++s) {
            const int qi = (u * U + s) * 4 + q;
            if (qi < a.quarters) {
                uint4 x[MG][2];
                const uint4 *at = smem + (WINDOW ? (set * U + s) * 4 + q : qi) * MG * 128;
#pragma unroll
                for (int g = 0; g < MG; ++g) x[g][0] = at[g * 128 + slot0], x[g][1] = at[g * 128 + slot1];
#pragma unroll
                for (int r = 0; r < RG; ++r) add_step<MG>(acc[r], w[s][r], x, false);
            }
            if constexpr (AS_FREED)
                if (more) load_seg(u + sets, s);
        }
#pragma unroll
        for (int r = 0; r < RG; ++r) {
            const float t = quarter_sum<MG>(acc[r], lane);
            if (mine && (WINDOW || u < units)) totals[((r * kept + (WINDOW ? set : u)) * 4 + q) * OUT + vi * 4 + xrow] = t;
        }
        if (!AS_FREED && more) {
#pragma unroll
            for (int s = 0; s < U; ++s) load_seg(u + sets, s);
        }
        if constexpr (WINDOW) {
            __syncthreads();  // every wavefront has read its part of the window and left its totals
            for (int v = trip; v < trip + SETS && v < units; ++v) add_unit(v);
            if (more) {
                keep_window<MG, SETS * U>(smem, xs, a);
                __syncthreads();
            }
        }
    }
    if constexpr (!WINDOW) {
        __syncthreads();
        for (int u = 0; u < units; ++u) add_unit(u);
    }
    if (fr < RG && fm < a.M && fn < a.N) a.y[(size_t)fm * a.N + fn] = (uint16_t)f32_to_bf16_bits(scale * total);
}

constexpr size_t LDS_BYTES = 160 * 1024;

template <int MG, int U, int XV, int WAVES, int PER_CU>
int launch_stream(const BatchArgs &a, hipStream_t st) {
    auto k = gemv_w8a16_stream_kernel<MG, U, XV, WAVES>;
    static std::atomic<uint64_t> devices{0};
    if (const int rc = reserve_lds(reinterpret_cast<const void *>(k), LDS_BYTES, devices, "cmi_gemv_w8a16")) return rc;
    const int blocks = (a.items + WAVES - 1) / WAVES;
    k<<<dim3(blocks < 256 * PER_CU ? blocks : 256 * PER_CU), dim3(64 * WAVES), (size_t)a.segs * MG * 8192, st>>>(a);
    return check_launch("cmi_gemv_w8a16");
}

template <int MG, int RG, int U, int SETS, bool ONE, bool WINDOW, int XV>
int launch_quarters(BatchArgs &a, hipStream_t st) {
    auto k = gemv_w8a16_quarters_kernel<MG, RG, U, SETS, ONE, WINDOW, XV>;
    static std::atomic<uint64_t> devices{0};
    if (const int rc = reserve_lds(reinterpret_cast<const void *>(k), LDS_BYTES, devices, "cmi_gemv_w8a16")) return rc;
    const size_t lds = (size_t)(WINDOW ? SETS * 4 * U : a.quarters) * MG * 2048 + (size_t)a.teams * (WINDOW ? SETS : a.units) * (RG * MG * 256);
    a.sets_rcp = (65536u + a.sets - 1) / a.sets;
    const int rows = 4 * RG * a.teams;
    k<<<dim3((a.N + rows - 1) / rows), dim3(256 * a.teams * a.sets), lds, st>>>(a);
    return check_launch("cmi_gemv_w8a16");
}

// Whether every activation row fits LDS as the stream kernel holds it.
bool stream_fits(int mg, int segs) { return (size_t)segs * mg * 8192 <= LDS_BYTES; }

constexpr int up(int v, int d) { return (v + d - 1) / d; }

// Only forms that some row count and K reach are built: with U segments a unit K is above (U - 1) * 1024, one unit is at most U * 1024, and
// units of three (unit_segments) are of 5, 6 or 9 segments.  A count outside what a form was built for is an error, never a short copy.
template <int MG>
constexpr int least_rows() { return MG == 1 ? 1 : MG == 2 ? 5 : 9; }

int unbuilt(const BatchArgs &a) { return fail(CMI_E_UNSUPPORTED, "cmi_gemv_w8a16: no kernel for %d rows of %d", a.M, a.K); }

template <int MG, int U>
int stream(const BatchArgs &a, hipStream_t st) {
    if constexpr (MG == 1)
        if (a.segs <= 6 && a.M * (a.K / 8) <= 8 * 512) return launch_stream<MG, U, 8, 8, 2>(a, st);
    if constexpr (MG > 1 || U >= 3) {
        constexpr int WAVES = MG == 4 && U == 4 ? 8 : 12;  // 16 rows and four segments in flight take more than 168 registers
        constexpr int LAST = WAVES == 8 ? 20 : 14;
        constexpr int LONGEST = U <= 2 ? U * 1024 : U == 3 && MG < 4 ? 9216 : 20480 / MG;  // stream_fits
        constexpr int LEAST = up(least_rows<MG>() * ((U - 1) * 128 + 2), 64 * WAVES), MOST = up(4 * MG * (LONGEST / 8), 64 * WAVES);
        const int need = up(a.M * (a.K / 8), 64 * WAVES);
        if constexpr (LEAST <= 3)
            if (need <= 3) return launch_stream<MG, U, 3, WAVES, 1>(a, st);
        if constexpr (MOST > 3)
            if (need <= 7) return launch_stream<MG, U, 7, WAVES, 1>(a, st);
        if constexpr (MOST > 7)
            if (need <= LAST) return launch_stream<MG, U, LAST, WAVES, 1>(a, st);
    }
    return unbuilt(a);
}

template <int MG, int RG, int U, bool ONE>
int by_vectors(BatchArgs &a, int need, hipStream_t st) {
    // most of one unit: of the smallest workgroup (run); of several: of three teams, as fewer have sets, or of sixteen wavefronts.  Least of several: of
    // sixteen wavefronts, which one block a wavefront at eight rows has above K = 8192
    constexpr int THREADS = 256 * (RG == 1 ? 1 : MG == 4 ? 3 : 2);
    constexpr int LEAST = ONE ? 1 : up(least_rows<MG>() * (U == 3 ? 514 : MG == 2 && RG == 1 ? 1026 : 770), 1024);
    constexpr int MOST = ONE ? up(MG * U * 512, THREADS) : MG == 1 && RG == 1 && U == 3 ? up(4 * 1152, 768) : 12;
    if constexpr (LEAST <= 4)
        if (need <= 4) return launch_quarters<MG, RG, U, 1, ONE, false, 4>(a, st);
    if constexpr (MOST > 4)
        if (need <= 8) return launch_quarters<MG, RG, U, 1, ONE, false, 8>(a, st);
    if constexpr (MOST > 8)
        if (need <= 12) return launch_quarters<MG, RG, U, 1, ONE, false, 12>(a, st);
    return unbuilt(a);
}

template <int MG, int U, int RG>
int quarters(BatchArgs &a, hipStream_t st) {
    auto need = [&] { return up(a.M * (a.K / 8), 256 * a.teams * a.sets); };
    const int rows = 4 * RG * a.teams;
    while (a.teams * a.sets < 4 && need() > 12) ++a.teams, a.sets = 1;
    if (a.sets > 1 && need() > 12) a.teams = 4, a.sets = 1;
    const size_t totals = (size_t)a.teams * a.units * (RG * MG * 256);
    // (what fits LDS is at most ten vectors a thread of sixteen wavefronts)
    if ((size_t)a.quarters * MG * 2048 + totals <= LDS_BYTES) {
        if constexpr (U == 3 || (U == 4 && MG < 4)) {  // (16 rows of several units of four segments do not fit)
            if constexpr (RG == 1) {
                if constexpr (MG < 4)
                    if (a.sets > 1 && need() <= 4) return launch_quarters<MG, RG, U, 0, false, false, 4>(a, st);
                if (a.sets > 1) return launch_quarters<MG, RG, U, 0, false, false, 12>(a, st);
            }
            if (a.units > 1) return by_vectors<MG, RG, U, false>(a, need(), st);
        }
        return by_vectors<MG, RG, U, true>(a, need(), st);
    }
    // long rows: windows of as many units as LDS takes and the row blocks leave wavefronts for (units of four segments: the only
    // longer rows of units of three are sixteen)
    constexpr bool LONG = U == 4 || (U == 3 && MG == 4);
    constexpr int XV = up(MG * U * 512, 1024);
    if constexpr (LONG && RG == 1) {
        if constexpr (MG == 1)
            if (rows <= 4) return a.teams = 1, a.sets = 4, launch_quarters<MG, RG, U, 4, false, true, 4 * XV>(a, st);
        if constexpr (MG <= 2)
            if (rows <= 8) return a.teams = 2, a.sets = 2, launch_quarters<MG, RG, U, 2, false, true, 2 * XV>(a, st);
    }
    a.teams = 4, a.sets = 1;
    if constexpr (LONG && (RG == 1 || MG <= 2)) return launch_quarters<MG, RG, U, 1, false, true, XV>(a, st);
    return unbuilt(a);
}

template <int MG, int U>
int run(BatchArgs &a, bool streamed, hipStream_t st) {
    if (streamed) return stream<MG, U>(a, st);
    const int rows = (a.N - 1) / 256 + 1;  // of a CU
    // Row blocks for every CU at once: 4 rg weight rows a team, up to four teams a workgroup.  Twelve rows a CU go one block a
    // wavefront (4096 -> 2560 at four rows 4.4 us, two blocks 4.9); above, two share the activation fragments.  Short rows and pairs of
    // rows want small workgroups (1024 -> 8192 at four rows 3.9 with two blocks, 4.3 with eight; 896 -> 1030 at three 2.62 with one
    // block, 2.73 with two; two rows of 2560 -> 6144 5.2 against 5.5), and so does everything beyond 32 rows a CU, where workgroups
    // follow each other (2560 -> 19456 12.0 with four blocks, 13.9 with eight).
    // Up to sixteen rows a CU of many units: four teams of one block (14336 -> 4096 at 4 / 8 rows 16.0 / 17.9 us, two of two 18.8 / 22.8, at two and
    // three rows 1 % the other way; 20480 -> 3600 at three rows 20.5, 29.8).  Of three units only from five rows on (9728 -> 3800 at eight rows
    // 12.6, 17.2; at four 11.5 against 11.2, 10240 -> 3800 12.3 against 11.8).
    int rg = 2;
    if (rows <= 12) rg = 1, a.teams = MG == 1 && a.K <= 1024 ? 1 : (rows + 3) / 4;
    else if (MG <= 2 && a.K <= 1024) a.teams = MG;
    else if (a.M <= 2 && a.units == 1 && rows <= 32) a.teams = 1;
    else if (rows <= 16) rg = MG == 4 || a.units > (MG == 1 ? 3 : 2) ? 1 : 2, a.teams = 4 / rg;
    else if (rows <= 32) a.teams = rows <= 24 ? 3 : 4;
    else a.teams = MG == 4 ? 4 : 2;
    // wavefronts left in a workgroup of sixteen share the units of a long K (12800 -> 1000 at four rows 11 -> 6.7 us)
    a.sets = rg == 1 ? 4 / a.teams : 1;
    if (a.sets > a.units) a.sets = a.units;
    // four groups whose rows go through LDS in windows have registers for one block
    const size_t whole = (size_t)a.quarters * MG * 2048 + (size_t)4 * a.units * (2 * MG * 256);
    if (MG == 4 && whole > LDS_BYTES) rg = 1;
    return rg == 1 ? quarters<MG, U, 1>(a, st) : quarters<MG, U, 2>(a, st);
}

template <int MG>
int by_unit(BatchArgs &a, int unit, bool streamed, hipStream_t st) {
    if (unit == 1) return run<MG, 1>(a, streamed, st);
    if (unit == 2) return run<MG, 2>(a, streamed, st);
    if (unit == 3) return run<MG, 3>(a, streamed, st);
    return run<MG, 4>(a, streamed, st);
}

}  // namespace

namespace cmi {
int gemv_w8a16_batch(const int8_t *wq, const float *ws, const void *x, void *y, int M, int N, int K, void *stream) {
    BatchArgs a;
    a.wq = wq;
    a.ws = ws;
    a.x = static_cast<const uint16_t *>(x);
    a.y = static_cast<uint16_t *>(y);
    a.M = M;
    a.N = N;
    a.K = K;
    a.nchunks = K / 16;
    a.quarters = (a.nchunks + 15) / 16;
    a.segs = (a.nchunks + 63) / 64;
    const int unit = unit_segments(a.segs);
    a.units = (a.segs + unit - 1) / unit;
    a.items = (N + 3) / 4;
    a.teams = a.sets = 1;
    a.xvecs_rcp = (uint32_t)(((1ull << 32) + (K / 8) - 1) / (K / 8));
    const int mg = M <= 4 ? 1 : M <= 8 ? 2 : 4;
    // Which kernel: the stream kernel where every CU's wavefronts get row blocks enough to pay for its copy of the activations.  Four groups: from 9216
    // outputs (16 rows of 2560 -> 9728 12.0 against 13.3 us, 2560 -> 6144 9.7 against 7.6); two: 16384 (2560 -> 19456 14.5 against 15.8, 4096 -> 14336 17.1
    // against 16.4); one: four rows of 128 MiB and more (2560 -> 151936 67 against 72; three rows of 3072 -> 100000 53.6
    // against 50.4).  K of several units: 8192 outputs at two groups (6400 -> 9000 19.1 against 21.2), 96 MiB at one (5120 -> 51200 44.6 against 56, 5120 ->
    // 10000 16.7 against 15.2).  Four groups whose copy leaves the quarters kernel no room (K of 4609..5120): from 4096 outputs (5120 -> 5120 14.2 against 18.8).
    const size_t bytes = (size_t)N * K;
    const bool many = mg == 4   ? N >= 9216 || (a.quarters * 4 * 2048 + 16384 > (int)LDS_BYTES && N >= 4096)
                      : mg == 2 ? N >= (a.units > 1 ? 8193 : 16384)
                                : bytes >= (a.units > 1 ? (size_t)96 << 20 : M < 4 ? SIZE_MAX : (size_t)128 << 20);
    const bool streamed = many && stream_fits(mg, a.segs);
    // Sixteen rows too long for LDS where eight are not: two launches stream (8192 -> 28672 at 16 rows 106 -> 83 us).
    if (mg == 4 && !stream_fits(4, a.segs) && stream_fits(2, a.segs) && N >= 16384) {
        const int rc = gemv_w8a16_batch(wq, ws, x, y, 8, N, K, stream);
        return rc ? rc : gemv_w8a16_batch(wq, ws, a.x + (size_t)8 * K, a.y + (size_t)8 * N, M - 8, N, K, stream);
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    return mg == 1 ? by_unit<1>(a, unit, streamed, st) : mg == 2 ? by_unit<2>(a, unit, streamed, st) : by_unit<4>(a, unit, streamed, st);
}
}  // namespace cmi
