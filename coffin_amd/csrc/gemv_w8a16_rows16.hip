// int8 weight-only GEMV for batches of up to 16 bf16 activation rows (batched
// decode, speculative verify).
//
//   y[m,n] = bf16( (sum_k x[m,k] * (float)wq[n,k]) * ws[n] )        fp32 sums
//
// int8 -> bf16 is exact
// and bf16 x bf16 products are exact in fp32, so v_mfma_f32_16x16x32_bf16
// forms the sums -- 16 weight rows x 16 activation rows x 32 k per instruction
// -- and the vector ALU only widens the weight bytes.  The kernel stays a GEMV
// in every other respect: the weight is read once, straight into registers, all
// of a wavefront's bytes requested before anything else.
//
// A workgroup owns 16 weight rows; its wavefronts split K by 128-byte lines of
// the weight rows (wavefront w takes lines w, w+WAVES, ..).  For the MFMA lane l
// holds k  32*(l/16) .. +31  of a line for weight row l%16 (two 16-byte pieces)
// and for activation row l%16 (four pieces); both are fetched as whole cache
// lines and rearranged through private LDS patches.  The fp32 partial tiles of
// the wavefronts are added in wavefront order through LDS, so a row's result
// depends on K only, not on the batch it came in -- but it is not the bit
// pattern of the kernels behind cmi_gemv_w8a16 (different fp32
// summation order), which is why this kernel has an entry point of its own:
// callers that owe their users "a batched row equals the single-row call"
// (static-batch decode) stay on cmi_gemv_w8a16.
//
// TAIL: rows that end inside a line.  Of the last line the activations past K are zeros that are not read, so what
// the weight's pieces hold there (bytes of the row again) does not matter.  Cold weights, against the kernels of cmi_gemv_w8a16, 16 rows a
// launch: 9 rows of 2624 -> 9728 11.4 us, 12.5 there; 63 rows 22.0, 47.2; 16 rows of 9792 -> 2560 14.3, 14.5; 50 rows of 1344 -> 1000 8.6, 14.2;
// 63 rows of 13888 -> 5120 80, 141.
#include "rows16_tile.hpp"

namespace {

using namespace cmi;
using namespace cmi::rows16;

typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int ROWS = 16;
constexpr int LINE = 128;           // k per line
constexpr int XPITCH = 256 + 16;    // activation patch: 16 rows x 256 bytes
constexpr int XPATCH_BYTES = 16 * XPITCH;

struct Args {
    const int8_t *wq;
    const float *ws;
    const uint16_t *x;
    uint16_t *y;
    int M, N, K;
};

// Four int8 of a dword -> four bf16 (two dwords); exact.
__device__ __forceinline__ void widen4(uint32_t w, uint32_t &lo, uint32_t &hi) {
    const float f0 = (float)(int8_t)(w);
    const float f1 = (float)(int8_t)(w >> 8);
    const float f2 = (float)(int8_t)(w >> 16);
    const float f3 = (float)(int8_t)(w >> 24);
    // integers up to 128 in magnitude live in the upper 16 bits of their fp32 pattern
    lo = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
    hi = __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u);
}

// How the sums of a row's lines meet.  A chain of MFMAs is less exact than the single-row order, which the rows that end inside a
// line left, and which sums in short chains: so for those the MFMAs of a line start from zero and their sums meet in pairs, and where
// a wavefront has many lines (LOW) what the additions round off is kept and added at the end.  Root mean square error of sums that
// cancel (activations N(0, 1), 1 % of them 20 times larger, weights N(0, 30)), in 2^-24 of the sum of magnitudes, K = 960 / 2624 / 9664 / 25536:
// single-row order 0.054 / 0.046 / 0.031 / 0.022, a chain 0.061 / 0.054 / 0.053 / 0.058, these 0.054 / 0.046 / 0.025 / 0.015 (a kept sum over up to three lines as well: 0.045 at 2624, and 63 rows of 2624 ->
// 9728 24.9 us instead of 22.1).
enum Sum { CHAIN, PAIRS, LOW };
constexpr Sum sum_of(bool tail, int nlp, int rounds) { return !tail ? CHAIN : rounds == 1 && nlp <= 3 ? PAIRS : LOW; }

// The 128 products of a line onto acc: x holds the activations, w0 and w1 the codes in the MFMA arrangement.
template <Sum S>
__device__ __forceinline__ void add_line(v4f32 &acc, v4f32 &low, const v4i32 (&x)[4], v4i32 w0, v4i32 w1) {
    const uint32_t d[8] = {(uint32_t)w0.x, (uint32_t)w0.y, (uint32_t)w0.z, (uint32_t)w0.w,
                           (uint32_t)w1.x, (uint32_t)w1.y, (uint32_t)w1.z, (uint32_t)w1.w};
    v4f32 sum[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {  // k = 32*kq + 8*s .. +7 of the line
        uint32_t b[4];
        widen4(d[2 * s], b[0], b[1]);
        widen4(d[2 * s + 1], b[2], b[3]);
        const v4i32 bw = {(int)b[0], (int)b[1], (int)b[2], (int)b[3]};
        const v4f32 from = S == CHAIN ? acc : v4f32{0.f, 0.f, 0.f, 0.f};
        sum[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[s]), __builtin_bit_cast(bf16x8, bw), from, 0, 0, 0);
        if (S == CHAIN) acc = sum[s];
    }
    if constexpr (S != CHAIN) {
        const v4f32 line = (sum[0] + sum[1]) + (sum[2] + sum[3]), next = acc + line;
        if (S == LOW) low += line - (next - acc);
        acc = next;
    }
}

// A wavefront's share of its sums.  One that is infinite stays that: what was kept beside it is a difference of infinities.
template <Sum S>
__device__ __forceinline__ v4f32 whole_sum(v4f32 acc, v4f32 low) {
    if constexpr (S == LOW) {
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] = fabsf(acc[v]) < INFINITY ? acc[v] + low[v] : acc[v];
    }
    return acc;
}

// Sixteen bytes of an activation row: zeros past the row's end (TAIL).
template <bool TAIL>
__device__ __forceinline__ v4i32 load_x(const uint8_t *x, int lane, int half, int first_row, int last_row, size_t row_bytes, int byte) {
    const v4i32 v = *reinterpret_cast<const v4i32 *>(x + tile_src<TAIL>(lane, half, first_row, last_row, row_bytes, byte));
    const v4i32 zero = {0, 0, 0, 0};
    return TAIL && byte + (lane & 7) * 16 >= (int)row_bytes ? zero : v;
}

// NLP: lines per wavefront and round.  WAVES: wavefronts per workgroup.  ROUNDS: 1, or 2 for
// K above 128*NLP*WAVES (the second round's bytes are requested line by line as the first
// round frees their registers; asking for all weight bytes at the start took 179 registers
// and measured slower), or 0: as many rounds as K takes, counted at run time (K above 10240).
// T: 16-row tiles of weight rows per workgroup (the activation tiles a wavefront fetched and
// rearranged serve all of them: at 16 rows they are two thirds of the bytes a wavefront asks for).
template <int NLP, int WAVES, int ROUNDS, int T, bool TAIL>
__global__ void __launch_bounds__(WAVES * 64)
gemv_w8a16_rows16_kernel(const Args a) {
    static_assert(T == 1 || ROUNDS == 1, "several tiles only in the single-round arrangement");
    constexpr Sum SUM = sum_of(TAIL, NLP, ROUNDS);
    extern __shared__ __align__(16) uint8_t lds[];
    float(*partial)[64][4] = reinterpret_cast<float(*)[64][4]>(lds);  // [T * WAVES][64][4]
    uint8_t *patches = lds + T * WAVES * 1024;                            // per wavefront: weights, activations

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4;
    const int n0 = blockIdx.x * (T * ROWS);
    const int lines = (a.K + LINE - 1) / LINE;
    uint8_t *wpatch = patches + wave * (PATCH_BYTES + XPATCH_BYTES), *xpatch = wpatch + PATCH_BYTES;
    const uint8_t *xbytes = reinterpret_cast<const uint8_t *>(a.x);
    auto line_of = [&](int r, int i) { return (r * NLP + i) * WAVES + wave; };

    // Activations first (L2 resident; memory answers in request order), then every weight byte.
    // An activation line is 256 bytes: parts 0 and 1, each fetched as two half tiles; rows past
    // M repeat the last one, their sums are dropped.
    v4i32 xr[NLP][4], wr[T][NLP][2];
    // One or two activation rows: every lane's row is one of two, so the MFMA arrangement (row
    // lane%16, bytes 64*kq .. +63 of the line) can be loaded as it is -- the requests collapse
    // onto a few cache lines -- and the LDS rearrangement is skipped.
    const bool direct_x = !TAIL && a.M <= 2;
    const uint8_t *xdirect = xbytes + (size_t)min(lane & 15, a.M - 1) * a.K * 2 + kq * 64;
    auto request_x = [&](int r, int i) {
        const int line = line_of(r, i);
        if (line >= lines) return;  // uniform per wavefront
        if (direct_x) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                xr[i][q] = *reinterpret_cast<const v4i32 *>(xdirect + line * 256 + q * 16);
            return;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            xr[i][q] = load_x<TAIL>(xbytes, lane, q & 1, 0, a.M - 1, (size_t)a.K * 2, line * 256 + (q >> 1) * 128);
    };
    auto request_w = [&](int r, int i) {
        const int line = line_of(r, i);
        if (line >= lines) return;
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                wr[t][i][h] = __builtin_nontemporal_load(reinterpret_cast<const v4i32 *>(
                    a.wq + tile_src<TAIL>(lane, h, n0 + t * ROWS, a.N - 1, a.K, line * LINE)));
    };
#pragma unroll
    for (int i = 0; i < NLP; ++i) request_x(0, i);
#pragma unroll
    for (int i = 0; i < NLP; ++i) request_w(0, i);
    // The row scale of the output this thread will finish, requested now, behind everything the
    // arithmetic waits for: asked for at the end it is a cold load under a saturated memory system
    // (1.4 us of every workgroup's 4.6 us, by in-kernel timestamps).
    float ws_out[T];
#pragma unroll
    for (int t = 0; t < T; ++t) ws_out[t] = a.ws[min(n0 + t * ROWS + (int)((threadIdx.x >> 2) & 15), a.N - 1)];

    // the accumulator of lane l holds (n = l%16, m = 4*kq + v), v = 0..3, per tile
    v4f32 acc[T], low[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = low[t] = v4f32{0.f, 0.f, 0.f, 0.f};
    const int rounds = ROUNDS > 0 ? ROUNDS : (lines + NLP * WAVES - 1) / (NLP * WAVES);
    constexpr int UNROLL = ROUNDS > 0 ? ROUNDS : 1;
#pragma unroll UNROLL
    for (int r = 0; r < rounds; ++r) {
        // activations into the MFMA arrangement: row lane%16, bytes 64*kq .. +63 of the line
#pragma unroll
        for (int i = 0; i < NLP; ++i) {
            if (direct_x || line_of(r, i) >= lines) break;
            uint8_t *p = xpatch + (lane >> 3) * XPITCH + (lane & 7) * 16;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<v4i32 *>(p + (q & 1) * 8 * XPITCH + (q >> 1) * 128) = xr[i][q];
            const uint8_t *t = xpatch + (lane & 15) * XPITCH + kq * 64;
#pragma unroll
            for (int q = 0; q < 4; ++q) xr[i][q] = *reinterpret_cast<const v4i32 *>(t + q * 16);
        }
        // weights: rearrange, widen, multiply
#pragma unroll
        for (int i = 0; i < NLP; ++i) {
            if (line_of(r, i) >= lines) break;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                tile_park(wpatch, lane, wr[t][i][0], wr[t][i][1]);
                const v4i32 w0 = tile_take(wpatch, lane, 2 * kq), w1 = tile_take(wpatch, lane, 2 * kq + 1);
                add_line<SUM>(acc[t], low[t], xr[i], w0, w1);
            }
            if (r + 1 < rounds) {
                request_x(r + 1, i);
                request_w(r + 1, i);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) *reinterpret_cast<v4f32 *>(&partial[t * WAVES + wave][lane][0]) = whole_sum<SUM>(acc[t], low[t]);
    __syncthreads();

    if (threadIdx.x < 256) {
        const int l = threadIdx.x >> 2, v = threadIdx.x & 3;
        const int m = 4 * (l >> 4) + v;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int n = n0 + t * ROWS + (l & 15);
            if (n < a.N && m < a.M) {
                float total = partial[t * WAVES][l][v];
#pragma unroll
                for (int wv = 1; wv < WAVES; ++wv) total += partial[t * WAVES + wv][l][v];
                a.y[(size_t)m * a.N + n] = (uint16_t)f32_to_bf16_bits(total * ws_out[t]);
            }
        }
    }
}

template <int NLP, int WAVES, int ROUNDS = 1, int T = 1>
int launch(const Args &a, hipStream_t st) {
    constexpr int LDS_BYTES = WAVES * (T * 1024 + PATCH_BYTES + XPATCH_BYTES);
    static std::atomic<uint64_t> devices[2];
    const auto run = [&](auto kernel, std::atomic<uint64_t> &done) {
        if (const int rc = reserve_lds(reinterpret_cast<const void *>(kernel), LDS_BYTES, done, "cmi_gemv_w8a16_mfma")) return rc;
        kernel<<<dim3((a.N + T * ROWS - 1) / (T * ROWS)), dim3(WAVES * 64), LDS_BYTES, st>>>(a);
        return check_launch("cmi_gemv_w8a16_mfma");
    };
    return a.K % LINE == 0 ? run(gemv_w8a16_rows16_kernel<NLP, WAVES, ROUNDS, T, false>, devices[0])
                           : run(gemv_w8a16_rows16_kernel<NLP, WAVES, ROUNDS, T, true>, devices[1]);
}


// 17..64 activation rows: the workgroup still asks for its 16 weight rows once and keeps them in
// registers in the MFMA arrangement (NLP*ROUNDS lines per wavefront); the activation rows go
// through in chunks of 16, each with the arithmetic of the kernel above -- so a row's bits are
// the same as in a 16-row call -- and only the activations (L2 resident) and the widening are
// paid again per chunk.  The activation registers hold NLP lines: with two rounds a chunk is two
// such batches, and the batch after the one in hand is requested line by line as its registers
// free up.  The partial tiles of all chunks meet in LDS behind one barrier.
constexpr int MAX_CHUNKS = 4;

// T: 16-row tiles of weight rows per workgroup (single-round arrangements only): every workgroup
// pulls all activation rows through L2 once per chunk, M * K * 2 bytes times N / (16 T) workgroups,
// which from three chunks up is what the launch waits for.
template <int NLP, int WAVES, int ROUNDS, int T, bool TAIL>
__global__ void __launch_bounds__(WAVES * 64)
gemv_w8a16_rows64_kernel(const Args a) {
    static_assert(T == 1 || ROUNDS == 1, "several tiles only in the single-round arrangement");
    constexpr Sum SUM = sum_of(TAIL, NLP, ROUNDS);
    extern __shared__ __align__(16) uint8_t lds[];
    float(*partial)[64][4] = reinterpret_cast<float(*)[64][4]>(lds);  // [(chunk * T + tile) * WAVES + wave][64][4]
    const int chunks = (a.M + ROWS - 1) / ROWS;
    uint8_t *patches = lds + chunks * T * WAVES * 1024;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4;
    const int n0 = blockIdx.x * (T * ROWS);
    const int lines = (a.K + LINE - 1) / LINE;
    uint8_t *wpatch = patches + wave * (PATCH_BYTES + XPATCH_BYTES), *xpatch = wpatch + PATCH_BYTES;
    const uint8_t *xbytes = reinterpret_cast<const uint8_t *>(a.x);
    auto line_of = [&](int r, int i) { return (r * NLP + i) * WAVES + wave; };

    v4i32 xr[NLP][4], wr[T][ROUNDS * NLP][2];
    auto request_x = [&](int c, int r, int i) {
        const int line = min(line_of(r, i), lines - 1);  // a slot past the last line is not used
#pragma unroll
        for (int q = 0; q < 4; ++q)
            xr[i][q] = load_x<TAIL>(xbytes, lane, q & 1, c * ROWS, a.M - 1, (size_t)a.K * 2, line * 256 + (q >> 1) * 128);
    };
#pragma unroll
    for (int i = 0; i < NLP; ++i) request_x(0, 0, i);
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r)
#pragma unroll
            for (int i = 0; i < NLP; ++i) {
                const int line = min(line_of(r, i), lines - 1);
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    wr[t][r * NLP + i][h] = __builtin_nontemporal_load(reinterpret_cast<const v4i32 *>(
                        a.wq + tile_src<TAIL>(lane, h, n0 + t * ROWS, a.N - 1, a.K, line * LINE)));
            }
    // the row scales of the outputs this thread will finish (n depends on the thread and the tile only),
    // requested behind the operands instead of cold at the end
    float ws_out[T];
#pragma unroll
    for (int t = 0; t < T; ++t) ws_out[t] = a.ws[min(n0 + t * ROWS + (int)((threadIdx.x >> 2) & 15), a.N - 1)];
    // weights into the MFMA arrangement, once
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < ROUNDS * NLP; ++i) {
            tile_park(wpatch, lane, wr[t][i][0], wr[t][i][1]);
            wr[t][i][0] = tile_take(wpatch, lane, 2 * kq);
            wr[t][i][1] = tile_take(wpatch, lane, 2 * kq + 1);
        }

#pragma unroll 1
    for (int c = 0; c < chunks; ++c) {
        v4f32 acc[T], low[T];
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t] = low[t] = v4f32{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            // this batch of activation lines into the MFMA arrangement: row lane%16, bytes 64*kq .. +63
#pragma unroll
            for (int i = 0; i < NLP; ++i) {
                uint8_t *p = xpatch + (lane >> 3) * XPITCH + (lane & 7) * 16;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<v4i32 *>(p + (q & 1) * 8 * XPITCH + (q >> 1) * 128) = xr[i][q];
                const uint8_t *t = xpatch + (lane & 15) * XPITCH + kq * 64;
#pragma unroll
                for (int q = 0; q < 4; ++q) xr[i][q] = *reinterpret_cast<const v4i32 *>(t + q * 16);
            }
#pragma unroll
            for (int i = 0; i < NLP; ++i) {
                if (line_of(r, i) < lines) {  // uniform per wavefront
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        v4i32 w0 = wr[t][r * NLP + i][0], w1 = wr[t][r * NLP + i][1];
                        // with two rounds or several tiles of weight registers the widened copies must
                        // not be kept across chunks (the compiler would hoist them out of the loop and spill)
                        if (ROUNDS > 1 || T > 1) asm volatile("" : "+v"(w0), "+v"(w1));
                        if constexpr (SUM != CHAIN) {
                            add_line<SUM>(acc[t], low[t], xr[i], w0, w1);
                        } else {
                            // (written out: through the function several tiles' accumulators are copied between registers, 64 rows
                            // of 4096 -> 14336 38.2 -> 38.8 us)
                            const uint32_t d[8] = {(uint32_t)w0.x, (uint32_t)w0.y, (uint32_t)w0.z, (uint32_t)w0.w,
                                                   (uint32_t)w1.x, (uint32_t)w1.y, (uint32_t)w1.z, (uint32_t)w1.w};
#pragma unroll
                            for (int s = 0; s < 4; ++s) {
                                uint32_t b[4];
                                widen4(d[2 * s], b[0], b[1]);
                                widen4(d[2 * s + 1], b[2], b[3]);
                                const v4i32 bw = {(int)b[0], (int)b[1], (int)b[2], (int)b[3]};
                                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xr[i][s]),
                                                                                 __builtin_bit_cast(bf16x8, bw), acc[t], 0, 0, 0);
                            }
                        }
                    }
                }
                // this line's activation registers are free: ask for the same slot of the next batch
                if (r + 1 < ROUNDS) request_x(c, r + 1, i);
                else if (c + 1 < chunks) request_x(c + 1, 0, i);
            }
        }
#pragma unroll
        for (int t = 0; t < T; ++t) *reinterpret_cast<v4f32 *>(&partial[(c * T + t) * WAVES + wave][lane][0]) = whole_sum<SUM>(acc[t], low[t]);
    }
    __syncthreads();

    for (int o = threadIdx.x; o < chunks * T * 256; o += WAVES * 64) {
        const int ct = o >> 8, c = ct / T, t = ct % T, l = (o >> 2) & 63, v = o & 3;
        const int n = n0 + t * ROWS + (l & 15), m = c * ROWS + 4 * (l >> 4) + v;
        if (n < a.N && m < a.M) {
            float total = partial[ct * WAVES][l][v];
#pragma unroll
            for (int wv = 1; wv < WAVES; ++wv) total += partial[ct * WAVES + wv][l][v];
            float scale = ws_out[0];
#pragma unroll
            for (int tt = 1; tt < T; ++tt) scale = t == tt ? ws_out[tt] : scale;
            a.y[(size_t)m * a.N + n] = (uint16_t)f32_to_bf16_bits(total * scale);
        }
    }
}

template <int NLP, int WAVES, int ROUNDS = 1, int T = 1>
int launch64(const Args &a, hipStream_t st) {
    constexpr int LDS_MAX = MAX_CHUNKS * T * WAVES * 1024 + WAVES * (PATCH_BYTES + XPATCH_BYTES);
    static std::atomic<uint64_t> devices[2];
    const int chunks = (a.M + ROWS - 1) / ROWS;
    const int lds_bytes = chunks * T * WAVES * 1024 + WAVES * (PATCH_BYTES + XPATCH_BYTES);
    const auto run = [&](auto kernel, std::atomic<uint64_t> &done) {
        if (const int rc = reserve_lds(reinterpret_cast<const void *>(kernel), LDS_MAX, done, "cmi_gemv_w8a16_mfma")) return rc;
        kernel<<<dim3((a.N + T * ROWS - 1) / (T * ROWS)), dim3(WAVES * 64), lds_bytes, st>>>(a);
        return check_launch("cmi_gemv_w8a16_mfma");
    };
    return a.K % LINE == 0 ? run(gemv_w8a16_rows64_kernel<NLP, WAVES, ROUNDS, T, false>, devices[0])
                           : run(gemv_w8a16_rows64_kernel<NLP, WAVES, ROUNDS, T, true>, devices[1]);
}

// 17..64 rows of more than 80 lines: the weight is asked for once, a round of NLP lines per wavefront at a time, and each
// round's lines meet every chunk of 16 activation rows before the next round's take their registers, so a row's bits are those of a
// 16-row call (its lines in the same order).  A launch per 16 rows, which this replaces, read the weight up to four
// times: 13824 -> 5120, 17 rows 50.2 -> 46.1 us, 32 rows 56.8 -> 46.8, 63 rows 112 -> 69.
template <int NLP, int WAVES, int CHUNKS, bool TAIL>
__global__ void __launch_bounds__(WAVES * 64)
gemv_w8a16_rows64_long_kernel(const Args a) {
    constexpr Sum SUM = sum_of(TAIL, NLP, 0);
    extern __shared__ __align__(16) uint8_t lds[];
    float(*partial)[64][4] = reinterpret_cast<float(*)[64][4]>(lds);  // [CHUNKS * WAVES][64][4]
    uint8_t *patches = lds + CHUNKS * WAVES * 1024;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4;
    const int n0 = blockIdx.x * ROWS;
    const int lines = (a.K + LINE - 1) / LINE, rounds = (lines + NLP * WAVES - 1) / (NLP * WAVES);
    uint8_t *wpatch = patches + wave * (PATCH_BYTES + XPATCH_BYTES), *xpatch = wpatch + PATCH_BYTES;
    const uint8_t *xbytes = reinterpret_cast<const uint8_t *>(a.x);
    auto line_of = [&](int r, int i) { return (r * NLP + i) * WAVES + wave; };

    v4i32 xr[NLP][4], wr[NLP][2];
    auto request_x = [&](int c, int r, int i) {
        const int line = min(line_of(r, i), lines - 1);  // a slot past the last line is not used
#pragma unroll
        for (int q = 0; q < 4; ++q)
            xr[i][q] = load_x<TAIL>(xbytes, lane, q & 1, c * ROWS, a.M - 1, (size_t)a.K * 2, line * 256 + (q >> 1) * 128);
    };
    auto request_w = [&](int r, int i) {
        const int line = min(line_of(r, i), lines - 1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
            wr[i][h] = __builtin_nontemporal_load(
                reinterpret_cast<const v4i32 *>(a.wq + tile_src<TAIL>(lane, h, n0, a.N - 1, a.K, line * LINE)));
    };
#pragma unroll
    for (int i = 0; i < NLP; ++i) request_x(0, 0, i);
#pragma unroll
    for (int i = 0; i < NLP; ++i) request_w(0, i);
    const float ws_out = a.ws[min(n0 + (int)((threadIdx.x >> 2) & 15), a.N - 1)];

    v4f32 acc[CHUNKS], low[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) acc[c] = low[c] = v4f32{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int r = 0; r < rounds; ++r) {
#pragma unroll
        for (int i = 0; i < NLP; ++i) {  // weights into the MFMA arrangement, once
            tile_park(wpatch, lane, wr[i][0], wr[i][1]);
            wr[i][0] = tile_take(wpatch, lane, 2 * kq);
            wr[i][1] = tile_take(wpatch, lane, 2 * kq + 1);
        }
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
#pragma unroll
            for (int i = 0; i < NLP; ++i) {
                uint8_t *p = xpatch + (lane >> 3) * XPITCH + (lane & 7) * 16;
#pragma unroll
                for (int q = 0; q < 4; ++q) *reinterpret_cast<v4i32 *>(p + (q & 1) * 8 * XPITCH + (q >> 1) * 128) = xr[i][q];
                const uint8_t *t = xpatch + (lane & 15) * XPITCH + kq * 64;
#pragma unroll
                for (int q = 0; q < 4; ++q) xr[i][q] = *reinterpret_cast<const v4i32 *>(t + q * 16);
            }
#pragma unroll
            for (int i = 0; i < NLP; ++i) {
                if (line_of(r, i) < lines) {  // uniform per wavefront
                    v4i32 w0 = wr[i][0], w1 = wr[i][1];
                    asm volatile("" : "+v"(w0), "+v"(w1));  // widened for each chunk: all copies at once would spill
                    add_line<SUM>(acc[c], low[c], xr[i], w0, w1);
                }
                if (c + 1 < CHUNKS) {
                    request_x(c + 1, r, i);
                } else if (r + 1 < rounds) {
                    request_x(0, r + 1, i);
                    request_w(r + 1, i);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) *reinterpret_cast<v4f32 *>(&partial[c * WAVES + wave][lane][0]) = whole_sum<SUM>(acc[c], low[c]);
    __syncthreads();

    for (int o = threadIdx.x; o < CHUNKS * 256; o += WAVES * 64) {
        const int c = o >> 8, l = (o >> 2) & 63, v = o & 3;
        const int n = n0 + (l & 15), m = c * ROWS + 4 * (l >> 4) + v;
        if (n < a.N && m < a.M) {
            float total = partial[c * WAVES][l][v];
#pragma unroll
            for (int wv = 1; wv < WAVES; ++wv) total += partial[c * WAVES + wv][l][v];
            a.y[(size_t)m * a.N + n] = (uint16_t)f32_to_bf16_bits(total * ws_out);
        }
    }
}

template <int CHUNKS>
int launch64_long(const Args &a, hipStream_t st) {
    constexpr int NLP = 5, WAVES = 8, LDS_BYTES = CHUNKS * WAVES * 1024 + WAVES * (PATCH_BYTES + XPATCH_BYTES);
    static std::atomic<uint64_t> devices[2];
    const auto run = [&](auto kernel, std::atomic<uint64_t> &done) {
        if (const int rc = reserve_lds(reinterpret_cast<const void *>(kernel), LDS_BYTES, done, "cmi_gemv_w8a16_mfma")) return rc;
        kernel<<<dim3((a.N + ROWS - 1) / ROWS), dim3(WAVES * 64), LDS_BYTES, st>>>(a);
        return check_launch("cmi_gemv_w8a16_mfma");
    };
    return a.K % LINE == 0 ? run(gemv_w8a16_rows64_long_kernel<NLP, WAVES, CHUNKS, false>, devices[0])
                           : run(gemv_w8a16_rows64_long_kernel<NLP, WAVES, CHUNKS, true>, devices[1]);
}

}  // namespace

namespace {

int run_mfma(const int8_t *wq, const float *ws, const void *x, void *y, int M, int N, int K, void *stream) {
    Args a;
    a.wq = wq;
    a.ws = ws;
    a.x = static_cast<const uint16_t *>(x);
    a.y = static_cast<uint16_t *>(y);
    a.M = M;
    a.N = N;
    a.K = K;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int lines = (K + LINE - 1) / LINE;
    if (lines > 80) {
        // rows longer than two rounds of registers hold: as many rounds as it takes
        return M <= 16 ? launch<5, 8, 0>(a, st) : M <= 32 ? launch64_long<2>(a, st) : M <= 48 ? launch64_long<3>(a, st) : launch64_long<4>(a, st);
    }
    if (M > ROWS) {
        if (lines <= 8) return launch64<2, 4>(a, st);
        if (lines <= 20 && (N + ROWS - 1) / ROWS > 2048) return launch64<5, 4>(a, st);
        // Several weight tiles per workgroup: the activation rows a workgroup pulls through L2 per
        // chunk then serve 32 or 48 weight rows.  A launch takes (rounds of 256 workgroups) x (time of
        // a workgroup), and a workgroup of T tiles about (2 T + 1) units -- fitted to 2560 -> 9728 /
        // 6144 / 19456 and 4096 -> 11008 / 14336 / 5120 at 32..64 rows, where the best T follows this
        // count every time (64 rows of 2560 -> 9728: 21.9 -> 16.6 us with three tiles, 2560 -> 6144
        // 15.2 -> 12.6 with two, 4096 -> 14336 44 -> 39 with two; three is what LDS holds).
        const int tiles = (N + ROWS - 1) / ROWS;
        int T = 1, best = 1 << 30;
        for (int t = 1; t <= 3; ++t) {
            const int cost = ((tiles + t - 1) / t + 255) / 256 * (2 * t + 1);
            if (cost < best) best = cost, T = t;
        }
        if (lines <= 24) return T == 3 ? launch64<3, 8, 1, 3>(a, st) : T == 2 ? launch64<3, 8, 1, 2>(a, st) : launch64<3, 8>(a, st);
        if (lines <= 40) return T == 3 ? launch64<5, 8, 1, 3>(a, st) : T == 2 ? launch64<5, 8, 1, 2>(a, st) : launch64<5, 8>(a, st);
        return launch64<5, 8, 2>(a, st);
    }
    // eight wavefronts (shorter chains of dependent steps) up to 2048 workgroups, four beyond
    // (2560 -> 151936: 72 us against 84)
    // From four rows and 300 tiles of weight rows up, a workgroup owns two tiles: the activation
    // tiles its wavefronts fetched and rearranged serve both (16 rows: 2560 -> 6144 6.9 -> 6.3 us,
    // 2560 -> 151936 86 -> 78 us; with fewer rows or tiles one tile per workgroup stays faster).
    const int tiles = (N + ROWS - 1) / ROWS;
    const bool two = M >= 4 && tiles >= 300;
    if (lines <= 8) return launch<2, 4>(a, st);
    if (lines <= 20 && tiles > 2048) return two ? launch<5, 4, 1, 2>(a, st) : launch<5, 4>(a, st);
    if (lines <= 24) return two ? launch<3, 8, 1, 2>(a, st) : launch<3, 8>(a, st);
    if (lines <= 40) return two ? launch<5, 8, 1, 2>(a, st) : launch<5, 8>(a, st);
    return launch<5, 8, 2>(a, st);
}

}  // namespace

extern "C" int cmi_gemv_w8a16_mfma(const int8_t *wq, const float *ws, const void *x, void *y, int M, int N,
                                   int K, void *stream) {
    CMI_REQUIRE(wq && ws && x && y, CMI_E_ARG, "cmi_gemv_w8a16_mfma: null pointer");
    CMI_REQUIRE(M >= 1 && M <= MAX_CHUNKS * ROWS, CMI_E_UNSUPPORTED, "cmi_gemv_w8a16_mfma: M=%d outside 1..64", M);
    CMI_REQUIRE(N >= 1 && K >= 1, CMI_E_ARG, "cmi_gemv_w8a16_mfma: bad shape N=%d K=%d", N, K);
    CMI_REQUIRE(K % LINE == 0, CMI_E_UNSUPPORTED, "cmi_gemv_w8a16_mfma: K=%d is not a multiple of 128 (use cmi_gemv_w8a16)", K);
    CMI_REQUIRE(aligned(wq, 16) && aligned(x, 16) && aligned(y, 2) && aligned(ws, 4), CMI_E_ARG,
                "cmi_gemv_w8a16_mfma: wq and x must be 16-byte aligned");
    return run_mfma(wq, ws, x, y, M, N, K, stream);
}

namespace {

// Few outputs of long rows that end inside a line: rows below this go to the kernels of cmi_gemv_w8a16.  A wavefront of this file takes every
// eighth line of its 16 weight rows, a chain that grows with K alone.  The line was measured against a kernel that is gone (5 rows of 12304 -> 300
// 10.9 us, 15.6 here).  The batch kernels in its place are the faster ones up to eight rows on both sides of it (5 rows of 12304 -> 1200
// 8.9 us, 16.4 here, of 16400 -> 300 10.4 / 19.0; 8 rows of 9200 -> 300 6.1 / 12.3, of 16368 -> 800 10.5 / 19.9; 9 rows of 12304 -> 300
// 15.5 / 16.1, of 2624 -> 9728 12.5 / 11.7); it stays: rows beyond it agree in their bits with
// those of a call of sixteen.
int rows_from(int N, int K) {
    if (K % LINE == 0 || K <= 8192) return 1;
    if (K <= 16384) return N <= 512 ? (K >= 12288 ? 9 : 7) : N <= 832 ? 7 : N <= 1024 ? 6 : 1;
    return K > 20480 && N <= 512 ? 6 : 1;
}

}  // namespace

extern "C" int cmi_linear_w8a16_rows(const int8_t *wq, const float *ws, const void *x, void *y, int M, int N, int K, void *stream) {
    CMI_REQUIRE(M >= 0 && N >= 1 && K >= LINE, CMI_E_ARG, "cmi_linear_w8a16_rows: bad shape M=%d N=%d K=%d", M, N, K);
    // (the bound of cmi_gemv_w8a16, which takes such rows one by one)
    CMI_REQUIRE(K % 16 == 0 && K <= 1 << 18, CMI_E_UNSUPPORTED, "cmi_linear_w8a16_rows: K=%d is not a multiple of 16 up to 262144", K);
    if (M == 0) return CMI_OK;
    CMI_REQUIRE(wq && ws && x && y, CMI_E_ARG, "cmi_linear_w8a16_rows: null pointer");
    CMI_REQUIRE(aligned(wq, 16) && aligned(x, 16) && aligned(y, 2) && aligned(ws, 4), CMI_E_ARG,
                "cmi_linear_w8a16_rows: wq and x must be 16-byte aligned");
    if (M < rows_from(N, K)) return cmi_gemv_w8a16(wq, ws, x, y, M, N, K, stream);
    const uint16_t *xr = static_cast<const uint16_t *>(x);
    uint16_t *yr = static_cast<uint16_t *>(y);
    for (int lo = 0; lo < M; lo += MAX_CHUNKS * ROWS) {
        const int m = M - lo < MAX_CHUNKS * ROWS ? M - lo : MAX_CHUNKS * ROWS;
        if (const int rc = run_mfma(wq, ws, xr + (size_t)lo * K, yr + (size_t)lo * N, m, N, K, stream)) return rc;
    }
    return CMI_OK;
}
