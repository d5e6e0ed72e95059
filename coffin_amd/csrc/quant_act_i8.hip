// Per-token symmetric int8 activation quantiser (bf16 in, int8 + fp32 scale out).
//
// One workgroup per row, or a part of a wavefront per short row.  The row is read once from
// HBM with 16-byte loads and kept in registers across the absmax reduction when it fits (VPT
// vectors per thread), so HBM traffic is the algorithmic 2 B in + 1 B out per element.
// The scale and the rounding follow the torch spec bit for bit: IEEE fp32
// division by the scale (not a reciprocal multiply), round-half-even, clamp.
#include "quant_math.hpp"

namespace {

using namespace cmi;

constexpr int QUANT_THREADS = 256;

// Block-wide max of non-negative values; every thread returns the result.
__device__ __forceinline__ float block_max(float v, float *smem) {
    v = wave_max_to_lane63(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63) smem[wave] = v;
    __syncthreads();
    float r = smem[0];
#pragma unroll
    for (int i = 1; i < QUANT_THREADS / 64; ++i) r = fmaxf(r, smem[i]);
    return r;
}

// How a row of K elements is read, eight at a time.  Whole: K % 8 == 0, rows 16-byte aligned (PADDED: rows of q are longer).
// Ragged: any K, any alignment of two bytes (a vector load needs no more on gfx950); the elements past K of the last vector are zeros and
// are not read.
template <bool P>
struct Whole {
    static constexpr bool PADDED = P;
    typedef uint4 T;
    const uint4 *x;
    int nvec;
    __device__ __forceinline__ uint4 load(int row, int idx) const {
        return idx < nvec ? x[(size_t)row * nvec + idx] : make_uint4(0, 0, 0, 0);
    }
    __device__ __forceinline__ int vecs() const { return nvec; }
};
struct Ragged {
    static constexpr bool PADDED = true;
    typedef uint16_t T;
    const uint16_t *x;
    int K;
    __device__ __forceinline__ uint4 load(int row, int idx) const {
        const uint16_t *p = x + (size_t)row * K + 8 * idx;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (8 * idx + 8 <= K) {
            __builtin_memcpy(&v, p, 16);
        } else if (8 * idx < K) {
            uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 7; ++e)
                if (8 * idx + e < K) w[e / 2] |= (uint32_t)p[e] << (16 * (e & 1));
            v = make_uint4(w[0], w[1], w[2], w[3]);
        }
        return v;
    }
    __device__ __forceinline__ int vecs() const { return (K + 7) / 8; }
};

// VPT > 0: the row fits in VPT vectors per thread and stays in registers; VPT == 0: generic, second pass re-reads.
// Rows of q have q_vecs vectors where they are padded; past the row's own they are zeros, as quant8 makes of zeros under every scale
// (rows padded to whole groups of an int4 weight).  Rows that are not know one count, and it and the row pointer are arguments of
// their own: with two counts, and a struct among the arguments, every launch took 1 .. 3 % longer (16 x 2560 2.49 -> 2.51 us, 65536 x 128
// 6.95 -> 7.15).  n: SRC's second member.
// zero / n_zero: a few ints of the caller's that the first workgroup clears on the way (the
// arrival counters of a split-K GEMM that follows in the stream), or null / 0.
template <int VPT, typename SRC>
__global__ void __launch_bounds__(QUANT_THREADS)
quant_act_i8_vec(const typename SRC::T *__restrict__ x_rows, uint2 *__restrict__ q, float *__restrict__ s, int n, int *__restrict__ zero,
                 int n_zero, int q_vecs) {
    const SRC x{x_rows, n};
    __shared__ float smem[QUANT_THREADS / 64];
    const int row = blockIdx.x;
    if (row == 0)
        for (int i = threadIdx.x; i < n_zero; i += QUANT_THREADS) zero[i] = 0;
    const int nvec = x.vecs(), pvec = SRC::PADDED ? q_vecs : nvec;
    uint2 *qr = q + (size_t)row * pvec;
    float amax = 0.f;
    if constexpr (VPT > 0) {
        uint4 v[VPT];
#pragma unroll
        for (int i = 0; i < VPT; ++i) v[i] = x.load(row, threadIdx.x + i * QUANT_THREADS);
#pragma unroll
        for (int i = 0; i < VPT; ++i) amax = absmax8(v[i], amax);
        amax = block_max(amax, smem);
        const RowScale rs = row_scale(amax);
        const float sc = rs.sc;
        if (threadIdx.x == 0) s[row] = sc;
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int idx = threadIdx.x + i * QUANT_THREADS;
            if (idx < pvec) qr[idx] = quant8(v[i], rs);
        }
    } else {
        for (int idx = threadIdx.x; idx < nvec; idx += QUANT_THREADS) amax = absmax8(x.load(row, idx), amax);
        amax = block_max(amax, smem);
        const RowScale rs = row_scale(amax);
        const float sc = rs.sc;
        if (threadIdx.x == 0) s[row] = sc;
        for (int idx = threadIdx.x; idx < pvec; idx += QUANT_THREADS) qr[idx] = quant8(x.load(row, idx), rs);
    }
}

// Max over the LANES lanes of a row's group; every lane of the group returns it.
template <int LANES>
__device__ __forceinline__ float group_max(float v) {
    static_assert(LANES == 8 || LANES == 16 || LANES == 32 || LANES == 64, "a power of two from 8");
    v = fmaxf(v, dpp_f32<0xB1, 0xf>(v));   // l ^ 1
    v = fmaxf(v, dpp_f32<0x4E, 0xf>(v));   // l ^ 2
    v = fmaxf(v, dpp_f32<0x141, 0xf>(v));  // the other quad of the half row
    if constexpr (LANES >= 16) v = fmaxf(v, dpp_f32<0x140, 0xf>(v));  // the other half of the row
    typedef unsigned u32x2_swap __attribute__((ext_vector_type(2)));
    if constexpr (LANES >= 32) {
        const u32x2_swap r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
    }
    if constexpr (LANES == 64) {
        const u32x2_swap r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
    }
    return v;
}

// Short rows (cache rows of 64 .. 576 elements): LANES lanes own a row, VPT vectors each, so a wavefront
// carries 64 / LANES rows at a time, R times, and reduces them without LDS or a barrier.  A workgroup per
// row left 15 of 16 lanes idle at 128 elements and was bound by the rate at which workgroups are started.
// Cold operands in a graph: 16384 x 128 13.1 -> 3.6 us (1.7 TB/s; 1.6 us of it are the launch), 65536 x 128
// 45.9 -> 7.8 us (3.2 TB/s), 8192 x 512 9.0 -> 5.6 us, 3000 x 1024 6.1 -> 4.5 us.  Same arithmetic, same bits.
template <int LANES, int VPT, int R, typename SRC>
__global__ void __launch_bounds__(QUANT_THREADS)
quant_act_i8_rows(const typename SRC::T *__restrict__ x_rows, uint2 *__restrict__ q, float *__restrict__ s, int n, int rows,
                  int *__restrict__ zero, int n_zero, int q_vecs) {
    const SRC x{x_rows, n};
    constexpr int STEP = QUANT_THREADS / LANES;
    const int pvec = SRC::PADDED ? q_vecs : x.vecs();
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < n_zero; i += QUANT_THREADS) zero[i] = 0;
    const int l = threadIdx.x % LANES;
    const int row0 = blockIdx.x * (STEP * R) + threadIdx.x / LANES;
    uint4 v[R][VPT];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = min(row0 + r * STEP, rows - 1);
#pragma unroll
        for (int i = 0; i < VPT; ++i) v[r][i] = x.load(row, l + i * LANES);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = row0 + r * STEP;
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < VPT; ++i) amax = absmax8(v[r][i], amax);
        const RowScale rs = row_scale(group_max<LANES>(amax));
        if (row >= rows) continue;  // a whole group of lanes; the next rows lie further on
        if (l == 0) s[row] = rs.sc;
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int idx = l + i * LANES;
            if (idx < pvec) q[(size_t)row * pvec + idx] = quant8(v[r][i], rs);
        }
    }
}

// Any K, any alignment of x and q.
__global__ void __launch_bounds__(QUANT_THREADS)
quant_act_i8_scalar(const uint16_t *__restrict__ x, int8_t *__restrict__ q,
                    float *__restrict__ s, int K, int *__restrict__ zero, int n_zero) {
    __shared__ float smem[QUANT_THREADS / 64];
    const int row = blockIdx.x;
    if (row == 0)
        for (int i = threadIdx.x; i < n_zero; i += QUANT_THREADS) zero[i] = 0;
    const uint16_t *xr = x + (size_t)row * K;
    int8_t *qr = q + (size_t)row * K;
    float amax = 0.f;
    for (int k = threadIdx.x; k < K; k += QUANT_THREADS)
        amax = fmaxf(amax, fabsf(bf16_bits_to_f32(xr[k])));
    amax = block_max(amax, smem);
    const RowScale rs = row_scale(amax);
    const float sc = rs.sc;
    if (threadIdx.x == 0) s[row] = sc;
    for (int k = threadIdx.x; k < K; k += QUANT_THREADS)
        qr[k] = (int8_t)quant1(bf16_bits_to_f32(xr[k]), rs);
}

// The vector kernels' launch: rows of pvec vectors in q.
template <typename SRC>
void launch_vectors(const void *x_rows, int n, int8_t *q, float *s, int M, int pvec, int *zero, int n_zero, hipStream_t st) {
    const dim3 grid(M), block(QUANT_THREADS);
    const auto *x = static_cast<const typename SRC::T *>(x_rows);
    uint2 *qv = reinterpret_cast<uint2 *>(q);
    const int vpt = (pvec + QUANT_THREADS - 1) / QUANT_THREADS;
    const auto rows_launch = [&](auto kernel, int rows_per_block) {
        kernel<<<dim3((M + rows_per_block - 1) / rows_per_block), block, 0, st>>>(x, qv, s, n, M, zero, n_zero, pvec);
    };
    const auto row_launch = [&](auto kernel) { kernel<<<grid, block, 0, st>>>(x, qv, s, n, zero, n_zero, pvec); };
    // Up to 1024 elements a wavefront or less owns a row.  Two rows per lane group once one each would
    // be more than two workgroups per CU: twice the bytes in flight per wavefront (65536 x 128: 9.8 ->
    // 7.8 us; below that the second row only lengthens the launch, 2048 x 576: 3.3 -> 3.9 us).
    // Two vectors a lane pay from 257 rows on; below, a workgroup per row is shorter (1 x 576 1.99 us against 2.16,
    // 256 x 576 2.40 against 2.55, 512 x 576 5 % the other way).
    const auto many = [&](int rows_per_block) { return M > 512 * rows_per_block; };
    if (pvec <= 8) many(32) ? rows_launch(quant_act_i8_rows<8, 1, 2, SRC>, 64) : rows_launch(quant_act_i8_rows<8, 1, 1, SRC>, 32);
    else if (pvec <= 16) many(16) ? rows_launch(quant_act_i8_rows<16, 1, 2, SRC>, 32) : rows_launch(quant_act_i8_rows<16, 1, 1, SRC>, 16);
    else if (pvec <= 32) many(8) ? rows_launch(quant_act_i8_rows<32, 1, 2, SRC>, 16) : rows_launch(quant_act_i8_rows<32, 1, 1, SRC>, 8);
    else if (pvec <= 64) many(4) ? rows_launch(quant_act_i8_rows<64, 1, 2, SRC>, 8) : rows_launch(quant_act_i8_rows<64, 1, 1, SRC>, 4);
    else if (pvec <= 128 && M > QUANT_THREADS) rows_launch(quant_act_i8_rows<64, 2, 1, SRC>, 4);
    else if (vpt <= 1) row_launch(quant_act_i8_vec<1, SRC>);
    else if (vpt <= 2) row_launch(quant_act_i8_vec<2, SRC>);
    else if (vpt <= 4) row_launch(quant_act_i8_vec<4, SRC>);
    else if (vpt <= 8) row_launch(quant_act_i8_vec<8, SRC>);
    else if (vpt <= 16) row_launch(quant_act_i8_vec<16, SRC>);
    else row_launch(quant_act_i8_vec<0, SRC>);
}

}  // namespace

int cmi::quant_act_i8_and_clear(const void *x, int8_t *q, float *s, int M, int K, int *zero, int n_zero,
                                void *stream) {
    CMI_REQUIRE(M >= 0 && K > 0, CMI_E_ARG, "cmi_quant_act_i8: bad shape M=%d K=%d", M, K);
    if (M == 0) return CMI_OK;  // an empty batch has no storage to point at
    CMI_REQUIRE(x && q && s, CMI_E_ARG, "cmi_quant_act_i8: null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (K % 8 == 0 && aligned(x, 16) && aligned(q, 8))
        launch_vectors<Whole<false>>(x, K / 8, q, s, M, K / 8, zero, n_zero, st);
    else
        quant_act_i8_scalar<<<dim3(M), dim3(QUANT_THREADS), 0, st>>>(static_cast<const uint16_t *>(x), q, s, K, zero, n_zero);
    return check_launch("cmi_quant_act_i8");
}

// Rows of an int4 weight whose K is not whole groups: the vector kernels as well, whatever K is, since the padded rows
// of q are whole vectors.  Element by element, each read twice, the projection behind it included: 9664 -> 2560, one
// row 15.2 -> 8.9 us, 16 rows 18.8 -> 12.5, 8000 rows 359 -> 280; 100 rows of 2497 -> 9000 21.7 -> 17.5.
int cmi::quant_act_i8_padded(const void *x, int8_t *q, float *s, int M, int K, int ldq, void *stream) {
    if (ldq == K) return quant_act_i8_and_clear(x, q, s, M, K, nullptr, 0, stream);
    CMI_REQUIRE(M >= 0 && K > 0 && ldq > K && ldq % 8 == 0, CMI_E_ARG, "cmi_quant_act_i8: bad shape M=%d K=%d pitch=%d", M, K, ldq);
    if (M == 0) return CMI_OK;
    CMI_REQUIRE(x && q && s, CMI_E_ARG, "cmi_quant_act_i8: null pointer");
    CMI_REQUIRE(aligned(q, 8), CMI_E_ARG, "cmi_quant_act_i8: rows must be 8-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (K % 8 == 0 && aligned(x, 16)) launch_vectors<Whole<true>>(x, K / 8, q, s, M, ldq / 8, nullptr, 0, st);
    else launch_vectors<Ragged>(x, K, q, s, M, ldq / 8, nullptr, 0, st);
    return check_launch("cmi_quant_act_i8");
}

extern "C" int cmi_quant_act_i8(const void *x, int8_t *q, float *s, int M, int K, void *stream) {
    return cmi::quant_act_i8_and_clear(x, q, s, M, K, nullptr, 0, stream);
}
