// Producers of quantised activations fused with the op in front of them:
//   silu_mul_quant   out = bf16(silu(gate)) * up (bf16), then the per-token int8 quantiser
//   rms_norm_i8      y = rms_norm(x) * w (bf16), then the quantiser
//   add_rms_norm_i8  x += add (bf16, written back), then the same
// Each equals "the op writing bf16, then cmi_quant_act_i8 reading it back" bit for bit: the
// absmax is taken over the narrowed bf16 values and the rounding is quant_math.hpp's.  What
// the fusion saves is the bf16 round trip through HBM in front of every W8A8 / W4A8
// projection (5 B per element instead of 9 for silu_mul_quant with the bf16 copy, 3 without).
//
// One workgroup per row; the row's results stay in registers across the absmax reduction
// (VPT 16-byte vectors per thread), so every input is read once and every output written once.
#include "quant_math.hpp"
#include <algorithm>

namespace {

using namespace cmi;

constexpr int THREADS = 256;       // per row when there are rows enough to fill the chip
constexpr int MAX_THREADS = 1024;  // per row for a few rows: the row is the only parallelism there is
constexpr int FEW_ROWS = 256;      // up to this many rows a row gets as many threads as it has vectors

typedef unsigned u32x2_swap __attribute__((ext_vector_type(2)));

// Butterfly sum of doubles over the wavefront, in every lane (DPP moves and row swaps: a shuffle is an LDS
// round trip).  The addends are sums of squares of bf16 values, which double holds exactly for any realistic
// row, so the order does not matter.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const u32x2_swap u = __builtin_bit_cast(u32x2_swap, v);
    const u32x2_swap r = {(unsigned)dpp_i32<CTRL, 0xf>((int)u.x), (unsigned)dpp_i32<CTRL, 0xf>((int)u.y)};
    return __builtin_bit_cast(double, r);
}

__device__ __forceinline__ double wave_sum(double v) {
    v += dpp_f64<0xB1>(v);   // l ^ 1
    v += dpp_f64<0x4E>(v);   // l ^ 2
    v += dpp_f64<0x141>(v);  // the other quad of the half row
    v += dpp_f64<0x140>(v);  // the other half of the row
    {
        const u32x2_swap u = __builtin_bit_cast(u32x2_swap, v);
        const u32x2_swap lo = __builtin_amdgcn_permlane16_swap(u.x, u.x, false, false);
        const u32x2_swap hi = __builtin_amdgcn_permlane16_swap(u.y, u.y, false, false);
        const u32x2_swap a = {lo.x, hi.x}, b = {lo.y, hi.y};
        v = __builtin_bit_cast(double, a) + __builtin_bit_cast(double, b);
    }
    const u32x2_swap u = __builtin_bit_cast(u32x2_swap, v);
    const u32x2_swap lo = __builtin_amdgcn_permlane32_swap(u.x, u.x, false, false);
    const u32x2_swap hi = __builtin_amdgcn_permlane32_swap(u.y, u.y, false, false);
    const u32x2_swap a = {lo.x, hi.x}, b = {lo.y, hi.y};
    return __builtin_bit_cast(double, a) + __builtin_bit_cast(double, b);
}

// Over the workgroup; `smem` (one slot per wavefront) is used by one reduction of a launch only.
__device__ __forceinline__ float block_max(float v, float *smem) {
    v = wave_max_to_lane63(v);
    if ((threadIdx.x & 63) == 63) smem[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = smem[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) r = fmaxf(r, smem[i]);
    return r;
}

__device__ __forceinline__ double block_sum(double v, double *smem) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = smem[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) r += smem[i];
    return r;
}

// A launch holds fewer than 2^32 threads: more rows than that allows run in slices of whole rows.
// launch(first row, rows) is called for each.
template <typename LAUNCH>
void in_row_slices(int M, long threads_per_row, LAUNCH launch) {
    const long step = std::max(1L, INT32_MAX / threads_per_row);
    for (long lo = 0; lo < M; lo += step) launch(lo, (int)std::min(step, M - lo));
}

// ----------------------------------------------------------------- silu

// silu(g) for a bf16 g as the fp32 value whose narrowing is the result: g / (1 + exp(-g))
// evaluated in fp32 with exp rounded once from its exact value.  The fast evaluation --
// exp(-g) = 2^p (1 + r) with p = -g log2(e) rounded and r = -g - p ln 2, v_exp_f32, v_rcp_f32 --
// is within 3 fp32 steps of that value for every bf16 g with |g| < 64 (measured over all of
// them); it is used unless it sits within 4 steps of a bf16 rounding boundary, where those few
// steps could change the narrowing: such inputs (0.014 %) and |g| >= 64, infinities and NaN take
// the double-precision exp and the correctly rounded division.
__device__ __forceinline__ float silu_exact_f32(float g) {
    const float e = (float)exp((double)(-g));
    return __fdiv_rn(g, 1.f + e);
}

__device__ __forceinline__ float silu_fast_f32(float g) {
    constexpr float LOG2E = 1.44269502e+00f, LN2 = 0.693147182f, LN2_LO = -1.90465421e-09f;
    const float p = __fmul_rn(-g, LOG2E);
    const float r = __fmaf_rn(-p, LN2_LO, __fmaf_rn(-p, LN2, -g));  // -g - p ln 2
    const float ep = __builtin_amdgcn_exp2f(p);
    return __fmul_rn(g, __builtin_amdgcn_rcpf(__fadd_rn(1.f, __fmaf_rn(ep, r, ep))));
}

// How far `fast` is past the lower edge of the window around a bf16 rounding boundary (in units of
// 2^16, the unsigned difference): at most NEAR inside the window.
constexpr uint32_t NEAR = 8u << 16;
__device__ __forceinline__ uint32_t boundary_offset(float fast) { return (__float_as_uint(fast) << 16) - ((0x8000u - 4u) << 16); }

__device__ __forceinline__ float silu_f32(float g) {
    const float fast = silu_fast_f32(g);
    return !(fabsf(g) < 64.f) || boundary_offset(fast) <= NEAR ? silu_exact_f32(g) : fast;
}

__device__ __forceinline__ uint32_t silu_bf16_bits(float g) { return pack2_bf16(silu_f32(g), 0.f) & 0xffffu; }

// product of two bf16 values as torch forms it: one fp32 multiply, one narrowing
__device__ __forceinline__ uint32_t mul_bf16_bits(uint32_t a_bits, float b) {
    return pack2_bf16(__fmul_rn(bf16_bits_to_f32(a_bits), b), 0.f) & 0xffffu;
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
constexpr unsigned short BF16_64 = 0x4280;  // 64 as bf16

// eight elements: bf16(bf16(silu(g)) * u), two per dword.  The fast evaluations of all eight run
// without a branch between them (their exponentials and reciprocals overlap) and one test per vector
// finds out whether any of them needs the exact one: with a branch per element 2048 x 9728 took
// 34 us, bound by the latency of one element's chain after the other.
__device__ __forceinline__ uint4 silu_mul8(const uint4 &g, const uint4 &u) {
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
    float x[8], f[8];
    uint32_t near = ~0u;
    u16x2 big = {0, 0};  // the largest magnitudes as bits, so that NaN counts as large
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        x[i] = i & 1 ? __uint_as_float(gw[i / 2] & 0xffff0000u) : bf16_bits_to_f32(gw[i / 2] & 0xffffu);
        f[i] = silu_fast_f32(x[i]);
        near = min(near, boundary_offset(f[i]));
        if (i & 1) big = __builtin_elementwise_max(big, __builtin_bit_cast(u16x2, gw[i / 2] & 0x7fff7fffu));
    }
    if (__builtin_expect(near <= NEAR || max(big.x, big.y) >= BF16_64, 0)) {
        uint32_t todo = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (!(fabsf(x[i]) < 64.f) || boundary_offset(f[i]) <= NEAR) todo |= 1u << i;
        // one copy of the exact evaluation, element by element (eight copies per vector outgrow the
        // instruction cache)
        for (; todo; todo &= todo - 1) {
            float one = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if ((todo & (0u - todo)) == 1u << i) one = x[i];
            one = silu_exact_f32(one);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if ((todo & (0u - todo)) == 1u << i) f[i] = one;
        }
    }
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t s2 = pack2_bf16(f[2 * i], f[2 * i + 1]);
        o[i] = pack2_bf16(__fmul_rn(bf16_bits_to_f32(s2 & 0xffffu), bf16_bits_to_f32(uw[i] & 0xffffu)),
                          __fmul_rn(__uint_as_float(s2 & 0xffff0000u), __uint_as_float(uw[i] & 0xffff0000u)));
    }
    return make_uint4(o[0], o[1], o[2], o[3]);
}

struct SiluArgs {
    const uint16_t *gate, *up;
    uint16_t *out;   // nullable
    int8_t *q;       // nullable together with s
    float *s;
    int K;
    long ldg, ldu, ldo;

    SiluArgs from_row(long r) const {
        return {gate + r * ldg, up + r * ldu, out ? out + r * ldo : nullptr, q ? q + r * K : nullptr, s ? s + r : nullptr,
                K, ldg, ldu, ldo};
    }
};

// K % 8 == 0, every row 16-byte aligned; the row fits VPT vectors per thread.  A workgroup per row, all
// of the row's inputs requested before the first is used.
template <int VPT>
__global__ void __launch_bounds__(MAX_THREADS) silu_mul_quant_vec(SiluArgs a) {
    __shared__ float smem[MAX_THREADS / 64];
    const int T = blockDim.x;
    const int row = blockIdx.x, nvec = a.K / 8;
    const uint4 *gr = reinterpret_cast<const uint4 *>(a.gate + (size_t)row * a.ldg);
    const uint4 *ur = reinterpret_cast<const uint4 *>(a.up + (size_t)row * a.ldu);
    uint4 *orow = a.out ? reinterpret_cast<uint4 *>(a.out + (size_t)row * a.ldo) : nullptr;
    uint4 v[VPT], u[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int idx = threadIdx.x + i * T;
        v[i] = u[i] = make_uint4(0, 0, 0, 0);
        if (idx < nvec) {
            v[i] = gr[idx];
            u[i] = ur[idx];
        }
    }
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int idx = threadIdx.x + i * T;
        if (idx < nvec) {  // wavefronts past the row skip the arithmetic
            v[i] = silu_mul8(v[i], u[i]);
            if (orow) orow[idx] = v[i];  // may overwrite up[idx]: read above by this same thread
            amax = absmax8(v[i], amax);
        }
    }
    amax = block_max(amax, smem);
    const RowScale rs = row_scale(amax);
    if (threadIdx.x == 0) a.s[row] = rs.sc;
    uint2 *qr = reinterpret_cast<uint2 *>(a.q + (size_t)row * a.K);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int idx = threadIdx.x + i * T;
        if (idx < nvec) qr[idx] = quant8(v[i], rs);
    }
}

// Without the quantised row nothing couples a row's elements: a workgroup per 256 vectors of a row
// (`chunks` per row), so that a single row is spread over several CUs (9728 elements: 3.3 -> 2.0 us).
__global__ void __launch_bounds__(THREADS) silu_mul_vec(SiluArgs a, int chunks) {
    const int row = blockIdx.x / chunks, idx = (blockIdx.x - row * chunks) * blockDim.x + threadIdx.x;
    if (idx >= a.K / 8) return;
    const uint4 g = reinterpret_cast<const uint4 *>(a.gate + (size_t)row * a.ldg)[idx];
    const uint4 u = reinterpret_cast<const uint4 *>(a.up + (size_t)row * a.ldu)[idx];
    reinterpret_cast<uint4 *>(a.out + (size_t)row * a.ldo)[idx] = silu_mul8(g, u);
}

// Any K, pitch and alignment; rows longer than the vector kernel holds.  Two passes: the
// product is recomputed for the quantiser (cheaper than depending on a bf16 copy that the
// caller may not have asked for).
__global__ void __launch_bounds__(THREADS) silu_mul_quant_scalar(SiluArgs a) {
    __shared__ float smem[MAX_THREADS / 64];
    const int row = blockIdx.x;
    const uint16_t *gr = a.gate + (size_t)row * a.ldg, *ur = a.up + (size_t)row * a.ldu;
    int8_t *qr = a.q ? a.q + (size_t)row * a.K : nullptr;
    // the quantised row must come from the inputs as they were: quantise before `out` (which may
    // alias `up`) is written
    float amax = 0.f;
    if (a.q) {
        for (int k = threadIdx.x; k < a.K; k += THREADS) {
            const uint32_t p = mul_bf16_bits(silu_bf16_bits(bf16_bits_to_f32(gr[k])), bf16_bits_to_f32(ur[k]));
            amax = fmaxf(amax, fabsf(bf16_bits_to_f32(p)));
        }
        amax = block_max(amax, smem);
    }
    const RowScale rs = row_scale(amax);
    if (a.q && threadIdx.x == 0) a.s[row] = rs.sc;
    uint16_t *orow = a.out ? a.out + (size_t)row * a.ldo : nullptr;
    for (int k = threadIdx.x; k < a.K; k += THREADS) {
        const uint32_t p = mul_bf16_bits(silu_bf16_bits(bf16_bits_to_f32(gr[k])), bf16_bits_to_f32(ur[k]));
        if (qr) qr[k] = (int8_t)quant1(bf16_bits_to_f32(p), rs);
        if (orow) orow[k] = (uint16_t)p;
    }
}

// ------------------------------------------------------------- rms norm

struct NormArgs {
    uint16_t *x;          // read; written back when add != nullptr
    const uint16_t *add;  // nullable
    const uint16_t *w;
    uint16_t *y;          // nullable: the bf16 normalised row
    int8_t *q;            // nullable together with s
    float *s;
    int N;
    long ldx, lda, ldy;
    float eps;
    double rcp_n;         // 1 / N, rounded

    NormArgs from_row(long r) const {
        return {x + r * ldx, add ? add + r * lda : nullptr, w, y ? y + r * ldy : nullptr, q ? q + r * N : nullptr,
                s ? s + r : nullptr, N, ldx, lda, ldy, eps, rcp_n};
    }
};

// The mean is the correctly rounded quotient: one Newton correction of ss * (1 / N) leaves an error near
// 2^-104, and a quotient of a 53-bit number by an N below 2^31 stays further than that from every
// rounding boundary.  A row with an infinity has an infinite mean and so the scale 0 (the correction would be
// inf - inf); a NaN stays one.
__device__ __forceinline__ float inv_rms(double ss, const NormArgs &a) {
    const double q = ss * a.rcp_n;
    const double mean = q < __builtin_inf() ? fma(fma(-q, (double)a.N, ss), a.rcp_n, q) : q;
    return __fdiv_rn(1.0f, __fsqrt_rn((float)mean + a.eps));
}

__device__ __forceinline__ uint32_t add_bf16_bits(float a, float b) { return pack2_bf16(__fadd_rn(a, b), 0.f) & 0xffffu; }

__device__ __forceinline__ uint32_t norm1(float x, float scale, float w) {
    return mul_bf16_bits(pack2_bf16(__fmul_rn(x, scale), 0.f) & 0xffffu, w);
}

// the two bf16 of a dword at once: bf16(bf16(x * scale) * w)
__device__ __forceinline__ uint32_t norm2(uint32_t xw, float scale, uint32_t gw) {
    const uint32_t t = pack2_bf16(__fmul_rn(bf16_bits_to_f32(xw & 0xffffu), scale),
                                  __fmul_rn(__uint_as_float(xw & 0xffff0000u), scale));
    return pack2_bf16(__fmul_rn(bf16_bits_to_f32(t & 0xffffu), bf16_bits_to_f32(gw & 0xffffu)),
                      __fmul_rn(__uint_as_float(t & 0xffff0000u), __uint_as_float(gw & 0xffff0000u)));
}

__device__ __forceinline__ uint32_t add2(uint32_t xw, uint32_t dw) {
    return pack2_bf16(__fadd_rn(bf16_bits_to_f32(xw & 0xffffu), bf16_bits_to_f32(dw & 0xffffu)),
                      __fadd_rn(__uint_as_float(xw & 0xffff0000u), __uint_as_float(dw & 0xffff0000u)));
}

__device__ __forceinline__ double add_squares(const uint4 &v, double ss) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double lo = (double)bf16_bits_to_f32(w[j] & 0xffffu), hi = (double)__uint_as_float(w[j] & 0xffff0000u);
        ss = fma(lo, lo, ss);
        ss = fma(hi, hi, ss);
    }
    return ss;
}

// N % 8 == 0, rows 16-byte aligned, VPT vectors per thread.  WAVE: a wavefront per row (four rows per
// workgroup), reduced without LDS or a barrier -- short rows; otherwise a workgroup of
// blockDim.x <= T_MAX threads per row.  The row, the addend and the gain are all requested before the first is
// used: with the gain fetched behind the reduction a launch of one row waited for memory twice.
template <int VPT, bool ADD, bool WAVE, int T_MAX = THREADS>
__global__ void __launch_bounds__(T_MAX) rms_norm_i8_vec(NormArgs a, int rows) {
    __shared__ double dsmem[WAVE ? 1 : MAX_THREADS / 64];
    __shared__ float smem[WAVE ? 1 : MAX_THREADS / 64];
    const int T = WAVE ? 64 : blockDim.x, t = WAVE ? threadIdx.x & 63 : threadIdx.x;
    const int row = WAVE ? blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6) : blockIdx.x;
    if (WAVE && row >= rows) return;  // whole wavefronts: nothing below synchronises across them
    const int nvec = a.N / 8;
    uint4 *xr = reinterpret_cast<uint4 *>(a.x + (size_t)row * a.ldx);
    const uint4 *ar = reinterpret_cast<const uint4 *>(a.add + (ADD ? (size_t)row * a.lda : 0));
    const uint4 *wr = reinterpret_cast<const uint4 *>(a.w);
    uint4 v[VPT], d[ADD ? VPT : 1], g[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int idx = t + i * T;
        v[i] = d[ADD ? i : 0] = g[i] = make_uint4(0, 0, 0, 0);
        if (idx < nvec) {
            v[i] = xr[idx];
            if constexpr (ADD) d[i] = ar[idx];
        }
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i)
        if (t + i * T < nvec) g[i] = wr[t + i * T];
    double ss = 0.0, ss1 = 0.0;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        if constexpr (ADD) {
            v[i] = make_uint4(add2(v[i].x, d[i].x), add2(v[i].y, d[i].y), add2(v[i].z, d[i].z), add2(v[i].w, d[i].w));
            if (t + i * T < nvec) xr[t + i * T] = v[i];  // the residual stream keeps the sum
        }
        if (i & 1) ss1 = add_squares(v[i], ss1);
        else ss = add_squares(v[i], ss);
    }
    ss += ss1;
    const float scale = inv_rms(WAVE ? wave_sum(ss) : block_sum(ss, dsmem), a);
    uint4 *yr = a.y ? reinterpret_cast<uint4 *>(a.y + (size_t)row * a.ldy) : nullptr;
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        v[i] = make_uint4(norm2(v[i].x, scale, g[i].x), norm2(v[i].y, scale, g[i].y), norm2(v[i].z, scale, g[i].z),
                          norm2(v[i].w, scale, g[i].w));
        if (yr && t + i * T < nvec) yr[t + i * T] = v[i];
        amax = absmax8(v[i], amax);
    }
    if (!a.q) return;
    amax = WAVE ? lane63(wave_max_to_lane63(amax)) : block_max(amax, smem);
    const RowScale rs = row_scale(amax);
    if (t == 0) a.s[row] = rs.sc;
    uint2 *qr = reinterpret_cast<uint2 *>(a.q + (size_t)row * a.N);
#pragma unroll
    for (int i = 0; i < VPT; ++i)
        if (t + i * T < nvec) qr[t + i * T] = quant8(v[i], rs);
}

// Any N, pitch and alignment.  Needs a bf16 destination for the normalised row when quantising
// (y, or the quantiser would have to recompute it a third time): the host passes one.
__global__ void __launch_bounds__(THREADS) rms_norm_i8_scalar(NormArgs a) {
    __shared__ double dsmem[MAX_THREADS / 64];
    __shared__ float smem[MAX_THREADS / 64];
    const int row = blockIdx.x;
    uint16_t *xr = a.x + (size_t)row * a.ldx;
    const uint16_t *ar = a.add ? a.add + (size_t)row * a.lda : nullptr;
    double ss = 0.0;
    for (int k = threadIdx.x; k < a.N; k += THREADS) {
        uint32_t b = xr[k];
        if (ar) {
            b = add_bf16_bits(bf16_bits_to_f32(b), bf16_bits_to_f32(ar[k]));
            xr[k] = (uint16_t)b;
        }
        const double v = (double)bf16_bits_to_f32(b);
        ss = fma(v, v, ss);
    }
    const float scale = inv_rms(block_sum(ss, dsmem), a);
    float amax = 0.f;
    for (int k = threadIdx.x; k < a.N; k += THREADS)   // xr[k] was written by this same thread
        amax = fmaxf(amax, fabsf(bf16_bits_to_f32(norm1(bf16_bits_to_f32(xr[k]), scale, bf16_bits_to_f32(a.w[k])))));
    amax = block_max(amax, smem);
    const RowScale rs = row_scale(amax);
    if (a.q && threadIdx.x == 0) a.s[row] = rs.sc;
    uint16_t *yr = a.y ? a.y + (size_t)row * a.ldy : nullptr;
    int8_t *qr = a.q ? a.q + (size_t)row * a.N : nullptr;
    for (int k = threadIdx.x; k < a.N; k += THREADS) {
        const uint32_t p = norm1(bf16_bits_to_f32(xr[k]), scale, bf16_bits_to_f32(a.w[k]));
        if (yr) yr[k] = (uint16_t)p;
        if (qr) qr[k] = (int8_t)quant1(bf16_bits_to_f32(p), rs);
    }
}

template <bool ADD>
void launch_norm(const NormArgs &a, int M, int waves, hipStream_t st) {
    const int nvec = a.N / 8;
    if (waves == 1) {
        const dim3 grid((M + THREADS / 64 - 1) / (THREADS / 64)), block(THREADS);
        if (nvec <= 64) rms_norm_i8_vec<1, ADD, true><<<grid, block, 0, st>>>(a, M);
        else if (nvec <= 128) rms_norm_i8_vec<2, ADD, true><<<grid, block, 0, st>>>(a, M);
        else if (nvec <= 192) rms_norm_i8_vec<3, ADD, true><<<grid, block, 0, st>>>(a, M);
        else rms_norm_i8_vec<4, ADD, true><<<grid, block, 0, st>>>(a, M);
        return;
    }
    const dim3 grid(M), block(64 * waves);
    const int vpt = (nvec + 64 * waves - 1) / (64 * waves);
    if (vpt <= 1) rms_norm_i8_vec<1, ADD, false, MAX_THREADS><<<grid, block, 0, st>>>(a, M);
    else if (vpt <= 2) rms_norm_i8_vec<2, ADD, false, MAX_THREADS><<<grid, block, 0, st>>>(a, M);
    else if (vpt <= 3) rms_norm_i8_vec<3, ADD, false, MAX_THREADS><<<grid, block, 0, st>>>(a, M);
    else rms_norm_i8_vec<4, ADD, false, MAX_THREADS><<<grid, block, 0, st>>>(a, M);
}

// Wavefronts per row: four up to 8192 elements (add + norm + quantiser on cold operands, 2560 elements: 500 rows
// 10.3 -> 6.0 us against a wavefront per row, 8192 rows 41.6 -> 36.5; two and eight are slower at
// most sizes), four per 8192 beyond, a single one -- four rows per workgroup -- for many rows of at
// most 1024 elements, where a workgroup per row is mostly its own start.  With the quantised row, whose second
// reduction is a second barrier, the single one also wins for many rows of up to 2048 elements (4096 x 1032 8.7 us
// against 12.2 with four, 8192 x 2048 22.5 against 24.4; 1024 rows lose), with the add up to 1536 or, from 4096 rows
// on, 1280 (2048 x 1536 9.1 against 9.9, 8192 x 1536 5 % the other way).
int norm_waves(int M, int nvec, bool add, bool quantised) {
    if (nvec <= 128) return M <= FEW_ROWS ? (nvec + 63) / 64 : 1;
    if (quantised && M > 1280 && nvec <= (!add ? 256 : M <= 4096 ? 192 : 160)) return 1;
    return nvec <= 1024 ? 4 : (nvec + 1023) / 1024 * 4;
}

int norm_entry(const char *who, uint16_t *x, const uint16_t *add, const void *w, void *y, int8_t *q, float *s,
               int M, int N, long ldx, long lda, long ldy, float eps, void *stream) {
    CMI_REQUIRE(M >= 0 && N > 0, CMI_E_ARG, "%s: bad shape M=%d N=%d", who, M, N);
    if (M == 0) return CMI_OK;
    CMI_REQUIRE(x && w && ((q && s) || y), CMI_E_ARG, "%s: null pointer (x, w and one of y or out_q + out_s)", who);
    CMI_REQUIRE((q == nullptr) == (s == nullptr), CMI_E_ARG, "%s: out_q and out_s go together", who);
    CMI_REQUIRE(ldx >= N && (!add || lda >= N) && (!y || ldy >= N), CMI_E_ARG, "%s: a row pitch is below N=%d", who, N);
    CMI_REQUIRE(eps >= 0.f, CMI_E_ARG, "%s: eps must not be negative", who);
    NormArgs a{x, add, static_cast<const uint16_t *>(w), static_cast<uint16_t *>(y), q, s, N, ldx, lda, ldy, eps, 1.0 / N};
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int nvec = N / 8;
    const bool vec = N % 8 == 0 && nvec <= 4 * MAX_THREADS && aligned(x, 16) && ldx % 8 == 0 && aligned(w, 16) &&
                     (!add || (aligned(add, 16) && lda % 8 == 0)) && (!y || (aligned(y, 16) && ldy % 8 == 0)) &&
                     (!q || aligned(q, 8));
    const int waves = vec ? norm_waves(M, nvec, add, q) : THREADS / 64;
    in_row_slices(M, 64 * waves, [&](long lo, int rows) {
        const NormArgs part = a.from_row(lo);
        if (!vec) rms_norm_i8_scalar<<<dim3(rows), dim3(THREADS), 0, st>>>(part);
        else if (add) launch_norm<true>(part, rows, waves, st);
        else launch_norm<false>(part, rows, waves, st);
    });
    return check_launch(who);
}

// Threads per row: one per 16-byte vector for a few rows (up to 512 of at most 2048 elements: 512 x 2048 5.1 us, 5.5 with
// two vectors each), one per two of them otherwise (2048 x 4096: 17.2 us with one each, 15.7 with two), more vectors where the row would need over 1024 threads; a power of two of
// wavefronts, so that the workgroup loads the four SIMDs alike (2048 x 14336: 45 us on 14, 41 on 16).
void launch_silu(const SiluArgs &a, int rows, int M, hipStream_t st) {
    const int nvec = a.K / 8;
    const int vpt = std::max(M <= (nvec <= 256 ? 2 : 1) * FEW_ROWS ? 1 : 2, (nvec + MAX_THREADS - 1) / MAX_THREADS);
    int threads = 64;
    while (threads * vpt < nvec) threads *= 2;
    const dim3 grid(rows), block(threads);
    if (vpt == 1) silu_mul_quant_vec<1><<<grid, block, 0, st>>>(a);
    else if (vpt == 2) silu_mul_quant_vec<2><<<grid, block, 0, st>>>(a);
    else if (vpt == 3) silu_mul_quant_vec<3><<<grid, block, 0, st>>>(a);
    else silu_mul_quant_vec<4><<<grid, block, 0, st>>>(a);
}

}  // namespace

extern "C" int cmi_silu_mul_quant(const void *gate, const void *up, void *out, int8_t *out_q, float *out_s,
                                  int M, int K, int64_t ld_gate, int64_t ld_up, int64_t ld_out, void *stream) {
    CMI_REQUIRE(M >= 0 && K > 0, CMI_E_ARG, "cmi_silu_mul_quant: bad shape M=%d K=%d", M, K);
    if (M == 0) return CMI_OK;
    CMI_REQUIRE(gate && up && (out || (out_q && out_s)), CMI_E_ARG,
                "cmi_silu_mul_quant: null pointer (gate, up and one of out or out_q + out_s)");
    CMI_REQUIRE((out_q == nullptr) == (out_s == nullptr), CMI_E_ARG, "cmi_silu_mul_quant: out_q and out_s go together");
    CMI_REQUIRE(ld_gate >= K && ld_up >= K && (!out || ld_out >= K), CMI_E_ARG,
                "cmi_silu_mul_quant: a row pitch is below K=%d", K);
    SiluArgs a{static_cast<const uint16_t *>(gate), static_cast<const uint16_t *>(up), static_cast<uint16_t *>(out),
               out_q, out_s, K, (long)ld_gate, (long)ld_up, (long)ld_out};
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int nvec = K / 8;
    const bool vec = K % 8 == 0 && aligned(gate, 16) && aligned(up, 16) && ld_gate % 8 == 0 &&
                     ld_up % 8 == 0 && (!out || (aligned(out, 16) && ld_out % 8 == 0)) && (!out_q || aligned(out_q, 8));
    // Vectors per workgroup of the plain product: the width from 256 down that leaves the fewest threads idle (320 and
    // 384 vectors a row: 8192 x 2560 29.6 us at 256, 25.2 at 64; 8192 x 3072 32.7 and 29.5).  Of equal ones the narrower where a row
    // is more than 256 vectors and not a whole number of them (4096 x 5120 26.4 us at 128, 25.1 at 64, 25.4 at 256), else the wider
    // (512 x 576 3.05 us at 128, 3.46 at 64; 600 x 6144 6.5 at 256, 6.7 at 64).
    int width = THREADS;
    const bool narrow = nvec > THREADS && nvec % THREADS;
    for (int t = THREADS - 64; t >= 64; t -= 64) {
        const int held = (nvec + t - 1) / t * t, best = (nvec + width - 1) / width * width;
        if (held < best || (narrow && held == best)) width = t;
    }
    const int chunks = (nvec + width - 1) / width;
    const bool plain = vec && !out_q, whole_rows = vec && out_q && nvec <= 4 * MAX_THREADS;
    in_row_slices(M, plain ? (long)chunks * width : whole_rows ? MAX_THREADS : THREADS, [&](long lo, int rows) {
        const SiluArgs part = a.from_row(lo);
        if (plain) silu_mul_vec<<<dim3(rows * chunks), dim3(width), 0, st>>>(part, chunks);
        else if (whole_rows) launch_silu(part, rows, M, st);
        else silu_mul_quant_scalar<<<dim3(rows), dim3(THREADS), 0, st>>>(part);
    });
    return check_launch("cmi_silu_mul_quant");
}

extern "C" int cmi_rms_norm_i8(const void *x, const void *w, void *y, int8_t *out_q, float *out_s, int M, int N,
                               int64_t ld_x, int64_t ld_y, float eps, void *stream) {
    return norm_entry("cmi_rms_norm_i8", const_cast<uint16_t *>(static_cast<const uint16_t *>(x)), nullptr, w, y,
                      out_q, out_s, M, N, (long)ld_x, 0, (long)ld_y, eps, stream);
}

extern "C" int cmi_add_rms_norm_i8(void *x, const void *add, const void *w, void *y, int8_t *out_q, float *out_s,
                                   int M, int N, int64_t ld_x, int64_t ld_add, int64_t ld_y, float eps, void *stream) {
    CMI_REQUIRE(add, CMI_E_ARG, "cmi_add_rms_norm_i8: null pointer (add)");
    return norm_entry("cmi_add_rms_norm_i8", static_cast<uint16_t *>(x), static_cast<const uint16_t *>(add), w, y,
                      out_q, out_s, M, N, (long)ld_x, (long)ld_add, (long)ld_y, eps, stream);
}
