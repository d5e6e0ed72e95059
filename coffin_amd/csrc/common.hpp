// Shared device helpers and host-side status plumbing for the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <stdint.h>

#include "../../include/coffin_mi355.h"

namespace cmi {

// ---------------------------------------------------------------- host status
void set_error(const char *fmt, ...);
int fail(int code, const char *fmt, ...);
int check_launch(const char *what);
// Raise a kernel's dynamic-LDS limit to `bytes` on the current device, once per device
// (`devices`: one bit per device ordinal, owned by the call site).  CMI_OK or CMI_E_HIP.
int reserve_lds(const void *kernel, int bytes, std::atomic<uint64_t> &devices, const char *who);

// Kernel-selection overrides (cmi_set_option / CMI_GEMM_TILE, CMI_GEMV_WHOLEROW read once).
int option_gemm_tile();      // 0 = the library chooses, else a tile code of cmi_set_option
int option_gemv_wholerow();  // -1 = the library chooses, 0 = never, 1 = where it can
int option_w4_decode_waves();  // 0 = the library chooses, else 4 or 16 wavefronts per workgroup
int option_w4_gemm_deep();     // 0 = the library chooses, 1 = never, else a tile code (gemm_w4a8_deep_code)
int option_w4_decode_chain();  // 0 = the library chooses, 1 = never, else a variant code of gemv_w4a8_chain

#define CMI_REQUIRE(cond, code, ...)                 \
    do {                                             \
        if (!(cond)) return cmi::fail(code, __VA_ARGS__); \
    } while (0)

// gemm_mfma.hip: register-staged W8A8 GEMM for rows under 128 elements or over 4 Mi, and for under 8 outputs (see gemm_w8a8.hip for the fast path).
int gemm_w8a8_generic(const int8_t *xq, const int8_t *wq, const float *xs, const float *ws, void *y,
                      int32_t *acc_out, int M, int N, int K, int ldy, void *stream);
// gemm_w8a8_rows16.hip: W8A8 for up to 128 rows with the weight read once (K % 16 == 0,
// 128 <= K <= 10240); CMI_E_UNSUPPORTED (no error text) outside that range.
int gemm_w8a8_rows16(const int8_t *xq, const int8_t *wq, const float *xs, const float *ws, void *y,
                     int32_t *acc_out, int M, int N, int K, int ldy, void *stream);
// gemm_w8a8.hip: cmi_gemm_w8a8 with room for split-K (arrival counters, 256 ints, zero; partial
// tiles, gemm_w8a8_split_bytes(M, N, K) bytes or fewer: the kernel choice adapts); both null = no split.
int gemm_w8a8_split(const int8_t *xq, const int8_t *wq, const float *xs, const float *ws, void *y,
                    int32_t *acc_out, int M, int N, int K, int ldy, int *arrivals, void *partials,
                    size_t partial_bytes, void *stream);
size_t gemm_w8a8_split_bytes(int M, int N, int K);
// quant_act_i8.hip: cmi_quant_act_i8 that also clears n_zero ints at `zero` (null / 0: none).
int quant_act_i8_and_clear(const void *x, int8_t *q, float *s, int M, int K, int *zero, int n_zero, void *stream);
// quant_act_i8.hip: the quantiser writing rows of pitch ldq >= K, the tail K .. ldq-1 cleared (rows
// of an int4 weight whose K is padded to whole groups on the device; ldq % 8 == 0 there).
int quant_act_i8_padded(const void *x, int8_t *q, float *s, int M, int K, int ldq, void *stream);
// 16-row weight tiles per workgroup (1 or 2) that gemm_w8a8_rows16 uses for 17..128 rows.
int gemm_w8a8_rows_tiles(int N);

// gemv_w8a16_batch.hip: cmi_gemv_w8a16 for 2..16 rows; arguments already checked.
int gemv_w8a16_batch(const int8_t *wq, const float *ws, const void *x, void *y, int M, int N, int K, void *stream);

// gemv_w4a8_decode.hip: W4A8 GEMV for 1..4 rows, K <= 10240, from bf16 activations (x) or
// quantised ones (xq, xs), groups of 64 and 256 for one row; returns CMI_E_UNSUPPORTED (no error text) for other shapes.
int gemv_w4a8_decode(const uint8_t *w4, const float *ws, const void *x, const int8_t *xq, const float *xs,
                     void *y, int32_t *group_acc, int8_t *xq_out, float *xs_out, int M, int N, int K, int gs,
                     void *stream);
// gemv_w4a8_chain.hip: the same for 1..2 rows with the fp32 chain in registers; `variant` = lanes per
// weight row (8, 16) + 100 * wavefronts sharing a row (1, 2, 4, 8) + 10000 * wavefronts per workgroup
// (4, 8, 16); groups of 64 and 256: one row, 16 lanes; CMI_E_UNSUPPORTED (no error text) outside the variant's range.
int gemv_w4a8_chain(const uint8_t *w4, const float *ws, const void *x, const int8_t *xq, const float *xs,
                    void *y, int32_t *group_acc, int8_t *xq_out, float *xs_out, int M, int N, int K,
                    int gs, int variant, void *stream);
// gemv_w4a8_rows16.hip: W4A8 GEMV for up to 16 quantised rows (xq, xs) or up to 4 bf16 rows (x,
// quantised in the kernel), K <= 10240, integer sums on the matrix pipe; groups of 64 and 256 up to 16 quantised rows;
// CMI_E_UNSUPPORTED (no error text) outside that range.
int gemv_w4a8_rows16(const uint8_t *w4, const float *ws, const int8_t *xq, const float *xs, const void *x,
                     void *y, int32_t *group_acc, int8_t *xq_out, float *xs_out, int M, int N, int K, int gs,
                     void *stream);
// gemv_w4a8_stream.hip: W4A8 GEMV of groups of 128 for the quantised rows of a large weight, and whether it is the one for a shape.
bool gemv_w4a8_streams(int M, int N, int K);
int gemv_w4a8_stream(const uint8_t *w4, const float *ws, const int8_t *xq, const float *xs, void *y, int M, int N, int K, void *stream);
// gemm_w4a8_tile.hip: W4A8 tile GEMM, arguments already checked by cmi_gemm_w4a8 / cmi_gemv_w4a8.  The cheapest tile for a
// shape and its modelled time (us), of all tiles and of those of four groups a step; the tile a gemm_tile
// option names; whether a w4_gemm_deep option names one; the launch.
double gemm_w4a8_tile_us(int M, int N, int K, int gs, int *tile);
double gemm_w4a8_deep_us(int M, int N, int K, int *tile);
int gemm_w4a8_forced_tile(int option, int gs);
// gemm_w4a8.hip: the two-stage kernel, which also writes the group sums where they are asked for; K whole steps of 128 and whole
// groups, arguments already checked, without the sums groups of 64 only.
int gemm_w4a8_two_stage(const uint8_t *w4, const float *ws, const int8_t *xq, const float *xs, void *y, int32_t *group_acc, int M, int N,
                        int K, int gs, void *stream);
// gemv_w4a8.hip: whether cmi_gemv_w4a8 gives rows of groups of 128 to a tile of four groups a step, and which.
bool w4a8_rows_take_tiles(int M, int N, int K, int *tile);
bool gemm_w4a8_deep_code(int code);
int gemm_w4a8_tile(const uint8_t *w4, const float *ws, const int8_t *xq, const float *xs, void *y, int M, int N,
                   int K, int gs, int tile, void *stream);
// linear_bf16.hip: quantiser + W4A8 GEMV / GEMM (or the GEMV that quantises by itself where that
// is faster) on bf16 rows, with xq int8 [M,K] / xs fp32 [M] as staging; arguments already checked.
int linear_w4a8_rows(const uint8_t *w4, const float *ws, const void *x, void *y, int M, int N, int K, int gs,
                     int8_t *xq, float *xs, void *stream);
static inline bool aligned(const void *p, uintptr_t a) {
    return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
}

// ------------------------------------------------------------- device helpers
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v16i32 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t v) {
    return __uint_as_float(v << 16);
}

// fp32 -> bf16 bit pattern, round to nearest even (finite inputs).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}

typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Two fp32 -> packed bf16 (lo in the low half), round to nearest even, one v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack2_bf16(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK,
                                                      0xf, false));
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xf, false);
}

// Sum over the 64 lanes of a wavefront in a fixed order; the total lands in
// lane 63 (other lanes hold partial sums).
__device__ __forceinline__ float wave_sum_to_lane63(float v) {
    v += dpp_f32<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
    v += dpp_f32<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
    v += dpp_f32<0x141, 0xf>(v);  // row_half_mirror
    v += dpp_f32<0x140, 0xf>(v);  // row_mirror
    v += dpp_f32<0x142, 0xa>(v);  // row_bcast15 into rows 1 and 3
    v += dpp_f32<0x143, 0xc>(v);  // row_bcast31 into rows 2 and 3
    return v;
}

// One level of a transposing reduction: of 2 H values a lane forms the sums with its partner (a DPP control) of one half and the
// partner those of the other, so the work halves per level.  The pairing is a plain tree's, and fp32 addition commutes: same bits.
template <int CTRL, int H>
__device__ __forceinline__ void transposed_level(const float (&in)[2 * H], float (&out)[H], bool upper) {
#pragma unroll
    for (int i = 0; i < H; ++i) {
        const float lo = in[i] + dpp_f32<CTRL, 0xf>(in[i]);
        const float hi = in[i + H] + dpp_f32<CTRL, 0xf>(in[i + H]);
        out[i] = upper ? hi : lo;
    }
}

// Rows 0 + 1 and 2 + 3 of the wavefront: even rows hold the sums of a, odd ones those of b.
__device__ __forceinline__ float swap16_add(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// The two halves of the wavefront, likewise.
__device__ __forceinline__ float swap32_add(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The wave sums of two values in one tree, with the pairing of wave_sum_to_lane63: lanes 0 and 1 end with the totals of a and b.
// Which of the two a lane keeps (bits 0 and 2 of its number differ: b) is the same for its partners of all later levels.
__device__ __forceinline__ float wave_sum_pair(float a, float b, int lane) {
    const float v[2] = {a, b};
    float t[1];
    transposed_level<0xB1, 1>(v, t, ((lane ^ (lane >> 2)) & 1) != 0);  // quad_perm [1,0,3,2]
    t[0] += dpp_f32<0x4E, 0xf>(t[0]);                                   // quad_perm [2,3,0,1]
    t[0] += dpp_f32<0x141, 0xf>(t[0]);                                  // row_half_mirror
    t[0] += dpp_f32<0x140, 0xf>(t[0]);                                  // row_mirror
    t[0] = swap16_add(t[0], t[0]);
    return swap32_add(t[0], t[0]);
}

// Max over the 64 lanes; every lane of row 3 ends with the wave maximum, lane
// 63 included.  Inputs must be >= 0 (masked lanes contribute 0).
__device__ __forceinline__ float wave_max_to_lane63(float v) {
    v = fmaxf(v, dpp_f32<0xB1, 0xf>(v));
    v = fmaxf(v, dpp_f32<0x4E, 0xf>(v));
    v = fmaxf(v, dpp_f32<0x141, 0xf>(v));
    v = fmaxf(v, dpp_f32<0x140, 0xf>(v));
    v = fmaxf(v, dpp_f32<0x142, 0xa>(v));
    v = fmaxf(v, dpp_f32<0x143, 0xc>(v));
    return v;
}

// Workgroups are handed to the eight XCDs round-robin.  Renumbered so that each XCD works on one
// contiguous run of row blocks, the 2-byte results of neighbouring rows -- one cache line holds 64 of
// them -- are written by one XCD and leave its L2 as whole lines when the launch ends (lines whose
// bytes are spread over eight L2s cost the step of 129 decode launches 5 %).
__device__ __forceinline__ int xcd_contiguous_block(int b, int nb) {
    const int x = b & 7, q = nb >> 3, r = nb & 7;
    return x * q + min(x, r) + (b >> 3);
}

// Items walked by wavefronts that stay: those of this XCD are one contiguous run, dealt to its workgroups in turn, a wavefront of each at a
// time (few items are spread over all workgroups).
struct XcdItems {
    int next, end, step;
};
__device__ __forceinline__ XcdItems xcd_items(int items, int wave, int waves) {
    const int xcd = blockIdx.x & 7, nq = gridDim.x >> 3, nr = gridDim.x & 7;
    const int nb = nq + (xcd < nr), before = xcd * nq + min(xcd, nr);
    const int first = (int)((uint64_t)items * before / gridDim.x), end = (int)((uint64_t)items * (before + nb) / gridDim.x);
    return {first + wave * nb + (int)(blockIdx.x >> 3), end, waves * nb};
}

__device__ __forceinline__ float lane63(float v) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

}  // namespace cmi
