// W4A8 GEMV for 3..16 quantised rows against a large weight (lm_head), groups of 128, K of 256..5120; arithmetic and bits of
// gemv_w4a8_rows16.hip.
//
// HBM-bound.  The kernels of the smaller weights give a workgroup 16 or 64 weight rows, and each of them fetches the activations
// again: half as many bytes through L2 as the weight itself (16 rows of 2560 -> 151936: 48 us).  Here one workgroup of 16 wavefronts per CU
// fetches them once, keeps them in LDS in the MFMA arrangement with -8 times their group sums (what the unsigned codes owe, the
// accumulators' first value), and each wavefront walks tiles of 16 weight rows over all of K: the fp32 chain stays in its
// registers, no sum goes through LDS, and D lines (2 KiB each) are on their way at any time, across tiles.  us before -> after at 3 / 8 / 16
// rows, dependent launches on cold weights: 2560 -> 151936 41.5 -> 36.9 / 43.0 -> 37.2 / 48.4 -> 38.3, 5120 -> 51200 35.8 ->
// 27.5 / 33.1 -> 28.0 / 34.5 -> 28.5.  A wavefront's tile takes 6 us whatever else runs, so weights of few tiles a
// wavefront keep the other kernels (4096 -> 28672 15.3 either way at 16 rows, 2560 -> 19456 9.8 against 10.0).
// Parking a line one step ahead of its sums changed nothing.
#include "rows16_tile.hpp"

namespace {

using namespace cmi;
using namespace cmi::rows16;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 16;   // weight rows per tile
constexpr int GS = 128;
constexpr int WAVES = 16;

struct Args {
    const uint8_t *w4;
    const float *ws;
    const int8_t *xq;
    const float *xs;
    uint16_t *y;
    int M, N, K;
    int G;          // groups: K / 128
    int lines;      // 128-byte lines of a weight row, two groups each: ceil(G / 2)
    int tiles;      // ceil(N / 16)
    uint32_t g_rcp; // ceil(2^32 / G), G >= 2
};

// activation pieces [G][2][64 lanes] 16 bytes, -8 * their sums [G][16]; per wavefront the scales of a tile [16][G + 1] and a patch
__host__ __device__ constexpr int shared_bytes(int G) { return G * 2048 + G * 64; }
__host__ __device__ constexpr int wave_bytes(int G) { return (TILE * (G + 1) * 4 + 15) / 16 * 16 + PATCH_BYTES; }

// D: lines on their way; XN: groups a wavefront stages; WSN: floats of a tile's scales per lane.
template <int D, int XN, int WSN>
__global__ void __launch_bounds__(WAVES * 64)
gemv_w4a8_stream_kernel(const Args a) {
    extern __shared__ __align__(16) uint8_t lds[];
    v4i32 *xf = reinterpret_cast<v4i32 *>(lds);
    int *cinit = reinterpret_cast<int *>(lds + a.G * 2048);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4, nn = lane & 15;
    uint8_t *mine = lds + shared_bytes(a.G) + wave * wave_bytes(a.G);
    float *wsl = reinterpret_cast<float *>(mine);
    uint8_t *patch = mine + wave_bytes(a.G) - PATCH_BYTES;

    // activations: 32 contiguous bytes of row nn per lane and group
    v4i32 xa[XN][2];
#pragma unroll
    for (int i = 0; i < XN; ++i) {
        const int g = min(wave + i * WAVES, a.G - 1);
        const v4i32 *p = reinterpret_cast<const v4i32 *>(a.xq + (size_t)min(nn, a.M - 1) * a.K + g * GS + kq * 32);
        xa[i][0] = p[0];
        xa[i][1] = p[1];
    }
    float xs[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) xs[v] = a.xs[min(4 * kq + v, a.M - 1)];

    const XcdItems tiles = xcd_items(a.tiles, wave, WAVES);
    const int end = tiles.end, step = tiles.step;
    int tile = tiles.next, line = 0;
    int ptile = tile, pline = 0;

    float wsr[WSN];
    auto request_ws = [&](int t) {
        const float *src = a.ws + (size_t)t * TILE * a.G;
        const int total = min(TILE, a.N - t * TILE) * a.G;
#pragma unroll
        for (int i = 0; i < WSN; ++i) {
            const int idx = lane + i * 64;
            wsr[i] = idx < total ? src[idx] : 0.f;
        }
    };
    auto keep_ws = [&] {
#pragma unroll
        for (int i = 0; i < WSN; ++i) {
            const int idx = lane + i * 64;
            if (idx < TILE * a.G) wsl[idx + __umulhi((uint32_t)idx, a.g_rcp)] = wsr[i];
        }
    };
    v4i32 w[D][2];
    const int half_k = a.K / 2;
    auto request = [&](int slot) {
        if (ptile < end) {
            const uint8_t *base = a.w4 + (size_t)ptile * TILE * half_k;
            const int last = a.N - 1 - ptile * TILE;
            const int off = min(pline * 128 + (lane & 7) * 16, half_k - 16);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                w[slot][j] = __builtin_nontemporal_load(reinterpret_cast<const v4i32 *>(base + (uint32_t)(min(8 * j + (lane >> 3), last) * half_k + off)));
            if (++pline == a.lines) pline = 0, ptile += step;
        }
    };
    if (tile < end) request_ws(tile);
#pragma unroll
    for (int s = 0; s < D; ++s) request(s);

    // activations into the MFMA arrangement, and what the -8 of the codes takes off each group sum
#pragma unroll
    for (int i = 0; i < XN; ++i) {
        const int g = wave + i * WAVES;
        if (g < a.G) {
            const v4i32 p = xa[i][0], q = xa[i][1];
            xf[g * 128 + lane] = v4i32{p.x, p.z, q.x, q.z};
            xf[g * 128 + 64 + lane] = v4i32{p.y, p.w, q.y, q.w};
            int s = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s = __builtin_amdgcn_sdot4(p[e], 0x01010101, s, false);
                s = __builtin_amdgcn_sdot4(q[e], 0x01010101, s, false);
            }
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (kq == 0) cinit[g * 16 + nn] = -8 * s;
        }
    }
    keep_ws();
    __syncthreads();

    float total[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    while (tile < end) {
#pragma unroll
        for (int s = 0; s < D; ++s) {
            if (tile >= end) break;
            if (line == 0 && tile + step < end) request_ws(tile + step);
            tile_park(patch, lane, w[s][0], w[s][1]);
            request(s);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int g = 2 * line + h;
                if (h == 0 || g < a.G) {
                    const u32x4 ww = __builtin_bit_cast(u32x4, tile_take(patch, lane, 4 * h + kq));
                    const u32x4 lo = ww & 0x0F0F0F0Fu, hi = (ww >> 4) & 0x0F0F0F0Fu;
                    v4i32 acc = *reinterpret_cast<const v4i32 *>(cinit + g * 16 + 4 * kq);
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(xf[g * 128 + lane], __builtin_bit_cast(v4i32, lo), acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(xf[g * 128 + 64 + lane], __builtin_bit_cast(v4i32, hi), acc, 0, 0, 0);
                    const float scale = wsl[nn * (a.G + 1) + g];
#pragma unroll
                    for (int v = 0; v < 4; ++v) total[v] = fmaf((float)acc[v], scale, total[v]);
                }
            }
            if (++line == a.lines) {
                const int n = tile * TILE + nn;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int m = 4 * kq + v;
                    if (n < a.N && m < a.M) a.y[(size_t)m * a.N + n] = (uint16_t)f32_to_bf16_bits(total[v] * xs[v]);
                    total[v] = 0.f;
                }
                line = 0;
                tile += step;
                keep_ws();
            }
        }
    }
}

template <int D, int MAX_G>
int launch(const Args &a, hipStream_t st) {
    auto k = gemv_w4a8_stream_kernel<D, (MAX_G + WAVES - 1) / WAVES, (TILE * MAX_G + 63) / 64>;
    static std::atomic<uint64_t> devices{0};
    if (const int rc = reserve_lds(reinterpret_cast<const void *>(k), shared_bytes(MAX_G) + WAVES * wave_bytes(MAX_G), devices, "cmi_gemv_w4a8"))
        return rc;
    // One workgroup per CU although some wavefronts of each then have no tile: as few workgroups as the tiles fill left 5120 -> 32768 to 128 CUs
    // (18.8 us, 23.6 so; 3968 -> 42281 21.8, 26.1).
    k<<<dim3(a.tiles < 256 ? a.tiles : 256), dim3(WAVES * 64), shared_bytes(a.G) + WAVES * wave_bytes(a.G), st>>>(a);
    return check_launch("cmi_gemv_w4a8");
}

}  // namespace

bool cmi::gemv_w4a8_streams(int M, int N, int K) {
    if (option_w4_gemm_deep() != 0) return false;  // the caller names the tile of 3..16 rows, or the GEMV
    if (M < 3 || M > 16 || K % GS != 0 || K < 2 * GS || K > 5120) return false;
    // From 80 MiB of codes; us, the kernels of the smaller weights against this one at 3 / 16 rows: 5120 -> 32768 18.7, 18.8 / 20.1, 19.8, 3072 -> 54613
    // 21.3, 19.6 / 26.1, 20.6, 512 -> 327680 24.8, 21.2 / 29.4, 22.9.  The others stay longer for few rows of few lines, each a
    // larger share of a tile's fixed steps: up to four rows to 88 MiB below K = 2560 (2048 -> 82432 at 3 rows 19.9, 20.7, 2304 -> 81920 23.3, 21.6),
    // up to eight to 112 at K = 1024 (184320 outputs at 3 rows 21.1, 22.7, 276480 30.1, 29.8), and where besides the last line is half empty always
    // (896 -> 315977 33.4, 35.9; 1152 -> 245760 34.0, 34.3, from five rows on 35.5, 34.8).
    const size_t codes = (size_t)N * K / 2, mib = (size_t)1 << 20;
    if (M <= 8 && K > 768 && K < 1280) return K % (2 * GS) == 0 ? codes >= 112 * mib : K > 1024 && M > 4 && codes >= 80 * mib;
    return codes >= (M <= 4 && K > 768 && K < 2560 ? 88 : 80) * mib;
}

int cmi::gemv_w4a8_stream(const uint8_t *w4, const float *ws, const int8_t *xq, const float *xs, void *y, int M, int N, int K, void *stream) {
    Args a{w4, ws, xq, xs, static_cast<uint16_t *>(y), M, N, K, K / GS, (K / GS + 1) / 2, (N - 1) / TILE + 1, 0};
    a.g_rcp = (uint32_t)(((1ull << 32) + a.G - 1) / a.G);
    hipStream_t st = static_cast<hipStream_t>(stream);
    return a.G <= 20 ? launch<6, 20>(a, st) : launch<4, 40>(a, st);  // 128 registers, 160 KB
}
