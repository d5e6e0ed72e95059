// int8 weight-only GEMV, y = bf16(ws[n] * sum_k wq[n,k] x[m,k]): one activation row, two rows of some shapes, and the entry point
// for 1..16 rows (the rest is gemv_w8a16_batch.hip's).
//
// HBM-bound: the only large stream is the int8 weight, read exactly once with
// 16-byte loads that are contiguous across the wavefront (1 KiB per
// wave-load).  int8 is widened in registers (SDWA convert + byte permute to
// packed bf16, exact for |w| <= 127); four products at a time are added to a
// lane's fp32 chain by v_mfma_f32_4x4x4_16b_bf16 (own_chain below).
//
// Canonical summation order (what makes a batched row bit-identical to the
// single-row call, whatever kernel and blocking the launcher picks); it depends on K only:
//   - K is cut into segments of 1024 (64 chunks of 16 elements);
//   - U consecutive segments form a unit (U = unit_segments(K), 1..4);
//   - chunk c of a unit's segments owns one fp32 chain that starts at 0.f: segments ascending, a
//     segment's sixteen products as four MFMA steps of four k each (what a step rounds off: chain_chunk);
//   - the 64 chains of a unit are summed by a fixed tree: chunks c ^ 1, c ^ 2, c ^ 4, c ^ 8, c ^ 16, c ^ 32
//     (wave_sum_to_lane63 where lane l holds chunk l);
//   - unit totals are added in ascending unit order, starting from unit 0's
//     total (not from 0.f);
//   - the per-row weight scale multiplies that sum once, then one bf16 rounding.
//
// Of the MFMA's 16 blocks of 4 x 4 outputs only the diagonal is wanted here, and it costs about what eight v_dot2 would (one
// row, chains of v_dot2 -> these: 2560 -> 151936 57.4 -> 56.8 us, 4096 -> 128256 78.2 -> 77.9, 3584 -> 120000 62.8 -> 62.7, and
// 1-2 % more where a launch is one round of latencies: 4608 -> 340 2.76 -> 2.82); with several activation rows every output is, and the
// kernels for those read the weight at the speed of one row.  (v_dot2 does the same with two products, so
// chains of both kinds cannot be mixed: the order is the MFMA's for every count.)
//
// Execution: one wavefront = (block of R weight rows, one unit of K).  All of a
// wavefront's weight loads are issued up front and there are many small
// wavefronts (R = 2: 2 KiB x CHT in flight each, ~70 VGPRs), which is what keeps
// HBM saturated from the first microsecond to the last: the hardware dispatcher
// back-fills retiring wavefronts, so late memory service of one wavefront never
// idles the rest.  The activations are the same few cache lines for every
// wavefront on the chip; fetched per wavefront they serialise on the L2
// channels that own those lines, so a workgroup (4 wavefronts)
// copies them into LDS once -- requested before the weights, because memory
// returns data in issue order -- and every wavefront reads its fragments from
// there.  When K spans several units the wavefronts of a team each take units
// of the same rows and the unit totals meet in LDS (summed in unit order by one
// lane per output); otherwise the lanes that hold the tree results scale and
// store them.  What a wavefront does after its last bytes have arrived is time in which it has none in flight: where that is a large
// share, two weight rows go through one tree and one store (pairs below).
// A single activation row against a K of two or three units (and against a
// mid-sized weight with K in one unit, from 2305 on) takes gemv_w8a16_wholerow_kernel instead: one
// wavefront per weight row, all units.

#include "gemv_w8a16_math.hpp"

namespace {

using namespace cmi;

struct GemvArgs {
    const int8_t *wq;
    const float *ws;
    const uint16_t *x;
    uint16_t *y;
    int M, N, K;
    int nchunks;    // K / 16
    int nseg;       // ceil(nchunks / 64)
    int unit;       // segments per unit (canonical, from K)
    int units;      // ceil(nseg / unit)
    int nblocks;    // ceil(N / R)
    int uw;         // wavefronts of a team (they stride over the units)
    uint32_t uw_rcp;  // ceil(2^16 / uw)
    int teams;      // row blocks per workgroup
};

// Wavefronts per workgroup (they share one LDS copy of the activations).
// (For one row and K in several units, 9728 -> 2560, that means one team of 3 wavefronts that
// stages the whole activation row for two weight rows; workgroups of 6, 9 and 12 wavefronts stage
// less and measured 8.6, 9.3 and 9.7 us against 7.3.)
constexpr int BLOCK_WAVES = 4;

// Wavefronts per SIMD the compiler is to leave room for.  Told of four, it forms the MFMA sums in ordinary registers instead of accumulation registers
// that each sum has to be copied out of: two activation rows of 6400 -> 9000 14.7 -> 13.8 us, of 2560 -> 151936 65.5 -> 61.1.  One row has no use for it
// (2560 -> 151936 57.2 -> 57.7: an eighth wavefront a SIMD does not help a stream).
constexpr int simd_waves(int m) { return m == 2 ? 4 : 1; }

// Whether two weight rows go through one tree (wave_sum_pair) and end in two lanes that store together: two activation rows, where it halves four trees,
// and short rows, of which the tail is a large share (one row of 1024 -> 151936 28.4 -> 26.7 us; 2560 -> 151936 56.8 against 57.2).
constexpr bool pairs(int m, int r, int cht) { return r == 2 && (m == 2 || cht <= 2); }

// uint4 vectors of the LDS copy of the activations.
//   K one unit: [row][segment][lane][half], i.e. a row as it is in memory, padded
//     with zeros to whole segments: no select, a lane's address is its own offset plus
//     constants.
//   Several units: [row][K] unpadded plus one zeroed 32-byte slot that dead chunks
//     are pointed at (padding whole dead segments would cost a workgroup per CU at K = 9728).
__host__ __device__ constexpr int xlds_vectors(int rows, int K, int segs, bool one_unit) {
    return one_unit ? rows * segs * 128 : rows * (K / 8) + 2;
}

// 16-byte vectors of activations each thread can carry from global memory to LDS: K of one unit is at most 4096, and 256 threads carry it.
constexpr int xstage_vectors(int m, bool multi) { return (multi ? 8 : 2) * m; }

template <int M, int CHT>
struct XStage {
    uint4 x[M][CHT][2];
};

template <int R, int CHT>
struct WStage {
    u32x4 w[R][CHT];
};

// MULTI: several units (totals via LDS); else K is one unit.  A unit is CHT segments, all its loads up front.
// XLDS: the workgroup stages the activations in LDS; otherwise each wavefront
//       reads them from global memory (only when they do not fit).
template <int M, int R, int CHT, bool MULTI, bool XLDS>
__global__ void __launch_bounds__(64 * BLOCK_WAVES, simd_waves(M))
gemv_w8a16_kernel(const GemvArgs a) {
    extern __shared__ uint4 smem[];  // staged activations (XLDS, see xlds_vectors), then unit totals
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: row addresses stay scalar
    // a single unit means one wavefront per team; otherwise wave / uw through a 16-bit reciprocal
    // (exact for the few wavefronts of a workgroup)
    const int team = !MULTI ? wave : (int)(((uint32_t)wave * a.uw_rcp) >> 16);
    const int rb = xcd_contiguous_block(blockIdx.x, gridDim.x) * a.teams + team;
    const bool idle = rb >= a.nblocks;  // only in the last workgroup
    int u = wave - team * a.uw;         // unit in hand; the team's wavefronts stride over the units
    const int xvecs = a.K / 8;          // uint4 per activation row
    const int segs = a.units * a.unit;  // segments the unit loop walks (>= nseg)
    float *unit_total = reinterpret_cast<float *>(smem + (XLDS ? xlds_vectors(a.M, a.K, segs, !MULTI) : 0)) +
                        team * a.units * (R * M);

    const int8_t *wrow[R];  // uniform per wavefront
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int n = rb * R + r;
        n = n < a.N ? n : a.N - 1;
        wrow[r] = a.wq + (size_t)n * a.K;
    }

    // Loads are unconditional: a dead chunk's address is clamped to the row's
    // last chunk and its activations are zeroed, so nothing branches between a
    // load and the arithmetic it overlaps.
    auto load_w = [&](WStage<R, CHT> &s, int unit_idx) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int j = 0; j < CHT; ++j) {
                const int chunk = (unit_idx * CHT + j) * 64 + lane;
                s.w[r][j] = __builtin_nontemporal_load(
                    reinterpret_cast<const u32x4 *>(wrow[r] + (uint32_t)min(chunk, a.nchunks - 1) * 16u));
            }
    };
    auto load_x = [&](XStage<M, CHT> &s, int unit_idx) {
        const int seg_end = min((unit_idx + 1) * CHT, a.nseg);
#pragma unroll
        for (int j = 0; j < CHT; ++j) {
            const int seg = unit_idx * CHT + j;
            const int chunk = seg * 64 + lane;
            const bool live = seg < seg_end && chunk < a.nchunks;
            const int safe = min(chunk, a.nchunks - 1);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int mrow = m < a.M ? m : a.M - 1;
                if constexpr (XLDS) {
                    // dead chunks read zeros: the LDS reads are unconditional
                    if constexpr (!MULTI) {
                        const int at = (mrow * segs + seg) * 128 + 2 * lane;
                        s.x[m][j][0] = smem[at];
                        s.x[m][j][1] = smem[at + 1];
                    } else {
                        // a select on the address, so the LDS reads stay unconditional
                        const int at = live ? mrow * xvecs + 2 * chunk : a.M * xvecs;
                        s.x[m][j][0] = smem[at];
                        s.x[m][j][1] = smem[at + 1];
                    }
                } else {
                    const uint4 *xp = reinterpret_cast<const uint4 *>(a.x + (size_t)mrow * a.K);
                    const uint4 lo = xp[2 * safe], hi = xp[2 * safe + 1];
                    s.x[m][j][0] = live ? lo : make_uint4(0, 0, 0, 0);
                    s.x[m][j][1] = live ? hi : make_uint4(0, 0, 0, 0);
                }
            }
        }
    };

    v4f32 acc[R][M];
    auto compute = [&](const WStage<R, CHT> &ws_, const XStage<M, CHT> &xs_) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < M; ++m) acc[r][m] = v4f32{0.f, 0.f, 0.f, 0.f};
        // two activation rows: the weight rows' chains side by side (one row: no faster)
#pragma unroll
        for (int i = 0; i < R * CHT; ++i) {
            const int r = M == 2 ? i % R : i / CHT, j = M == 2 ? i / R : i % CHT;
            const Chunk w = widen_chunk(ws_.w[r][j]);
#pragma unroll
            for (int m = 0; m < M; ++m) acc[r][m] = chain_chunk(acc[r][m], w, xs_.x[m][j][0], xs_.x[m][j][1]);
        }
    };

    // Activation fetch first (memory returns data in issue order, so whatever a
    // wavefront waits for must have been requested before the long weight
    // stream), then all first-trip weights, then the LDS hand-over: the copy and
    // its barrier run in the shadow of the weight latency.
    constexpr int XV = xstage_vectors(M, MULTI);
    uint4 xstage[XV];
    const int xtotal = a.M * xvecs;
    if constexpr (XLDS) {
        const uint4 *xg = reinterpret_cast<const uint4 *>(a.x);
        // (the zero of the idle threads also keeps the compiler from moving a load down to the
        // predicated LDS store that consumes it, behind the weight requests)
#pragma unroll
        for (int j = 0; j < XV; ++j) {
            const int idx = threadIdx.x + j * blockDim.x;
            xstage[j] = idx < xtotal ? xg[idx] : make_uint4(0, 0, 0, 0);
        }
    }
    WStage<R, CHT> w0;
    load_w(w0, min(u, a.units - 1));
    // The scales of the outputs that this lane stores, requested behind the weights and by vector loads (the
    // opaque zero keeps a uniform address in a vector register).  As scalar loads they would share the
    // LDS counter and sit in front of the barrier of the activation hand-over.
    constexpr bool PAIR = pairs(M, R, CHT);
    constexpr int ROWS = PAIR ? 1 : R;  // weight rows of a lane that holds totals: lanes 0 and 1 (PAIR), or lane 63
    int vzero = 0;
    asm volatile("" : "+v"(vzero));
    float scale[MULTI ? 1 : ROWS];
#pragma unroll
    for (int i = 0; i < (MULTI ? 1 : ROWS); ++i) {
        const int row = MULTI ? min(lane / M, R - 1) : PAIR ? lane & 1 : i;
        scale[i] = a.ws[min(rb * R + row, a.N - 1) + (MULTI ? 0 : vzero)];
    }
    if constexpr (XLDS) {
#pragma unroll
        for (int j = 0; j < XV; ++j) {
            const int idx = threadIdx.x + j * blockDim.x;
            // memory order; the second row starts at its padded offset
            const int row = idx >= xvecs ? 1 : 0;
            const int pad = !MULTI ? segs * 128 - xvecs : 0;
            if (idx < xtotal) smem[idx + row * pad] = xstage[j];
        }
        if constexpr (!MULTI) {
            const int pad = segs * 128 - xvecs;  // zero vectors behind each row (< 128)
            for (int i = threadIdx.x; i < a.M * pad; i += blockDim.x) {
                const int row = i >= pad ? 1 : 0;
                smem[row * segs * 128 + xvecs + i - row * pad] = make_uint4(0, 0, 0, 0);
            }
        } else {
            if (threadIdx.x < 2) smem[xtotal + threadIdx.x] = make_uint4(0, 0, 0, 0);
        }
        __syncthreads();
    }

    auto holds = [&] { return PAIR ? lane < 2 : lane == 63; };
    float tot[ROWS][M];
#pragma unroll 1
    for (; u < a.units; u += a.uw) {
        if (idle) break;
        XStage<M, CHT> x0;
        load_x(x0, u);
        compute(w0, x0);
        if (MULTI && u + a.uw < a.units) load_w(w0, u + a.uw);  // next unit of this wavefront
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if constexpr (PAIR) tot[0][m] = wave_sum_pair(own_chain(acc[0][m], lane), own_chain(acc[1][m], lane), lane);
            else
#pragma unroll
                for (int i = 0; i < ROWS; ++i) tot[i][m] = wave_sum_to_lane63(own_chain(acc[i][m], lane));
        }
        if constexpr (!MULTI) break;
        // unit totals meet in LDS; one lane per output adds them in unit order below
        if (holds()) {
#pragma unroll
            for (int i = 0; i < ROWS; ++i)
#pragma unroll
                for (int m = 0; m < M; ++m) unit_total[u * (R * M) + (PAIR ? lane : i) * M + m] = tot[i][m];
        }
    }

    if constexpr (!MULTI) {
        if (!idle && holds()) {
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                const int n = rb * R + (PAIR ? lane : i);
                if (n < a.N) {
#pragma unroll
                    for (int m = 0; m < M; ++m)
                        if (m < a.M) a.y[(size_t)m * a.N + n] = (uint16_t)f32_to_bf16_bits(scale[i] * tot[i][m]);
                }
            }
        }
    } else {
        __syncthreads();
        if (!idle && wave == team * a.uw && lane < R * M) {
            const int r = lane / M, m = lane - r * M;
            const int n = rb * R + r;
            if (n < a.N && m < a.M) {
                float total = unit_total[lane];
                for (int v = 1; v < a.units; ++v) total += unit_total[v * (R * M) + lane];
                a.y[(size_t)m * a.N + n] = (uint16_t)f32_to_bf16_bits(scale[0] * total);
            }
        }
    }
}

// One activation row, K in up to three units: a wavefront owns a whole
// weight row -- all units, every byte requested up front -- and adds its unit totals in lane
// 63 in the canonical order, so there is no exchange through LDS and no second barrier, and a
// workgroup of W wavefronts stages the activation row once for W weight rows (the team
// arrangement of the general kernel stages it once per two rows).  Same bits.
template <int CHT, int NU, int XV>
__global__ void __launch_bounds__(256)
gemv_w8a16_wholerow_kernel(const GemvArgs a) {
    extern __shared__ uint4 smem[];  // the activation row, then one zeroed 32-byte slot
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int n_raw = xcd_contiguous_block(blockIdx.x, gridDim.x) * waves + wave;
    const int n = n_raw < a.N ? n_raw : a.N - 1;
    const int8_t *wrow = a.wq + (size_t)n * a.K;
    const int xvecs = a.K / 8;

    uint4 xstage[XV];
    const uint4 *xg = reinterpret_cast<const uint4 *>(a.x);
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int idx = threadIdx.x + j * blockDim.x;
        xstage[j] = idx < xvecs ? xg[idx] : make_uint4(0, 0, 0, 0);
    }
    u32x4 w[NU][CHT];
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int j = 0; j < CHT; ++j) {
            const int chunk = ((u * CHT + j) * 64 + lane);
            w[u][j] = __builtin_nontemporal_load(
                reinterpret_cast<const u32x4 *>(wrow + (uint32_t)min(chunk, a.nchunks - 1) * 16u));
        }
    int vzero = 0;
    asm volatile("" : "+v"(vzero));
    const float scale = a.ws[n + vzero];
#pragma unroll
    for (int j = 0; j < XV; ++j) {
        const int idx = threadIdx.x + j * blockDim.x;
        if (idx < xvecs) smem[idx] = xstage[j];
    }
    if (threadIdx.x < 2) smem[xvecs + threadIdx.x] = make_uint4(0, 0, 0, 0);
    __syncthreads();

    float total = 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int seg_end = min((u + 1) * CHT, a.nseg);
        v4f32 v4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < CHT; ++j) {
            const int seg = u * CHT + j;
            const int chunk = seg * 64 + lane;
            const bool live = seg < seg_end && chunk < a.nchunks;
            const int at = live ? 2 * chunk : xvecs;
            const uint4 x0 = smem[at], x1 = smem[at + 1];
            v4 = chain_chunk(v4, widen_chunk(w[u][j]), x0, x1);
        }
        const float v = wave_sum_to_lane63(own_chain(v4, lane));
        total = u == 0 ? v : total + v;
    }
    if (lane == 63 && n_raw < a.N) a.y[n] = (uint16_t)f32_to_bf16_bits(scale * total);
}

//: Wavefronts per workgroup of the whole-row kernel (2, 3, 5, 6 and 8 measured slower:
//: 9728 -> 2560 takes 7.2, 7.5, 7.3, 7.7 and 8.0 us against 6.7).
constexpr int WHOLEROW_WAVES = 4;
//: 16-byte vectors of the activation row per thread: K <= 12288, which three units cannot exceed.
constexpr int WHOLEROW_XV = 6;

template <int CHT, int NU>
int launch_wholerow(const GemvArgs &a, hipStream_t st) {
    const size_t lds = 16 * (size_t)(a.K / 8 + 2);
    const dim3 grid((a.N + WHOLEROW_WAVES - 1) / WHOLEROW_WAVES), block(64 * WHOLEROW_WAVES);
    gemv_w8a16_wholerow_kernel<CHT, NU, WHOLEROW_XV><<<grid, block, lds, st>>>(a);
    return check_launch("cmi_gemv_w8a16");
}

// CMI_E_UNSUPPORTED (no error text) when the shape is not one this kernel takes.
int dispatch_wholerow(const GemvArgs &a, hipStream_t st) {
    if (a.K / 8 > WHOLEROW_XV * 64 * WHOLEROW_WAVES) return CMI_E_UNSUPPORTED;
    if (a.units == 1) {
        // K in one unit: the general kernel is as good or better for small launches (one weight row per
        // wavefront there too, padded activation copy without selects: 4096 -> 2560 3.85 against 3.91 us)
        // and for very tall weights; in between this kernel is 1-4 % faster (2560 -> 19456 10.1 -> 9.7 us, 3072 -> 40000 21.1 -> 20.4)
        // while a row is long enough to keep the memory busy by itself.  Up to 2304 the general kernel's two rows a wavefront are
        // (2048 -> 40000 16.4 -> 14.6 us, 1536 -> 60000 20.3 -> 16.4, 1040 -> 126030 34.3 -> 25.3, 2112 -> 39718 16.3 -> 15.2;
        // 2304 -> 56888 23.6 -> 23.1, 2432 -> 53894 22.5 against 23.2).
        const size_t wbytes = (size_t)a.N * a.K;
        if (a.K <= 2304 || wbytes <= ((size_t)20 << 20) || wbytes > ((size_t)128 << 20)) return CMI_E_UNSUPPORTED;
        return a.unit == 4 ? launch_wholerow<4, 1>(a, st) : launch_wholerow<3, 1>(a, st);
    }
    if (a.units == 2) {
        if (a.unit == 4) return launch_wholerow<4, 2>(a, st);
        if (a.unit == 3) return launch_wholerow<3, 2>(a, st);
    } else if (a.units == 3) {
        if (a.unit == 4) return launch_wholerow<4, 3>(a, st);
        if (a.unit == 3) return launch_wholerow<3, 3>(a, st);
    }
    return CMI_E_UNSUPPORTED;
}

//: Most K-units one launch handles (LDS holds one total per unit and output).
constexpr int MAX_UNITS = 64;
//: LDS of a workgroup of which a CU holds six.
constexpr size_t SIX_PER_CU = 26 * 1024;
//: Activations up to this many bytes are staged in LDS.
constexpr size_t XLDS_MAX_BYTES = 128 * 1024;

// Two weight rows per wavefront share the activation fragments.  A single row of a small
// weight is latency-bound instead: one row per wavefront halves the arithmetic left to do
// when a wavefront's last bytes arrive (4096 -> 2560: 4.4 -> 4.1 us); from ~20 MB on the
// launch is throughput-bound and the shared fragments win.  (Blocking never changes results.)
int weight_rows(int M, int N, int K, int units) {
    return M == 1 && units == 1 && (size_t)N * K <= ((size_t)20 << 20) ? 1 : 2;
}

template <int M, int R, int CHT, bool MULTI, bool XLDS>
int launch_x(const GemvArgs &a, const dim3 grid, const dim3 block, size_t lds, hipStream_t st) {
    static std::atomic<uint64_t> devices{0};
    if (const int rc = reserve_lds(reinterpret_cast<const void *>(gemv_w8a16_kernel<M, R, CHT, MULTI, XLDS>), 128 * 1024, devices,
                                   "cmi_gemv_w8a16"))
        return rc;
    gemv_w8a16_kernel<M, R, CHT, MULTI, XLDS><<<grid, block, lds, st>>>(a);
    return check_launch("cmi_gemv_w8a16");
}

// Whether a workgroup can carry the activations into LDS.
bool x_fits_lds(int M, int K, int units, int segs) {
    const int uw = units < 4 ? units : 4;
    const int teams = BLOCK_WAVES / uw;
    // the unit totals share the allocation: one float per (team, unit, weight row, activation row)
    const size_t lds = 16 * (size_t)xlds_vectors(M, K, segs, units == 1) + (units > 1 ? sizeof(float) * teams * units * 4 * M : 0);
    return lds <= XLDS_MAX_BYTES && (size_t)M * K * 2 <= 16 * (size_t)xstage_vectors(M, units > 1) * (64 * uw * teams);
}

// Two rows that this file's kernel, which has a wavefront for every two weight rows and unit, takes faster than the batch kernels (us, batch
// kernel -> this one).
//   One unit: more outputs than fit the chip's workgroups of the batch kernel at once, K > 1024 (1280 -> 8400 5.5 -> 4.7, 2560 -> 10000
//   8.1 -> 7.1, 4096 -> 10000 11.3 -> 10.0, 2560 -> 151936 79.6 -> 63.4; 1728 -> 6000 4.1 against 4.3, 1024 -> 20000 5.9 against 6.8).  Short rows
//   that do not start on whole lines only up to 16384 (1088 -> 12000 5.3 -> 5.2, 1088 -> 50000 14.8 against 15.5, 1152 -> 50000 17.6 -> 15.7).
//   Several units: outputs too few for the batch kernel to stream (5120 -> 10000 14.3 -> 13.0, 6400 -> 9000 17.0 -> 14.9), or so few that a
//   wavefront of it walks several units: 768 of three, 1152 of four (12800 -> 512 5.5 -> 4.4, 16384 -> 300 5.7 -> 4.4), and where it then has one
//   workgroup for two CUs (1025..1536: 8320 -> 1200 6.4 -> 5.4, 9728 -> 1100 7.3 -> 6.0, 14336 -> 1300 8.5 -> 7.8;
//   8320 -> 900 4.3 against 4.5, 9728 -> 1800 8.0 -> 7.4 but 11264 -> 1800 8.25 against 8.3, 16384 -> 1600 9.3 against 10.3).
bool two_rows_stay(int N, int K, int units, int segs) {
    if (units == 1) return K > 1024 && N > 8192 && (N <= 16384 || K % 128 == 0 || K > 2048);
    if (!x_fits_lds(2, K, units, segs)) return false;
    return (N > 8192 && (size_t)N * K < ((size_t)96 << 20)) || (units > 2 && (N <= 384 * (units - 1) || (N > 1024 && N <= 1536)));
}

template <int M, int R, int CHT, bool MULTI>
int launch(GemvArgs &a, hipStream_t st) {
    a.nblocks = (a.N + R - 1) / R;
    a.uw = a.units < 4 ? a.units : 4;
    a.uw_rcp = (65536u + a.uw - 1) / a.uw;
    a.teams = BLOCK_WAVES / a.uw;
    const dim3 grid((a.nblocks + a.teams - 1) / a.teams);
    const dim3 block(64 * a.uw * a.teams);
    const size_t totals = MULTI ? sizeof(float) * a.teams * a.units * R * M : 0;
    const int segs = a.units * a.unit;
    if constexpr (MULTI && M == 1 && CHT == 4)  // (units of three segments fit, and two rows that do not are the batch kernels')
        if (!x_fits_lds(a.M, a.K, a.units, segs)) return launch_x<M, R, CHT, MULTI, false>(a, grid, block, totals, st);
    size_t lds = 16 * (size_t)xlds_vectors(a.M, a.K, segs, !MULTI) + totals;
    // One row of a large weight of several segments, mostly full: six workgroups a CU have 100..200 KB in flight, and a seventh only takes turns with them.
    // Seven or eight -> six: 2048 -> 151936 48.6 -> 47.4 us, 3584 -> 120000 65.4 -> 64.9, 4096 -> 151936 92.1 -> 91.4, 2560 -> 151936 58.8 -> 58.6 (five 59.7);
    // 2176 -> 128256, its third segment an eighth full, 43.9 against 45.1, 1024 -> 151936 27.3 / 28.4.  Up to 128 MiB it makes no difference.
    if constexpr (M == 1 && R == 2 && CHT >= 2 && !MULTI)
        if ((size_t)a.N * a.K > (size_t)128 << 20 && a.nchunks * 5 >= segs * 256) lds = lds < SIX_PER_CU ? SIX_PER_CU : lds;
    return launch_x<M, R, CHT, MULTI, true>(a, grid, block, lds, st);
}

template <int M, int R>
int by_unit(GemvArgs &a, hipStream_t st) {
    if (a.units > 1) {  // unit_segments: several units are of three or four segments
        if constexpr (R == 2) return a.unit == 3 ? launch<M, R, 3, true>(a, st) : launch<M, R, 4, true>(a, st);
        return fail(CMI_E_UNSUPPORTED, "cmi_gemv_w8a16: no kernel for %d weight rows and several units", R);
    }
    if constexpr (M == 1)  // (two rows that short are the batch kernels')
        if (a.unit == 1) return launch<M, R, 1, false>(a, st);
    if (a.unit == 2) return launch<M, R, 2, false>(a, st);
    if (a.unit == 3) return launch<M, R, 3, false>(a, st);
    return launch<M, R, 4, false>(a, st);
}

}  // namespace

extern "C" int cmi_gemv_w8a16(const int8_t *wq, const float *ws, const void *x, void *y,
                              int M, int N, int K, void *stream) {
    CMI_REQUIRE(wq && ws && x && y, CMI_E_ARG, "cmi_gemv_w8a16: null pointer");
    CMI_REQUIRE(M >= 1 && M <= 16, CMI_E_UNSUPPORTED, "cmi_gemv_w8a16: M=%d outside 1..16", M);
    CMI_REQUIRE(N >= 1 && K >= 16, CMI_E_ARG, "cmi_gemv_w8a16: bad shape N=%d K=%d", N, K);
    CMI_REQUIRE(K % 16 == 0, CMI_E_UNSUPPORTED, "cmi_gemv_w8a16: K=%d is not a multiple of 16", K);
    CMI_REQUIRE(aligned(wq, 16) && aligned(x, 16) && aligned(y, 2) && aligned(ws, 4), CMI_E_ARG,
                "cmi_gemv_w8a16: wq and x must be 16-byte aligned");
    GemvArgs a;
    a.wq = wq;
    a.ws = ws;
    a.x = static_cast<const uint16_t *>(x);
    a.y = static_cast<uint16_t *>(y);
    a.M = M;
    a.N = N;
    a.K = K;
    a.nchunks = K / 16;
    a.nseg = (a.nchunks + 63) / 64;
    a.unit = unit_segments(a.nseg);
    a.units = (a.nseg + a.unit - 1) / a.unit;
    CMI_REQUIRE(a.units <= MAX_UNITS, CMI_E_UNSUPPORTED, "cmi_gemv_w8a16: K=%d above %d", K,
                MAX_UNITS * 4096);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (M > 2 || (M == 2 && !two_rows_stay(N, K, a.units, a.units * a.unit)))
        return gemv_w8a16_batch(wq, ws, x, y, M, N, K, stream);
    // One row of a long K (two or three units), or of a mid-sized weight with K in one unit: a
    // wavefront per weight row.  CMI_GEMV_WHOLEROW=0 keeps the general kernel (the tests compare
    // the two bit for bit).
    if (M == 1 && option_gemv_wholerow() != 0) {
        const int rc = dispatch_wholerow(a, st);
        if (rc != CMI_E_UNSUPPORTED) return rc;
    }
    if (M == 2) return by_unit<2, 2>(a, st);
    return weight_rows(M, N, K, a.units) == 1 ? by_unit<1, 1>(a, st) : by_unit<1, 2>(a, st);
}
