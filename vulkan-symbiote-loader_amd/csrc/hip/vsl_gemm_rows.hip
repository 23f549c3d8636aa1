// vsl_gemm_rows.hip -- prompt-pass GEMM of few rows: C[M][N] = A[M][K] * B[N][K]^T for short chunks
// (a chat turn, the tail chunk of a prompt), where the product streams the weights once and the matrix
// work is small.
//
// HBM-bound: at M = 45 a 28672 x 4096 product moves 235 MB of weights for 21 GFLOP of matrix work. The
// tiles of the general kernels (vsl_gemm_dma.hip) pad such a chunk to 64 or 128 rows, carry the padding
// through L2 and LDS, and meet at a block barrier every 64 columns. Here the waves share nothing inside
// the main loop: a block owns 16 NF weight rows, its four waves (one per SIMD, up to 512 registers each;
// eight where a block has one fragment and at most 32 activation rows) take every fourth (eighth)
// 64-column unit of K, load its weight and activation rows by whole 128-byte lines one unit ahead, and turn
// each unit into v_mfma_f32_16x16x32_f16 operands in LDS of their own. The waves' sums meet once, in wave
// order. The activations are re-read per block, from L2 (16 MT rows x 2 planes against 16 NF weight rows):
// loads of eight whole lines fetch them at 18 TB/s, loads in the operand layout (64 bytes of each of 16
// rows, adjacent lanes in different rows) at 8 TB/s.
//
// The weights of the wide blocks are loaded non-temporally (8B layer of 45 rows 140.6 -> 133.4 us, of 3 rows
// 117.0 -> 105.3). With two row blocks (65 to 128 rows) each line is read twice and not kept between (1B down
// of 128 rows fetches 77.7 MB for 33.6 MB of weights); plain loads are level there, weights from memory, us, plain
// / non-temporal: 3072 x 2048 of 128 rows 15.4 / 15.4, 2048 x 8192 25.0 / 24.8, 8192 x 2048 23.7 / 22.4, 2048 x
// 14336 33.6 / 34.5. The narrow shapes' weights (NF = 1) are small and keep plain loads (45.0 against 47.1).
//
// A layer's prompt pass, before (the tiles of vsl_gemm_dma.hip) -> with this kernel, us: 8B 45 rows 170.3 ->
// 133.4, 3 rows 158.6 -> 105.3, 64 rows 177.5 -> 149.4; 1B 45 rows 99.2 -> 76.3, 7 rows 89.3 -> 61.8, 128 rows
// 108.1 -> 96.8; 70B 40 rows 624.6 -> 357.0; d 768 with 30 rows 88.6 -> 45.0.
#include <hip/hip_runtime.h>

#include "vsl_device.h"
#include "vsl_internal.h"

namespace {

constexpr int kPartials = -1;  // in place of an epilogue: the chunk sums for a later launch
constexpr uint32_t kUnit = 64;      // columns of K per wave step: one 128-byte line of each row
constexpr uint32_t kRowCUs = 256;   // MI355X compute units

// Eight e4m3 codes times 2^-12 as binary16, exactly (the smallest is 2^-21).
__device__ __forceinline__ half8 lo8_to_f16(uint2 c) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(c.x, 0x1p-12f, false);
    const h2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(c.x, 0x1p-12f, true);
    const h2 d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(c.y, 0x1p-12f, false);
    const h2 e = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(c.y, 0x1p-12f, true);
    return half8{a[0], a[1], b[0], b[1], d[0], d[1], e[0], e[1]};
}

// MT 16-row tiles of A per block (blocks of consecutive rows when M > 16 MT), NF 16-row fragments of B.
// SW: B holds [Wgate; Wup] (2 N rows); row i of a fragment is gate row (i % 4 < 2) or up row of output
// 2 (i / 4) + i % 2 of the fragment's eight, so that a lane's four sums are two gate/up pairs. Otherwise
// the k chunk's sums go to ws[chunk][M][N].
// F8: the lo plane is VSL_DT_F16F8's bytes, widened to binary16 (exactly) before the matrix product, so
// it meets the fp16 weights themselves rather than their e4m3 roundings.
template <int MT, int NF, int WAVES, bool SW, bool F8>
__global__ __launch_bounds__(64 * WAVES, 1) void k_gemm_rows(const vsl_half* __restrict__ A,
                                                                 const vsl_half* __restrict__ B, uint32_t M, uint32_t N,
                                                                 uint32_t K, uint32_t n_m, uint32_t ksplit,
                                                                 float* __restrict__ ws, void* __restrict__ Cv, int epi, int cm) {
    // one unit per wave (halfs): A's hi rows, its lo rows (or lo codes), the weight rows; after the last
    // unit each wave leaves its sums there (1 KB per fragment)
    constexpr int kPlane = MT * 16 * (int)kUnit, kB = F8 ? kPlane + kPlane / 2 : 2 * kPlane;
    constexpr int kStage = kB + NF * 16 * (int)kUnit;
    constexpr int kWaveBuf = kStage > NF * MT * 512 ? kStage : NF * MT * 512;
    __shared__ __attribute__((aligned(16))) vsl_half lds[WAVES][kWaveBuf];
    const uint32_t lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr uint32_t kOut = SW ? 8 * NF : 16 * NF;  // output columns of the block
    // each XCD takes a contiguous range of items, row blocks fastest (they share the weight rows), then
    // the n tiles of one k chunk (they share the activations)
    const uint32_t n_items = n_m * (N / kOut) * ksplit, per = (n_items + 7) >> 3;
    const uint32_t item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || item >= n_items) return;
    const uint32_t m0 = item % n_m * (16 * MT), kn = item / n_m;
    const uint32_t kc = kn % ksplit, nt = kn / ksplit, n0 = nt * kOut;
    const uint32_t kspan = K / ksplit, units = kspan / kUnit;
    const uint32_t nu = wave < units ? (units - 1 - wave) / WAVES + 1 : 0;
    const uint32_t rot = nt % units;

    const vsl_half* Ak = A + (size_t)kc * kspan;
    const vsl_half* Bk = B + (size_t)kc * kspan;
    const uint8_t* A8 = reinterpret_cast<const uint8_t*>(A + (size_t)M * K) + (size_t)kc * kspan;
    // element offsets of this lane's sources (rows * K < 2^31 is checked by the launcher). Load j takes
    // eight rows' whole lines (lo codes: 16 half lines), eight (four) lanes per row; its lanes store their
    // chunks side by side, chunk c of row r at position c ^ ((r >> 1) & 7) (c ^ ((r >> 2) & 3)) of its row, so
    // that the 16 rows of a fragment read fall in distinct banks. Rows past M re-read row M - 1 and are not stored.
    uint32_t a_off[2 * MT], l_off[F8 ? MT : 1], b_off[2 * NF];
    auto a_row = [&](uint32_t r) { return (m0 + r < M ? m0 + r : M - 1) * K; };
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) {
        const uint32_t r = 8 * j + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        a_off[j] = a_row(r) + 8 * c;
    }
    if constexpr (F8) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const uint32_t r = 16 * j + (lane >> 2), c = (lane & 3) ^ ((r >> 2) & 3);
            l_off[j] = a_row(r) + 16 * c;
        }
    }
#pragma unroll
    for (int j = 0; j < 2 * NF; ++j) {
        const uint32_t r = 8 * j + (lane >> 3), i = r & 15, c = (lane & 7) ^ ((r >> 1) & 7);
        uint32_t row;
        if constexpr (SW) row = ((i & 3) < 2 ? 0u : N) + n0 + 8 * (r >> 4) + 2 * (i >> 2) + (i & 1);
        else row = n0 + r;
        b_off[j] = row * K + 8 * c;
    }
    struct Unit {
        uint4 b[2 * NF], hi[2 * MT], lo[F8 ? MT : 2 * MT];
    };
    vsl_half* const L = lds[wave];
    auto load = [&](Unit& u, uint32_t i) {
        uint32_t un = wave + i * WAVES + rot;
        un = un >= units ? un - units : un;
        const uint32_t k0 = un * kUnit;
#pragma unroll
        for (int j = 0; j < 2 * MT; ++j) u.hi[j] = load16<false>(Ak + k0 + a_off[j]);
        if constexpr (F8) {
#pragma unroll
            for (int j = 0; j < MT; ++j) u.lo[j] = load16<false>(A8 + k0 + l_off[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 2 * MT; ++j) u.lo[j] = load16<false>(Ak + (size_t)M * K + k0 + a_off[j]);
        }
#pragma unroll
        for (int j = 0; j < 2 * NF; ++j) u.b[j] = load16<(NF > 1)>(Bk + k0 + b_off[j]);
        __builtin_amdgcn_sched_barrier(0);
    };
    float4v acc[NF][MT];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[f][m] = float4v{0.f, 0.f, 0.f, 0.f};
    // The wave's LDS accesses execute in order; the fences keep the compiler's order too.
    auto lds_order = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    auto stage = [&](const Unit& u) {
#pragma unroll
        for (int j = 0; j < 2 * MT; ++j) *reinterpret_cast<uint4*>(L + j * 512 + lane * 8) = u.hi[j];
#pragma unroll
        for (int j = 0; j < (F8 ? MT : 2 * MT); ++j) *reinterpret_cast<uint4*>(L + kPlane + j * 512 + lane * 8) = u.lo[j];
#pragma unroll
        for (int j = 0; j < 2 * NF; ++j) *reinterpret_cast<uint4*>(L + kB + j * 512 + lane * 8) = u.b[j];
        lds_order();
    };
    auto compute = [&]() {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint32_t c = 4 * t + g;
            half8 b[NF];
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const uint32_t r = 16 * f + r16;
                b[f] = *reinterpret_cast<const half8*>(L + kB + r * kUnit + (c ^ ((r >> 1) & 7)) * 8);
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const uint32_t r = 16 * m + r16;
                const half8 hi = *reinterpret_cast<const half8*>(L + r * kUnit + (c ^ ((r >> 1) & 7)) * 8);
#pragma unroll
                for (int f = 0; f < NF; ++f)
                    acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[f], hi, acc[f][m], 0, 0, 0);
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const uint32_t r = 16 * m + r16;
                half8 lo;
                if constexpr (F8) {
                    // this lane's eight codes: bytes lo8_pos(8 g) .. + 7 of the 32-column block's 32
                    const uint32_t p = lo8_pos(8 * g), q = 2 * t + (p >> 4);
                    lo = lo8_to_f16(*reinterpret_cast<const uint2*>(L + kPlane + r * (kUnit / 2) +
                                                                    ((q ^ ((r >> 2) & 3)) * 8 + (p & 15) / 2)));
                } else {
                    lo = *reinterpret_cast<const half8*>(L + kPlane + r * kUnit + (c ^ ((r >> 1) & 7)) * 8);
                }
#pragma unroll
                for (int f = 0; f < NF; ++f)
                    acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[f], lo, acc[f][m], 0, 0, 0);
            }
        }
        lds_order();
        __builtin_amdgcn_sched_barrier(0);
    };

    // one unit in registers ahead of the one in LDS: the registers are refilled as soon as they are stored
    if (nu) {
        Unit u;
        load(u, 0);
        for (uint32_t i = 1; i < nu; ++i) {
            stage(u);
            load(u, i);
            compute();
        }
        stage(u);
        compute();
    }
    auto red = [&](uint32_t w, uint32_t q) -> float4v* { return reinterpret_cast<float4v*>(lds[w] + q * 512) + lane; };
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int m = 0; m < MT; ++m) *red(wave, f * MT + m) = acc[f][m];
    __syncthreads();
#pragma unroll
    for (int q0 = 0; q0 < NF * MT; q0 += WAVES) {
        const uint32_t q = q0 + wave;
        if (q >= (uint32_t)(NF * MT)) break;
        float4v s = *red(0, q);
#pragma unroll
        for (int w = 1; w < WAVES; ++w) s += *red(w, q);
        const uint32_t f = q / MT, row = m0 + q % MT * 16 + r16;
        if (row >= M) continue;
        if constexpr (SW) {
            const uint32_t col = n0 + 8 * f + 2 * g;
            const float h0 = silu(s[0]) * s[2], h1 = silu(s[1]) * s[3];
            vsl_half* C = static_cast<vsl_half*>(Cv);
            vsl_half* c = C + (size_t)row * N + col;
            if (cm == kGemmCF8) {
                vsl_half a, b;
                uint32_t l0, l1;
                split_f16_f8(h0, a, l0);
                split_f16_f8(h1, b, l1);
                *reinterpret_cast<half2v*>(c) = half2v{a, b};
                *reinterpret_cast<uint16_t*>(reinterpret_cast<uint8_t*>(C + (size_t)M * N) + (size_t)row * N + lo8_pos(col)) =
                    (uint16_t)(l0 | (l1 << 8));
            } else if (cm == kGemmCX2) {
                vsl_half a, b, l0, l1;
                split_f16(h0, a, l0);
                split_f16(h1, b, l1);
                *reinterpret_cast<half2v*>(c) = half2v{a, b};
                *reinterpret_cast<half2v*>(c + (size_t)M * N) = half2v{l0, l1};
            } else {
                *reinterpret_cast<half2v*>(c) = half2v{(vsl_half)h0, (vsl_half)h1};
            }
        } else {
            const size_t o = (size_t)row * N + n0 + 16 * f + 4 * g;
            if (epi == kPartials) {
                *reinterpret_cast<float4v*>(ws + (size_t)kc * M * N + o) = s;
            } else if (epi == VSL_EPI_STORE_F16) {
                *reinterpret_cast<half4*>(static_cast<vsl_half*>(Cv) + o) =
                    half4{(vsl_half)s[0], (vsl_half)s[1], (vsl_half)s[2], (vsl_half)s[3]};
            } else {
                float4v* c = reinterpret_cast<float4v*>(static_cast<float*>(Cv) + o);
                *c = epi == VSL_EPI_RESID ? *c + s : s;
            }
        }
    }
}

struct RowsArgs {
    hipStream_t s;
    const vsl_half *a, *b;
    uint32_t M, N, K, n_m, ks;
    float* ws;
    void* c;
    int epi, cm;
};

template <int MT, int NF, int WAVES, bool SW, bool F8>
void launch(const RowsArgs& r) {
    const uint32_t items = r.n_m * (r.N / (SW ? 8 * NF : 16 * NF)) * r.ks;
    k_gemm_rows<MT, NF, WAVES, SW, F8><<<(items + 7) / 8 * 8, 64 * WAVES, 0, r.s>>>(  // whole XCD ranges
        r.a, r.b, r.M, r.N, r.K, r.n_m, r.ks, r.ws, r.c, r.epi, r.cm);
}

template <int MT, bool SW, bool F8>
void launch_nf(int nf, const RowsArgs& r) {
    if (nf == 8) launch<MT, 8, 4, SW, F8>(r);
    else if (nf == 4) launch<MT, 4, 4, SW, F8>(r);
    else if constexpr (SW) launch<MT, 7, 4, SW, F8>(r);
    else if (nf == 6) launch<MT, 6, 4, SW, F8>(r);
    else launch<MT, 1, MT <= 2 ? 8 : 4, SW, F8>(r);
}

template <bool SW, bool F8>
void launch_mt(int mt, int nf, const RowsArgs& r) {
    switch (mt) {
        case 1: launch_nf<1, SW, F8>(nf, r); break;
        case 2: launch_nf<2, SW, F8>(nf, r); break;
        case 3: launch_nf<3, SW, F8>(nf, r); break;
        default: launch_nf<4, SW, F8>(nf, r); break;
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

struct RowsPlan {
    int nf = 0;  // 0: not served
    int mt = 0;
    uint32_t n_m = 0, ks = 0;
};

// The block's weight rows (16 nf) and, for the K-split form, the chunks: the least cost of rounds of 256
// blocks x columns x (weight rows + activation rows, two planes of 16 mt) at the rate of one CU, plus the
// partials' traffic (written and read, 4 bytes) shared by all. One wide block per CU beats two narrow ones
// (4 x 16 rows everywhere: 8B layer of 45 rows 143 -> 171-188 us, of 3 rows 117 -> 133). More than 64 rows
// run as two row blocks that share their weights through L2, in one round of blocks and for the narrow
// models' products only (N or K up to 2048: the 1B layer's QKV of 128 rows 22.4 -> 15.8 us, O 22.1 -> 15.6,
// down 27.7 -> 25.5); past that the activations read by every block outweigh what the general tiles
// waste (5120 x 3072 of 96 rows 22.1 -> 31.6, 6144 x 4096 25.6 either way, 4096 x 14336 45.7 -> 50.4, 5120 x 5120
// 40.8 -> 53.1). Widths of 2304 to 3072 on both sides and 4096 x 4096 would gain (2560 x 2560 of 96 rows 38.9 ->
// 22.5, 3072 x 3072 27.8 -> 23.8, 4096 x 4096 27.3 -> 23.1) and are not served.
RowsPlan rows_plan(uint32_t M, uint32_t N, uint32_t K, bool sw, int am, uint32_t max_ks) {
    RowsPlan best;
    const uint64_t brows = sw ? 2ull * N : N;
    if (M == 0 || M > (am == kGemmAF8 ? kRowsMaxM8 : kRowsMaxM) || K % 128) return best;
    if (((uint64_t)M * K) >> 31 || (brows * K) >> 31) return best;  // 32-bit element offsets
    if (M > 64 && N > 2048 && K > 2048) return best;
    const uint32_t n_m = (M + 63) / 64, mt = ((M + n_m - 1) / n_m + 15) / 16;
    double cost = 0;
    for (int nf : {8, sw ? 7 : 6, 4}) {
        const uint32_t out = sw ? 8 * nf : 16 * nf;
        if (N % out) continue;
        for (uint32_t ks = 1; ks <= max_ks; ks *= 2) {
            if (K % (ks * kUnit) || (ks > 1 && K / ks < 4 * kUnit)) break;
            const uint64_t items = (uint64_t)n_m * (N / out) * ks;
            if (n_m > 1 && items > kRowCUs) continue;
            const double c = (double)((items + kRowCUs - 1) / kRowCUs) * (K / ks) * (16 * nf + 32 * mt) * 2 +
                             (sw ? 0.0 : 8.0 * ks * M * N / kRowCUs);
            if (!best.nf || c < cost) {
                cost = c;
                best.nf = nf;
                best.mt = (int)mt;
                best.n_m = n_m;
                best.ks = ks;
            }
        }
    }
    return best;
}

}  // namespace

uint32_t vsl_gemm_rows_split(uint32_t M, uint32_t N, uint32_t K, int am, uint32_t max_ks) {
    return am == kGemmA1 ? 0 : rows_plan(M, N, K, false, am, max_ks).ks;
}

bool vsl_gemm_rows_partials(uint32_t ks, void* stream, const void* A, const void* B, uint32_t M, uint32_t N, uint32_t K,
                            int am, float* ws) {
    if (am == kGemmA1 || !aligned16(A) || !aligned16(B)) return false;
    const RowsPlan p = rows_plan(M, N, K, false, am, ks);
    if (!p.nf || p.ks != ks) return false;
    const RowsArgs r{static_cast<hipStream_t>(stream), static_cast<const vsl_half*>(A), static_cast<const vsl_half*>(B),
                     M, N, K, p.n_m, ks, ws, nullptr, kPartials, kGemmC1};
    if (am == kGemmAF8) launch_mt<false, true>(p.mt, p.nf, r);
    else launch_mt<false, false>(p.mt, p.nf, r);
    return true;
}

bool vsl_gemm_rows_direct(void* stream, const void* A, const void* B, uint32_t M, uint32_t N, uint32_t K, void* C, int epi,
                          int am, int cm) {
    if (am == kGemmA1 || !aligned16(A) || !aligned16(B) || !aligned16(C)) return false;
    const bool sw = epi == VSL_EPI_SWIGLU;
    RowsPlan p = rows_plan(M, N, K, sw, am, 1);
    if (!p.nf) return false;
    if (!sw) p.nf = 1;  // narrow shapes that no K split serves: as many blocks as there are fragments
    const RowsArgs r{static_cast<hipStream_t>(stream), static_cast<const vsl_half*>(A), static_cast<const vsl_half*>(B),
                     M, N, K, p.n_m, 1, nullptr, C, epi, cm};
    if (sw && am == kGemmAF8) launch_mt<true, true>(p.mt, p.nf, r);
    else if (sw) launch_mt<true, false>(p.mt, p.nf, r);
    else if (am == kGemmAF8) launch_mt<false, true>(p.mt, p.nf, r);
    else launch_mt<false, false>(p.mt, p.nf, r);
    return true;
}
