// vsl_skinny.hip -- Y[N][B] = W[N][K] X[K][B] for 2 <= B <= 16 fp16 columns, X row-major (element (k, b)
// at k * B + b): the skinny product of vsl_gemv.
//
// HBM-bound: W streams once, 2 B flops per 2 weight bytes against a ridge of ~300. On the matrix cores
// (v_mfma_f32_16x16x32_f16, A = 16 rows of W) the operand of X is, per lane, eight consecutive k of one
// column, which this layout scatters B elements apart: gathered from memory, eight 2-byte loads per
// fragment for every one or two 16-byte loads of W, their issue bounds the kernel. Here a wave loads the 64
// rows of X of its unit as they lie (contiguous, 16 bytes per lane) and the weights by whole 128-byte lines
// (eight lanes per row), one unit ahead, and turns both in its own piece of LDS: no block barrier until the
// waves' sums meet. Block = 16 NF rows of W; its WAVES waves take every WAVES-th 64-column unit of K, and
// the 16 NF rows share each X unit: NF = 4 where that still gives three quarters of the CUs a block, else 2
// or 1 with as many more waves. The weights of the wide blocks are loaded non-temporally; those of one
// fragment per block (up to 6128 rows) are not: a product repeated over one such matrix finds it in the cache,
// while matrices that come from memory each time lose (plain / non-temporal, us, repeated: 4096 x 4096, 16 6.6 /
// 7.0, 4096 x 14336, 16 19.9 / 22.4; from memory: 8.8 / 8.4, 25.0 / 23.2; both under the gathering kernel's). The
// blocks of an XCD start at different units, three apart: rows of a power-of-two stride put one unit of
// all rows on few memory channels.
// N x K, B (gathering kernel -> this one, us; one matrix repeated | matrices from memory): 14336 x 4096, 16
// 23.5 -> 19.4 | 30.4 -> 20.2; 4096 x 4096, 9 8.0 -> 6.4 | 10.6 -> 8.5; 1000 x 14336, 4 20.4 -> 12.8 | 28.7 -> 15.9;
// 32000 x 2048, 16 24.8 -> 21.3 | 32.7 -> 21.8; 8000 x 8192, 12 25.9 -> 23.2 | 34.5 -> 24.0 (graphs of one product after
// another).
#include <hip/hip_runtime.h>

#include "vsl_device.h"
#include "vsl_internal.h"

namespace {

constexpr uint32_t kUnit = 64;     // columns of K per wave step
constexpr uint32_t kSkinnyCUs = 256;  // MI355X compute units
static_assert(kSkinnyOneFragN == (3 * kSkinnyCUs / 2 - 1) * 16, "two fragments per block from three quarters of the CUs");

template <int NF, int WAVES, typename YT>
__global__ __launch_bounds__(WAVES * 64) void k_skinny_rows(const vsl_half* __restrict__ W, uint32_t N, uint32_t K,
                                                            const vsl_half* __restrict__ X, uint32_t B, YT* __restrict__ Y) {
    constexpr uint32_t ROWS = 16 * NF;
    // a wave's unit: the rows of X as they lie, then the weight rows (chunk c of row r at position
    // c ^ ((r >> 1) & 7), so that the 16 rows of a fragment read fall in distinct banks)
    __shared__ __attribute__((aligned(16))) vsl_half xs[WAVES][kUnit * 16 * (1 + NF)];
    __shared__ float part[WAVES][ROWS][17];
    const uint32_t lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t units = K / kUnit, nu = wave < units ? (units - 1 - wave) / WAVES + 1 : 0;
    const uint32_t rot = (blockIdx.x >> 3) * 3 % units;
    const uint32_t col = r16 < B ? r16 : B - 1;  // columns past B are not stored
    const vsl_half* wrow[2 * NF];  // load j: eight rows' whole lines, eight lanes per row
#pragma unroll
    for (int j = 0; j < 2 * NF; ++j) {
        const uint32_t r = 8 * j + (lane >> 3), row = blockIdx.x * ROWS + r;  // rows past N re-read row N - 1, not stored
        wrow[j] = W + (size_t)(row < N ? row : N - 1) * K + 8 * ((lane & 7) ^ ((r >> 1) & 7));
    }
    const uint32_t chunks = 8 * B;  // 16-byte chunks of a unit of X (64 B halfs)
    uint32_t xc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) xc[j] = 8 * (lane + 64 * j < chunks ? lane + 64 * j : chunks - 1);

    struct Unit {
        uint4 w[2 * NF], x[2];
    };
    auto load = [&](Unit& u, uint32_t i) {
        uint32_t un = wave + i * WAVES + rot;
        un = un >= units ? un - units : un;
        const uint32_t k0 = un * kUnit;
#pragma unroll
        for (int j = 0; j < 2; ++j) u.x[j] = load16<false>(X + (size_t)k0 * B + xc[j]);
#pragma unroll
        for (int j = 0; j < 2 * NF; ++j) u.w[j] = load16<(NF > 1)>(wrow[j] + k0);
        __builtin_amdgcn_sched_barrier(0);
    };
    float4v acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = float4v{0.f, 0.f, 0.f, 0.f};
    // The wave's LDS accesses execute in order; the fences keep the compiler's order too.
    auto lds_order = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    auto compute = [&](const Unit& u) {
#pragma unroll
        for (int j = 0; j < 2; ++j) *reinterpret_cast<uint4*>(&xs[wave][xc[j]]) = u.x[j];
        vsl_half* const ws = &xs[wave][kUnit * 16];
#pragma unroll
        for (int j = 0; j < 2 * NF; ++j) *reinterpret_cast<uint4*>(ws + j * 512 + lane * 8) = u.w[j];
        lds_order();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            half8 x;
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = xs[wave][(32 * t + 8 * g + i) * B + col];
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const half8 w = *reinterpret_cast<const half8*>(ws + f * 1024 + r16 * kUnit + ((4 * t + g) ^ (r16 >> 1)) * 8);
                acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x, acc[f], 0, 0, 0);
            }
        }
        lds_order();
        __builtin_amdgcn_sched_barrier(0);
    };
    // two register sets, unconditional loads inside the loop, the last two or three units peeled
    Unit u0, u1;
    if (nu == 1) {
        load(u0, 0);
        compute(u0);
    } else if (nu > 1) {
        load(u0, 0);
        load(u1, 1);
        uint32_t i = 0;
        for (; i + 3 < nu; i += 2) {
            compute(u0);
            load(u0, i + 2);
            compute(u1);
            load(u1, i + 3);
        }
        compute(u0);
        if (nu - i == 3) load(u0, i + 2);
        compute(u1);
        if (nu - i == 3) compute(u0);
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[wave][16 * f + 4 * g + v][r16] = acc[f][v];
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < ROWS * 16; e += WAVES * 64) {
        const uint32_t m = e >> 4, n = e & 15, row = blockIdx.x * ROWS + m;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) v += part[w][m][n];
        if (row < N && n < B) store_elem(Y + (size_t)row * B + n, v);
    }
}

template <typename YT>
void launch(const vsl_half* w, uint32_t N, uint32_t K, const vsl_half* x, uint32_t B, YT* y, hipStream_t s) {
    const uint32_t frags = (N + 15) / 16;
    if (frags >= 3 * kSkinnyCUs) k_skinny_rows<4, 4, YT><<<(frags + 3) / 4, 256, 0, s>>>(w, N, K, x, B, y);
    else if (N > kSkinnyOneFragN) k_skinny_rows<2, 8, YT><<<(frags + 1) / 2, 512, 0, s>>>(w, N, K, x, B, y);
    else k_skinny_rows<1, 16, YT><<<frags, 1024, 0, s>>>(w, N, K, x, B, y);
}

}  // namespace

void vsl_skinny_rows(const void* W, uint32_t N, uint32_t K, const void* X, uint32_t B, void* Y, bool y16, void* stream) {
    const vsl_half *w = static_cast<const vsl_half*>(W), *x = static_cast<const vsl_half*>(X);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (y16) launch(w, N, K, x, B, static_cast<vsl_half*>(Y), s);
    else launch(w, N, K, x, B, static_cast<float*>(Y), s);
}
