// Single-precision matrix product for the true 32-bit path:
// C[M,N] = A[M,K] . B[N,K]^T on the float matrix instructions (products and sums in float, fused; no reduced-precision
// mode).  The reference's scalar backend folds each output left to right in float (crates/leone/src/cpu.rs:1379-1405,
// 1622-1640); here an output is one such chain, or the sum of a few (below), in an order that the sizes alone fix, so that a
// launch repeats bit for bit.  (Off the 64-bit product by 1e-7 to 1e-6 of its norm over 1 to 1024 rows and K of 512 to 6144,
// never more than the single chain that stood here: 4e-7 to 1.4e-6.)
//
// Two kernels.  Few rows (decoding): a product reads every weight once for 2 M operations, so the weights' bytes are the
// bound and what matters is how much of them is in flight: a workgroup owns 16 rows of B, its waves share out K, and a wave
// keeps eight 1 KB loads in the air.  Many rows (prompt portions): tiles staged through shared memory, bound by the matrix
// instructions (256 operations a cycle and compute unit).  With few tiles K is cut into parts, whose results (planes in
// a buffer of the caller's) a second kernel adds in order.
#include "common.h"
#include "leone_hip.h"

namespace leone {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Four elements of a row from element `at` on, zeros from `k` on; kVec: the row is aligned to 16 bytes and k is a multiple of 4.
template <bool kVec>
__device__ inline f32x4 load_four(const float* __restrict__ row, int at, int k) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (kVec) {
        if (at < k) v = *reinterpret_cast<const f32x4*>(row + at);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (at + i < k) v[i] = row[at + i];
    }
    return v;
}

// ---- few rows ------------------------------------------------------------------------------------------------------
// Lane l of a wave holds, of 16 rows of B, row l % 16's elements 4 (l / 16) .. + 3 of every run of 16: one 16-byte load
// a lane is 64 bytes of each of 16 rows, and the element j of all lanes is one 16 x 16 x 4 instruction.  A's rows lie the
// same way, out of the caches (rows past the last are the last one again and not written).
constexpr int kStreamTile = 16;                        // rows of B a workgroup
constexpr int kStreamRun = 64;                         // elements of K a wave takes at a time
constexpr int kStreamLoads = kStreamRun / 16;

template <int kTilesM, int kWaves, bool kVec>
__global__ void __launch_bounds__(kWaves * kWave)
gemm_f32_stream_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k) {
    __shared__ float sums[kWaves][kTilesM][kStreamTile * kStreamTile];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int n0 = blockIdx.x * kStreamTile;
    const int r = lane % 16, h = (lane / 16) * 4;
    const float* brow = b + static_cast<long>(n0 + r < n ? n0 + r : n - 1) * k;
    const float* arow[kTilesM];
#pragma unroll
    for (int t = 0; t < kTilesM; ++t) arow[t] = a + static_cast<long>(t * 16 + r < m ? t * 16 + r : m - 1) * k;
    // sums side by side, put together at the end: short chains, and what is added rounds at a smaller sum's size (sixteen waves
    // have registers for two)
    constexpr int kSums = kWaves == 16 ? 2 : 4;
    f32x4 acc[kTilesM][kSums] = {};
    f32x4 w[2][kStreamLoads], x[2][kTilesM][kStreamLoads];
    auto fetch = [&](int at, int into) {
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i) w[into][i] = load_four<kVec>(brow, at + i * 16 + h, k);
#pragma unroll
        for (int t = 0; t < kTilesM; ++t)
#pragma unroll
            for (int i = 0; i < kStreamLoads; ++i) x[into][t][i] = load_four<kVec>(arow[t], at + i * 16 + h, k);
    };
    auto multiply = [&](int from) {
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < kTilesM; ++t)
                    acc[t][j % kSums] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[from][t][i][j], w[from][i][j], acc[t][j % kSums], 0, 0, 0);
    };
    // two runs' registers take turns: a run is asked for before the one ahead of it is multiplied
    constexpr int kStep = kWaves * kStreamRun;
    int at = wave * kStreamRun;
    if (at < k) {
        fetch(at, 0);
        for (; at + kStep < k; at += 2 * kStep) {
            fetch(at + kStep, 1);
            multiply(0);
            if (at + 2 * kStep < k) {
                fetch(at + 2 * kStep, 0);
                multiply(1);
            } else {
                multiply(1);
                at += 2 * kStep;
                break;
            }
        }
        if (at < k) multiply(0);
    }
#pragma unroll
    for (int t = 0; t < kTilesM; ++t) {
        f32x4 sum = acc[t][0] + acc[t][1];
        if constexpr (kSums == 4) sum += acc[t][2] + acc[t][3];
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[wave][t][(h + i) * kStreamTile + r] = sum[i];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kTilesM * 256; e += kWaves * kWave) {
        const int t = e / 256, row = t * 16 + e % 256 / 16, col = n0 + e % 16;
        if (row >= m || col >= n) continue;
        float total = sums[0][t][e % 256];
#pragma unroll
        for (int v = 1; v < kWaves; ++v) total += sums[v][t][e % 256];
        c[static_cast<long>(row) * n + col] = total;
    }
}

// ---- many rows -----------------------------------------------------------------------------------------------------
// A tile of kEdge x kEdge outputs, four waves of a quarter each (32 x 32 x 2 instructions, kEdge / 64 squared of them a
// wave).  Slabs of K in shared memory, rows 4 floats further apart than they are long (16-byte reads of 8 neighbouring
// rows then touch every bank once); the next slab is on its way into registers while one is multiplied, and is long enough
// (2048 cycles of instructions and more a wave) to arrive meanwhile.  Of every 8 elements the
// even ones lie first and then the odd ones: half-wave h reads its four at once, and the four instructions take elements 0
// and 1, 2 and 3, .. of them, so that an output is one chain of fused products, k ascending.
constexpr int slab_of(int edge) { return edge == 128 ? 32 : 64; }

template <int kEdge, bool kVec>
__global__ void __launch_bounds__(256)
gemm_f32_tile_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k,
                     int part_k) {
    constexpr int kSlab = slab_of(kEdge);
    constexpr int kFrag = kEdge / 64;                  // 32 x 32 squares along an edge of a wave's quarter
    constexpr int kLoads = kEdge * kSlab / 4 / 256;    // 16-byte loads a thread, matrix and slab
    __shared__ float as[2][kEdge][kSlab + 4];
    __shared__ float bs[2][kEdge][kSlab + 4];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const long m0 = static_cast<long>(blockIdx.y) * kEdge, n0 = static_cast<long>(blockIdx.x) * kEdge;
    const int k_first = blockIdx.z * part_k, k_end = k_first + part_k < k ? k_first + part_k : k;
    c += static_cast<long>(blockIdx.z) * m * n;
    const int wm = (wave / 2) * (kEdge / 2), wn = (wave % 2) * (kEdge / 2);
    f32x16 acc[kFrag][kFrag] = {};
    f32x4 ra[kLoads], rb[kLoads];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int idx = threadIdx.x + i * 256, row = idx / (kSlab / 4), at = k0 + (idx % (kSlab / 4)) * 4;
            const long gm = m0 + row < m ? m0 + row : m - 1, gn = n0 + row < n ? n0 + row : n - 1;
            ra[i] = load_four<kVec>(a + gm * k, at, k_end);
            rb[i] = load_four<kVec>(b + gn * k, at, k_end);
        }
    };
    auto keep = [&](int into) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int idx = threadIdx.x + i * 256, row = idx / (kSlab / 4), at = (idx % (kSlab / 4)) * 4;
            const int even = at / 8 * 8 + at % 8 / 2;
            *reinterpret_cast<f32x2*>(&as[into][row][even]) = f32x2{ra[i][0], ra[i][2]};
            *reinterpret_cast<f32x2*>(&as[into][row][even + 4]) = f32x2{ra[i][1], ra[i][3]};
            *reinterpret_cast<f32x2*>(&bs[into][row][even]) = f32x2{rb[i][0], rb[i][2]};
            *reinterpret_cast<f32x2*>(&bs[into][row][even + 4]) = f32x2{rb[i][1], rb[i][3]};
        }
    };
    fetch(k_first);
    keep(0);
    int at = 0;
    for (int k0 = k_first; k0 < k_end; k0 += kSlab, at ^= 1) {
        const bool more = k0 + kSlab < k_end;
        if (more) fetch(k0 + kSlab);
        __syncthreads();
        const int row = lane % 32, h = (lane / 32) * 4;
#pragma unroll
        for (int s = 0; s < kSlab; s += 8) {
            f32x4 av[kFrag], bv[kFrag];
#pragma unroll
            for (int i = 0; i < kFrag; ++i) {
                av[i] = *reinterpret_cast<const f32x4*>(&as[at][wm + i * 32 + row][s + h]);
                bv[i] = *reinterpret_cast<const f32x4*>(&bs[at][wn + i * 32 + row][s + h]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < kFrag; ++i)
#pragma unroll
                    for (int j = 0; j < kFrag; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i][e], bv[j][e], acc[i][j], 0, 0, 0);
        }
        if (more) keep(at ^ 1);        // read last two slabs ago, and every wave has passed a barrier since
    }
#pragma unroll
    for (int i = 0; i < kFrag; ++i)
#pragma unroll
        for (int j = 0; j < kFrag; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const long gm = m0 + wm + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4, gn = n0 + wn + j * 32 + lane % 32;
                if (gm < m && gn < n) c[gm * n + gn] = acc[i][j][e];
            }
}

// C = the planes' sum, in order.
__global__ void __launch_bounds__(256) gemm_f32_sum_kernel(const float* __restrict__ planes, float* __restrict__ c, long count, int parts) {
    const long at = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (at + 4 <= count && count % 4 == 0) {
        f32x4 total = *reinterpret_cast<const f32x4*>(planes + at);
        for (int p = 1; p < parts; ++p) total += *reinterpret_cast<const f32x4*>(planes + p * count + at);
        *reinterpret_cast<f32x4*>(c + at) = total;
        return;
    }
    for (long e = at; e < at + 4 && e < count; ++e) {
        float total = planes[e];
        for (int p = 1; p < parts; ++p) total += planes[p * count + e];
        c[e] = total;
    }
}

// Up to here a product is a stream of weights.  Measured against 2048 x 2048 weights (us, streamed : tiled): 14.6 : about 20 at 24
// rows; at 64 rows the stream's reads of A, four times the weights', make it 46 : 16.
constexpr int kStreamRows = 32;
constexpr int kStreamK = 256;          // a shorter K is no work to share out over four waves
constexpr int kPartMin = 256;          // elements of K in a part at least
constexpr int kPartsMax = 16;

struct F32Plan {
    int edge = 0, parts = 1, part_k = 0;               // edge 0: the streaming kernel
};

// The tile and the number of parts that keep the chip busiest.  A compute unit's matrix instructions run at one rate however
// many tiles it holds, so what is lost is what tiles cover past the edges and what the fullest of the 256 units has more than
// the others; one tile a unit leaves a wave a SIMD and its waits in the open (measured at two thirds of the rate of three);
// every part writes and reads a plane.
F32Plan f32_plan(int m, int n, int k) {
    F32Plan best;
    best.part_k = k;
    if (m <= kStreamRows && k >= kStreamK) return best;
    constexpr long kUnits = 256;
    double most = 0.0;
    for (int edge : {128, 64}) {
        const long tiles = static_cast<long>(ceil_div(m, edge)) * ceil_div(n, edge);
        const double inside = static_cast<double>(m) * n / (static_cast<double>(tiles) * edge * edge);
        for (int wanted = 1; wanted <= kPartsMax && (wanted == 1 || k / wanted >= kPartMin); ++wanted) {
            const int part_k = ceil_div(ceil_div(k, wanted), 64) * 64, parts = ceil_div(k, part_k);
            const long each = (tiles * parts + kUnits - 1) / kUnits;                     // of the fullest unit
            const double busy = static_cast<double>(tiles) * k / (static_cast<double>(each) * kUnits * part_k);
            const double hidden = edge == 128 ? 1.0 : each >= 3 ? 0.9 : each == 2 ? 0.8 : 0.65;
            const double worth = inside * busy * hidden / (1.0 + 0.04 * (parts - 1));
            if (worth > most * 1.001) {
                most = worth;
                best.edge = edge;
                best.parts = parts;
                best.part_k = parts == 1 ? k : part_k;
            }
        }
    }
    return best;
}

}  // namespace leone

using namespace leone;

// How many planes [m, n] of floats leone_gemm_f32 needs beside C (0: none).
extern "C" int leone_gemm_f32_planes(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0) return 0;
    const F32Plan p = f32_plan(m, n, k);
    return p.parts > 1 ? p.parts : 0;
}

// planes: room for leone_gemm_f32_planes(m, n, k) results (null if that is 0).
extern "C" int leone_gemm_f32(const float* a, const float* b, float* c, float* planes, int m, int n, int k, hipStream_t stream) {
    LEONE_REQUIRE(a && b && c, "gemm_f32: null pointer");
    LEONE_REQUIRE(m > 0 && n > 0 && k > 0, "gemm_f32: sizes %d x %d x %d must be positive", m, n, k);
    const F32Plan p = f32_plan(m, n, k);
    LEONE_REQUIRE(p.parts == 1 || planes, "gemm_f32: %d planes are needed for %d x %d x %d", p.parts, m, n, k);
    const bool vec = k % 4 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0 && reinterpret_cast<uintptr_t>(b) % 16 == 0;
    if (p.edge == 0) {
        const int blocks = ceil_div(n, kStreamTile);
        // waves share out K in runs of 64; sixteen of them where the workgroups are few, so that the chip has loads enough in flight
        const int runs = ceil_div(k, kStreamRun);
        const int tiles = m <= 16 ? 1 : 2;
        const int waves = runs >= 16 && tiles == 1 && blocks < 512 && vec ? 16 : runs >= 8 ? 8 : 4;
#define LEONE_STREAM(T, W)                                                                                                \
    (vec ? gemm_f32_stream_kernel<T, W, true><<<blocks, W * kWave, 0, stream>>>(a, b, c, m, n, k)                          \
         : gemm_f32_stream_kernel<T, W, false><<<blocks, W * kWave, 0, stream>>>(a, b, c, m, n, k))
#define LEONE_STREAM_TILES(T) (waves == 8 ? LEONE_STREAM(T, 8) : LEONE_STREAM(T, 4))
        if (tiles == 1) {
            if (waves == 16) gemm_f32_stream_kernel<1, 16, true><<<blocks, 16 * kWave, 0, stream>>>(a, b, c, m, n, k);
            else LEONE_STREAM_TILES(1);
        } else {
            LEONE_STREAM_TILES(2);
        }
#undef LEONE_STREAM_TILES
#undef LEONE_STREAM
        LEONE_LAUNCH_CHECK("gemm_f32");
        return 0;
    }
    const int grid_y = ceil_div(m, p.edge);
    LEONE_REQUIRE(grid_y <= 65535, "gemm_f32: %d rows exceed the launch limit", m);
    const dim3 grid(ceil_div(n, p.edge), grid_y, p.parts);
    float* into = p.parts > 1 ? planes : c;
#define LEONE_TILE(E, V) gemm_f32_tile_kernel<E, V><<<grid, 256, 0, stream>>>(a, b, into, m, n, k, p.part_k)
    if (p.edge == 128) {
        if (vec) LEONE_TILE(128, true);
        else LEONE_TILE(128, false);
    } else {
        if (vec) LEONE_TILE(64, true);
        else LEONE_TILE(64, false);
    }
#undef LEONE_TILE
    LEONE_LAUNCH_CHECK("gemm_f32");
    if (p.parts > 1) {
        const long count = static_cast<long>(m) * n;
        gemm_f32_sum_kernel<<<ceil_div(count, 1024), 256, 0, stream>>>(planes, c, count, p.parts);
        LEONE_LAUNCH_CHECK("gemm_f32 sum");
    }
    return 0;
}
