// Single-precision matrix product for the true 32-bit path:
// C[M,N] = A[M,K] . B[N,K]^T on the float matrix instructions (products and sums in float, fused; no reduced-precision
// mode).  The reference's scalar backend folds each output left to right in float (crates/leone/src/cpu.rs:1379-1405,
// 1622-1640).
//
// An output's bits depend on its row of A, its row of B and K alone, never on the rows that share the launch (what a request gets
// does not depend on who is beside it): K is cut into segments by a rule on K (f32_segments), a segment's sum is that of chains of
// 16 fused products, k ascending, added in order, and so is the segments' sum.  Both kernels below work that way.  What is added rounds
// at the sum's size, so the short sums are also off by less than one chain over K (error against 64 bits over the result's norm, 1 to 1,024 rows:
// K 512 1.0e-7, 2048 1.2e-7, 6144 1.6e-7; one chain 2.9e-7, 8.1e-7 and 9.9e-7).  A K below 256 is one chain, the scalar backend's fold.
//
// Few rows (decoding): a product reads every weight once for 2 M operations, so the weights' bytes are the
// bound and what matters is how much of them is in flight: a workgroup owns 16 rows of B, its waves take a segment each, and a
// wave keeps eight 1 KB loads of B in the air.  Many rows (prompt portions): tiles staged through shared memory, bound by
// the matrix instructions (256 operations a cycle and compute unit).  With few tiles the segments are shared out over
// workgroups, which leave them as planes in a buffer of the caller's for a second kernel to add.
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

// The same where all four lie before the row's end.
template <bool kVec>
__device__ inline f32x4 load_whole(const float* __restrict__ at) {
    if (kVec) return *reinterpret_cast<const f32x4*>(at);
    return f32x4{at[0], at[1], at[2], at[3]};
}

// ---- few rows ------------------------------------------------------------------------------------------------------
// Lane l of a wave loads, of 16 rows of B, row l % 16's elements 4 (l / 16) .. + 3 of every run of 16: one 16-byte load
// a lane is 64 bytes of each of 16 rows.  A's rows lie the same way, out of the caches (rows past the last are the last one again
// and not written).  The 16 x 16 x 4 instruction adds its four products in the order of the lanes' quarters, so the four quarters'
// registers are transposed by lane swaps first: instruction j then takes elements 4 j .. 4 j + 3 in turn.
constexpr int kStreamTile = 16;                        // rows of B a workgroup
constexpr int kStreamRun = 64;                         // elements of K a wave takes at a time
constexpr int kStreamLoads = kStreamRun / 16;
constexpr int kChain = 16;                             // elements of K a chain of products: what a wave's 16-byte loads bring

// Register j of quarter g becomes register g of quarter j.
__device__ inline f32x4 transpose_quarters(const f32x4 v) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const auto bits = [](float f) { return __float_as_uint(f); };
    const u32x2 p = __builtin_amdgcn_permlane32_swap(bits(v[0]), bits(v[2]), false, false);
    const u32x2 q = __builtin_amdgcn_permlane32_swap(bits(v[1]), bits(v[3]), false, false);
    const u32x2 r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    const u32x2 s = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    return f32x4{__uint_as_float(r[0]), __uint_as_float(r[1]), __uint_as_float(s[0]), __uint_as_float(s[1])};
}

template <int kTilesM, int kWaves, int kDepth, bool kVec>
__global__ void __launch_bounds__(kWaves * kWave)
gemm_f32_stream_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k, int segment) {
    __shared__ float sums[kWaves][kTilesM][kStreamTile * kStreamTile];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int n0 = blockIdx.x * kStreamTile;
    const int r = lane % 16, h = (lane / 16) * 4;
    const float* brow = b + static_cast<long>(n0 + r < n ? n0 + r : n - 1) * k;
    const float* arow[kTilesM];
#pragma unroll
    for (int t = 0; t < kTilesM; ++t) arow[t] = a + static_cast<long>(t * 16 + r < m ? t * 16 + r : m - 1) * k;
    f32x4 sum[kTilesM] = {};
    f32x4 w[kDepth][kStreamLoads], x[kDepth][kTilesM][kStreamLoads];
    const int first = wave * segment, end = first + segment < k ? first + segment : k;
    const auto fetch = [&](int at, int into) {         // a run that lies whole before the segment's end
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i) w[into][i] = load_whole<kVec>(brow + at + i * 16 + h);
#pragma unroll
        for (int t = 0; t < kTilesM; ++t)
#pragma unroll
            for (int i = 0; i < kStreamLoads; ++i) x[into][t][i] = load_whole<kVec>(arow[t] + at + i * 16 + h);
    };
    const auto multiply = [&](int from) {
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i) {
            const f32x4 wt = transpose_quarters(w[from][i]);
            f32x4 xt[kTilesM];
#pragma unroll
            for (int t = 0; t < kTilesM; ++t) xt[t] = transpose_quarters(x[from][t][i]);
            f32x4 acc[kTilesM] = {};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < kTilesM; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xt[t][j], wt[j], acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < kTilesM; ++t) sum[t] += acc[t];
        }
    };
    // whole runs, kDepth of them on their way at a time; the loop's body asks for a run on every pass, so that the compiler can
    // count the loads in flight
    int left = end > first ? (end - first) / kStreamRun : 0, at = first;
    if (left >= kDepth) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) fetch(at + d * kStreamRun, d);
        for (; left >= 2 * kDepth; left -= kDepth, at += kDepth * kStreamRun)
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                multiply(d);
                fetch(at + (kDepth + d) * kStreamRun, d);
            }
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            multiply(d);
            if (kDepth + d < left) fetch(at + (kDepth + d) * kStreamRun, d);
        }
        left -= kDepth, at += kDepth * kStreamRun;
    } else {
#pragma unroll
        for (int d = 0; d < kDepth - 1; ++d)
            if (d < left) fetch(at + d * kStreamRun, d);
    }
#pragma unroll
    for (int d = 0; d < kDepth - 1; ++d)
        if (d < left) multiply(d);
    at += left * kStreamRun;
    if (at < end) {                                    // the rest of the last segment, filled up with zeros
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i) w[0][i] = load_four<kVec>(brow, at + i * 16 + h, end);
#pragma unroll
        for (int t = 0; t < kTilesM; ++t)
#pragma unroll
            for (int i = 0; i < kStreamLoads; ++i) x[0][t][i] = load_four<kVec>(arow[t], at + i * 16 + h, end);
        multiply(0);
    }
#pragma unroll
    for (int t = 0; t < kTilesM; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[wave][t][(h + i) * kStreamTile + r] = sum[t][i];
    __syncthreads();
    for (int e = threadIdx.x; e < kTilesM * 256; e += kWaves * kWave) {
        const int t = e / 256, row = t * 16 + e % 256 / 16, col = n0 + e % 16;
        if (row >= m || col >= n) continue;
        float total = sums[0][t][e % 256];
#pragma unroll
        for (int v = 1; v < kWaves; ++v) total += sums[v][t][e % 256];        // (segments past K's end are zeros)
        c[static_cast<long>(row) * n + col] = total;
    }
}

// ---- many rows -----------------------------------------------------------------------------------------------------
// A tile of kRows x 64 outputs, four waves of a quarter each (32 x 32 x 2 instructions, kRows / 64 of them a wave).  Slabs of K in
// shared memory, rows 4 floats further apart than they are long (16-byte reads of 8 neighbouring
// rows then touch every bank once); the next slab is on its way into registers while one is multiplied, and is long enough
// (2048 cycles of instructions a wave) to arrive meanwhile.  Of every 8 elements the
// even ones lie first and then the odd ones: half-wave h reads its four at once, and the four instructions take elements 0
// and 1, 2 and 3, .. of them: k ascending.  A chain, a segment's sum of chains and the sum of segments each have registers of their
// own, which is what bounds the tile: 128 x 128 would need more than the 256 that two waves a SIMD leave each other.  1,024 rows
// against 12288 x 2048: 470 us, 110 TFLOP/s (one chain an output in tiles of 128 x 128: 452); 777 rows 440 (408).
//
// kCut: blockIdx.z takes `each` segments and leaves a plane of c for every one of them; else one workgroup walks them all.  kChains:
// segments are sums of chains of kChain elements, else one chain.
constexpr int slab_of(int rows) { return rows == 128 ? 32 : 64; }
constexpr int kTileCols = 64;

template <int kRows, bool kVec, bool kCut, bool kChains>
__global__ void __launch_bounds__(256, 2)
gemm_f32_tile_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k,
                     int segment, int each) {
    constexpr int kSlab = slab_of(kRows);
    constexpr int kFrag = kRows / 64;                  // 32 x 32 squares of a wave, one under the other
    constexpr int kLoadsA = kRows * kSlab / 4 / 256, kLoadsB = kTileCols * kSlab / 4 / 256;    // 16-byte loads a thread and slab
    __shared__ float as[2][kRows][kSlab + 4];
    __shared__ float bs[2][kTileCols][kSlab + 4];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int m0 = blockIdx.y * kRows, n0 = blockIdx.x * kTileCols;
    const long part = static_cast<long>(segment) * each;
    const int k_first = static_cast<int>(blockIdx.z * part), k_end = k - k_first > part ? static_cast<int>(k_first + part) : k;
    const int wm = (wave / 2) * (kRows / 2), wn = (wave % 2) * (kTileCols / 2);
    f32x16 acc[kFrag] = {}, sum[kFrag] = {}, total[kFrag] = {};
    f32x4 ra[kLoadsA], rb[kLoadsB];
    const auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) {
            const int idx = threadIdx.x + i * 256, row = m0 + idx / (kSlab / 4), at = k0 + (idx % (kSlab / 4)) * 4;
            ra[i] = load_four<kVec>(a + static_cast<long>(row < m ? row : m - 1) * k, at, k_end);
        }
#pragma unroll
        for (int i = 0; i < kLoadsB; ++i) {
            const int idx = threadIdx.x + i * 256, row = n0 + idx / (kSlab / 4), at = k0 + (idx % (kSlab / 4)) * 4;
            rb[i] = load_four<kVec>(b + static_cast<long>(row < n ? row : n - 1) * k, at, k_end);
        }
    };
    const auto put = [&](float* row, int at, const f32x4& v) {
        const int even = at / 8 * 8 + at % 8 / 2;
        *reinterpret_cast<f32x2*>(row + even) = f32x2{v[0], v[2]};
        *reinterpret_cast<f32x2*>(row + even + 4) = f32x2{v[1], v[3]};
    };
    const auto keep = [&](int into) {
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) {
            const int idx = threadIdx.x + i * 256;
            put(as[into][idx / (kSlab / 4)], (idx % (kSlab / 4)) * 4, ra[i]);
        }
#pragma unroll
        for (int i = 0; i < kLoadsB; ++i) {
            const int idx = threadIdx.x + i * 256;
            put(bs[into][idx / (kSlab / 4)], (idx % (kSlab / 4)) * 4, rb[i]);
        }
    };
    const auto store = [&](const f32x16 (&of)[kFrag], float* to) {
        const int col = n0 + wn + lane % 32;
#pragma unroll
        for (int i = 0; i < kFrag; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + wm + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
                if (row < m && col < n) to[static_cast<long>(row) * n + col] = of[i][e];
            }
    };
    fetch(k_first);
    keep(0);
    int at = 0, segment_left = segment;                // segments are whole slabs
    float* plane = c + static_cast<long>(blockIdx.z) * each * m * n;
    for (int k0 = k_first; k0 < k_end; k0 += kSlab, at ^= 1) {
        const bool more = k0 + kSlab < k_end;
        if (more) fetch(k0 + kSlab);
        __syncthreads();
        const int row = lane % 32, h = (lane / 32) * 4;
#pragma unroll
        for (int s = 0; s < kSlab; s += 8) {
            f32x4 av[kFrag];
            const f32x4 bv = *reinterpret_cast<const f32x4*>(&bs[at][wn + row][s + h]);
#pragma unroll
            for (int i = 0; i < kFrag; ++i) av[i] = *reinterpret_cast<const f32x4*>(&as[at][wm + i * 32 + row][s + h]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < kFrag; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i][e], bv[e], acc[i], 0, 0, 0);
            if (kChains && (s + 8) % kChain == 0) {
#pragma unroll
                for (int i = 0; i < kFrag; ++i) {
                    sum[i] += acc[i];
                    acc[i] = f32x16{};
                }
            }
        }
        if (more) keep(at ^ 1);        // read last two slabs ago, and every wave has passed a barrier since
        segment_left -= kSlab;
        if (segment_left == 0 || !more) {
            segment_left = segment;
            if constexpr (kCut) {
                store(sum, plane);
                plane += static_cast<long>(m) * n;
            }
#pragma unroll
            for (int i = 0; i < kFrag; ++i) {
                if constexpr (!kCut) total[i] += kChains ? sum[i] : acc[i];
                sum[i] = f32x16{};
            }
        }
    }
    if constexpr (!kCut) store(total, c);
}

// C = the planes' sum, in order.  kVec: planes and c are aligned to 16 bytes and `count` is a multiple of 4.
template <bool kVec>
__global__ void __launch_bounds__(256) gemm_f32_sum_kernel(const float* __restrict__ planes, float* __restrict__ c, long count, int parts) {
    const long at = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (kVec) {
        if (at >= count) return;
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

// Up to here a product is a stream of weights.  Measured against 2048 x 2048 and 12288 x 2048 weights (us, streamed : tiled): 14.1 :
// 14.3 and 40 : 43 at 24 rows, 15 : 14.5 and 43 : 44 at 32; beyond, the stream's reads of A, then four times the weights', cost more.
constexpr int kStreamRows = 32;
constexpr int kStreamK = 256;          // a shorter K is no work to share out over four waves: one segment, in tiles whatever the rows

// The segments of K: by K alone.  Eight from 512 elements on (a wave each of a streaming workgroup), four from 256, multiples
// of 64 elements (a streaming wave's run, and whole slabs of a tile).
struct F32Segments {
    int length, count;
};
F32Segments f32_segments(int k) {
    const int wanted = k < kStreamK ? 1 : k < 2 * kStreamK ? 4 : 8;
    const int length = ceil_div(ceil_div(k, wanted), kStreamRun) * kStreamRun;
    return {length, ceil_div(k, length)};
}

struct F32Plan {
    int rows = 0, parts = 1, each = 1;                 // rows of a tile, 0: the streaming kernel; parts workgroups of `each` segments along K
};

// The tile and the cut of K that take least time.  A compute unit's matrix instructions run at one rate however many tiles it
// holds, so the product takes as long as the fullest of the 256 units has work for; one tile a unit leaves a wave a SIMD and
// its waits in the open.  A cut K costs a plane written and read for every segment (mostly in the caches) and a second launch.
// Constants fitted to every tile and cut timed at 33 to 1,024 rows against 512 x 512 to 32768 x 2048 and 2048 x 6144 weights: the
// choice is within 6 % of the best at each.
F32Plan f32_plan(int m, int n, int k) {
    F32Plan best;
    const F32Segments segments = f32_segments(k);
    best.each = segments.count;
    if (m <= kStreamRows && k >= kStreamK) return best;
    constexpr long kUnits = 256;
    constexpr double kUnitRate = 0.6e6, kPlaneRate = 30e6, kLaunch = 6.0;      // operations and bytes a microsecond; microseconds
    double least = 0.0;
    for (int rows : {128, 64}) {
        const long tiles = static_cast<long>(ceil_div(m, rows)) * ceil_div(n, kTileCols);
        for (int wanted = 1; wanted <= segments.count; wanted *= 2) {
            const int each = ceil_div(segments.count, wanted), parts = ceil_div(segments.count, each);
            const long held = (tiles * parts + kUnits - 1) / kUnits;           // of the fullest unit
            const double hidden = rows == 128 ? (held >= 2 ? 0.87 : 0.4) : (held >= 2 ? 0.82 : 0.65);
            const double product = 2.0 * held * rows * kTileCols * segments.length * each / (kUnitRate * hidden);
            const double planes = parts == 1 ? 0.0 : kLaunch + 8.0 * segments.count * m * n / kPlaneRate;
            if (best.rows == 0 || product + planes < least * 0.999) {
                least = product + planes;
                best.rows = rows, best.parts = parts, best.each = each;
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
    return p.parts > 1 ? f32_segments(k).count : 0;
}

// planes: room for leone_gemm_f32_planes(m, n, k) results (null if that is 0).
extern "C" int leone_gemm_f32(const float* a, const float* b, float* c, float* planes, int m, int n, int k, hipStream_t stream) {
    LEONE_REQUIRE(a && b && c, "gemm_f32: null pointer");
    LEONE_REQUIRE(m > 0 && n > 0 && k > 0, "gemm_f32: sizes %d x %d x %d must be positive", m, n, k);
    const F32Plan p = f32_plan(m, n, k);
    const F32Segments segments = f32_segments(k);
    LEONE_REQUIRE(p.parts == 1 || planes, "gemm_f32: %d planes are needed for %d x %d x %d", segments.count, m, n, k);
    const auto aligned = [](const void* at) { return reinterpret_cast<uintptr_t>(at) % 16 == 0; };
    const bool vec = k % 4 == 0 && aligned(a) && aligned(b);
    if (p.rows == 0) {
        const int blocks = ceil_div(n, kStreamTile);
#define LEONE_STREAM(T, W, D)                                                                                                          \
    (vec ? gemm_f32_stream_kernel<T, W, D, true><<<blocks, W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length)                  \
         : gemm_f32_stream_kernel<T, W, D, false><<<blocks, W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length))
        // Runs on their way a wave: two leave room for more waves, whose loads count as well (one row against 12288 x 2048 18.4 us,
        // with four 24.4); two tiles of A take long enough over a run for three (24 rows against 2048 x 6144 37.8, with four 43.1).
        if (segments.count <= 4) {
            if (m <= kStreamTile) LEONE_STREAM(1, 4, 2);
            else LEONE_STREAM(2, 4, 3);
        } else {
            if (m <= kStreamTile) LEONE_STREAM(1, 8, 2);
            else LEONE_STREAM(2, 8, 3);
        }
#undef LEONE_STREAM
        LEONE_LAUNCH_CHECK("gemm_f32");
        return 0;
    }
    const int grid_y = ceil_div(m, p.rows);
    LEONE_REQUIRE(grid_y <= 65535, "gemm_f32: %d rows exceed the launch limit", m);
    const dim3 grid(ceil_div(n, kTileCols), grid_y, p.parts);
#define LEONE_TILE_CHAIN(E, V, CHAIN)                                                                                                  \
    (p.parts > 1 ? gemm_f32_tile_kernel<E, V, true, CHAIN><<<grid, 256, 0, stream>>>(a, b, planes, m, n, k, segments.length, p.each)   \
                 : gemm_f32_tile_kernel<E, V, false, CHAIN><<<grid, 256, 0, stream>>>(a, b, c, m, n, k, segments.length, p.each))
#define LEONE_TILE(E, V)                                                                                                               \
    (segments.count > 1 ? LEONE_TILE_CHAIN(E, V, true)                                                                               \
                        : gemm_f32_tile_kernel<E, V, false, false><<<grid, 256, 0, stream>>>(a, b, c, m, n, k, segments.length, p.each))
    if (p.rows == 128) {
        if (vec) LEONE_TILE(128, true);
        else LEONE_TILE(128, false);
    } else {
        if (vec) LEONE_TILE(64, true);
        else LEONE_TILE(64, false);
    }
#undef LEONE_TILE_CHAIN
#undef LEONE_TILE
    LEONE_LAUNCH_CHECK("gemm_f32");
    if (p.parts > 1) {
        const long count = static_cast<long>(m) * n;
        const int blocks = ceil_div(count, 1024);
        if (count % 4 == 0 && aligned(planes) && aligned(c))
            gemm_f32_sum_kernel<true><<<blocks, 256, 0, stream>>>(planes, c, count, segments.count);
        else
            gemm_f32_sum_kernel<false><<<blocks, 256, 0, stream>>>(planes, c, count, segments.count);
        LEONE_LAUNCH_CHECK("gemm_f32 sum");
    }
    return 0;
}
