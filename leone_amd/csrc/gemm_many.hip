// Matrix products of many rows: a step's prompt portions, the prompts of a few requests, decode steps of 17 requests and more.  Y[M,N] = X[M,K] . W[N,K]^T for bfloat16 X and the tiled copy of bfloat16 W (see leone_hip.h).
//
// A workgroup of four waves (or two, or three) takes 32 kMT rows and 32 kNT columns a wave, in parts of 32.  The wave's own elements
// of W come from memory as its instruction (32 x 32 x 16) wants them, one to four stages of 64 elements of K ahead, and pass neither through
// shared memory nor a barrier.  X, which all waves read, goes through shared memory, a stage's 128 bytes of a row turned about by the row's
// number so that the same piece of 16 rows lies in 16 places; a stage is written while the one before it is worked on.
//
// What bounds it: with few tiles the time one takes (0.28 us a stage for 64 x 128, 0.33 for 96 x 128, 0.40 for 128 x 128, 0.53 for 96 x 256,
// which a second tile on the same unit doubles), so a product with fewer tiles than units is cut along K, into planes, where its caller
// takes them; with many, the chip's power, where the vendor library with its 256 x 256 tiles is as good or better (6,144 x 4,096 for 2,048 rows: 81
// us here, 67 there).  ops.many_plan chooses; its comment has both sides' figures.
//
// kDeep, for up to 128 rows: what bounds it is memory, that is, the bytes that a unit has asked for and not yet got.  Four stages of W are on their way (64
// KB of 128 columns, where the kernel of gemm_rows.hip has 32 KB), asked for with the hint that they are read once, and the last four stages ask for
// nothing; workgroups of two or three waves take 64 or 96 columns where 128 would leave units without work.  us, 64 rows, gemm_rows.hip and here: 4,096 x
// 12,288 24.3 and 21.3 (4.7 TB/s), 6,144 x 4,096 16.5 and 11.7, 4,096 x 4,096 12.4 and 10.1, 2,048 x 2,048 6.7 and 5.4, gated 24,576 x 4,096 41.9 and 37.2.
// Beyond 64 rows there are one or two rows of tiles, whatever is faster; with two, W is asked for twice, by workgroups that work side by side.  The hint
// is worth its while there too (128 rows in two rows of tiles, with it and without: 6,144 x 4,096 17.5 and 18.8, 4,096 x 4,096 13.1 and 13.9, 4,096 x 12,288
// 31.5 and 32.6, gated 12,288 x 2,048 20.6 and 21.6), but not for the smallest matrices (1,024 x 3,072 5.6 and 5.0; 64 rows 5.2 and 4.6).
// ops.deep_plan chooses.
//
// The walk along the stages and the turned stores stand in moe_product_many_kernel (routed.hip) as well: what is mended in one is mended in both.
#include "common.h"

#include <type_traits>

namespace leone {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

enum ManyOut : int { kManyStore = 0, kManyResidual = 1, kManyGated = 2, kManyPlanes = 3 };

struct ManyArgs {
    const bf16_t* x;
    const bf16_t* w;
    void* y;
    long plane;                  // elements from plane to plane
    int m, n, k, tiles_m, tiles_n, splits, per, act;
    float limit;
};

template <int kMT, int kNT, int kWaves, bool kDeep, int kOut, typename TOut>
__global__ void __launch_bounds__(kWaves * kWave, kDeep ? (kMT == 1 || (kMT == 2 && kWaves == 4) ? 3 : 2) : kNT == 1 ? 3 : 2)
gemm_many_kernel(ManyArgs a) {
    constexpr int kThreads = kWaves * kWave, kRows = 32 * kMT, kPieces = kRows * 8, kCopies = (kPieces + kThreads - 1) / kThreads;
    // stages of W and of X on their way in registers; stages that the loop takes at a time
    constexpr int kWAhead = kDeep ? 4 : kNT == 1 ? 2 : 1, kAhead = kMT <= 2 ? 2 : 1, kTurns = kDeep ? 4 : 2;
    __shared__ uint4 sx[2][kPieces > kWaves * 128 ? kPieces : kWaves * 128];
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int c = lane & 31, hi = lane >> 5;
    const int tiles = a.tiles_m * a.tiles_n, total = tiles * a.splits;
    // Workgroups go to the eight dies in turn: a die gets a run of neighbouring tiles, of eight rows of tiles a block of columns after the
    // other, whose pieces of X and W it then reads from its own cache.
    const int xcd = blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
    int at = xcd * q8 + (xcd < r8 ? xcd : r8) + static_cast<int>(blockIdx.x >> 3);
    const int split = at / tiles;
    at -= split * tiles;
    constexpr int kGroup = 8;
    const int group = at / (kGroup * a.tiles_n), in_group = at - group * kGroup * a.tiles_n;
    const int rows_here = a.tiles_m - group * kGroup < kGroup ? a.tiles_m - group * kGroup : kGroup;
    const int tn = in_group / rows_here, tm = group * kGroup + in_group % rows_here;
    const int all = a.k / 64, s0 = split * a.per, count = s0 + a.per < all ? a.per : all - s0;
    const bf16_t* wp[kNT];
#pragma unroll
    for (int u = 0; u < kNT; ++u) {
        // the lane's row of W (gated: gate and up rows take turns by eights); past the last the last again, not written
        const int want = ((tn * kWaves + wave) * kNT + u) * 2 + (c >> 4), t16 = want < a.n / 16 ? want : a.n / 16 - 1;
        wp[u] = a.w + (static_cast<long>(t16) * all + s0) * 1024 + hi * 128 + (c & 15) * 8;
    }
    const bf16_t* x_from[kCopies];
    int x_to[kCopies];
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
        const int q = (i * kThreads + tid) % kPieces, row = q >> 3, part = q & 7;         // (past the last piece one again: the same bytes)
        const int wanted = tm * kRows + row, gr = wanted < a.m ? wanted : a.m - 1;
        x_from[i] = a.x + static_cast<long>(gr) * a.k + s0 * 64 + part * 8;
        x_to[i] = row * 8 + (part ^ ((row >> 1) & 7));
    }
    const auto inside = [&](int s) { return s < count ? s : count - 1; };                // (past the end the last stage again, unused)
    const auto load_x = [&](int s, int i) { return *reinterpret_cast<const uint4*>(x_from[i] + static_cast<long>(inside(s)) * 64); };
    const auto load_w = [&](int s, int j, int u) {
        const bf16_t* from = wp[u] + static_cast<long>(inside(s)) * 1024 + (j >> 1) * 512 + (j & 1) * 256;
        if constexpr (kDeep) return load_streamed16(from);
        else return *reinterpret_cast<const uint4*>(from);
    };
    floatx16 acc[kMT][kNT];
#pragma unroll
    for (int t = 0; t < kMT; ++t)
#pragma unroll
        for (int u = 0; u < kNT; ++u)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][u][i] = 0.f;
    uint4 held[kAhead][kCopies], wr[kWAhead][4][kNT];
    bf16x8 xb[2][kMT];
    const auto read_x = [&](const uint4* from, int j, int t) {
        const int row = 32 * t + c, ch = 4 * (j & 1) + 2 * hi + (j >> 1);              // (the elements that the copy of W holds there)
        return __builtin_bit_cast(bf16x8, from[row * 8 + (ch ^ ((row >> 1) & 7))]);
    };
    // The i-th copy belongs to this place among a stage's 4 kMT pairs of a read and an instruction: within the first three quarters, behind
    // which the stage's barrier stands.  The loads ahead of the loop are asked for in the loop's order, or the compiler, which counts the
    // loads in flight, would wait for younger ones.
    const auto place_of = [&](int i) { return i * 3 * kMT / kCopies; };
    {
        uint4 first[kCopies];
#pragma unroll
        for (int i = 0; i < kCopies; ++i) first[i] = load_x(0, i);
#pragma unroll
        for (int v = 0; v < kTurns; ++v)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int i = 0; i < kCopies; ++i)
                    if (place_of(i) / kMT == j && v >= kTurns - kAhead) held[(v + 1 + kAhead) % kAhead][i] = load_x(v + 1 - kTurns + kAhead, i);
                if (v >= kTurns - kWAhead)
#pragma unroll
                    for (int u = 0; u < kNT; ++u) wr[v % kWAhead][j][u] = load_w(v - kTurns + kWAhead, j, u);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int i = 0; i < kCopies; ++i) sx[0][x_to[i]] = first[i];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kMT; ++t) xb[0][t] = read_x(sx[0], 0, t);
    const auto stage = [&](int s, auto number, auto last) {
        constexpr int at_turn = decltype(number)::value, p = at_turn & 1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j == 3) {                                // the next stage lies in shared memory, and everyone has read this one
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            }
#pragma unroll
            for (int t = 0; t < kMT; ++t) {
                xb[(j + 1) & 1][t] = j < 3 ? read_x(sx[p], j + 1, t) : read_x(sx[p ^ 1], 0, t);
#pragma unroll
                for (int i = 0; i < kCopies; ++i)
                    if (place_of(i) == j * kMT + t) {
                        sx[p ^ 1][x_to[i]] = held[(p + 1) % kAhead][i];
                        held[(p + 1) % kAhead][i] = load_x(s + 1 + kAhead, i);
                    }
#pragma unroll
                for (int u = 0; u < kNT; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wr[at_turn % kWAhead][j][u]), xb[j & 1][t], acc[t][u], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!decltype(last)::value)
#pragma unroll
                for (int u = 0; u < kNT; ++u) wr[at_turn % kWAhead][j][u] = load_w(s + kWAhead, j, u);
        }
    };
    int s = 0;
    if constexpr (kDeep) {
        const std::false_type more;
        const std::true_type last;                       // (of W nothing is asked for any more)
        for (; s + kTurns < count; s += kTurns) {
            stage(s, std::integral_constant<int, 0>{}, more);
            stage(s + 1, std::integral_constant<int, 1>{}, more);
            stage(s + 2, std::integral_constant<int, 2>{}, more);
            stage(s + 3, std::integral_constant<int, 3>{}, more);
        }
        stage(s, std::integral_constant<int, 0>{}, last);
        if (s + 1 < count) {
            stage(s + 1, std::integral_constant<int, 1>{}, last);
            if (s + 2 < count) {
                stage(s + 2, std::integral_constant<int, 2>{}, last);
                if (s + 3 < count) stage(s + 3, std::integral_constant<int, 3>{}, last);
            }
        }
    } else {
        const std::false_type more;
        for (; s + 1 < count; s += 2) {
            stage(s, std::integral_constant<int, 0>{}, more);
            stage(s + 1, std::integral_constant<int, 1>{}, more);
        }
        if (s < count) stage(s, std::integral_constant<int, 0>{}, more);
    }
    // Lane (c, hi) holds, of row c of every t, columns 8 q + 4 hi .. + 3 of each of the wave's 32.  They are turned in shared memory, a wave's
    // own part of it, so that a store covers whole runs of a row (straight from the registers it would be 16 bytes of 32 rows).
    __syncthreads();                                     // the last stage has been read
    constexpr bool kGate = kOut == kManyGated;
    constexpr int kBytes = kOut == kManyStore || kGate ? static_cast<int>(sizeof(TOut)) : 4;
    constexpr int kPart = kGate ? 16 : 32;                           // results of one of the wave's parts
    constexpr int kAtOnce = kBytes == 4 ? 1 : kNT;                   // of these parts
    constexpr int kRun = kPart * kAtOnce * kBytes / 16;              // 16-byte pieces of a row at once
    static_assert(kRun * 32 * 16 <= sizeof(sx) / kWaves && (kRun == 2 || kRun == 4 || kRun == 8), "a wave's part of the stages' memory");
    uint4* mine = &sx[0][0] + wave * (kRun * 32);
    const auto turn = [](int r) { return (kRun == 8 ? r >> 1 : kRun == 4 ? r >> 2 : r >> 3) & (kRun - 1); };
    const int width = kGate ? a.n / 2 : a.n;
    const int col0 = (tn * kWaves + wave) * kNT * kPart;
    char* out = static_cast<char*>(a.y) + (kOut == kManyPlanes ? split * a.plane * 4 : 0);
#pragma unroll
    for (int t = 0; t < kMT; ++t)
#pragma unroll
        for (int u0 = 0; u0 < kNT; u0 += kAtOnce) {
            const int row_t = tm * kRows + 32 * t;
            float4 old[kOut == kManyResidual ? kRun / 2 : 1];
            if constexpr (kOut == kManyResidual) {
#pragma unroll
                for (int i = 0; i < kRun / 2; ++i) {
                    const int row = row_t + i * (64 / kRun) + lane / kRun, col = col0 + u0 * kPart + lane % kRun * 4;
                    old[i] = *reinterpret_cast<const float4*>(out + (static_cast<long>(row < a.m ? row : a.m - 1) * width + (col < width ? col : 0)) * 4);
                }
            }
#pragma unroll
            for (int u = u0; u < u0 + kAtOnce; ++u)
#pragma unroll
                for (int q = 0; q < 4; q += kGate ? 2 : 1) {
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[j] = acc[t][u][4 * q + j];
                        if constexpr (kGate) {
                            float gate = v[j], up = acc[t][u][(4 * q + 4 + j) & 15];
                            if constexpr (!kDeep) {                  // both rounded first, as they are where a kernel of its own does this
                                gate = to_float(from_float<bf16_t>(gate));
                                up = to_float(from_float<bf16_t>(up));
                            }
                            v[j] = glu_value(gate, up, a.act, a.limit);
                        }
                    }
                    const int first = (u - u0) * kPart + (kGate ? 4 * q : 8 * q) + 4 * hi, piece = (first * kBytes / 16) ^ turn(c);
                    if constexpr (kBytes == 4) {
                        mine[c * kRun + piece] = __builtin_bit_cast(uint4, float4{v[0], v[1], v[2], v[3]});
                    } else {
                        uint2 pk;
                        pk.x = bf16_bits_from_float(v[0]) | (unsigned(bf16_bits_from_float(v[1])) << 16);
                        pk.y = bf16_bits_from_float(v[2]) | (unsigned(bf16_bits_from_float(v[3])) << 16);
                        reinterpret_cast<uint2*>(mine)[2 * (c * kRun + piece) + hi] = pk;
                    }
                }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < kRun / 2; ++i) {
                const int r = i * (64 / kRun) + lane / kRun, piece = lane % kRun, row = row_t + r, col = col0 + u0 * kPart + piece * (16 / kBytes);
                uint4 whole = mine[r * kRun + (piece ^ turn(r))];
                if constexpr (kOut == kManyResidual) {
                    float4 f = __builtin_bit_cast(float4, whole);
                    f.x += old[i].x;
                    f.y += old[i].y;
                    f.z += old[i].z;
                    f.w += old[i].w;
                    whole = __builtin_bit_cast(uint4, f);
                }
                if (row < a.m && col < width)
                    *reinterpret_cast<uint4*>(out + (static_cast<long>(row) * width + col) * kBytes) = whole;
            }
            __builtin_amdgcn_wave_barrier();
        }
}

template <int kMT, int kNT, int kWaves, bool kDeep>
void launch_many(ManyArgs a, int out_mode, int out_dtype, hipStream_t stream) {
    a.tiles_m = ceil_div(a.m, 32 * kMT);
    a.tiles_n = ceil_div(a.n, 32 * kWaves * kNT);
    const int groups = a.tiles_m * a.tiles_n * a.splits, threads = kWaves * kWave;
    if (out_mode == kManyResidual) gemm_many_kernel<kMT, kNT, kWaves, kDeep, kManyResidual, float><<<groups, threads, 0, stream>>>(a);
    else if (out_mode == kManyGated) gemm_many_kernel<kMT, kNT, kWaves, kDeep, kManyGated, bf16_t><<<groups, threads, 0, stream>>>(a);
    else if (out_mode == kManyPlanes) gemm_many_kernel<kMT, kNT, kWaves, kDeep, kManyPlanes, float><<<groups, threads, 0, stream>>>(a);
    else if (out_dtype == kF32) gemm_many_kernel<kMT, kNT, kWaves, kDeep, kManyStore, float><<<groups, threads, 0, stream>>>(a);
    else gemm_many_kernel<kMT, kNT, kWaves, kDeep, kManyStore, bf16_t><<<groups, threads, 0, stream>>>(a);
}

}  // namespace leone

using namespace leone;

extern "C" int leone_gemm_many_bf16(const void* x, const void* w, void* y, int out_mode, int out_dtype, int m, int n, int k, int splits,
                                    long plane, int tile_rows, int tile_columns, int deep, int act, float limit, hipStream_t stream) {
    LEONE_REQUIRE(x && w && y, "gemm_many: null pointer");
    LEONE_REQUIRE(m > 0 && n > 0 && k > 0 && n % 16 == 0 && k % 64 == 0, "gemm_many: bad sizes %d x %d x %d", m, n, k);
    LEONE_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y)) % 16 == 0,
                  "gemm_many: operands must begin at a multiple of 16 bytes");
    LEONE_REQUIRE(out_mode >= kManyStore && out_mode <= kManyPlanes, "gemm_many: unknown kind of output %d", out_mode);
    LEONE_REQUIRE(out_mode != kManyStore || out_dtype == kF32 || out_dtype == kBF16, "gemm_many: unknown output type");
    LEONE_REQUIRE(out_mode != kManyGated || act == kGateSilu || act == kGateGeluTanh || (act == kGateClampedSwish && limit > 0.f),
                  "gemm_many: unknown activation %d (limit %g)", act, limit);
    const int stages = k / 64;
    LEONE_REQUIRE(splits >= 1 && splits <= stages && (splits == 1 || out_mode == kManyPlanes), "gemm_many: %d ranges of K", splits);
    const int per = ceil_div(stages, splits);
    LEONE_REQUIRE(per * (splits - 1) < stages, "gemm_many: %d ranges of K would leave one empty (%d stages)", splits, stages);
    LEONE_REQUIRE(out_mode != kManyPlanes || (plane >= static_cast<long>(m) * n && plane % 4 == 0), "gemm_many: planes overlap");
    LEONE_REQUIRE(static_cast<long>(ceil_div(m, 32)) * ceil_div(n, 64) * splits < (1l << 30), "gemm_many: %d x %d is too large", m, n);
    const ManyArgs a{static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), y, plane, m, n, k, 0, 0, splits, per, act, limit};
    if (deep) {
        switch (tile_rows * 1000 + tile_columns) {
            case 32064: launch_many<1, 1, 2, true>(a, out_mode, out_dtype, stream); break;
            case 64064: launch_many<2, 1, 2, true>(a, out_mode, out_dtype, stream); break;
            case 32096: launch_many<1, 1, 3, true>(a, out_mode, out_dtype, stream); break;
            case 64096: launch_many<2, 1, 3, true>(a, out_mode, out_dtype, stream); break;
            case 64128: launch_many<2, 1, 4, true>(a, out_mode, out_dtype, stream); break;
            case 96128: launch_many<3, 1, 4, true>(a, out_mode, out_dtype, stream); break;
            case 128128: launch_many<4, 1, 4, true>(a, out_mode, out_dtype, stream); break;
            default: set_error("gemm_many: tiles of %d x %d are not built", tile_rows, tile_columns); return 1;
        }
    } else if (tile_rows == 64 && tile_columns == 128) launch_many<2, 1, 4, false>(a, out_mode, out_dtype, stream);
    else if (tile_rows == 96 && tile_columns == 128) launch_many<3, 1, 4, false>(a, out_mode, out_dtype, stream);
    else if (tile_rows == 128 && tile_columns == 128) launch_many<4, 1, 4, false>(a, out_mode, out_dtype, stream);
    else if (tile_rows == 96 && tile_columns == 256) launch_many<3, 2, 4, false>(a, out_mode, out_dtype, stream);
    else {
        set_error("gemm_many: tiles of %d x %d are not built", tile_rows, tile_columns);
        return 1;
    }
    LEONE_LAUNCH_CHECK("gemm_many");
    return 0;
}
