// Single-precision matrix product for the true 32-bit path: C[M,N] = A[M,K] . B[N,K]^T, operands, products and sums with a float's 24
// bits (no reduced-precision mode).  A K below 256 goes to the float matrix instructions; from there on to those of bfloat16, every
// number taken apart into three.  The reference's scalar backend folds each output left to right in float (crates/leone/src/cpu.rs:1379-1405,
// 1622-1640).
//
// An output's bits depend on its row of A, its row of B and K alone, never on the rows that share the launch (what a request gets
// does not depend on who is beside it): K is cut into segments by a rule on K (f32_segments), a segment's sum is that of the sums of 32
// products, k ascending, added in order, and so is the segments' sum.  A K below 256 is one chain of float products, the scalar
// backend's fold.
//
// The matrix instructions take floats at a sixteenth of the rate of bfloat16.  From a K of 256 on, numbers are therefore taken apart
// into three bfloat16 each, which hold all of their 24 bits, and a product is made of eight of the nine products of parts (the method is
// published: Henry, Tang, Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations", 2019):
// twice the float rate.  The sums of 32 round less often than chains of float products do (error against 64 bits over the
// result's norm, 1 to 1,024 rows: K 512 0.7e-7, 2048 0.9e-7, 6144 1.1e-7; chains of 16 float products 1.0e-7, 1.2e-7 and 1.6e-7), and a
// row's only product is rounded as a float product is (at most 1.003 of 2^-24 off, 0.15 % not to the nearest).
//
// Few rows (decoding): a product reads every weight once for 2 M operations, so the weights' bytes are the
// bound and what matters is how much of them is in flight: a workgroup owns 16 rows of B, its waves take a segment each, and a
// wave keeps its next loads of B in the air.  Many rows (prompt portions): tiles, whose rows of A are staged through shared memory.
// With few tiles the segments are shared out over workgroups, which leave them as planes in a buffer of the caller's for a second
// kernel to add.
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

// ---- three parts a number --------------------------------------------------------------------------------------------
// The 16 x 16 x 32 instruction takes eight bfloat16 a lane and adds in float.  A float is the sum of three bfloat16 (8 bits each,
// rounded to nearest, so that what is left is at most half of the last bit and of either sign).  Of the nine products of two floats' parts the
// one of both last parts is left out: it is at most 2^-32 of the product.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// The next part of two numbers, taken off them.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ inline unsigned next_part(float& a, float& b) {
    unsigned bits = __builtin_bit_cast(unsigned, bf16x2{static_cast<__bf16>(a), static_cast<__bf16>(b)});
    asm("" : "+v"(bits));          // (one conversion of both, not another of each for what is taken off)
    a -= __uint_as_float(bits << 16);
    b -= __uint_as_float(bits & 0xffff0000u);
    return bits;
}
// Four numbers' parts, highest first.
struct FourParts {
    u32x2 part[3];
};
__device__ inline FourParts parts_of(f32x4 v) {
    FourParts r;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        float a = v[0], b = v[1], c = v[2], d = v[3];
        const unsigned low = next_part(a, b), high = next_part(c, d);
        r.part[p] = u32x2{low, high};
        v = f32x4{a, b, c, d};
    }
    return r;
}
// A lane's operand of one instruction: eight numbers in three parts.
struct Operand {
    bf16x8 part[3];
};
__device__ inline Operand operand_of(const f32x4& first, const f32x4& second) {
    const FourParts a = parts_of(first), b = parts_of(second);
    Operand r;
#pragma unroll
    for (int p = 0; p < 3; ++p) r.part[p] = __builtin_bit_cast(bf16x8, u32x4{a.part[p][0], a.part[p][1], b.part[p][0], b.part[p][1]});
    return r;
}
// The sum of 32 products: those of lower parts, the smallest first, and those of both highest parts, which a float addition rounds (added to
// the others by the instruction, a fifth of lone products came out one off).  What the instruction loses when it brings its products to one exponent it takes
// off, whatever their sign (sums of 2,048 come out 5e-8 of their root mean square too low), so every other 32 elements of a segment
// are multiplied with A's sign turned and their sum is subtracted.
constexpr int kTerms = 7, kTermA[kTerms] = {2, 1, 2, 0, 1, 1, 0}, kTermB[kTerms] = {1, 2, 0, 2, 1, 0, 1};
__device__ inline f32x4 add_term(int term, const Operand& a, const Operand& b, const f32x4& sum) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.part[kTermA[term]], b.part[kTermB[term]], sum, 0, 0, 0);
}
__device__ inline f32x4 highest_term(const Operand& a, const Operand& b) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.part[0], b.part[0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
}
// An infinity has no parts (what is left of it is not a number), and neither have numbers that round to one; and what lies below
// bfloat16's least number, 2^-133, is lost from the parts of a number below 2^-110, and from the products of parts what lies below a
// float's, which counts where the other factor is large.  A segment's sum that comes out infinite or NaN, or so small beside the largest
// numbers of its row of A and its row of B that what is lost could count, is therefore made again on the float instructions.  For
// largest numbers a and b less than 2^-132 max(a, 1) max(b, 1) is lost a product (half of 2^-133 of either factor times the other, and eight
// products' 2^-149); a sum is in doubt below 2^-90 max(a, 1) max(b, 1), so that others lose less than half of a float's last bit up to
// segments of 2^17.  Rows of zeros are not in doubt.
// A row's share of the limit below which a sum is in doubt (0: never); the sum's own: their product.
__device__ inline float least_of(float largest) { return largest > 0.f ? fmaxf(largest, 1.0f) * 0x1p-45f : 0.f; }
__device__ inline bool in_doubt(float v, float least_a, float least_b) {
    return fmaf(-least_a, least_b, fabsf(v)) < 0.f || !(fabsf(v) <= 3.402823466e38f);
}
// No sum is in doubt where no factor lies above the one bound and every sum is a number not below the other (seen without a word between
// the lanes; the limit of factors of 2^30 is 2^-30).
__device__ inline bool beyond_doubt(float largest, float least_sum, float no_number) {
    return largest <= 0x1p30f && least_sum >= 0x1p-30f && no_number == 0.f;
}
// The largest absolute value so far (of NaN any: it spoils its sum).  Two instructions for four numbers; from fmaxf and fabsf the
// compiler makes more, to quiet NaN first.
__device__ inline float largest_of(float so_far, const f32x4& v) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(so_far) : "v"(v[0]), "v"(v[1]));
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(so_far) : "v"(v[2]), "v"(v[3]));
    return so_far;
}
// Register j of quarter g becomes register g of quarter j.
__device__ inline f32x4 transpose_quarters(const f32x4 v) {
    const auto bits = [](float f) { return __float_as_uint(f); };
    const u32x2 p = __builtin_amdgcn_permlane32_swap(bits(v[0]), bits(v[2]), false, false);
    const u32x2 q = __builtin_amdgcn_permlane32_swap(bits(v[1]), bits(v[3]), false, false);
    const u32x2 r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    const u32x2 s = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    return f32x4{__uint_as_float(r[0]), __uint_as_float(r[1]), __uint_as_float(s[0]), __uint_as_float(s[1])};
}
// Elements of a normed row, rounded as the norm's own kernel rounds them (not taken into a subtraction of what follows).
__device__ inline f32x4 normed(const f32x4& v, const f32x4& gain, float inv) {
#pragma clang fp contract(off)
    return v * gain * inv;
}
// The segment's sums of a square of 16 x 16 outputs on the float instructions: 16 products a chain, k ascending, and the chains' sums
// added in order.  This lane's row of A and row of B are those of number lane % 16 of the square; what comes out lies as the bfloat16
// instruction's results do, and depends on an output's own two rows alone.  The 16 x 16 x 4 instruction adds its four products in the
// order of the lanes' quarters, so the four quarters' registers are transposed by lane swaps: instruction j takes elements 4 j .. 4 j + 3
// in turn; the next run is on its way meanwhile.  (By a loop over K for every output in doubt, a row that is not a number held up whoever
// shared its launch.  us, all sums ordinary, one row NaN, all rows: one row against 2048 x 2048 6.5, 14, 14 (by a loop 100); five against 32768 x
// 2048 44, 94, 90; 200 against 3072 x 2048 36, 48, 113 (79 and 2842); 777 against 12288 x 2048 298, 344, 1408 (287 and 38668).)
constexpr int kPlainRun = 16;                          // elements of K on their way at a time
// kNormed: A's elements are (a * gain) * inv.
template <bool kVec, bool kNormed = false>
__device__ inline f32x4 plain_square(const float* __restrict__ arow, const float* __restrict__ brow, int first, int end, int g,
                                     const float* __restrict__ gain = nullptr, float inv = 1.0f) {
    const auto of_a = [&](int at) {
        f32x4 v = load_four<kVec>(arow, at, end);
        if constexpr (kNormed) v = normed(v, load_four<kVec>(gain, at, end), inv);
        return v;
    };
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    constexpr int kLoads = kPlainRun / 16;
    f32x4 x[kLoads], y[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) x[i] = of_a(first + i * 16 + 4 * g), y[i] = load_four<kVec>(brow, first + i * 16 + 4 * g, end);
#pragma unroll 1
    for (int at = first; at < end; at += kPlainRun) {
        f32x4 next_x[kLoads], next_y[kLoads];
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            next_x[i] = of_a(at + kPlainRun + i * 16 + 4 * g);
            next_y[i] = load_four<kVec>(brow, at + kPlainRun + i * 16 + 4 * g, end);
        }
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const f32x4 xt = transpose_quarters(x[i]), yt = transpose_quarters(y[i]);
            f32x4 chain = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; ++j) chain = __builtin_amdgcn_mfma_f32_16x16x4f32(xt[j], yt[j], chain, 0, 0, 0);
            sum += chain;
            x[i] = next_x[i], y[i] = next_y[i];
        }
    }
    return sum;
}

// What is done with finished sums: nothing, or (B's rows are 8 gates, their 8 ups, and so on) act(gate) * up of every pair.
struct Epilogue {
    int gated = 0, act = 0;
    float limit = 0.f;
};

// ---- few rows ------------------------------------------------------------------------------------------------------
// Lane l of a wave loads, of 16 rows of B, row l % 16's elements 4 (l / 16) .. + 3 of every run of 16: one 16-byte load
// a lane is 64 bytes of each of 16 rows.  A's rows lie the same way, out of the caches (rows past the last are the last one again
// and not written).  Two such runs are a lane's eight numbers of an instruction.
constexpr int kStreamTile = 16;                        // rows of B a workgroup
constexpr int kStreamRun = 32;                         // elements of K a wave takes at a time
constexpr int kStreamLoads = kStreamRun / 16;
constexpr int kChain = 32;                             // elements of K whose products are added up before they meet a sum

// The waves' sums of the workgroup's tiles, added and stored.
// kAdds (one tile): what lay in c before, of the thread's one element, is added.
// kCols: of the tile's 16 columns the first so many count.
template <int kTilesM, int kTilesN, int kWaves, bool kAdds = false, int kCols = kStreamTile>
__device__ inline void add_segments(const float (&sums)[kWaves][kTilesM][kTilesN][kStreamTile * kStreamTile], float* __restrict__ c, int m, int n,
                                    int n0, const Epilogue& then, float before = 0.f) {
    static_assert(!kAdds || (kTilesM == 1 && kTilesN == 1 && kWaves * kWave >= 256), "an element a thread");
    if (then.gated) {                                  // a tile's 16 rows of B are eight gates and their ups (n is whole tiles)
        for (int e = threadIdx.x; e < kTilesM * kTilesN * 128; e += kWaves * kWave) {
            const int t = e / (kTilesN * 128), j = e / 128 % kTilesN, row = t * 16 + e % 128 / 8, at = e % 128 / 8 * kStreamTile + e % 8;
            if (row >= m || n0 + j * kStreamTile >= n) continue;
            float gate = sums[0][t][j][at], up = sums[0][t][j][at + 8];
#pragma unroll
            for (int v = 1; v < kWaves; ++v) gate += sums[v][t][j][at], up += sums[v][t][j][at + 8];
            c[static_cast<long>(row) * (n / 2) + n0 / 2 + j * 8 + e % 8] = glu_value(gate, up, then.act, then.limit);
        }
        return;
    }
    for (int e = threadIdx.x; e < kTilesM * kTilesN * 256; e += kWaves * kWave) {
        const int t = e / (kTilesN * 256), j = e / 256 % kTilesN, row = t * 16 + e % 256 / 16, col = n0 + j * kStreamTile + e % 16;
        if (row >= m || col >= n || (kCols < kStreamTile && e % 16 >= kCols)) continue;
        float total = sums[0][t][j][e % 256];
#pragma unroll
        for (int v = 1; v < kWaves; ++v) total += sums[v][t][j][e % 256];     // (segments past K's end are zeros)
        c[static_cast<long>(row) * n + col] = kAdds ? before + total : total;
    }
}

template <int kTilesM, int kTilesN, int kWaves, int kDepth, int kEach, bool kVec>
__global__ void __launch_bounds__(kWaves * kWave, kEach)
gemm_f32_stream_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k, int segment,
                       Epilogue then) {
    __shared__ float sums[kWaves][kTilesM][kTilesN][kStreamTile * kStreamTile];
    static_assert(kDepth % 2 == 0, "a register's runs are all even ones or all odd ones");
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int n0 = blockIdx.x * kTilesN * kStreamTile;
    const int r = lane % 16, h = (lane / 16) * 4;
    const float *brow[kTilesN], *arow[kTilesM];
#pragma unroll
    for (int j = 0; j < kTilesN; ++j) brow[j] = b + static_cast<long>(n0 + j * 16 + r < n ? n0 + j * 16 + r : n - 1) * k;
#pragma unroll
    for (int t = 0; t < kTilesM; ++t) arow[t] = a + static_cast<long>(t * 16 + r < m ? t * 16 + r : m - 1) * k;
    f32x4 sum[kTilesM][kTilesN] = {};
    float largest_b[kTilesN] = {}, largest_a[kTilesM] = {};
    f32x4 w[kDepth][kTilesN][kStreamLoads], x[kDepth][kTilesM][kStreamLoads];
    const int first = wave * segment, end = first + segment < k ? first + segment : k;
    const auto fetch = [&](int at, int into) {         // a run that lies whole before the segment's end
#pragma unroll
        for (int j = 0; j < kTilesN; ++j)
#pragma unroll
            for (int i = 0; i < kStreamLoads; ++i) w[into][j][i] = load_whole<kVec>(brow[j] + at + i * 16 + h);
#pragma unroll
        for (int t = 0; t < kTilesM; ++t)
#pragma unroll
            for (int i = 0; i < kStreamLoads; ++i) x[into][t][i] = load_whole<kVec>(arow[t] + at + i * 16 + h);
    };
    const auto multiply = [&](int from, bool odd) {     // (see kTerms)
#pragma unroll
        for (int i = 0; i < kStreamLoads; i += 2) {
            Operand wp[kTilesN];
#pragma unroll
            for (int j = 0; j < kTilesN; ++j) {
                wp[j] = operand_of(w[from][j][i], w[from][j][i + 1]);
                largest_b[j] = largest_of(largest_of(largest_b[j], w[from][j][i]), w[from][j][i + 1]);
            }
#pragma unroll
            for (int t = 0; t < kTilesM; ++t) {
                largest_a[t] = largest_of(largest_of(largest_a[t], x[from][t][i]), x[from][t][i + 1]);
                const Operand xp = odd ? operand_of(-x[from][t][i], -x[from][t][i + 1]) : operand_of(x[from][t][i], x[from][t][i + 1]);
                f32x4 acc[kTilesN] = {};
#pragma unroll
                for (int e = 0; e < kTerms; ++e)
#pragma unroll
                    for (int j = 0; j < kTilesN; ++j) acc[j] = add_term(e, xp, wp[j], acc[j]);
#pragma unroll
                for (int j = 0; j < kTilesN; ++j) {
                    acc[j] += highest_term(xp, wp[j]);
                    sum[t][j] = odd ? sum[t][j] - acc[j] : sum[t][j] + acc[j];
                }
                __builtin_amdgcn_sched_barrier(0);     // (interleaved with the next ones' products the waves' number would not fit the registers)
            }
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
                multiply(d, d % 2);
                fetch(at + (kDepth + d) * kStreamRun, d);
            }
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            multiply(d, d % 2);
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
        if (d < left) multiply(d, d % 2);
    at += left * kStreamRun;
    if (at < end) {                                    // the rest of the last segment, filled up with zeros
#pragma unroll
        for (int j = 0; j < kTilesN; ++j)
#pragma unroll
            for (int i = 0; i < kStreamLoads; ++i) w[0][j][i] = load_four<kVec>(brow[j], at + i * 16 + h, end);
#pragma unroll
        for (int t = 0; t < kTilesM; ++t)
#pragma unroll
            for (int i = 0; i < kStreamLoads; ++i) x[0][t][i] = load_four<kVec>(arow[t], at + i * 16 + h, end);
        left % 2 ? multiply(0, true) : multiply(0, false);
    }
    float largest = 0.f, least_sum = INFINITY, no_number = 0.f;
#pragma unroll
    for (int t = 0; t < kTilesM; ++t) {
        largest = fmaxf(largest, largest_a[t]);
#pragma unroll
        for (int j = 0; j < kTilesN; ++j) {
            largest = fmaxf(largest, largest_b[j]);
#pragma unroll
            for (int i = 0; i < 4; ++i) least_sum = fminf(least_sum, fabsf(sum[t][j][i])), no_number = fmaf(sum[t][j][i], 0.f, no_number);
        }
    }
    if (!__all(beyond_doubt(largest, least_sum, no_number))) {
        float least_b[kTilesN];
#pragma unroll
        for (int j = 0; j < kTilesN; ++j) least_b[j] = least_of(max_lanes<16>(max_lanes<32>(largest_b[j])));
#pragma unroll
        for (int t = 0; t < kTilesM; ++t) {
            const float least_a = least_of(max_lanes<16>(max_lanes<32>(largest_a[t])));
            float least[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) least[i] = __shfl(least_a, h + i, kWave);
#pragma unroll
            for (int j = 0; j < kTilesN; ++j) {
                const auto doubt = [&](int i) { return in_doubt(sum[t][j][i], least[i], least_b[j]); };
                if (!__any(doubt(0) || doubt(1) || doubt(2) || doubt(3))) continue;
                const f32x4 plain = plain_square<kVec>(arow[t], brow[j], first, end, lane / 16);
#pragma unroll
                for (int i = 0; i < 4; ++i) sum[t][j][i] = doubt(i) ? plain[i] : sum[t][j][i];
            }
        }
    }
#pragma unroll
    for (int t = 0; t < kTilesM; ++t)
#pragma unroll
        for (int j = 0; j < kTilesN; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) sums[wave][t][j][(h + i) * kStreamTile + r] = sum[t][j][i];
    __syncthreads();
    add_segments<kTilesM, kTilesN, kWaves>(sums, c, m, n, n0, then);
}

// Up to eight rows: half of the instruction's 16 rows of A are taken for the run after, so that A is asked for and taken apart
// once for two runs (a third of the taking apart, which is most of a wave's instructions).  Of the first run's products rows 0 .. 7 count, of
// the second's (whose B has its sign turned, see kTerms) rows 8 .. 15, which the other half of the wave holds.
constexpr int kFewRows = 8;
constexpr long kManyTiles = 1024;

// kFold, what else the launch does: 0 nothing; kFoldAdds: the product is added to what lies in C; from 2 on: A's rows are normed first, every
// element (a * gain) / sqrt(mean(a^2) + eps), rows of up to 256 kFold elements.  A workgroup needs the sums of squares of all rows: a wave
// asks for a whole row ahead of its first weights and adds up while those are on their way, in the order of the norm's own kernel
// (add_rmsnorm_vec_kernel), so that results are the same bits as of two launches.
constexpr int kFoldAdds = 1;

// kNarrow: the workgroup owns eight rows of B, not 16, and the instruction's 16 columns too are taken for two runs: twice as many
// workgroups where 16 rows each would leave units idle.  Of the products the first run's lie in rows and columns 0 .. 7, the second's in 8 .. 15.
template <int kWaves, int kAhead, bool kVec, int kFold, bool kNarrow = false>
__device__ inline void few_rows(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k, int segment,
                                const Epilogue& then, const float* __restrict__ gain, float eps) {
    constexpr int kPair = 2 * kStreamRun;
    constexpr bool kNorm = kFold >= 2;
    static_assert(kVec || kFold == 0, "what is folded goes with aligned rows");
    __shared__ float sums[kWaves][1][1][kStreamTile * kStreamTile];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    constexpr int kCols = kNarrow ? kStreamTile / 2 : kStreamTile, kRuns = kNarrow ? 1 : 2;
    const int n0 = blockIdx.x * kCols;
    const int r = lane % 16, h = (lane / 16) * 4, later = r < kFewRows ? 0 : kStreamRun;
    const float* brow = b + static_cast<long>(n0 + r % kCols < n ? n0 + r % kCols : n - 1) * k + (kNarrow ? later : 0);
    const float* arow = a + static_cast<long>(r % kFewRows < m ? r % kFewRows : m - 1) * k;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};                  // (of the lower half of the wave)
    float largest_a = 0.f, largest_b = 0.f;
    f32x4 w[kAhead][kRuns][kStreamLoads], x[kAhead][kStreamLoads];
    [[maybe_unused]] f32x4 gains[kNorm ? kAhead : 1][kStreamLoads];
    [[maybe_unused]] float inv = 1.0f, before = 0.f;
    // the whole rows of this wave: the norm's threads 64 v + lane take four elements of every 4 kThreads
    constexpr int kThreads = kFold == 2 ? 64 : 256, kTurns = kThreads / 64, kChunks = kNorm ? kFold / kTurns : 1, kRowsEach = kFewRows / kWaves;
    [[maybe_unused]] __shared__ float inverses[kFewRows];
    [[maybe_unused]] f32x4 whole[kNorm ? kRowsEach : 1][kNorm ? kFold : 1];
    const auto place = [&](int q) { return 4 * ((q / kChunks) * 64 + lane + (q % kChunks) * kThreads); };
    if constexpr (kNorm) {
#pragma unroll
        for (int e = 0; e < kRowsEach; ++e) {
            const int row = wave + e * kWaves;
            const float* from = a + static_cast<long>(row < m ? row : m - 1) * k;
#pragma unroll
            for (int q = 0; q < kFold; ++q) whole[e][q] = *reinterpret_cast<const f32x4*>(from + (place(q) < k ? place(q) : 0));
        }
    }
    if constexpr (kFold == kFoldAdds) {                // the one element that this thread writes (see add_segments)
        const int row = threadIdx.x / 16, col = n0 + threadIdx.x % kCols;
        before = c[static_cast<long>(row < m ? row : m - 1) * n + (col < n ? col : n - 1)];
    }
    const auto settle = [&] {                          // the rows' factors, once the first weights are on their way
        if constexpr (kNorm) {
#pragma unroll
            for (int e = 0; e < kRowsEach; ++e) {
                float total = 0.f;
#pragma unroll
                for (int v = 0; v < kTurns; ++v) {
                    float ss = 0.f;
#pragma unroll
                    for (int i = 0; i < kChunks; ++i) {
                        const int q = v * kChunks + i;
                        float with = ss;
#pragma unroll
                        for (int j = 0; j < 4; ++j) with = fmaf(whole[e][q][j], whole[e][q][j], with);
                        ss = place(q) < k ? with : ss;
                    }
                    total += wave_sum(ss);
                }
                if (lane == 0) inverses[wave + e * kWaves] = 1.0f / sqrtf(total / static_cast<float>(k) + eps);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");        // (__syncthreads waits for the weights)
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            inv = inverses[r % kFewRows < m ? r % kFewRows : m - 1];
        }
    };
    const int first = wave * segment, end = first + segment < k ? first + segment : k;
    const auto fetch_a = [&](int at, int into) {       // a pair of runs that lies whole before the segment's end
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i) {
            x[into][i] = load_whole<kVec>(arow + at + later + i * 16 + h);
            if constexpr (kNorm) gains[into][i] = load_whole<kVec>(gain + at + later + i * 16 + h);
        }
    };
    const auto fetch_b = [&](int at, int into, int run) {
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i) w[into][run][i] = load_whole<kVec>(brow + at + run * kStreamRun + i * 16 + h);
    };
    const auto fetch_pair = [&](int at, int into) {
#pragma unroll
        for (int run = 0; run < kRuns; ++run) fetch_b(at, into, run);
    };
    [[maybe_unused]] const unsigned sign = kNarrow && later ? 0x80000000u : 0u;
    [[maybe_unused]] const auto turned = [&](const f32x4& v) {
        f32x4 t;
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = __uint_as_float(__float_as_uint(v[e]) ^ sign);
        return t;
    };
    // the pair in the registers `of`; another one from `next` on is asked for as they become free
    const auto multiply = [&](int of, bool more, int next) {
        f32x4 x0 = x[of][0], x1 = x[of][1];
        if constexpr (kNorm) x0 = normed(x0, gains[of][0], inv), x1 = normed(x1, gains[of][1], inv);
        const Operand xp = operand_of(x0, x1);
        largest_a = largest_of(largest_of(largest_a, x0), x1);
        if (more) fetch_a(next, of);
        f32x4 acc[kRuns];
#pragma unroll
        for (int run = 0; run < kRuns; ++run) {
            const f32x4 w0 = w[of][run][0], w1 = w[of][run][1];
            const Operand wp = kNarrow ? operand_of(turned(w0), turned(w1)) : run ? operand_of(-w0, -w1) : operand_of(w0, w1);
            largest_b = largest_of(largest_of(largest_b, w0), w1);
            if (more) fetch_b(next, of, run);
            acc[run] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < kTerms; ++e) acc[run] = add_term(e, xp, wp, acc[run]);
            acc[run] += highest_term(xp, wp);
            if (run == 0) sum += acc[0];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {                  // (the upper half's results to the lower one, of columns 8 .. 15 to 0 .. 7)
            const unsigned first = __float_as_uint(acc[0][e]), second = __float_as_uint(acc[kRuns - 1][e]);
            const unsigned upper = __builtin_amdgcn_permlane32_swap(second, first, false, false)[1];
            sum[e] -= __uint_as_float(kNarrow ? of_lane<0x128>(upper) : upper);
        }
    };
    int left = end > first ? (end - first) / kPair : 0, at = first;
    if (left >= kAhead) {
#pragma unroll
        for (int d = 0; d < kAhead; ++d) fetch_a(at + d * kPair, d), fetch_pair(at + d * kPair, d);
        settle();
        for (; left >= 2 * kAhead; left -= kAhead, at += kAhead * kPair)
#pragma unroll
            for (int d = 0; d < kAhead; ++d) multiply(d, true, at + (kAhead + d) * kPair);
#pragma unroll
        for (int d = 0; d < kAhead; ++d) multiply(d, kAhead + d < left, at + (kAhead + d) * kPair);
        left -= kAhead, at += kAhead * kPair;
    } else {
#pragma unroll
        for (int d = 0; d < kAhead - 1; ++d)
            if (d < left) fetch_a(at + d * kPair, d), fetch_pair(at + d * kPair, d);
        settle();
    }
#pragma unroll
    for (int d = 0; d < kAhead - 1; ++d)
        if (d < left) multiply(d, false, 0);
    at += left * kPair;
    if (at < end) {                                    // the rest of the last segment, filled up with zeros
#pragma unroll
        for (int i = 0; i < kStreamLoads; ++i) {
            x[0][i] = load_four<kVec>(arow, at + later + i * 16 + h, end);
            if constexpr (kNorm) gains[0][i] = load_four<kVec>(gain, at + later + i * 16 + h, end);
#pragma unroll
            for (int run = 0; run < kRuns; ++run) w[0][run][i] = load_four<kVec>(brow, at + run * kStreamRun + i * 16 + h, end - (kNarrow ? later : 0));
        }
        multiply(0, false, 0);
    }
    const bool mine = lane < kWave / 2 && r < kCols;
    float least_sum = INFINITY, no_number = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) least_sum = fminf(least_sum, fabsf(sum[i])), no_number = fmaf(sum[i], 0.f, no_number);
    if (!__all(beyond_doubt(fmaxf(largest_a, largest_b), mine ? least_sum : 1.0f, mine ? no_number : 0.f))) {
        float largest_of_b = max_lanes<16>(max_lanes<32>(largest_b));
        if constexpr (kNarrow) largest_of_b = max_lanes<8>(largest_of_b);
        const float least_b = least_of(largest_of_b);
        const float least_a = least_of(max_lanes<8>(max_lanes<16>(max_lanes<32>(largest_a))));
        float least[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) least[i] = __shfl(least_a, h + i, kWave);
        const auto doubt = [&](int i) { return mine && in_doubt(sum[i], least[i], least_b); };
        if (__any(doubt(0) || doubt(1) || doubt(2) || doubt(3))) {
            const f32x4 plain = plain_square<kVec, kNorm>(arow, brow - (kNarrow ? later : 0), first, end, lane / 16, gain, inv);
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[i] = doubt(i) ? plain[i] : sum[i];
        }
    }
    if (mine) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[wave][0][0][(h + i) * kStreamTile + r] = sum[i];
    }
    __syncthreads();
    add_segments<1, 1, kWaves, kFold == kFoldAdds, kCols>(sums, c, m, n, n0, then, before);
}

template <int kWaves, int kAhead, int kEach, bool kVec>
__global__ void __launch_bounds__(kWaves * kWave, kEach)
gemm_f32_few_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k, int segment,
                    Epilogue then) {
    few_rows<kWaves, kAhead, kVec, 0>(a, b, c, m, n, k, segment, then, nullptr, 0.f);
}

// The same with a neighbour folded in.
template <int kWaves, int kAhead, int kEach, int kFold>
__global__ void __launch_bounds__(kWaves * kWave, kEach)
gemm_f32_folded_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k, int segment,
                       Epilogue then, const float* __restrict__ gain, float eps) {
    few_rows<kWaves, kAhead, true, kFold>(a, b, c, m, n, k, segment, then, gain, eps);
}

// Eight rows of B a workgroup.
template <int kWaves, int kAhead, int kEach, int kFold>
__global__ void __launch_bounds__(kWaves * kWave, kEach)
gemm_f32_narrow_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k, int segment,
                       Epilogue then, const float* __restrict__ gain, float eps) {
    few_rows<kWaves, kAhead, true, kFold, true>(a, b, c, m, n, k, segment, then, gain, eps);
}

// ---- many rows -----------------------------------------------------------------------------------------------------
// A tile of 64 x kCols outputs, four waves side by side.  A wave's columns are its own: it takes their elements of B from memory as
// the kernel above does, and takes them apart in registers.  All four waves need A's rows: slabs of 32 elements of K in shared memory,
// in parts (64 bytes a row and part); a lane's eight numbers of an instruction, elements 4 g .. + 3 and 16 + 4 g .. + 3 of the slab for
// g = lane / 16, lie together, and the four lanes' places of a row change with every second row, so that eight neighbouring lanes touch
// every bank once.  While a slab is multiplied, A's next one is taken apart between the instructions, and the one after that and B's
// next one are on their way into registers.
//
// What bounds it is that the matrix instructions (eight for what one product of floats needs), the taking apart (half of the vector
// instructions) and the trips through shared memory follow one another within a wave; three workgroups a unit make up for it to half of
// the instructions' rate.  Columns of their own keep B out of shared memory (777 rows against 12288 x 2048, with six products of parts:
// 243 us, with both operands in shared memory 303).  With eight 777 rows take 300 to 320 us there and 170 against 2048 x 6144 (with six on the
// same card 266 and 148; on the float instructions 440 and 219).
//
// kCut: blockIdx.z takes `each` segments and leaves a plane of c for every one of them; else one workgroup walks them all.
constexpr int kSlab = kChain;
constexpr int kTileRows = 64;

template <int kCols, bool kVec, bool kCut>
__global__ void __launch_bounds__(256, 3)
gemm_f32_tile_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k,
                     int segment, int each, Epilogue then) {
    constexpr int kFragA = kTileRows / 16, kFragB = kCols / 64;                      // 16 x 16 squares of a wave
    constexpr int kLoadsA = kTileRows / 32;                                          // 16-byte loads a thread and slab
    constexpr int kSquares = kFragA * kFragB;
    constexpr int kHeld = kFragB > 1 ? 2 : kSquares;                                 // squares whose totals are in registers,
    constexpr int kAway = kCut ? 0 : kSquares - kHeld;                               // and in shared memory (with all of them a wave would spill)
    __shared__ u32x2 slabs[2][3][kTileRows][8];
    __shared__ f32x4 away[kAway ? kAway : 1][kAway ? 256 : 1];
    __shared__ __align__(16) float least_a[2][kTileRows];       // (see least_of) of this segment's rows of A and, by turns, the next one's
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;       // (a scalar register)
    const int m0 = blockIdx.y * kTileRows, n0 = blockIdx.x * kCols + wave * (kCols / 4);
    const int r = lane % 16, g = lane / 16;
    const long part = static_cast<long>(segment) * each;
    const int k_first = static_cast<int>(blockIdx.z * part), k_end = k - k_first > part ? static_cast<int>(k_first + part) : k;
    const int four = threadIdx.x % 8, from_row = threadIdx.x / 8;                // this thread's four elements of every 32nd row of A
    // A number whose uses are computed where they stand: held in registers throughout, they would leave the sums none.
    const auto here = [](int v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    const auto arow = [&](int i) {
        const int row = m0 + i * 32 + here(from_row);
        return a + static_cast<long>(row < m ? row : m - 1) * k;
    };
    const auto brow = [&](int j) {
        const int row = n0 + j * 16 + here(r);
        return b + static_cast<long>(row < n ? row : n - 1) * k;
    };
    f32x4 sum[kFragA][kFragB] = {};
    [[maybe_unused]] f32x4 total[kHeld] = {};
    f32x4 ra[kLoadsA], rb[kFragB][2];
    float largest_a[kLoadsA] = {}, largest_b[kFragB] = {};
    // (past the last element of a row: its last ones, and not used)
    const auto load_at = [&](const float* row, int at) {
        if (kVec) return *reinterpret_cast<const f32x4*>(row + (at < k ? at : k - 4));
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = row[at + e < k ? at + e : k - 1];
        return v;
    };
    const auto fetch_a = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) ra[i] = load_at(arow(i), k0 + four * 4);
    };
    const auto fetch_b = [&](int k0) {
#pragma unroll
        for (int j = 0; j < kFragB; ++j)
#pragma unroll
            for (int half = 0; half < 2; ++half) rb[j][half] = load_at(brow(j), k0 + half * 16 + g * 4);
    };
    const auto cut_off = [&](int k0) {                  // what lies past K in a slab of A counts as zero
        if (k0 + kSlab <= k) return;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (k0 + four * 4 + e >= k) {
#pragma unroll
                for (int i = 0; i < kLoadsA; ++i) ra[i][e] = 0.f;
            }
    };
    const auto cut_off_b = [&](int k0) {                // and of B
        if (k0 + kSlab <= k) return;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (k0 + half * 16 + g * 4 + e >= k) {
#pragma unroll
                    for (int j = 0; j < kFragB; ++j) rb[j][half][e] = 0.f;
                }
    };
    const auto place = [](int row, int of) { return of ^ (row / 2 % 4); };       // of lane group `of`'s sixteen bytes
    const int kept_at = place(from_row, four % 4) * 2 + four / 4;                // (32 rows further it is the same)
    const auto keep = [&](int into, int i, float sign) {
        largest_a[i] = largest_of(largest_a[i], ra[i]);
        const FourParts v = parts_of(ra[i] * sign);
#pragma unroll
        for (int p = 0; p < 3; ++p) slabs[into][p][from_row + i * 32][kept_at] = v.part[p];
    };
    const int col = n0 + r;                                                      // of the first square; rows 4 g .. + 3
    const auto row_of = [&](int i, int e) { return m0 + i * 16 + 4 * g + e; };
    const auto store = [&](const f32x4 (&of)[kFragA][kFragB], float* to) {
        const int left_m = m - m0, left_n = n - n0, row0 = here(4 * g), column = here(r);
#pragma unroll
        for (int i = 0; i < kFragA; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < kFragB; ++j)
                    if (row0 + i * 16 + e < left_m && column + j * 16 < left_n)
                        to[static_cast<long>(m0 + row0 + i * 16 + e) * n + n0 + column + j * 16] = of[i][j][e];
    };
    // the slab of A that was kept ends its segment: the segment's rows are known (eight threads have one)
    int kept_turn = 0, kept_end = k_first + segment;
    const auto kept = [&](int k0) {
        if (k0 + kSlab < kept_end && k0 + kSlab < k_end) return;
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) {
            const float least = least_of(join_span<8>(largest_a[i], [](float x, float y) { return fmaxf(x, y); }));
            const int thread = here(threadIdx.x);
            if (thread % 8 == 0) least_a[kept_turn][thread / 8 + i * 32] = least;
            largest_a[i] = 0.f;
        }
        kept_turn ^= 1, kept_end += segment;
    };
    if constexpr (kAway > 0) {
#pragma unroll
        for (int i = 0; i < kAway; ++i) away[i][threadIdx.x] = f32x4{0.f, 0.f, 0.f, 0.f};       // (a thread's own)
    }
    fetch_a(k_first);
    fetch_b(k_first);
    cut_off(k_first);
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i) keep(0, i, 1.0f);
    kept(k_first);
    fetch_a(k_first + kSlab);
    float sign = 1.0f;                                 // of the slab that is multiplied (see kTerms)
    int at = 0, turn = 0, segment_first = k_first;     // segments are an even number of slabs
    float* plane = c + static_cast<long>(blockIdx.z) * each * m * n;
    const int mine = place(r, g) * 2;
    for (int k0 = k_first; k0 < k_end; k0 += kSlab, at ^= 1) {
        cut_off_b(k0);
        Operand bp[kFragB];
#pragma unroll
        for (int j = 0; j < kFragB; ++j) {
            bp[j] = operand_of(rb[j][0], rb[j][1]);
            largest_b[j] = largest_of(largest_of(largest_b[j], rb[j][0]), rb[j][1]);
        }
        fetch_b(k0 + kSlab);
        __syncthreads();               // this slab is there, and nobody reads the one before it any more
        cut_off(k0 + kSlab);
#pragma unroll
        for (int i = 0; i < kFragA; ++i) {
            Operand ap;
#pragma unroll
            for (int p = 0; p < 3; ++p)
                ap.part[p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&slabs[at][p][i * 16 + r][mine]));
#pragma unroll
            for (int l = i * kLoadsA / kFragA; l < (i + 1) * kLoadsA / kFragA; ++l) keep(at ^ 1, l, -sign);
            f32x4 acc[kFragB] = {};
#pragma unroll
            for (int e = 0; e < kTerms; ++e)
#pragma unroll
                for (int j = 0; j < kFragB; ++j) acc[j] = add_term(e, ap, bp[j], acc[j]);
#pragma unroll
            for (int j = 0; j < kFragB; ++j) acc[j] += highest_term(ap, bp[j]);
#pragma unroll
            for (int j = 0; j < kFragB; ++j) sum[i][j] = acc[j] * sign + sum[i][j];        // (one instruction, and exact)
            if constexpr (kFragB > 1) __builtin_amdgcn_sched_barrier(0);             // (the next one's operands ahead of these sums would not fit the registers)
        }
        if (k0 + kSlab < k_end) kept(k0 + kSlab);
        fetch_a(k0 + 2 * kSlab);
        sign = -sign;
        if (k0 + kSlab >= k_end || k0 + kSlab == segment_first + segment) {
            // (that segment's rows of A were written before the slab's barrier, and are written again behind the next one at the earliest)
            const int row0 = here(4 * g), column0 = here(r);
            float least_b[kFragB], least = 0.f, odd = 0.f;       // least: below 0 if a sum is in doubt; odd: NaN if one is no finite number
#pragma unroll
            for (int j = 0; j < kFragB; ++j) {
                least_b[j] = least_of(max_lanes<16>(max_lanes<32>(largest_b[j])));
                largest_b[j] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < kFragA; ++i) {
                const f32x4 of = *reinterpret_cast<const f32x4*>(&least_a[turn][i * 16 + row0]);
#pragma unroll
                for (int j = 0; j < kFragB; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        least = fminf(least, fmaf(-of[e], least_b[j], fabsf(sum[i][j][e])));
                        odd = fmaf(sum[i][j][e], 0.f, odd);
                    }
            }
            if (__any(least < 0.f || odd != 0.f)) {
                const int end = segment_first + segment < k_end ? segment_first + segment : k_end;
#pragma unroll 1
                for (int x = 0; x < kFragA * kFragB; ++x) {
                    f32x4 v = sum[0][0];
                    float of_b = least_b[0];
#pragma unroll
                    for (int y = 1; y < kFragA * kFragB; ++y) v = x == y ? sum[y / kFragB][y % kFragB] : v;
#pragma unroll
                    for (int j = 1; j < kFragB; ++j) of_b = x % kFragB == j ? least_b[j] : of_b;
                    const f32x4 of = *reinterpret_cast<const f32x4*>(&least_a[turn][x / kFragB * 16 + row0]);
                    const auto doubt = [&](int e) { return in_doubt(v[e], of[e], of_b); };
                    if (!__any(doubt(0) || doubt(1) || doubt(2) || doubt(3))) continue;
                    const int row = m0 + x / kFragB * 16 + column0, column = n0 + x % kFragB * 16 + column0;
                    const f32x4 plain = plain_square<kVec>(a + static_cast<long>(row < m ? row : m - 1) * k,
                                                           b + static_cast<long>(column < n ? column : n - 1) * k, segment_first, end, row0 / 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = doubt(e) ? plain[e] : v[e];
#pragma unroll
                    for (int y = 0; y < kFragA * kFragB; ++y) sum[y / kFragB][y % kFragB] = x == y ? v : sum[y / kFragB][y % kFragB];
                }
            }
            turn ^= 1;
            segment_first += segment;
            if constexpr (kCut) {
                store(sum, plane);
                plane += static_cast<long>(m) * n;
            }
#pragma unroll
            for (int i = 0; i < kFragA; ++i)
#pragma unroll
                for (int j = 0; j < kFragB; ++j) {
                    if constexpr (!kCut) {
                        constexpr int kRoom = kAway ? kAway : 1;
                        const int x = i * kFragB + j;
                        if (x < kHeld) total[x % kHeld] += sum[i][j];
                        else away[(x - kHeld) % kRoom][threadIdx.x] += sum[i][j];
                    }
                    sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
    }
    if constexpr (!kCut) {
        const auto total_of = [&](int x) { return x < kHeld ? total[x % kHeld] : away[(x - kHeld) % (kAway ? kAway : 1)][threadIdx.x]; };
#pragma unroll
        for (int i = 0; i < kFragA; ++i)
#pragma unroll
            for (int j = 0; j < kFragB; ++j) sum[i][j] = total_of(i * kFragB + j);
        if (!then.gated) return store(sum, c);
        // lanes 0 .. 7 of a row of 16 hold gates, the lane eight further its up
#pragma unroll
        for (int i = 0; i < kFragA; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < kFragB; ++j) {
                    const float up = lane_pair<8>(sum[i][j][e]).b;
                    if (r < 8 && row_of(i, e) < m && col + j * 16 < n)
                        c[static_cast<long>(row_of(i, e)) * (n / 2) + (n0 + j * 16) / 2 + r] =
                            glu_value(sum[i][j][e], up, then.act, then.limit);
                }
    }
}

// ---- a short K -----------------------------------------------------------------------------------------------------
// K below 256 is one chain of float products, k ascending, in tiles of kRows x 64 outputs whatever the rows: 32 x 32 x 2 instructions
// on the floats themselves, a quarter of the tile a wave.  Slabs of K in shared memory, rows 4 floats further apart than they are long (16-byte reads of 8
// neighbouring rows then touch every bank once).  Of every 8 elements the even ones lie first and then the odd ones: half-wave h
// reads its four at once, and the four instructions take elements 0 and 1, 2 and 3, .. of them.
constexpr int kChainCols = 64;
constexpr int chain_slab_of(int rows) { return rows == 128 ? 32 : 64; }

template <int kRows, bool kVec>
__global__ void __launch_bounds__(256, 2)
gemm_f32_chain_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, int m, int n, int k) {
    constexpr int kLong = chain_slab_of(kRows);
    constexpr int kFrag = kRows / 64;                  // 32 x 32 squares of a wave, one under the other
    constexpr int kLoadsA = kRows * kLong / 4 / 256, kLoadsB = kChainCols * kLong / 4 / 256;    // 16-byte loads a thread and slab
    __shared__ float as[2][kRows][kLong + 4];
    __shared__ float bs[2][kChainCols][kLong + 4];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int m0 = blockIdx.y * kRows, n0 = blockIdx.x * kChainCols;
    const int wm = (wave / 2) * (kRows / 2), wn = (wave % 2) * (kChainCols / 2);
    f32x16 acc[kFrag] = {};
    f32x4 ra[kLoadsA], rb[kLoadsB];
    const auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) {
            const int idx = threadIdx.x + i * 256, row = m0 + idx / (kLong / 4), at = k0 + (idx % (kLong / 4)) * 4;
            ra[i] = load_four<kVec>(a + static_cast<long>(row < m ? row : m - 1) * k, at, k);
        }
#pragma unroll
        for (int i = 0; i < kLoadsB; ++i) {
            const int idx = threadIdx.x + i * 256, row = n0 + idx / (kLong / 4), at = k0 + (idx % (kLong / 4)) * 4;
            rb[i] = load_four<kVec>(b + static_cast<long>(row < n ? row : n - 1) * k, at, k);
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
            put(as[into][idx / (kLong / 4)], (idx % (kLong / 4)) * 4, ra[i]);
        }
#pragma unroll
        for (int i = 0; i < kLoadsB; ++i) {
            const int idx = threadIdx.x + i * 256;
            put(bs[into][idx / (kLong / 4)], (idx % (kLong / 4)) * 4, rb[i]);
        }
    };
    fetch(0);
    keep(0);
    int at = 0;
    for (int k0 = 0; k0 < k; k0 += kLong, at ^= 1) {
        const bool more = k0 + kLong < k;
        if (more) fetch(k0 + kLong);
        __syncthreads();
        const int row = lane % 32, h = (lane / 32) * 4;
#pragma unroll
        for (int s = 0; s < kLong; s += 8) {
            f32x4 av[kFrag];
            const f32x4 bv = *reinterpret_cast<const f32x4*>(&bs[at][wn + row][s + h]);
#pragma unroll
            for (int i = 0; i < kFrag; ++i) av[i] = *reinterpret_cast<const f32x4*>(&as[at][wm + i * 32 + row][s + h]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < kFrag; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i][e], bv[e], acc[i], 0, 0, 0);
        }
        if (more) keep(at ^ 1);        // read last two slabs ago, and every wave has passed a barrier since
    }
    const int col = n0 + wn + lane % 32;
#pragma unroll
    for (int i = 0; i < kFrag; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = m0 + wm + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
            if (row < m && col < n) c[static_cast<long>(row) * n + col] = acc[i][e];
        }
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

// The same of sums that are gates and ups: four results a thread, of rows of n / 2.  kVec: planes and c are aligned to 16 bytes.
template <bool kVec>
__global__ void __launch_bounds__(256)
gemm_f32_sum_gated_kernel(const float* __restrict__ planes, float* __restrict__ c, long count, int n, int parts, Epilogue then) {
    const long at = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (at >= count / 2) return;
    const long row = at / (n / 2);
    const int col = static_cast<int>(at - row * (n / 2));                   // n / 2 is a multiple of 8
    const float* from = planes + row * n + col / 8 * 16 + col % 8;
    const auto four = [](const float* p) { return kVec ? *reinterpret_cast<const f32x4*>(p) : f32x4{p[0], p[1], p[2], p[3]}; };
    f32x4 gate = four(from), up = four(from + 8), result;
    for (int p = 1; p < parts; ++p) gate += four(from + p * count), up += four(from + p * count + 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) result[e] = glu_value(gate[e], up[e], then.act, then.limit);
    if (kVec) {
        *reinterpret_cast<f32x4*>(c + at) = result;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) c[at + e] = result[e];
    }
}

// Up to here a product is a stream of weights.  Measured (us, streamed : tiled) against 2048 x 2048 weights 10.7 : 12.4 at 17 rows,
// 13.1 : 13.1 at 32, 3072 x 512 5.5 : 10.1 at 32, 6144 x 1024 13.2 : 15.7, 12288 x 2048 36.0 : 35.2, 32768 x 2048 74.7 : 77.9 and 89.9 : 83.2 at 17
// and 32; beyond, the stream's reads of A, then four times the weights', cost more.  A long K leaves the tiles' workgroups enough to do
// from the second tile of rows on: with six products of parts 1024 x 3072 15.1 : 14.6 and 18.9 : 15.0 at 17 and 32 rows, 2048 x 6144 27.9 : 26.4
// and 35.5 : 26.8.
constexpr int kStreamRows = 32;
constexpr int kStreamLongK = 3072;
constexpr int kStreamK = 256;          // a shorter K is no work to share out over four waves: one chain, in tiles whatever the rows

// The segments of K: by K alone.  Eight from 512 elements on (a wave each of a streaming workgroup), four from 256, multiples
// of 64 elements (whole slabs of a tile).
struct F32Segments {
    int length, count;
};
F32Segments f32_segments(int k) {
    const int wanted = k < kStreamK ? 1 : k < 2 * kStreamK ? 4 : 8;
    const int length = ceil_div(ceil_div(k, wanted), 64) * 64;
    return {length, ceil_div(k, length)};
}

struct F32Plan {
    int rows = 0, cols = 0, parts = 1, each = 1;       // of a tile, no rows: the streaming kernel; parts workgroups of `each` segments along K
};

// A short K: the tile that takes least time.  A compute unit's float instructions run at one rate however many tiles it holds, so the
// product takes as long as the fullest of the 256 units has work for; one tile a unit leaves a wave a SIMD and its waits in the open.
F32Plan f32_chain_plan(int m, int n) {
    F32Plan best;
    double least = 0.0;
    for (int rows : {128, 64}) {
        const long held = (static_cast<long>(ceil_div(m, rows)) * ceil_div(n, kChainCols) + 255) / 256;
        const double time = held * rows / (rows == 128 ? (held >= 2 ? 0.87 : 0.4) : (held >= 2 ? 0.82 : 0.65));
        if (best.rows == 0 || time < least * 0.999) {
            least = time;
            best.rows = rows, best.cols = kChainCols;
        }
    }
    return best;
}

// The tile's width and the cut of K that take least time.  Up to four workgroups of a unit work side by side: a slab takes them the longer
// of a workgroup's own way through it and of what they ask of the unit together.  A cut K costs a plane written and read for every
// segment (mostly in the caches) and a second launch.  Constants (microseconds; bytes a microsecond) fitted to both tiles and every cut
// timed at 17 to 2,048 rows against the matrices of layers of 512, 1,024, 2,048 and 4,096 channels: the choice is 0.5 % off the best on
// average and 8 % at worst (512 rows against 4096 x 12288 408 us, 378 with every segment a workgroup).
F32Plan f32_plan(int m, int n, int k) {
    F32Plan best;
    if (k < kStreamK) return f32_chain_plan(m, n);
    const F32Segments segments = f32_segments(k);
    best.each = segments.count;
    if (m <= (k < kStreamLongK ? kStreamRows : kStreamTile)) return best;
    constexpr long kUnits = 256, kBeside = 4;
    constexpr double kPlaneRate = 8.5e6, kLaunch = 4.4;
    double least = 0.0;
    for (int cols : {128, 64}) {
        const double own = cols == 128 ? 1.06 : 0.66, shared = cols == 128 ? 0.76 : 0.47;
        const long tiles = static_cast<long>(ceil_div(m, kTileRows)) * ceil_div(n, cols);
        for (int wanted = 1; wanted <= segments.count; wanted *= 2) {
            const int each = ceil_div(segments.count, wanted), parts = ceil_div(segments.count, each);
            const long held = (tiles * parts + kUnits - 1) / kUnits;           // of the fullest unit
            const double slabs = static_cast<double>(segments.length) * each / kSlab;
            const auto side_by_side = [&](long workgroups) { return workgroups * shared > own ? workgroups * shared : own; };
            const double product = slabs * ((held / kBeside) * side_by_side(kBeside) + (held % kBeside ? side_by_side(held % kBeside) : 0.0));
            const double planes = parts == 1 ? 0.0 : kLaunch + 8.0 * segments.count * m * n / kPlaneRate;
            if (best.rows == 0 || product + planes < least * 0.999) {
                least = product + planes;
                best.rows = kTileRows, best.cols = cols, best.parts = parts, best.each = each;
            }
        }
    }
    return best;
}

// Up to eight rows one pair of runs on its way a wave; of a large matrix two, for two waves a SIMD (us, one and two pairs: one row
// against 12288 x 2048 19.6 and 18.8, five against 24576 x 4096 72.5 and 69.7, 32768 x 2048 49.5 and 47.7; but 4096 x 2048 7.6 and 7.8,
// 32768 x 1024 26.8 and 27.4).  Beyond, two runs; where there are many tiles and more than eight rows or short segments, two tiles
// of B share what A's parts cost (one and two tiles: 16 rows against 32768 x 2048 64.6 and 53.5, 24576 x 4096 96.3 and 76.8, one row against
// 32768 x 512 16.6 and 14.6; but 16 against 12288 x 2048 26.6 and 27.0, 4096 x 2048 9.8 and 13.6).
bool large_matrix(const F32Segments& segments, int n, int k) { return segments.length >= 256 && static_cast<long>(n) * k >= 16l << 20; }
bool many_tiles(const F32Segments& segments, int m, int n) { return n >= kManyTiles * kStreamTile && (m > kFewRows || segments.length <= 64); }

// Products of at most eight rows with a neighbour folded in: which ones, and their launch.
constexpr int kFoldedK = 4096;         // longest row that a product norms
// Up to here a workgroup owns eight rows of B, not 16, so that every unit has at most one: a unit without one asks for nothing (us, 16 and
// eight, 1 row and 8: 512 x 512 3.7 and 3.3, 4.0 and 3.6; 1024 x 3072 8.7 and 6.8, 10.7 and 8.4; 2048 x 2048 6.8 and 5.7, 8.1 and 6.7; 2048 x 6144
// 16.1 and 12.4, 19.7 and 14.7; but 3072 x 2048 6.9 and 8.5, 8.1 and 10.2, 4096 x 4096 14.6 and 15.1, 15.1 and 18.3).
constexpr int kNarrowColumns = 2048;
bool folds(int m, int n, int k, bool norm) {
    return m > 0 && m <= kFewRows && n > 0 && k >= kStreamK && k % 4 == 0 && (!norm || k <= kFoldedK) && !many_tiles(f32_segments(k), m, n);
}
bool narrow(int n) { return n <= kNarrowColumns; }
int launch_narrow(int fold, const float* a, const float* b, float* c, int m, int n, int k, const float* gain, float eps, hipStream_t stream) {
    const F32Segments segments = f32_segments(k);
#define LEONE_NARROW(W, D, E, F) \
    gemm_f32_narrow_kernel<W, D, E, F><<<ceil_div(n, kStreamTile / 2), W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length, Epilogue{}, gain, eps)
    if (segments.count <= 4) fold == 0 ? LEONE_NARROW(4, 1, 4, 0) : fold == kFoldAdds ? LEONE_NARROW(4, 1, 4, kFoldAdds) : LEONE_NARROW(4, 1, 4, 2);
    else if (fold < 2) fold == 0 ? LEONE_NARROW(8, 2, 4, 0) : LEONE_NARROW(8, 2, 4, kFoldAdds);
    else if (fold == 2) LEONE_NARROW(8, 1, 4, 2);
    else fold == 8 ? LEONE_NARROW(8, 2, 4, 8) : LEONE_NARROW(8, 1, 4, 16);
#undef LEONE_NARROW
    LEONE_LAUNCH_CHECK("gemm_f32_narrow");
    return 0;
}
int launch_folded(const float* a, const float* b, float* c, int m, int n, int k, const Epilogue& then, const float* gain, float eps, hipStream_t stream) {
    const F32Segments segments = f32_segments(k);
    const bool large = large_matrix(segments, n, k);
    const int fold = !gain ? kFoldAdds : k <= 512 ? 2 : k <= 2048 ? 8 : 16;
    if (!then.gated && narrow(n)) return launch_narrow(fold, a, b, c, m, n, k, gain, eps, stream);
#define LEONE_FOLDED(W, D, E, F)                                                                                                       \
    gemm_f32_folded_kernel<W, D, E, F><<<ceil_div(n, kStreamTile), W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length, then, gain, eps)
    if (segments.count <= 4) fold == kFoldAdds ? LEONE_FOLDED(4, 1, 4, kFoldAdds) : LEONE_FOLDED(4, 1, 4, 2);
    else if (large) fold == kFoldAdds ? LEONE_FOLDED(8, 2, 2, kFoldAdds) : fold == 8 ? LEONE_FOLDED(8, 2, 2, 8) : LEONE_FOLDED(8, 2, 2, 16);
    else if (fold <= 2) fold == kFoldAdds ? LEONE_FOLDED(8, 1, 4, kFoldAdds) : LEONE_FOLDED(8, 1, 4, 2);
    else fold == 8 ? LEONE_FOLDED(8, 1, 4, 8) : LEONE_FOLDED(8, 1, 4, 16);
#undef LEONE_FOLDED
    LEONE_LAUNCH_CHECK("gemm_f32_folded");
    return 0;
}

int launch_f32(const F32Plan& p, const float* a, const float* b, float* c, float* planes, int m, int n, int k, const Epilogue& then,
               hipStream_t stream) {
    const F32Segments segments = f32_segments(k);
    LEONE_REQUIRE(p.parts == 1 || planes, "gemm_f32: %d planes are needed for %d x %d x %d", segments.count, m, n, k);
    const auto aligned = [](const void* at) { return reinterpret_cast<uintptr_t>(at) % 16 == 0; };
    const bool vec = k % 4 == 0 && aligned(a) && aligned(b);
    if (p.rows == 0) {
#define LEONE_FEW(W, D, E)                                                                                                             \
    (vec ? gemm_f32_few_kernel<W, D, E, true><<<ceil_div(n, kStreamTile), W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length, then) \
         : gemm_f32_few_kernel<W, D, E, false><<<ceil_div(n, kStreamTile), W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length, then))
#define LEONE_STREAM(T, N, W, D, E)                                                                                                    \
    (vec ? gemm_f32_stream_kernel<T, N, W, D, E, true><<<ceil_div(n, N * kStreamTile), W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length, then)  \
         : gemm_f32_stream_kernel<T, N, W, D, E, false><<<ceil_div(n, N * kStreamTile), W * kWave, 0, stream>>>(a, b, c, m, n, k, segments.length, then))
        const bool large = large_matrix(segments, n, k), many = many_tiles(segments, m, n);
        if (vec && m <= kFewRows && !then.gated && narrow(n)) return launch_narrow(0, a, b, c, m, n, k, nullptr, 0.f, stream);
        if (segments.count <= 4) {
            if (m <= kFewRows) LEONE_FEW(4, 1, 4);
            else if (m <= kStreamTile) LEONE_STREAM(1, 1, 4, 2, 4);
            else LEONE_STREAM(2, 1, 4, 2, 2);
        } else if (m > kStreamTile) {
            LEONE_STREAM(2, 1, 8, 2, 2);
        } else if (many) {
            LEONE_STREAM(1, 2, 8, 2, 4);
        } else if (m > kFewRows) {
            LEONE_STREAM(1, 1, 8, 2, 4);
        } else if (large) {
            LEONE_FEW(8, 2, 2);
        } else {
            LEONE_FEW(8, 1, 4);
        }
#undef LEONE_FEW
#undef LEONE_STREAM
        LEONE_LAUNCH_CHECK("gemm_f32");
        return 0;
    }
    const int grid_y = ceil_div(m, p.rows);
    LEONE_REQUIRE(grid_y <= 65535, "gemm_f32: %d rows exceed the launch limit", m);
    const dim3 grid(ceil_div(n, p.cols), grid_y, p.parts);
#define LEONE_CHAIN(R)                                                                                                                 \
    (vec ? gemm_f32_chain_kernel<R, true><<<grid, 256, 0, stream>>>(a, b, c, m, n, k)                                                  \
         : gemm_f32_chain_kernel<R, false><<<grid, 256, 0, stream>>>(a, b, c, m, n, k))
#define LEONE_TILE_CUT(C, V)                                                                                                           \
    (p.parts > 1 ? gemm_f32_tile_kernel<C, V, true><<<grid, 256, 0, stream>>>(a, b, planes, m, n, k, segments.length, p.each, then)    \
                 : gemm_f32_tile_kernel<C, V, false><<<grid, 256, 0, stream>>>(a, b, c, m, n, k, segments.length, p.each, then))
#define LEONE_TILE(C) (vec ? LEONE_TILE_CUT(C, true) : LEONE_TILE_CUT(C, false))
    if (k < kStreamK) p.rows == 128 ? LEONE_CHAIN(128) : LEONE_CHAIN(64);
    else p.cols == 128 ? LEONE_TILE(128) : LEONE_TILE(64);
#undef LEONE_CHAIN
#undef LEONE_TILE
#undef LEONE_TILE_CUT
    LEONE_LAUNCH_CHECK("gemm_f32");
    if (p.parts > 1) {
        const long count = static_cast<long>(m) * n;
        if (then.gated) {
            const int blocks = ceil_div(count / 2, 1024);
            if (aligned(planes) && aligned(c)) gemm_f32_sum_gated_kernel<true><<<blocks, 256, 0, stream>>>(planes, c, count, n, segments.count, then);
            else gemm_f32_sum_gated_kernel<false><<<blocks, 256, 0, stream>>>(planes, c, count, n, segments.count, then);
            LEONE_LAUNCH_CHECK("gemm_f32 sum");
            return 0;
        }
        const int blocks = ceil_div(count, 1024);
        if (count % 4 == 0 && aligned(planes) && aligned(c))
            gemm_f32_sum_kernel<true><<<blocks, 256, 0, stream>>>(planes, c, count, segments.count);
        else
            gemm_f32_sum_kernel<false><<<blocks, 256, 0, stream>>>(planes, c, count, segments.count);
        LEONE_LAUNCH_CHECK("gemm_f32 sum");
    }
    return 0;
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
    return launch_f32(f32_plan(m, n, k), a, b, c, planes, m, n, k, Epilogue{}, stream);
}

// Whether leone_gemm_f32_glu takes a matrix: whole tiles of eight gates and their ups, and a K that is no chain.
extern "C" int leone_gemm_f32_glu_fits(int n, int k) { return n > 0 && n % 16 == 0 && k >= kStreamK; }

// C[M, N / 2] = act(gate) * up of the same product, B's rows being eight gates, their eight ups, and so on (act, limit: as leone_glu).
// The bits are those of the product and leone_glu behind it; one launch and the product's way to memory and back are saved (us, two launches
// and one: one row against 12288 x 2048 22.7 and 20.5, five against 3072 x 512 7.0 and 4.2, 200 20.6 and 18.6, 777 against 12288 x 2048
// 271 and 264).
extern "C" int leone_gemm_f32_glu(const float* a, const float* b, float* c, float* planes, int m, int n, int k, int act, float limit,
                                  hipStream_t stream) {
    LEONE_REQUIRE(a && b && c, "gemm_f32_glu: null pointer");
    LEONE_REQUIRE(m > 0 && leone_gemm_f32_glu_fits(n, k), "gemm_f32_glu: sizes %d x %d x %d", m, n, k);
    LEONE_REQUIRE(act == kGateSilu || act == kGateGeluTanh || (act == kGateClampedSwish && limit > 0.f),
                  "gemm_f32_glu: unknown activation %d (limit %g)", act, limit);
    return launch_f32(f32_plan(m, n, k), a, b, c, planes, m, n, k, Epilogue{1, act, limit}, stream);
}

// What else a product of few rows can do in its launch, to the bit what the launches give one by one: 1: C += A . B^T; 2: A's rows are
// normed first, (a * gain) / sqrt(mean(a^2) + eps) with float gains, and the product may be gated as leone_gemm_f32_glu's is (n whole tiles).
extern "C" int leone_gemm_f32_folds(int m, int n, int k, int kind) { return (kind == 1 || kind == 2) && folds(m, n, k, kind == 2); }

// gain: null for kind 1; act -1: the product is not gated.
extern "C" int leone_gemm_f32_folded(const float* a, const float* b, float* c, int m, int n, int k, const float* gain, float eps, int act,
                                     float limit, hipStream_t stream) {
    LEONE_REQUIRE(a && b && c, "gemm_f32_folded: null pointer");
    LEONE_REQUIRE(folds(m, n, k, gain != nullptr), "gemm_f32_folded: sizes %d x %d x %d", m, n, k);
    for (const void* at : {static_cast<const void*>(a), static_cast<const void*>(b), static_cast<const void*>(gain)})
        LEONE_REQUIRE(reinterpret_cast<uintptr_t>(at) % 16 == 0, "gemm_f32_folded: operands must be aligned to 16 bytes");
    LEONE_REQUIRE(!gain || (eps > 0.f && eps == eps), "gemm_f32_folded: eps must be positive");
    LEONE_REQUIRE(act < 0 || (gain && n % 16 == 0), "gemm_f32_folded: a gated product goes with a norm and %d columns", n);
    LEONE_REQUIRE(act < 0 || act == kGateSilu || act == kGateGeluTanh || (act == kGateClampedSwish && limit > 0.f),
                  "gemm_f32_folded: unknown activation %d (limit %g)", act, limit);
    return launch_folded(a, b, c, m, n, k, act < 0 ? Epilogue{} : Epilogue{1, act, limit}, gain, eps, stream);
}
