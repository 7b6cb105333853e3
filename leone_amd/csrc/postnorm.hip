// A norm on what a sublayer hands back, folded into the residual sum.
//
// A block whose norms stand behind its sublayers (x <- x + norm(sublayer(x)), the sublayer reading x itself)
// needs, between two sublayers, the RMS norm of the sublayer's result, the sum into the float32 stream and
// the stream's rows in the type the next product reads.  One launch does all three; for the model's last rows
// it also does the norm that stands before the output head.  Sums of squares, the scaling and the residual
// sum are float whatever the type that is written.
#include "common.h"
#include "leone_hip.h"

#include <math.h>

namespace leone {

constexpr int kPostThreads = 256;

// One workgroup a row.  `row` (dynamic shared memory, `hidden` floats) holds the summed planes of the delta,
// then the new row of the stream.
//   x[r] += (delta[r] / sqrt(mean(delta[r]^2) + eps)) * gain          (delta == nullptr: nothing is added)
//   gain2 == nullptr:  y[r] = x[r] in TY                               (y == nullptr: nothing is written)
//   gain2 != nullptr:  y[i] = (x[r] / sqrt(mean(x[r]^2) + eps2)) * gain2, r = rows ? rows[i] : i
// With `rows` the stream itself is left as it was (only some rows are looked at).
// kVec: elements a thread takes at a time (4 where the row's length and the addresses allow whole 16-byte runs).
template <int kVec>
__device__ inline void load_run(const float* p, float out[kVec]) {
    if constexpr (kVec == 4) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
    } else {
        out[0] = p[0];
    }
}
template <int kVec>
__device__ inline void store_run(float* p, const float v[kVec]) {
    if constexpr (kVec == 4) *reinterpret_cast<float4*>(p) = float4{v[0], v[1], v[2], v[3]};
    else p[0] = v[0];
}
template <int kVec>
__device__ inline void store_run(bf16_t* p, const float v[kVec]) {
    if constexpr (kVec == 4) {
        uint2 packed;
        packed.x = bf16_bits_from_float(v[0]) | (static_cast<uint32_t>(bf16_bits_from_float(v[1])) << 16);
        packed.y = bf16_bits_from_float(v[2]) | (static_cast<uint32_t>(bf16_bits_from_float(v[3])) << 16);
        *reinterpret_cast<uint2*>(p) = packed;
    } else {
        p[0] = from_float<bf16_t>(v[0]);
    }
}

template <typename TY, int kVec>
__global__ void __launch_bounds__(kPostThreads)
add_normed_kernel(float* __restrict__ x, const float* __restrict__ delta, int planes, long plane, AnyVec gain, float eps,
                  TY* __restrict__ y, AnyVec gain2, float eps2, const int* __restrict__ rows, int hidden) {
    extern __shared__ float row[];
    __shared__ float scratch[kPostThreads / kWave];
    const int out_row = blockIdx.x;
    const long in_row = rows ? rows[out_row] : out_row;
    float* xr = x + in_row * hidden;
    float inv = 0.f;
    if (delta != nullptr) {
        const float* dr = delta + in_row * hidden;
        float ss = 0.f;
        for (int c = kVec * threadIdx.x; c < hidden; c += kVec * kPostThreads) {
            float d[kVec];
            load_run<kVec>(dr + c, d);
            for (int p = 1; p < planes; ++p) {                 // planes of a product cut along K, in order
                float more[kVec];
                load_run<kVec>(dr + p * plane + c, more);
#pragma unroll
                for (int i = 0; i < kVec; ++i) d[i] += more[i];
            }
#pragma unroll
            for (int i = 0; i < kVec; ++i) {
                row[c + i] = d[i];
                ss = fmaf(d[i], d[i], ss);
            }
        }
        inv = 1.0f / sqrtf(block_sum<kPostThreads>(ss, scratch) / static_cast<float>(hidden) + eps);
    }
    float ss2 = 0.f;
    for (int c = kVec * threadIdx.x; c < hidden; c += kVec * kPostThreads) {
        float v[kVec];
        load_run<kVec>(xr + c, v);
        if (delta != nullptr) {
#pragma unroll
            for (int i = 0; i < kVec; ++i) v[i] += (row[c + i] * inv) * load_any(gain, c + i);
            if (!rows) store_run<kVec>(xr + c, v);
        }
        if (gain2.ptr != nullptr) {
#pragma unroll
            for (int i = 0; i < kVec; ++i) {
                row[c + i] = v[i];
                ss2 = fmaf(v[i], v[i], ss2);
            }
        } else if (y != nullptr) {
            store_run<kVec>(y + static_cast<long>(out_row) * hidden + c, v);
        }
    }
    if (gain2.ptr == nullptr) return;
    const float inv2 = 1.0f / sqrtf(block_sum<kPostThreads>(ss2, scratch) / static_cast<float>(hidden) + eps2);
    for (int c = kVec * threadIdx.x; c < hidden; c += kVec * kPostThreads) {
        float v[kVec];
#pragma unroll
        for (int i = 0; i < kVec; ++i) v[i] = (row[c + i] * inv2) * load_any(gain2, c + i);
        store_run<kVec>(y + static_cast<long>(out_row) * hidden + c, v);
    }
}

// The same for rows of up to 1,024 kPer elements in whole 16-byte runs: the stream's row, what is added to it and the gains are all
// asked for before the first sum, and the row stays in registers.  Few rows are a chain of trips to memory and launches, many rows
// are bound by their bytes.  Sums in the other kernel's order: the same bits.
// The delta is the sum of `places` rows of `delta`, place_stride apart, in order.  kPairs: the places of a row are what its routed
// experts gave, chosen[row, place] and weight[row, place] the router's choice: an index from `experts` on stands for weight times
// the row of `from` instead, a negative one for nothing; `extra`, if there, is added behind them (as moe_combine does it, without a
// launch and without the sums' way through memory).  Places are read before it is known which of them count.
// us with cold caches, 2,048 wide (before): 8 rows of 6 places, with their sum a launch of its own, 7.8 (15.5); 2,114 rows 46.7
// (70.4); 8 rows without places 6.2 (7.4), 2,114 rows 14.3 (17.0).
template <typename TY, int kPer, int kPlaces, bool kPairs>
__global__ void __launch_bounds__(kPostThreads)
add_normed_held_kernel(float* __restrict__ x, const float* __restrict__ delta, int places, long place_stride, long row_stride,
                       const int* __restrict__ chosen, const float* __restrict__ weight, AnyVec from, const float* __restrict__ extra,
                       int experts, AnyVec gain, float eps, TY* __restrict__ y, AnyVec gain2, float eps2,
                       const int* __restrict__ rows, int hidden) {
    __shared__ float scratch[kPostThreads / kWave];
    const int out_row = blockIdx.x;
    const long in_row = rows ? rows[out_row] : out_row;
    float* xr = x + in_row * hidden;
    int at[kPer];
    bool in[kPer];
#pragma unroll
    for (int n = 0; n < kPer; ++n) {
        at[n] = 4 * (static_cast<int>(threadIdx.x) + n * kPostThreads);
        in[n] = at[n] < hidden;
        if (!in[n]) at[n] = 0;
    }
    // Four elements of a vector of either type, unpacked where they are used.
    struct Raw {
        uint4 bits;
        __device__ inline void load(const AnyVec& v, long i) {
            if (v.dtype == kF32) {
                bits = *reinterpret_cast<const uint4*>(static_cast<const float*>(v.ptr) + i);
            } else {
                const uint2 two = *reinterpret_cast<const uint2*>(static_cast<const bf16_t*>(v.ptr) + i);
                bits.x = two.x, bits.y = two.y;
            }
        }
        __device__ inline float get(const AnyVec& v, int i) const {
            if (v.dtype == kF32) return __uint_as_float(i == 0 ? bits.x : i == 1 ? bits.y : i == 2 ? bits.z : bits.w);
            const unsigned word = i / 2 ? bits.y : bits.x;
            return __uint_as_float(i % 2 ? word & 0xffff0000u : word << 16);
        }
    };
    float v[kPer][4], d[kPer][4] = {};
    Raw by[kPer], by2[kPer], came[kPer];
    float more[kPer][4] = {};
#pragma unroll
    for (int n = 0; n < kPer; ++n) load_run<4>(xr + at[n], v[n]);
    if (delta != nullptr) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) by[n].load(gain, at[n]);
    }
    if (gain2.ptr != nullptr) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) by2[n].load(gain2, at[n]);
    }
    if constexpr (kPairs) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) came[n].load(from, in_row * hidden + at[n]);
        if (extra != nullptr) {
#pragma unroll
            for (int n = 0; n < kPer; ++n) load_run<4>(extra + in_row * hidden + at[n], more[n]);
        }
    }
    if (delta != nullptr) {
        const float* dr = delta + in_row * row_stride;
        for (int j0 = 0; j0 < places; j0 += kPlaces) {
            float part[kPlaces][kPer][4];
            int which[kPlaces];
            float share[kPlaces];
#pragma unroll
            for (int u = 0; u < kPlaces; ++u) {
                if (j0 + u >= places) continue;
#pragma unroll
                for (int n = 0; n < kPer; ++n) load_run<4>(dr + (j0 + u) * place_stride + at[n], part[u][n]);
                if constexpr (kPairs) {
                    which[u] = chosen[in_row * places + j0 + u];
                    share[u] = weight[in_row * places + j0 + u];
                }
            }
#pragma unroll
            for (int u = 0; u < kPlaces; ++u) {
                if (j0 + u >= places) continue;
#pragma unroll
                for (int n = 0; n < kPer; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (!kPairs) d[n][i] += part[u][n][i];
                        else if (which[u] >= experts) d[n][i] += share[u] * came[n].get(from, i);
                        else if (which[u] >= 0) d[n][i] += part[u][n][i];
                    }
            }
        }
        float ss = 0.f;
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (kPairs && extra != nullptr) d[n][i] += more[n][i];
                if (in[n]) ss = fmaf(d[n][i], d[n][i], ss);
            }
        const float inv = 1.0f / sqrtf(block_sum<kPostThreads>(ss, scratch) / static_cast<float>(hidden) + eps);
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[n][i] += (d[n][i] * inv) * by[n].get(gain, i);
            if (!rows && in[n]) store_run<4>(xr + at[n], v[n]);
        }
    }
    if (y == nullptr) return;
    TY* yr = y + static_cast<long>(out_row) * hidden;
    if (gain2.ptr != nullptr) {
        float ss = 0.f;
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (in[n]) ss = fmaf(v[n][i], v[n][i], ss);
        const float inv = 1.0f / sqrtf(block_sum<kPostThreads>(ss, scratch) / static_cast<float>(hidden) + eps2);
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[n][i] = (v[n][i] * inv) * by2[n].get(gain2, i);
    }
#pragma unroll
    for (int n = 0; n < kPer; ++n)
        if (in[n]) store_run<4>(yr + at[n], v[n]);
}

constexpr int kHeldRow = 4096;                       // the longest row of add_normed_held_kernel

template <bool kPairs>
void launch_add_normed_held(float* x, const float* delta, int places, long place_stride, long row_stride, const int* chosen,
                            const float* weight, const AnyVec& from, const float* extra, int experts, const AnyVec& gain, float eps,
                            void* y, int y_dtype, const AnyVec& gain2, float eps2, const int* rows, int n_rows, int hidden,
                            hipStream_t stream) {
    // A thread has as many runs as the row asks for: of 512, with room for 2,048, half the threads asked for elements that nobody has
    // (2,048 rows of 512 5.4 us, so 4.5; of 256 4.8 and 4.0; the kernel without held rows 5.0 and 4.3).
    constexpr int kFew = kPairs ? 8 : 2, kMany = kPairs ? 4 : 2;         // places on their way at a time
#define LEONE_HELD_NORMED(TY, PER, PLACES)                                                                                      \
    add_normed_held_kernel<TY, PER, PLACES, kPairs><<<n_rows, kPostThreads, 0, stream>>>(                                        \
        x, delta, places, place_stride, row_stride, chosen, weight, from, extra, experts, gain, eps, static_cast<TY*>(y), gain2, eps2, \
        rows, hidden)
#define LEONE_HELD_NORMED_SIZE(TY) \
    (hidden <= 1024 ? LEONE_HELD_NORMED(TY, 1, kFew) : hidden <= 2048 ? LEONE_HELD_NORMED(TY, 2, kFew) : LEONE_HELD_NORMED(TY, 4, kMany))
    if (y_dtype == kBF16 && y) LEONE_HELD_NORMED_SIZE(bf16_t);
    else LEONE_HELD_NORMED_SIZE(float);
#undef LEONE_HELD_NORMED_SIZE
#undef LEONE_HELD_NORMED
}

static bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace leone

using namespace leone;

extern "C" int leone_add_normed_pairs(float* x, const float* pair_out, const int* chosen, const float* weight, int top, const void* from,
                                      int from_dtype, const float* extra, int experts, const void* gain, int gain_dtype, float eps,
                                      void* y, int y_dtype, const void* gain2, int gain2_dtype, float eps2, const int* rows, int n_rows,
                                      int hidden, hipStream_t stream) {
    LEONE_REQUIRE(x && pair_out && chosen && weight && from, "add_normed_pairs: null pointer");
    LEONE_REQUIRE(n_rows > 0 && top > 0 && experts >= 0 && leone_add_normed_pairs_fits(hidden),
                  "add_normed_pairs: rows %d, %d places, hidden %d (multiples of 4 up to %d)", n_rows, top, hidden, kHeldRow);
    LEONE_REQUIRE(gain && eps > 0.f && (gain_dtype == kF32 || gain_dtype == kBF16) && (from_dtype == kF32 || from_dtype == kBF16),
                  "add_normed_pairs: needs its norm's gain, a positive eps and known types");
    LEONE_REQUIRE(!gain2 || (y && eps2 > 0.f && eps2 == eps2 && (gain2_dtype == kF32 || gain2_dtype == kBF16)),
                  "add_normed_pairs: the second norm needs an output, a gain and a positive eps");
    LEONE_REQUIRE(!y || y_dtype == kF32 || y_dtype == kBF16, "add_normed_pairs: unknown output type %d", y_dtype);
    LEONE_REQUIRE(!rows || gain2, "add_normed_pairs: picked rows come with the second norm");
    LEONE_REQUIRE(aligned16(x) && aligned16(pair_out) && aligned16(from) && aligned16(extra) && aligned16(gain) && aligned16(gain2) && aligned16(y),
                  "add_normed_pairs: operands are aligned to 16 bytes");
    launch_add_normed_held<true>(x, pair_out, top, hidden, static_cast<long>(top) * hidden, chosen, weight, AnyVec{from, from_dtype}, extra,
                                 experts, AnyVec{gain, gain_dtype}, eps, y, y_dtype, AnyVec{gain2, gain2_dtype}, eps2, rows, n_rows, hidden,
                                 stream);
    LEONE_LAUNCH_CHECK("add_normed_pairs");
    return 0;
}
extern "C" int leone_add_normed_pairs_fits(int hidden) { return hidden > 0 && hidden % 4 == 0 && hidden <= kHeldRow; }

extern "C" int leone_add_normed(float* x, const float* delta, int delta_planes, long delta_plane, const void* gain,
                                int gain_dtype, float eps, void* y, int y_dtype, const void* gain2, int gain2_dtype,
                                float eps2, const int* rows, int n_rows, int hidden, hipStream_t stream) {
    LEONE_REQUIRE(x, "add_normed: null pointer");
    LEONE_REQUIRE(n_rows > 0 && hidden > 0 && hidden <= 12288, "add_normed: rows %d, hidden %d (at most 12288)", n_rows, hidden);
    LEONE_REQUIRE(!delta || (gain && eps > 0.f && eps == eps && (gain_dtype == kF32 || gain_dtype == kBF16)),
                  "add_normed: a delta needs its norm's gain and a positive eps");
    LEONE_REQUIRE(!delta || (delta_planes >= 1 && delta_planes <= 64 && (delta_planes == 1 || delta_plane >= static_cast<long>(n_rows) * hidden)),
                  "add_normed: %d planes of what is to be added", delta_planes);
    LEONE_REQUIRE(!gain2 || (y && eps2 > 0.f && eps2 == eps2 && (gain2_dtype == kF32 || gain2_dtype == kBF16)),
                  "add_normed: the second norm needs an output, a gain and a positive eps");
    LEONE_REQUIRE(!y || y_dtype == kF32 || y_dtype == kBF16, "add_normed: unknown output type %d", y_dtype);
    LEONE_REQUIRE(!rows || gain2, "add_normed: picked rows come with the second norm");
    LEONE_REQUIRE(delta || y, "add_normed: nothing to do");
    const AnyVec g1{gain, gain_dtype}, g2{gain2, gain2_dtype};
    const size_t shared = static_cast<size_t>(hidden) * sizeof(float);
    // whole 16-byte runs where the row's length, the planes' distance and every address allow them
    const bool runs = hidden % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                      (!delta || (reinterpret_cast<uintptr_t>(delta) % 16 == 0 && (delta_planes == 1 || delta_plane % 4 == 0))) &&
                      (!y || reinterpret_cast<uintptr_t>(y) % 16 == 0);
    if (runs && hidden <= kHeldRow && aligned16(gain) && aligned16(gain2)) {
        launch_add_normed_held<false>(x, delta, delta_planes, delta_plane, hidden, nullptr, nullptr, AnyVec{}, nullptr, 0, g1, eps, y, y_dtype,
                                      g2, eps2, rows, n_rows, hidden, stream);
        LEONE_LAUNCH_CHECK("add_normed");
        return 0;
    }
#define LEONE_ADD_NORMED(TY, V)                                                                                        \
    add_normed_kernel<TY, V><<<n_rows, kPostThreads, shared, stream>>>(x, delta, delta_planes, delta_plane, g1, eps,  \
                                                                       static_cast<TY*>(y), g2, eps2, rows, hidden)
    if (y_dtype == kBF16 && y) {
        if (runs) LEONE_ADD_NORMED(bf16_t, 4);
        else LEONE_ADD_NORMED(bf16_t, 1);
    } else {
        if (runs) LEONE_ADD_NORMED(float, 4);
        else LEONE_ADD_NORMED(float, 1);
    }
#undef LEONE_ADD_NORMED
    LEONE_LAUNCH_CHECK("add_normed");
    return 0;
}
