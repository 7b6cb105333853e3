// Row-wise kernels of layers that keep a short history of their own inputs:
//
//   add_layernorm     x += LayerNorm_a(delta) (if a delta comes), y = LayerNorm_b(x): the norm after one
//                     sublayer, the residual sum and the norm before the next in one pass over the row
//   entry_spans       first row and end of every entry of a step, and its state slot, from the row -> entry map
//   causal_conv       out[t] = (in[t] if asked) + sum_j w[c, j] * in[t - (taps - 1) + j], per channel, the
//                     rows before a portion taken from the request's state (its last taps - 1 inputs)
//   causal_conv_state leaves the last taps - 1 inputs of every entry behind as the new state
//   head_norm_gate    per head: (read-out / denominator) / rms * gain * act(gate)
//   rms_mix           scale * sum_b rms(branch_b) * gain_b over the model width
//   relu_squared      max(x, 0)^2
//
// Sums, means and variances are float whatever the storage type.
#include "common.h"
#include "leone_hip.h"

#include <math.h>

#include <type_traits>

namespace leone {

// Threads a row.  Few rows (decode steps): 1,024, so that a thread has few elements and a row is a handful of trips to
// memory, not one per element.  Many rows (prompt portions): 256, so that many rows are in flight on a compute unit.
constexpr int kNormThreadsFew = 1024;
constexpr int kNormThreadsMany = 256;
constexpr int kNormManyRows = 512;
constexpr int kMaxTaps = 16;

// Mean and inverse deviation of n values read through f(i); every thread gets both.
template <int kNormThreads, typename F>
__device__ inline void mean_rstd(F value, int n, float eps, float* scratch, float& mean, float& rstd) {
    float s = 0.f;
    for (int i = threadIdx.x; i < n; i += kNormThreads) s += value(i);
    mean = block_sum<kNormThreads>(s, scratch) / static_cast<float>(n);
    float q = 0.f;
    for (int i = threadIdx.x; i < n; i += kNormThreads) {
        const float d = value(i) - mean;
        q = fmaf(d, d, q);
    }
    const float var = block_sum<kNormThreads>(q, scratch) / static_cast<float>(n);
    rstd = 1.0f / sqrtf(var + eps);
}

__device__ inline void store_four(float* to, const float (&v)[4]) { *reinterpret_cast<float4*>(to) = float4{v[0], v[1], v[2], v[3]}; }
__device__ inline void store_four(bf16_t* to, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(to) = uint2{bf16_bits_from_float(v[0]) | static_cast<unsigned>(bf16_bits_from_float(v[1])) << 16,
                                          bf16_bits_from_float(v[2]) | static_cast<unsigned>(bf16_bits_from_float(v[3])) << 16};
}

// One workgroup a row; the row lies in shared memory between the passes.
template <typename TOut, int kNormThreads>
__global__ void __launch_bounds__(kNormThreads)
add_layernorm_kernel(float* __restrict__ x, const float* __restrict__ delta, AnyVec dw, AnyVec db, float deps,
                     AnyVec w, AnyVec b, float eps, TOut* __restrict__ y, const int* __restrict__ rows, int hidden,
                     AnyVec conv, int taps, float* __restrict__ conv_state, int write_state,
                     const int* __restrict__ positions, const int* __restrict__ row_entry, const int* __restrict__ entry_slots,
                     int stage_delta) {
    extern __shared__ float row_buf[];          // the row; behind it, if there is room, the delta's row
    __shared__ float scratch[kNormThreads / kWave];
    const long src = rows ? rows[blockIdx.x] : blockIdx.x;
    float* xr = x + src * hidden;
    if (delta) {
        const float* dr = delta + src * hidden;
        // both rows are fetched once, side by side; the passes after that read shared memory
        float* staged = stage_delta ? row_buf + hidden : nullptr;
        for (int i = threadIdx.x; i < hidden; i += kNormThreads) {
            row_buf[i] = xr[i];
            if (staged) staged[i] = dr[i];
        }
        __syncthreads();
        float mean = 0.f, rstd = 1.f;
        if (dw.ptr) {
            if (staged) mean_rstd<kNormThreads>([&](int i) { return staged[i]; }, hidden, deps, scratch, mean, rstd);
            else mean_rstd<kNormThreads>([&](int i) { return dr[i]; }, hidden, deps, scratch, mean, rstd);
        }
        for (int i = threadIdx.x; i < hidden; i += kNormThreads) {
            float d = staged ? staged[i] : dr[i];
            if (dw.ptr) d = (d - mean) * rstd * load_any(dw, i) + load_any(db, i);
            const float t = row_buf[i] + d;
            row_buf[i] = t;
            if (!rows) xr[i] = t;
        }
    } else {
        for (int i = threadIdx.x; i < hidden; i += kNormThreads) row_buf[i] = xr[i];
    }
    if (!y) return;
    __syncthreads();
    float mean, rstd;
    mean_rstd<kNormThreads>([&](int i) { return row_buf[i]; }, hidden, eps, scratch, mean, rstd);
    TOut* yr = y + static_cast<long>(blockIdx.x) * hidden;
    if (!conv.ptr) {
        for (int i = threadIdx.x; i < hidden; i += kNormThreads)
            yr[i] = from_float<TOut>((row_buf[i] - mean) * rstd * load_any(w, i) + load_any(b, i));
        return;
    }
    // A step of single rows, every row another request: the input convolution of the sublayer that reads this
    // norm is done here, h + conv(h) over the request's last inputs, and its state moved on by this row.
    const int pos = positions[blockIdx.x];
    float* keep = conv_state + static_cast<long>(entry_slots[row_entry[blockIdx.x]]) * (taps - 1) * hidden;
    for (int i = threadIdx.x; i < hidden; i += kNormThreads) {
        const float h = (row_buf[i] - mean) * rstd * load_any(w, i) + load_any(b, i);
        float acc = 0.f;
        for (int j = 0; j + 1 < taps; ++j) {                 // oldest input first
            const float old = pos - (taps - 1 - j) < 0 ? 0.f : keep[static_cast<long>(j) * hidden + i];
            acc = fmaf(load_any(conv, static_cast<long>(i) * taps + j), old, acc);
            if (write_state && j > 0) keep[static_cast<long>(j - 1) * hidden + i] = old;
        }
        acc = fmaf(load_any(conv, static_cast<long>(i) * taps + taps - 1), h, acc);
        if (write_state) keep[static_cast<long>(taps - 2) * hidden + i] = h;
        yr[i] = from_float<TOut>(h + acc);
    }
}

// Eight neighbouring elements of a row that is aligned to 16 bytes and holds whole runs, as they were loaded: a value is unpacked
// where it is used, so that no load is waited for by its own conversion.
constexpr int kRun = 8;
template <typename T>
struct Run;
template <>
struct Run<float> {
    float4 v[2];
    __device__ inline void load(const float* __restrict__ row, int at, int length) {
        const float4* from = reinterpret_cast<const float4*>(row + (at < length ? at : 0));
        v[0] = from[0];
        v[1] = from[1];
    }
    __device__ inline float get(int i) const {
        const float4 half = v[i / 4];
        return i % 4 == 0 ? half.x : i % 4 == 1 ? half.y : i % 4 == 2 ? half.z : half.w;
    }
};
template <>
struct Run<bf16_t> {
    uint4 v;
    __device__ inline void load(const bf16_t* __restrict__ row, int at, int length) {
        v = *reinterpret_cast<const uint4*>(row + (at < length ? at : 0));
    }
    __device__ inline float get(int i) const {
        const unsigned word = i / 2 == 0 ? v.x : i / 2 == 1 ? v.y : i / 2 == 2 ? v.z : v.w;
        return __uint_as_float(i % 2 ? word & 0xffff0000u : word << 16);
    }
};
template <typename T>
__device__ inline void store_run(T* __restrict__ row, int at, int length, const float (&v)[kRun]) {
    if (at >= length) return;
    if constexpr (sizeof(T) == 4) {
        reinterpret_cast<float4*>(row + at)[0] = float4{v[0], v[1], v[2], v[3]};
        reinterpret_cast<float4*>(row + at)[1] = float4{v[4], v[5], v[6], v[7]};
    } else {
        unsigned w[kRun / 2];
#pragma unroll
        for (int i = 0; i < kRun / 2; ++i)
            w[i] = bf16_bits_from_float(v[2 * i]) | static_cast<unsigned>(bf16_bits_from_float(v[2 * i + 1])) << 16;
        *reinterpret_cast<uint4*>(row + at) = uint4{w[0], w[1], w[2], w[3]};
    }
}

// The same for few rows of up to 1,024 kPer elements, a thread an element of every 1,024.  A step of few rows is a chain of trips to
// memory, about two microseconds each when the lines are cold: here the row, the delta, the gains, the biases, the filter's taps and
// the state's last inputs are all asked for before the first sum (each at an index held inside the row, so that no branch stands
// between the loads), and the row stays in registers.  One type for all of the norm's and the filter's vectors, so that a load is
// not followed by its conversion.  Sums run in the other kernel's order: the results are the same bits.
constexpr int kHeldTaps = 4;
template <typename TOut, typename TW, int kPer>
__global__ void __launch_bounds__(kNormThreadsFew)
add_layernorm_single_kernel(float* __restrict__ x, const float* __restrict__ delta, const TW* __restrict__ dw, const TW* __restrict__ db,
                          float deps, const TW* __restrict__ w, const TW* __restrict__ b, float eps, TOut* __restrict__ y,
                          const int* __restrict__ rows, int hidden, const TW* __restrict__ conv, int taps, float* conv_state,
                          int write_state, const int* __restrict__ positions, const int* __restrict__ row_entry,
                          const int* __restrict__ entry_slots) {
    __shared__ float scratch[kNormThreadsFew / kWave];
    const int tid = threadIdx.x;
    const long src = rows ? rows[blockIdx.x] : blockIdx.x;
    float* xr = x + src * hidden;
    int at[kPer];
    bool in[kPer];
#pragma unroll
    for (int n = 0; n < kPer; ++n) {
        in[n] = tid + n * kNormThreadsFew < hidden;
        at[n] = in[n] ? tid + n * kNormThreadsFew : hidden - 1;
    }
    float v[kPer], d[kPer], old[kHeldTaps - 1][kPer];
    TW gd[kPer], bd[kPer], g[kPer], o[kPer], f[kHeldTaps][kPer];
    int pos = 0, entry = 0;
    if (conv) {
        pos = positions[blockIdx.x];
        entry = row_entry[blockIdx.x];
    }
#pragma unroll
    for (int n = 0; n < kPer; ++n) v[n] = xr[at[n]];
    if (delta) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) d[n] = delta[src * hidden + at[n]];
    }
    if (dw) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
            gd[n] = dw[at[n]];
            bd[n] = db[at[n]];
        }
    }
    if (y) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
            g[n] = w[at[n]];
            o[n] = b[at[n]];
        }
    }
    float* keep = nullptr;
    if (conv) {
#pragma unroll
        for (int j = 0; j < kHeldTaps; ++j)
#pragma unroll
            for (int n = 0; n < kPer; ++n)
                if (j < taps) f[j][n] = conv[static_cast<long>(at[n]) * taps + j];
        keep = conv_state + static_cast<long>(entry_slots[entry]) * (taps - 1) * hidden;
#pragma unroll
        for (int j = 0; j + 1 < kHeldTaps; ++j)
#pragma unroll
            for (int n = 0; n < kPer; ++n)
                if (j + 1 < taps) old[j][n] = keep[static_cast<long>(j) * hidden + at[n]];
    }
    auto mean_of = [&](const float (&values)[kPer], float eps_, float& mean, float& rstd) {
        float sum = 0.f;
#pragma unroll
        for (int n = 0; n < kPer; ++n) sum += in[n] ? values[n] : 0.f;
        mean = block_sum<kNormThreadsFew>(sum, scratch) / static_cast<float>(hidden);
        float q = 0.f;
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
            const float off = in[n] ? values[n] - mean : 0.f;
            q = fmaf(off, off, q);
        }
        rstd = 1.0f / sqrtf(block_sum<kNormThreadsFew>(q, scratch) / static_cast<float>(hidden) + eps_);
    };
    float mean = 0.f, rstd = 1.f;
    if (delta) {
        if (dw) mean_of(d, deps, mean, rstd);
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
            const float more = dw ? (d[n] - mean) * rstd * to_float(gd[n]) + to_float(bd[n]) : d[n];
            v[n] += more;
            if (!rows && in[n]) xr[at[n]] = v[n];
        }
    }
    if (!y) return;
    mean_of(v, eps, mean, rstd);
    TOut* yr = y + static_cast<long>(blockIdx.x) * hidden;
#pragma unroll
    for (int n = 0; n < kPer; ++n) {
        if (!in[n]) continue;
        const float h = (v[n] - mean) * rstd * to_float(g[n]) + to_float(o[n]);
        if (!conv) {
            yr[at[n]] = from_float<TOut>(h);
            continue;
        }
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < kHeldTaps; ++j) {                // oldest input first, the row itself under the last tap
            if (j + 1 < taps) {
                const float was = pos - (taps - 1 - j) < 0 ? 0.f : old[j < kHeldTaps - 1 ? j : 0][n];
                acc = fmaf(to_float(f[j][n]), was, acc);
                if (write_state && j > 0) keep[static_cast<long>(j - 1) * hidden + at[n]] = was;
            } else if (j + 1 == taps) {
                acc = fmaf(to_float(f[j][n]), h, acc);
                if (write_state) keep[static_cast<long>(j - 1) * hidden + at[n]] = h;
            }
        }
        yr[at[n]] = from_float<TOut>(h + acc);
    }
}

// The same for rows of up to 1,024 kPer elements, a workgroup of two waves a row, in runs of 8 elements a thread.  A step of few rows
// is a chain of trips to memory, about two microseconds each when the lines are cold: here the row, the delta, the gains, the
// biases, the filter's taps and the state's last inputs are all asked for before the first sum, and the row stays in registers.
// Sums run in the other kernel's order with 1,024 threads, so that few rows get the bits they get there: elements 1,024 apart in
// turn, then those 32, 16, .. 1 apart meet, then every 64's sums in turn.  The runs of 64 elements lie on the eight lanes so that
// each of the lanes' three meetings is an operand's permutation.
// kTaps: of the folded filter; 0: none.
// Eight rows of 2,048 with two norms and a filter of 4 taps, in bfloat16: 6.1 us (7.8 with 1,024 threads of single elements).
constexpr int kHeldThreads = 128;
template <typename TOut, typename TW, int kPer, int kTaps>
__global__ void __launch_bounds__(kHeldThreads)
add_layernorm_held_kernel(float* __restrict__ x, const float* __restrict__ delta, const TW* __restrict__ dw, const TW* __restrict__ db,
                          float deps, const TW* __restrict__ w, const TW* __restrict__ b, float eps, TOut* __restrict__ y,
                          const int* __restrict__ rows, int hidden, const TW* __restrict__ conv, float* conv_state, int write_state,
                          const int* __restrict__ positions, const int* __restrict__ row_entry, const int* __restrict__ entry_slots) {
    constexpr int kLanes = 64 / kRun, kGroups = kHeldThreads / kLanes;        // lanes that share 64 elements, sums of 64 elements
    __shared__ float4 scratch[4][kGroups / 4];
    const long src = rows ? rows[blockIdx.x] : blockIdx.x;
    float* xr = x + src * hidden;
    const int sub = threadIdx.x % kLanes, place = threadIdx.x - sub + (sub & 1) * 4 + (sub & 2) + sub / 4;
    int at[kPer];
#pragma unroll
    for (int n = 0; n < kPer; ++n) at[n] = (n * kHeldThreads + place) * kRun;
    constexpr bool filtered = kTaps > 0;
    static_assert(kTaps == 0 || kTaps == 4, "a channel's taps are half a run");
    int pos = 0, entry = 0;
    if (filtered) {
        pos = positions[blockIdx.x];
        entry = row_entry[blockIdx.x];
    }
    Run<float> stream[kPer], more[kPer], old[kTaps == 0 ? 1 : kTaps - 1][kPer];
    Run<TW> delta_gain[kPer], delta_bias[kPer], gain[kPer], bias[kPer], filter[kTaps == 0 ? 1 : kTaps][kPer];
#pragma unroll
    for (int n = 0; n < kPer; ++n) stream[n].load(xr, at[n], hidden);
    if (delta) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) more[n].load(delta + src * hidden, at[n], hidden);
    }
    if (dw) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
            delta_gain[n].load(dw, at[n], hidden);
            delta_bias[n].load(db, at[n], hidden);
        }
    }
    if (y) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
            gain[n].load(w, at[n], hidden);
            bias[n].load(b, at[n], hidden);
        }
    }
    float* keep = nullptr;
    if (filtered) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
#pragma unroll
            for (int j = 0; j < kTaps; ++j)          // a channel's taps lie side by side: four runs of two channels each
                filter[j][n].load(conv, at[n] < hidden ? at[n] * kTaps + j * kRun : 0, hidden * kTaps);
        }
        keep = conv_state + static_cast<long>(entry_slots[entry]) * (kTaps - 1) * hidden;
#pragma unroll
        for (int j = 0; j + 1 < kTaps; ++j)
#pragma unroll
            for (int n = 0; n < kPer; ++n) old[j][n].load(keep + static_cast<long>(j) * hidden, at[n], hidden);
    }
    const auto inside = [&](int n) { return at[n] < hidden; };
    const auto row_sum = [&](float (&part)[kRun], float4* meet) {
#pragma unroll
        for (int i = 0; i < kRun; ++i) {
            constexpr int kSwap1 = 0xb1, kSwap2 = 0x4e, kMirror8 = 0x141;     // elements 32, 16 and 8 apart
            part[i] += of_lane<kSwap1>(part[i]);
            part[i] += of_lane<kSwap2>(part[i]);
            part[i] += of_lane<kMirror8>(part[i]);
        }
#pragma unroll
        for (int off = kRun / 2; off > 0; off /= 2)
#pragma unroll
            for (int i = 0; i < off; ++i) part[i] += part[i + off];
        if (sub == 0) reinterpret_cast<float*>(meet)[threadIdx.x / kLanes] = part[0];
        __syncthreads();
        float total = 0.f;
#pragma unroll
        for (int q = 0; q < kGroups / 4; ++q) {
            const float4 four = meet[q];
            total += four.x;
            total += four.y;
            total += four.z;
            total += four.w;
        }
        return total;
    };
    const auto moments = [&](const float (&v)[kPer][kRun], float of_eps, float4 (*meet)[kGroups / 4], float& mean, float& rstd) {
        float part[kRun] = {};
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < kRun; ++i) part[i] += inside(n) ? v[n][i] : 0.f;
        mean = row_sum(part, meet[0]) / static_cast<float>(hidden);
#pragma unroll
        for (int i = 0; i < kRun; ++i) part[i] = 0.f;
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < kRun; ++i) {
                const float off = inside(n) ? v[n][i] - mean : 0.f;
                part[i] = fmaf(off, off, part[i]);
            }
        rstd = 1.0f / sqrtf(row_sum(part, meet[1]) / static_cast<float>(hidden) + of_eps);
    };
    float v[kPer][kRun];
#pragma unroll
    for (int n = 0; n < kPer; ++n)
#pragma unroll
        for (int i = 0; i < kRun; ++i) v[n][i] = stream[n].get(i);
    if (delta) {
        float d[kPer][kRun], mean = 0.f, rstd = 1.f;
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < kRun; ++i) d[n][i] = more[n].get(i);
        if (dw) moments(d, deps, scratch, mean, rstd);
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
#pragma unroll
            for (int i = 0; i < kRun; ++i) v[n][i] += dw ? (d[n][i] - mean) * rstd * delta_gain[n].get(i) + delta_bias[n].get(i) : d[n][i];
            if (!rows) store_run<float>(xr, at[n], hidden, v[n]);
        }
    }
    if (!y) return;
    float mean, rstd;
    moments(v, eps, scratch + 2, mean, rstd);
    TOut* yr = y + static_cast<long>(blockIdx.x) * hidden;
#pragma unroll
    for (int n = 0; n < kPer; ++n) {
        float h[kRun];
#pragma unroll
        for (int i = 0; i < kRun; ++i) h[i] = (v[n][i] - mean) * rstd * gain[n].get(i) + bias[n].get(i);
        if (filtered) {
            // A step of single rows, every row another request: oldest input first, the row itself under the last tap
            float acc[kRun] = {};
#pragma unroll
            for (int j = 0; j < kTaps; ++j) {
                float in[kRun];
#pragma unroll
                for (int i = 0; i < kRun; ++i) {
                    if (j + 1 < kTaps) in[i] = pos - (kTaps - 1 - j) < 0 ? 0.f : old[j < kTaps - 1 ? j : 0][n].get(i);
                    else in[i] = h[i];
                    acc[i] = fmaf(filter[i / 2][n].get(i % 2 * kTaps + j), in[i], acc[i]);
                }
                if (write_state && j > 0) store_run<float>(keep + static_cast<long>(j - 1) * hidden, at[n], hidden, in);
            }
#pragma unroll
            for (int i = 0; i < kRun; ++i) h[i] += acc[i];
        }
        store_run<TOut>(yr, at[n], hidden, h);
    }
}

// The same for many rows of up to 256 kPer elements in whole 16-byte runs, a wave a row, without a barrier: what bounds them are
// their bytes, so every row is on its way at once.  Sums in the general kernel's order with 256 threads, for its bits: a lane adds
// elements 256 apart in turn, those 32, 16, .. 1 apart meet, and the sums of every 64 neighbours are added in turn.  A lane has four
// neighbours, so the first four meetings are between lanes of a row of 16, the last two in its own registers.
// With cold caches, two norms (us, before): 2,048 rows of 2,048 20.8 (33.6), of 1,024 12.3 (18.6), 512 rows of 2,048 12.6 (20.0).
constexpr int kRowThreads = 256;                 // four rows
template <typename TOut, typename TW, int kPer>
__global__ void __launch_bounds__(kRowThreads)
add_layernorm_wave_kernel(float* __restrict__ x, const float* __restrict__ delta, const TW* __restrict__ dw, const TW* __restrict__ db,
                          float deps, const TW* __restrict__ w, const TW* __restrict__ b, float eps, TOut* __restrict__ y,
                          const int* __restrict__ rows, int n_out, int hidden) {
    const int lane = threadIdx.x % kWave;
    const int out_row = blockIdx.x * (kRowThreads / kWave) + threadIdx.x / kWave;
    if (out_row >= n_out) return;
    const long src = rows ? rows[out_row] : out_row;
    float* xr = x + src * hidden;
    float v[kPer][4], d[kPer][4];
    const auto at = [&](int n) { return n * 256 + lane * 4; };
    const auto place = [&](int n) { return at(n) < hidden ? at(n) : 0; };
    const auto fetch = [](const float* p, float (&to)[4]) {
        const float4 four = *reinterpret_cast<const float4*>(p);
        to[0] = four.x, to[1] = four.y, to[2] = four.z, to[3] = four.w;
    };
#pragma unroll
    for (int n = 0; n < kPer; ++n) fetch(xr + place(n), v[n]);
    if (delta) {
#pragma unroll
        for (int n = 0; n < kPer; ++n) fetch(delta + src * hidden + place(n), d[n]);
    }
    const auto row_sum = [&](float (&part)[4]) {
        constexpr int kRotate8 = 0x128, kRotate4 = 0x124, kSwap1 = 0xb1, kSwap2 = 0x4e;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            part[i] += of_lane<kRotate8>(part[i]);
            part[i] += of_lane<kRotate4>(part[i]);
            part[i] += of_lane<kSwap2>(part[i]);
            part[i] += of_lane<kSwap1>(part[i]);
        }
        const float mine = (part[0] + part[2]) + (part[1] + part[3]);
        float total = 0.f;
#pragma unroll
        for (int sixteen = 0; sixteen < 4; ++sixteen)
            total += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine), sixteen * 16));
        return total;
    };
    const auto moments = [&](const float (&of)[kPer][4], float of_eps, float& mean, float& rstd) {
        float part[4] = {};
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) part[i] += at(n) < hidden ? of[n][i] : 0.f;
        mean = row_sum(part) / static_cast<float>(hidden);
#pragma unroll
        for (int i = 0; i < 4; ++i) part[i] = 0.f;
#pragma unroll
        for (int n = 0; n < kPer; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float off = at(n) < hidden ? of[n][i] - mean : 0.f;
                part[i] = fmaf(off, off, part[i]);
            }
        rstd = 1.0f / sqrtf(row_sum(part) / static_cast<float>(hidden) + of_eps);
    };
    if (delta) {
        float mean = 0.f, rstd = 1.f;
        if (dw) moments(d, deps, mean, rstd);
#pragma unroll
        for (int n = 0; n < kPer; ++n) {
            if (at(n) >= hidden) continue;
            Four<TW> gain, bias;
            if (dw) {
                gain.load(dw + at(n));
                bias.load(db + at(n));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) v[n][i] += dw ? (d[n][i] - mean) * rstd * gain.get(i) + bias.get(i) : d[n][i];
            if (!rows) *reinterpret_cast<float4*>(xr + at(n)) = float4{v[n][0], v[n][1], v[n][2], v[n][3]};
        }
    }
    if (!y) return;
    float mean, rstd;
    moments(v, eps, mean, rstd);
    TOut* yr = y + static_cast<long>(out_row) * hidden;
#pragma unroll
    for (int n = 0; n < kPer; ++n) {
        if (at(n) >= hidden) continue;
        Four<TW> gain, bias;
        gain.load(w + at(n));
        bias.load(b + at(n));
        float h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = (v[n][i] - mean) * rstd * gain.get(i) + bias.get(i);
        store_four(yr + at(n), h);
    }
}

__global__ void entry_spans_kernel(const int* __restrict__ row_entry, const int* __restrict__ positions,
                                   const int* __restrict__ entry_slots, int rows, int* __restrict__ spans) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int e = row_entry[r];
    if (r == 0 || row_entry[r - 1] != e) {
        spans[4 * e] = r;
        spans[4 * e + 2] = positions[r] == 0 ? -1 : entry_slots[e];     // a sequence's start: from zeros
        spans[4 * e + 3] = entry_slots[e];
    }
    if (r == rows - 1 || row_entry[r + 1] != e) spans[4 * e + 1] = r + 1;
}

enum Activation : int { kActNone = 0, kActSigmoid = 1, kActSilu = 2 };

__device__ inline float activate(float v, int act) {
    if (act == kActNone) return v;
    const float s = 1.0f / (1.0f + expf(-v));
    return act == kActSigmoid ? s : v * s;
}

constexpr int kConvRows = 8;     // consecutive rows a workgroup takes in a step of many rows: what it must know of a row is
                                 // fetched once for all of them; a step of few rows has a workgroup a row

template <typename TIn, typename TOut>
__global__ void causal_conv_kernel(const TIn* __restrict__ in, long in_stride, TOut* __restrict__ out, long out_stride,
                                   AnyVec w, AnyVec bias, const float* __restrict__ state, const int* __restrict__ positions,
                                   const int* __restrict__ row_entry, const int* __restrict__ entry_slots, int rows,
                                   int channels, int taps, int add_input, int act, float* __restrict__ own_state, int per_block) {
    __shared__ int s_inside[kConvRows], s_pos[kConvRows], s_slot[kConvRows];
    const int c = blockIdx.y * blockDim.x + threadIdx.x;
    const int r0 = blockIdx.x * per_block;
    if (threadIdx.x < per_block && r0 + threadIdx.x < rows) {
        const int r = r0 + threadIdx.x;
        const int e = row_entry[r];
        int inside = 0;      // rows of this request that stand before row r in this step, as far as the taps reach
        while (inside < taps - 1 && r - inside - 1 >= 0 && row_entry[r - inside - 1] == e) ++inside;
        s_inside[threadIdx.x] = inside;
        s_pos[threadIdx.x] = positions[r];
        s_slot[threadIdx.x] = entry_slots[e];
    }
    __syncthreads();
    if (c >= channels) return;
    for (int k = 0; k < per_block && r0 + k < rows; ++k) {
        const int r = r0 + k;
        const int pos = s_pos[k], inside = s_inside[k];
        const float* mine = state + (static_cast<long>(s_slot[k]) * (taps - 1)) * channels + c;
        float acc = 0.f;
        for (int back = taps - 1; back >= 0; --back) {          // oldest input first
            float h;
            if (pos - back < 0) h = 0.f;                          // before the sequence's start
            else if (back <= inside) h = to_float(in[static_cast<long>(r - back) * in_stride + c]);
            else h = mine[static_cast<long>(taps - 1 - (back - inside)) * channels];
            acc = fmaf(load_any(w, static_cast<long>(c) * taps + (taps - 1 - back)), h, acc);
        }
        const float now = to_float(in[static_cast<long>(r) * in_stride + c]);
        if (add_input) acc += now;
        if (bias.ptr) acc += load_any(bias, c);
        out[static_cast<long>(r) * out_stride + c] = from_float<TOut>(activate(acc, act));
        if (own_state) {      // a step of single rows, every row another request: this thread alone touches (slot, channel)
            float* keep = own_state + (static_cast<long>(s_slot[k]) * (taps - 1)) * channels + c;
            for (int j = 0; j + 2 < taps; ++j)
                keep[static_cast<long>(j) * channels] = pos - (taps - 2 - j) < 0 ? 0.f : keep[static_cast<long>(j + 1) * channels];
            keep[static_cast<long>(taps - 2) * channels] = now;
        }
    }
}

// The same for steps of many rows with four taps, four channels a thread: a row is read once, the inputs before it stay in registers
// as a window that moves on with every row of the same request, and the rows of a workgroup are all asked for before the first is
// worked on.  Sums in the other kernel's order: the same bits.  What bounds it are the bytes, read and written once.
// With cold caches, 2,048 rows of 4,096 channels, float to float: 17.2 us (54.4 with a load for every tap of a row); of 2,048, float
// to bfloat16: 12.3 (26.5); 600 rows of those 9.6 (19.7).
constexpr int kWindowTaps = 4;
constexpr int kWindowThreads = 256;
constexpr int kWindowChannels = 4;
template <typename TIn, typename TOut>
__global__ void __launch_bounds__(kWindowThreads)
causal_conv_window_kernel(const TIn* __restrict__ in, long in_stride, TOut* __restrict__ out, long out_stride, AnyVec w, AnyVec bias,
                          const float* __restrict__ state, const int* __restrict__ positions, const int* __restrict__ row_entry,
                          const int* __restrict__ entry_slots, int rows, int channels, int add_input, int act) {
    constexpr int kBefore = kWindowTaps - 1;
    const int c = (blockIdx.y * kWindowThreads + threadIdx.x) * kWindowChannels;
    const int r0 = blockIdx.x * kConvRows, count = min(kConvRows, rows - r0);
    if (c >= channels) return;
    Four<TIn> mine[kConvRows];
#pragma unroll
    for (int k = 0; k < kConvRows; ++k) mine[k].load(in + static_cast<long>(r0 + (k < count ? k : 0)) * in_stride + c);
    int entries[kConvRows], places[kConvRows];
#pragma unroll
    for (int k = 0; k < kConvRows; ++k) {
        entries[k] = row_entry[r0 + (k < count ? k : 0)];
        places[k] = positions[r0 + (k < count ? k : 0)];
    }
    static_assert(kWindowChannels * kWindowTaps == 16, "a thread's taps are two runs of eight");
    float taps[kWindowChannels * kWindowTaps], add[kWindowChannels], window[kBefore][kWindowChannels];
    load_any8(w, static_cast<long>(c) * kWindowTaps, taps);
    load_any8(w, static_cast<long>(c) * kWindowTaps + 8, taps + 8);
#pragma unroll
    for (int i = 0; i < kWindowChannels; ++i) add[i] = bias.ptr ? load_any(bias, c + i) : 0.f;
    int last_entry = -1, last_pos = 0;
#pragma unroll
    for (int k = 0; k < kConvRows; ++k) {
        if (k >= count) break;
        const int r = r0 + k, entry = entries[k], pos = places[k];
        if (k == 0 || entry != last_entry || pos != last_pos + 1) {
            // a request's first row here: its last inputs are rows of this step as far as there are some, and then its state
            int inside = 0;
            while (inside < kBefore && r - inside - 1 >= 0 && row_entry[r - inside - 1] == entry) ++inside;
            const float* kept = state + static_cast<long>(entry_slots[entry]) * kBefore * channels + c;
#pragma unroll
            for (int back = kBefore; back > 0; --back) {
                if (pos - back < 0) {                           // before the sequence's start
#pragma unroll
                    for (int i = 0; i < kWindowChannels; ++i) window[kBefore - back][i] = 0.f;
                } else if (back <= inside) {
                    Four<TIn> row;
                    row.load(in + static_cast<long>(r - back) * in_stride + c);
#pragma unroll
                    for (int i = 0; i < kWindowChannels; ++i) window[kBefore - back][i] = row.get(i);
                } else {
                    Four<float> was;
                    was.load(kept + static_cast<long>(kBefore - (back - inside)) * channels);
#pragma unroll
                    for (int i = 0; i < kWindowChannels; ++i) window[kBefore - back][i] = was.get(i);
                }
            }
        }
        last_entry = entry, last_pos = pos;
        float result[kWindowChannels];
#pragma unroll
        for (int i = 0; i < kWindowChannels; ++i) {
            const float now = mine[k].get(i);
            float acc = 0.f;
#pragma unroll
            for (int j = 0; j < kBefore; ++j) acc = fmaf(taps[i * kWindowTaps + j], window[j][i], acc);        // oldest input first
            acc = fmaf(taps[i * kWindowTaps + kBefore], now, acc);
            if (add_input) acc += now;
            if (bias.ptr) acc += add[i];
            result[i] = activate(acc, act);
#pragma unroll
            for (int j = 0; j + 1 < kBefore; ++j) window[j][i] = window[j + 1][i];
            window[kBefore - 1][i] = now;
        }
        store_four(out + static_cast<long>(r) * out_stride + c, result);
    }
}

template <typename TIn>
__global__ void causal_conv_state_kernel(const TIn* __restrict__ in, long in_stride, float* __restrict__ state,
                                         const int* __restrict__ spans, const int* __restrict__ entry_slots,
                                         const int* __restrict__ positions, int channels, int taps) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int e = blockIdx.y;
    if (c >= channels) return;
    const int first = spans[4 * e], n = spans[4 * e + 1] - first;
    const int start = positions[first];
    float* mine = state + (static_cast<long>(entry_slots[e]) * (taps - 1)) * channels + c;
    float keep[kMaxTaps - 1];
    for (int j = 0; j < taps - 1; ++j) {
        const int back = taps - 1 - j;                        // how far before the end of the portion
        if (back <= n) keep[j] = to_float(in[static_cast<long>(first + n - back) * in_stride + c]);
        else if (start + n - back < 0) keep[j] = 0.f;
        else keep[j] = mine[static_cast<long>(taps - 1 - (back - n)) * channels];
    }
    for (int j = 0; j < taps - 1; ++j) mine[static_cast<long>(j) * channels] = keep[j];
}

// Where the new running maximum of exponential gates made in a step of single rows (outer_step) goes: row r's is top's, in the state of the
// slot that the r-th span writes.  Kernels that keep none have no such argument (asked for at run time it cost them up to 6 %).
struct KeepTop {
    float* state;                // the first slot's first maximum
    long slot_stride, head_stride;
    const int* spans;            // [rows, 4]
};
// The slot, a span's fourth word, is asked for with a row's first loads by the fourth lane, as a vector load that comes back among them, and written
// to at the row's end (as the scalar that it is, it is waited for before anything else).  Eight rows of four heads of 512 in a decode step: 4.9 us.
constexpr int kKeeper = 3;
__device__ inline int slot_to_keep(int row, int lane, const KeepTop& keep) { return keep.spans[4 * row + lane % 4]; }
__device__ inline void keep_top(int slot, int head, float value, const KeepTop& keep) {
    if (slot >= 0) keep.state[slot * keep.slot_stride + head * keep.head_stride] = value;
}

// One wave per (row, head).
template <typename TOut, int kKept, typename... Keep>
__global__ void head_norm_gate_kernel(const float* __restrict__ o, const float* __restrict__ dot, const float* __restrict__ top,
                                      AnyVec gain, int gain_per_head, const float* __restrict__ gate, long gate_stride,
                                      int act, float eps, TOut* __restrict__ out, int heads, int vdim, int gate_first, Keep... keep) {
    const int row = blockIdx.x;
    const int head = blockIdx.y * (blockDim.x / kWave) + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (head >= heads) return;
    const long at = static_cast<long>(row) * heads + head;
    const float* src = o + at * vdim;
    const float* gate_row = gate ? gate + static_cast<long>(row) * gate_stride + static_cast<long>(head) * vdim : nullptr;
    // Few rows are a chain of trips to memory: the run, its gate, its gains and what divides it are asked for side by side
    // (at indexes held inside the run, so that no branch stands between the loads).  Eight rows of four heads of 512: 4.8 us (8.8 before).
    // kKept: the values a lane keeps between the two passes.
    const long gain_at = gain_per_head ? static_cast<long>(head) * vdim : 0;
    float kept[kKept], open[kKept] = {}, by[kKept];
    const float read = dot ? dot[at] : 0.f, highest = dot ? top[at] : 0.f;
    [[maybe_unused]] int slot = -1;
    if constexpr (sizeof...(Keep) > 0) slot = slot_to_keep(row, lane, keep...);
    auto within = [&](int n) { return min(lane + n * kWave, vdim - 1); };
#pragma unroll
    for (int n = 0; n < kKept; ++n) kept[n] = src[within(n)];
    if (gate_row) {
#pragma unroll
        for (int n = 0; n < kKept; ++n) open[n] = gate_row[within(n)];
    }
    if (gain.ptr && gain.dtype == kF32) {
#pragma unroll
        for (int n = 0; n < kKept; ++n) by[n] = static_cast<const float*>(gain.ptr)[gain_at + within(n)];
    } else if (gain.ptr) {
        bf16_t raw[kKept];
#pragma unroll
        for (int n = 0; n < kKept; ++n) raw[n] = static_cast<const bf16_t*>(gain.ptr)[gain_at + within(n)];
#pragma unroll
        for (int n = 0; n < kKept; ++n) by[n] = to_float(raw[n]);
    }
    float under = 1.f;
    if (dot) under = fmaxf(fabsf(read), expf(-highest)) + 1e-6f;
    // with gate_first the gate multiplies ahead of the norm, and the root mean square is that of the gated values
    if (gate_row) {                                            // (once for both places: a fifth less code, which a decode step fetches anew every time: 5.4 us, so 4.9)
#pragma unroll
        for (int n = 0; n < kKept; ++n)
            if (n * kWave < vdim) open[n] = activate(open[n], act);
    }
    auto gate_of = [&](int j) { return gate_row ? activate(gate_row[j], act) : 0.f; };
    auto opened = [&](float v, float g) {
        v /= under;
        return (gate_first && gate_row) ? v * g : v;
    };
    float ss = 0.f;
#pragma unroll
    for (int n = 0; n < kKept; ++n) {
        kept[n] = lane + n * kWave < vdim ? opened(kept[n], open[n]) : 0.f;
        ss = fmaf(kept[n], kept[n], ss);
    }
    for (int j = lane + kKept * kWave; j < vdim; j += kWave) {
        const float v = opened(src[j], gate_first ? gate_of(j) : 0.f);
        ss = fmaf(v, v, ss);
    }
    const float inv = 1.0f / sqrtf(wave_sum(ss) / static_cast<float>(vdim) + eps);
    TOut* dst = out + at * vdim;
    auto finish = [&](int j, float v, float by_gain, float g) {
        v *= inv;
        if (gain.ptr) v *= by_gain;
        if (gate_row && !gate_first) v *= g;
        dst[j] = from_float<TOut>(v);
    };
#pragma unroll
    for (int n = 0; n < kKept; ++n)
        if (lane + n * kWave < vdim) finish(lane + n * kWave, kept[n], by[n], open[n]);
    for (int j = lane + kKept * kWave; j < vdim; j += kWave) {
        const float g = gate_of(j);
        finish(j, opened(src[j], g), gain.ptr ? load_any(gain, gain_at + j) : 1.f, g);
    }
    if constexpr (sizeof...(Keep) > 0)
        if (lane == kKeeper) keep_top(slot, head, highest, keep...);
}

// The same for runs too long for a wave: a workgroup a (row, head), the values kept in registers between the passes where they
// fit, sums added in a fixed order.
constexpr int kWideHeadFrom = 1024;                            // runs of more columns go here
template <typename TOut, int kThreads, typename... Keep>
__global__ void __launch_bounds__(kThreads)
head_norm_gate_wide_kernel(const float* __restrict__ o, const float* __restrict__ dot, const float* __restrict__ top, AnyVec gain,
                           int gain_per_head, const float* __restrict__ gate, long gate_stride, int act, float eps,
                           TOut* __restrict__ out, int heads, int vdim, int gate_first, Keep... keep) {
    __shared__ float scratch[kThreads / kWave];
    const int row = blockIdx.x, head = blockIdx.y;
    const long at = static_cast<long>(row) * heads + head;
    [[maybe_unused]] int slot = -1;
    if constexpr (sizeof...(Keep) > 0) slot = slot_to_keep(row, threadIdx.x, keep...);
    const float* src = o + at * vdim;
    const float under = dot ? fmaxf(fabsf(dot[at]), expf(-top[at])) + 1e-6f : 1.f;
    const float* gate_row = gate ? gate + static_cast<long>(row) * gate_stride + static_cast<long>(head) * vdim : nullptr;
    auto fetch = [&](int j) {
        const float v = src[j] / under;
        return (gate_first && gate_row) ? v * activate(gate_row[j], act) : v;
    };
    constexpr int kKept = 4;
    float kept[kKept], open[kKept];
    float ss = 0.f;
#pragma unroll
    for (int n = 0; n < kKept; ++n) {
        const int j = threadIdx.x + n * kThreads;
        kept[n] = j < vdim ? fetch(j) : 0.f;
        open[n] = (gate_row && !gate_first && j < vdim) ? gate_row[j] : 0.f;     // asked for ahead of the sum
        ss = fmaf(kept[n], kept[n], ss);
    }
    for (int j = threadIdx.x + kKept * kThreads; j < vdim; j += kThreads) {
        const float v = fetch(j);
        ss = fmaf(v, v, ss);
    }
    const float inv = 1.0f / sqrtf(block_sum<kThreads>(ss, scratch) / static_cast<float>(vdim) + eps);
    TOut* dst = out + at * vdim;
    auto finish = [&](int j, float v, float g) {
        v *= inv;
        if (gain.ptr) v *= load_any(gain, gain_per_head ? static_cast<long>(head) * vdim + j : j);
        if (gate_row && !gate_first) v *= activate(g, act);
        dst[j] = from_float<TOut>(v);
    };
#pragma unroll
    for (int n = 0; n < kKept; ++n)
        if (threadIdx.x + n * kThreads < static_cast<unsigned>(vdim)) finish(threadIdx.x + n * kThreads, kept[n], open[n]);
    for (int j = threadIdx.x + kKept * kThreads; j < vdim; j += kThreads) finish(j, fetch(j), gate_row && !gate_first ? gate_row[j] : 0.f);
    if constexpr (sizeof...(Keep) > 0)
        if (threadIdx.x == kKeeper) keep_top(slot, head, top[at], keep...);
}

constexpr int kMaxBranches = 4;
struct Branches {
    const float* rows[kMaxBranches];
    AnyVec gain[kMaxBranches];
};

template <int kNormThreads>
__global__ void __launch_bounds__(kNormThreads)
rms_mix_kernel(Branches in, int branches, float eps, float scale, float* __restrict__ out, int hidden) {
    __shared__ float scratch[kNormThreads / kWave];
    const long row = blockIdx.x;
    float inv[kMaxBranches];
    for (int b = 0; b < branches; ++b) {
        const float* src = in.rows[b] + row * hidden;
        float ss = 0.f;
        for (int i = threadIdx.x; i < hidden; i += kNormThreads) ss = fmaf(src[i], src[i], ss);
        inv[b] = 1.0f / sqrtf(block_sum<kNormThreads>(ss, scratch) / static_cast<float>(hidden) + eps);
    }
    for (int i = threadIdx.x; i < hidden; i += kNormThreads) {
        float total = 0.f;
        for (int b = 0; b < branches; ++b) total += in.rows[b][row * hidden + i] * inv[b] * load_any(in.gain[b], i);
        out[row * hidden + i] = total * scale;
    }
}

// out = sum_b weight_b * branch_b, nothing normed.
__global__ void weighted_mix_kernel(Branches in, int branches, float w0, float w1, float w2, float w3, float* __restrict__ out, long n) {
    const float weight[kMaxBranches] = {w0, w1, w2, w3};
    for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * blockDim.x) {
        float total = 0.f;
        for (int b = 0; b < branches; ++b) total = fmaf(weight[b], in.rows[b][i], total);
        out[i] = total;
    }
}

template <typename T>
__global__ void relu_squared_kernel(const T* __restrict__ in, T* __restrict__ out, long n) {
    for (long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * blockDim.x) {
        const float v = fmaxf(to_float(in[i]), 0.f);
        out[i] = from_float<T>(v * v);
    }
}

// Per-head sigmoid gates on attention's output: out[r, h, :] *= sigmoid(gate[r * stride + h]).
template <typename T>
__global__ void head_gate_kernel(T* __restrict__ out, const float* __restrict__ gate, long gate_stride, int heads, int vdim, long n) {
    const long i = blockIdx.x * static_cast<long>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    const long row = i / (static_cast<long>(heads) * vdim);
    const int head = static_cast<int>((i / vdim) % heads);
    out[i] = from_float<T>(to_float(out[i]) * activate(gate[row * gate_stride + head], kActSigmoid));
}

// The same in runs of eight elements of a row (`runs` of them), which have one gate (kEach: a gate each).  What bounds it are its
// bytes: 2,114 rows of 2,048 with cold caches, a gate an element 15.0 us, a gate a head of 128 7.8 (element by element, with two
// divisions each, 22.6 and 16.9).
// A gate an element is eight exponentials one after the other in a thread, which few values wait for: up to so many go element by element.
// (us with warm caches, runs and elements: in bfloat16 16 x 2,048 2.8 and 2.4, 128 x 2,048 2.9 and 2.7, 192 x 2,048 3.0 and 3.0, 512 x 512 3.0
// and 2.7; in float 384 x 512 2.6 and 2.6, 128 x 2,048 2.6 and 2.7.  A gate a head: 16 x 2,048 2.4 and 2.4.)
static bool gates_in_runs(int dtype, bool each, long n) { return !each || n >= (dtype == kBF16 ? 192L << 11 : 96L << 11); }
template <typename T, bool kEach>
__global__ void __launch_bounds__(256)
head_gate_runs_kernel(T* __restrict__ out, const float* __restrict__ gate, long gate_stride, int runs, int vdim, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int row = i / runs, at = (i - row * runs) * kRun, length = runs * kRun;
    const float* gates = gate + row * gate_stride;
    T* mine = out + static_cast<long>(row) * length;
    Run<T> v;
    v.load(mine, at, length);
    Run<float> each;
    float one = 0.f;
    if constexpr (kEach) each.load(gates, at, length);
    else one = gates[at / vdim];
    float result[kRun];
#pragma unroll
    for (int k = 0; k < kRun; ++k) result[k] = v.get(k) * activate(kEach ? each.get(k) : one, kActSigmoid);
    store_run<T>(mine, at, length, result);
}

static bool known(int dtype) { return dtype == kF32 || dtype == kBF16; }

}  // namespace leone

using namespace leone;

extern "C" int leone_add_layernorm(float* x, const float* delta, const void* dw, const void* db, float deps,
                                   const void* w, const void* b, int w_dtype, float eps, void* y, int y_dtype,
                                   const int* rows, int n_out, int hidden, const void* conv, int conv_dtype, int taps,
                                   float* conv_state, int write_state, const int* positions, const int* row_entry,
                                   const int* entry_slots, hipStream_t stream) {
    LEONE_REQUIRE(!conv || (y && !rows && conv_state && positions && row_entry && entry_slots && taps >= 2 && taps <= kMaxTaps &&
                            known(conv_dtype)), "add_layernorm: a folded convolution needs its state, the rows' places and 2..%d taps", kMaxTaps);
    const AnyVec vconv{conv, conv_dtype};
    LEONE_REQUIRE(x && n_out > 0 && hidden > 0, "add_layernorm: needs a stream and positive sizes");
    LEONE_REQUIRE(known(w_dtype) && known(y_dtype), "add_layernorm: unknown element type");
    LEONE_REQUIRE((dw == nullptr) == (db == nullptr), "add_layernorm: the delta's gain and bias come together");
    LEONE_REQUIRE(!dw || (delta && deps > 0.f), "add_layernorm: a norm of the delta needs a delta and an eps");
    LEONE_REQUIRE(!y || (w && b && eps > 0.f), "add_layernorm: the output norm needs gain, bias and eps");
    LEONE_REQUIRE(y || (delta && !rows), "add_layernorm: nothing to do");
    LEONE_REQUIRE(static_cast<size_t>(hidden) * sizeof(float) <= 64 * 1024, "add_layernorm: rows of %d elements are too long", hidden);
    const AnyVec vdw{dw, w_dtype}, vdb{db, w_dtype}, vw{w, w_dtype}, vb{b, w_dtype};
    const int stage_delta = (delta && static_cast<size_t>(hidden) * 2 * sizeof(float) <= 64 * 1024) ? 1 : 0;
    const size_t shared = static_cast<size_t>(hidden) * sizeof(float) * (stage_delta ? 2 : 1);
#define LEONE_LAYERNORM(T, THREADS)                                                                                        \
    add_layernorm_kernel<T, THREADS><<<n_out, THREADS, shared, stream>>>(x, delta, vdw, vdb, deps, vw, vb, eps, static_cast<T*>(y), \
                                                                         rows, hidden, vconv, taps, conv_state, write_state,   \
                                                                         positions, row_entry, entry_slots, stage_delta)
    const bool many = n_out >= kNormManyRows;
    // Rows that fit registers, one type of vectors throughout: few rows by a workgroup each, many rows by a wave each where they lie in
    // whole 16-byte runs.  Few rows go in such runs too where they lie so, a filter in four taps, and else element by element: in runs
    // that were loaded by elements a thread takes 490 registers and neighbours lie 32 bytes apart (us, element by element: 8 rows of
    // 2,049 10.1, so 5.2, of 4,095 12.9, 5.3, of 4,096 with three taps 25.2, 8.1).  Rows of more than 2,048 without a filter go element by
    // element up to one a compute unit: a thread with four runs of everything is the longer chain (8 rows of 4,096, two norms, vectors in
    // bfloat16 and in float: in runs 6.2 and 6.5, so 5.4 and 5.1; 256 rows 7.2 and 7.5, 6.5 and 6.4), and with two workgroups a unit
    // the runs are ahead (384 rows 8.8 and 9.5, so 12.2 and 12.1).
    const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    const bool vec = hidden % kRun == 0 && aligned(x) && aligned(delta) && aligned(dw) && aligned(db) && aligned(w) && aligned(b) &&
                     aligned(y) && (!conv || (taps == kHeldTaps && aligned(conv) && aligned(conv_state)));
    if (!many && hidden <= 4 * kNormThreadsFew && (!conv || (taps <= kHeldTaps && conv_dtype == w_dtype))) {
        constexpr int kTwoRuns = 2 * kRun * kHeldThreads, kSingleRows = 256;
        static_assert(kTwoRuns == 2 * kNormThreadsFew, "both kernels hold the same rows");
        const bool single = !vec || (!conv && hidden > kTwoRuns && n_out <= kSingleRows);
#define LEONE_SINGLE(T, TW, PER)                                                                                                \
    add_layernorm_single_kernel<T, TW, PER><<<n_out, kNormThreadsFew, 0, stream>>>(                                             \
        x, delta, static_cast<const TW*>(dw), static_cast<const TW*>(db), deps, static_cast<const TW*>(w), static_cast<const TW*>(b), eps, \
        static_cast<T*>(y), rows, hidden, static_cast<const TW*>(conv), taps, conv_state, write_state, positions, row_entry, entry_slots)
#define LEONE_HELD(T, TW, PER, TAPS)                                                                                            \
    add_layernorm_held_kernel<T, TW, PER, TAPS><<<n_out, kHeldThreads, 0, stream>>>(                                            \
        x, delta, static_cast<const TW*>(dw), static_cast<const TW*>(db), deps, static_cast<const TW*>(w), static_cast<const TW*>(b), eps, \
        static_cast<T*>(y), rows, hidden, static_cast<const TW*>(conv), conv_state, write_state, positions, row_entry, entry_slots)
#define LEONE_FEW_PER(T, TW, PER)                                                                                               \
    (single ? LEONE_SINGLE(T, TW, PER) : conv ? LEONE_HELD(T, TW, PER, kHeldTaps) : LEONE_HELD(T, TW, PER, 0))
#define LEONE_FEW(T, TW) (hidden <= kTwoRuns ? LEONE_FEW_PER(T, TW, 2) : LEONE_FEW_PER(T, TW, 4))
        if (y_dtype == kF32 && w_dtype == kF32) LEONE_FEW(float, float);
        else if (y_dtype == kF32) LEONE_FEW(float, bf16_t);
        else if (w_dtype == kF32) LEONE_FEW(bf16_t, float);
        else LEONE_FEW(bf16_t, bf16_t);
#undef LEONE_FEW
#undef LEONE_FEW_PER
#undef LEONE_HELD
#undef LEONE_SINGLE
        LEONE_LAUNCH_CHECK("add_layernorm");
        return 0;
    }
    if (many && vec && !conv && hidden <= 4096) {
#define LEONE_WAVE(T, TW, PER)                                                                                                    \
    add_layernorm_wave_kernel<T, TW, PER><<<ceil_div(n_out, kRowThreads / kWave), kRowThreads, 0, stream>>>(                      \
        x, delta, static_cast<const TW*>(dw), static_cast<const TW*>(db), deps, static_cast<const TW*>(w), static_cast<const TW*>(b), eps, \
        static_cast<T*>(y), rows, n_out, hidden)
#define LEONE_WAVE_PER(T, TW) (hidden <= 1024 ? LEONE_WAVE(T, TW, 4) : hidden <= 2048 ? LEONE_WAVE(T, TW, 8) : LEONE_WAVE(T, TW, 16))
        if (y_dtype == kF32 && w_dtype == kF32) LEONE_WAVE_PER(float, float);
        else if (y_dtype == kF32) LEONE_WAVE_PER(float, bf16_t);
        else if (w_dtype == kF32) LEONE_WAVE_PER(bf16_t, float);
        else LEONE_WAVE_PER(bf16_t, bf16_t);
#undef LEONE_WAVE_PER
#undef LEONE_WAVE
        LEONE_LAUNCH_CHECK("add_layernorm");
        return 0;
    }
    if (y_dtype == kF32) {
        if (many) LEONE_LAYERNORM(float, kNormThreadsMany);
        else LEONE_LAYERNORM(float, kNormThreadsFew);
    } else {
        if (many) LEONE_LAYERNORM(bf16_t, kNormThreadsMany);
        else LEONE_LAYERNORM(bf16_t, kNormThreadsFew);
    }
#undef LEONE_LAYERNORM
    LEONE_LAUNCH_CHECK("add_layernorm");
    return 0;
}

extern "C" int leone_entry_spans(const int* row_entry, const int* positions, const int* entry_slots, int rows, int* spans,
                                 hipStream_t stream) {
    LEONE_REQUIRE(row_entry && positions && entry_slots && spans && rows > 0, "entry_spans: needs a row map");
    entry_spans_kernel<<<ceil_div(rows, 256), 256, 0, stream>>>(row_entry, positions, entry_slots, rows, spans);
    LEONE_LAUNCH_CHECK("entry_spans");
    return 0;
}

extern "C" int leone_causal_conv(const void* in, int in_dtype, long in_stride, void* out, int out_dtype, long out_stride,
                                 const void* w, int w_dtype, float* state, int write_state, const int* spans, int entries,
                                 const int* positions, const int* row_entry, const int* entry_slots, int rows,
                                 int channels, int taps, int add_input, int act, int single_rows, hipStream_t stream) {
    return leone_causal_conv_biased(in, in_dtype, in_stride, out, out_dtype, out_stride, w, nullptr, w_dtype, state, write_state,
                                    spans, entries, positions, row_entry, entry_slots, rows, channels, taps, add_input, act,
                                    single_rows, stream);
}

// bias: one value a channel ([channels], of the filters' type) added to the filter's sum ahead of the activation; may be null.
extern "C" int leone_causal_conv_biased(const void* in, int in_dtype, long in_stride, void* out, int out_dtype, long out_stride,
                                        const void* w, const void* bias, int w_dtype, float* state, int write_state,
                                        const int* spans, int entries, const int* positions, const int* row_entry,
                                        const int* entry_slots, int rows, int channels, int taps, int add_input, int act,
                                        int single_rows, hipStream_t stream) {
    LEONE_REQUIRE(in && out && w && state && positions && row_entry && entry_slots, "causal_conv: null pointer");
    LEONE_REQUIRE(known(in_dtype) && known(out_dtype) && known(w_dtype), "causal_conv: unknown element type");
    LEONE_REQUIRE(rows > 0 && channels > 0 && ceil_div(channels, 256) <= 65535 && in_stride >= channels && out_stride >= channels,
                  "causal_conv: %d rows of %d channels", rows, channels);
    LEONE_REQUIRE(taps >= 2 && taps <= kMaxTaps, "causal_conv: %d taps, the kernel takes 2..%d", taps, kMaxTaps);
    LEONE_REQUIRE(act >= kActNone && act <= kActSilu, "causal_conv: unknown activation %d", act);
    LEONE_REQUIRE(!write_state || single_rows || (spans && entries > 0 && entries <= 65535),
                  "causal_conv: the state's update needs the entries' spans");
    const AnyVec vw{w, w_dtype};
    const AnyVec vbias{bias, w_dtype};
    const int per_block = rows >= kNormManyRows ? kConvRows : 1;
    const dim3 grid(ceil_div(rows, per_block), ceil_div(channels, 256));
    float* const own_state = (write_state && single_rows) ? state : nullptr;
    // Four channels a thread where rows of the inputs, the outputs and the state can be read and written so, in steps whose workgroups take
    // eight rows.  That line, in rows alone, is right for rows of some 1,500 channels: with a row a workgroup and with the window, us, 64
    // rows of 2,048 3.6 and 5.9, 256 5.2 and 5.9, 511 8.1 and 6.1; of 4,096 128 rows 5.3 and 5.2, 511 18.3 and 6.5; of 512 511 rows 4.3 and
    // 5.9, where eight rows a workgroup without the window take 10.3.
    const auto fours = [&](const void* p, long stride, int size) {
        return stride % kWindowChannels == 0 && reinterpret_cast<uintptr_t>(p) % (kWindowChannels * size) == 0;
    };
    const bool window = per_block > 1 && taps == kWindowTaps && !own_state && fours(in, in_stride, in_dtype == kF32 ? 4 : 2) &&
                        fours(out, out_stride, out_dtype == kF32 ? 4 : 2) && fours(state, channels, 4) &&
                        reinterpret_cast<uintptr_t>(w) % 16 == 0;
    const dim3 window_grid(grid.x, ceil_div(channels, kWindowThreads * kWindowChannels));
#define LEONE_CONV(TIN, TOUT)                                                                                         \
    (window ? causal_conv_window_kernel<TIN, TOUT><<<window_grid, kWindowThreads, 0, stream>>>(                           \
                  static_cast<const TIN*>(in), in_stride, static_cast<TOUT*>(out), out_stride, vw, vbias, state, positions, \
                  row_entry, entry_slots, rows, channels, add_input, act)                                             \
            : causal_conv_kernel<TIN, TOUT><<<grid, 256, 0, stream>>>(static_cast<const TIN*>(in), in_stride, static_cast<TOUT*>(out), \
                                                                      out_stride, vw, vbias, state, positions, row_entry, entry_slots, \
                                                                      rows, channels, taps, add_input, act, own_state, per_block))
    if (in_dtype == kF32 && out_dtype == kF32) LEONE_CONV(float, float);
    else if (in_dtype == kF32) LEONE_CONV(float, bf16_t);
    else if (out_dtype == kF32) LEONE_CONV(bf16_t, float);
    else LEONE_CONV(bf16_t, bf16_t);
#undef LEONE_CONV
    LEONE_LAUNCH_CHECK("causal_conv");
    if (write_state && !single_rows) {
        const dim3 sgrid(ceil_div(channels, 256), entries);
        if (in_dtype == kF32)
            causal_conv_state_kernel<float><<<sgrid, 256, 0, stream>>>(static_cast<const float*>(in), in_stride, state, spans,
                                                                       entry_slots, positions, channels, taps);
        else
            causal_conv_state_kernel<bf16_t><<<sgrid, 256, 0, stream>>>(static_cast<const bf16_t*>(in), in_stride, state, spans,
                                                                        entry_slots, positions, channels, taps);
        LEONE_LAUNCH_CHECK("causal_conv_state");
    }
    return 0;
}

extern "C" int leone_head_norm_gate(const float* o, const float* dot, const float* top, const void* gain, int gain_dtype,
                                    int gain_per_head, const float* gate, long gate_stride, int act, float eps, void* out,
                                    int out_dtype, int rows, int heads, int vdim, hipStream_t stream) {
    return leone_head_norm_gate_ordered(o, dot, top, gain, gain_dtype, gain_per_head, gate, gate_stride, act, 0, eps, out,
                                        out_dtype, rows, heads, vdim, stream);
}

// keep_state (may be null): see KeepTop.
// gate_first: the gate multiplies ahead of the norm (the root mean square is taken of the gated values) instead of behind it.
extern "C" int leone_head_norm_gate_kept(const float* o, const float* dot, const float* top, const void* gain, int gain_dtype,
                                         int gain_per_head, const float* gate, long gate_stride, int act, int gate_first,
                                         float eps, void* out, int out_dtype, int rows, int heads, int vdim,
                                         float* keep_state, long keep_slot_stride, long keep_head_stride,
                                         const int* keep_spans, hipStream_t stream) {
    LEONE_REQUIRE(!keep_state || (top && keep_spans), "head_norm_gate: a maximum that is kept needs its value and the rows' slots");
    const KeepTop keep{keep_state, keep_slot_stride, keep_head_stride, keep_spans};
    LEONE_REQUIRE(o && out && rows > 0 && heads > 0 && vdim > 0, "head_norm_gate: needs read-outs and positive sizes");
    LEONE_REQUIRE(known(out_dtype) && (!gain || known(gain_dtype)), "head_norm_gate: unknown element type");
    LEONE_REQUIRE((dot == nullptr) == (top == nullptr), "head_norm_gate: the denominator's two parts come together");
    LEONE_REQUIRE(act >= kActNone && act <= kActSilu && eps > 0.f, "head_norm_gate: activation %d, eps %g", act, eps);
    LEONE_REQUIRE(rows <= 0x7fffffff && ceil_div(heads, 4) <= 65535, "head_norm_gate: too many heads");
    const AnyVec vg{gain, gain_dtype};
    if (vdim > kWideHeadFrom) {
        LEONE_REQUIRE(heads <= 65535, "head_norm_gate: too many heads");
        // few rows: a row in as few trips to memory as threads allow; many rows: more rows in flight a compute unit
        const auto launch = [&](auto* to, auto... kept) {
            using T = std::remove_pointer_t<decltype(to)>;
            if (rows >= kNormManyRows)
                head_norm_gate_wide_kernel<T, kNormThreadsMany><<<dim3(rows, heads), kNormThreadsMany, 0, stream>>>(
                    o, dot, top, vg, gain_per_head, gate, gate_stride, act, eps, to, heads, vdim, gate_first, kept...);
            else
                head_norm_gate_wide_kernel<T, kNormThreadsFew><<<dim3(rows, heads), kNormThreadsFew, 0, stream>>>(
                    o, dot, top, vg, gain_per_head, gate, gate_stride, act, eps, to, heads, vdim, gate_first, kept...);
        };
        if (out_dtype == kF32) keep_state ? launch(static_cast<float*>(out), keep) : launch(static_cast<float*>(out));
        else keep_state ? launch(static_cast<bf16_t*>(out), keep) : launch(static_cast<bf16_t*>(out));
        LEONE_LAUNCH_CHECK("head_norm_gate");
        return 0;
    }
    const dim3 grid(rows, ceil_div(heads, 4));
    // Heads of 64 and 128 hold one and two values a lane: asking for eight reads the same ones again (us, 2,048 rows of 32 heads of
    // 64, eight and one: 26.8 and 19.6; 16 of 128, eight and two: 17.9 and 14.1).
    const auto launch = [&](auto* to, auto... kept) {
        using T = std::remove_pointer_t<decltype(to)>;
        const auto of = [&](auto values) {
            head_norm_gate_kernel<T, decltype(values)::value><<<grid, 4 * kWave, 0, stream>>>(o, dot, top, vg, gain_per_head, gate, gate_stride, act, eps,
                                                                                              to, heads, vdim, gate_first, kept...);
        };
        if (vdim <= kWave) of(std::integral_constant<int, 1>{});
        else if (vdim <= 2 * kWave) of(std::integral_constant<int, 2>{});
        else of(std::integral_constant<int, 8>{});
    };
    if (out_dtype == kF32) keep_state ? launch(static_cast<float*>(out), keep) : launch(static_cast<float*>(out));
    else keep_state ? launch(static_cast<bf16_t*>(out), keep) : launch(static_cast<bf16_t*>(out));
    LEONE_LAUNCH_CHECK("head_norm_gate");
    return 0;
}

extern "C" int leone_head_norm_gate_ordered(const float* o, const float* dot, const float* top, const void* gain, int gain_dtype,
                                            int gain_per_head, const float* gate, long gate_stride, int act, int gate_first,
                                            float eps, void* out, int out_dtype, int rows, int heads, int vdim,
                                            hipStream_t stream) {
    return leone_head_norm_gate_kept(o, dot, top, gain, gain_dtype, gain_per_head, gate, gate_stride, act, gate_first, eps, out, out_dtype,
                                     rows, heads, vdim, nullptr, 0, 0, nullptr, stream);
}

extern "C" int leone_rms_mix(const float* const* branch_rows, const void* const* gains, int gain_dtype, int branches,
                             float eps, float scale, float* out, int rows, int hidden, hipStream_t stream) {
    LEONE_REQUIRE(branch_rows && gains && out && rows > 0 && hidden > 0, "rms_mix: needs branches and positive sizes");
    LEONE_REQUIRE(branches >= 1 && branches <= kMaxBranches, "rms_mix: %d branches, the kernel takes 1..%d", branches, kMaxBranches);
    LEONE_REQUIRE(known(gain_dtype) && eps > 0.f, "rms_mix: unknown gain type or eps");
    Branches in{};
    for (int b = 0; b < branches; ++b) {
        LEONE_REQUIRE(branch_rows[b] && gains[b], "rms_mix: branch %d is missing", b);
        in.rows[b] = branch_rows[b];
        in.gain[b] = AnyVec{gains[b], gain_dtype};
    }
    if (rows >= kNormManyRows) rms_mix_kernel<kNormThreadsMany><<<rows, kNormThreadsMany, 0, stream>>>(in, branches, eps, scale, out, hidden);
    else rms_mix_kernel<kNormThreadsFew><<<rows, kNormThreadsFew, 0, stream>>>(in, branches, eps, scale, out, hidden);
    LEONE_LAUNCH_CHECK("rms_mix");
    return 0;
}

extern "C" int leone_weighted_mix(const float* const* branch_rows, const float* weights, int branches, float* out, long n,
                                  hipStream_t stream) {
    LEONE_REQUIRE(branch_rows && weights && out && n > 0, "weighted_mix: needs branches and a positive size");
    LEONE_REQUIRE(branches >= 1 && branches <= kMaxBranches, "weighted_mix: %d branches, the kernel takes 1..%d", branches, kMaxBranches);
    Branches in{};
    float w[kMaxBranches] = {0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < branches; ++b) {
        LEONE_REQUIRE(branch_rows[b], "weighted_mix: branch %d is missing", b);
        in.rows[b] = branch_rows[b];
        w[b] = weights[b];
    }
    const long blocks = (n + 255) / 256;
    weighted_mix_kernel<<<static_cast<int>(blocks < 4096 ? blocks : 4096), 256, 0, stream>>>(in, branches, w[0], w[1], w[2], w[3], out, n);
    LEONE_LAUNCH_CHECK("weighted_mix");
    return 0;
}

extern "C" int leone_relu_squared(const void* in, void* out, int dtype, long n, hipStream_t stream) {
    LEONE_REQUIRE(in && out && n > 0 && known(dtype), "relu_squared: needs values of a known type");
    const long blocks = (n + 255) / 256;
    const int grid = static_cast<int>(blocks < 8192 ? blocks : 8192);
    if (dtype == kF32) relu_squared_kernel<float><<<grid, 256, 0, stream>>>(static_cast<const float*>(in), static_cast<float*>(out), n);
    else relu_squared_kernel<bf16_t><<<grid, 256, 0, stream>>>(static_cast<const bf16_t*>(in), static_cast<bf16_t*>(out), n);
    LEONE_LAUNCH_CHECK("relu_squared");
    return 0;
}

extern "C" int leone_gates_in_runs(int dtype, int each, long n) { return gates_in_runs(dtype, each != 0, n); }
extern "C" int leone_head_gate(void* out, int dtype, const float* gate, long gate_stride, int rows, int heads, int vdim,
                               hipStream_t stream) {
    LEONE_REQUIRE(out && gate && known(dtype) && rows > 0 && heads > 0 && vdim > 0, "head_gate: needs values and gates");
    const long n = static_cast<long>(rows) * heads * vdim;
    LEONE_REQUIRE((n + 255) / 256 <= 0x7fffffffL, "head_gate: too many values");
    // Runs of eight where a row's elements and its gates can be read so: every run in one head, or a gate an element.
    const bool each = vdim == 1, aligned = reinterpret_cast<uintptr_t>(out) % 16 == 0;
    if (aligned && n <= 0x7fffffffL && gates_in_runs(dtype, each, n) &&
        (each ? heads % kRun == 0 && gate_stride % 4 == 0 && reinterpret_cast<uintptr_t>(gate) % 16 == 0 : vdim % kRun == 0)) {
        const int runs = static_cast<int>(static_cast<long>(heads) * vdim / kRun), items = static_cast<int>(n / kRun), blocks = ceil_div(items, 256);
#define LEONE_GATE_RUNS(T, EACH) \
    head_gate_runs_kernel<T, EACH><<<blocks, 256, 0, stream>>>(static_cast<T*>(out), gate, gate_stride, runs, vdim, items)
        if (dtype == kF32) each ? LEONE_GATE_RUNS(float, true) : LEONE_GATE_RUNS(float, false);
        else each ? LEONE_GATE_RUNS(bf16_t, true) : LEONE_GATE_RUNS(bf16_t, false);
#undef LEONE_GATE_RUNS
        LEONE_LAUNCH_CHECK("head_gate");
        return 0;
    }
    const int grid = static_cast<int>((n + 255) / 256);
    if (dtype == kF32) head_gate_kernel<float><<<grid, 256, 0, stream>>>(static_cast<float*>(out), gate, gate_stride, heads, vdim, n);
    else head_gate_kernel<bf16_t><<<grid, 256, 0, stream>>>(static_cast<bf16_t*>(out), gate, gate_stride, heads, vdim, n);
    LEONE_LAUNCH_CHECK("head_gate");
    return 0;
}
