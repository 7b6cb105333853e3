// Mixers that keep a matrix memory per request and head instead of a cache of keys: S is [dim, vdim] float,
// carried from token to token in the request's state slot.
//
//   outer_scan   S_t = a_t S_(t-1) + b_t k_t v_t^T,  o_t = S_t^T q_t
//                a_t, b_t per head and token: a fixed decay with b = 1 (retention), or exponential gates with a
//                running maximum m_t = max(f_t + m_(t-1), i_t), a_t = exp(f_t + m_(t-1) - m_t),
//                b_t = exp(i_t - m_t), together with the normaliser n_t = a_t n_(t-1) + b_t k_t carried as one
//                more column of S (a value that is always 1), whose read-out n_t . q_t and m_t go out beside o
//                for the division that follows.  Rotary positions on q and k if tables come; q, k and v through silu first if
//                asked for.
//   delta_scan   S <- g_t * S (g per key channel, or one a head);  u = beta_t (v_t - S^T k_t);  S <- S + k_t u^T;  o_t = S^T q_t
//                with q and k made unit vectors per head first.
//
// A workgroup of four waves owns a run of columns of one head of one segment (a request's rows in the step, or a
// chunk of them) and walks the segment's rows in order (steps of single rows have kernels of
// their own, outer_step and delta_step, where the size allows).  A column's dim elements are spread over 1, 2, 4 or 8 lanes, 32 to a lane in registers (so that several
// waves fit a SIMD and hide each other's waits); the lanes of a column add their parts of a read-out by shuffles.
// The vectors every lane needs (q_t, k_t, the decays) are prepared 16 tokens at a time in shared memory.
// Everything here is float.
#include "common.h"
#include "leone_hip.h"

#include <math.h>

#include <type_traits>

namespace leone {

constexpr int kScanTokens = 16;
constexpr int kLaneRows = 32;       // key channels a lane holds
constexpr int kScanThreads = 256;
constexpr int kLaneCols = 2;        // columns a lane holds in the outer-product scan: every q and k it reads serves both

// Over how many lanes a column of `dim` key channels is spread: 1, 2, 4 or 8 (dim up to 256).
inline int lane_groups(int dim) { return dim <= 32 ? 1 : dim <= 64 ? 2 : dim <= 128 ? 4 : 8; }

// A segment is a run of consecutive rows of one request that one wave walks in order: rows [first, end), the
// state it starts from (index `in` into the launch's input states, negative: zeros) and where the state it ends
// with goes (index `out` into the launch's output states, negative: nowhere).  A decoded token or a short portion
// is one segment from and into the request's state slot; long portions go through chunked_memory.hip.  What that does not take,
// the delta rule over more than 128 key channels, is cut into chunks that are walked side
// by side, three launches instead of one: every chunk from zeros (what the chunk's own rows write, and what they
// read of it), then the chunks' end states chained into the state each chunk starts from (delta_chain), then every
// chunk once more from that state with nothing written into it (`no_input`), added to the first walk's read-outs.
struct Segment {
    int first, end, in, out;
};

struct OuterScanArgs {
    const float* proj;          // [rows, stride]
    long stride;
    int q_off, k_off, v_off;    // columns of head 0; head h of q and k at + h * dim, of v at + h * vdim
    const float* coef;          // [rows, heads, 2]: a_t and b_t, or null: a = decay[head], b = 1
    const float* decay;         // [heads]
    int norm_column;            // one more column whose value is always 1 (the normaliser), read out into dot
    float q_scale, k_scale;
    int silu;                   // q, k and v pass through silu first
    const float* cos_table;     // [table_positions, rot_half] or null
    const float* sin_table;
    int rot_half, table_positions;
    const int* positions;
    const Segment* segments;
    const float* state_in;      // [index, heads, head_stride]
    long in_stride;
    float* state_out;
    long out_stride;
    long head_stride;           // floats from head to head in a state: S [dim, vdim], then the normaliser [dim]
    float* out;                 // [rows, heads, vdim]
    float* dot;                 // [rows, heads]
    int heads, dim, vdim;
};

// outer_step with exponential gates, made where they are used, in place of coef and decay.  (Arguments and kernels of their own: as a run-time
// question they cost a step without them up to 6 %.)
struct GatedStepArgs : OuterScanArgs {
    AnyVec i_bias, f_bias;      // [heads]
    int i_off, f_off;           // the first columns of their pre-activations in a row of proj
    float cap;
    long top_at;                // the running maximum's place in a head's state, which is read; the new one goes to top
    float* top;                 // [rows, heads]
};

__device__ inline float silu_if(float x, int silu) { return silu ? x / (1.0f + expf(-x)) : x; }

__device__ inline float rotated(const float* src, int i, int silu, const float* cos_row, const float* sin_row, int rot_half) {
    const float x = silu_if(src[i], silu);
    if (!cos_row || i >= 2 * rot_half) return x;
    if (i < rot_half) return x * cos_row[i] - silu_if(src[i + rot_half], silu) * sin_row[i];
    return x * cos_row[i - rot_half] + silu_if(src[i - rot_half], silu) * sin_row[i - rot_half];
}

__device__ inline float soft_cap_f(float z, float cap) { return cap * tanhf(z / cap); }
__device__ inline float log_sigmoid_f(float z) { return z >= 0.f ? -log1pf(expf(-z)) : z - log1pf(expf(z)); }

// The exponential gates of an entry's rows, a workgroup per (entry, head): log gates i_t = soft_cap(pre_i + bias_i),
// f_t = logsigmoid(soft_cap(pre_f + bias_f)); running maximum m_t = max(f_t + m_(t-1), i_t) from the request's
// state (0 at a sequence's start); a_t = exp(f_t + m_(t-1) - m_t), b_t = exp(i_t - m_t).  coef[row, head] = (a, b),
// top[row, head] = m_t; the last m goes back into the state.
// m -> max(A + m, B) is what a row does to the maximum; rows compose as (A2, B2) after (A1, B1) = (A1 + A2, max(A2 + B1, B2)), so a
// wave walks 64 rows by a prefix scan over its lanes, the waves side by side, and what they do to the maximum is then taken in the
// waves' order.  A portion is bound by one workgroup's chain of trips to memory a head: as many rows a trip as a workgroup may have
// threads, the next trip's rows asked for ahead of this one's scan.  2,048 rows of 4 heads: 10.4 us (28.2 with one wave scanning the
// 256 rows of a trip).
//
// How many threads, by the longest entry's rows: as many waves as it has 64 rows, which scan side by side, and up to 1,024 threads
// while every workgroup has a compute unit of its own.  More workgroups share units with each other, and threads without rows hold
// them up (us with 64, 256, 512 and 1,024 threads): one portion of 2,000 rows beside 8 single ones, 16 heads 41, 15.2, 11.9, 10.4, beside 63
// 40, 22.9, 18.7, 25.6; beside 128, 32 heads 43, 19.1, 21.3, 42; 64 entries of 2 rows, 16 heads 3.7, 3.9, 5.6, 9.7; one of 128 rows 4.7, 3.7,
// 3.8, 3.9.
constexpr int kGateUnits = 256;
__host__ inline int gate_threads(int longest, long groups) {
    if (longest <= kWave) return kWave;
    if (longest <= 256 || groups > 8 * kGateUnits) return 256;
    return groups > kGateUnits ? 512 : 1024;
}
template <int kThreads>
__global__ void __launch_bounds__(kThreads)
exp_gates_kernel(const float* __restrict__ proj, long stride, int i_off, int f_off, AnyVec i_bias, AnyVec f_bias, float cap,
                 const int* __restrict__ spans, float* __restrict__ state, long slot_stride, long head_stride, long top_at,
                 int write_state, float* __restrict__ coef, float* __restrict__ top, int heads) {
    constexpr int kWaves = kThreads / kWave;
    __shared__ float2 done[2][kWaves];              // what every wave's rows do to the maximum
    const int e = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int first = spans[4 * e], end = spans[4 * e + 1], in = spans[4 * e + 2], out = spans[4 * e + 3];
    float m = in < 0 ? 0.f : state[in * slot_stride + head * head_stride + top_at];
    const float bi = load_any(i_bias, head), bf = load_any(f_bias, head);
    float raw_i = 0.f, raw_f = 0.f;
    const auto fetch = [&](int r) {
        const float* base = proj + static_cast<long>(r < end ? r : end - 1) * stride;
        raw_i = base[i_off + head];
        raw_f = base[f_off + head];
    };
    if (first < end) fetch(first + tid);             // (an entry without rows has no last row to take instead)
    for (int r0 = first, turn = 0; r0 < end; r0 += kThreads, turn ^= 1) {
        const int r = r0 + tid;
        float li = -INFINITY, lf = 0.f;
        if (r < end) {
            li = soft_cap_f(raw_i + bi, cap);
            lf = log_sigmoid_f(soft_cap_f(raw_f + bf, cap));
        }
        if (r0 + kThreads < end) fetch(r + kThreads);
        float A = lf, B = li;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const float Ap = __shfl_up(A, off, kWave), Bp = __shfl_up(B, off, kWave);
            if (lane >= off) {
                B = fmaxf(A + Bp, B);
                A = A + Ap;
            }
        }
        float before = m;                           // the maximum ahead of this wave's rows
        const int last_lane = min(kWave - 1, end - 1 - (r0 + wave * kWave));
        if constexpr (kWaves > 1) {
            if (lane == last_lane) done[turn][wave] = float2{A, B};
            __syncthreads();                        // (the other turn's places were read before the barrier of the trip between)
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                if (w == wave) before = m;
                if (r0 + w * kWave < end) m = fmaxf(done[turn][w].x + m, done[turn][w].y);
            }
        }
        const float mine_m = fmaxf(A + before, B);
        float last = __shfl_up(mine_m, 1, kWave);
        if (lane == 0) last = before;
        if (r < end) {
            const long at = static_cast<long>(r) * heads + head;
            coef[2 * at] = expf(lf + last - mine_m);
            coef[2 * at + 1] = expf(li - mine_m);
            top[at] = mine_m;
        }
        if constexpr (kWaves == 1) m = __shfl(mine_m, last_lane, kWave);
    }
    if (write_state && out >= 0 && tid == 0) state[out * slot_stride + head * head_stride + top_at] = m;
}

__global__ void __launch_bounds__(kScanThreads) outer_scan_kernel(OuterScanArgs p, int groups) {
    extern __shared__ __align__(16) float scan_lds[];
    const int dkp = groups * kLaneRows;
    float* sq = scan_lds;                       // [kScanTokens][dkp]
    float* sk = sq + kScanTokens * dkp;
    float* sa = sk + kScanTokens * dkp;         // [kScanTokens]
    float* sb = sa + kScanTokens;
    const int head = blockIdx.y, tid = threadIdx.x, lane = tid % kWave;
    const Segment seg = p.segments[blockIdx.x];
    const int per_wave = kWave / groups;                       // lanes a wave has for columns; each holds kLaneCols of them
    const int part = lane / per_wave;                          // which 32 key channels of its columns this lane holds
    const int cols = p.vdim + (p.norm_column ? 1 : 0);
    int col[kLaneCols];
    bool is_value[kLaneCols], is_norm[kLaneCols];
#pragma unroll
    for (int c = 0; c < kLaneCols; ++c) {
        col[c] = ((blockIdx.z * (kScanThreads / kWave) + tid / kWave) * kLaneCols + c) * per_wave + lane % per_wave;
        is_value[c] = col[c] < p.vdim;
        is_norm[c] = p.norm_column && col[c] == p.vdim;
    }
    const int first = seg.first, n = seg.end - seg.first;
    const int ch0 = part * kLaneRows;
    const float* from = seg.in < 0 ? nullptr : p.state_in + seg.in * p.in_stride + head * p.head_stride;

    float S[kLaneCols][kLaneRows];
#pragma unroll
    for (int c = 0; c < kLaneCols; ++c) {
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i) {
            float v = 0.f;
            if (from && ch0 + i < p.dim) {
                if (is_value[c]) v = from[static_cast<long>(ch0 + i) * p.vdim + col[c]];
                else if (is_norm[c]) v = from[static_cast<long>(p.dim) * p.vdim + ch0 + i];
            }
            S[c][i] = v;
        }
    }
    const float fixed = p.coef ? 0.f : p.decay[head];

    for (int t0 = 0; t0 < n; t0 += kScanTokens) {
        const int here = min(kScanTokens, n - t0);
        for (int idx = tid; idx < here * dkp; idx += kScanThreads) {
            const int t = idx / dkp, i = idx % dkp;
            const long row = first + t0 + t;
            float qv = 0.f, kv = 0.f;
            if (i < p.dim) {
                const int pos = min(p.positions[row], p.table_positions - 1);
                const float* c = p.cos_table ? p.cos_table + static_cast<long>(pos) * p.rot_half : nullptr;
                const float* s = p.cos_table ? p.sin_table + static_cast<long>(pos) * p.rot_half : nullptr;
                const float* base = p.proj + row * p.stride;
                qv = rotated(base + p.q_off + head * p.dim, i, p.silu, c, s, p.rot_half) * p.q_scale;
                kv = rotated(base + p.k_off + head * p.dim, i, p.silu, c, s, p.rot_half) * p.k_scale;
            }
            sq[idx] = qv;
            sk[idx] = kv;
        }
        if (tid < here) {
            const long at = static_cast<long>(first + t0 + tid) * p.heads + head;
            sa[tid] = p.coef ? p.coef[2 * at] : fixed;
            sb[tid] = p.coef ? p.coef[2 * at + 1] : 1.f;
        }
        __syncthreads();
        if (col[0] < cols) {                                   // the lanes of a column are in or out together
            for (int t = 0; t < here; ++t) {
                const long row = first + t0 + t;
                const float a = sa[t];
                const float* kt = sk + t * dkp + ch0;
                const float* qt = sq + t * dkp + ch0;
                float acc[kLaneCols], bv[kLaneCols];
#pragma unroll
                for (int c = 0; c < kLaneCols; ++c) {
                    const float v = is_value[c] ? silu_if(p.proj[row * p.stride + p.v_off + head * p.vdim + col[c]], p.silu) : 1.f;
                    bv[c] = sb[t] * v;
                    acc[c] = 0.f;
                }
#pragma unroll
                for (int i = 0; i < kLaneRows; ++i) {
                    const float k = kt[i], q = qt[i];
#pragma unroll
                    for (int c = 0; c < kLaneCols; ++c) {
                        S[c][i] = fmaf(a, S[c][i], k * bv[c]);
                        acc[c] = fmaf(S[c][i], q, acc[c]);
                    }
                }
#pragma unroll
                for (int c = 0; c < kLaneCols; ++c) {
                    for (int off = per_wave; off < kWave; off <<= 1) acc[c] += __shfl_xor(acc[c], off, kWave);
                    if (part == 0 && col[c] < cols) {
                        const long at = row * p.heads + head;
                        *(is_value[c] ? p.out + at * p.vdim + col[c] : p.dot + at) = acc[c];
                    }
                }
            }
        }
        __syncthreads();
    }
    if (!p.state_out || seg.out < 0) return;
    float* to = p.state_out + seg.out * p.out_stride + head * p.head_stride;
#pragma unroll
    for (int c = 0; c < kLaneCols; ++c) {
        if (col[c] >= cols) continue;
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i) {
            if (ch0 + i < p.dim) {
                if (is_value[c]) to[static_cast<long>(ch0 + i) * p.vdim + col[c]] = S[c][i];
                else to[static_cast<long>(p.dim) * p.vdim + ch0 + i] = S[c][i];
            }
        }
    }
}

// The same for segments of single rows (decode steps), where the state's bytes in and out are the bound and the chain of trips to
// memory in front of them is what costs.  A workgroup takes 64 columns of a head, so that a wave's loads are whole lines of
// 256 bytes (the other kernel's are pieces of 32), and its waves take 32 key channels each; a row's q and k are made by
// the lanes of the wave that needs them.  A segment's row, gates, values and state are
// all asked for before the first is used.  The waves' sums meet in shared memory in the order in which the other kernel's
// lanes meet.  Eight rows of four heads of 256 x 512 with a normaliser: 9.6 us (18.3 walked).  Exponential gates are made here as well
// (eight rows of four heads: this launch 9.3 us and 10.7 with them, theirs was 4.9): every workgroup of a head reads the running maximum, so none of
// them may write the new one into the state; head_norm_gate, the next launch, does.
// The float at a wave's own row (in bytes from a base that all waves share) and a lane's own column: one base and one offset of 32
// bits a load, so that no row needs an address of its own.
__device__ inline const float& float_at(const float* base, unsigned row_bytes, unsigned col_bytes) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + (row_bytes + col_bytes));
}
__device__ inline float& float_at(float* base, unsigned row_bytes, unsigned col_bytes) {
    return *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + (row_bytes + col_bytes));
}

template <int kGroups>
__device__ inline float sum_groups(const float* of, int stride) {
    float v[kGroups];
#pragma unroll
    for (int g = 0; g < kGroups; ++g) v[g] = of[g * stride];
#pragma unroll
    for (int step = 1; step < kGroups; step <<= 1)
#pragma unroll
        for (int g = 0; g + step < kGroups; g += 2 * step) v[g] += v[g + step];
    return v[0];
}

// x turned by its row's angle, from loads that are already under way
struct Turned {
    float own, other, c, s;
};
__device__ inline float turn(const Turned& t, int i, int silu, int rot_half) {
    const float x = silu_if(t.own, silu);
    if (i >= 2 * rot_half) return x;
    return i < rot_half ? x * t.c - silu_if(t.other, silu) * t.s : x * t.c + silu_if(t.other, silu) * t.s;
}

template <int kGroups, bool kGated>
__global__ void __launch_bounds__(kGroups * kWave) outer_step_kernel(std::conditional_t<kGated, GatedStepArgs, OuterScanArgs> p) {
    __shared__ float sums[2][kGroups][kWave + 1];             // the columns' shares; one more for the normaliser's
    __shared__ __align__(16) float2 skq[kGroups][kLaneRows];  // a wave's own k and q
    __shared__ float snorm[kGroups][kLaneRows];
    const int head = blockIdx.y, tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);      // one for all lanes: the state's rows have one address a wave
    const Segment seg = p.segments[blockIdx.x];
    const int first = seg.first, n = seg.end - seg.first;
    const int ch0 = wave * kLaneRows;
    const int col = blockIdx.z * kWave + lane;
    const int ccol = min(col, p.vdim - 1);
    const unsigned row_bytes = 4u * p.vdim;
    const bool norm = p.norm_column && blockIdx.z == 0;
    const int ch = ch0 + lane % kLaneRows;                    // the channel whose q, k and normaliser this lane holds
    const int half = p.rot_half;
    const int other = ch < half ? ch + half : ch < 2 * half ? ch - half : ch;
    const int turned = ch < half ? ch : ch < 2 * half ? ch - half : 0;
    const float* from = seg.in < 0 ? nullptr : p.state_in + seg.in * p.in_stride + head * p.head_stride;
    float S[kLaneRows], N = 0.f;
    [[maybe_unused]] float fixed = 0.f, m = 0.f, bi = 0.f, bf = 0.f;
    if constexpr (!kGated) {
        fixed = p.coef ? 0.f : p.decay[head];
    } else {
        m = from ? from[p.top_at] : 0.f;
        bi = load_any(p.i_bias, head);
        bf = load_any(p.f_bias, head);
    }
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i) S[i] = 0.f;

    for (int t = 0; t < n; ++t) {
        const long row = first + t;
        const float* base = p.proj + row * p.stride;
        const float* qs = base + p.q_off + head * p.dim;
        const float* ks = base + p.k_off + head * p.dim;
        int pos = 0;
        if (p.cos_table) pos = p.positions[row];
        Turned q{qs[ch], qs[other], 1.f, 0.f}, k{ks[ch], ks[other], 1.f, 0.f};
        const float v_raw = base[p.v_off + head * p.vdim + ccol];
        const long at = row * p.heads + head;
        float a = fixed, b = 1.f;
        [[maybe_unused]] float raw_i = 0.f, raw_f = 0.f;
        if constexpr (!kGated) {
            if (p.coef) {
                a = p.coef[2 * at];
                b = p.coef[2 * at + 1];
            }
        } else {
            raw_i = base[p.i_off + head];
            raw_f = base[p.f_off + head];
        }
        if (p.cos_table) {
            const long angle = static_cast<long>(min(pos, p.table_positions - 1)) * half + turned;
            q.c = k.c = p.cos_table[angle];
            q.s = k.s = p.sin_table[angle];
        }
        if (t == 0 && from) {
#pragma unroll
            for (int i = 0; i < kLaneRows; ++i) S[i] = float_at(from, (ch0 + i) * row_bytes, 4u * ccol);
            if (norm) N = from[static_cast<long>(p.dim) * p.vdim + ch];
        }
        if constexpr (kGated) {                                // as exp_gates_kernel makes them, to the bit: no product joins a sum
#pragma clang fp contract(off)
            const float li = soft_cap_f(raw_i + bi, p.cap), lf = log_sigmoid_f(soft_cap_f(raw_f + bf, p.cap));
            const float next = fmaxf(lf + m, li);
            a = expf(lf + m - next);
            b = expf(li - next);
            m = next;
            if (blockIdx.z == 0 && tid == 0) p.top[at] = m;
        }
        const float qv = turn(q, ch, p.silu, half) * p.q_scale;
        const float kv = turn(k, ch, p.silu, half) * p.k_scale;
        const float bv = b * silu_if(v_raw, p.silu);
        if (lane < kLaneRows) skq[wave][lane] = float2{kv, qv};
        if (norm) {
            N = fmaf(a, N, kv * b);
            if (lane < kLaneRows) snorm[wave][lane] = N;
        }
        __syncthreads();
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i) {
            const float2 kq = skq[wave][i];
            S[i] = fmaf(a, S[i], kq.x * bv);
            acc = fmaf(S[i], kq.y, acc);
        }
        float (*to)[kWave + 1] = sums[t & 1];                  // read behind one barrier, written again behind the next
        to[wave][lane] = acc;
        if (norm) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < kLaneRows; ++i) sum = fmaf(snorm[wave][i], skq[wave][i].y, sum);
            if (lane == 0) to[wave][kWave] = sum;
        }
        __syncthreads();
        if (wave == 0 && col < p.vdim) p.out[at * p.vdim + col] = sum_groups<kGroups>(&to[0][lane], kWave + 1);
        if (norm && tid == kGroups * kWave - 1) p.dot[at] = sum_groups<kGroups>(&to[0][kWave], kWave + 1);
    }
    if (!p.state_out || seg.out < 0 || n <= 0) return;         // (a segment without rows leaves its state as it is)
    float* into = p.state_out + seg.out * p.out_stride + head * p.head_stride;
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i)
        if (col < p.vdim) float_at(into, (ch0 + i) * row_bytes, 4u * ccol) = S[i];
    if (norm && lane < kLaneRows) into[static_cast<long>(p.dim) * p.vdim + ch] = N;
}

struct DeltaScanArgs {
    const float* qkv;           // [rows, stride]: q and k heads (kv_heads x dim each), then v heads (heads x vdim)
    long stride;
    int q_off, k_off, v_off;
    const float* beta;          // [rows, beta_stride]: pre-activation of the write strength, one a head
    long beta_stride;
    const float* step;          // [rows, step_stride]: pre-activation of the step size, heads x dim, or one a head
    long step_stride;
    int per_head;               // one step size, and so one decay, a head
    AnyVec rate_log;            // [heads]: decay = exp(-exp(rate_log) * softplus(step + step_bias))
    AnyVec step_bias;           // [heads * dim], per_head: [heads]
    float q_scale, unit_eps;
    int no_input;               // v is taken as 0: what a state carries through the rows, and what is read of it
    int accumulate;             // read-outs are added to what out holds
    const Segment* segments;
    const float* state_in;      // [index, heads, dim, vdim]
    long in_stride;
    float* state_out;
    long out_stride;
    float* transition;          // [segments, heads, dim, dim] or null: what the segment's rows do to a state that comes
                                // in, as a matrix: dim more columns that start as the unit vectors and are given v = 0;
                                // stored [unit vector j][channel i], the order in which the chain reads it
    float* out;                 // [rows, heads, vdim]
    int heads, kv_heads, dim, vdim;
};

__device__ inline float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }

__global__ void __launch_bounds__(kScanThreads) delta_scan_kernel(DeltaScanArgs p, int groups) {
    extern __shared__ __align__(16) float scan_lds[];
    const int dkp = groups * kLaneRows;
    float* sq = scan_lds;                       // [kScanTokens][dkp] each
    float* sk = sq + kScanTokens * dkp;
    float* sg = sk + kScanTokens * dkp;
    float* sbeta = sg + kScanTokens * dkp;      // [kScanTokens]
    const int head = blockIdx.y, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const Segment seg = p.segments[blockIdx.x];
    const int kvh = head / (p.heads / p.kv_heads);
    const int per_wave = kWave / groups;
    const int part = lane / per_wave;
    const int col = (blockIdx.z * (kScanThreads / kWave) + wave) * per_wave + lane % per_wave;
    const bool is_value = col < p.vdim;
    const int unit = (p.transition && !is_value && col < p.vdim + p.dim) ? col - p.vdim : -1;   // a unit vector's column
    const bool live = is_value || unit >= 0;
    const int ch0 = part * kLaneRows;
    const int first = seg.first, n = seg.end - seg.first;
    const long head_size = static_cast<long>(p.dim) * p.vdim;
    const float* from = seg.in < 0 ? nullptr : p.state_in + seg.in * p.in_stride + head * head_size;
    const float rate = expf(load_any(p.rate_log, head));

    float S[kLaneRows];
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i) {
        float v = 0.f;
        if (is_value && from && ch0 + i < p.dim) v = from[static_cast<long>(ch0 + i) * p.vdim + col];
        if (unit >= 0 && ch0 + i == unit) v = 1.f;
        S[i] = v;
    }

    for (int t0 = 0; t0 < n; t0 += kScanTokens) {
        const int here = min(kScanTokens, n - t0);
        {   // sixteen lanes prepare a row's vectors, all rows of the chunk at once
            constexpr int kRowLanes = kScanThreads / kScanTokens;
            const int t = tid / kRowLanes, sub = tid % kRowLanes;
            if (t < here) {
                const long row = first + t0 + t;
                const float* base = p.qkv + row * p.stride;
                const float* qs = base + p.q_off + kvh * p.dim;
                const float* ks = base + p.k_off + kvh * p.dim;
                float qq = 0.f, kk = 0.f;
                for (int i = sub; i < p.dim; i += kRowLanes) {
                    qq = fmaf(qs[i], qs[i], qq);
                    kk = fmaf(ks[i], ks[i], kk);
                }
                // (on a chunk's last rows only some of the lanes are here, whole rows of 16 of them)
                static_assert(kRowLanes <= 16 && 16 % kRowLanes == 0, "a row's lanes meet within a row of 16 lanes");
                qq = add_span<kRowLanes>(qq);
                kk = add_span<kRowLanes>(kk);
                const float qinv = p.q_scale / sqrtf(qq + p.unit_eps);
                const float kinv = 1.0f / sqrtf(kk + p.unit_eps);
                const float head_decay = p.per_head
                    ? expf(-rate * softplus_f(p.step[row * p.step_stride + head] + load_any(p.step_bias, head))) : 1.f;
                for (int i = sub; i < dkp; i += kRowLanes) {
                    const bool in = i < p.dim;
                    sq[t * dkp + i] = in ? qs[i] * qinv : 0.f;
                    sk[t * dkp + i] = in ? ks[i] * kinv : 0.f;
                    const long ch = static_cast<long>(head) * p.dim + i;
                    if (p.per_head) sg[t * dkp + i] = head_decay;
                    else sg[t * dkp + i] = in ? expf(-rate * softplus_f(p.step[row * p.step_stride + ch] + load_any(p.step_bias, ch))) : 1.f;
                }
                if (sub == 0) sbeta[t] = 1.0f / (1.0f + expf(-p.beta[row * p.beta_stride + head]));
            }
        }
        __syncthreads();
        if (live) {                                            // the lanes of a column are in or out together
            for (int t = 0; t < here; ++t) {
                const long row = first + t0 + t;
                const float v = (is_value && !p.no_input) ? p.qkv[row * p.stride + p.v_off + head * p.vdim + col] : 0.f;
                const float* gt = sg + t * dkp + ch0;
                const float* kt = sk + t * dkp + ch0;
                const float* qt = sq + t * dkp + ch0;
                float seen = 0.f;
#pragma unroll
                for (int i = 0; i < kLaneRows; ++i) {
                    S[i] *= gt[i];
                    seen = fmaf(S[i], kt[i], seen);
                }
                for (int off = per_wave; off < kWave; off <<= 1) seen += __shfl_xor(seen, off, kWave);
                const float u = sbeta[t] * (v - seen);
                float acc = 0.f;
#pragma unroll
                for (int i = 0; i < kLaneRows; ++i) {
                    S[i] = fmaf(kt[i], u, S[i]);
                    acc = fmaf(S[i], qt[i], acc);
                }
                for (int off = per_wave; off < kWave; off <<= 1) acc += __shfl_xor(acc, off, kWave);
                if (part == 0 && is_value) {
                    float* dst = p.out + (row * p.heads + head) * p.vdim + col;
                    *dst = p.accumulate ? *dst + acc : acc;
                }
            }
        }
        __syncthreads();
    }
    if (unit >= 0) {
        float* to = p.transition + (static_cast<long>(blockIdx.x) * p.heads + head) * p.dim * p.dim;
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i)
            if (ch0 + i < p.dim) to[static_cast<long>(unit) * p.dim + ch0 + i] = S[i];
        return;
    }
    if (!p.state_out || seg.out < 0 || !is_value) return;
    float* to = p.state_out + seg.out * p.out_stride + head * head_size;
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i)
        if (ch0 + i < p.dim) to[static_cast<long>(ch0 + i) * p.vdim + col] = S[i];
}

// The same for segments of single rows (decode steps), split as in outer_step_kernel: 64 columns of a head a workgroup, 32 key
// channels a wave, everything asked for before the first use.  Eight rows of 16 heads of 128 x 128: 8.9 us (14.5 walked).
template <int kGroups>
__global__ void __launch_bounds__(kGroups * kWave) delta_step_kernel(DeltaScanArgs p) {
    constexpr int kRowLanes = kScanThreads / kScanTokens;     // lanes that share a row's sums of squares, as in the other kernel
    constexpr int kOwn = kGroups * kLaneRows / kRowLanes;
    __shared__ float saw[kGroups][kWave], sums[kGroups][kWave];
    __shared__ float4 sgkq[kGroups][kLaneRows];               // a wave's own decays, k and q
    const int head = blockIdx.y, tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const Segment seg = p.segments[blockIdx.x];
    const int first = seg.first, n = seg.end - seg.first;
    const int kvh = head / (p.heads / p.kv_heads);
    const int ch0 = wave * kLaneRows;
    const int col = blockIdx.z * kWave + lane;
    const int ccol = min(col, p.vdim - 1);
    const unsigned row_bytes = 4u * p.vdim;
    const int ch = ch0 + lane % kLaneRows;
    const long head_size = static_cast<long>(p.dim) * p.vdim;
    const float* from = seg.in < 0 ? nullptr : p.state_in + seg.in * p.in_stride + head * head_size;
    const long step_at = p.per_head ? head : static_cast<long>(head) * p.dim + ch;
    float S[kLaneRows];
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i) S[i] = 0.f;

    for (int t = 0; t < n; ++t) {
        const long row = first + t;
        const float* base = p.qkv + row * p.stride;
        const float* qs = base + p.q_off + kvh * p.dim;
        const float* ks = base + p.k_off + kvh * p.dim;
        float qr[kOwn], kr[kOwn];
#pragma unroll
        for (int m = 0; m < kOwn; ++m) {
            qr[m] = qs[lane % kRowLanes + m * kRowLanes];
            kr[m] = ks[lane % kRowLanes + m * kRowLanes];
        }
        const float q_raw = qs[ch], k_raw = ks[ch];
        const float v = base[p.v_off + head * p.vdim + ccol];
        const float step_raw = p.step[row * p.step_stride + step_at], beta_raw = p.beta[row * p.beta_stride + head];
        if (t == 0 && from) {
#pragma unroll
            for (int i = 0; i < kLaneRows; ++i) S[i] = float_at(from, (ch0 + i) * row_bytes, 4u * ccol);
        }
        const float rate = expf(load_any(p.rate_log, head)), bias = load_any(p.step_bias, step_at);
        float qq = 0.f, kk = 0.f;
#pragma unroll
        for (int m = 0; m < kOwn; ++m) {
            qq = fmaf(qr[m], qr[m], qq);
            kk = fmaf(kr[m], kr[m], kk);
        }
        qq = add_span<kRowLanes>(qq);
        kk = add_span<kRowLanes>(kk);
        const float qinv = p.q_scale / sqrtf(qq + p.unit_eps);
        const float kinv = 1.0f / sqrtf(kk + p.unit_eps);
        const float gv = expf(-rate * softplus_f(step_raw + bias));
        if (lane < kLaneRows) sgkq[wave][lane] = float4{gv, k_raw * kinv, q_raw * qinv, 0.f};
        __syncthreads();
        const float strength = 1.0f / (1.0f + expf(-beta_raw));
        float seen = 0.f;
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i) {
            const float4 gkq = sgkq[wave][i];
            S[i] *= gkq.x;
            seen = fmaf(S[i], gkq.y, seen);
        }
        saw[wave][lane] = seen;                                // last read ahead of the barrier that the row before ended with
        __syncthreads();
        const float u = strength * (v - sum_groups<kGroups>(&saw[0][lane], kWave));
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i) {
            const float4 gkq = sgkq[wave][i];
            S[i] = fmaf(gkq.y, u, S[i]);
            acc = fmaf(S[i], gkq.z, acc);
        }
        sums[wave][lane] = acc;
        __syncthreads();
        if (wave == 0 && col < p.vdim) p.out[(row * p.heads + head) * p.vdim + col] = sum_groups<kGroups>(&sums[0][lane], kWave);
    }
    if (!p.state_out || seg.out < 0 || n <= 0 || col >= p.vdim) return;
    float* to = p.state_out + seg.out * p.out_stride + head * head_size;
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i)
        float_at(to, (ch0 + i) * row_bytes, 4u * ccol) = S[i];
}

// The chunks of a long portion chained for the delta rule, its chunks [g0, g1) of `work`: a chunk's rows turn a state S that comes
// in into transition[chunk] . S + (what the chunk holds: its end state from zeros).  From the request's state on (zeros at a
// sequence's start) every chunk's place in `work` ends up holding the state the chunk starts from, and the last state is the
// request's new one.  links[l] = (slot, fresh, g0, g1).
// A workgroup owns a run of columns of one head; a column's channels are spread over lanes as in the scans, and
// the whole column passes through shared memory so that every lane sees all of it.
__global__ void __launch_bounds__(kScanThreads)
delta_chain_kernel(const int* __restrict__ links, float* __restrict__ work, long work_stride, const float* __restrict__ transition,
                   float* __restrict__ state, long slot_stride, int heads, int dim, int vdim, int groups, int tile, int write_state) {
    extern __shared__ __align__(16) float chain_lds[];
    const int dkp = groups * kLaneRows;
    const int l = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int per_wave = kWave / groups, per_block = (kScanThreads / kWave) * per_wave;
    float* sS = chain_lds;                      // [dkp][columns a workgroup]: the state that comes in
    float* sT = chain_lds + dkp * per_block;    // [tile][dkp]: `tile` columns of the transition, turned
    const int part = lane / per_wave, local = wave * per_wave + lane % per_wave;
    const int col = blockIdx.z * per_block + local;
    const bool live = col < vdim;
    const int ch0 = part * kLaneRows;
    const int slot = links[4 * l], fresh = links[4 * l + 1], g0 = links[4 * l + 2], g1 = links[4 * l + 3];
    const long head_size = static_cast<long>(dim) * vdim;
    float* mine = state + slot * slot_stride + head * head_size;
    float S[kLaneRows];
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i)
        S[i] = (!fresh && live && ch0 + i < dim) ? mine[static_cast<long>(ch0 + i) * vdim + col] : 0.f;
    for (int g = g0; g < g1; ++g) {
        float* held = work + g * work_stride + head * head_size;
        const float* T = transition + (static_cast<long>(g) * heads + head) * dim * dim;
        float next[kLaneRows];
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i) {
            const bool in = live && ch0 + i < dim;
            next[i] = in ? held[static_cast<long>(ch0 + i) * vdim + col] : 0.f;
            if (in) held[static_cast<long>(ch0 + i) * vdim + col] = S[i];
            sS[(ch0 + i) * per_block + local] = S[i];
        }
        for (int j0 = 0; j0 < dim; j0 += tile) {
            __syncthreads();
            for (int idx = tid; idx < tile * dkp; idx += kScanThreads) {
                const int jj = idx / dkp, i = idx % dkp;
                sT[idx] = (i < dim && j0 + jj < dim) ? T[static_cast<long>(j0 + jj) * dim + i] : 0.f;
            }
            __syncthreads();
            const int width = min(tile, dim - j0);
            for (int jj = 0; jj < width; ++jj) {
                const float s = sS[(j0 + jj) * per_block + local];
                const float* column = sT + jj * dkp + ch0;
#pragma unroll
                for (int i = 0; i < kLaneRows; ++i) next[i] = fmaf(column[i], s, next[i]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kLaneRows; ++i) S[i] = next[i];
    }
    if (!write_state || !live) return;
#pragma unroll
    for (int i = 0; i < kLaneRows; ++i)
        if (ch0 + i < dim) mine[static_cast<long>(ch0 + i) * vdim + col] = S[i];
}

static bool known_vec(int dtype) { return dtype == kF32 || dtype == kBF16; }

}  // namespace leone

using namespace leone;

extern "C" int leone_scan_max_dim() { return 256; }
extern "C" int leone_exp_gates_threads(int longest, int entries, int heads) { return gate_threads(longest, static_cast<long>(entries) * heads); }

extern "C" int leone_exp_gates(const float* proj, long stride, int i_off, int f_off, const void* i_bias, const void* f_bias,
                               int bias_dtype, float cap, const int* spans, int entries, float* state, long slot_stride,
                               long head_stride, long top_at, int write_state, float* coef, float* top, int longest,
                               int heads, hipStream_t stream) {
    LEONE_REQUIRE(proj && i_bias && f_bias && spans && state && coef && top, "exp_gates: null pointer");
    LEONE_REQUIRE(known_vec(bias_dtype) && cap > 0.f, "exp_gates: unknown bias type or cap %g", cap);
    LEONE_REQUIRE(entries > 0 && longest > 0 && heads > 0 && heads <= 65535 && i_off >= 0 && f_off >= 0 && stride >= i_off + heads &&
                  stride >= f_off + heads, "exp_gates: %d entries, %d heads, rows of %ld", entries, heads, stride);
    LEONE_REQUIRE(top_at >= 0 && top_at < head_stride && slot_stride >= heads * head_stride, "exp_gates: the maximum's place %ld", top_at);
#define LEONE_GATES(THREADS)                                                                                                \
    exp_gates_kernel<THREADS><<<dim3(entries, heads), THREADS, 0, stream>>>(proj, stride, i_off, f_off, AnyVec{i_bias, bias_dtype}, \
                                                                            AnyVec{f_bias, bias_dtype}, cap, spans, state, slot_stride, \
                                                                            head_stride, top_at, write_state, coef, top, heads)
    switch (gate_threads(longest, static_cast<long>(entries) * heads)) {
        case kWave: LEONE_GATES(kWave); break;
        case 256: LEONE_GATES(256); break;
        case 512: LEONE_GATES(512); break;
        default: LEONE_GATES(1024); break;
    }
#undef LEONE_GATES
    LEONE_LAUNCH_CHECK("exp_gates");
    return 0;
}

// Whether heads of such sizes are taken by the kernels for single rows: waves of 32 key channels each, without a rest (of 1, 2, 4
// or 8 waves), offsets within a head's state of 32 bits.  Other heads are walked by the general kernels in single rows too.
extern "C" int leone_step_fits(int dim, int vdim) {
    return dim == lane_groups(dim) * kLaneRows && ceil_div(vdim, kWave) <= 65535 && static_cast<long>(dim) * vdim < (1L << 30);
}

static int run_outer_scan(bool single, const float* proj, long stride, int q_off, int k_off, int v_off, const float* coef,
                                const float* decay, int norm_column, float q_scale, float k_scale, int silu,
                                const float* cos_table, const float* sin_table, int rotary_dim, int table_positions,
                                const int* positions, const int* segments, int n_segments, const float* state_in,
                                long in_stride, float* state_out, long out_stride, long head_stride, float* out, float* dot,
                                int heads, int dim, int vdim, hipStream_t stream, const GatedStepArgs* gates = nullptr) {
    LEONE_REQUIRE(proj && positions && segments && out, "outer_scan: null pointer");
    LEONE_REQUIRE(n_segments > 0 && heads > 0 && heads <= 65535 && dim > 0 && vdim > 0, "outer_scan: %d segments, %d heads of %d x %d",
                  n_segments, heads, dim, vdim);
    LEONE_REQUIRE(dim <= leone_scan_max_dim(), "outer_scan: heads of %d key channels, the kernel takes up to %d", dim, leone_scan_max_dim());
    LEONE_REQUIRE(coef || decay || gates, "outer_scan: neither per-row coefficients nor a fixed decay");
    LEONE_REQUIRE(!norm_column || dot, "outer_scan: the normaliser's read-out needs a place");
    LEONE_REQUIRE((cos_table == nullptr) == (sin_table == nullptr), "outer_scan: cos and sin tables come together");
    LEONE_REQUIRE(!cos_table || (rotary_dim > 0 && rotary_dim % 2 == 0 && rotary_dim <= dim && table_positions > 0),
                  "outer_scan: rotary_dim %d must be even, positive and at most %d", rotary_dim, dim);
    const long per_head = static_cast<long>(dim) * vdim + (norm_column ? dim : 0);
    LEONE_REQUIRE(head_stride >= per_head && (!state_in || in_stride >= heads * head_stride) &&
                  (!state_out || out_stride >= heads * head_stride), "outer_scan: states of %ld floats a head do not fit", head_stride);
    LEONE_REQUIRE(stride >= q_off + heads * dim && stride >= k_off + heads * dim && stride >= v_off + heads * vdim &&
                  q_off >= 0 && k_off >= 0 && v_off >= 0, "outer_scan: the projection's rows of %ld do not hold the named columns", stride);
    OuterScanArgs a{proj, stride, q_off, k_off, v_off, coef, decay, norm_column, q_scale, k_scale,
                    silu, cos_table, sin_table, cos_table ? rotary_dim / 2 : 0, cos_table ? table_positions : 1, positions,
                    reinterpret_cast<const Segment*>(segments), state_in, in_stride, state_out, out_stride, head_stride,
                    out, dot, heads, dim, vdim};
    const int groups = lane_groups(dim);
    const int per_block = (kScanThreads / kWave) * (kWave / groups) * kLaneCols;          // columns a workgroup
    const dim3 grid(n_segments, heads, ceil_div(vdim + (norm_column ? 1 : 0), per_block));
    const size_t shared = (2 * kScanTokens * groups * kLaneRows + 2 * kScanTokens) * sizeof(float);
    if (single) {
        LEONE_REQUIRE(leone_step_fits(dim, vdim), "outer_step: heads have 32, 64, 128 or 256 key channels (not %d x %d)", dim, vdim);
        const dim3 columns(n_segments, heads, ceil_div(vdim, kWave));
        const auto launch = [&](auto gated, const auto& args) {
            constexpr bool kGated = decltype(gated)::value;
            if (groups == 1) outer_step_kernel<1, kGated><<<columns, kWave, 0, stream>>>(args);
            else if (groups == 2) outer_step_kernel<2, kGated><<<columns, 2 * kWave, 0, stream>>>(args);
            else if (groups == 4) outer_step_kernel<4, kGated><<<columns, 4 * kWave, 0, stream>>>(args);
            else outer_step_kernel<8, kGated><<<columns, 8 * kWave, 0, stream>>>(args);
        };
        if (gates) {
            GatedStepArgs with = *gates;
            static_cast<OuterScanArgs&>(with) = a;
            launch(std::true_type{}, with);
        } else {
            launch(std::false_type{}, a);
        }
        LEONE_LAUNCH_CHECK("outer_step");
        return 0;
    }
    outer_scan_kernel<<<grid, kScanThreads, shared, stream>>>(a, groups);
    LEONE_LAUNCH_CHECK("outer_scan");
    return 0;
}

extern "C" int leone_outer_scan(const float* proj, long stride, int q_off, int k_off, int v_off, const float* coef,
                                const float* decay, int norm_column, float q_scale, float k_scale, int silu,
                                const float* cos_table, const float* sin_table, int rotary_dim, int table_positions,
                                const int* positions, const int* segments, int n_segments, const float* state_in,
                                long in_stride, float* state_out, long out_stride, long head_stride, float* out, float* dot,
                                int heads, int dim, int vdim, hipStream_t stream) {
    return run_outer_scan(false, proj, stride, q_off, k_off, v_off, coef, decay, norm_column, q_scale, k_scale, silu, cos_table,
        sin_table, rotary_dim, table_positions, positions, segments, n_segments, state_in, in_stride, state_out, out_stride,
        head_stride, out, dot, heads, dim, vdim, stream);
}

// leone_outer_scan where every segment is a single row.
extern "C" int leone_outer_step(const float* proj, long stride, int q_off, int k_off, int v_off, const float* coef,
                                const float* decay, int norm_column, float q_scale, float k_scale, int silu,
                                const float* cos_table, const float* sin_table, int rotary_dim, int table_positions,
                                const int* positions, const int* segments, int n_segments, const float* state_in,
                                long in_stride, float* state_out, long out_stride, long head_stride, float* out, float* dot,
                                int heads, int dim, int vdim, hipStream_t stream) {
    return run_outer_scan(true, proj, stride, q_off, k_off, v_off, coef, decay, norm_column, q_scale, k_scale, silu, cos_table,
        sin_table, rotary_dim, table_positions, positions, segments, n_segments, state_in, in_stride, state_out, out_stride,
        head_stride, out, dot, heads, dim, vdim, stream);
}

// leone_outer_step with a normaliser and exponential gates made in the launch (what leone_exp_gates writes to coef and top, but the state's
// maximum stays as it is: leone_head_norm_gate_kept writes it).
extern "C" int leone_outer_step_gated(const float* proj, long stride, int q_off, int k_off, int v_off, int i_off, int f_off,
                                      const void* i_bias, const void* f_bias, int bias_dtype, float cap, long top_at, float* top,
                                      float q_scale, float k_scale, int silu, const float* cos_table, const float* sin_table, int rotary_dim,
                                      int table_positions, const int* positions, const int* segments, int n_segments, const float* state_in,
                                      long in_stride, float* state_out, long out_stride, long head_stride, float* out, float* dot, int heads,
                                      int dim, int vdim, hipStream_t stream) {
    LEONE_REQUIRE(i_bias && f_bias && top && state_in, "outer_step: the gates' operands are missing");
    LEONE_REQUIRE(known_vec(bias_dtype) && cap > 0.f, "outer_step: unknown bias type or cap %g", cap);
    LEONE_REQUIRE(i_off >= 0 && f_off >= 0 && stride >= i_off + heads && stride >= f_off + heads, "outer_step: rows of %ld do not hold the gates", stride);
    LEONE_REQUIRE(top_at >= 0 && top_at < head_stride, "outer_step: the maximum's place %ld", top_at);
    GatedStepArgs gates{};
    gates.i_bias = AnyVec{i_bias, bias_dtype}, gates.f_bias = AnyVec{f_bias, bias_dtype};
    gates.i_off = i_off, gates.f_off = f_off, gates.cap = cap, gates.top_at = top_at, gates.top = top;
    return run_outer_scan(true, proj, stride, q_off, k_off, v_off, nullptr, nullptr, 1, q_scale, k_scale, silu, cos_table,
        sin_table, rotary_dim, table_positions, positions, segments, n_segments, state_in, in_stride, state_out, out_stride,
        head_stride, out, dot, heads, dim, vdim, stream, &gates);
}

static int run_delta_scan(bool single, const float* qkv, long stride, int q_off, int k_off, int v_off, const float* beta,
                                long beta_stride, const float* step, long step_stride, int per_head, const void* rate_log,
                                const void* step_bias, int vec_dtype, float q_scale, float unit_eps, int no_input,
                                int accumulate, const int* segments, int n_segments, const float* state_in, long in_stride,
                                float* state_out, long out_stride, float* transition, float* out, int heads, int kv_heads,
                                int dim, int vdim, hipStream_t stream) {
    LEONE_REQUIRE(qkv && beta && step && rate_log && step_bias && segments && out, "delta_scan: null pointer");
    LEONE_REQUIRE(known_vec(vec_dtype), "delta_scan: unknown element type");
    LEONE_REQUIRE(n_segments > 0 && heads > 0 && heads <= 65535 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0,
                  "delta_scan: %d segments, %d heads over %d key heads of %d x %d", n_segments, heads, kv_heads, dim, vdim);
    LEONE_REQUIRE(dim <= leone_scan_max_dim(), "delta_scan: heads of %d key channels, the kernel takes up to %d", dim, leone_scan_max_dim());
    const long per_slot = static_cast<long>(heads) * dim * vdim;
    LEONE_REQUIRE((!state_in || in_stride >= per_slot) && (!state_out || out_stride >= per_slot),
                  "delta_scan: states of %ld floats do not fit", per_slot);
    LEONE_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && stride >= q_off + kv_heads * dim && stride >= k_off + kv_heads * dim &&
                  stride >= v_off + heads * vdim && beta_stride >= heads && step_stride >= static_cast<long>(heads) * (per_head ? 1 : dim),
                  "delta_scan: rows too short for the named columns");
    DeltaScanArgs a{qkv, stride, q_off, k_off, v_off, beta, beta_stride, step, step_stride, per_head, AnyVec{rate_log, vec_dtype},
                    AnyVec{step_bias, vec_dtype}, q_scale, unit_eps, no_input, accumulate,
                    reinterpret_cast<const Segment*>(segments), state_in, in_stride, state_out, out_stride, transition, out,
                    heads, kv_heads, dim, vdim};
    const int groups = lane_groups(dim);
    const dim3 grid(n_segments, heads, ceil_div(vdim + (transition ? dim : 0), (kScanThreads / kWave) * (kWave / groups)));
    const size_t shared = (3 * kScanTokens * groups * kLaneRows + kScanTokens) * sizeof(float);
    if (single) {
        LEONE_REQUIRE(leone_step_fits(dim, vdim), "delta_step: heads have 32, 64, 128 or 256 key channels (not %d x %d)", dim, vdim);
        const dim3 columns(n_segments, heads, ceil_div(vdim, kWave));
        if (groups == 1) delta_step_kernel<1><<<columns, kWave, 0, stream>>>(a);
        else if (groups == 2) delta_step_kernel<2><<<columns, 2 * kWave, 0, stream>>>(a);
        else if (groups == 4) delta_step_kernel<4><<<columns, 4 * kWave, 0, stream>>>(a);
        else delta_step_kernel<8><<<columns, 8 * kWave, 0, stream>>>(a);
        LEONE_LAUNCH_CHECK("delta_step");
        return 0;
    }
    delta_scan_kernel<<<grid, kScanThreads, shared, stream>>>(a, groups);
    LEONE_LAUNCH_CHECK("delta_scan");
    return 0;
}

extern "C" int leone_delta_scan(const float* qkv, long stride, int q_off, int k_off, int v_off, const float* beta,
                                long beta_stride, const float* step, long step_stride, int per_head, const void* rate_log,
                                const void* step_bias, int vec_dtype, float q_scale, float unit_eps, int no_input,
                                int accumulate, const int* segments, int n_segments, const float* state_in, long in_stride,
                                float* state_out, long out_stride, float* transition, float* out, int heads, int kv_heads,
                                int dim, int vdim, hipStream_t stream) {
    return run_delta_scan(false, qkv, stride, q_off, k_off, v_off, beta, beta_stride, step, step_stride, per_head,
        rate_log, step_bias, vec_dtype, q_scale, unit_eps, no_input, accumulate, segments, n_segments, state_in,
        in_stride, state_out, out_stride, transition, out, heads, kv_heads, dim, vdim, stream);
}

// leone_delta_scan where every segment is a single row.
extern "C" int leone_delta_step(const float* qkv, long stride, int q_off, int k_off, int v_off, const float* beta,
                                long beta_stride, const float* step, long step_stride, int per_head, const void* rate_log,
                                const void* step_bias, int vec_dtype, float q_scale, float unit_eps, const int* segments,
                                int n_segments, const float* state_in, long in_stride, float* state_out, long out_stride,
                                float* out, int heads, int kv_heads, int dim, int vdim, hipStream_t stream) {
    return run_delta_scan(true, qkv, stride, q_off, k_off, v_off, beta, beta_stride, step, step_stride, per_head,
        rate_log, step_bias, vec_dtype, q_scale, unit_eps, 0, 0, segments, n_segments, state_in,
        in_stride, state_out, out_stride, nullptr, out, heads, kv_heads, dim, vdim, stream);
}

extern "C" int leone_delta_chain(const int* links, int n_links, float* work, long work_stride, const float* transition,
                                 float* state, long slot_stride, int heads, int dim, int vdim, int write_state,
                                 hipStream_t stream) {
    LEONE_REQUIRE(links && work && transition && state && n_links > 0 && heads > 0 && heads <= 65535 && dim > 0 && vdim > 0,
                  "delta_chain: null pointer or empty sizes");
    LEONE_REQUIRE(dim <= leone_scan_max_dim(), "delta_chain: heads of %d key channels, the kernel takes up to %d", dim, leone_scan_max_dim());
    const long per_slot = static_cast<long>(heads) * dim * vdim;
    LEONE_REQUIRE(work_stride >= per_slot && slot_stride >= per_slot, "delta_chain: states of %ld floats do not fit", per_slot);
    const int groups = lane_groups(dim);
    const int per_block = (kScanThreads / kWave) * (kWave / groups);
    const int dkp = groups * kLaneRows;
    const int tile = 8192 / dkp;                                   // 32 KB of the transition at a time
    const size_t shared = static_cast<size_t>(dkp) * (per_block + tile) * sizeof(float);
    delta_chain_kernel<<<dim3(n_links, heads, ceil_div(vdim, per_block)), kScanThreads, shared, stream>>>(
        links, work, work_stride, transition, state, slot_stride, heads, dim, vdim, groups, tile, write_state);
    LEONE_LAUNCH_CHECK("delta_chain");
    return 0;
}
