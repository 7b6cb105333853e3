// Matrix memories over long portions, as products on the matrix cores (float throughout).
//
//   S_t = g_t S_(t-1) + k_t u_t^T,  o_t = S_t^T q_t                                       S is [dim, vdim]
//   fixed decays:   g a constant of the head, u_t = v_t
//   gates:          g_t and a factor b_t of a row and head, u_t = b_t v_t; the normaliser n_t = g_t n_(t-1) + b_t k_t is one
//                   more column of S, whose value is always 1
//   delta rule:     u_t = beta_t (v_t - (g_t S_(t-1))^T k_t), g_t one a head or one for every key channel
//
// Over a chunk of 64 rows, with L_t the product of the chunk's decays up to and with row t and S0 the state it starts from,
//   S_t = L_t S0 + sum_(i <= t) (L_t / L_i) k_i u_i^T,
// so with A_ti = beta_t (L_t / L_i) k_t.k_i (i < t) and M_ti = (L_t / L_i) q_t.k_i (i <= t), one row a token,
//   (1 + A) U = diag(beta) V - diag(beta L) K S0,   O = diag(L) Q S0 + M U,   S_end = L_end S0 + (diag(L_end / L) K)^T U.
// chunk_prepare makes everything that does not hold S0, all chunks and heads side by side: U0 and W, the solutions of the
// triangular system for diag(beta) V and diag(beta L) K (forward substitution, 16 rows at a time: the rows before leave them
// as products), M, and Q and K with their decays.  chunk_walk then goes through a portion's chunks in order, a workgroup a head
// and 16 columns of S: U = U0 - W S, O, S.  With fixed decays and gates there is no system: U = V or diag(b) V.
//
// With a decay for every key channel L_t and L_t / L_i are vectors, and the decays between two rows belong inside the dot
// products of their k and q.  chunk_prepare_channel makes them a tile of 16 x 16 rows at a time.  Between different tiles the
// decays from the end of the key's tile back to the key ride on the key, those from the start of the query's tile on the
// query, and the tiles between are a product of their own: every factor is a product of decays, so none is above 1 and none is
// made by a division.  Within a tile a lane takes a key's channels through the rows behind it, a decay at a time.
//
// Against the recurrences walked row by row in chunks side by side, three walks of every chunk or two and a product of
// matrices (us a layer of 2,048 rows, before): gates, 4 heads of 256 x 512 165 (566); fixed decays with rotation, 4 heads of
// 128 x 256 110 (250); a decay a channel, 16 heads of 128 x 128 241 (1034).
//
// A row's read-out holds nothing of the rows behind it, not even where those are infinite or not numbers, and a decay that is not
// a number makes the memory none from its row on, as the recurrences do row by row.
//
// Products are v_mfma_f32_16x16x4_f32.  Lane l = 16 g + c holds A[row c][k-slot g], B[k-slot g][column c] and rows 4 g + v of
// column c of the result in register v.  Which inner element a k-slot stands for is free as long as both operands agree:
// instruction v of a run of 16 takes element 4 g + v for slot g, so that an operand is one 16-byte read a lane, and a result
// in registers (S, U) is the next product's second operand as it lies.  Decays travel as logarithms summed over the chunk, in
// double: a row that forgets everything must not blur the small decays behind it.
#include "common.h"
#include "leone_hip.h"

#include <math.h>

namespace leone {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

constexpr int kChunkRows = 64;
constexpr int kChunkThreads = 256;
constexpr int kChunkMaxDim = 256;       // key channels: four tiles of 16 a wave
constexpr int kChunkMaxDeltaDim = 128;  // the delta rule holds twice as much of a chunk
constexpr int kChunkTiles = 10;         // tiles of 16 x 16 of a chunk's rows by rows on and below the diagonal
constexpr int kPartStride = 20;         // of a row of 16 in shared memory: rows four apart lie in banks of their own

struct ChunkArgs {
    const float* rows;          // [rows, stride]: q and k heads (kv_heads x dim each), v heads (heads x vdim)
    long stride;
    int q_off, k_off, v_off;
    int silu;                   // q, k and v pass through silu first
    float q_scale, k_scale;
    float unit_eps;             // delta rule: q and k are made unit vectors a head first, this under the root
    const float* beta;          // delta rule: [rows, beta_stride] pre-activation of the write strength, one a head
    long beta_stride;
    const float* step;          // delta rule: [rows, step_stride] pre-activation of the step size, one a head
    long step_stride;
    AnyVec rate_log, step_bias; // delta rule: [heads]; decay = exp(-exp(rate_log) * softplus(step + step_bias))
                                // (a decay for every channel: step [rows, >= heads * dim], step_bias [heads * dim])
    const float* decay;         // fixed decays: [heads]
    const float* coef;          // gates: [rows, heads, 2], g_t and b_t
    const float* cos_table;     // rotation of q and k: [table_positions, rot_half] or null
    const float* sin_table;
    const int* positions;
    int rot_half, table_positions;
    const int* chunks;          // [chunks, 4]: first row, end, -, -
    const int* links;           // [links, 4]: state slot, whether the sequence starts here, first chunk, end
    float* q_in;                // [chunks, heads, 64 x dim_p]: q_t L_t, in the order chunk_walk reads
    float* k_out;               // [chunks, heads, dim_p x 64]: k_t L_end / L_t, likewise
    float* mix;                 // [chunks, heads, 64 x 64]: M, likewise (tiles above the diagonal are not written)
    float* solved_k;            // delta rule: [chunks, heads, 64 x dim_p]: W, likewise
    float* values;              // [chunks, heads, 64, vdim_p]: U0, or V
    float* total;               // [chunks, heads]: L_end (a decay for every channel: [chunks, heads, dim_p])
    float* state;               // [slots, heads, head_stride]: [dim, vdim], then with gates the normaliser [dim]
    long slot_stride, head_stride;
    int write_state;
    float* out;                 // [rows, heads, vdim]
    float* dot;                 // gates: [rows, heads], the normaliser's read-out; else null
    int heads, kv_heads, dim, vdim, dim_p, vdim_p;      // _p: filled up to whole tiles (vdim_p: with the normaliser's column)
};

__device__ inline float chunk_act(float x, int silu) { return silu ? x / (1.0f + expf(-x)) : x; }
__device__ inline float chunk_softplus(float z) { return z > 20.f ? z : log1pf(expf(z)); }
constexpr float kNothingLeft = -1e4f;   // a logarithm whose exponential is zero and of which 64 add up without overflow
// exp(later - earlier), the difference's rounding to float made good (an exponential in double took a chunk's tiles 0.4 us longer;
// read-outs and states are as far from 64 bits either way).
__device__ inline float between(double later, double earlier) {
    const double of = later - earlier;
    const float rounded = static_cast<float>(of), result = expf(rounded);
    return result == INFINITY ? result : fmaf(result, static_cast<float>(of - rounded), result);
}
__device__ inline float element(const float4& f, int v) { return v == 0 ? f.x : v == 1 ? f.y : v == 2 ? f.z : f.w; }
__device__ inline floatx4 mfma4(float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Where the four elements that a lane of chunk_walk reads at once stand in the chunk's rows: its operands lie in the order of
// [wave][tile of rows][tile of channels][lane], so that a wave reads 1,024 bytes in a row.
struct Place { int row, channel; };
template <int kT>
__device__ inline Place place_of(int idx) {
    const int lane = idx % kWave, tile = idx / kWave;
    return {16 * (tile / kT % 4) + (lane & 15), 16 * (tile / (4 * kT) * kT + tile % kT) + 4 * (lane >> 4)};
}

// The triangular system solved for a chunk's right sides, in their place: a block of value columns in sq, the keys in sk (rows
// of kDim + 4), sa -A in tiles.  The solved values go to `values` (columns `block` ..), the solved keys to `solved_k` (null:
// another workgroup stores them).
template <int kT>
__device__ inline void solve_chunk(float* sq, float* sk, const float* sa, float* values, int vdim_p, int block, float* solved_k) {
    constexpr int kDim = 64 * kT, row_p = kDim + 4;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, c = lane & 15, g = lane >> 4;
    static_assert(2 * kDim <= kChunkThreads, "a thread takes one column");
    const bool is_key = tid >= kDim;
    const int mine = is_key ? tid - kDim : tid;
    float* column = (is_key ? sk : sq) + mine;
    float* to = values + block + mine;
    const bool stores = !is_key && block + mine < vdim_p;
#pragma unroll 1
    for (int b = 0; b < kChunkRows / 16; ++b) {
        // 16 rows at a time: the solved rows leave them as products,
        const float* tiles = sa + 256 * (b * (b + 1) / 2);
        if (b > 0) {
            for (int at16 = wave; at16 < 2 * kDim / 16; at16 += kChunkThreads / kWave) {
                float* x = (at16 < kDim / 16 ? sq + 16 * at16 : sk + 16 * at16 - kDim) + c;
                floatx4 sums[4] = {};
                for (int s = 0; s < b; ++s) {
                    const float4 a = *reinterpret_cast<const float4*>(tiles + 256 * s + 16 * c + 4 * g);
                    const float* solved = x + (16 * s + 4 * g) * row_p;
#pragma unroll
                    for (int v = 0; v < 4; ++v) sums[v] = mfma4(element(a, v), solved[v * row_p], sums[v]);
                }
                const floatx4 sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
#pragma unroll
                for (int v = 0; v < 4; ++v) x[(16 * b + 4 * g + v) * row_p] += sum[v];
            }
            __syncthreads();
        }
        // then a column a thread among themselves
        if (tid < 2 * kDim) {
            float x[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) x[t] = column[(16 * b + t) * row_p];
#pragma unroll
            for (int t = 1; t < 16; ++t) {
                float4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i4 = 0; 4 * i4 < t; ++i4) {
                    const float4 a = *reinterpret_cast<const float4*>(tiles + 256 * b + 16 * t + 4 * i4);
                    sum.x = fmaf(a.x, x[4 * i4], sum.x);
                    if (4 * i4 + 1 < t) sum.y = fmaf(a.y, x[4 * i4 + 1], sum.y);
                    if (4 * i4 + 2 < t) sum.z = fmaf(a.z, x[4 * i4 + 2], sum.z);
                    if (4 * i4 + 3 < t) sum.w = fmaf(a.w, x[4 * i4 + 3], sum.w);
                }
                x[t] += (sum.x + sum.y) + (sum.z + sum.w);
            }
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                column[(16 * b + t) * row_p] = x[t];
                if (stores) to[(16 * b + t) * vdim_p] = x[t];
            }
        }
        __syncthreads();
    }
    if (solved_k != nullptr)
#pragma unroll 4
        for (int idx = tid; idx < kChunkRows * kDim / 4; idx += kChunkThreads) {
            const Place a = place_of<kT>(idx);
            reinterpret_cast<float4*>(solved_k)[idx] = *reinterpret_cast<const float4*>(sk + a.row * row_p + a.channel);
        }
}

// kT: tiles of 16 key channels a wave of chunk_walk holds; 64 kT channels, the last ones zeros.
template <bool kDelta, int kT>
__global__ void __launch_bounds__(kChunkThreads, 2) chunk_prepare_kernel(ChunkArgs p) {
    extern __shared__ __align__(16) float chunk_lds[];
    constexpr int kDim = 64 * kT, row_p = kDim + 4;
    float* sq = chunk_lds;                              // [64][row_p]
    float* sk = sq + kChunkRows * row_p;
    float* sa = sk + kChunkRows * row_p;                // delta rule: -A in tiles of 16 x 16, those on and below the diagonal
    __shared__ double cum[kChunkRows];
    __shared__ float strength[kChunkRows], q_norm[kChunkRows], k_norm[kChunkRows], so_far[kChunkRows], to_end[kChunkRows];
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int chunk = blockIdx.x, head = blockIdx.y, kvh = head / (p.heads / p.kv_heads);
    const int first = p.chunks[4 * chunk], n = p.chunks[4 * chunk + 1] - first;
    const long at = static_cast<long>(chunk) * p.heads + head;
    const int block = blockIdx.z * kDim;        // delta rule: the value columns solved here; the first workgroup writes all the rest

    // Reads in batches, of the last row or channel again where there is none, so that no read waits for the one before; the first
    // batch is on its way while wave 0 makes the decays, a logarithm in double among them.
    constexpr int kBatch = 8;
    static_assert(kChunkRows * kDim % (kBatch * kChunkThreads) == 0, "whole batches");
    float q_read[kBatch], k_read[kBatch];
    const auto read_rows = [&](int from) {
#pragma unroll
        for (int e = 0; e < kBatch; ++e) {
            const int t = (from + e * kChunkThreads) / kDim, i = (from + e * kChunkThreads) % kDim;
            const float* base = p.rows + static_cast<long>(first + min(t, n - 1)) * p.stride + kvh * p.dim + min(i, p.dim - 1);
            q_read[e] = base[p.q_off], k_read[e] = base[p.k_off];
        }
    };
    read_rows(tid);
    if (wave == 0) {
        // the decays' logarithms summed up over the chunk; rows past its end decay nothing and write nothing
        double l = 0.;
        if (lane < n) {
            const long row = first + lane;
            if (kDelta) {
                l = -expf(load_any(p.rate_log, head)) * chunk_softplus(p.step[row * p.step_stride + head] + load_any(p.step_bias, head));
                strength[lane] = 1.0f / (1.0f + expf(-p.beta[row * p.beta_stride + head]));
            } else {
                const float d = p.coef ? p.coef[2 * (row * p.heads + head)] : p.decay[head];
                l = d <= 0.f ? static_cast<double>(kNothingLeft) : log(static_cast<double>(d));
                strength[lane] = p.coef ? p.coef[2 * (row * p.heads + head) + 1] : 1.f;
            }
            if (l < kNothingLeft) l = kNothingLeft;              // (a decay that is not a number stays one)
        } else {
            strength[lane] = 0.f;
        }
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const double before = __shfl_up(l, off, kWave);
            if (lane >= off) l += before;
        }
        cum[lane] = l;
        so_far[lane] = between(l, 0.);
        to_end[lane] = between(__shfl(l, kWave - 1, kWave), l);
    }
    for (int from = tid; from < kChunkRows * kDim; from += kBatch * kChunkThreads) {
        if (from != tid) read_rows(from);
#pragma unroll
        for (int e = 0; e < kBatch; ++e) {
            const int t = (from + e * kChunkThreads) / kDim, i = (from + e * kChunkThreads) % kDim;
            const bool there = t < n && i < p.dim;
            sq[t * row_p + i] = there ? chunk_act(q_read[e], p.silu) : 0.f;
            sk[t * row_p + i] = there ? chunk_act(k_read[e], p.silu) : 0.f;
        }
    }
    __syncthreads();
    if (!kDelta && p.cos_table != nullptr) {
        for (int idx = tid; idx < n * p.rot_half; idx += kChunkThreads) {
            const int t = idx / p.rot_half, i = idx % p.rot_half;
            const long at = static_cast<long>(min(p.positions[first + t], p.table_positions - 1)) * p.rot_half + i;
            const float cs = p.cos_table[at], sn = p.sin_table[at];
            float* q = sq + t * row_p + i;
            float* k = sk + t * row_p + i;
            const float q0 = q[0], q1 = q[p.rot_half], k0 = k[0], k1 = k[p.rot_half];
            q[0] = q0 * cs - q1 * sn, q[p.rot_half] = q1 * cs + q0 * sn;
            k[0] = k0 * cs - k1 * sn, k[p.rot_half] = k1 * cs + k0 * sn;
        }
        __syncthreads();
    }
    {   // four lanes a row
        const int t = tid / 4, sub = tid % 4;
        float qq = 0.f, kk = 0.f;
        if (kDelta) {
            for (int i = sub; i < p.dim; i += 4) {
                qq = fmaf(sq[t * row_p + i], sq[t * row_p + i], qq);
                kk = fmaf(sk[t * row_p + i], sk[t * row_p + i], kk);
            }
            qq = add_lanes<1>(qq);
            kk = add_lanes<1>(kk);
            qq = add_lanes<2>(qq);
            kk = add_lanes<2>(kk);
        }
        if (sub == 0) {
            q_norm[t] = kDelta ? p.q_scale / sqrtf(qq + p.unit_eps) : p.q_scale;
            k_norm[t] = kDelta ? p.k_scale / sqrtf(kk + p.unit_eps) : p.k_scale;
        }
    }
    __syncthreads();
    if (tid == 0 && block == 0) p.total[at] = so_far[kChunkRows - 1];

    // k_t.k_i and q_t.k_i, the ten tiles of 16 x 16 on and below the diagonal shared out over the waves
    float* mix = p.mix + at * kChunkRows * kChunkRows;
    const int c = lane & 15, g = lane >> 4;
    for (int pair = wave; pair < kChunkTiles; pair += kChunkThreads / kWave) {
        const int ti = pair < 1 ? 0 : pair < 3 ? 1 : pair < 6 ? 2 : 3, tj = pair - ti * (ti + 1) / 2;
        const float* rq = sq + (16 * ti + c) * row_p + 4 * g;
        const float* rk = sk + (16 * ti + c) * row_p + 4 * g;
        const float* ck = sk + (16 * tj + c) * row_p + 4 * g;
        // Four sums side by side over 64 channels at a time: short chains, of which less rounds at the result's size.  (Over all 256
        // channels read-outs were off by 2.2e-7 of their norm, more than those of the rows walked one by one: 2.0e-7.)
        floatx4 kk = {}, qk = {};
#pragma unroll
        for (int from = 0; from < kDim; from += 64) {
            floatx4 kks[4] = {}, qks[4] = {};
#pragma unroll
            for (int d = from; d < from + 64; d += 16) {
                const float4 b = *reinterpret_cast<const float4*>(ck + d), aq = *reinterpret_cast<const float4*>(rq + d);
#pragma unroll
                for (int v = 0; v < 4; ++v) qks[v] = mfma4(element(aq, v), element(b, v), qks[v]);
                if (kDelta) {
                    const float4 ak = *reinterpret_cast<const float4*>(rk + d);
#pragma unroll
                    for (int v = 0; v < 4; ++v) kks[v] = mfma4(element(ak, v), element(b, v), kks[v]);
                }
            }
            qk += (qks[0] + qks[1]) + (qks[2] + qks[3]);
            kk += (kks[0] + kks[1]) + (kks[2] + kks[3]);
        }
        const int i = 16 * tj + c;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 16 * ti + 4 * g + v;
            // (chosen and not multiplied by zero: what is not finite in a later row's key is none of an earlier row's)
            const float decayed = between(cum[t], cum[i]) * k_norm[i];
            if (block == 0) mix[4 * ((ti * 4 + tj) * kWave + 16 * (c / 4) + 4 * g + v) + c % 4] = t >= i ? decayed * q_norm[t] * qk[v] : 0.f;
            if (kDelta) sa[256 * pair + 16 * (4 * g + v) + c] = t >= i ? -decayed * k_norm[t] * strength[t] * kk[v] : 0.f;
        }
    }
    float* q_in = p.q_in + at * kChunkRows * kDim;
    float* k_out = p.k_out + at * kChunkRows * kDim;
    if (block == 0) {
#pragma unroll 4
        for (int idx = tid; idx < kChunkRows * kDim / 4; idx += kChunkThreads) {
            const Place a = place_of<kT>(idx);
            const float4 x = *reinterpret_cast<const float4*>(sq + a.row * row_p + a.channel);
            const float f = q_norm[a.row] * so_far[a.row];
            reinterpret_cast<float4*>(q_in)[idx] = float4{x.x * f, x.y * f, x.z * f, x.w * f};
            const int ki = 16 * (idx / kWave / 4) + c, kt = 16 * (idx / kWave % 4) + 4 * g;
            float4 y;
            y.x = sk[kt * row_p + ki] * (k_norm[kt] * to_end[kt]);
            y.y = sk[(kt + 1) * row_p + ki] * (k_norm[kt + 1] * to_end[kt + 1]);
            y.z = sk[(kt + 2) * row_p + ki] * (k_norm[kt + 2] * to_end[kt + 2]);
            y.w = sk[(kt + 3) * row_p + ki] * (k_norm[kt + 3] * to_end[kt + 3]);
            reinterpret_cast<float4*>(k_out)[idx] = y;
        }
    }
    float* values = p.values + at * kChunkRows * p.vdim_p;
    const float* v_base = p.rows + static_cast<long>(first) * p.stride + p.v_off + head * p.vdim;
    const auto read_v = [&](int t, int j) { return v_base[min(t, n - 1) * p.stride + min(j, p.vdim - 1)]; };
    const auto taken_v = [&](float v, int t, int j) { return t < n && j < p.vdim ? chunk_act(v, p.silu) : 0.f; };
    if constexpr (!kDelta) {
        constexpr int kRows = kChunkThreads / kWave, kEach = kChunkRows / kRows;
        const int norm = p.dot != nullptr ? p.vdim : -1;        // the normaliser's column
        float by[kEach];
#pragma unroll
        for (int e = 0; e < kEach; ++e) by[e] = strength[wave + kRows * e];
        for (int j = lane; j < p.vdim_p; j += kWave) {
            if (j == norm) continue;
            float v[kEach];
#pragma unroll
            for (int e = 0; e < kEach; ++e) v[e] = read_v(wave + kRows * e, j);
#pragma unroll
            for (int e = 0; e < kEach; ++e) {
                const int t = wave + kRows * e;
                values[t * p.vdim_p + j] = taken_v(v[e], t, j) * by[e];
            }
        }
        if (norm >= 0 && tid < kChunkRows) values[tid * p.vdim_p + norm] = strength[tid];      // (0 past the chunk's end)
    } else {
        float* solved_k = p.solved_k + at * kChunkRows * kDim;
        __syncthreads();                    // M is made and K written: their places take the right sides, K and a block of V
        for (int from = tid; from < kChunkRows * kDim; from += kBatch * kChunkThreads) {
            float v[kBatch];
#pragma unroll
            for (int e = 0; e < kBatch; ++e) v[e] = read_v((from + e * kChunkThreads) / kDim, block + (from + e * kChunkThreads) % kDim);
#pragma unroll
            for (int e = 0; e < kBatch; ++e) {
                const int t = (from + e * kChunkThreads) / kDim, i = (from + e * kChunkThreads) % kDim;
                sk[t * row_p + i] *= strength[t] * so_far[t] * k_norm[t];
                sq[t * row_p + i] = strength[t] * taken_v(v[e], t, block + i);
            }
        }
        __syncthreads();
        solve_chunk<kT>(sq, sk, sa, values, p.vdim_p, block, block == 0 ? solved_k : nullptr);
    }
}

// The same for the delta rule with a decay for every key channel (see the head of this file).
template <int kT>
__global__ void __launch_bounds__(kChunkThreads, 1) chunk_prepare_channel_kernel(ChunkArgs p) {
    extern __shared__ __align__(16) float chunk_lds[];
    constexpr int kDim = 64 * kT, row_p = kDim + 4, kTiles = kChunkRows / 16;
    float* sq = chunk_lds;                              // [64][row_p]: q, then q times the decays since its tile's start
    float* sk = sq + kChunkRows * row_p;                // k, then likewise
    float* sg = sk + kChunkRows * row_p;                // the decays, then k times the decays behind it up to its tile's end
    float* sa = sg + kChunkRows * row_p;                // -A in tiles of 16 x 16, those on and below the diagonal
    float* whole = sa + kChunkTiles * 256;              // [tiles][kDim]: a tile's decays multiplied up
    float* earlier = whole + kTiles * kDim;             // of the tiles before it
    float* later = earlier + kTiles * kDim;             // of the tiles behind it
    __shared__ float strength[kChunkRows], q_norm[kChunkRows], k_norm[kChunkRows];
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, c = lane & 15, g = lane >> 4;
    const int chunk = blockIdx.x, head = blockIdx.y, kvh = head / (p.heads / p.kv_heads);
    const int first = p.chunks[4 * chunk], n = p.chunks[4 * chunk + 1] - first;
    const long at = static_cast<long>(chunk) * p.heads + head;
    const int block = blockIdx.z * kDim;                // the value columns solved here; the first workgroup writes all the rest
    const float rate = expf(load_any(p.rate_log, head));

    constexpr int kBatch = 8;
    static_assert(kChunkRows * kDim % (kBatch * kChunkThreads) == 0, "whole batches");
    for (int from = tid; from < kChunkRows * kDim; from += kBatch * kChunkThreads) {
        float q[kBatch], k[kBatch], d[kBatch];
#pragma unroll
        for (int e = 0; e < kBatch; ++e) {
            const int t = (from + e * kChunkThreads) / kDim, i = min((from + e * kChunkThreads) % kDim, p.dim - 1);
            const long row = first + min(t, n - 1);
            const float* base = p.rows + row * p.stride + kvh * p.dim + i;
            q[e] = base[p.q_off], k[e] = base[p.k_off];
            d[e] = p.step[row * p.step_stride + static_cast<long>(head) * p.dim + i];
        }
#pragma unroll
        for (int e = 0; e < kBatch; ++e) {
            const int t = (from + e * kChunkThreads) / kDim, i = (from + e * kChunkThreads) % kDim;
            const bool there = t < n && i < p.dim;                 // nothing decays, is written or read elsewhere
            sq[t * row_p + i] = there ? chunk_act(q[e], p.silu) : 0.f;
            sk[t * row_p + i] = there ? chunk_act(k[e], p.silu) : 0.f;
            sg[t * row_p + i] = there ? expf(-rate * chunk_softplus(d[e] + load_any(p.step_bias, static_cast<long>(head) * p.dim + i))) : 1.f;
        }
    }
    if (tid < kChunkRows) strength[tid] = tid < n ? 1.0f / (1.0f + expf(-p.beta[(first + tid) * p.beta_stride + head])) : 0.f;
    __syncthreads();
    {   // four lanes a row
        const int t = tid / 4, sub = tid % 4;
        float qq = 0.f, kk = 0.f;
        for (int i = sub; i < p.dim; i += 4) {
            qq = fmaf(sq[t * row_p + i], sq[t * row_p + i], qq);
            kk = fmaf(sk[t * row_p + i], sk[t * row_p + i], kk);
        }
        qq = add_lanes<1>(qq);
        kk = add_lanes<1>(kk);
        qq = add_lanes<2>(qq);
        kk = add_lanes<2>(kk);
        if (sub == 0) {
            q_norm[t] = p.q_scale / sqrtf(qq + p.unit_eps);
            k_norm[t] = p.k_scale / sqrtf(kk + p.unit_eps);
        }
    }
    __syncthreads();
    for (int idx = tid; idx < kChunkRows * kDim; idx += kChunkThreads) {
        const int t = idx / kDim, i = idx % kDim;
        sq[t * row_p + i] *= q_norm[t];
        sk[t * row_p + i] *= k_norm[t];
    }
    __syncthreads();

    float* mix = p.mix + at * kChunkRows * kChunkRows;
    {   // within a tile, a wave each: lane (c, g) takes a quarter of key c's channels through the rows from c on
        constexpr int kShare = kDim / 4;
        const float* tile_q = sq + 16 * wave * row_p + kShare * g;
        const float* tile_k = sk + 16 * wave * row_p + kShare * g;
        const float* tile_g = sg + 16 * wave * row_p + kShare * g;
        float4 key[kShare / 4];
#pragma unroll
        for (int j = 0; j < kShare / 4; ++j) key[j] = *reinterpret_cast<const float4*>(tile_k + c * row_p + 4 * j);
        float* to_a = sa + 256 * (wave * (wave + 1) / 2 + wave);
#pragma unroll 1
        for (int t = 0; t < 16; ++t) {
            float4 qs = {0.f, 0.f, 0.f, 0.f}, ks = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < kShare / 4; ++j) {
                const float4 d = *reinterpret_cast<const float4*>(tile_g + t * row_p + 4 * j);
                const float4 x = *reinterpret_cast<const float4*>(tile_q + t * row_p + 4 * j);
                const float4 y = *reinterpret_cast<const float4*>(tile_k + t * row_p + 4 * j);
                if (t > c) key[j].x *= d.x, key[j].y *= d.y, key[j].z *= d.z, key[j].w *= d.w;
                qs.x = fmaf(x.x, key[j].x, qs.x), qs.y = fmaf(x.y, key[j].y, qs.y);
                qs.z = fmaf(x.z, key[j].z, qs.z), qs.w = fmaf(x.w, key[j].w, qs.w);
                ks.x = fmaf(y.x, key[j].x, ks.x), ks.y = fmaf(y.y, key[j].y, ks.y);
                ks.z = fmaf(y.z, key[j].z, ks.z), ks.w = fmaf(y.w, key[j].w, ks.w);
            }
            float qk = (qs.x + qs.y) + (qs.z + qs.w), kk = (ks.x + ks.y) + (ks.z + ks.w);
            qk = add_lanes<16>(qk);
            kk = add_lanes<16>(kk);
            qk = add_lanes<32>(qk);
            kk = add_lanes<32>(kk);
            if (g == 0) {
                if (block == 0) mix[4 * ((wave * 4 + wave) * kWave + 16 * (c / 4) + t) + c % 4] = t >= c ? qk : 0.f;
                to_a[16 * t + c] = t > c ? -strength[16 * wave + t] * kk : 0.f;
            }
        }
    }
    __syncthreads();
    // the decays up to a row and behind it, within its tile, onto the rows: a thread a channel and tile
    for (int idx = tid; idx < kTiles * kDim; idx += kChunkThreads) {
        const int tile = idx / kDim, i = idx % kDim;
        float k[16], d[16], so_far = 1.f, behind = 1.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int place = (16 * tile + r) * row_p + i;
            k[r] = sk[place], d[r] = sg[place];
            so_far *= d[r];
            sq[place] *= so_far;
            sk[place] = k[r] * so_far;
        }
#pragma unroll
        for (int r = 15; r >= 0; --r) {
            sg[(16 * tile + r) * row_p + i] = k[r] * behind;
            behind *= d[r];
        }
        whole[idx] = behind;
    }
    __syncthreads();
    if (tid < kDim) {
        float so_far = 1.f, behind = 1.f;
#pragma unroll
        for (int tile = 0; tile < kTiles; ++tile) {
            earlier[tile * kDim + tid] = so_far;
            so_far *= whole[tile * kDim + tid];
        }
#pragma unroll
        for (int tile = kTiles - 1; tile >= 0; --tile) {
            later[tile * kDim + tid] = behind;
            behind *= whole[tile * kDim + tid];
        }
        if (block == 0) p.total[at * kDim + tid] = so_far;
    }
    __syncthreads();
    // between tiles: the six below the diagonal shared out over the waves
    for (int pair = wave; pair < 6; pair += kChunkThreads / kWave) {
        const int ti = pair < 1 ? 1 : pair < 3 ? 2 : 3, tj = pair - ti * (ti - 1) / 2;
        const float* rq = sq + (16 * ti + c) * row_p + 4 * g;
        const float* rk = sk + (16 * ti + c) * row_p + 4 * g;
        const float* ck = sg + (16 * tj + c) * row_p + 4 * g;
        floatx4 kks[4] = {}, qks[4] = {};
#pragma unroll
        for (int d = 0; d < kDim; d += 16) {
            float4 b = *reinterpret_cast<const float4*>(ck + d);
            for (int tile = tj + 1; tile < ti; ++tile) {
                const float4 w = *reinterpret_cast<const float4*>(whole + tile * kDim + 4 * g + d);
                b.x *= w.x, b.y *= w.y, b.z *= w.z, b.w *= w.w;
            }
            const float4 aq = *reinterpret_cast<const float4*>(rq + d), ak = *reinterpret_cast<const float4*>(rk + d);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                qks[v] = mfma4(element(aq, v), element(b, v), qks[v]);
                kks[v] = mfma4(element(ak, v), element(b, v), kks[v]);
            }
        }
        const floatx4 qk = (qks[0] + qks[1]) + (qks[2] + qks[3]), kk = (kks[0] + kks[1]) + (kks[2] + kks[3]);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 16 * ti + 4 * g + v;
            if (block == 0) mix[4 * ((ti * 4 + tj) * kWave + 16 * (c / 4) + 4 * g + v) + c % 4] = qk[v];
            sa[256 * (ti * (ti + 1) / 2 + tj) + 16 * (4 * g + v) + c] = -strength[t] * kk[v];
        }
    }
    if (block == 0) {
        float* q_in = p.q_in + at * kChunkRows * kDim;
        float* k_out = p.k_out + at * kChunkRows * kDim;
#pragma unroll 4
        for (int idx = tid; idx < kChunkRows * kDim / 4; idx += kChunkThreads) {
            const Place a = place_of<kT>(idx);
            const float4 x = *reinterpret_cast<const float4*>(sq + a.row * row_p + a.channel);
            const float4 f = *reinterpret_cast<const float4*>(earlier + a.row / 16 * kDim + a.channel);
            reinterpret_cast<float4*>(q_in)[idx] = float4{x.x * f.x, x.y * f.y, x.z * f.z, x.w * f.w};
            const int ki = 16 * (idx / kWave / 4) + c, kt = 16 * (idx / kWave % 4) + 4 * g;
            const float h = later[kt / 16 * kDim + ki];
            float4 y;
            y.x = sg[kt * row_p + ki] * h;
            y.y = sg[(kt + 1) * row_p + ki] * h;
            y.z = sg[(kt + 2) * row_p + ki] * h;
            y.w = sg[(kt + 3) * row_p + ki] * h;
            reinterpret_cast<float4*>(k_out)[idx] = y;
        }
    }
    __syncthreads();                        // q and k are used up: their places take the right sides, K and a block of V
    const float* v_base = p.rows + static_cast<long>(first) * p.stride + p.v_off + head * p.vdim;
    for (int from = tid; from < kChunkRows * kDim; from += kBatch * kChunkThreads) {
        float v[kBatch];
#pragma unroll
        for (int e = 0; e < kBatch; ++e) {
            const int t = (from + e * kChunkThreads) / kDim, j = block + (from + e * kChunkThreads) % kDim;
            v[e] = v_base[min(t, n - 1) * p.stride + min(j, p.vdim - 1)];
        }
#pragma unroll
        for (int e = 0; e < kBatch; ++e) {
            const int t = (from + e * kChunkThreads) / kDim, i = (from + e * kChunkThreads) % kDim;
            sk[t * row_p + i] *= strength[t] * earlier[t / 16 * kDim + i];
            sq[t * row_p + i] = t < n && block + i < p.vdim ? strength[t] * chunk_act(v[e], p.silu) : 0.f;
        }
    }
    __syncthreads();
    solve_chunk<kT>(sq, sk, sa, p.values + at * kChunkRows * p.vdim_p, p.vdim_p, block,
                    block == 0 ? p.solved_k + at * kChunkRows * kDim : nullptr);
}

// Workgroups of chunk_walk a compute unit, where its registers allow: 256 a lane for two of them.  (Eight portions of 512 rows with
// one workgroup and with two a unit, us: fixed decays, 4 heads of 128 x 256, 69 and 58; the delta rule, 8 heads of 64 x 128, 90 and 80.)
template <bool kDelta, int kT>
constexpr int kWalkers = kT * (kDelta ? 2 : 1) <= 2 ? 2 : 1;

// What a wave needs of a chunk, all of it asked for a chunk ahead.
template <bool kDelta, int kT, bool kChannel>
struct ChunkOperands {
    float4 w[kDelta ? 4 : 1][kT], q[4][kT], k[kT][4], m[4], totals[kChannel ? kT : 1];
    float u[4], total;
    int first, end;
};

template <bool kDelta, int kT, bool kChannel>
__device__ inline void fetch_chunk(const ChunkArgs& p, int chunk, int head, int wave, int c, int g, int col,
                                   ChunkOperands<kDelta, kT, kChannel>& o) {
    const long at = static_cast<long>(chunk) * p.heads + head;
    constexpr int kDim = 64 * kT;
    const int lane = 16 * g + c;
    const float4* q_in = reinterpret_cast<const float4*>(p.q_in + at * kChunkRows * kDim) + wave * 4 * kT * kWave + lane;
    const float4* k_out = reinterpret_cast<const float4*>(p.k_out + at * kChunkRows * kDim) + wave * 4 * kT * kWave + lane;
    const float4* mix = reinterpret_cast<const float4*>(p.mix + at * kChunkRows * kChunkRows) + wave * 4 * kWave + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < kT; ++t) {
            if constexpr (kDelta)
                o.w[r][t] = (reinterpret_cast<const float4*>(p.solved_k + at * kChunkRows * kDim) + wave * 4 * kT * kWave + lane)[(r * kT + t) * kWave];
            o.q[r][t] = q_in[(r * kT + t) * kWave];
        }
    o.first = p.chunks[4 * chunk];
    o.end = p.chunks[4 * chunk + 1];
    if constexpr (kChannel) {
#pragma unroll
        for (int t = 0; t < kT; ++t) o.totals[t] = *reinterpret_cast<const float4*>(p.total + at * kDim + 16 * (wave * kT + t) + 4 * g);
    } else {
        o.total = p.total[at];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) o.u[v] = p.values[at * kChunkRows * p.vdim_p + (16 * wave + 4 * g + v) * p.vdim_p + col];
#pragma unroll
    for (int s = 0; s < 4; ++s) o.m[s] = s <= wave ? mix[s * kWave] : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) o.k[t][r] = k_out[(t * 4 + r) * kWave];
}

// What the walk shares over a workgroup.
template <bool kDelta>
struct WalkShared {
    float part[kDelta ? 2 : 1][kChunkThreads / kWave][kChunkRows * kPartStride];
    float u[kChunkRows * kPartStride];
};

// A workgroup walks the chunks of one portion for one head and 16 columns; wave w holds key channels 16 kT w .. of the columns
// and makes what they give to every row of W S and Q S; the parts meet in shared memory, where wave w takes rows 16 w ..
// Returns whether a read-out of this lane came out as no number.  Not kCareful: if only because M's zeros met an infinity or a
// NaN of a later row, which is none of the row's; kCareful: such sums are made without the rows behind.
template <bool kDelta, int kT, bool kChannel, bool kCareful>
__device__ inline bool walk_chunks(const ChunkArgs& p, WalkShared<kDelta>& shared, int g0, int g1, int head, int wave, int c, int g, int col,
                                   bool held, bool is_norm, floatx4 (&S)[kT]) {
    constexpr int kWaves = kChunkThreads / kWave;
    auto& part = shared.part;
    float* su = shared.u;
    bool odd = false;
    ChunkOperands<kDelta, kT, kChannel> ahead;
    if constexpr (!kCareful) fetch_chunk<kDelta, kT, kChannel>(p, g0, head, wave, c, g, col, ahead);
    for (int chunk = g0; chunk < g1; ++chunk) {
        if constexpr (kCareful) fetch_chunk<kDelta, kT, kChannel>(p, chunk, head, wave, c, g, col, ahead);
        const ChunkOperands<kDelta, kT, kChannel> now = ahead;
        if constexpr (!kCareful) fetch_chunk<kDelta, kT, kChannel>(p, chunk + 1 < g1 ? chunk + 1 : chunk, head, wave, c, g, col, ahead);
        // Sums are kept short and put together at the end (two a row of W S and Q S, one a tile of M U, the chunk's own part of S
        // by itself): what is added to a sum is rounded at the sum's size.
        // (sums of all four tiles of rows side by side take registers that a second workgroup a unit needs)
        constexpr int kSide = kWalkers<kDelta, kT> == 1 ? 4 : kDelta ? 1 : 2;
#pragma unroll
        for (int r0 = 0; r0 < 4; r0 += kSide) {
            floatx4 ws[kSide][2] = {}, qs[kSide][2] = {};
#pragma unroll
            for (int t = 0; t < kT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int r = 0; r < kSide; ++r) {
                        if constexpr (kDelta) ws[r][v / 2] = mfma4(element(now.w[r0 + r][t], v), S[t][v], ws[r][v / 2]);
                        qs[r][v / 2] = mfma4(element(now.q[r0 + r][t], v), S[t][v], qs[r][v / 2]);
                    }
#pragma unroll
            for (int r = 0; r < kSide; ++r) {
                const floatx4 w = ws[r][0] + ws[r][1], q = qs[r][0] + qs[r][1];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    part[0][wave][(16 * (r0 + r) + 4 * g + v) * kPartStride + c] = q[v];
                    if constexpr (kDelta) part[kDelta ? 1 : 0][wave][(16 * (r0 + r) + 4 * g + v) * kPartStride + c] = w[v];
                }
            }
        }
        __syncthreads();
        floatx4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int spot = (16 * wave + 4 * g + v) * kPartStride + c;
            static_assert(kWaves == 4, "four parts");
            float seen = 0.f;
            o[v] = (part[0][0][spot] + part[0][1][spot]) + (part[0][2][spot] + part[0][3][spot]);
            if constexpr (kDelta) {
                constexpr int kW = kDelta ? 1 : 0;
                seen = (part[kW][0][spot] + part[kW][1][spot]) + (part[kW][2][spot] + part[kW][3][spot]);
            }
            su[spot] = now.u[v] - seen;
        }
        __syncthreads();
        float u[4][4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v) u[s][v] = su[(16 * s + 4 * g + v) * kPartStride + c];
        floatx4 mu[4] = {}, wrote[kT] = {};
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                mu[s] = mfma4(element(now.m[s], v), u[s][v], mu[s]);    // tiles above the diagonal are zeros
#pragma unroll
                for (int t = 0; t < kT; ++t) wrote[t] = mfma4(element(now.k[t][s], v), u[s][v], wrote[t]);
            }
        [[maybe_unused]] const floatx4 before = o;
        o += (mu[0] + mu[1]) + (mu[2] + mu[3]);
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if constexpr (kChannel) S[t][v] = fmaf(S[t][v], element(now.totals[t], v), wrote[t][v]);
                else S[t][v] = fmaf(S[t][v], now.total, wrote[t][v]);
            }
        const bool none = o[0] != o[0] || o[1] != o[1] || o[2] != o[2] || o[3] != o[3];
        if constexpr (!kCareful) {
            odd = odd || none;
        } else if (__any(none)) {
            // the same sums an element at a time, M from memory
            const float* mix = p.mix + (static_cast<long>(chunk) * p.heads + head) * kChunkRows * kChunkRows + 16 * wave * kChunkRows;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float sums[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll 1
                    for (int e = 0; e < 16; ++e) {
                        const int i = 4 * (e % 4) + e / 4;                                // in the order of the instructions
                        if (16 * s + i <= 16 * wave + 4 * g + v)
                            sums[s] = fmaf(mix[4 * (s * kWave + 16 * (e % 4) + 4 * g + v) + e / 4], su[(16 * s + i) * kPartStride + c], sums[s]);
                    }
                o[v] = before[v] + ((sums[0] + sums[1]) + (sums[2] + sums[3]));
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = 16 * wave + 4 * g + v;
            const long row_head = static_cast<long>(now.first + t) * p.heads + head;
            if (now.first + t < now.end && held) *(is_norm ? p.dot + row_head : p.out + row_head * p.vdim + col) = o[v];
        }
    }
    return odd;
}

template <bool kDelta, int kT, bool kChannel>
__global__ void __launch_bounds__(kChunkThreads, (kWalkers<kDelta, kT>)) chunk_walk_kernel(ChunkArgs p) {
    __shared__ WalkShared<kDelta> shared;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, c = lane & 15, g = lane >> 4;
    const int link = blockIdx.x, head = blockIdx.y, col = 16 * blockIdx.z + c;
    const int slot = p.links[4 * link], fresh = p.links[4 * link + 1], g0 = p.links[4 * link + 2], g1 = p.links[4 * link + 3];
    float* state = p.state + slot * p.slot_stride + head * p.head_stride;
    const bool is_norm = p.dot != nullptr && col == p.vdim, held = col < p.vdim || is_norm;
    const auto place = [&](int i) { return is_norm ? static_cast<long>(p.dim) * p.vdim + i : static_cast<long>(i) * p.vdim + col; };
    floatx4 S[kT];
    const auto load = [&]() {
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = 16 * (wave * kT + t) + 4 * g + v;
                S[t][v] = (!fresh && i < p.dim && held) ? state[place(i)] : 0.f;
            }
    };
    if (g0 >= g1) return;
    load();
    // (once more from the start where a read-out is no number: a look at every chunk within the walk cost it 4 %)
    if (__syncthreads_or(walk_chunks<kDelta, kT, kChannel, false>(p, shared, g0, g1, head, wave, c, g, col, held, is_norm, S))) {
        load();
        walk_chunks<kDelta, kT, kChannel, true>(p, shared, g0, g1, head, wave, c, g, col, held, is_norm, S);
    }
    if (!p.write_state) return;
#pragma unroll
    for (int t = 0; t < kT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * (wave * kT + t) + 4 * g + v;
            if (i < p.dim && held) state[place(i)] = S[t][v];
        }
}

static int chunk_tiles(int dim) { return dim <= 64 ? 1 : dim <= 128 ? 2 : 4; }      // tiles of 16 key channels a wave

enum ChunkRule : int { kChunkOuter = 0, kChunkDelta = 1, kChunkDeltaChannel = 2 };

template <typename K>
static int launch_prepare(K kernel, const dim3& grid, size_t shared, const ChunkArgs& a, hipStream_t stream) {
    if (shared > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(shared));
        LEONE_REQUIRE(e == hipSuccess, "chunked_memory: %zu bytes of shared memory were refused: %s", shared, hipGetErrorString(e));
    }
    kernel<<<grid, kChunkThreads, shared, stream>>>(a);
    LEONE_LAUNCH_CHECK("chunk_prepare");
    return 0;
}

}  // namespace leone

using namespace leone;

extern "C" int leone_chunk_rows() { return kChunkRows; }
extern "C" int leone_chunk_max_dim() { return kChunkMaxDim; }
extern "C" int leone_chunk_max_delta_dim() { return kChunkMaxDeltaDim; }

// Floats of workspace a chunk and head needs; rule: 0 fixed decays or gates (with gates vdim counts the normaliser's column), 1
// the delta rule with one decay a head, 2 with one for every key channel.
extern "C" long leone_chunk_workspace(int dim, int vdim, int rule) {
    const long dim_p = 64L * chunk_tiles(dim), vdim_p = ceil_div(vdim, 16) * 16L;
    return kChunkRows * (dim_p * (rule != kChunkOuter ? 3 : 2) + vdim_p + kChunkRows) + (rule == kChunkDeltaChannel ? dim_p : 4);
}

// A long portion's rows through a memory.  beta, step, rate_log and step_bias belong to the delta rule (all null: fixed decays
// from `decay`, or gates from `coef` [rows, heads, 2] with the normaliser's read-out into `dot`); the delta rule makes q and k
// unit vectors first; step_each: a step size, and so a decay, for every key channel.  cos_table: q and k are rotated first (not
// for the delta rule).  chunks and links: the portions' chunks of leone_chunk_rows() rows as the other recurrences list them.
// workspace: n_chunks * heads * leone_chunk_workspace() floats.  state: heads of head_stride floats, [dim, vdim] and, with
// gates, the normaliser [dim].
extern "C" int leone_chunked_memory(const float* rows, long stride, int q_off, int k_off, int v_off, int silu, float q_scale,
                                    float k_scale, float unit_eps, const float* beta, long beta_stride, const float* step,
                                    long step_stride, int step_each, const void* rate_log, const void* step_bias, int vec_dtype,
                                    const float* decay, const float* coef, const float* cos_table, const float* sin_table,
                                    int rotary_dim, int table_positions, const int* positions, const int* chunks, int n_chunks,
                                    const int* links, int n_links, float* workspace, float* state, long slot_stride,
                                    long head_stride, int write_state, float* out, float* dot, int heads, int kv_heads, int dim,
                                    int vdim, hipStream_t stream) {
    const int rule = beta == nullptr ? kChunkOuter : step_each ? kChunkDeltaChannel : kChunkDelta;
    const bool delta = rule != kChunkOuter;
    LEONE_REQUIRE(rows && chunks && links && workspace && state && out && n_chunks > 0 && n_links > 0, "chunked_memory: null pointer or no chunks");
    LEONE_REQUIRE(delta ? (step && rate_log && step_bias && unit_eps > 0.f && (vec_dtype == kF32 || vec_dtype == kBF16) && !coef && !decay && !cos_table)
                        : ((decay != nullptr) != (coef != nullptr)),
                  "chunked_memory: the delta rule needs strengths, step sizes and rates, anything else fixed decays or gates");
    LEONE_REQUIRE((coef != nullptr) == (dot != nullptr), "chunked_memory: gates come with a place for the normaliser's read-out");
    LEONE_REQUIRE((cos_table == nullptr) == (sin_table == nullptr) &&
                      (!cos_table || (positions && rotary_dim > 0 && rotary_dim % 2 == 0 && rotary_dim <= dim && table_positions > 0)),
                  "chunked_memory: a rotation of %d of %d elements from tables of %d positions", rotary_dim, dim, table_positions);
    LEONE_REQUIRE(heads > 0 && heads <= 65535 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && dim <= (delta ? kChunkMaxDeltaDim : kChunkMaxDim) &&
                      vdim > 0 && vdim < 16 * 65535,
                  "chunked_memory: %d heads over %d key heads of %d x %d (at most %d key channels)", heads, kv_heads, dim, vdim,
                  delta ? kChunkMaxDeltaDim : kChunkMaxDim);
    LEONE_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && stride >= q_off + static_cast<long>(kv_heads) * dim &&
                  stride >= k_off + static_cast<long>(kv_heads) * dim && stride >= v_off + static_cast<long>(heads) * vdim &&
                  (!delta || (beta_stride >= heads && step_stride >= static_cast<long>(heads) * (step_each ? dim : 1))),
                  "chunked_memory: rows of %ld do not hold the named columns", stride);
    LEONE_REQUIRE(head_stride >= static_cast<long>(dim) * vdim + (coef ? dim : 0) && slot_stride >= heads * head_stride,
                  "chunked_memory: states of %ld floats do not fit", slot_stride);
    LEONE_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0, "chunked_memory: the workspace must be aligned to 16 bytes");
    ChunkArgs a{};
    a.rows = rows, a.stride = stride, a.q_off = q_off, a.k_off = k_off, a.v_off = v_off, a.silu = silu;
    a.q_scale = q_scale, a.k_scale = k_scale, a.unit_eps = unit_eps;
    a.beta = beta, a.beta_stride = beta_stride, a.step = step, a.step_stride = step_stride;
    a.rate_log = AnyVec{rate_log, vec_dtype}, a.step_bias = AnyVec{step_bias, vec_dtype}, a.decay = decay, a.coef = coef;
    a.cos_table = cos_table, a.sin_table = sin_table, a.positions = positions, a.rot_half = rotary_dim / 2, a.table_positions = table_positions;
    a.chunks = chunks, a.links = links, a.state = state, a.slot_stride = slot_stride, a.head_stride = head_stride;
    a.write_state = write_state, a.out = out, a.dot = dot;
    a.heads = heads, a.kv_heads = kv_heads, a.dim = dim, a.vdim = vdim;
    const int tiles = chunk_tiles(dim);
    a.dim_p = 64 * tiles, a.vdim_p = ceil_div(vdim + (dot ? 1 : 0), 16) * 16;
    const long each = static_cast<long>(n_chunks) * heads * kChunkRows;
    a.q_in = workspace;
    a.k_out = a.q_in + each * a.dim_p;
    a.values = a.k_out + each * a.dim_p;
    a.mix = a.values + each * a.vdim_p;
    a.solved_k = a.mix + each * kChunkRows;
    a.total = a.solved_k + (delta ? each * a.dim_p : 0);
    const size_t row = (a.dim_p + 4) * sizeof(float);
    const dim3 prepare(n_chunks, heads, delta ? ceil_div(a.vdim_p, a.dim_p) : 1), walk(n_links, heads, a.vdim_p / 16);
    if (rule == kChunkDeltaChannel) {
        const size_t shared = 3 * kChunkRows * row + (kChunkTiles * 256 + 3 * (kChunkRows / 16) * a.dim_p) * sizeof(float);
        if (tiles == 1 ? launch_prepare(chunk_prepare_channel_kernel<1>, prepare, shared, a, stream)
                       : launch_prepare(chunk_prepare_channel_kernel<2>, prepare, shared, a, stream)) return 1;
        if (tiles == 1) chunk_walk_kernel<true, 1, true><<<walk, kChunkThreads, 0, stream>>>(a);
        else chunk_walk_kernel<true, 2, true><<<walk, kChunkThreads, 0, stream>>>(a);
    } else if (rule == kChunkDelta) {
        const size_t shared = 2 * kChunkRows * row + kChunkTiles * 256 * sizeof(float);
        if (tiles == 1 ? launch_prepare(chunk_prepare_kernel<true, 1>, prepare, shared, a, stream)
                       : launch_prepare(chunk_prepare_kernel<true, 2>, prepare, shared, a, stream)) return 1;
        if (tiles == 1) chunk_walk_kernel<true, 1, false><<<walk, kChunkThreads, 0, stream>>>(a);
        else chunk_walk_kernel<true, 2, false><<<walk, kChunkThreads, 0, stream>>>(a);
    } else {
        const size_t shared = 2 * kChunkRows * row;
        if (tiles == 1 ? launch_prepare(chunk_prepare_kernel<false, 1>, prepare, shared, a, stream)
            : tiles == 2 ? launch_prepare(chunk_prepare_kernel<false, 2>, prepare, shared, a, stream)
                         : launch_prepare(chunk_prepare_kernel<false, 4>, prepare, shared, a, stream)) return 1;
        if (tiles == 1) chunk_walk_kernel<false, 1, false><<<walk, kChunkThreads, 0, stream>>>(a);
        else if (tiles == 2) chunk_walk_kernel<false, 2, false><<<walk, kChunkThreads, 0, stream>>>(a);
        else chunk_walk_kernel<false, 4, false><<<walk, kChunkThreads, 0, stream>>>(a);
    }
    LEONE_LAUNCH_CHECK("chunk_walk");
    return 0;
}
