// Attention over the paged cache in single precision, on the float matrix instructions: the function of
// attention_rows_kernel (attention.hip; scores, softmax and sums in float) for heads of 64 or 128 elements.
//
// A query row alone reads every key for itself, which bounds a row by the walk along its keys (one dot product and one
// step of the softmax a key).  Here a workgroup takes up to 16 queries that read the same keys - the query heads of one
// kv head, of a few neighbouring rows of one request - and its waves share out the keys, 16 at a time, in eight shares with a
// running softmax each; the shares' results are merged through shared memory in a fixed order.  What bounds it is
// the matrix instructions: 64 of 32 cycles for 16 keys of 128 elements, whose loads (16 KB a wave) are in flight meanwhile.
//
// A row's result depends on its own query and on the keys that it sees alone, to the bit, whichever rows share the workgroup or the
// launch: a tile of keys belongs to a share by the keys' positions, a share's tiles are taken in their order, and tiles that a row
// does not see add nothing to it.
//
// Lane l of a wave holds, of a product, row or column l % 16, and inner elements 4 (l / 16) .. + 3 of every 16: with the
// cache's runs of 8 a 16-byte load a lane brings 16 keys x 16 elements, or 16 value elements x 16 tokens.  Scores are made
// as keys x queries, so that a lane's four scores belong to its own query and to the four keys it holds values of: they
// are the operand of the second product as they stand.
//
// Everything that is the same for a wave (its share, the tile, the page) is in scalar registers, and a tile that every row sees whole
// needs neither masks nor a look for values that are no numbers: of the instructions between the products, which the other wave of a
// SIMD has to cover, that is a third.
//
// Measured (us; with those, the row kernel of attention.hip): 16 heads over 4 of 128 elements, one row at 780 keys 23.5 (24.9, 314; 15.1 with a
// workgroup a share, below), a prompt
// of 777 rows 64 (71, 1375), of 2,048 rows 260 (292, 8589).
#include "common.h"
#include "leone_hip.h"
#include "score_shape.h"

#include <math.h>

namespace leone {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kQueries = 16;
constexpr int kKeys = 16;
constexpr int kShares = 8;

struct AttentionF32Args {
    const float* q;
    float* out;
    const float* k_pool;
    const float* v_pool;
    const int* positions;
    const int* row_entry;
    const int* block_table;
    int max_blocks, rows, q_heads, kv_heads, group, most;      // most: rows that a workgroup takes
    unsigned multiples_inverse;                                // 2^32 / (rows / most, rounded up), rounded up; 0: divide
    int page_tokens, page_shift;                               // page_shift: -1 if page_tokens is no power of two
    float scale;
    int window;
    const float* gate;
    long gate_stride;
    int keep_first, gate_each;
    const float* slopes;
    float temp_coef;
    int temp_every;
    ScoreShape shape;
    int chunk;
};

// The end of a row: its query's sums over the denominator, turned back, behind their gate.  Lane l of a wave has elements h .. h + 3, h = 4 (l /
// 16), of the kCount runs of 16 from `first` on, kStep runs apart (a run's partner for turning is kCount / 2 further).
template <int kDim, int kCount, int kStep>
__device__ inline void finish_row(const AttentionF32Args& g, f32x4 (&result)[kCount], int first, float denom, int row, int head, int pos,
                                  int lane, bool real) {
    static_assert(kCount * kStep * 16 == kDim, "the runs are every kStep-th of the head's");
    const int h = (lane / 16) * 4;
#pragma unroll
    for (int i = 0; i < kCount; ++i) result[i] /= denom;
    if (g.shape.turn_cos) {
        f32x4 turned[kCount];
#pragma unroll
        for (int i = 0; i < kCount; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float partner = g.shape.turn_pairing ? result[i][r ^ 1] : result[(i + kCount / 2) % kCount][r];
                turned[i][r] = turned_back(result[i][r], partner, (first + i * kStep) * 16 + h + r, kDim, pos, g.shape);
            }
#pragma unroll
        for (int i = 0; i < kCount; ++i) result[i] = turned[i];
    }
    if (!real) return;
    float* orow = g.out + (static_cast<long>(row) * g.q_heads + head) * kDim;
    const float* gate_row = g.gate ? g.gate + static_cast<long>(row) * g.gate_stride + (g.gate_each ? static_cast<long>(head) * kDim : head) : nullptr;
    const float open_head = (g.gate && !g.gate_each) ? 1.0f / (1.0f + expf(-gate_row[0])) : 1.0f;
#pragma unroll
    for (int i = 0; i < kCount; ++i) {
        const int at = (first + i * kStep) * 16 + h;
        f32x4 open = {open_head, open_head, open_head, open_head};
        if (g.gate && g.gate_each) {
#pragma unroll
            for (int r = 0; r < 4; ++r) open[r] = 1.0f / (1.0f + expf(-gate_row[at + r]));
        }
        *reinterpret_cast<f32x4*>(orow + at) = result[i] * open;
    }
}

// kWaves waves with kShares / kWaves shares each.
template <int kDim, int kWaves>
__global__ void __launch_bounds__(kWaves * kWave, kDim == 64 ? 3 : 2) attention_f32_kernel(const AttentionF32Args g) {
    constexpr int kRuns = kDim / 16, kOwn = kShares / kWaves;
    __shared__ float sm_m[kShares][kQueries], sm_l[kShares][kQueries];
    __shared__ f32x4 sm_acc[kWaves / 2][kRuns][kWave];

    // The rows of this workgroup: from this one on, those of the same request up to the next multiple of `most`; the
    // workgroups of the rows that another one takes have nothing to do.  Rows are numbered so that those at the multiples come first,
    // one behind the other: workgroups go to the eight dies in turn, and every 4th or 16th would have left the work of a portion to one
    // or two of them (2,048 rows of 16 heads over 4 of 128: 1330 us, numbered so 295).
    const int group = g.group, most = g.most;
    const int multiples = (g.rows + most - 1) / most;
    const int turn = multiples == 1 ? blockIdx.x : g.multiples_inverse ? __umulhi(blockIdx.x, g.multiples_inverse) : blockIdx.x / multiples;
    const int first_row = (blockIdx.x - turn * multiples) * most + turn, kvh = blockIdx.y;       // (turn 0: a multiple of `most`)
    if (first_row >= g.rows) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int mine = lane % 16, h = (lane / 16) * 4;

    // A lane's query, if the workgroup takes so many rows (past the last row it is the last one again), is asked for ahead of what the
    // rows are; that comes by scalar loads where, as in decoding, the row is alone.
    const auto clamped = [&](int row) { return row < g.rows ? row : g.rows - 1; };
    const int place = mine / group;                           // which of the rows this lane's query belongs to
    const int row = clamped(first_row + place), head = kvh * group + (mine - place * group);
    const int entry = g.row_entry[first_row], entry_before = g.row_entry[first_row > 0 ? first_row - 1 : 0];
    const int entry_after = g.row_entry[clamped(first_row + 1)], first_pos = g.positions[first_row];
    if (turn != 0 && entry_before == entry) return;
    // rows of the same request, one behind the other, up to the next multiple
    const int room = most - turn < g.rows - first_row ? most - turn : g.rows - first_row;
    int count = 1, pos = first_pos;
    if (room > 1 && entry_after == entry) {
        const unsigned others = static_cast<unsigned>(__ballot(g.row_entry[clamped(first_row + mine)] != entry)) & 0xffffu;
        const int same = others ? __builtin_ctz(others) : 16;
        count = same < room ? same : room;
        pos = g.positions[first_row + (place < count ? place : count - 1)];
    }
    // lanes past the last query stand where the last row does and write nothing
    const bool real = mine < count * group;
    f32x4 q[kRuns];
    {
        const float* qr = g.q + (static_cast<long>(row) * g.q_heads + head) * kDim;
#pragma unroll
        for (int i = 0; i < kRuns; ++i) q[i] = *reinterpret_cast<const f32x4*>(qr + i * 16 + h);
    }
    float scale = g.scale;
    if (g.temp_every > 0) scale *= 1.0f + g.temp_coef * logf(static_cast<float>((pos + 1) / g.temp_every + 1));
    const float slope = g.slopes ? g.slopes[head] : 0.f;
    const int first = first_key(pos, g.window, g.chunk);

    // what the rows together see: tiles of 16 keys from the earliest row's first one on, and those of the kept first keys
    // and what each of them sees: a tile between the two needs no masks
    int low = __builtin_amdgcn_readfirstlane(first), high = __builtin_amdgcn_readfirstlane(pos), whole_from = low, whole_to = high;
    if (count > 1) {
        const auto least = [](int v) { return __builtin_amdgcn_readfirstlane(join_span<16>(v, [](int a, int b) { return min(a, b); })); };
        const auto most_of = [](int v) { return __builtin_amdgcn_readfirstlane(join_span<16>(v, [](int a, int b) { return max(a, b); })); };
        low = least(first), high = most_of(pos), whole_from = most_of(first), whole_to = least(pos);
    }
    const int low_tile = low / kKeys;
    const int kept_tiles = min((g.keep_first + kKeys - 1) / kKeys, low_tile);
    const int tiles = high / kKeys + 1;
    const int* table = g.block_table + static_cast<long>(entry) * g.max_blocks;
    const long page_floats = static_cast<long>(g.page_tokens) * kDim;
    const auto page_of = [&](int key) { return g.page_shift >= 0 ? key >> g.page_shift : key / g.page_tokens; };

    f32x4 kf[kRuns], vf[kRuns], acc[kRuns] = {};
    [[maybe_unused]] f32x4 ready[kOwn == 2 ? kRuns : 1];      // the first of two shares
    float m = -INFINITY, l = 0.f;
    bool mapped = true, mapped_next = true;
    // share n's tiles are those whose number is n modulo kShares, wave w has the shares that are w modulo kWaves; past the kept
    // tiles, from the first that a row sees on
    const auto skip = [&](int t) { return t < kept_tiles || t >= low_tile ? t : t + (low_tile - t + kShares - 1) / kShares * kShares; };
    int in_page = 0;                              // of the tile that is fetched: its first key's place in its page
    const auto block_of = [&](int start, bool& there) {
        const int block = page_of(start), page = table[block];
        in_page = start - block * g.page_tokens;
        there = page >= 0;
        return (static_cast<long>(there ? page : 0) * g.kv_heads + kvh) * page_floats;
    };
    const long run_step = 2l * g.page_tokens * 8;             // from a key's 16 elements to its next
    const int key_lane = (h / 8) * g.page_tokens * 8 + mine * 8 + h % 8, value_lane = ((h / 8) * kDim + mine) * 8 + h % 8;
    const auto fetch_keys = [&](long block) {
        const float* at = g.k_pool + block + in_page * 8 + key_lane;
#pragma unroll
        for (int i = 0; i < kRuns; ++i) kf[i] = *reinterpret_cast<const f32x4*>(at + i * run_step);
    };
    const auto fetch_values = [&](long block, int first_place) {
        const float* at = g.v_pool + block + static_cast<long>(first_place) * kDim + value_lane;      // (a tile begins a run of 8)
#pragma unroll
        for (int i = 0; i < kRuns; ++i) vf[i] = *reinterpret_cast<const f32x4*>(at + i * 128);
    };
#pragma unroll 1
    for (int own = wave; own < kShares; own += kWaves) {
        if constexpr (kOwn == 2) {
            if (own != wave) {
#pragma unroll
                for (int i = 0; i < kRuns; ++i) {
                    ready[i] = acc[i];
                    acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                m = -INFINITY, l = 0.f;
                mapped = true;
            }
        }
        int t = skip(own);
        long block = 0;
        if (t < tiles) {
            block = block_of(t * kKeys, mapped);
            fetch_keys(block);
        }
        while (t < tiles) {
            const int start = t * kKeys;
            t = skip(t + kShares);
            fetch_values(block, in_page);
            // whether every row sees all of the tile's keys
            const bool whole = mapped && start + kKeys - 1 <= whole_to && (start >= whole_from || start + kKeys <= g.keep_first);
            f32x4 dots[4] = {};                   // four sums side by side: no instruction waits for the one before it
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) dots[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][j], q[i][j], dots[j], 0, 0, 0);
            f32x4 s = (dots[0] + dots[1]) + (dots[2] + dots[3]);
            if (t < tiles) {                      // the keys' registers are free: the next tile's are on their way from here on
                block = block_of(t * kKeys, mapped_next);
                fetch_keys(block);
            }
            float top = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = start + h + r;
                const bool seen = whole || (key <= pos && (key >= first || key < g.keep_first));
                float v = s[r] * scale;
                if (g.shape.cap > 0.f) v = g.shape.cap * tanhf(v / g.shape.cap);
                v -= slope * static_cast<float>(pos - key);
                // an unmapped block poisons the result of every row that sees it
                s[r] = seen ? (mapped ? v : __builtin_nanf("")) : -INFINITY;
                top = fmaxf(top, s[r]);
            }
            top = max_lanes<16>(top);
            top = max_lanes<32>(top);
            const float m_new = fmaxf(m, top);
            const float reference = m_new == -INFINITY ? 0.f : m_new;      // nothing seen yet: every weight is 0
            const float alpha = expf(m - reference);
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[r] = expf(s[r] - reference);
                sum += s[r];
            }
            sum = add_lanes<16>(sum);
            sum = add_lanes<32>(sum);
            l = l * alpha + sum;
            m = m_new;
            if (!mapped || start + kKeys > high + 1) {       // places nobody has written: their weight is 0, but not what they may hold
#pragma unroll
                for (int i = 0; i < kRuns; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (!mapped || start + h + r > high) vf[i][r] = 0.f;
            }
            {
#pragma unroll
                for (int i = 0; i < kRuns; ++i) acc[i] *= alpha;
            }
            bool odd_value = false;
            if (!whole) {
                f32x4 odd = {0.f, 0.f, 0.f, 0.f};            // stays 0 unless a value is infinite or NaN
#pragma unroll
                for (int i = 0; i < kRuns; ++i) odd += vf[i] * 0.f;
                odd_value = __any(!(odd[0] + odd[1] + odd[2] + odd[3] == 0.f));
            }
            if (odd_value) {
                // such a value is for the rows that see it, and no weight of 0 keeps it from the others: one key after the other, in
                // the order of the instructions below
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll 1
                    for (int from = 0; from < 4; ++from) {
                        const int key = start + 4 * from + j;
                        const bool seen = key <= pos && (key >= first || key < g.keep_first);
                        const float p = __shfl(s[j], from * 16 + mine, kWave);
#pragma unroll
                        for (int i = 0; i < kRuns; ++i)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const float v = __shfl(vf[i][j], from * 16 + h + r, kWave);
                                if (seen) acc[i][r] = fmaf(p, v, acc[i][r]);
                            }
                    }
            } else {
#pragma unroll
                for (int i = 0; i < kRuns; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][j], s[j], acc[i], 0, 0, 0);
            }
            mapped = mapped_next;
        }
        if (lane < kQueries) {
            sm_m[own][lane] = m;
            sm_l[own][lane] = l;
        }
    }

    // ---- the shares' results, merged: by halves, a share's result rounded before it is added --------------------------
    __syncthreads();
    float top = sm_m[0][mine];
#pragma unroll
    for (int w = 1; w < kShares; ++w) top = fmaxf(top, sm_m[w][mine]);
    const float sink = g.shape.sinks ? g.shape.sinks[head] : -INFINITY;
    top = fmaxf(top, sink);
    const auto weight = [&](float of) { return of == -INFINITY ? 0.f : expf(of - top); };
    float denom = g.shape.sinks ? expf(sink - top) : 0.f;
#pragma unroll
    for (int w = 0; w < kShares; ++w) denom += sm_l[w][mine] * weight(sm_m[w][mine]);
    f32x4 result[kRuns];
    {
#pragma clang fp contract(off)
        static_assert(kOwn <= 2 && kShares == kOwn * kWaves, "a wave's two shares are the first halves that meet");
        const float own = weight(m);
#pragma unroll
        for (int i = 0; i < kRuns; ++i) result[i] = acc[i] * own;
        if constexpr (kOwn == 2) {
            const float first_own = weight(sm_m[wave][mine]);
#pragma unroll
            for (int i = 0; i < kRuns; ++i) result[i] = ready[i] * first_own + result[i];
        }
#pragma unroll
        for (int half = kWaves / 2; half > 0; half /= 2) {
            if (wave >= half && wave < 2 * half) {
#pragma unroll
                for (int i = 0; i < kRuns; ++i) sm_acc[wave - half][i][lane] = result[i];
            }
            __syncthreads();
            if (wave < half) {
#pragma unroll
                for (int i = 0; i < kRuns; ++i) result[i] += sm_acc[wave][i][lane];
            }
            __syncthreads();
        }
    }
    if (wave != 0) return;
    finish_row<kDim, kRuns, 1>(g, result, 0, denom, row, head, pos, lane, real);
}

// ---- few rows: a workgroup a share -----------------------------------------------------------------------------------------
//
// With a workgroup a row and kv head a step of one request uses as many units as there are kv heads.  Here every share of a row's keys has a
// workgroup of its own, and what bounds it are the instructions of its waves, each alone on its SIMD (some five cycles apiece): so its four
// waves take four tiles at a time, make the scores of one each, tell each other the tiles' highest scores, weigh their own tile, and then add up
// the values of all four, a quarter of the runs each.  (All four waves on one tile, a quarter of each product apiece, repeated the softmax in
// every wave: 18.7 us where this takes 15.1.)  16 heads over 4 of 128 elements, one row at 300, 780 and 4,000 keys, both launches: 10.5, 15.1 and
// 42 us; with a workgroup a row and kv head 13.2, 23.5 and 88.  Sums, shares and the order in which they are merged are attention_f32_kernel's: the results are the same bits.
constexpr int kPartWaves = 4;

// Waits for what this wave has put into shared memory and read from it, not for its loads from memory.
__device__ inline void shares_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int kDim>
__global__ void __launch_bounds__(kPartWaves * kWave) attention_f32_share_kernel(const AttentionF32Args g, float* part_acc, float* part_ml) {
    constexpr int kRuns = kDim / 16, kOwnRuns = kRuns / kPartWaves;
    __shared__ float sm_top[kPartWaves][kQueries], sm_alpha[kPartWaves][kQueries], sm_sum[kPartWaves][kQueries];
    __shared__ f32x4 sm_s[kPartWaves][kWave];
    const int own = blockIdx.x, row = blockIdx.y, kvh = blockIdx.z, group = g.group;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int mine = lane % 16, h = (lane / 16) * 4;
    const int entry = g.row_entry[row], pos = g.positions[row];
    const int head = kvh * group + (mine < group ? mine : group - 1);
    f32x4 q[kRuns];
    {
        const float* qr = g.q + (static_cast<long>(row) * g.q_heads + head) * kDim + h;
#pragma unroll
        for (int i = 0; i < kRuns; ++i) q[i] = *reinterpret_cast<const f32x4*>(qr + i * 16);
    }
    float scale = g.scale;
    if (g.temp_every > 0) scale *= 1.0f + g.temp_coef * logf(static_cast<float>((pos + 1) / g.temp_every + 1));
    const float slope = g.slopes ? g.slopes[head] : 0.f;
    const int first = first_key(pos, g.window, g.chunk);
    const int low_tile = first / kKeys, kept_tiles = min((g.keep_first + kKeys - 1) / kKeys, low_tile), tiles = pos / kKeys + 1;
    // the share's tiles, numbered: first those of the kept keys, then those from the first that the row sees
    const int kept = own < kept_tiles ? (kept_tiles - own + kShares - 1) / kShares : 0;
    const int base = own >= low_tile ? own : own + (low_tile - own + kShares - 1) / kShares * kShares;
    const int count = kept + (base < tiles ? (tiles - base + kShares - 1) / kShares : 0);
    const auto start_of = [&](int n) { return (n < kept ? own + kShares * n : base + kShares * (n - kept)) * kKeys; };

    f32x4 acc[kOwnRuns] = {};
    float m = -INFINITY, l = 0.f;
    if (count > 0) {
        const int* table = g.block_table + static_cast<long>(entry) * g.max_blocks;
        const long page_floats = static_cast<long>(g.page_tokens) * kDim, run_step = 2l * g.page_tokens * 8;
        const auto page_of = [&](int key) { return g.page_shift >= 0 ? key >> g.page_shift : key / g.page_tokens; };
        const int key_lane = (h / 8) * g.page_tokens * 8 + mine * 8 + h % 8, value_lane = ((h / 8) * kDim + mine) * 8 + h % 8 + wave * kOwnRuns * 128;
        f32x4 kf[kRuns], vf[kPartWaves][kOwnRuns];
        // four tiles: their starts, their pages' places, whether they have one (past the last tile that one again, unused)
        struct Four {
            int start[kPartWaves], in_page[kPartWaves];
            long block[kPartWaves];
            bool mapped[kPartWaves];
        };
        int pages = 0;                                        // of 64 tiles, a lane each
        const auto four_from = [&](int n0) {
            if (n0 % kWave == 0) {
                pages = table[page_of(start_of(min(n0 + lane, count - 1)))];
                asm volatile("" : "+v"(pages));               // waited for here: behind a join, every load in flight would be waited for
            }
            Four f;
#pragma unroll
            for (int t = 0; t < kPartWaves; ++t) {
                const int n = min(n0 + t, count - 1), page = __builtin_amdgcn_readlane(pages, n % kWave);
                f.start[t] = start_of(n);
                f.in_page[t] = f.start[t] - page_of(f.start[t]) * g.page_tokens;
                f.mapped[t] = page >= 0;
                f.block[t] = (static_cast<long>(page >= 0 ? page : 0) * g.kv_heads + kvh) * page_floats;
            }
            return f;
        };
        const auto pick = [&](const auto& of) { return wave == 0 ? of[0] : wave == 1 ? of[1] : wave == 2 ? of[2] : of[3]; };
        const auto fetch_keys = [&](const Four& f) {
            const float* at = g.k_pool + pick(f.block) + pick(f.in_page) * 8 + key_lane;
#pragma unroll
            for (int i = 0; i < kRuns; ++i) kf[i] = *reinterpret_cast<const f32x4*>(at + i * run_step);
        };
        const auto fetch_values = [&](const Four& f) {
#pragma unroll
            for (int t = 0; t < kPartWaves; ++t) {
                const float* at = g.v_pool + f.block[t] + static_cast<long>(f.in_page[t]) * kDim + value_lane;
#pragma unroll
                for (int i = 0; i < kOwnRuns; ++i) vf[t][i] = *reinterpret_cast<const f32x4*>(at + i * 128);
            }
        };
        Four four = four_from(0);
        fetch_keys(four);
        fetch_values(four);
        for (int n0 = 0; n0 < count; n0 += kPartWaves) {
            const int here = min(count - n0, kPartWaves);
            f32x4 dots[4] = {};
#pragma unroll
            for (int i = 0; i < kRuns; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) dots[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][j], q[i][j], dots[j], 0, 0, 0);
            f32x4 s = (dots[0] + dots[1]) + (dots[2] + dots[3]);
            const bool more = n0 + kPartWaves < count;
            Four next = four;
            if (more) {
                next = four_from(n0 + kPartWaves);
                fetch_keys(next);
            }
            const int start = pick(four.start);
            const bool there = pick(four.mapped);
            const auto whole_at = [&](int at, bool is) { return is && at + kKeys - 1 <= pos && (at >= first || at + kKeys <= g.keep_first); };
            const bool whole = whole_at(start, there);
            float top = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = s[r] * scale;
                if (g.shape.cap > 0.f) v = g.shape.cap * tanhf(v / g.shape.cap);
                if (g.slopes) v -= slope * static_cast<float>(pos - (start + h + r));
                s[r] = v;
            }
            if (!whole) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = start + h + r;
                    const bool seen = key <= pos && (key >= first || key < g.keep_first);
                    s[r] = seen ? (there ? s[r] : __builtin_nanf("")) : -INFINITY;
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) top = fmaxf(top, s[r]);
            top = max_lanes<16>(top);
            top = max_lanes<32>(top);
            if (lane < kQueries) sm_top[wave][lane] = top;
            shares_barrier();
            // the running maximum through the four tiles; this wave's tile is weighed by what it has come to there
            float m_before = m, m_own = m;
#pragma unroll
            for (int t = 0; t < kPartWaves; ++t) {
                if (t == wave) m_before = m;
                if (t < here) m = fmaxf(m, sm_top[t][mine]);
                if (t == wave) m_own = m;
            }
            const float reference = m_own == -INFINITY ? 0.f : m_own;      // nothing seen yet: every weight is 0
            const float alpha = expf(m_before - reference);
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[r] = expf(s[r] - reference);
                sum += s[r];
            }
            sum = add_lanes<16>(sum);
            sum = add_lanes<32>(sum);
            sm_s[wave][lane] = s;
            if (lane < kQueries) {
                sm_alpha[wave][lane] = alpha;
                sm_sum[wave][lane] = sum;
            }
            shares_barrier();
#pragma unroll
            for (int t = 0; t < kPartWaves; ++t) {
                if (t >= here) break;
                const float alpha_t = sm_alpha[t][mine];
                const f32x4 s_t = sm_s[t][lane];
                l = l * alpha_t + sm_sum[t][mine];
                f32x4 (&v)[kOwnRuns] = vf[t];
                const int at = four.start[t];
                const bool whole_t = whole_at(at, four.mapped[t]);
                bool odd_value = false;
                if (!whole_t) {
                    if (!four.mapped[t] || at + kKeys > pos + 1) {         // places nobody has written
#pragma unroll
                        for (int i = 0; i < kOwnRuns; ++i)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (!four.mapped[t] || at + h + r > pos) v[i][r] = 0.f;
                    }
                    f32x4 odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int i = 0; i < kOwnRuns; ++i) odd += v[i] * 0.f;
                    odd_value = __any(!(odd[0] + odd[1] + odd[2] + odd[3] == 0.f));
                }
#pragma unroll
                for (int i = 0; i < kOwnRuns; ++i) acc[i] *= alpha_t;
                if (odd_value) {                              // not a number where the row does not see it: see above
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll 1
                        for (int from = 0; from < 4; ++from) {
                            const int key = at + 4 * from + j;
                            const bool seen = key <= pos && (key >= first || key < g.keep_first);
                            const float p = __shfl(s_t[j], from * 16 + mine, kWave);
#pragma unroll
                            for (int i = 0; i < kOwnRuns; ++i)
#pragma unroll
                                for (int r = 0; r < 4; ++r) {
                                    const float each = __shfl(v[i][j], from * 16 + h + r, kWave);
                                    if (seen) acc[i][r] = fmaf(p, each, acc[i][r]);
                                }
                        }
                } else {
#pragma unroll
                    for (int i = 0; i < kOwnRuns; ++i)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i][j], s_t[j], acc[i], 0, 0, 0);
                }
            }
            if (more) fetch_values(next);
            four = next;
        }
    }
    const long place = (static_cast<long>(row) * g.kv_heads + kvh) * kShares + own;
    if (wave == 0 && lane < kQueries) {
        part_ml[(place * 2) * kQueries + lane] = m;
        part_ml[(place * 2 + 1) * kQueries + lane] = l;
    }
#pragma unroll
    for (int i = 0; i < kOwnRuns; ++i)
        reinterpret_cast<f32x4*>(part_acc)[(place * kRuns + wave * kOwnRuns + i) * kWave + lane] = acc[i];
}

// The shares' results of a row and kv head, merged as attention_f32_kernel merges them; wave w takes runs w and w + half of them.
template <int kDim>
__global__ void __launch_bounds__(kDim / 32 * kWave) attention_f32_join_kernel(const AttentionF32Args g, const float* part_acc, const float* part_ml) {
    constexpr int kRuns = kDim / 16;
    const int row = blockIdx.x, kvh = blockIdx.y, group = g.group;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, mine = lane % 16;
    const int head = kvh * group + (mine < group ? mine : group - 1);
    const long place = (static_cast<long>(row) * g.kv_heads + kvh) * kShares;
    f32x4 acc[kShares][2];
    float ms[kShares], ls[kShares];
#pragma unroll
    for (int w = 0; w < kShares; ++w) {
        ms[w] = part_ml[((place + w) * 2) * kQueries + mine];
        ls[w] = part_ml[((place + w) * 2 + 1) * kQueries + mine];
    }
#pragma unroll
    for (int w = 0; w < kShares; ++w)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            acc[w][i] = reinterpret_cast<const f32x4*>(part_acc)[((place + w) * kRuns + wave + i * (kRuns / 2)) * kWave + lane];
    const int pos = g.positions[row];
    float top = ms[0];
#pragma unroll
    for (int w = 1; w < kShares; ++w) top = fmaxf(top, ms[w]);
    const float sink = g.shape.sinks ? g.shape.sinks[head] : -INFINITY;
    top = fmaxf(top, sink);
    const auto weight = [&](float of) { return of == -INFINITY ? 0.f : expf(of - top); };
    float denom = g.shape.sinks ? expf(sink - top) : 0.f;
    float weights[kShares];
#pragma unroll
    for (int w = 0; w < kShares; ++w) {
        weights[w] = weight(ms[w]);
        denom += ls[w] * weights[w];
    }
    {
#pragma clang fp contract(off)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int w = 0; w < kShares; ++w) acc[w][i] = acc[w][i] * weights[w];
#pragma unroll
            for (int half = kShares / 2; half > 0; half /= 2)
#pragma unroll
                for (int w = 0; w < half; ++w) acc[w][i] = acc[w][i] + acc[w + half][i];
        }
    }
    finish_row<kDim, 2, kRuns / 2>(g, acc[0], wave, denom, row, head, pos, lane, mine < group);
}

// Whether the kernel takes this shape: 16-byte rows of q and of the results follow from the head's size, tiles of 16 keys lie
// within a page, and a kv head's query heads fit one tile.  Everything else is the row kernel's.
bool attention_f32_takes(const void* q, const void* out, const void* k_pool, const void* v_pool, int q_heads, int kv_heads, int head_dim,
                         int v_dim, int page_tokens) {
    const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return (head_dim == 64 || head_dim == 128) && v_dim == head_dim && page_tokens % kKeys == 0 && q_heads / kv_heads <= kQueries &&
           kv_heads <= 65535 && aligned(q) && aligned(out) && aligned(k_pool) && aligned(v_pool);
}

void launch_attention_f32(const float* q, float* out, const float* k_pool, const float* v_pool, const int* positions, const int* row_entry,
                          const int* block_table, int max_blocks, int rows, int q_heads, int kv_heads, int head_dim, int page_tokens,
                          float scale, int window, const float* gate, long gate_stride, int keep_first, int gate_each,
                          const float* slopes, float temp_coef, int temp_every, const ScoreShape& shape, int chunk, float* part_acc,
                          float* part_ml, hipStream_t stream) {
    const int group = q_heads / kv_heads, most = kQueries / group;
    const long multiples = ceil_div(rows, most);
    const int page_shift = (page_tokens & (page_tokens - 1)) == 0 ? __builtin_ctz(page_tokens) : -1;
    const AttentionF32Args args{q, out, k_pool, v_pool, positions, row_entry, block_table, max_blocks, rows, q_heads, kv_heads,
                                group, most, multiples > 1 && multiples * (rows + kQueries) < 1l << 32 ? static_cast<unsigned>(((1ull << 32) + multiples - 1) / multiples) : 0u,
                                page_tokens, page_shift, scale, window, gate, gate_stride, keep_first, gate_each, slopes, temp_coef, temp_every,
                                shape, chunk};
    if (part_acc && part_ml && rows <= 65535) {
        const dim3 shares(kShares, rows, kv_heads), joined(rows, kv_heads);
        if (head_dim == 128) {
            attention_f32_share_kernel<128><<<shares, kPartWaves * kWave, 0, stream>>>(args, part_acc, part_ml);
            attention_f32_join_kernel<128><<<joined, 4 * kWave, 0, stream>>>(args, part_acc, part_ml);
        } else {
            attention_f32_share_kernel<64><<<shares, kPartWaves * kWave, 0, stream>>>(args, part_acc, part_ml);
            attention_f32_join_kernel<64><<<joined, 2 * kWave, 0, stream>>>(args, part_acc, part_ml);
        }
        return;
    }
    const dim3 grid(ceil_div(rows, most) * most, kv_heads);
    // Eight waves, a share each, where the launch is small or heads are of 128 elements; four waves with two shares each for many
    // rows of 64, whose workgroups are short (us, eight waves and four: 8 heads over 2, 1,500 rows 66 and 58, 300 decoded rows at 500
    // keys 38 and 32; 16 over 8, 777 rows 57 and 45; but 300 rows behind 1,200 keys of 8 over 2 30 and 48, which the host cannot tell
    // from decoded rows).  As many workgroups are launched as there are rows: those of the rows that share one leave at once.
    if (head_dim == 128) attention_f32_kernel<128, 8><<<grid, 8 * kWave, 0, stream>>>(args);
    else if (static_cast<long>(rows) * kv_heads < 512) attention_f32_kernel<64, 8><<<grid, 8 * kWave, 0, stream>>>(args);
    else attention_f32_kernel<64, 4><<<grid, 4 * kWave, 0, stream>>>(args);
}

}  // namespace leone
