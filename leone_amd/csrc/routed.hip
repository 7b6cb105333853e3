// A feed-forward of routed experts: the router's choice, the rows sorted by expert, the experts' products.
//
//   route_topk   scores s = softmax(z) over all router outputs (float); choice scores s + correction; experts in
//                equal groups of neighbours, a group's score its best choice score, only the best `keep` groups
//                stay open (the others count as minus infinity); the `top` best open choice scores win; the
//                weights are the winners' s over their sum (+ 1e-20).
//   moe_plan     the (row, place) pairs of every expert gathered into tiles of pairs of one expert.
//   route_plan   both in one launch of one workgroup, for steps of few rows; experts that every row takes with
//                weight 1 (a shared expert cut to the experts' size) may stand behind the routed ones.
//   moe_product  gated: act(W_gate x) * (W_up x) of every pair, by its expert's matrices; plain (experts without a gate):
//                act(W_up x), or act(W_up (weight x)) where the pair's weight multiplies what the expert reads; else
//                W_down of that, times the pair's weight if there is one, float.  Four kernels: any type and size (float sums of 8-element runs a lane);
//                bfloat16 on the matrix cores from registers (tiles of 16 pairs, the inner size shared out over a
//                workgroup's waves); bfloat16 on the matrix cores through shared memory (tiles of 64 and of 128 pairs).
//   moe_combine  a row's pairs summed in the order of its places; a router output beyond the experts with
//                matrices hands the row itself on (times its weight); a delta that comes along is added.
//
// Every grid is fixed by the step's row count alone (tiles that turn out unused end at once), so a step that is
// recorded once can be replayed with other choices.  Products accumulate in float from operands of the engine's
// type; the router, its softmax and the weights are float.
#include "common.h"
#include "leone_hip.h"

#include <math.h>
#include <type_traits>

namespace leone {

constexpr int kRouteSlots = 8;                 // router outputs a lane holds: up to 512 experts
constexpr int kTilePairs = 8;                  // pairs of one expert a workgroup of the products takes
constexpr int kMoeThreads = 256;
constexpr int kMoeWaves = kMoeThreads / kWave;
constexpr int kColsPerWave = 4;
constexpr int kMoeCols = kMoeWaves * kColsPerWave;

// The best (value, index) of a wave: the larger value, the lower index among equals; what has no index (0x7fffffff) loses.
template <int kSpan = kWave>
__device__ inline void wave_best(float& v, int& at) {
    const Pair<float> of = lane_pair<kSpan / 2>(v);
    const Pair<int> where = lane_pair<kSpan / 2>(at);
    const bool second = of.b > of.a || (of.b == of.a && where.b < where.a) || where.a == 0x7fffffff;
    v = second ? of.b : of.a;
    at = second ? where.b : where.a;
    if constexpr (kSpan > 2) wave_best<kSpan / 2>(v, at);
}

// One wave a row; a lane holds kSlots router outputs (kSlots * 64 >= total).
// How a router scores and weighs: `score` 0 softmax over all outputs, 1 a sigmoid of each; `group_best` how many of a
// group's best choice scores make the group's score (their sum; 1: the best alone); `renorm` 1: the winners' scores over
// their sum, 0: the scores themselves; `scale` multiplies the weights either way.
struct RouteRule {
    int score, group_best, renorm;
    float scale;
};

// The choice of a row with one router output a lane, whose groups count by their best alone: a lane ranks its group among
// the groups and its output among the open ones by counting those ahead of it (higher, or the lower index among equals),
// each read from its lane by one instruction.  Scores are compared as integers in the order of the floats, so that what is
// not a number has a place too and every rank is some lane's.  Returns the lane's place among the winners, `top` and more if
// it is none of them.  (Winner after winner by exchanges over the wave, a dozen of them each, and the tiles' places by one thread, the
// choice and the plan of 8 rows over 35 outputs in 7 groups took 18.5 us; by ranks 6.6, recorded one behind the other; what
// route_plan_kernel says of its waits made it 5.4.)
__device__ inline unsigned route_order(float v) {
    const unsigned bits = __float_as_uint(v + 0.0f);           // -0 counts as 0
    return bits & 0x80000000u ? ~bits : bits | 0x80000000u;
}
__device__ inline int route_rank(float choice, int lane, int total, int group_count, int group_keep) {
    unsigned mine = lane < total ? route_order(choice) : 0u;
    if (group_count > 1) {
        const int size = total / group_count, group = lane / size;
        unsigned best = 0u;
        for (int i = 0; i < size; ++i) {
            const unsigned other = __shfl(mine, group * size + i, kWave);
            best = other > best ? other : best;
        }
        int ahead = 0;
        for (int h = 0; h < group_count; ++h) {
            const unsigned other = __builtin_amdgcn_readlane(best, h * size);
            ahead += other > best || (other == best && h < group) ? 1 : 0;
        }
        if (ahead >= group_keep) mine = route_order(-INFINITY);
    }
    int ahead = 0;
    for (int o = 0; o < total; ++o) {
        const unsigned other = __builtin_amdgcn_readlane(mine, o);
        ahead += other > mine || (other == mine && o < lane) ? 1 : 0;
    }
    return lane < total ? ahead : total;
}

template <int kSlots>
__device__ inline void route_row(int row, int lane, const float* __restrict__ logits, const AnyVec& correction,
                                 int* __restrict__ chosen, float* __restrict__ weight, int total, int top, int group_count,
                                 int group_keep, const RouteRule rule, int shift_from = 0x7fffffff, int always = 0,
                                 int* here = nullptr, int room = 0) {
    // `always` experts that every row takes with weight 1 stand behind the routed ones in the matrices (indices
    // shift_from .. shift_from + always - 1): a row's places are its `top` choices and then these; a chosen router
    // output from shift_from on (one that hands the row on) is numbered behind them.
    // here: a second copy of the first `room` choices of all rows, for the workgroup's own use (not with kRouteSlots outputs a lane).
    const int places = top + always;
    const auto choose = [&](int place, int e) {
        const long at = static_cast<long>(row) * places + place;
        chosen[at] = e;
        if constexpr (kSlots < kRouteSlots)
            if (at < room) here[at] = e;
    };
    const float* z = logits + static_cast<long>(row) * total;
    float s[kSlots], choice[kSlots];
    bool taken[kSlots];
    float top_z = -INFINITY;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
        const int e = lane + i * kWave;
        s[i] = e < total ? z[e] : -INFINITY;
        if constexpr (kSlots > 1) top_z = fmaxf(top_z, s[i]);
    }
    float early = 0.f;                                     // one output a lane: the correction on its way together with the logits
    if constexpr (kSlots == 1) {
        early = lane < total && correction.ptr ? load_any(correction, lane) : 0.f;
        top_z = fmaxf(top_z, s[0]);
    }
    top_z = wave_max(top_z);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
        const int e = lane + i * kWave;
        if (rule.score == 1) s[i] = e < total ? 1.0f / (1.0f + expf(-s[i])) : 0.f;
        else s[i] = e < total ? expf(s[i] - top_z) : 0.f;
        sum += s[i];
    }
    sum = rule.score == 1 ? 1.0f : wave_sum(sum);
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
        const int e = lane + i * kWave;
        s[i] = s[i] / sum;
        choice[i] = e < total ? s[i] + (kSlots == 1 ? early : correction.ptr ? load_any(correction, e) : 0.f) : -INFINITY;
        taken[i] = e >= total;
    }
    if (kSlots == 1 && (group_count == 1 || rule.group_best == 1)) {
        const int rank = route_rank(choice[0], lane, total, group_count, group_keep);
        const bool won = rank < top;
        // the winners' scores are added in the order of their ranks
        float picked = 0.f;
        for (int i = 0; i < top; ++i) {
            const unsigned long long who = __ballot(rank == i);
            picked += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s[0]), __ffsll(who) - 1));
        }
        const float by = rule.renorm ? picked + 1e-20f : 1.0f;
        if (won) {
            choose(rank, lane >= shift_from ? lane + always : lane);
            weight[static_cast<long>(row) * places + rank] = s[0] / by * rule.scale;
        }
        for (int i = lane; i < always; i += kWave) {
            choose(top + i, shift_from + i);
            weight[static_cast<long>(row) * places + top + i] = 1.0f;
        }
        return;
    }
    if (group_count > 1) {
        // a group's score: lane g % 64 keeps group g's in its place g / 64 (there are no more groups than outputs)
        const int size = total / group_count;
        int group_of[kSlots];
#pragma unroll
        for (int i = 0; i < kSlots; ++i) group_of[i] = (lane + i * kWave) / size;
        float mine[kSlots];
        bool mine_taken[kSlots];
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            mine[i] = -INFINITY;
            mine_taken[i] = lane + i * kWave >= group_count;
        }
        for (int g = 0; g < group_count; ++g) {
            float best = 0.f;
            int used[kSlots];                              // the group's outputs already counted into its score
#pragma unroll
            for (int i = 0; i < kSlots; ++i) used[i] = 0;
            for (int n = 0; n < rule.group_best && n < size; ++n) {
                float v = -INFINITY;
                int at = 0x7fffffff;
#pragma unroll
                for (int i = 0; i < kSlots; ++i) {
                    const int e = lane + i * kWave;
                    if (e < total && group_of[i] == g && !used[i] && (at == 0x7fffffff || choice[i] > v)) {
                        v = choice[i];
                        at = e;
                    }
                }
                wave_best(v, at);
#pragma unroll
                for (int i = 0; i < kSlots; ++i)
                    if (lane + i * kWave == at) used[i] = 1;
                best = n == 0 ? v : best + v;
            }
#pragma unroll
            for (int i = 0; i < kSlots; ++i)
                if (lane + i * kWave == g) mine[i] = best;
        }
        unsigned open = 0u;                                   // bit i: group lane + 64 i stays open
        for (int n = 0; n < group_keep; ++n) {
            float v = -INFINITY;
            int at = 0x7fffffff;
#pragma unroll
            for (int i = 0; i < kSlots; ++i)
                if (!mine_taken[i] && (at == 0x7fffffff || mine[i] > v)) {
                    v = mine[i];
                    at = lane + i * kWave;
                }
            wave_best(v, at);
            if (at == 0x7fffffff) break;
#pragma unroll
            for (int i = 0; i < kSlots; ++i)
                if (lane + i * kWave == at) {
                    mine_taken[i] = true;
                    open |= 1u << i;
                }
        }
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            const int e = lane + i * kWave;
            const int g = e < total ? group_of[i] : 0;
            const unsigned theirs = __shfl(open, g % kWave, kWave);
            if (e < total && !((theirs >> (g / kWave)) & 1u)) choice[i] = -INFINITY;
        }
    }
    float picked_sum = 0.f;
    float my_s = 0.f;
    int my_e = 0;
    for (int n = 0; n < top; ++n) {
        float v = -INFINITY;
        int at = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            const int e = lane + i * kWave;
            if (!taken[i] && (at == 0x7fffffff || choice[i] > v)) {
                v = choice[i];
                at = e;
            }
        }
        wave_best(v, at);
        float got = 0.f;
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            const int e = lane + i * kWave;
            if (e == at) {
                taken[i] = true;
                got = s[i];
            }
        }
        got = wave_sum(got);               // one lane held it
        picked_sum += got;
        if (lane == n % kWave && n < kWave) {
            my_s = got;
            my_e = at;
        }
        if (n >= kWave && lane == 0) {       // more than 64 places: written as they come, scaled below
            choose(n, at >= shift_from ? at + always : at);
            weight[static_cast<long>(row) * places + n] = got;
        }
    }
    const float denom = rule.renorm ? picked_sum + 1e-20f : 1.0f;
    if (lane < top && lane < kWave) {
        choose(lane, my_e >= shift_from ? my_e + always : my_e);
        weight[static_cast<long>(row) * places + lane] = my_s / denom * rule.scale;
    }
    if (top > kWave && lane == 0)
        for (int n = kWave; n < top; ++n)
            weight[static_cast<long>(row) * places + n] = weight[static_cast<long>(row) * places + n] / denom * rule.scale;
    for (int i = lane; i < always; i += kWave) {
        choose(top + i, shift_from + i);
        weight[static_cast<long>(row) * places + top + i] = 1.0f;
    }
}

template <int kSlots>
__global__ void __launch_bounds__(kWave)
route_topk_kernel(const float* __restrict__ logits, AnyVec correction, int* __restrict__ chosen, float* __restrict__ weight,
                  int total, int top, int group_count, int group_keep, RouteRule rule) {
    route_row<kSlots>(blockIdx.x, threadIdx.x, logits, correction, chosen, weight, total, top, group_count, group_keep, rule);
}

// One workgroup.  counts and places live in shared memory (experts <= 1024).  clear_tiles, the choices, a barrier, plan_tiles.
__device__ inline void clear_tiles(int experts, int* __restrict__ tile_expert, int* __restrict__ tile_pairs, int max_tiles, int tile,
                                   int* count, int first_thread = 0) {
    const int mine = threadIdx.x - first_thread, all = blockDim.x - first_thread;
    for (int e = mine; e < experts; e += all) count[e] = 0;
    for (int t = mine; t < max_tiles; t += all) tile_expert[t] = -1;
    for (long i = mine; i < static_cast<long>(max_tiles) * tile; i += all) tile_pairs[i] = -1;
}

__device__ inline void plan_tiles(const int* chosen, int pairs, int experts, int* __restrict__ tile_expert,
                                  int* __restrict__ tile_pairs, int max_tiles, int tile, int* count, int* first_tile) {
    for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
        const int e = chosen[p];
        if (e >= 0 && e < experts) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (threadIdx.x < kWave) {                          // the first wave: a run of experts a lane, the runs added up over the lanes
        const int run = (experts + kWave - 1) / kWave, begin = threadIdx.x * run;
        const int end = begin + run < experts ? begin + run : experts;
        int tiles = 0;
        for (int e = begin; e < end; ++e) tiles += (count[e] + tile - 1) / tile;
        int at = tiles;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int before = __shfl_up(at, off, kWave);
            if (static_cast<int>(threadIdx.x) >= off) at += before;
        }
        at -= tiles;
        for (int e = begin; e < end; ++e) {
            first_tile[e] = at;
            const int mine = (count[e] + tile - 1) / tile;
            for (int t = 0; t < mine && at + t < max_tiles; ++t) tile_expert[at + t] = e;
            at += mine;
            count[e] = 0;
        }
    }
    __syncthreads();
    // Which place of its expert's tiles a pair gets does not matter to its result: every pair is worked out by itself.
    for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
        const int e = chosen[p];
        if (e >= 0 && e < experts) {
            const int at = atomicAdd(&count[e], 1);
            const long place = static_cast<long>(first_tile[e]) * tile + at;
            if (place < static_cast<long>(max_tiles) * tile) tile_pairs[place] = p;
        }
    }
}

__global__ void __launch_bounds__(1024)
moe_plan_kernel(const int* __restrict__ chosen, int pairs, int experts, int* __restrict__ tile_expert,
                int* __restrict__ tile_pairs, int max_tiles, int tile) {
    __shared__ int count[1024];
    __shared__ int first_tile[1024];
    clear_tiles(experts, tile_expert, tile_pairs, max_tiles, tile, count);
    __syncthreads();
    plan_tiles(chosen, pairs, experts, tile_expert, tile_pairs, max_tiles, tile, count, first_tile);
}

// The router's choice and the tiles in one launch, for steps of few rows (a wave a row, 16 waves in turn).  One workgroup and so
// bound by its chain of waits: the waves without a row clear the tiles meanwhile (a wave with one would wait for its stores along with
// its logits), and the choices are handed to the plan through shared memory (kPlanPairs of them; more are read back from where
// they were written).  kSlots: outputs a lane; each number is a kernel of its own, without the others' registers.  One behind the
// other in a recording: 8 rows over 64 outputs 7.5 -> 6.1 us, 64 rows over 64 in 8 groups 28.4 -> 26.0, 64 over 256 (4 outputs a lane,
// not 8) 47.7 -> 36.5.  With 8 outputs a lane the copy in shared memory gave nothing and is not made, and of 16 and more rows the tiles are
// cleared behind a barrier of their own (64 over 512 as before 50.2, without the barrier 50.6, with the copy 51.1).
constexpr int kPlanPairs = 2048;

template <int kSlots>
__global__ void __launch_bounds__(1024)
route_plan_kernel(const float* __restrict__ logits, AnyVec correction, int* __restrict__ chosen, float* __restrict__ weight,
                  int rows, int total, int top, int group_count, int group_keep, int experts, int* __restrict__ tile_expert,
                  int* __restrict__ tile_pairs, int max_tiles, int tile, int always, RouteRule rule) {
    constexpr int kWaves = 1024 / kWave;
    const int routed = experts - always;               // experts the router chooses among; the others every row takes
    __shared__ int count[1024];
    __shared__ int first_tile[1024];
    __shared__ int here[kPlanPairs];
    const int pairs = rows * (top + always), room = kSlots < kRouteSlots && pairs <= kPlanPairs ? pairs : 0;
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    for (int row = wave; row < rows; row += kWaves)
        route_row<kSlots>(row, lane, logits, correction, chosen, weight, total, top, group_count, group_keep, rule, routed, always, here, room);
    if (kSlots == kRouteSlots && rows >= kWaves) __syncthreads();
    if (rows >= kWaves) clear_tiles(experts, tile_expert, tile_pairs, max_tiles, tile, count);
    else if (wave >= rows) clear_tiles(experts, tile_expert, tile_pairs, max_tiles, tile, count, rows * kWave);
    __syncthreads();                                   // the choices are written; the same workgroup reads them
    if (room > 0) plan_tiles(here, pairs, experts, tile_expert, tile_pairs, max_tiles, tile, count, first_tile);
    else plan_tiles(chosen, pairs, experts, tile_expert, tile_pairs, max_tiles, tile, count, first_tile);
}

template <typename T>
__device__ inline void load8f(const T* __restrict__ p, int k, int limit, bool runs, float out[8]);

template <>
__device__ inline void load8f<float>(const float* __restrict__ p, int k, int limit, bool runs, float out[8]) {
    if (runs && k + 8 <= limit) {
        const float4 a = *reinterpret_cast<const float4*>(p + k);
        const float4 b = *reinterpret_cast<const float4*>(p + k + 4);
        out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w;
        out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = k + i < limit ? p[k + i] : 0.f;
}

template <>
__device__ inline void load8f<bf16_t>(const bf16_t* __restrict__ p, int k, int limit, bool runs, float out[8]) {
    if (runs && k + 8 <= limit) {
        const uint4 t = *reinterpret_cast<const uint4*>(p + k);
        const unsigned w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            out[2 * i] = __uint_as_float(w[i] << 16);
            out[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = k + i < limit ? to_float(p[k + i]) : 0.f;
}

// A tile's pairs against kMoeCols rows of its expert's matrices: a wave takes kColsPerWave rows, its lanes runs of
// eight elements of the inner size; sums over the lanes at the end.
//   kMoeGated: w = [experts][2][n][k] (gate rows, then up rows), y[pair][col] = act(gate) * up in T
//   kMoePlain: w = [experts][n][k], y[pair][col] = act(weight[pair] * product) in T (a product of weight[pair] * x)
//   kMoeDown:  w = [experts][n][k], y[pair][col] = weight[pair] * product in float
// x: kMoeDown: row pair of [pairs][k]; else row pair / top of [rows][k].  Without weights they count as 1.
enum MoeMode : int { kMoeDown = 0, kMoeGated = 1, kMoePlain = 2 };

template <typename T, int kMode>
__global__ void __launch_bounds__(kMoeThreads)
moe_product_kernel(const T* __restrict__ x, const T* __restrict__ w, void* __restrict__ y, const float* __restrict__ pair_weight,
                   const int* __restrict__ tile_expert, const int* __restrict__ tile_pairs, int top, int n, int k, int act,
                   float limit, int runs) {
    constexpr bool kGated = kMode == kMoeGated;
    const int tile = blockIdx.x;
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int col0 = blockIdx.y * kMoeCols + wave * kColsPerWave;
    if (col0 >= n) return;
    int pair[kTilePairs];
#pragma unroll
    for (int p = 0; p < kTilePairs; ++p) pair[p] = tile_pairs[static_cast<long>(tile) * kTilePairs + p];
    float acc[kColsPerWave][kTilePairs], acc2[kGated ? kColsPerWave : 1][kTilePairs];
#pragma unroll
    for (int c = 0; c < kColsPerWave; ++c)
#pragma unroll
        for (int p = 0; p < kTilePairs; ++p) {
            acc[c][p] = 0.f;
            if constexpr (kGated) acc2[c][p] = 0.f;
        }
    const long matrix = static_cast<long>(n) * k;
    const T* w_first = w + static_cast<long>(e) * (kGated ? 2 : 1) * matrix;
    for (int at = 8 * lane; at < k; at += 8 * kWave) {
        float xv[kTilePairs][8];
#pragma unroll
        for (int p = 0; p < kTilePairs; ++p) {
            if (pair[p] >= 0) {
                load8f<T>(x + static_cast<long>(kMode != kMoeDown ? pair[p] / top : pair[p]) * k, at, k, runs != 0, xv[p]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) xv[p][i] = 0.f;
            }
        }
#pragma unroll
        for (int c = 0; c < kColsPerWave; ++c) {
            const int col = col0 + c;
            if (col >= n) continue;
            float wv[8], wv2[8];
            load8f<T>(w_first + static_cast<long>(col) * k, at, k, runs != 0, wv);
            if constexpr (kGated) load8f<T>(w_first + matrix + static_cast<long>(col) * k, at, k, runs != 0, wv2);
#pragma unroll
            for (int p = 0; p < kTilePairs; ++p)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    acc[c][p] = fmaf(wv[i], xv[p][i], acc[c][p]);
                    if constexpr (kGated) acc2[c][p] = fmaf(wv2[i], xv[p][i], acc2[c][p]);
                }
        }
    }
    // lane c * kTilePairs + p writes (column c, pair p)
    float mine = 0.f, mine2 = 0.f;
#pragma unroll
    for (int c = 0; c < kColsPerWave; ++c)
#pragma unroll
        for (int p = 0; p < kTilePairs; ++p) {
            const float total = wave_sum(acc[c][p]);
            float total2 = 0.f;
            if constexpr (kGated) total2 = wave_sum(acc2[c][p]);
            if (lane == c * kTilePairs + p) {
                mine = total;
                mine2 = total2;
            }
        }
    if (lane < kColsPerWave * kTilePairs) {
        const int c = lane / kTilePairs, p = lane % kTilePairs;
        const int col = col0 + c;
        // the pair of this lane, without indexing the register array by a lane's value
        int which = -1;
#pragma unroll
        for (int q = 0; q < kTilePairs; ++q)
            if (q == p) which = pair[q];
        if (col < n && which >= 0) {
            if constexpr (kGated)
                static_cast<T*>(y)[static_cast<long>(which) * n + col] = from_float<T>(glu_value(mine, mine2, act, limit));
            else if constexpr (kMode == kMoePlain)
                static_cast<T*>(y)[static_cast<long>(which) * n + col] =
                    from_float<T>(plain_act(pair_weight ? mine * pair_weight[which] : mine, act));
            else
                static_cast<float*>(y)[static_cast<long>(which) * n + col] = pair_weight ? mine * pair_weight[which] : mine;
        }
    }
}


// The same products on the matrix cores, bfloat16 (v_mfma_f32_16x16x32_bf16: rows of the matrix are one operand, 16 pairs the
// other; lane (c, g) holds elements 8 g .. 8 g + 7 of a step of 32 of row c and of pair c, and gets rows 4 g .. 4 g + 3 of
// pair c).  Inner sizes are multiples of 8; what lies beyond the inner size counts as zeros.
typedef __bf16 moe_bf16x8 __attribute__((ext_vector_type(8)));
typedef float moe_floatx4 __attribute__((ext_vector_type(4)));

__device__ inline moe_bf16x8 moe_load8(const bf16_t* p) {
    return __builtin_bit_cast(moe_bf16x8, *reinterpret_cast<const uint4*>(p));
}
__device__ inline moe_bf16x8 moe_zero8() {
    const uint4 z = {0u, 0u, 0u, 0u};
    return __builtin_bit_cast(moe_bf16x8, z);
}

// Tiles of 16 pairs, bfloat16 (steps of few rows): every matrix of a chosen expert is read once for a handful of pairs, so
// its bytes are the bound.  A workgroup takes 16 rows of the matrix (gated: and their up rows) and its four waves share out
// the inner size, each with eight steps of 32 on their way at a time; their sums meet in shared memory, in the waves' order.
// (A wave that walked the whole inner size by itself had a quarter of the loads in flight and four times the chain.)
// Eight rows of 2,048 over 34 experts of 768, four routed places and two for every row (us; with loads that the compiler could not
// count, for which it waited one by one; one wave an item): gated 30 (38, 47), down 18 (19, 24).
//
// A load is half of a line in 16 rows; the other half comes with the load behind it.  kStreamed: loads marked as not to be kept, which
// leaves the caches to others (a decoding step of a model with 32 experts of 2,048 x 768: 6.96 ms, unmarked 7.09, its first products alone unmarked
// 7.14); with longer rows some lines came twice (32 experts of 4,096 x 1,024, both products, 16 rows 172 us, the first one
// unmarked 158; 8 of 1,024 x 4,096, eight rows 58, the second one unmarked 46 to 56).
//
// kTiled: the matrices come as a copy laid out as the waves ask for them (16 rows at a time, steps of 32 elements one after the other, a
// step lane by lane), so that a load is one kilobyte in one piece; same numbers in the same places, same bits.
constexpr int kStreamedInner = 2048;

enum MoeLayout : int { kMoeKept = 0, kMoeStreamed = 1, kMoeTiled = 2 };
template <int kMode, int kLayout>
__global__ void __launch_bounds__(kMoeThreads, 4)
moe_product_stream_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ y,
                          const float* __restrict__ pair_weight, const int* __restrict__ tile_expert,
                          const int* __restrict__ tile_pairs, int top, int n, int k, int act, float limit) {
    constexpr bool kGated = kMode == kMoeGated, kTiled = kLayout == kMoeTiled;
    constexpr int kDepth = 8, kStep = kTiled ? 512 : 32;         // elements from a step of the matrix to the next
    __shared__ moe_floatx4 sums[kGated ? 2 : 1][kMoeWaves][kWave];
    const int tile = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int c = lane & 15, g = lane >> 4;
    const int* my_pairs = tile_pairs + static_cast<long>(tile) * 16;
    const int own = my_pairs[c], first_pair = my_pairs[0];
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int row0 = blockIdx.y * 16;
    const long matrix = static_cast<long>(n) * k;
    // Lanes past the last row take that one again, lanes without a pair the tile's first: their results are not written.  Nothing
    // stands between the loads: behind one that may not have been asked for the compiler cannot count those in flight and waits for all.
    const bf16_t* wa = w + static_cast<long>(e) * (kGated ? 2 : 1) * matrix +
                       (kTiled ? static_cast<long>(row0) * k + 8 * lane : static_cast<long>(row0 + c < n ? row0 + c : n - 1) * k + 8 * g);
    const int pair = own < 0 ? first_pair : own;
    const bf16_t* xrow = x + static_cast<long>(kMode != kMoeDown ? pair / top : pair) * k;
    const int steps = (k + 31) / 32, share = (steps + kMoeWaves - 1) / kMoeWaves;
    const int first = wave * share, last = first + share < steps ? first + share : steps;
    moe_floatx4 acc = {0.f, 0.f, 0.f, 0.f}, acc2 = {0.f, 0.f, 0.f, 0.f};
    moe_bf16x8 a[kDepth], a2[kGated ? kDepth : 1], xb[kDepth];
    const auto weights = [](const bf16_t* p) { return kLayout != kMoeKept ? __builtin_bit_cast(moe_bf16x8, load_streamed16(p)) : moe_load8(p); };
    const auto ask = [&](int d, const bf16_t* of_w, const bf16_t* of_x) {
        a[d] = weights(of_w);
        if constexpr (kGated) a2[d] = weights(of_w + matrix);
        xb[d] = moe_load8(of_x);
    };
    const auto multiply = [&](int d) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d], xb[d], acc, 0, 0, 0);
        if constexpr (kGated) acc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[d], xb[d], acc2, 0, 0, 0);
    };
    const int whole = last * 32 <= k ? last : last - 1;          // steps without the inner size's end
    const bf16_t *from_w = wa + static_cast<long>(kStep) * first, *from_x = xrow + 32 * first + 8 * g;
    int left = whole > first ? whole - first : 0;
    if (left >= kDepth) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) ask(d, from_w + kStep * d, from_x + 32 * d);
        for (; left >= 2 * kDepth; left -= kDepth) {
            from_w += kStep * kDepth, from_x += 32 * kDepth;
#pragma unroll
            for (int d = 0; d < kDepth; ++d) {
                multiply(d);
                ask(d, from_w + kStep * d, from_x + 32 * d);
            }
        }
#pragma unroll
        for (int d = 0; d < kDepth; ++d) multiply(d);
        from_w += kStep * kDepth, from_x += 32 * kDepth, left -= kDepth;
    }
    const auto rest = [&](auto count) {
#pragma unroll
        for (int d = 0; d < decltype(count)::value; ++d) ask(d, from_w + kStep * d, from_x + 32 * d);
#pragma unroll
        for (int d = 0; d < decltype(count)::value; ++d) multiply(d);
    };
    switch (left) {
        case 7: rest(std::integral_constant<int, 7>{}); break;
        case 6: rest(std::integral_constant<int, 6>{}); break;
        case 5: rest(std::integral_constant<int, 5>{}); break;
        case 4: rest(std::integral_constant<int, 4>{}); break;
        case 3: rest(std::integral_constant<int, 3>{}); break;
        case 2: rest(std::integral_constant<int, 2>{}); break;
        case 1: rest(std::integral_constant<int, 1>{}); break;
        default: break;
    }
    if (!kTiled && first < last && whole < last) {                 // the step that holds the inner size's end; zeros beyond it
        const int wanted = 32 * whole + 8 * g, at = wanted < k ? wanted : k - 8;
        ask(0, wa + at - 8 * g, xrow + at);
        if (wanted >= k) {
            a[0] = xb[0] = moe_zero8();
            if constexpr (kGated) a2[0] = moe_zero8();
        }
        multiply(0);
    }
    sums[0][wave][lane] = acc;
    if constexpr (kGated) sums[1][wave][lane] = acc2;
    __syncthreads();
    // thread t: row t % 16 of pair t / 16, which lane 16 (row / 4) + pair of every wave holds at row % 4
    const int row = threadIdx.x % 16, which = threadIdx.x / 16;
    const int to = tile_pairs[static_cast<long>(tile) * 16 + which], r = row0 + row;
    if (to < 0 || r >= n) return;
    const int from = 16 * (row / 4) + which, j = row % 4;
    float total = 0.f, total2 = 0.f;
#pragma unroll
    for (int v = 0; v < kMoeWaves; ++v) {
        total += sums[0][v][from][j];
        if constexpr (kGated) total2 += sums[1][v][from][j];
    }
    const long at = static_cast<long>(to) * n + r;
    if constexpr (kGated) static_cast<bf16_t*>(y)[at] = from_float<bf16_t>(glu_value(total, total2, act, limit));
    else if constexpr (kMode == kMoePlain)
        static_cast<bf16_t*>(y)[at] = from_float<bf16_t>(plain_act(pair_weight ? total * pair_weight[to] : total, act));
    else static_cast<float*>(y)[at] = pair_weight ? total * pair_weight[to] : total;
}

// Tiles of 64 pairs, bfloat16: a workgroup takes a tile and 128 rows of its expert's matrix (gated: 64 gate rows and their
// up rows), in chunks of 64 of the inner size that go through shared memory: a row's chunk is one line of 128 bytes, fetched
// whole by eight neighbouring threads (rows of a matrix lie a power of two apart, so lines that are only half used at a time
// push one another out of the caches before their other half is asked for).  In shared memory a chunk lies as two halves of 32
// elements, rows one after the other within a half: the 16 rows of an operand are one kilobyte that the 64 lanes read in one
// piece.  The four waves take 64 rows x 32 pairs each.
//
// What bounds it is the way from memory: a chunk is worked off in half a microsecond and takes two to arrive.  So two chunks
// are on their way in registers while a third is worked on and a fourth lies ready behind it in shared memory, and the tile
// is small enough for two to three workgroups a compute unit.  (One chunk ahead, with tiles of 128 pairs x 256 rows, had 0.34
// PFLOP/s; tiles of 64 pairs straight from memory into registers were slower still; tiles of 128 pairs worked this way take
// eight waves, of which fewer workgroups fit: 312 us at the largest of these.)  Measured, both products of 32 experts, width
// 2,048 and 768, in a model's pass (us; with loads that the compiler could not count): 7,700 pairs 181 (199).  Alone, matrices not
// in the caches: 1,160 pairs 128 (131), 2,800 pairs 143 (161), 8,456 pairs 259 (279).
constexpr int kBigPairs = 64;
constexpr int kBigRows = 128;
constexpr int kBigChunk = 64;

// Where 16-byte piece `quarter` of a row's half chunk lies in its half: rows of four pieces, the pieces of every fourth row turned
// about, so that the same piece of 16 neighbouring rows lies in 16 places of the 256 bytes that shared memory gives at a time.  The
// second half begins 128 bytes past the first one's end: a row's two halves, written side by side, then meet in no bank either.
// (Rows one after the other as they came: half of shared memory's time went to conflicts, and it was busy for 55 % of the first
// product's: 121 us for 7,700 pairs, 32 experts of 2,048 x 768.)
__device__ inline int piece_at(int row, int quarter) { return row * 4 + (quarter ^ ((row >> 2) & 3)); }
constexpr int half_pieces(int rows) { return rows * 4 + 8; }

// Rows r .. r + 3 of a pair's result, r < n.
template <int kMode>
__device__ inline void store_rows(void* y, int pair, int r, int n, const float (&v)[4]) {
    const bool whole = r + 3 < n && n % 4 == 0;
    if constexpr (kMode != kMoeDown) {
        bf16_t* to = static_cast<bf16_t*>(y) + static_cast<long>(pair) * n + r;
        if (whole) {
            uint2 packed;
            packed.x = bf16_bits_from_float(v[0]) | (static_cast<uint32_t>(bf16_bits_from_float(v[1])) << 16);
            packed.y = bf16_bits_from_float(v[2]) | (static_cast<uint32_t>(bf16_bits_from_float(v[3])) << 16);
            *reinterpret_cast<uint2*>(to) = packed;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (r + j < n) to[j] = from_float<bf16_t>(v[j]);
        }
    } else {
        float* to = static_cast<float*>(y) + static_cast<long>(pair) * n + r;
        if (whole) {
            *reinterpret_cast<float4*>(to) = float4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (r + j < n) to[j] = v[j];
        }
    }
}

// One chunk is on its way at a time, not two, where the experts' matrices give nearly every unit one workgroup (7/8 of the units up to all of
// them) and their rows lie whole multiples of 4 KB apart: the units then walk the inner size abreast, and what more they ask for falls on
// the same channels.  Both products from memory, us (one chunk, two): 8 experts of 4,096 x 2,048, 16 pairs an expert 116 and 130, 50 pairs
// 126 and 143, 150 pairs 152 and 162; 16 of 8,192 x 1,024, 16 pairs 205 and 254; 16 of 2,048 x 1,024 62 and 67.  With rows
// 12 KB apart (6,144) 166 and 170, 10 KB (5,120) 136 and 138; with half the workgroups (4 of 4,096 x 2,048) 87 and 65, with twice as many (32
// of 4,096 x 1,024) 189 and 173; matrices of few rows (32 of 4,096 x 512) 100 and 96.
constexpr int kMoeUnits = 256;
static bool one_chunk_ahead(int experts, int blocks, int n, int k) {
    const long groups = static_cast<long>(experts) * blocks;
    return 8 * groups > 7 * kMoeUnits && groups <= kMoeUnits && k % 2048 == 0 && n >= 1024;
}

template <int kMode>
__global__ void __launch_bounds__(kMoeThreads, 3)
moe_product_tiled_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ y,
                         const float* __restrict__ pair_weight, const int* __restrict__ tile_expert,
                         const int* __restrict__ tile_pairs, int top, int n, int k, int act, float limit, int n_tiles, int n_blocks,
                         int one_ahead) {
    constexpr bool kGated = kMode == kMoeGated;
    constexpr int kOwnRows = kGated ? kBigRows / 2 : kBigRows;        // rows of the result
    constexpr int kBring = kMoeThreads / 8;                           // rows of 8 pieces that the workgroup brings at once
    constexpr int kXPieces = kBigPairs / kBring;                         // 16-byte pieces of x a thread brings per chunk
    constexpr int kWPieces = kBigRows / kBring;
    constexpr int kPB = 2;                                            // blocks of 16 pairs a wave
    constexpr int kXHalf = half_pieces(kBigPairs), kWHalf = half_pieces(kBigRows);
    __shared__ uint4 sx[2][2 * kXHalf];                                  // [chunk][half][piece_at]
    __shared__ uint4 sw[2][2 * kWHalf];
    // Workgroups go to the eight dies in turn, and each die has a cache of its own: the work is numbered so that a
    // die gets a run of neighbouring (row block, tile) places, tiles fastest: the tiles of one expert, which read the
    // same rows of its matrix, then lie on one die.  (Groups of two or four tiles with all their row blocks measured the same.)
    const int per_die = (n_tiles * n_blocks + 7) / 8;
    const int place = static_cast<int>(blockIdx.x % 8) * per_die + static_cast<int>(blockIdx.x / 8);
    if (place >= n_tiles * n_blocks) return;
    const int tile = place % n_tiles;
    const int row_block = place / n_tiles;
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid % kWave;
    const int c = lane & 15, g = lane >> 4;
    const int wr = wave / 2, wp = wave % 2;               // a wave's 64 rows and 32 pairs
    const int row_base = row_block * kOwnRows;
    const long matrix = static_cast<long>(n) * k;
    const int* my_pairs = tile_pairs + static_cast<long>(tile) * kBigPairs;

    // what this thread brings: part tid % 8 of every kBring-th row from tid / 8 on
    const int part = tid & 7;
    const int half = part >> 2, quarter = part & 3;
    const bf16_t* x_from[kXPieces];
    const bf16_t* w_from[kWPieces];
#pragma unroll
    for (int i = 0; i < kXPieces; ++i) {                                  // (in place of no pair or row, another one: not written)
        const int own = my_pairs[tid / 8 + kBring * i], pair = own < 0 ? my_pairs[0] : own;
        x_from[i] = x + static_cast<long>(kMode != kMoeDown ? pair / top : pair) * k;
    }
#pragma unroll
    for (int i = 0; i < kWPieces; ++i) {
        const int local = tid / 8 + kBring * i;                           // gated: rows 0..63 gate, 64..127 up
        const int row = row_base + local % kOwnRows;
        w_from[i] = w + static_cast<long>(e) * (kGated ? 2 : 1) * matrix + (local >= kOwnRows ? matrix : 0) +
                    static_cast<long>(row < n ? row : n - 1) * k;
    }
    struct Pieces {
        uint4 x[kXPieces], w[kWPieces];
    };
    const int chunks = (k + kBigChunk - 1) / kBigChunk;
    // Every call loads, past the inner size's end its last piece again, and in place of no pair the tile's first one: behind a load
    // that may not have been asked for the compiler cannot count those in flight, and waited for both chunks where one was needed.
    auto bring = [&](int chunk, Pieces& to) {
        const int wanted = chunk * kBigChunk + 8 * part, at = wanted < k ? wanted : k - 8;
#pragma unroll
        for (int i = 0; i < kWPieces; ++i) to.w[i] = *reinterpret_cast<const uint4*>(w_from[i] + at);
#pragma unroll
        for (int i = 0; i < kXPieces; ++i) to.x[i] = *reinterpret_cast<const uint4*>(x_from[i] + at);
    };
    auto put = [&](Pieces& from, int chunk, int at) {
        if (chunk >= chunks - 1 && chunk * kBigChunk + 8 * part >= k) {      // beyond the inner size: zeros
#pragma unroll
            for (int i = 0; i < kXPieces; ++i) from.x[i] = uint4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < kWPieces; ++i) from.w[i] = uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < kXPieces; ++i) sx[at][half * kXHalf + piece_at(tid / 8 + kBring * i, quarter)] = from.x[i];
#pragma unroll
        for (int i = 0; i < kWPieces; ++i) sw[at][half * kWHalf + piece_at(tid / 8 + kBring * i, quarter)] = from.w[i];
    };
    // a wave's four blocks of 16 rows: gated, two of gate rows and two of their up rows
    auto row_of = [&](int t) { return kGated ? (t / 2) * kOwnRows + 32 * wr + 16 * (t % 2) : 64 * wr + 16 * t; };
    moe_floatx4 acc[4][kPB] = {};
    auto work = [&](int at) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            moe_bf16x8 a[4], b[kPB];
#pragma unroll
            for (int t = 0; t < 4; ++t) a[t] = __builtin_bit_cast(moe_bf16x8, sw[at][h * kWHalf + piece_at(row_of(t) + c, g)]);
#pragma unroll
            for (int t = 0; t < kPB; ++t) b[t] = __builtin_bit_cast(moe_bf16x8, sx[at][h * kXHalf + piece_at(32 * wp + 16 * t + c, g)]);
#pragma unroll
            for (int ta = 0; ta < 4; ++ta)
#pragma unroll
                for (int tb = 0; tb < kPB; ++tb) acc[ta][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ta], b[tb], acc[ta][tb], 0, 0, 0);
        }
    };
    Pieces even, odd;                                  // chunks 1, 3, .. of the loop below come in `odd`, 2, 4, .. in `even`
    bring(0, even);
    bring(1, odd);
    put(even, 0, 0);
    bring(2, even);
    int ck = 0;
    for (; ck + 4 < chunks; ck += 2) {
        __syncthreads();                               // chunk ck lies ready, and nobody reads the other place any more
        if (one_ahead) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        put(odd, ck + 1, 1);
        __builtin_amdgcn_sched_barrier(0);             // asked for earlier a chunk would take registers of its own, later it would come late
        bring(ck + 3, odd);
        __builtin_amdgcn_sched_barrier(0);
        work(0);
        __syncthreads();
        if (one_ahead) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        put(even, ck + 2, 0);
        __builtin_amdgcn_sched_barrier(0);
        bring(ck + 4, even);
        __builtin_amdgcn_sched_barrier(0);
        work(1);
    }
    // the last one to four chunks; behind an odd number of them one of zeros
    __syncthreads();
    put(odd, ck + 1, 1);
    if (ck + 3 < chunks) bring(ck + 3, odd);
    work(0);
    __syncthreads();
    put(even, ck + 2, 0);
    work(1);
    if (ck + 2 < chunks) {
        __syncthreads();
        put(odd, ck + 3, 1);
        work(0);
        __syncthreads();
        work(1);
    }
    // lane (c, g) holds rows 4 g .. 4 g + 3 of pair c of every (ta, tb)
#pragma unroll
    for (int tb = 0; tb < kPB; ++tb) {
        const int pair = my_pairs[32 * wp + 16 * tb + c];
        if (pair < 0) continue;
        const float scale = kGated || !pair_weight ? 1.f : pair_weight[pair];
#pragma unroll
        for (int ta = 0; ta < (kGated ? 2 : 4); ++ta) {
            const int r = row_base + row_of(ta) + 4 * g;
            if (r >= n) continue;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = kGated ? glu_value(acc[ta][tb][j], acc[kGated ? ta + 2 : ta][tb][j], act, limit)
                              : kMode == kMoePlain ? plain_act(acc[ta][tb][j] * scale, act) : acc[ta][tb][j] * scale;
            store_rows<kMode>(y, pair, r, n, v);
        }
    }
}

// Tiles of 128 pairs, bfloat16, where an expert gets hundreds: 128 rows of the matrix (gated: and their up rows), whose chunks
// lie in shared memory as above, one at a time, the next on its way in registers.  The four waves take 64 rows x 64 pairs each,
// four and four operands (gated: eight and four) for 16 (32) matrix instructions, and a matrix is read half as often: with many
// tiles an expert that counts for more than chunks in flight.  Both products, us, tiles of 64 and of 128: 32 experts of 2,048 x
// 768, 300 pairs an expert 247 and 257, 500 388 and 351, 700 533 and 468; of 4,096 x 1,024, 500 910 and 790; 64 of 2,048 x
// 1,408, 700 1594 and 1332.
constexpr int kWidePairs = 128;
constexpr int kWideRows = 128;

template <int kMode>
__global__ void __launch_bounds__(kMoeThreads, 2)
moe_product_wide_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ y,
                         const float* __restrict__ pair_weight, const int* __restrict__ tile_expert,
                         const int* __restrict__ tile_pairs, int top, int n, int k, int act, float limit, int n_tiles, int n_blocks, int) {
    constexpr bool kGated = kMode == kMoeGated;
    constexpr int kWRows = kGated ? 2 * kWideRows : kWideRows;          // rows of the matrix in a chunk
    constexpr int kXPieces = kWidePairs * 8 / kMoeThreads;             // 16-byte pieces of x a thread brings per chunk
    constexpr int kWPieces = kWRows * 8 / kMoeThreads;
    constexpr int kXHalf = half_pieces(kWidePairs), kWHalf = half_pieces(kWRows);
    __shared__ uint4 sx[2 * kXHalf];                                   // [half][piece_at]
    __shared__ uint4 sw[2 * kWHalf];
    // Workgroups go to the eight dies in turn, and each die has a cache of its own: the work is numbered so that a
    // die gets a run of neighbouring (row block, tile) places, tiles fastest: the tiles of one expert, which read the
    // same rows of its matrix, then lie on one die.
    const int per_die = (n_tiles * n_blocks + 7) / 8;
    const int place = static_cast<int>(blockIdx.x % 8) * per_die + static_cast<int>(blockIdx.x / 8);
    if (place >= n_tiles * n_blocks) return;
    const int tile = place % n_tiles;
    const int row_block = place / n_tiles;
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid % kWave;
    const int c = lane & 15, g = lane >> 4;
    const int wr = wave >> 1, wp = wave & 1;
    const int row_base = row_block * kWideRows;
    const long matrix = static_cast<long>(n) * k;
    const int* my_pairs = tile_pairs + static_cast<long>(tile) * kWidePairs;

    // what this thread brings: piece p = tid + 256 i is part p % 8 of row p / 8 (row tid / 8 + 32 i)
    const int part = tid & 7;
    const int half = part >> 2, quarter = part & 3;
    const bf16_t* x_from[kXPieces];
    const bf16_t* w_from[kWPieces];
#pragma unroll
    for (int i = 0; i < kXPieces; ++i) {
        const int pair = my_pairs[tid / 8 + 32 * i];
        x_from[i] = pair < 0 ? nullptr : x + static_cast<long>(kMode != kMoeDown ? pair / top : pair) * k + 8 * part;
    }
#pragma unroll
    for (int i = 0; i < kWPieces; ++i) {
        const int local = tid / 8 + 32 * i;                           // gated: rows 0..127 gate, 128..255 up
        const int row = row_base + (local % kWideRows);
        w_from[i] = row >= n ? nullptr
                             : w + static_cast<long>(e) * (kGated ? 2 : 1) * matrix + (local >= kWideRows ? matrix : 0) +
                                   static_cast<long>(row) * k + 8 * part;
    }
    uint4 hx[kXPieces], hw[kWPieces];

    moe_floatx4 acc[4][4], acc2[kGated ? 4 : 1][4];
#pragma unroll
    for (int ta = 0; ta < 4; ++ta)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) {
            acc[ta][tb] = moe_floatx4{0.f, 0.f, 0.f, 0.f};
            if constexpr (kGated) acc2[ta][tb] = moe_floatx4{0.f, 0.f, 0.f, 0.f};
        }
    const int chunks = (k + kBigChunk - 1) / kBigChunk;
#define LEONE_MOE_BRING(K0)                                                                                              \
    {                                                                                                                    \
        const bool in = (K0) + 8 * part < k;                                                                             \
        _Pragma("unroll") for (int i = 0; i < kXPieces; ++i) {                                                           \
            hx[i] = uint4{0u, 0u, 0u, 0u};                                                                               \
            if (x_from[i] && in) hx[i] = *reinterpret_cast<const uint4*>(x_from[i] + (K0));                              \
        }                                                                                                                \
        _Pragma("unroll") for (int i = 0; i < kWPieces; ++i) {                                                           \
            hw[i] = uint4{0u, 0u, 0u, 0u};                                                                               \
            if (w_from[i] && in) hw[i] = *reinterpret_cast<const uint4*>(w_from[i] + (K0));                              \
        }                                                                                                                \
    }
    LEONE_MOE_BRING(0)
    for (int ck = 0; ck < chunks; ++ck) {
#pragma unroll
        for (int i = 0; i < kXPieces; ++i) sx[half * kXHalf + piece_at(tid / 8 + 32 * i, quarter)] = hx[i];
#pragma unroll
        for (int i = 0; i < kWPieces; ++i) sw[half * kWHalf + piece_at(tid / 8 + 32 * i, quarter)] = hw[i];
        __syncthreads();
        if (ck + 1 < chunks) LEONE_MOE_BRING((ck + 1) * kBigChunk)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            moe_bf16x8 a[4], a2[kGated ? 4 : 1], b[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                a[t] = __builtin_bit_cast(moe_bf16x8, sw[h * kWHalf + piece_at(64 * wr + 16 * t + c, g)]);
                if constexpr (kGated) a2[t] = __builtin_bit_cast(moe_bf16x8, sw[h * kWHalf + piece_at(kWideRows + 64 * wr + 16 * t + c, g)]);
                b[t] = __builtin_bit_cast(moe_bf16x8, sx[h * kXHalf + piece_at(64 * wp + 16 * t + c, g)]);
            }
#pragma unroll
            for (int ta = 0; ta < 4; ++ta)
#pragma unroll
                for (int tb = 0; tb < 4; ++tb) {
                    acc[ta][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ta], b[tb], acc[ta][tb], 0, 0, 0);
                    if constexpr (kGated) acc2[ta][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[ta], b[tb], acc2[ta][tb], 0, 0, 0);
                }
        }
        __syncthreads();                               // everyone has read the chunk before the next is put down
    }
#undef LEONE_MOE_BRING
    // lane (c, g) holds rows 4 g .. 4 g + 3 of pair c of every (ta, tb)
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
        const int pair = my_pairs[64 * wp + 16 * tb + c];
        if (pair < 0) continue;
        const float scale = kGated || !pair_weight ? 1.f : pair_weight[pair];
#pragma unroll
        for (int ta = 0; ta < 4; ++ta) {
            const int r = row_base + 64 * wr + 16 * ta + 4 * g;
            if (r >= n) continue;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = kGated ? glu_value(acc[ta][tb][j], acc2[kGated ? ta : 0][tb][j], act, limit)
                              : kMode == kMoePlain ? plain_act(acc[ta][tb][j] * scale, act) : acc[ta][tb][j] * scale;
            store_rows<kMode>(y, pair, r, n, v);
        }
    }
}

// Tiles of 64 and 128 pairs from the matrices' second copies (kMoeTiled), inner sizes that are multiples of 64: a workgroup takes a tile of
// pairs and 128 kNT rows of its expert's matrix (gated: half as many gate rows and their up rows), a wave a quarter of them in parts of 32, whose
// elements it takes from memory as its instruction (32 x 32 x 16) wants them, one or two stages of 64 ahead: they pass neither through shared memory
// nor a barrier.  The pairs' rows, which all four waves read, go through shared memory, a stage's 128 bytes of a row turned about by the row's
// number so that the same piece of 16 rows lies in 16 places; a stage is written while the one before it is worked on.  (The walk along the stages and the
// turned stores are gemm_many_kernel's: what is mended in one is mended in both.)
//
// What bounds it is the power of the chip (matrix instructions alone, on all units, run at two thirds of the clock) and what goes through
// shared memory: hence 256 rows a workgroup, which read a piece of the pairs' rows half as often, wherever that leaves work for the units (see
// many_rows), and results turned in shared memory so that stores are whole lines (as 16 bytes of 32 rows they took a third of the
// second product).  With the matrices row by row the same kernel takes 1.4 times as long (half a line of 32 rows a load).
// And a workgroup walks a whole inner size: with few of them that is what takes the time, and ops._copied_tile leaves such products to the kernels above.
// Both products, us, best tiles of moe_product_tiled_kernel and moe_product_wide_kernel and now: 32 experts of 2,048 x 768, 40 pairs each 79 and 63, 100
// pairs 109 and 75, 240 pairs 176 and 132, 400 pairs 256 and 181, 700 pairs 358 and 277; 32 of 4,096 x 1,024, 240 pairs 413 and 306; 64 of 2,048 x 1,408,
// 100 pairs 322 and 250; 32 of 1,024 x 384, 100 pairs 37 and 26.
typedef float moe_floatx16 __attribute__((ext_vector_type(16)));
constexpr int kTogether = 2;
template <int kMode, int kMT, int kNT>
__global__ void __launch_bounds__(kMoeThreads, kNT == 1 ? 3 : 2)
moe_product_many_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ y, const float* __restrict__ pair_weight,
                        const int* __restrict__ tile_expert, const int* __restrict__ tile_pairs, int top, int n, int k, int act, float limit,
                        int n_tiles, int n_blocks) {
    constexpr bool kGated = kMode == kMoeGated;
    constexpr int kPairs = 32 * kMT, kOwnRows = (kGated ? 64 : 128) * kNT, kWAhead = kNT == 1 ? 2 : 1, kCopies = kPairs * 8 / kMoeThreads;
    __shared__ uint4 sx[2][kPairs * 8];
    __shared__ int s_pairs[kPairs];
    __shared__ float s_scale[kPairs];
    // Workgroups go to the eight dies in turn: a die gets every eighth run of kTogether tiles, with all blocks of their matrices' rows, the
    // tiles of a run fastest.  The pairs' rows are then read from the die's own cache by all blocks but the first, and a block of rows by the tiles
    // of one expert at about the same time.
    const int place = static_cast<int>(blockIdx.x / 8), run = place / (kTogether * n_blocks), within = place % (kTogether * n_blocks);
    const int tile = (run * 8 + static_cast<int>(blockIdx.x % 8)) * kTogether + within % kTogether, row_block = within / kTogether;
    if (tile >= n_tiles) return;
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int c = lane & 31, hi = lane >> 5;
    const long matrix = static_cast<long>(n) * k;
    const int* my_pairs = tile_pairs + static_cast<long>(tile) * kPairs;
    const int stages = k / 64;

    // this lane's row of the matrix: of 32, the first 16 and the others are a tile each (gated: gate rows and their up rows)
    const bf16_t* wp[kNT];
#pragma unroll
    for (int u = 0; u < kNT; ++u) {
        const int wanted = kGated ? (row_block * 4 + wave) * kNT + u : ((row_block * 4 + wave) * kNT + u) * 2 + (c >> 4);
        const int tile16 = wanted < n / 16 ? wanted : n / 16 - 1;
        wp[u] = w + static_cast<long>(e) * (kGated ? 2 : 1) * matrix + (kGated ? (c >> 4) * matrix : 0) +
                static_cast<long>(tile16) * 16 * k + hi * 128 + (c & 15) * 8;
    }
    const bf16_t* x_from[kCopies];
    int x_to[kCopies];
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {                  // (in place of no pair the tile's first one: not written)
        const int q = i * kMoeThreads + tid, row = q >> 3, part = q & 7;
        const int own = my_pairs[row], pair = own < 0 ? my_pairs[0] : own;
        x_from[i] = x + static_cast<long>(kMode != kMoeDown ? pair / top : pair) * k + 8 * part;
        x_to[i] = row * 8 + (part ^ ((row >> 1) & 7));
    }
    if (tid < kPairs) {                                  // the pairs again, for the end
        const int own = my_pairs[tid];
        s_pairs[tid] = own;
        if (!kGated && pair_weight) s_scale[tid] = pair_weight[own < 0 ? my_pairs[0] : own];
    }
    const auto inside = [&](int s) { return s < stages ? s : stages - 1; };              // (past the end the last stage again, unused)
    const auto load_x = [&](int s, int i) { return *reinterpret_cast<const uint4*>(x_from[i] + static_cast<long>(inside(s)) * 64); };
    const auto load_w = [&](int s, int j, int u) {
        return *reinterpret_cast<const uint4*>(wp[u] + static_cast<long>(inside(s)) * 1024 + j * 256);
    };
    moe_floatx16 acc[kMT][kNT];
#pragma unroll
    for (int t = 0; t < kMT; ++t)
#pragma unroll
        for (int u = 0; u < kNT; ++u)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][u][i] = 0.f;
    constexpr int kAhead = kMT <= 2 ? 2 : 1;             // stages of the pairs' rows on their way in registers
    uint4 held[kAhead][kCopies], weights[kWAhead][4][kNT];
    moe_bf16x8 xb[2][kMT];
    const auto read_x = [&](const uint4* from, int j, int t) {
        const int row = 32 * t + c;
        return __builtin_bit_cast(moe_bf16x8, from[row * 8 + ((2 * j + hi) ^ ((row >> 1) & 7))]);
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
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int i = 0; i < kCopies; ++i)
                    if (place_of(i) / kMT == j && v >= 2 - kAhead) held[(v + 1 + kAhead) % kAhead][i] = load_x(v - 1 + kAhead, i);
                if (v >= 2 - kWAhead)
#pragma unroll
                    for (int u = 0; u < kNT; ++u) weights[v % kWAhead][j][u] = load_w(v - 2 + kWAhead, j, u);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int i = 0; i < kCopies; ++i) sx[0][x_to[i]] = first[i];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kMT; ++t) xb[0][t] = read_x(sx[0], 0, t);
    const auto stage = [&](int s, auto parity) {
        constexpr int p = decltype(parity)::value;
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
                    acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(moe_bf16x8, weights[p % kWAhead][j][u]), xb[j & 1][t], acc[t][u], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int u = 0; u < kNT; ++u) weights[p % kWAhead][j][u] = load_w(s + kWAhead, j, u);
        }
    };
    int s = 0;
    for (; s + 1 < stages; s += 2) {
        stage(s, std::integral_constant<int, 0>{});
        stage(s + 1, std::integral_constant<int, 1>{});
    }
    if (s < stages) stage(s, std::integral_constant<int, 0>{});
    // Lane (c, hi) holds, of pair c of every t, rows 8 q + 4 hi .. + 3 of each of the wave's 32.  They are turned in shared memory, a wave's
    // own part of it, so that a store covers whole runs of a pair's rows (straight from the registers it would be 16 bytes of 32 rows).
    __syncthreads();                                     // the last stage has been read
    constexpr int kBytes = kMode == kMoeDown ? 4 : 2, kWaveRows = kOwnRows / 4;
    constexpr int kAtOnce = kMode == kMoeDown ? 1 : kNT;             // of the wave's parts of 32 (gated: 16) rows
    constexpr int kRun = kWaveRows / kNT * kAtOnce * kBytes / 16;    // 16-byte pieces of a pair's rows at once
    static_assert(kRun * 32 * 16 <= sizeof(sx) / 4 && (kRun == 2 || kRun == 4 || kRun == 8), "a wave's part of the stages' memory");
    uint4* mine = &sx[0][0] + wave * (kRun * 32);
    const auto turn = [](int pair) { return (kRun == 8 ? pair >> 1 : kRun == 4 ? pair >> 2 : pair >> 3) & (kRun - 1); };
    const int row0 = row_block * kOwnRows + wave * kWaveRows;
#pragma unroll
    for (int t = 0; t < kMT; ++t) {
        const float scale = kGated || !pair_weight ? 1.f : s_scale[32 * t + c];
#pragma unroll
        for (int u0 = 0; u0 < kNT; u0 += kAtOnce) {
#pragma unroll
            for (int u = u0; u < u0 + kAtOnce; ++u)
#pragma unroll
                for (int q = 0; q < (kGated ? 2 : 4); ++q) {
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float value = acc[t][u][4 * q + j];
                        v[j] = kGated ? glu_value(value, acc[t][u][(4 * q + j + 8) & 15], act, limit)
                                      : kMode == kMoePlain ? plain_act(value * scale, act) : value * scale;
                    }
                    const int at = (u - u0) * (kWaveRows / kNT) + 8 * q + 4 * hi;        // the first of the four rows
                    const int piece = (at * kBytes / 16) ^ turn(c);
                    if constexpr (kBytes == 4) {
                        mine[c * kRun + piece] = __builtin_bit_cast(uint4, float4{v[0], v[1], v[2], v[3]});
                    } else {
                        uint2 packed;
                        packed.x = bf16_bits_from_float(v[0]) | (static_cast<uint32_t>(bf16_bits_from_float(v[1])) << 16);
                        packed.y = bf16_bits_from_float(v[2]) | (static_cast<uint32_t>(bf16_bits_from_float(v[3])) << 16);
                        reinterpret_cast<uint2*>(mine)[2 * (c * kRun + piece) + hi] = packed;
                    }
                }
            __builtin_amdgcn_wave_barrier();             // (the wave's own writes, read by its other lanes: in order in shared memory)
#pragma unroll
            for (int i = 0; i < kRun / 2; ++i) {
                const int pair = i * (kWave / kRun) + lane / kRun, piece = lane % kRun;
                const uint4 whole = mine[pair * kRun + (piece ^ turn(pair))];
                const int to = s_pairs[32 * t + pair], r = row0 + u0 * (kWaveRows / kNT) + piece * (16 / kBytes);
                if (to >= 0 && r < n) *reinterpret_cast<uint4*>(static_cast<char*>(y) + (static_cast<long>(to) * n + r) * kBytes) = whole;
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// 256 rows of the matrix a workgroup (gated: 128 and their up rows) where tiles are of 128 pairs and that leaves some 200 workgroups, by the tiles
// that are likely to be used: us, 256 and 128 rows: 32 experts of 2,048 x 768, first product, 100 pairs each (246 workgroups) 52 and 55, 240 pairs (456) 79 and 85; second, 240
// pairs 52 and 50, 400 pairs 70 and 80; 8 of 4,096 x 2,048, 150 pairs (208) 75 and 83; but 32 of 1,024 x 384, 100 pairs (198) 18.0 and 16.2; 16 of
// 2,048 x 1,024, 16 pairs (96) 31 and 26; second product of 8 of 1,024 x 4,096, 300 pairs (88) 43 and 35.
static bool many_rows(int tiles, int n, bool gated) { return static_cast<long>(tiles) * ceil_div(n, gated ? 128 : 256) >= 200; }

// A workgroup takes 256 columns of a row; a thread one column.
template <typename T>
__global__ void __launch_bounds__(256)
moe_combine_kernel(const float* __restrict__ pair_out, const int* __restrict__ chosen, const float* __restrict__ weight,
                   const T* __restrict__ x, const float* __restrict__ extra, float* __restrict__ out, int top, int experts,
                   int hidden) {
    const int row = blockIdx.x;
    const int c = blockIdx.y * 256 + threadIdx.x;
    if (c >= hidden) return;
    const int* ch = chosen + static_cast<long>(row) * top;
    const float* wt = weight + static_cast<long>(row) * top;
    const long at = static_cast<long>(row) * hidden + c;
    float sum = 0.f;
    for (int j = 0; j < top; ++j) {                       // in the order of the row's places, whatever the tiles were
        const int e = ch[j];
        if (e >= experts)
            sum += wt[j] * to_float(x[at]);               // hands the row on as it came
        else if (e >= 0)
            sum += pair_out[(static_cast<long>(row) * top + j) * hidden + c];
    }
    if (extra != nullptr) sum += extra[at];
    out[at] = sum;
}

}  // namespace leone

using namespace leone;

extern "C" int leone_moe_tile_pairs() { return kTilePairs; }
extern "C" int leone_route_max_outputs() { return kRouteSlots * kWave; }

extern "C" int leone_route_topk(const float* logits, const void* correction, int correction_dtype, int* chosen, float* weight,
                                int rows, int total, int top, int group_count, int group_keep, int score, int group_best,
                                int renorm, float weight_scale, hipStream_t stream) {
    LEONE_REQUIRE(logits && chosen && weight, "route_topk: null pointer");
    LEONE_REQUIRE((score == 0 || score == 1) && group_best >= 1 && (renorm == 0 || renorm == 1),
                  "route_topk: score kind %d, %d best of a group, renorm %d", score, group_best, renorm);
    LEONE_REQUIRE(rows > 0 && total > 0 && total <= kRouteSlots * kWave, "route_topk: rows %d, %d router outputs (at most %d)",
                  rows, total, kRouteSlots * kWave);
    LEONE_REQUIRE(top > 0 && top <= total, "route_topk: %d of %d outputs", top, total);
    LEONE_REQUIRE(!correction || correction_dtype == kF32 || correction_dtype == kBF16, "route_topk: unknown type of the correction");
    LEONE_REQUIRE(group_count >= 1 && total % group_count == 0 && group_keep >= 1 && group_keep <= group_count,
                  "route_topk: %d groups (dividing %d outputs), %d kept", group_count, total, group_keep);
    const auto kernel = total <= kWave ? route_topk_kernel<1> : total <= 2 * kWave ? route_topk_kernel<2>
                        : total <= 4 * kWave ? route_topk_kernel<4> : route_topk_kernel<kRouteSlots>;
    kernel<<<rows, kWave, 0, stream>>>(logits, AnyVec{correction, correction_dtype}, chosen, weight, total, top, group_count, group_keep,
                                       RouteRule{score, group_best, renorm, weight_scale});
    LEONE_LAUNCH_CHECK("route_topk");
    return 0;
}

// leone_route_topk and leone_moe_plan in one launch (one workgroup: for steps of few rows).  `always`: the last so many
// of the `experts` are taken by every row with weight 1 (a shared expert cut to the experts' size): chosen and weight are
// [rows, top + always], a row's choices and then these; a chosen router output that stands for no matrix (from
// experts - always on in the router's numbering) is numbered from `experts` on.
extern "C" int leone_route_plan(const float* logits, const void* correction, int correction_dtype, int* chosen, float* weight,
                                int rows, int total, int top, int group_count, int group_keep, int experts, int* tile_expert,
                                int* tile_pairs, int max_tiles, int tile, int always, int score, int group_best, int renorm,
                                float weight_scale, hipStream_t stream) {
    LEONE_REQUIRE((score == 0 || score == 1) && group_best >= 1 && (renorm == 0 || renorm == 1),
                  "route_plan: score kind %d, %d best of a group, renorm %d", score, group_best, renorm);
    LEONE_REQUIRE(always >= 0 && always < experts, "route_plan: %d of %d experts for every row", always, experts);
    LEONE_REQUIRE(logits && chosen && weight && tile_expert && tile_pairs, "route_plan: null pointer");
    LEONE_REQUIRE(rows > 0 && rows <= 256 && total > 0 && total <= kRouteSlots * kWave, "route_plan: rows %d (at most 256), %d router outputs",
                  rows, total);
    LEONE_REQUIRE(top > 0 && top <= total, "route_plan: %d of %d outputs", top, total);
    LEONE_REQUIRE(!correction || correction_dtype == kF32 || correction_dtype == kBF16, "route_plan: unknown type of the correction");
    LEONE_REQUIRE(group_count >= 1 && total % group_count == 0 && group_keep >= 1 && group_keep <= group_count,
                  "route_plan: %d groups (dividing %d outputs), %d kept", group_count, total, group_keep);
    LEONE_REQUIRE(experts > 0 && experts <= 1024, "route_plan: %d experts (at most 1024)", experts);
    LEONE_REQUIRE(tile == kTilePairs || tile == 16 || tile == kBigPairs || tile == kWidePairs, "route_plan: tiles of %d pairs", tile);
    const long pairs = static_cast<long>(rows) * (top + always);
    const long needed = pairs / tile + experts;
    LEONE_REQUIRE(max_tiles >= (needed < pairs ? needed : pairs), "route_plan: %d tiles cannot hold %ld pairs of %d experts", max_tiles,
                  pairs, experts);
    const auto kernel = total <= kWave ? route_plan_kernel<1> : total <= 2 * kWave ? route_plan_kernel<2>
                        : total <= 4 * kWave ? route_plan_kernel<4> : route_plan_kernel<kRouteSlots>;
    kernel<<<1, 1024, 0, stream>>>(logits, AnyVec{correction, correction_dtype}, chosen, weight, rows, total, top, group_count, group_keep,
                                   experts, tile_expert, tile_pairs, max_tiles, tile, always, RouteRule{score, group_best, renorm, weight_scale});
    LEONE_LAUNCH_CHECK("route_plan");
    return 0;
}

// Whether tiles of 128 pairs that read the matrices' copies take 256 rows of a matrix a workgroup, not 128 (see many_rows).
extern "C" int leone_moe_many_rows(int max_tiles, int experts, int n, int gated) { return many_rows(max_tiles - experts / 2, n, gated == kMoeGated); }

extern "C" int leone_moe_one_chunk_ahead(int experts, int gated, int n, int k) {
    return one_chunk_ahead(experts, ceil_div(n, gated == kMoeGated ? kBigRows / 2 : kBigRows), n, k);
}

extern "C" int leone_moe_plan(const int* chosen, int pairs, int experts, int* tile_expert, int* tile_pairs, int max_tiles,
                              int tile, hipStream_t stream) {
    LEONE_REQUIRE(tile == kTilePairs || tile == 16 || tile == kBigPairs || tile == kWidePairs, "moe_plan: tiles of %d pairs", tile);
    LEONE_REQUIRE(chosen && tile_expert && tile_pairs, "moe_plan: null pointer");
    LEONE_REQUIRE(pairs > 0 && experts > 0 && experts <= 1024, "moe_plan: %d pairs, %d experts (at most 1024)", pairs, experts);
    const long needed = static_cast<long>(pairs) / tile + experts;
    LEONE_REQUIRE(max_tiles >= (needed < pairs ? needed : pairs), "moe_plan: %d tiles cannot hold %d pairs of %d experts", max_tiles,
                  pairs, experts);
    moe_plan_kernel<<<1, 1024, 0, stream>>>(chosen, pairs, experts, tile_expert, tile_pairs, max_tiles, tile);
    LEONE_LAUNCH_CHECK("moe_plan");
    return 0;
}

// gated != 0: x [rows, k], w [experts, 2, n, k], y [pairs, n] of dtype = act(gate) * up (act: GateAct).
// gated == 0: x [pairs, k], w [experts, n, k], y float32 [pairs, n] = pair_weight[pair] * product (null: 1).
// gated == 2: x [rows, k], w [experts, n, k], y [pairs, n] of dtype = act(pair_weight[pair] * product) (null: 1).
// experts: how many there are, for the rule that looks at how many workgroups their matrices give (see one_chunk_ahead).
// tile: pairs a tile holds, as leone_moe_plan was told: leone_moe_tile_pairs() for the kernel that takes any type and
// size; 16, 64 or 128 for the matrix-core kernels (bfloat16, n and k multiples of 8).
static int run_moe_product(const void* x, const void* w, int w_tiled, void* y, const float* pair_weight, int dtype, int gated,
                           const int* tile_expert, const int* tile_pairs, int max_tiles, int tile, int experts, int top, int n, int k,
                           int act, float limit, hipStream_t stream) {
    LEONE_REQUIRE(!w_tiled || (n % 16 == 0 && (tile == 16 ? k % 32 == 0 : (tile == kBigPairs || tile == kWidePairs) && k % 64 == 0)),
                  "moe_product: matrices in tiles do not go with tiles of %d pairs and sizes %d x %d", tile, n, k);
    LEONE_REQUIRE(gated >= kMoeDown && gated <= kMoePlain, "moe_product: unknown kind of product %d", gated);
    LEONE_REQUIRE(act == kGateSilu || act == kGateGeluTanh || (act == kGateClampedSwish && limit > 0.f && gated != kMoePlain) ||
                      (act == kActReluSquared && gated != kMoeGated),
                  "moe_product: unknown activation %d (limit %g)", act, limit);
    if (tile != kTilePairs) {
        LEONE_REQUIRE(tile == 16 || tile == kBigPairs || tile == kWidePairs, "moe_product: tiles of %d pairs", tile);
        LEONE_REQUIRE(dtype == kBF16 && k % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0,
                      "moe_product: the matrix-core kernel takes bfloat16 with an inner size that is a multiple of 8, not %d", k);
        LEONE_REQUIRE(x && w && y && tile_expert && tile_pairs, "moe_product: null pointer");
        LEONE_REQUIRE(max_tiles > 0 && top > 0 && n > 0 && k > 0, "moe_product: %d tiles, sizes %d x %d", max_tiles, n, k);
        if (tile == 16) {
            const dim3 grid(max_tiles, ceil_div(n, 16));
            LEONE_REQUIRE(grid.y <= 65535, "moe_product: %d rows of a matrix are too many", n);
            const bool streamed = k <= kStreamedInner;
#define LEONE_MOE_LAID(MODE, LAYOUT)                                                                                           \
    moe_product_stream_kernel<MODE, LAYOUT><<<grid, kMoeThreads, 0, stream>>>(                                                 \
        static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), y, pair_weight, tile_expert, tile_pairs, top, n, k, act, limit)
#define LEONE_MOE_STREAM(MODE)                                                                                                 \
    (w_tiled ? LEONE_MOE_LAID(MODE, kMoeTiled) : streamed ? LEONE_MOE_LAID(MODE, kMoeStreamed) : LEONE_MOE_LAID(MODE, kMoeKept))
            if (gated == kMoeGated) LEONE_MOE_STREAM(kMoeGated);
            else if (gated == kMoePlain) LEONE_MOE_STREAM(kMoePlain);
            else LEONE_MOE_STREAM(kMoeDown);
#undef LEONE_MOE_STREAM
#undef LEONE_MOE_LAID
        } else if (w_tiled) {
            const bool many = tile == kWidePairs && leone_moe_many_rows(max_tiles, experts, n, gated);
            const int blocks = ceil_div(n, (gated == kMoeGated ? 64 : 128) * (many ? 2 : 1));
            const long places = static_cast<long>(ceil_div(max_tiles, 8 * kTogether)) * 8 * kTogether * blocks;
            LEONE_REQUIRE(places <= 0x7fffffffL, "moe_product: too many tiles");
            const int grid = static_cast<int>(places);
#define LEONE_MOE_MANY(MODE, MT, NT)                                                                                          \
    moe_product_many_kernel<MODE, MT, NT><<<grid, kMoeThreads, 0, stream>>>(                                                   \
        static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), y, pair_weight, tile_expert, tile_pairs, top, n, k, act, limit, max_tiles, blocks)
#define LEONE_MOE_PAIRS(MODE)                                                                                                  \
    (tile == kBigPairs ? LEONE_MOE_MANY(MODE, 2, 1) : many ? LEONE_MOE_MANY(MODE, 4, 2) : LEONE_MOE_MANY(MODE, 4, 1))
            if (gated == kMoeGated) LEONE_MOE_PAIRS(kMoeGated);
            else if (gated == kMoePlain) LEONE_MOE_PAIRS(kMoePlain);
            else LEONE_MOE_PAIRS(kMoeDown);
#undef LEONE_MOE_PAIRS
#undef LEONE_MOE_MANY
        } else {
            const int blocks = ceil_div(n, tile == kWidePairs ? kWideRows : gated == kMoeGated ? kBigRows / 2 : kBigRows);
            const long places = static_cast<long>(max_tiles) * blocks;
            LEONE_REQUIRE(places + 7 <= 0x7fffffffL, "moe_product: too many tiles");
            const int grid = static_cast<int>((places + 7) / 8 * 8), one_ahead = one_chunk_ahead(experts, blocks, n, k);
#define LEONE_MOE_TILED(KERNEL, MODE)                                                                                         \
    KERNEL<MODE><<<grid, kMoeThreads, 0, stream>>>(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), y, pair_weight,   \
                                                   tile_expert, tile_pairs, top, n, k, act, limit, max_tiles, blocks, one_ahead)
#define LEONE_MOE_TILES(MODE)                                                                                                 \
    (tile == kBigPairs ? LEONE_MOE_TILED(moe_product_tiled_kernel, MODE) : LEONE_MOE_TILED(moe_product_wide_kernel, MODE))
            if (gated == kMoeGated) LEONE_MOE_TILES(kMoeGated);
            else if (gated == kMoePlain) LEONE_MOE_TILES(kMoePlain);
            else LEONE_MOE_TILES(kMoeDown);
#undef LEONE_MOE_TILES
#undef LEONE_MOE_TILED
        }
        LEONE_LAUNCH_CHECK("moe_product");
        return 0;
    }
    LEONE_REQUIRE(dtype == kF32 || dtype == kBF16, "moe_product: unknown element type %d", dtype);
    LEONE_REQUIRE(x && w && y && tile_expert && tile_pairs, "moe_product: null pointer");
    LEONE_REQUIRE(max_tiles > 0 && top > 0 && n > 0 && k > 0, "moe_product: %d tiles, sizes %d x %d", max_tiles, n, k);
    const uintptr_t run = 8 * (dtype == kF32 ? sizeof(float) : sizeof(bf16_t));
    const int runs = k % 8 == 0 && reinterpret_cast<uintptr_t>(x) % run == 0 && reinterpret_cast<uintptr_t>(w) % run == 0;
    const dim3 grid(max_tiles, ceil_div(n, kMoeCols));
    LEONE_REQUIRE(grid.y <= 65535, "moe_product: %d rows of a matrix are too many", n);
#define LEONE_MOE(T, G)                                                                                                   \
    moe_product_kernel<T, G><<<grid, kMoeThreads, 0, stream>>>(static_cast<const T*>(x), static_cast<const T*>(w), y, pair_weight, \
                                                               tile_expert, tile_pairs, top, n, k, act, limit, runs)
    if (dtype == kF32) {
        if (gated == kMoeGated) LEONE_MOE(float, kMoeGated);
        else if (gated == kMoePlain) LEONE_MOE(float, kMoePlain);
        else LEONE_MOE(float, kMoeDown);
    } else {
        if (gated == kMoeGated) LEONE_MOE(bf16_t, kMoeGated);
        else if (gated == kMoePlain) LEONE_MOE(bf16_t, kMoePlain);
        else LEONE_MOE(bf16_t, kMoeDown);
    }
#undef LEONE_MOE
    LEONE_LAUNCH_CHECK("moe_product");
    return 0;
}

extern "C" int leone_moe_product(const void* x, const void* w, void* y, const float* pair_weight, int dtype, int gated,
                                 const int* tile_expert, const int* tile_pairs, int max_tiles, int tile, int experts, int top, int n,
                                 int k, int act, float limit, hipStream_t stream) {
    return run_moe_product(x, w, 0, y, pair_weight, dtype, gated, tile_expert, tile_pairs, max_tiles, tile, experts, top, n, k, act, limit, stream);
}

// The same for tiles of 16, 64 and 128 pairs with w as the copy [experts (, 2)][n / 16][k / 32][4][16][8]: element e of lane 16 g + c of step s of tile
// t is row 16 t + c's element 32 s + 8 g + e.  n a multiple of 16, k of 32 (of 64 beyond 16 pairs).
extern "C" int leone_moe_product_tiles(const void* x, const void* w, void* y, const float* pair_weight, int gated, const int* tile_expert,
                                       const int* tile_pairs, int max_tiles, int tile, int experts, int top, int n, int k, int act,
                                       float limit, hipStream_t stream) {
    LEONE_REQUIRE(tile != kTilePairs, "moe_product: matrices in tiles do not go with tiles of %d pairs", tile);
    return run_moe_product(x, w, 1, y, pair_weight, kBF16, gated, tile_expert, tile_pairs, max_tiles, tile, experts, top, n, k, act, limit, stream);
}

extern "C" int leone_moe_combine(const float* pair_out, const int* chosen, const float* weight, const void* x, int dtype,
                                 const float* extra, float* out, int rows, int top, int experts, int hidden, hipStream_t stream) {
    LEONE_REQUIRE(dtype == kF32 || dtype == kBF16, "moe_combine: unknown element type %d", dtype);
    LEONE_REQUIRE(pair_out && chosen && weight && x && out, "moe_combine: null pointer");
    LEONE_REQUIRE(rows > 0 && top > 0 && experts >= 0 && hidden > 0, "moe_combine: rows %d, top %d, hidden %d", rows, top, hidden);
    const dim3 grid(rows, ceil_div(hidden, 256));
    LEONE_REQUIRE(grid.y <= 65535, "moe_combine: rows of %d are too wide", hidden);
    if (dtype == kF32)
        moe_combine_kernel<float><<<grid, 256, 0, stream>>>(pair_out, chosen, weight, static_cast<const float*>(x), extra, out, top,
                                                            experts, hidden);
    else
        moe_combine_kernel<bf16_t><<<grid, 256, 0, stream>>>(pair_out, chosen, weight, static_cast<const bf16_t*>(x), extra, out, top,
                                                             experts, hidden);
    LEONE_LAUNCH_CHECK("moe_combine");
    return 0;
}
