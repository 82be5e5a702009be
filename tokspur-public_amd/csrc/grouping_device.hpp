// Device code shared by grouping.hip, gemm.hip and moe_few.hip: an expert's routes, the task list of the grouped GEMMs and the
// union records of a step of at most eight tokens.
#pragma once
#include "tsp_common.hpp"

namespace tsp {

// Inclusive sums over the 512 values of a block of 512 threads (one per thread), two or three sequences at once: each wave
// scans its 64 values with six shuffles, the eight wave totals meet in LDS (`totals`: 8 words per sequence), one barrier on
// the way in and one on the way out, where a step-by-step scan through LDS takes eighteen. Returns the scan at this thread;
// `grand[i]` receives the sum of all 512.
template <int N>
__device__ __forceinline__ void scan512(uint32_t (&v)[N], uint32_t (&grand)[N], uint32_t* totals) {
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
#pragma unroll
    for (int i = 0; i < N; ++i) {
#pragma unroll
        for (int step = 1; step < kWave; step <<= 1) {
            const uint32_t below = uint32_t(__shfl_up(int(v[i]), step, kWave));
            if (lane >= uint32_t(step)) v[i] += below;
        }
    }
    __syncthreads();  // whoever still reads `totals` from an earlier call has left
    if (lane == kWave - 1)
#pragma unroll
        for (int i = 0; i < N; ++i) totals[i * 8 + wave] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        uint32_t before = 0, all = 0;
#pragma unroll
        for (uint32_t w = 0; w < 8; ++w) { const uint32_t t = totals[i * 8 + w]; if (w < wave) before += t; all += t; }
        v[i] += before;
        grand[i] = all;
    }
}

// A workgroup of THREADS threads writes one expert's routes: token_map[e*T + k] = t*S + slot for the k-th token (ascending) that names e once,
// counts[e] = how many do. `wave_totals`: a word of LDS per wave.
template <uint32_t THREADS>
__device__ __forceinline__ void expert_routes_block(const uint32_t* __restrict__ ids, uint32_t* __restrict__ token_map, uint32_t* __restrict__ counts, uint32_t expert,
                                                    uint32_t experts, uint32_t selected, uint32_t tokens, uint32_t* error_word, uint32_t* wave_totals) {
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    uint32_t accumulated = 0, bad = 0;
    for (uint32_t base = 0; base < tokens; base += THREADS) {
        const uint32_t token = base + tid;
        uint32_t slot = 0xffffffffu, matches = 0;
        if (token < tokens) {
            const uint32_t* row = ids + uint64_t(token) * selected;
            if (selected % 2 == 0 && reinterpret_cast<uintptr_t>(ids) % 8 == 0) {  // 8-byte aligned rows of an even number of ids: half as many loads
                for (uint32_t i = 0; i < selected; i += 2) {
                    const uint2 pair = *reinterpret_cast<const uint2*>(row + i);
                    if (pair.x >= experts || pair.y >= experts) bad = TSP_ERRBIT_INDEX;
                    if (pair.x == expert) { slot = i; ++matches; }
                    if (pair.y == expert) { slot = i + 1; ++matches; }
                }
            } else {
                for (uint32_t i = 0; i < selected; ++i) {
                    const uint32_t id = row[i];
                    if (id >= experts) bad = TSP_ERRBIT_INDEX;
                    if (id == expert) { slot = i; ++matches; }
                }
            }
        }
        if (matches > 1) bad = TSP_ERRBIT_INDEX;
        const bool found = matches == 1;
        const uint64_t mask = __builtin_amdgcn_ballot_w64(found);
        const uint32_t prefix = __builtin_popcountll(mask & ((1ull << lane) - 1ull));
        if (lane == 0) wave_totals[wave] = __builtin_popcountll(mask);
        __syncthreads();
        uint32_t before = 0, chunk = 0;
        for (uint32_t w = 0; w < THREADS / kWave; ++w) { if (w < wave) before += wave_totals[w]; chunk += wave_totals[w]; }
        if (found) token_map[uint64_t(expert) * tokens + accumulated + before + prefix] = token * selected + slot;
        accumulated += chunk;
        __syncthreads();
    }
    if (tid == 0) counts[expert] = accumulated;
    publish_error(bad, error_word);
}

// The same counts of at most 512 tokens, for all experts, by one workgroup of 512 threads, which then need not wait for the experts' workgroups. What is
// wrong with the ids is theirs to report. `counted`: 2048 words of LDS, 16-byte aligned, the counts in the first 512; an expert has four
// counters, by lane, since lanes that add to the same one take turns.
__device__ __forceinline__ void count_routes_block(const uint32_t* __restrict__ ids, uint32_t experts, uint32_t selected, uint32_t tokens, uint32_t* counted) {
    const uint32_t tid = threadIdx.x;
    reinterpret_cast<uint4*>(counted)[tid] = uint4{0, 0, 0, 0};
    uint32_t id[16];
    if (tid < tokens) {
        const uint32_t* const row = ids + tid * selected;
        const bool pairs = selected % 2 == 0 && reinterpret_cast<uintptr_t>(ids) % 8 == 0;
#pragma unroll
        for (uint32_t i = 0; i < 16; i += 2) {
            if (i < selected && pairs) {
                const uint2 two = *reinterpret_cast<const uint2*>(row + i);
                id[i] = two.x; id[i + 1] = two.y;
            } else {
                if (i < selected) id[i] = row[i];
                if (i + 1 < selected) id[i + 1] = row[i + 1];
            }
        }
    }
    __syncthreads();
    if (tid < tokens) {
        bool wrong = id[0] >= experts;
#pragma unroll
        for (uint32_t i = 1; i < 16; ++i)
            if (i < selected) {
                wrong |= id[i] >= experts;
#pragma unroll
                for (uint32_t j = 0; j < i; ++j) wrong |= id[i] == id[j];
            }
        auto count = [&](uint32_t e) { atomicAdd(&counted[e * 4 + tid % 4], 1u); };
        if (!__builtin_amdgcn_ballot_w64(wrong)) {
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i)
                if (i < selected) count(id[i]);
        } else {  // an id counts if it is an expert's and no other of the token's
#pragma unroll 1
            for (uint32_t i = 0; i < selected; ++i) {
                const uint32_t mine = ids[tid * selected + i];
                uint32_t alike = 0;
#pragma unroll 1
                for (uint32_t j = 0; j < selected; ++j) alike += ids[tid * selected + j] == mine ? 1 : 0;
                if (mine < experts && alike == 1) count(mine);
            }
        }
    }
    __syncthreads();
    const uint4 four = reinterpret_cast<const uint4*>(counted)[tid];
    __syncthreads();
    counted[tid] = (four.x + four.y) + (four.z + four.w);
    __syncthreads();
}

// One block of 512 threads writes one list; experts <= 512. tiles(e) = ceil(min(counts[e], T) / tile), exclusive scan over
// the experts, task i of expert e is (e, i * tile); unused slots up to the bound are 0xFFFFFFFF. `totals`: LDS of
// the scans, eight words for each of two (three in the class lists).
// `every_token` appends ceil(tokens / tile) tasks (experts, i * tile) after the experts' own: an always-on expert whose rows
// are the tokens themselves (the bound grows by that many slots).
__device__ __forceinline__ void grouped_tasks_block(const uint32_t* __restrict__ counts, uint32_t* __restrict__ tasks, uint32_t tile,
                                                    uint32_t experts, uint32_t selected, uint32_t tokens, uint32_t* error_word,
                                                    uint32_t* totals, bool every_token = false) {
    const uint32_t tid = threadIdx.x;
    const uint32_t extra = every_token ? (tokens + tile - 1) / tile : 0;
    const uint32_t bound = tokens * selected / tile + experts + extra;
    uint32_t bad = 0;
    const uint32_t count = tid < experts ? counts[tid] : 0;
    if (count > tokens) bad = TSP_ERRBIT_INDEX;
    const uint32_t n = ((count < tokens ? count : tokens) + tile - 1) / tile;
    uint32_t scans[2] = {n, count}, sums[2];
    scan512(scans, sums, totals);
    const uint32_t total = sums[0], routes = sums[1];
    const uint32_t offset = scans[0] - n;
    for (uint32_t i = total + extra + tid; i < bound; i += 512) { tasks[2 + 2 * i] = 0xffffffffu; tasks[3 + 2 * i] = 0xffffffffu; }
    if (tid < experts)
        for (uint32_t i = 0; i < n; ++i)
            if (offset + i < bound) { tasks[2 + 2 * (offset + i)] = tid; tasks[3 + 2 * (offset + i)] = i * tile; }
    for (uint32_t i = tid; i < extra; i += 512)
        if (total + i < bound) { tasks[2 + 2 * (total + i)] = experts; tasks[3 + 2 * (total + i)] = i * tile; }
    if (tid == 0) {
        tasks[0] = total + extra < bound ? total + extra : bound;
        tasks[1] = routes;
        if (total + extra > bound || routes != tokens * selected) bad = TSP_ERRBIT_INDEX;
    }
    publish_error(bad, error_word);
}

// The tasks of a 64-row list sorted into two index lists by their number of rows: out[0] = tasks of at most 32 rows, out[1] =
// tasks of 33..64 rows, out[2 .. 2 + bound) the first kind's task indices in list order, out[2 + bound .. 2 + 2 bound) the
// second kind's. Of an expert's tasks only the last can have fewer than 64 rows, so the lists follow from the counts alone:
// the same block of 512 threads that wrote the task list writes them, from three more scans (experts <= 512).
__device__ __forceinline__ void task_class_lists_block(const uint32_t* __restrict__ counts, uint32_t* __restrict__ out, uint32_t experts,
                                                       uint32_t selected, uint32_t tokens, bool every_token, uint32_t* totals) {
    constexpr uint32_t tile = 64;
    const uint32_t tid = threadIdx.x;
    const uint32_t extra = every_token ? (tokens + tile - 1) / tile : 0;
    const uint32_t bound = tokens * selected / tile + experts + extra;
    const uint32_t count = tid < experts ? (counts[tid] < tokens ? counts[tid] : tokens) : 0;
    const uint32_t n = (count + tile - 1) / tile;
    const uint32_t small = n && count - (n - 1) * tile <= 32 ? 1 : 0;  // the last task is a small one
    uint32_t scans[3] = {n, small, n - small}, sums[3];
    scan512(scans, sums, totals);
    const uint32_t total = sums[0], total_small = sums[1], total_large = sums[2];
    const uint32_t first = scans[0] - n, first_small = scans[1] - small, first_large = scans[2] - (n - small);
    uint32_t* list_small = out + 2;
    uint32_t* list_large = out + 2 + bound;
    for (uint32_t i = 0; i < n; ++i) {
        if (first + i >= bound) break;
        if (small && i + 1 == n) list_small[first_small] = first + i;
        else list_large[first_large + i] = first + i;
    }
    const uint32_t extra_small = extra && tokens - (extra - 1) * tile <= 32 ? 1 : 0;
    for (uint32_t i = tid; i < extra; i += 512) {
        if (total + i >= bound) break;
        if (extra_small && i + 1 == extra) list_small[total_small] = total + i;
        else list_large[total_large + i] = total + i;
    }
    if (tid == 0) {
        const bool fits = total + extra <= bound;  // otherwise the task list itself is flagged as broken and nobody reads these
        out[0] = fits ? total_small + extra_small : 0;
        out[1] = fits ? total_large + extra - extra_small : 0;
    }
}

// The tasks of a 64-row list in the order in which a launch with a workgroup per (task, column tile) takes them: eight runs, one per XCD, of
// `order_pitch` places each; a place holds the whole task, so that a workgroup knows from its id alone where to look and asks once, or zero.
// A task of more than 32 rows takes about half as long again as one of fewer. Every XCD gets an eighth of either kind, the large ones at even distances
// among the small ones (products of the one beside the other's weights on their way), and its last `tail` are small: what is left running alone when
// the others have nothing more is short. 2048 tokens, 512 experts, gate/up: 2048 x 512 195 -> 190 us, 2560 x 640 287 -> 281 against list order; no tail 193
// and 281, all large ones first 200 and 294.
struct OrderedTask { uint32_t what, task; };  // what: 1 << 31 | rows << 16 | (first row / 64) << 10 | expert; task: index in the list
constexpr uint32_t order_pitch(uint32_t bound) { return bound / 8 + 2; }
// One block of 512 threads; experts <= 512, tokens <= 2048. `kinds`: 56 words of LDS, `totals` those of the scans. The thread of an expert of 2000 rows places
// thirty tasks one after the other, the longest chain of its launch: reciprocals made once where each place took two divisions (tasks_and_rows, 2048 tokens: 2560 columns
// 9.2 -> 8.3 us, 2048 8.1 -> 7.8, 1024 and 64 experts 6.1 -> 5.8; without the order 8.0, 8.4 and 5.4).
__device__ __forceinline__ void task_order_block(const uint32_t* __restrict__ counts, OrderedTask* __restrict__ out, uint32_t tail, uint32_t experts,
                                                 uint32_t selected, uint32_t tokens, bool every_token, uint32_t* totals, uint32_t* kinds) {
    constexpr uint32_t tile = 64;
    const uint32_t tid = threadIdx.x;
    const uint32_t extra = every_token ? (tokens + tile - 1) / tile : 0;
    const uint32_t bound = tokens * selected / tile + experts + extra, pitch = order_pitch(bound);
    const uint32_t raw = tid < experts ? counts[tid] : 0, count = raw < tokens ? raw : tokens;
    const uint32_t n = (count + tile - 1) / tile;
    const uint32_t small = n && count - (n - 1) * tile <= 32 ? 1 : 0;
    uint32_t scans[3] = {n, small, raw}, sums[3];
    scan512(scans, sums, totals);
    const uint32_t extra_small = extra && tokens - (extra - 1) * tile <= 32 ? 1 : 0;
    const uint32_t total = sums[0], all_small = sums[1] + extra_small, all_large = total + extra - all_small;
    const uint32_t first = scans[0] - n, first_small = scans[1] - small, first_large = first - first_small;
    const bool whole = sums[2] == tokens * selected && total + extra <= bound;  // else the list's block flags the batch, and no task is taken up
    // XCD x has the small tasks from ceil(x all / 8) on and the large ones likewise
    auto begin = [](uint32_t all, uint32_t x) { return (all * x + 7) / 8; };
    struct Run { uint32_t small0, large0, early, large; float per_early, per_large; };  // early: small tasks ahead of the tail; per: one over their number
    Run* const runs = reinterpret_cast<Run*>(kinds);
    if (tid < 8) {
        const uint32_t s0 = begin(all_small, tid), l0 = begin(all_large, tid), s = begin(all_small, tid + 1) - s0;
        const uint32_t early = s > tail ? s - tail : 0, large = begin(all_large, tid + 1) - l0;
        runs[tid] = Run{s0, l0, early, large, 1.0f / float(early), 1.0f / float(large)};
        kinds[48 + tid] = whole ? s + large : 0;
    }
    __syncthreads();
    // floor(a / b) from b's rounded reciprocal: exact where a < 2^16 and b < 2^9, and for a = 8 rank, rank < b < 2^14 (all of them tried)
    auto over = [](uint32_t a, float per_b) { return uint32_t((float(a) + 0.5f) * per_b); };
    const float per_small = 1.0f / float(all_small), per_large = 1.0f / float(all_large);
    auto put_small = [&](uint32_t rank, OrderedTask t) {
        const uint32_t x = over(rank * 8, per_small);
        const Run run = runs[x];
        const uint32_t i = rank - run.small0;
        uint32_t before = run.large;  // large ones ahead of this one
        if (i < run.early) { before = over((i + 1) * run.large + run.early - 1, run.per_early); before = before < run.large ? before : run.large; }
        out[x * pitch + i + before] = t;
    };
    auto put_large = [&](uint32_t rank, OrderedTask t) {
        const uint32_t x = over(rank * 8, per_large);
        const Run run = runs[x];
        const uint32_t i = rank - run.large0;
        out[x * pitch + over(i * (run.large + run.early), run.per_large)] = t;
    };
    auto ordered = [&](uint32_t expert, uint32_t i, uint32_t rows, uint32_t task) { return OrderedTask{1u << 31 | (rows < tile ? rows : tile) << 16 | i << 10 | expert, task}; };
    if (whole) {
        for (uint32_t i = 0; i < n; ++i) {
            const OrderedTask t = ordered(tid, i, count - i * tile, first + i);
            if (small && i + 1 == n) put_small(first_small, t);
            else put_large(first_large + i, t);
        }
        for (uint32_t i = tid; i < extra; i += 512) {
            const OrderedTask t = ordered(experts, i, tokens - i * tile, total + i);
            if (extra_small && i + 1 == extra) put_small(sums[1], t);
            else put_large(total - sums[1] + i, t);
        }
    }
    for (uint32_t x = tid / kWave; x < 8; x += 512 / kWave)
        for (uint32_t i = kinds[48 + x] + tid % kWave; i < pitch; i += kWave) out[x * pitch + i] = OrderedTask{0, 0};
}

// The union records of at most 128 routes (T <= 8 tokens x S <= 16 slots): records (expert, <= cap routes) in first-use
// order. Block layout in 32-bit words: [0..7] header, +8 experts[128], +136 counts[128], +264 tokens[128][8],
// +1288 routes[128][8]. Thread f < 128 owns flat route f and brings its expert id (`mine`, anything when f >= T S); threads
// from 128 on help clear the scratch and keep the barriers company. `scratch`: kUnionScratchWords of LDS, 16-byte aligned.
// `store(word, value)` puts a word of the block wherever the caller wants it. Returns false, with the header zeroed and
// `raise()` called by thread 0, when the shape or an id is out of range. Uniform over the workgroup; every thread must call.
//
// A route's rank among the routes of its expert is a population count: every expert has a 128-bit set of its routes (bit f:
// route f), filled by LDS atomics whose result does not depend on their order, and route f counts the bits below its own. The
// route that opened a record is found the same way, as the n-th set bit of the expert's set, so nothing scans the routes.
constexpr uint32_t kUnionScratchWords = 512 * 4 + 128 + 4;
__device__ __forceinline__ uint32_t nth_set_bit(uint32_t word, uint32_t n) {  // position of the (n + 1)-th set bit; it must exist
    uint32_t pos = 0;
#pragma unroll
    for (uint32_t half = 16; half >= 1; half >>= 1) {
        const uint32_t low = word & ((1u << half) - 1u), in_low = __builtin_popcount(low);
        if (n < in_low) { word = low; } else { n -= in_low; word >>= half; pos += half; }
    }
    return pos;
}
template <typename Store, typename Raise>
__device__ __forceinline__ bool union_block(uint32_t mine, uint32_t f, uint32_t threads, uint32_t experts, uint32_t selected, uint32_t tokens,
                                            uint32_t hidden, uint32_t channels, uint32_t* scratch, Store store, Raise raise) {
    uint32_t* const sets = scratch;                  // [512][4]
    uint32_t* const record_of = scratch + 2048;      // [128]: the record a route opened
    uint32_t* const wave_leaders = scratch + 2176;   // [2]
    uint32_t* const any_bad = scratch + 2178;
    const uint32_t total = tokens * selected;
    const bool shape_ok = experts && experts <= 512 && experts % 2 == 0 && selected && selected <= 16 && selected <= experts &&
                          tokens && tokens <= 8 && hidden && channels;
    for (uint32_t i = f; i < 2048; i += threads) sets[i] = 0;
    if (f == 0) *any_bad = shape_ok ? 0u : 1u;
    __syncthreads();
    const bool live = shape_ok && f < total;
    if (live) {
        if (mine >= experts) *any_bad = 1u;
        else atomicOr(&sets[mine * 4 + f / 32], 1u << (f % 32));
    }
    __syncthreads();
    if (*any_bad) {
        if (f < 8) store(f, 0u);
        if (f == 0) raise();
        return false;
    }
    const uint32_t cap = tokens <= 4 ? 4u : 8u;
    uint32_t set[4] = {0, 0, 0, 0}, rank = 0, same = 0;
    if (live) {
        const uint4 four = *reinterpret_cast<const uint4*>(&sets[mine * 4]);
        set[0] = four.x; set[1] = four.y; set[2] = four.z; set[3] = four.w;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            same += __builtin_popcount(set[w]);
            const uint32_t below = w < f / 32 ? set[w] : w == f / 32 ? set[w] & ((1u << (f % 32)) - 1u) : 0u;
            rank += __builtin_popcount(below);
        }
    }
    const bool leader = live && rank % cap == 0;
    const uint64_t mask = __builtin_amdgcn_ballot_w64(leader);
    const uint32_t lane = f % kWave, wave = f / kWave;
    if (lane == 0 && wave < 2) wave_leaders[wave] = __builtin_popcountll(mask);
    __syncthreads();
    const uint32_t record = (wave ? wave_leaders[0] : 0u) + __builtin_popcountll(mask & ((1ull << lane) - 1ull));
    const uint32_t records = wave_leaders[0] + wave_leaders[1];
    if (leader) record_of[f] = record;
    __syncthreads();
    if (live) {
        uint32_t rec = record;
        if (!leader) {
            // my record is the one opened by the route of my expert whose rank is rank - rank % cap
            uint32_t n = rank - rank % cap, opener = 0;
            bool found = false;
#pragma unroll
            for (uint32_t w = 0; w < 4; ++w) {
                const uint32_t here = __builtin_popcount(set[w]);
                if (!found && n < here) { opener = 32 * w + nth_set_bit(set[w], n); found = true; }
                if (!found) n -= here;
            }
            rec = record_of[opener];
        }
        const uint32_t slot = rank % cap;
        store(264 + rec * 8 + slot, f / selected);
        store(1288 + rec * 8 + slot, f);
        if (leader) {
            const uint32_t members = same - rank < cap ? same - rank : cap;
            store(8 + rec, mine);
            store(136 + rec, members);
            for (uint32_t k = members; k < 8; ++k) { store(264 + rec * 8 + k, f / selected); store(1288 + rec * 8 + k, f); }
        }
    }
    if (f == 0) {
        store(0, (hidden + 7) / 8); store(1, records); store(2, 1u);
        store(3, (channels + 15) / 16); store(4, records); store(5, 1u);
        store(6, records); store(7, 0u);
    }
    return true;
}

}  // namespace tsp
